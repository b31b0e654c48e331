"""GEMM tile choices (needs an MI355X): row and column counts on both sides of every block edge (32, 64,
128, 256) and slot counts that move the choice between the K-sliced and the ring kernels, every output
against the oracle.  tests/test_gemm_blocks.py asserts which blocks the sizes reach."""
import dataclasses

import numpy as np
import pytest

from aideen_amd import synth
from aideen_amd.backend import GpuDeqBackend
from test_gpu_parity import ATOL, RTOL, assert_forward_parity

pytestmark = pytest.mark.gpu

# (d, H, V, B, T): the Q|K|V, W_o, signal, readout and LM-head products of B * T rows
SHAPES = [
    (64, 1, 65, 1, 5),      # fewer steps of K than waves
    (64, 4, 31, 1, 31),     # one partial row block, one partial column block
    (64, 16, 129, 1, 33),   # one row past a 32-row block
    (256, 8, 300, 1, 24),   # the few-row head's 128-column blocks
    (192, 8, 65, 1, 128),   # whole blocks, narrow head
    (128, 2, 257, 1, 129),  # one row and one column past a block
    (320, 3, 300, 1, 65),   # K not a power of two, H not a power of two
    (64, 2, 8300, 1, 33),   # the 64x256 head, one row past the few-row kernel and a partial last block
    (64, 2, 8300, 1, 64),   # the same, whole row blocks
    (256, 8, 16500, 1, 97),  # a wide head on 128x128 blocks
    (192, 16, 513, 3, 171),  # 64x128 ring Q|K|V and head, 32x64 K-sliced W_o
    (512, 8, 130, 1, 250),  # 128x128 ring Q|K|V, 32x64 K-sliced W_o
    (192, 8, 130, 1, 810),  # 64x64 K-sliced Q|K|V, 64x128 ring W_o
    (256, 16, 130, 1, 777),  # 128x128 ring W_o
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("flags", [0, synth.F_GEMM_BF16X3], ids=["f16x3", "bf16x3"])
def test_tiles_match_oracle(shape, flags):
    from oracle import pyoracle
    d, H, V, B, T = shape
    mc = synth.ModelConfig(d=d, H=H, V=V, N=4, max_iters=3, eps=0.0, qk_bias=True, flags=synth.F_SCAN_SELECTIVE | flags)
    w = synth.make_token_sensitive_weights(mc)
    toks = synth.make_tokens("uniform", B, T, V, seed=1)
    be = GpuDeqBackend(mc, B, T)
    be.upload_weights(w)
    got = be.forward(toks)
    be.close()
    ref = pyoracle.Oracle(dataclasses.replace(mc, flags=synth.F_SCAN_SELECTIVE), w).forward(toks, nthreads=8)
    for k in ("h_star", "pooled", "logits", "scan_y", "scan_state"):
        np.testing.assert_allclose(got[k], ref[k], rtol=RTOL, atol=ATOL, err_msg=k)
    # the fused arg-max is the last-max of the stored logits
    lg = got["logits"].reshape(-1, V)
    assert np.array_equal(got["argmax"].ravel(), V - 1 - np.argmax(lg[:, ::-1], axis=1))


# tokens on both sides of the attention's and the update's few-token limits, padded slot counts and
# rows beyond 1024 floats
@pytest.mark.parametrize("d,H,n", [(64, 3, 385), (128, 5, 641), (64, 8, 1024), (64, 8, 1025), (192, 12, 128),
                                   (128, 12, 129), (64, 16, 256), (64, 16, 257), (320, 6, 1030), (320, 8, 24),
                                   (384, 5, 70), (448, 8, 33), (448, 16, 9), (512, 6, 24), (1024, 16, 40),
                                   (1536, 3, 70), (2048, 2, 129), (2048, 9, 12)])
def test_token_limits_match_oracle(d, H, n):
    from oracle import pyoracle
    mc = synth.ModelConfig(d=d, H=H, V=33, N=1, max_iters=2, eps=0.0)
    w = synth.make_token_sensitive_weights(mc)
    toks = synth.make_tokens("uniform", 1, n, mc.V, seed=1)
    be = GpuDeqBackend(mc, 1, n)
    be.upload_weights(w)
    got = be.forward(toks, want=("h_star", "iters"))
    be.close()
    # the tokens of one id are alike: every row against the oracle's solve of its id
    ids, inv = np.unique(toks[0], return_inverse=True)
    ref = pyoracle.Oracle(mc, w).forward(ids[None].astype(np.int32), nthreads=8, want_scan=False)
    np.testing.assert_allclose(got["h_star"][0], ref["h_star"][0][inv], rtol=RTOL, atol=ATOL)
    assert (got["iters"] == 2).all()


# 64x128 blocks throughout; Q|K|V alone on 128x256; every product on 128x256
BF16_SHAPES = [(128, 8, 257, 1, 1500), (256, 16, 1025, 3, 331), (256, 16, 2100, 1, 3001)]


@pytest.mark.parametrize("shape", BF16_SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_bf16_blocks_match_fp32_gemms(shape):
    """bf16-input products on the ring blocks up to 128x256 (partial last row and column blocks) against
    the fp32 products of the same model: one bf16 rounding of each operand, 2^-8 relative a product, well
    inside 2e-2 of outputs of order one after two contracting steps."""
    d, H, V, B, T = shape
    toks = synth.make_tokens("uniform", B, T, V, seed=1)
    got = {}
    for f in (synth.F_GEMM_BF16, synth.F_GEMM_FP32):
        mc = synth.ModelConfig(d=d, H=H, V=V, N=1, max_iters=2, eps=0.0, flags=synth.F_SCAN_SELECTIVE | f)
        be = GpuDeqBackend(mc, B, T)
        be.upload_weights(synth.make_token_sensitive_weights(mc))
        got[f] = be.forward(toks, want=("h_star", "logits", "argmax"))
        be.close()
    a, b = got[synth.F_GEMM_BF16], got[synth.F_GEMM_FP32]
    for k in ("h_star", "logits"):
        assert np.abs(a[k] - b[k]).max() <= 2e-2 * max(1.0, np.abs(b[k]).max()), k
    lg = a["logits"].reshape(-1, V)
    assert np.array_equal(a["argmax"].ravel(), V - 1 - np.argmax(lg[:, ::-1], axis=1))


# more than 128 tokens per slot at 16 slots: the update with a wave per token, unrolled over 16 slots up
# to 512 floats and walking them at run time beyond, its L2 exit and active list among them
@pytest.mark.parametrize("d,n,flags,eps", [(64, 2049, 0, 0.0), (128, 2200, synth.F_RESID_L2, 1e-4),
                                           (512, 2100, 0, 1e-4), (1024, 2050, synth.F_RESID_L2, 1e-4),
                                           (1024, 2077, 0, 0.0)])
def test_many_tokens_of_16_slots_match_oracle(d, n, flags, eps):
    from oracle import pyoracle
    mc = synth.ModelConfig(d=d, H=16, V=33, N=1, max_iters=20 if eps else 2, eps=eps, flags=flags)
    w = synth.make_token_sensitive_weights(mc)
    toks = synth.make_tokens("uniform", 1, n, mc.V, seed=1)
    be = GpuDeqBackend(mc, 1, n)
    be.upload_weights(w)
    got = be.forward(toks, want=("h_star", "iters", "converged"))
    be.close()
    ids, inv = np.unique(toks[0], return_inverse=True)
    ref = pyoracle.Oracle(mc, w).forward(ids[None].astype(np.int32), nthreads=8, want_scan=False)
    assert_forward_parity({k: v[0] for k, v in got.items()}, {k: ref[k][0][inv] for k in ("h_star", "iters", "converged")})


# (d, H, T, few, many): sequences of T tokens solved in batches of `few` and of `many`, both up to 32
# rows or both above: 256 rows beside 2304 as one document window beside a throughput batch
EXIT_SHAPES = [(512, 8, 256, 1, 9), (192, 8, 128, 1, 17), (128, 4, 2048, 1, 3), (1024, 16, 177, 1, 3), (320, 6, 9, 5, 40),
               (256, 8, 5, 1, 6), (64, 16, 1, 5, 32)]


@pytest.mark.parametrize("shape", EXIT_SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("flags", [0, synth.F_GEMM_BF16X3, synth.F_GEMM_BF16], ids=["f16x3", "bf16x3", "bf16"])
def test_exit_steps_do_not_depend_on_the_batch(shape, flags):
    """Tokens exit on a tolerance: a sequence's fixed points and iteration counts are the same bits
    whatever else is solved beside it, since a residual within rounding of the tolerance would
    otherwise move a token by one update."""
    check_exit_steps(shape, flags=synth.F_SCAN_SELECTIVE | flags, eps=1e-4)


@pytest.mark.parametrize("shape,kw", [
    ((512, 8, 256, 1, 9), dict(anderson_m=3, sigma=0.7, eps=1e-3)), ((128, 4, 64, 1, 40), dict(anderson_m=4, eps=1e-3)),
    ((1024, 4, 50, 1, 12), dict(anderson_m=3, eps=1e-3)), ((512, 8, 256, 1, 9), dict(flags=synth.F_RESID_L2, eps=1e-4)),
    ((512, 8, 256, 1, 9), dict(flags=synth.F_RESID_RELRMS | synth.F_HOMEOSTATIC_EXIT, eps=1e-4)),
    ((512, 8, 256, 1, 9), dict(flags=synth.F_RESID_RELRMS | synth.F_HOMEOSTATIC_EXIT, eps=0.0)),
    ((1536, 5, 60, 1, 8), dict(eps=1e-4))], ids=["anderson", "narrow", "wide-anderson", "l2", "plateau", "plateau-alone", "wide"])
def test_exit_forms_do_not_depend_on_the_batch(shape, kw):
    check_exit_steps(shape, **kw)


def check_exit_steps(shape, **kw):
    d, H, T, few, many = shape
    mc = synth.ModelConfig(d=d, H=H, V=97, N=1, max_iters=16, **kw)
    w = synth.make_token_sensitive_weights(mc)
    toks = synth.make_tokens("uniform", many, T, mc.V, seed=1)
    be = GpuDeqBackend(mc, many, T)
    be.upload_weights(w)
    want = ("h_star", "iters", "converged")
    a, b = be.forward(toks[:few], want=want), be.forward(toks, want=want)
    be.close()
    for k in want:
        assert np.array_equal(a[k], b[k][:few]), k


# batches of `few` and of `many`, their rows (and B * T signal rows) both up to 32 or both above
@pytest.mark.parametrize("d,H,T,few,many", [(128, 4, 4, 5, 8), (512, 8, 2, 33, 300)])
def test_memory_exits_do_not_depend_on_the_batch(d, H, T, few, many):
    """The memory-coupled solve, where a position's history also goes through W_hist and the readout."""
    mc = synth.ModelConfig(d=d, H=H, V=97, N=1, max_iters=16, eps=1e-4, flags=synth.F_MEMORY)
    w = {**synth.make_token_sensitive_weights(mc), **synth.make_hist_weights(mc, seed=11, strong=True)}
    toks = synth.make_tokens("uniform", many, T, mc.V, seed=1)
    be = GpuDeqBackend(mc, many, T)
    be.upload_weights(w)
    want = ("h_star", "iters", "scan_y")
    a, b = be.forward(toks[:few], want=want), be.forward(toks, want=want)
    be.close()
    for k in want:
        assert np.array_equal(a[k], b[k][:few]), k


@pytest.mark.parametrize("d,V", [(192, 300), (512, 8300), (1024, 515)])
def test_few_row_logits_do_not_depend_on_the_batch(d, V):
    """The LM head up to 32 rows sums K in one order, the shares of the few-row kernel's waves: a
    row's logits are the same bits at 3, 24 and 32 rows.  One slot and an exit test, so that
    everything before the head is the same bits too (the softmax over one slot is 1)."""
    mc = synth.ModelConfig(d=d, H=1, V=V, N=1, max_iters=3, eps=1e-4)
    toks = synth.make_tokens("uniform", 32, 1, V, seed=1)
    be = GpuDeqBackend(mc, 32, 1)
    be.upload_weights(synth.make_token_sensitive_weights(mc))
    got = [be.forward(toks[:n], want=("pooled", "logits", "argmax")) for n in (3, 24, 32)]
    be.close()
    for g in got[1:]:
        for k in ("pooled", "logits", "argmax"):
            assert np.array_equal(g[k][:3], got[0][k]), k
