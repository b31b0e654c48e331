"""The persistent 256x256 blocks with partial last row and column blocks (needs an MI355X): every
product of 3500 tokens at 8 slots of 512 and a vocabulary of 4100, against the oracle.  The tokens are
of a few ids, whose fixed points the oracle solves once."""
import dataclasses

import numpy as np
import pytest

from aideen_amd import synth
from aideen_amd.backend import GpuDeqBackend, gemm_blocks
from test_gpu_graph import capture_and_replay
from test_gpu_parity import ATOL, RTOL, assert_forward_parity, last_max
from test_gpu_range import G, scaled_model

pytestmark = pytest.mark.gpu

D, H, V, B, T = 512, 8, 4100, 28, 125  # 13 whole row blocks of 256 and 172 rows


def assert_reached(mc):
    for stage in ("signal_gemm", "qkv_gemm", "wo_gemm", "lmhead_gemm", "readout_gemm"):
        blk = gemm_blocks(mc, stage, B * T, mc.eps > 0)
        assert blk[:2] == (256, 256), (stage, blk)
        if stage in ("wo_gemm", "lmhead_gemm") and not mc.flags & synth.F_GEMM_BF16X3:
            assert blk[3] == 1, stage


def few_ids(n, seed):
    rng = np.random.default_rng(seed)
    return rng.choice(V, n, replace=False)[rng.integers(0, n, (B, T))].astype(np.int32)


def by_id(o, toks):
    """The oracle's forward of every token of toks (any shape), each id solved once."""
    ids, inv = np.unique(toks, return_inverse=True)
    ref = o.forward(ids[None].astype(np.int32), nthreads=8, want_scan=False)
    return {k: ref[k][0][inv.reshape(toks.shape)] for k in ("h_star", "pooled", "logits", "argmax", "iters", "converged")}


@pytest.mark.parametrize("flags,anderson_m", [(0, 0), (0, 3), (synth.F_GEMM_BF16X3, 0)], ids=["f16x3", "anderson", "bf16x3"])
def test_every_output_matches_oracle(oracle_lib, flags, anderson_m):
    kw = dict(anderson_m=3, eps=0.0, max_iters=6) if anderson_m else {}
    mc = synth.ModelConfig(d=D, H=H, V=V, N=4, flags=synth.F_SCAN_SELECTIVE | flags, **kw)
    assert_reached(mc)
    w = synth.make_token_sensitive_weights(mc)
    toks = few_ids(61, 1)
    be = GpuDeqBackend(mc, B, T)
    be.upload_weights(w)
    got = be.forward(toks)
    be.close()
    o = oracle_lib.Oracle(dataclasses.replace(mc, flags=synth.F_SCAN_SELECTIVE), w)
    assert_forward_parity({k: v for k, v in got.items() if not k.startswith("scan")}, by_id(o, toks), str(flags))
    assert np.array_equal(got["argmax"], last_max(got["logits"]))
    for b in (0, 13, B - 1):
        y, st = o.scan(got["h_star"][b])
        np.testing.assert_allclose(got["scan_y"][b], y, rtol=RTOL, atol=ATOL, err_msg=f"scan_y[{b}]")
        np.testing.assert_allclose(got["scan_state"][b], st, rtol=RTOL, atol=ATOL, err_msg=f"scan_state[{b}]")


def test_operands_beyond_fp16_range(oracle_lib):
    """States beyond 65504: the mix and the pooled row are written pre-split at the scale that the
    product derives for itself."""
    mc, w = scaled_model(synth.F_SCAN_SELECTIVE, 0, d=D, H=H, V=V)
    assert_reached(mc)
    toks = few_ids(23, 2)
    be = GpuDeqBackend(mc, B, T)
    be.upload_weights(w)
    got = be.forward(toks)
    be.close()
    o = oracle_lib.Oracle(mc, w)
    ref = by_id(o, toks)
    assert np.abs(got["h_star"]).max() > 65504
    for k, v in got.items():
        if v.dtype.kind == "f":
            assert np.isfinite(v).all(), k
    assert np.abs(got["iters"].astype(int) - ref["iters"]).max() <= 1
    for k in ("h_star", "pooled", "logits"):
        np.testing.assert_allclose(got[k] / G, ref[k] / G, rtol=RTOL, atol=ATOL, err_msg=k)
    assert np.array_equal(got["argmax"], ref["argmax"])
    for b in (0, B - 1):
        y, st = o.scan(got["h_star"][b])
        np.testing.assert_allclose(got["scan_y"][b] / 4e4, y / 4e4, rtol=RTOL, atol=ATOL, err_msg=f"scan_y[{b}]")


def test_nonfinite_rows(oracle_lib):
    """A NaN element and an all-inf row, the latter last in the partial row block: those two tokens run
    to the cap unconverged with non-finite states, the others match the oracle."""
    mc = synth.ModelConfig(d=D, H=H, V=V, N=4, flags=synth.F_SCAN_SELECTIVE, max_iters=16)
    assert_reached(mc)
    w = synth.make_token_sensitive_weights(mc)
    toks = few_ids(37, 3)
    s_in = np.ascontiguousarray(w["embed"][toks])
    s_in[5, 100, 300] = np.nan
    s_in[B - 1, T - 1, :] = -np.inf
    be = GpuDeqBackend(mc, B, T)
    be.upload_weights(w)
    got = be.forward(s_in=s_in, want=("h_star", "pooled", "logits", "argmax", "iters", "converged"))
    be.close()
    bad = np.zeros((B, T), bool)
    bad[5, 100] = bad[B - 1, T - 1] = True
    assert (got["iters"][bad] == 16).all() and (got["converged"][bad] == 0).all()
    assert not np.isfinite(got["h_star"][bad]).any()
    ref = by_id(oracle_lib.Oracle(mc, w), toks[~bad])
    assert_forward_parity({k: got[k][~bad] for k in got}, ref, "finite tokens")


@pytest.mark.parametrize("anderson_m", [0, 3])
def test_graph_replays_match_eager(anderson_m):
    mc = synth.ModelConfig(d=D, H=H, V=V, N=4, anderson_m=anderson_m, max_iters=12)
    assert_reached(mc)
    capture_and_replay(mc, synth.make_token_sensitive_weights(mc), B, T, few_ids(500, 4))
