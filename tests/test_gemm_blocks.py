"""The blocks that a product's sizes choose (host-only): the sizes of the GPU tests reach the kernels
that their texts name, and products that an exit test follows keep one order of summation."""
import ctypes as C

import numpy as np
import pytest

from aideen_amd import _lib, synth
from aideen_amd.backend import gemm_blocks
import test_gpu_graph as graph
import test_gpu_parity as parity
import test_gpu_tiles as tiles
import test_gpu_token_sensitive as sensitive

PRODUCTS = ("signal_gemm", "qkv_gemm", "wo_gemm", "lmhead_gemm", "readout_gemm")


def model(d, H, V, **kw):
    return synth.ModelConfig(d=d, H=H, V=V, N=4, **kw)


def blocks(shape, rows, exits, flags=0):
    mc = model(*shape, flags=flags)
    return {s: gemm_blocks(mc, s, rows, exits) for s in PRODUCTS}


def test_tile_shapes_reach_every_block():
    got = {s: blocks(s[:3], s[3] * s[4], False) for s in tiles.SHAPES}
    seen = {b[:3] for g in got.values() for b in g.values()}
    for want in ((32, 32, 8), (32, 64, 4), (64, 64, 4), (64, 128, 1), (64, 256, 1), (128, 128, 1), (32, 128, 2)):
        assert want in seen, want
    # W_o pre-split on 64x128 and 128x128 blocks, the head on all its pre-split blocks
    assert {g["wo_gemm"][:2] for g in got.values() if g["wo_gemm"][3]} >= {(64, 128), (128, 128)}
    assert {g["lmhead_gemm"][:2] for g in got.values() if g["lmhead_gemm"][3]} >= {(64, 128), (64, 256), (128, 128)}


def test_bf16_shapes_reach_the_128x256_blocks():
    got = [blocks(s[:3], s[3] * s[4], False, synth.F_GEMM_BF16) for s in tiles.BF16_SHAPES]
    for stage in PRODUCTS:
        assert any(g[stage][:2] == (128, 256) for g in got), stage


def test_exit_shapes_cross_the_block_choice():
    """The batches that must agree bit for bit run their products on different blocks."""
    n = 0
    for d, H, T, few, many in tiles.EXIT_SHAPES:
        a, b = (blocks((d, H, 97), B * T, True) for B in (few, many))
        n += any(a[s] != b[s] for s in PRODUCTS[:3])
    assert n >= 4


@pytest.mark.parametrize("var", parity.PRESPLIT_SHAPES, ids=lambda v: f"d{v['d']}H{v['H']}")
def test_presplit_shapes_are_presplit(var):
    var = dict(var)
    rows = var.pop("B", 4) * var.pop("T", 256)
    mc = synth.ModelConfig(**var)
    assert gemm_blocks(mc, "wo_gemm", rows, mc.eps > 0)[3] == 1
    assert gemm_blocks(mc, "lmhead_gemm", rows, mc.eps > 0)[3] == 1


@pytest.mark.parametrize("var", parity.LARGE + sensitive.LARGE_TS)
def test_large_shapes_run_on_ring_blocks(var):
    var = dict(var)
    rows = var.pop("B") * var.pop("T")
    mc = synth.ModelConfig(**var)
    assert all(gemm_blocks(mc, s, rows, mc.eps > 0)[2] == 1 for s in PRODUCTS)


def test_graph_shape_is_presplit():
    mc = synth.ModelConfig(d=512, H=2, V=700, N=4)
    assert gemm_blocks(mc, "wo_gemm", 1200, True)[3] == 1 and gemm_blocks(mc, "lmhead_gemm", 1200, True)[3] == 1
    assert graph.capture_and_replay


def test_products_before_an_exit_test_sum_in_one_order():
    rng = np.random.default_rng(1)
    for _ in range(400):
        d, H = int(rng.integers(1, 33)) * 64, int(rng.integers(1, 17))
        mc = model(d, H, 97, flags=int(rng.choice([0, synth.F_GEMM_BF16X3, synth.F_GEMM_BF16])))
        rows = int(np.exp(rng.uniform(0, np.log(20000))))
        few = {gemm_blocks(mc, s, min(rows, 32), True)[2] for s in PRODUCTS[:3]}
        assert few == {gemm_blocks(mc, "qkv_gemm", 1, True)[2]}
        assert all(gemm_blocks(mc, s, max(rows, 33), True)[2] == 1 for s in PRODUCTS[:3] + ("hist_gemm",))


def test_presplit_only_for_fp16_halves_on_ring_blocks():
    rng = np.random.default_rng(2)
    for _ in range(400):
        d, H, V = int(rng.integers(1, 33)) * 64, int(rng.integers(1, 17)), int(rng.integers(1, 60000))
        flags = int(rng.choice([0, 0, synth.F_GEMM_BF16X3, synth.F_GEMM_BF16, synth.F_GEMM_FP32]))
        rows, exits = int(np.exp(rng.uniform(0, np.log(20000)))), bool(rng.random() < 0.5)
        for stage, b in blocks((d, H, V), rows, exits, flags).items():
            ring = b[2] == 1 and b[:2] != (128, 64) and rows > (32 if stage == "lmhead_gemm" or exits else 4)
            if stage in ("wo_gemm", "lmhead_gemm") and flags == 0:
                assert b[3] == int(ring), (stage, d, H, V, rows, exits, b)
            else:
                assert b[3] == 0


def test_bad_arguments_are_errors():
    L, out = _lib.lib(), (C.c_int32 * 4)()
    cfg = _lib.AdnConfig(128, 4, 512, 16, 32, 1, 8, 0, 0)
    q = _lib.STAGES.index("qkv_gemm")
    assert L.adn_gemm_blocks(None, q, 5, 0, out) == _lib.ADN_E_INVALID
    assert L.adn_gemm_blocks(C.byref(cfg), q, 5, 0, None) == _lib.ADN_E_INVALID
    for stage, rows in ((_lib.STAGES.index("attn"), 5), (99, 5), (-1, 5), (q, 0), (q, -3)):
        assert L.adn_gemm_blocks(C.byref(cfg), stage, rows, 0, out) == _lib.ADN_E_INVALID
    cfg.d_r = 100
    assert L.adn_gemm_blocks(C.byref(cfg), q, 5, 0, out) == _lib.ADN_E_INVALID
