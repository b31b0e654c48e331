"""embed_context on both sides of its chunk rules (needs an MI355X): few and many blocks, sequences
whose chunk prefixes are summed in the window kernel or scanned, partial last chunks, sliding windows,
every width bucket, against a float64 brute force."""
import numpy as np
import pytest

from aideen_amd import synth
from aideen_amd.backend import GpuDeqBackend

pytestmark = pytest.mark.gpu

# (d, B, T, ctx)
SHAPES = [(64, 1, 1, 1), (192, 1, 129, 40), (256, 2, 1025, 100), (256, 3, 2050, 2050), (512, 1, 257, 256),
          (512, 5, 205, 33), (512, 1, 1030, 7), (1024, 1, 66, 66), (1024, 9, 70, 20), (1536, 1, 19, 5), (2048, 20, 17, 6)]


@pytest.mark.parametrize("d,B,T,ctx", SHAPES)
def test_embed_context_matches_brute_force(d, B, T, ctx):
    mc = synth.ModelConfig(d=d, H=1, V=97, N=1)
    w = synth.make_token_sensitive_weights(mc)
    toks = synth.make_tokens("uniform", B, T, mc.V, seed=3)
    be = GpuDeqBackend(mc, B, T)
    be.upload_weights(w)
    got = be.embed_context(toks, ctx)
    be.close()
    e = w["embed"].astype(np.float64)[toks]  # [B][T][d]
    for i in sorted({0, 1 % T, min(ctx, T) - 1, min(ctx, T - 1), T // 2, (T - 1) // 8 * 8, T - 1}):
        s = max(0, i - ctx + 1)
        r = (e[:, s:i + 1] * np.arange(1, i - s + 2)[None, :, None]).sum(1) / (i - s + 1)
        n = np.linalg.norm(r, axis=-1, keepdims=True)
        np.testing.assert_allclose(got[:, i], np.where(n > 1e-6, r / n, r), atol=1e-6, err_msg=f"position {i}")
