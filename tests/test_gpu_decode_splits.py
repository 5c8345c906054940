"""Batched decode attention (kernels_attn.hip, attn_decode_mfma_kernel) where its splits, tiles and the step's own row meet: positions at
the edges of a 32-key tile, of a wave's second tile and of a split, splits behind the position, an appended row behind or before the
attended ones.  Against float64 attention over the same bf16 values."""
import numpy as np
import pytest

from parity import hip_run
from test_gpu_gemm_tiles import bf16, program
from gptrs_amd import functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,dh,cap", [(8, 2, 128, 4096), (16, 2, 64, 16384), (4, 4, 64, 96), (32, 4, 128, 70)])
def test_positions(hip, hq, hkv, dh, cap):
    cfg = F.AttentionConfig(hq * dh, hq, hkv, dh)
    P = cfg.total_projection_dim
    rng = np.random.default_rng(cap)
    kv = ("Bf16", [hkv, cap, dh])
    p = program([("Bf16", [1, P]), kv, kv, ("Si32", [3]), ("Si32", [1])], lambda a, k, v, us, qs: list(F.attention_decode_cache(cfg, a, k, v, us, qs)))
    qkv, ck, cv = (bf16(rng.standard_normal(s, dtype=np.float32)) for s in ((1, P), (hkv, cap, dh), (hkv, cap, dh)))
    q = qkv[0, :hq * dh].reshape(hq, dh).astype(np.float64)
    knew, vnew = qkv[0, hq * dh:].reshape(2, hkv, dh)
    edges = [0, 1, 31, 32, 63, 64, 127, 128, 160, 255, 256, 257, 1000, cap // 2, cap - 2, cap - 1]
    for pos, upd in [(e, e) for e in edges if 0 <= e < cap] + [(cap // 2, cap - 1), (cap - 2, 33), (cap // 3, cap // 3 + 1)]:
        ctx, k, v = hip_run(hip, p, [qkv, ck, cv, np.array([0, upd, 0], np.int32), np.array([pos], np.int32)])
        wk, wv = ck.copy(), cv.copy()
        wk[:, upd], wv[:, upd] = knew, vnew
        assert np.array_equal(k, wk) and np.array_equal(v, wv)
        keys, vals = (np.repeat(c[:, :pos + 1].astype(np.float64), hq // hkv, axis=0) for c in (wk, wv))
        s = np.einsum("hd,htd->ht", q, keys) * dh ** -0.5
        w = np.exp(s - s.max(axis=1, keepdims=True))
        w /= w.sum(axis=1, keepdims=True)
        want = np.einsum("ht,htd->hd", w, vals)
        # scores are f32 sums of dh products (sqrt(dh) roundings of their magnitudes), which moves a weight by that much of itself;
        # sums over the keys likewise, and one rounding to bf16
        err = 2.0 ** -24 * (8 * np.sqrt(dh) * (np.abs(q).sum(axis=1).max() * np.abs(keys).max() * dh ** -0.5) + 4 * np.sqrt(pos + 1) + 16)
        assert (np.abs(ctx.reshape(hq, dh) - want) <= 2.0 ** -8 * np.abs(want) + err * np.einsum("ht,htd->hd", w, np.abs(vals)) + 1e-6).all(), (pos, upd)
