"""Batched decode attention (kernels_attn.hip, attn_decode_mfma_kernel) where its splits, tiles and the step's own row meet: positions at
the edges of a 32-key tile, of a wave's second tile and of a split, splits behind the position, an appended row behind or before the
attended ones.  Against float64 attention over the same bf16 values."""
import numpy as np
import pytest

from parity import hip_run
from test_gpu_gemm_tiles import bf16, program
from gptrs_amd import functional as F
from gptrs_amd.ptir import FunctionBuilder, Program

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


def test_empty_splits_in_front(hip):
    """Keys whose products overflow to minus infinity have no weight; ten splits of nothing else (32 keys each at these sizes) leave the maximum
    to the ones behind them, however far below zero their scores lie."""
    hq, dh, cap, pos = 1, 64, 512, 400
    cfg = F.AttentionConfig(hq * dh, hq, hq, dh)
    rng = np.random.default_rng(3)
    fb = FunctionBuilder("main", "F32")
    kv = ("F32", [hq, cap, dh])
    fb.set_results(list(F.attention_decode_cache(cfg, *(fb.param(*s) for s in (("F32", [1, 3 * dh]), kv, kv, ("Si32", [3]), ("Si32", [1]))))))
    qkv = rng.standard_normal((1, 3 * dh), dtype=np.float32)
    qkv[0, :2 * dh] = 0
    qkv[0, 0], qkv[0, dh] = 1e20, -1.7e-17
    ck, cv = np.zeros((1, cap, dh), np.float32), rng.standard_normal((1, cap, dh), dtype=np.float32)
    ck[0, :320, 0], ck[0, 320:, 0] = -1e20, rng.uniform(-1.8e-17, -1.6e-17, cap - 320)
    got = hip_run(hip, Program(fb), [qkv, ck, cv, np.array([0, pos, 0], np.int32), np.array([pos], np.int32)])[0]
    ck[0, pos], cv[0, pos] = qkv[0, dh:2 * dh], qkv[0, 2 * dh:]
    s = (np.float64(qkv[0, 0]) * ck[0, 320:pos + 1, 0]) * dh ** -0.5
    w = np.exp(s - s.max())
    want = (w / w.sum()) @ cv[0, 320:pos + 1].astype(np.float64)
    # scores of about -212: three roundings each move a weight by 212 * 3 * 2^-24, sums of 81 terms by far less
    assert np.abs(got[0] - want).max() <= 2 * 212 * 3 * 2.0 ** -24 * np.abs(cv).max()
