"""Prompt attention whose workgroups are dealt to the chip's eight dies: heads that divide among them, pairs of head and sequence (or
group of query heads) that do, neither.  A wrong deal leaves rows out or computes them twice, so every row is compared with float64."""
import numpy as np
import pytest

from parity import hip_run
from test_gpu_gemm_tiles import bf16, program
from gptrs_amd import functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["Bf16", "F32"])
@pytest.mark.parametrize("hq,hkv,dh,t", [(16, 8, 64, 333), (32, 16, 64, 70), (32, 4, 64, 161), (32, 2, 128, 70), (12, 12, 64, 97), (6, 2, 128, 260), (8, 8, 128, 31)])
def test_every_row(hip, dtype, hq, hkv, dh, t):
    cfg = F.AttentionConfig(hq * dh, hq, hkv, dh)
    P = cfg.total_projection_dim
    qkv = np.random.default_rng(t).standard_normal((t, P), dtype=np.float32)
    qkv = bf16(qkv) if dtype == "Bf16" else qkv
    got = hip_run(hip, program([(dtype, [t, P])], lambda a: list(F.attention(cfg, a, None))), [qkv])[0].reshape(t, hq, dh)
    x = qkv.astype(np.float64)
    q, k, v = x[:, :hq * dh].reshape(t, hq, dh), x[:, hq * dh:(hq + hkv) * dh].reshape(t, hkv, dh), x[:, (hq + hkv) * dh:].reshape(t, hkv, dh)
    for h in range(hq):
        s = q[:, h] @ k[:, h * hkv // hq].T * dh ** -0.5
        s[np.triu_indices(t, 1)] = -np.inf
        w = np.exp(s - s.max(axis=1, keepdims=True))
        w /= w.sum(axis=1, keepdims=True)
        vh = v[:, h * hkv // hq]
        mags = w @ np.abs(vh)
        # bf16: probabilities rounded to 2^-9 of themselves, and the result; f32: scores off by 2 sqrt(dh) roundings of their magnitudes
        # move a weight by as much of itself, and the sums over the keys add 2 sqrt(t) more
        score = 2.0 ** -24 * 2 * np.sqrt(dh) * (np.abs(q[:, h]) @ np.abs(k[:, h * hkv // hq]).T).max() * dh ** -0.5
        tol = (2.0 ** -8 if dtype == "Bf16" else 0) + 2 * score + 2.0 ** -24 * (2 * np.sqrt(t) + 16)
        assert (np.abs(got[:, h] - w @ vh) <= tol * (mags + np.abs(w @ vh)) + 1e-6).all(), h


# 65 to 128 keys: a wave group of four without a tile, one with a part of one; groups of 1, 2, 4 and 8 query heads; the last launch of four key
# groups (256 workgroups) and the first beyond
@pytest.mark.parametrize("hq,hkv,dh,t", [(4, 4, 32, 65), (5, 5, 128, 96), (8, 4, 64, 97), (8, 4, 32, 128), (16, 2, 32, 129), (16, 2, 128, 65),
                                         (32, 8, 128, 100), (32, 8, 128, 512), (32, 8, 128, 513), (8, 8, 64, 2000)])
def test_four_key_groups(hip, hq, hkv, dh, t):
    test_every_row(hip, "Bf16", hq, hkv, dh, t)
