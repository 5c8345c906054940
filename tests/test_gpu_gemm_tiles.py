"""The LDS-direct bf16 GEMM (kernels_mfma.hip, gemm_tile_kernel) at the edges of its tiles and splits over k: rows against
float64 sums of the same bf16 values, every output against the register-staged kernel."""
import numpy as np
import pytest

from parity import hip_run
from gptrs_amd import functional as F
from gptrs_amd.ptir import FunctionBuilder, Program, bf16_bits_to_f32, f32_to_bf16_bits

pytestmark = pytest.mark.gpu


def bf16(a):
    return bf16_bits_to_f32(f32_to_bf16_bits(np.asarray(a, np.float32)))


def program(specs, body):
    fb = FunctionBuilder("main", "Bf16")
    fb.set_results(body(*[fb.param(dt, dims) for dt, dims in specs]))
    return Program(fb)


# one row over and under the tiles' 64, 128 and 256 rows; columns that end inside a fragment, a tile and a group of 8; one
# k tile, fewer k tiles than the ring holds, k that does not divide among the splits; the layer sizes on each tile and split
@pytest.mark.parametrize("m,k,n", [(17, 64, 8), (33, 128, 41), (64, 192, 130), (65, 3072, 1000), (127, 4096, 3072), (129, 1088, 3075), (200, 9216, 1536),
                                   (255, 3072, 6144), (257, 320, 520), (333, 3072, 6176), (513, 2048, 4100), (1000, 9216, 768), (1025, 448, 9216), (2049, 256, 3008)])
def test_tiles_and_splits(hip, m, k, n):
    rng = np.random.default_rng(m * 7 + k + n)
    x = bf16(rng.standard_normal((m, k), dtype=np.float32))
    w, w2 = (bf16(rng.standard_normal((k, n), dtype=np.float32) * np.float32(k ** -0.5)) for _ in range(2))
    bias, res = bf16(rng.standard_normal(n)), rng.standard_normal((m, n), dtype=np.float32)
    mat, vec = ("Bf16", [k, n]), ("Bf16", [n])
    progs = [program([("Bf16", [m, k]), mat, ("F32", [m, n])], lambda a, b, r: [F.linear(a, b, out_dtype="F32") + r]),
             program([("Bf16", [m, k]), mat, vec], lambda a, b, c: [F.linear(a, b, c)]),
             program([("Bf16", [m, k]), mat, mat], lambda a, b, c: [F.swiglu(F.linear(a, b), F.linear(a, c))])]
    args = [[x, w, res], [x, w, bias], [x, w, w2]]
    got = [hip_run(hip, p, a)[0] for p, a in zip(progs, args)]
    again = [hip_run(hip, p, a)[0] for p, a in zip(progs, args)]
    for a, b in zip(got, again):
        assert np.array_equal(a, b)          # partial sums are added in a fixed order
    hip.set_option("gemm_lds_direct", 0)
    try:
        staged = [hip_run(hip, p, a)[0] for p, a in zip(progs, args)]
    finally:
        hip.set_option("gemm_lds_direct", 1)
    rows = sorted({r for r in (0, 31, 63, 64, 127, 128, 255, 256, m - 1) if r < m})
    x64, w64 = x[rows].astype(np.float64), w.astype(np.float64)
    s, t = x64 @ w64, x64 @ w2.astype(np.float64)
    # f32 sums of k exact products, in any order: off by at most k * 2^-24 of the sum of magnitudes (the order decides how
    # much; 2 sqrt(k) is four times what a random walk of roundings gives)
    bound = 2 * np.sqrt(k) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64)) + 1e-6
    bound2 = 2 * np.sqrt(k) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w2.astype(np.float64))) + 1e-6
    assert (np.abs(got[0][rows] - (s + res[rows])) <= bound + 2.0 ** -23 * np.abs(s + res[rows])).all()
    assert (np.abs(got[1][rows] - (s + bias)) <= bound + 2.0 ** -8 * np.abs(s + bias) + 2.0 ** -8 * np.abs(s)).all()    # the sum and the biased sum are bf16
    sig = 1 / (1 + np.exp(-s))
    # each sum rounded to bf16 where the program says so, at most; |d silu / ds| < 1.1
    pair = (bound + 2.0 ** -8 * np.abs(s)) * 1.1 * np.abs(t) + (bound2 + 2.0 ** -8 * np.abs(t)) * np.abs(s * sig) + 2.0 ** -7 * np.abs(s * sig * t) + 1e-6
    assert (np.abs(got[2][rows] - s * sig * t) <= pair).all()
    for a, b in zip(got, staged):           # two orders of the same sums, one rounding apart in bf16
        assert (np.abs(a - b) <= 2.0 ** -6 * np.maximum(np.abs(a), np.abs(b)) + 4e-4 * np.sqrt(k) / 16).all()
