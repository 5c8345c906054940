"""The LDS-direct bf16 GEMM (kernels_mfma.hip, gemm_tile_kernel) at the edges of its tiles and splits over k: rows against
float64 sums of the same bf16 values, every output against the register-staged kernel."""
import time

import numpy as np
import pytest

from parity import hip_run, to_bytes
from test_gemm_plans import lib, regions
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
                                   (255, 3072, 6144), (257, 320, 520), (333, 3072, 6176), (513, 2048, 4100), (1000, 9216, 768), (1025, 448, 9216), (2049, 256, 3008),
                                   # 192 x 192 tiles: one round, ragged rows and columns, k tiles that divide by the ring and that do not
                                   (2881, 9216, 2900), (2753, 5120, 3050), (3072, 5184, 3072),
                                   # 128 x 192 tiles, whole and in 2, 4 and 8 splits, then for the pair whole and in 2, 3 and 4: ragged rows and columns
                                   (1227, 1536, 3985), (913, 9216, 2673), (230, 9216, 5883), (2025, 9216, 368), (687, 3072, 3335), (615, 9216, 1602)])
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


# layers that take two launches, of the layer itself or of the pair: split between columns and between rows, ragged in both
@pytest.mark.parametrize("m,k,n", [(2824, 1088, 5398), (2075, 1088, 7699), (609, 1792, 6587), (1555, 1088, 5027), (857, 2624, 5157)])
def test_two_launches(hip, m, k, n):
    assert any(regions(m, k, n, dual) is not None for dual in (False, True))
    test_tiles_and_splits(hip, m, k, n)


# the same kernel in f32, of up to 128 rows (64 x 64 tiles): tile edges, columns that are no multiple of 8, one k tile, k tiles that do not divide among
# the splits (13 in 3, 25 in 6 and in 3, 35 in 6, 65 in 8, 97 in 4); three layers of more rows, which gemm_split_kernel takes, against the same bounds
@pytest.mark.parametrize("m,k,n", [(17, 32, 8), (40, 768, 41), (63, 96, 130), (65, 3072, 768), (66, 416, 130), (97, 1120, 1290), (100, 2080, 1000), (127, 800, 2307), (128, 800, 700),
                                   (128, 3104, 2000), (129, 800, 2307), (300, 4096, 192), (700, 256, 3072)])
def test_f32_tiles_and_splits(hip, m, k, n):
    rng = np.random.default_rng(m + k + n)
    x, w, w2 = (rng.standard_normal(s, dtype=np.float32) for s in ((m, k), (k, n), (k, n)))
    w, w2 = w * np.float32(k ** -0.5), w2 * np.float32(k ** -0.5)
    bias, res = rng.standard_normal(n, dtype=np.float32), rng.standard_normal((m, n), dtype=np.float32)
    f32, mat = "F32", ("F32", [k, n])

    def run(specs, body, args):
        fb = FunctionBuilder("main", f32)
        fb.set_results([body(*[fb.param(dt, dims) for dt, dims in specs])])
        p = Program(fb)
        got = hip_run(hip, p, args)[0]
        assert np.array_equal(got, hip_run(hip, p, args)[0])
        return got

    def all_three():
        return (run([(f32, [m, k]), mat, (f32, [m, n])], lambda a, b, r: F.linear(a, b) + r, [x, w, res]),
                run([(f32, [m, k]), mat, (f32, [n])], lambda a, b, c: F.linear(a, b, c), [x, w, bias]),
                run([(f32, [m, k]), mat, mat], lambda a, b, c: F.swiglu(F.linear(a, b), F.linear(a, c)), [x, w, w2]))

    tiles = all_three()
    hip.set_option("gemm_lds_direct", 0)
    try:
        staged = all_three()
    finally:
        hip.set_option("gemm_lds_direct", 1)
    assert not np.array_equal(tiles[0], staged[0]) or k <= 32      # another order of the sums: the switch has taken the other kernel
    x64, w64, v64 = x.astype(np.float64), w.astype(np.float64), w2.astype(np.float64)
    s, t = x64 @ w64, x64 @ v64
    # as above: 2 sqrt(k) roundings of the sum of magnitudes, and one for each operation behind the sum
    bs, bt = (2 * np.sqrt(k) * 2.0 ** -24 * (np.abs(x64) @ np.abs(v)) + 1e-6 for v in (w64, v64))
    g = s / (1 + np.exp(-s))
    for plain, biased, pair in (tiles, staged):
        assert (np.abs(plain - (s + res)) <= bs + 2.0 ** -23 * np.abs(s + res)).all()
        assert (np.abs(biased - (s + bias)) <= bs + 2.0 ** -23 * np.abs(s + bias)).all()
        assert (np.abs(pair - g * t) <= 1.1 * bs * np.abs(t) + bt * np.abs(g) + 2.0 ** -20 * np.abs(g * t) + 1e-6).all()


def test_f32_sums_in_two_chains(hip):
    """An f32 rounding is off by 0.42 * 2^-24 of its value in the mean square (uniform over half an ulp, an ulp being 2^-23 to 2^-24 of it), and
    a chain of n terms of one size rounds partial sums of sqrt(i): sqrt(n / 2) of that over the sum's own sqrt(n).  Two chains of k / 2:
    sqrt(k / 4).  A fifth is left for the sample of values; one chain would be 1.41 times the value.  128 rows are the most that f32 products take, and
    this layer's tiles fill the chip without splits, which would be chains of their own."""
    m, k, n = 128, 768, 8192
    assert lib()[1](0, m, k, n, False, 0) == 0      # no partial sums
    rng = np.random.default_rng(11)
    x, w = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    fb = FunctionBuilder("main", "F32")
    fb.set_results([F.linear(fb.param("F32", [m, k]), fb.param("F32", [k, n]))])
    got, want = hip_run(hip, Program(fb), [x, w])[0], x.astype(np.float64) @ w.astype(np.float64)
    assert np.linalg.norm(got - want) <= 1.2 * 0.42 * 2.0 ** -24 * np.sqrt(k / 4) * np.linalg.norm(want)


def f32_layers(hip, x, w, w2, bias, res):
    """x.w + res, x.w + bias and silu(x.w) * (x.w2), each run twice"""
    def run(specs, body, args):
        fb = FunctionBuilder("main", "F32")
        fb.set_results([body(*[fb.param("F32", dims) for dims in specs])])
        got = [hip_run(hip, Program(fb), args)[0] for _ in range(2)]
        assert np.array_equal(got[0], got[1], equal_nan=True)
        return got[0]

    (m, k), n = x.shape, w.shape[1]
    return (run([(m, k), (k, n), (m, n)], lambda a, b, r: F.linear(a, b) + r, [x, w, res]), run([(m, k), (k, n), (n,)], lambda a, b, c: F.linear(a, b, c), [x, w, bias]),
            run([(m, k), (k, n), (k, n)], lambda a, b, c: F.swiglu(F.linear(a, b), F.linear(a, c)), [x, w, w2]))


# f32 of more than 128 rows as six bf16 products (fewer: f32 products): rows around the tiles' 64, 128 and 256, columns around 64 and 96 and no multiples of 8, two k tiles,
# fewer and more than the ring, whole and in splits.  `scale` takes the rows far from 1, up and down
@pytest.mark.parametrize("m,k,n,scale", [(129, 32, 8, 1.0), (130, 96, 63, 1e18), (160, 3072, 97, 1.0), (191, 64, 193, 1.0), (193, 800, 770, 1e-29), (255, 768, 2304, 1.0), (511, 3072, 767, 1.0),
                                         (700, 736, 3070, 1e-18), (1025, 1536, 1000, 1.0), (1473, 768, 2309, 1.0), (2047, 768, 3073, 1.0), (2305, 3104, 769, 1.0)])
def test_f32_as_bf16_products(hip, m, k, n, scale):
    rng = np.random.default_rng(m + k + n)
    x, w, w2 = (rng.standard_normal(s, dtype=np.float32) for s in ((m, k), (k, n), (k, n)))
    x, w, w2 = x * np.float32(scale), w * np.float32(k ** -0.5), w2 * np.float32(k ** -0.5)
    bias, res = (rng.standard_normal(s, dtype=np.float32) * np.float32(scale) for s in ((n,), (m, n)))
    plain, biased, pair = f32_layers(hip, x, w, w2, bias, res)
    rows = sorted({r for r in (0, 31, 63, 64, 95, 96, 127, 128, 255, 256, 1000, m - 2, m - 1) if r < m})
    x64, w64, v64 = x[rows].astype(np.float64), w.astype(np.float64), w2.astype(np.float64)
    s, t = x64 @ w64, x64 @ v64
    # every term is off by 2^-23.9 at the most, and 2 sqrt(k) roundings of the sum of magnitudes as above
    bs, bt = (2 * (np.sqrt(k) + 1) * 2.0 ** -24 * (np.abs(x64) @ np.abs(v)) for v in (w64, v64))
    assert (np.abs(plain[rows] - (s + res[rows])) <= bs + 2.0 ** -23 * np.abs(s + res[rows])).all()
    assert (np.abs(biased[rows] - (s + bias)) <= bs + 2.0 ** -23 * np.abs(s + bias)).all()
    if scale == 1.0:
        g = s / (1 + np.exp(-s))
        assert (np.abs(pair[rows] - g * t) <= 1.1 * bs * np.abs(t) + bt * np.abs(g) + 2.0 ** -20 * np.abs(g * t) + 1e-12).all()
    # in the mean: a chain of n = k / 8 roundings of 0.42 * 2^-24 each is (n + 1) / 2 of their squares away (see test_f32_sums_in_two_chains), the sum
    # of the large and the small products 1 and the residual, which doubles the value's square, 2.  A quotient of two norms of so many values is itself
    # 1 / sqrt(values) uncertain: three of those, beside that test's fifth
    far = np.linalg.norm(plain[rows] - (s + res[rows])) / np.linalg.norm(s)
    assert far <= (1.2 + 3 / np.sqrt(s.size)) * 0.42 * 2.0 ** -24 * np.sqrt((k / 8 + 1) / 2 + 3)


# rows and weights of any size: subnormal values and up to where the split kernel's scaled sums leave f32's range (from 2^80 on), which f32 products then form.
# What f32 products hold, and no bits less
@pytest.mark.parametrize("m,k,n", [(129, 96, 70), (300, 3072, 130), (1100, 768, 1500)])
@pytest.mark.parametrize("sx,sw", [(-120, 0), (-112, 100), (-104, 0), (-140, 60), (0, -124), (90, -135), (-60, -50), (60, 0), (50, 40), (110, -100), (-90, 105)])
def test_f32_as_bf16_products_of_any_size(hip, m, k, n, sx, sw):
    rng = np.random.default_rng(m + 200 + sx)
    x, w = (rng.uniform(0.5, 1, s).astype(np.float32) * rng.choice([-1, 1], s).astype(np.float32) for s in ((m, k), (k, n)))
    x, w = np.ldexp(x, sx), np.ldexp(w, sw)
    fb = FunctionBuilder("main", "F32")
    fb.set_results([F.linear(fb.param("F32", [m, k]), fb.param("F32", [k, n]))])
    rows = sorted({0, 31, 32, 63, 64, 127, 128, m // 2, m - 1})
    got, x64, w64 = hip_run(hip, Program(fb), [x, w])[0][rows].astype(np.float64), x[rows].astype(np.float64), w.astype(np.float64)
    s = x64 @ w64
    assert (np.abs(got - s) <= 2 * (np.sqrt(k) + 1) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64)) + 2.0 ** -149).all()
    # in the mean as two chains of f32 sums (see test_f32_sums_in_two_chains); the split kernel's sums are nearer
    assert np.linalg.norm(got - s) <= (1.2 + 3 / np.sqrt(s.size)) * 0.42 * 2.0 ** -24 * np.sqrt(k / 4 + 3) * np.linalg.norm(s)


# infinities, NaN and values that round to infinity in bf16: what f32 products give, whole tiles and splits, both matrices of a pair
@pytest.mark.parametrize("m,k,n", [(129, 64, 40), (140, 3072, 100), (300, 96, 193), (2100, 64, 3000)])
def test_f32_as_bf16_products_not_finite(hip, m, k, n):
    rng = np.random.default_rng(m)
    x, w, w2 = (rng.uniform(0.5, 1, s).astype(np.float32) * rng.choice([-1, 1], s).astype(np.float32) for s in ((m, k), (k, n), (k, n)))
    w, w2 = w / np.float32(k), w2 / np.float32(k)
    x[3, 5], x[7, k - 1], x[m - 1, 0], x[20, 3], x[20, 4], x[33] = np.inf, np.nan, -np.inf, np.inf, -np.inf, np.float32(3.4e38)
    w[11, 2], w[k - 1, n - 1], w2[5, 6], w[9, 8] = -np.inf, np.nan, np.inf, np.float32(3.4e38)
    x[33, 1::2] *= -1                                      # terms of 3.4e38 / k, a sum that no order takes out of range
    x[33, [9, 11, k - 1]] = 0.0
    plain, biased, pair = f32_layers(hip, x, w, w2, np.zeros(n, np.float32), np.zeros((m, n), np.float32))
    with np.errstate(all="ignore"):
        s, t = ((x.astype(np.float64) @ v.astype(np.float64)).astype(np.float32) for v in (w, w2))
        both = (s.astype(np.float64) / (1 + np.exp(-s.astype(np.float64))) * t).astype(np.float32)
    odd = ~np.isfinite(s)
    scale = np.abs(np.where(np.isfinite(x), x, 0)).max(1, keepdims=True) * np.ones(n)
    scale[:, 8] = 3.4e38
    for got in (plain, biased):
        assert np.array_equal(got[odd], s[odd], equal_nan=True)
        assert (np.abs(got[~odd].astype(np.float64) - s[~odd]) <= 1e-5 * scale[~odd]).all()
    clear = np.isfinite(s) & np.isfinite(t) & np.isfinite(both)
    assert odd.sum() > 2 * n and np.isfinite(pair[clear]).all()
    gone = np.isnan(both)
    assert gone.any() and np.isnan(pair[gone & ~np.isneginf(s)]).all()      # (silu of an infinite negative gate: either zero or NaN)


# such sums are formed again by whole fragments on the f32 cores: all of a layer's take 2.7 times the layer, one row's 2.6 (one lane a sum, a term after
# another: 200 and 180 times)
@pytest.mark.parametrize("m,k,n", [(2048, 768, 3072), (512, 3072, 768)])
def test_f32_sums_not_finite_are_formed_again_quickly(hip, m, k, n):
    rng = np.random.default_rng(m)
    x, w = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    fb = FunctionBuilder("main", "F32")
    fb.set_results([F.linear(fb.param("F32", [m, k]), fb.param("F32", [k, n]))])
    p = Program(fb)
    row, every = x.copy(), np.full_like(x, np.nan)
    row[5, 7] = np.nan
    weights = hip.materialize(p.param_specs[1], to_bytes(w, "F32"))

    def us(rows):
        args = [hip.materialize(p.param_specs[0], to_bytes(rows, "F32")), weights]
        out, took = hip.to_numpy(hip.run_program(p, args)[0]), []
        for _ in range(5):
            hip.synchronize()
            t = time.perf_counter()
            for _ in range(8):
                hip.run_program(p, args)
            hip.synchronize()
            took.append(time.perf_counter() - t)
        return min(took) / 8 * 1e6, out

    (plain, a), (one, b), (all_nan, c) = (us(rows) for rows in (x, row, every))
    assert np.isnan(b[5]).all() and np.array_equal(np.delete(a, 5, 0), np.delete(b, 5, 0)) and np.isnan(c).all()
    assert max(one, all_nan) <= 5 * plain, (plain, one, all_nan)


# codes converted on the way to the matrix pipes: odd columns, one k tile pair, k tiles that split in the middle of an int4 group, rows
# around the tiles' 64 and 128
@pytest.mark.parametrize("scheme", ["w8", "w4g128"])
@pytest.mark.parametrize("m,k,n", [(17, 128, 9), (63, 384, 130), (65, 640, 137), (129, 1920, 391), (200, 2176, 260), (257, 9216, 72)])
def test_codes_equal_the_dequantised_matrix(hip, scheme, m, k, n):
    from test_gpu_quant import code_spec, dequantize_host, quantize, scale_dims
    rng = np.random.default_rng(m + k + n)
    x = bf16(rng.standard_normal((m, k), dtype=np.float32))
    (q, s), (q2, s2) = (quantize(rng.standard_normal((k, n), dtype=np.float32) * np.float32(k ** -0.5), scheme) for _ in range(2))
    rows, cs, ss, mat = ("Bf16", [m, k]), code_spec(scheme, k, n), ("Bf16", scale_dims(scheme, k, n)), ("Bf16", [k, n])
    codes = [program([rows, cs, ss], lambda a, b, c: [F.linear_quantized(a, b, c)]),
             program([rows, cs, ss, cs, ss], lambda a, b, bs, c, cs_: [F.swiglu(F.linear_quantized(a, b, bs), F.linear_quantized(a, c, cs_))])]
    plain = [program([rows, mat], lambda a, b: [F.linear(a, b)]), program([rows, mat, mat], lambda a, b, c: [F.swiglu(F.linear(a, b), F.linear(a, c))])]
    got = [hip_run(hip, p, a)[0] for p, a in zip(codes, ([x, q, s], [x, q, s, q2, s2]))]
    w, w2 = dequantize_host(q, s, scheme), dequantize_host(q2, s2, scheme)
    hip.set_option("gemm_lds_direct", 0)
    try:
        want = [hip_run(hip, p, a)[0] for p, a in zip(plain, ([x, w], [x, w, w2]))]
        staged = [hip_run(hip, p, a)[0] for p, a in zip(codes, ([x, q, s], [x, q, s, q2, s2]))]
    finally:
        hip.set_option("gemm_lds_direct", 1)
    for g, v, r in zip(got, want, staged):
        assert np.array_equal(g, v)      # the same products, added in the same order
        assert np.array_equal(r, v)      # so does the register-staged kernel over codes


# a pair's gate is one function for prompts and for decode steps (kernels_skinny.hip), also far below zero, where e^-g nears the largest
# f32.  Each sum has two exact products, so both kernels combine the same gates; a split over k meets in gemm_reduce_kernel
@pytest.mark.parametrize("kind", ["silu", "clamped"])
@pytest.mark.parametrize("m,k", [(17, 64), (300, 64), (300, 3072)])
def test_pair_is_the_decode_steps_function(hip, kind, m, k):
    rng = np.random.default_rng(k + m)
    n = 4096
    glu = F.swiglu if kind == "silu" else lambda a, b: F.clamped_glu(a, b, 60.0, 1.25)
    w, w2 = np.zeros((k, n), np.float32), np.zeros((k, n), np.float32)
    at = (0, k - 1)                                       # the two products of a sum lie as far apart as k allows
    w[at[0]], w[at[1]] = bf16(np.linspace(-100, 100, n)), bf16(rng.uniform(-1, 1, n))
    w2[at[0]] = bf16(rng.standard_normal(n) * 2.0 ** rng.uniform(-4, 60, n))
    x = np.zeros((m, k), np.float32)
    x[:, at[0]], x[:, at[1]] = bf16(np.linspace(1.0, 0.25, m)), 2.0 ** -8
    mat = ("Bf16", [k, n])
    run = lambda rows: hip_run(hip, program([("Bf16", [len(rows), k]), mat, mat], lambda a, b, c: [glu(F.linear(a, b), F.linear(a, c))]), [rows, w, w2])[0]
    got = run(x)
    for r in range(0, m, 16):
        rows = x[r:r + 16] if r + 16 <= m else x[m - 16:]
        first = r if r + 16 <= m else m - 16
        assert np.array_equal(got[first:first + 16], run(rows)), first


# the launch that adds a layer's splits takes the RMS norm behind it along: the same bits as the norm by itself, with every value of the
# program between its ends in reused memory; widths under and over a thread's 8 values, 64, 256 and 512 threads; more rows than splits are made for
@pytest.mark.parametrize("m,k,n", [(17, 1088, 264), (64, 9216, 3072), (129, 4096, 4160), (333, 9216, 3072), (333, 9216, 3084), (40, 2048, 8192), (40, 2048, 8200), (2100, 512, 3072)])
def test_norm_behind_splits(hip, m, k, n):
    rng = np.random.default_rng(m + k + n)
    x, w = bf16(rng.standard_normal((m, k), dtype=np.float32)), bf16(rng.standard_normal((k, n), dtype=np.float32) * np.float32(k ** -0.5))
    w2 = bf16(rng.standard_normal((n, 256), dtype=np.float32) * np.float32(n ** -0.5))
    res, gain = rng.standard_normal((m, n), dtype=np.float32), 1 + rng.standard_normal(n, dtype=np.float32) / 8
    rows, mat, f32, vec = ("Bf16", [m, k]), ("Bf16", [k, n]), ("F32", [m, n]), ("F32", [n])

    def norm(y, g):
        return F.rms_norm(y, g, 1e-5)[0].cast("Bf16")

    def block(a, b, r, g, c):
        y = F.linear(a, b, out_dtype="F32") + r
        return [F.linear(norm(y, g), c), y]

    layer = program([rows, mat, f32], lambda a, b, r: [F.linear(a, b, out_dtype="F32") + r])
    alone = program([f32, vec], lambda y, g: [norm(y, g)])
    head = program([("Bf16", [m, n]), ("Bf16", [n, 256])], lambda a, b: [F.linear(a, b)])
    both = program([rows, mat, f32, vec], lambda a, b, r, g: (lambda y: [norm(y, g), y])(F.linear(a, b, out_dtype="F32") + r))
    whole = program([rows, mat, f32, vec, ("Bf16", [n, 256])], block)
    no_res = program([rows, mat, vec], lambda a, b, g: [norm(F.linear(a, b, out_dtype="F32"), g)])
    y = hip_run(hip, layer, [x, w, res])[0]
    z = hip_run(hip, alone, [y, gain])[0]
    for _ in range(2):
        got = hip_run(hip, both, [x, w, res, gain])
        assert np.array_equal(got[1], y) and np.array_equal(got[0], z)
        got = hip_run(hip, whole, [x, w, res, gain, w2])
        assert np.array_equal(got[1], y) and np.array_equal(got[0], hip_run(hip, head, [z, w2])[0])
    plain = hip_run(hip, program([rows, mat], lambda a, b: [F.linear(a, b, out_dtype="F32")]), [x, w])[0]
    assert np.array_equal(hip_run(hip, no_res, [x, w, gain])[0], hip_run(hip, alone, [plain, gain])[0])
