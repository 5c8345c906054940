"""Linear layers of 2 to 16 rows (kernels_skinny.hip) at the edges of their launch rule: layers of at most 256 column tiles, of up to
768 and beyond; tiles of 12 and of 16 columns, 8 rows and more; few tiles, whose steps are split over workgroups; steps that do not divide among the waves, and fewer steps than
waves.  Rows against float64 sums of the same values, codes against the dequantised matrix."""
import numpy as np
import pytest

from parity import hip_run
from test_gpu_gemm_tiles import bf16, program
from gptrs_amd import backend, functional as F

pytestmark = pytest.mark.gpu


def bounds(x, w, dtype):
    """float64 sums, and what f32 sums of k products in any order (2 sqrt(k) roundings of the sum of magnitudes, four times what a
    random walk of roundings gives), rounded to the layer's type, may be off by."""
    s = x.astype(np.float64) @ w.astype(np.float64)
    mags = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64)
    return s, 2 * np.sqrt(x.shape[1]) * 2.0 ** -24 * mags + (2.0 ** -8 if dtype == "Bf16" else 2.0 ** -23) * np.abs(s) + 1e-6


SIZES = [(2, 32, 16), (3, 96, 130), (7, 3072, 40), (16, 1568, 700), (8, 9216, 304), (5, 288, 4096), (16, 544, 4112), (9, 160, 12272), (4, 192, 12304),
         # tiles of 12 columns: one to a CU, a last tile of 4, two to a CU; splits of 12 steps and more
         (8, 96, 3072), (9, 64, 3064), (16, 224, 6144), (3, 352, 4108), (2, 12288, 36),
         # tiles of 16 columns, two to a CU with up to 8 rows, and four with more
         (6, 160, 8190), (13, 96, 12304)]


@pytest.mark.parametrize("dtype", ["Bf16", "F32"])
@pytest.mark.parametrize("m,k,n", SIZES)
def test_plain_and_pair(hip, dtype, m, k, n):
    rng = np.random.default_rng(m + k + n)
    cast = bf16 if dtype == "Bf16" else np.float32
    x = cast(rng.standard_normal((m, k), dtype=np.float32))
    w, w2 = (cast(rng.standard_normal((k, n), dtype=np.float32) * np.float32(k ** -0.5)) for _ in range(2))
    rows, mat = (dtype, [m, k]), (dtype, [k, n])
    progs = [program([rows, mat], lambda a, b: [F.linear(a, b)]), program([rows, mat, mat], lambda a, b, c: [F.swiglu(F.linear(a, b), F.linear(a, c))])]
    got = [hip_run(hip, p, a)[0] for p, a in zip(progs, ([x, w], [x, w, w2]))]
    for p, a, g in zip(progs, ([x, w], [x, w, w2]), got):
        assert np.array_equal(g, hip_run(hip, p, a)[0])      # partial sums are added in a fixed order
    (s, bs), (t, bt) = (bounds(x, v, dtype) for v in (w, w2))
    assert (np.abs(got[0] - s) <= bs).all()
    g = s / (1 + np.exp(-s))
    # |d silu / ds| < 1.1, one more rounding each for silu and the product
    assert (np.abs(got[1] - g * t) <= 1.1 * bs * np.abs(t) + bt * np.abs(g) + (2.0 ** -7 if dtype == "Bf16" else 2.0 ** -20) * np.abs(g * t) + 1.1 * bs * bt + 1e-6).all()


@pytest.mark.parametrize("m,k,n", [(2, 16, 16), (7, 768, 2304), (16, 1008, 700), (9, 240, 3073), (16, 256, 4096), (3, 1008, 50), (16, 1024, 40), (5, 768, 4112)])
def test_f32_layer_norm_inside(hip, m, k, n):
    """LayerNorm, layer, bias and GELU in one launch (up to 1008 values and a tile for each CU), at the edges of that rule, against float64.  A normed value is off by
    the rounding of its mean, its difference from it and two products: 8 units of 1 + |value|; a sum as in `bounds`."""
    rng = np.random.default_rng(m + k + n)
    x = rng.standard_normal((m, k), dtype=np.float32) * 2 + 1
    g, b = rng.standard_normal(k, dtype=np.float32) * 0.1 + 1, rng.standard_normal(k, dtype=np.float32)
    w, bias = rng.standard_normal((k, n), dtype=np.float32) * np.float32(k ** -0.5), rng.standard_normal(n, dtype=np.float32)
    args = [("F32", list(a.shape)) for a in (x, g, b, w, bias)]
    p = program(args, lambda a, gg, bb, ww, c: [F.linear(F.layer_norm(a, gg, bb, 1e-5)[0], ww, c)])
    got = hip_run(hip, p, [x, g, b, w, bias])[0]
    x64 = x.astype(np.float64)
    c = x64 - x64.mean(1, keepdims=True)
    z = c / np.sqrt((c * c).mean(1, keepdims=True) + 1e-5)
    xn = z * g + b
    s, bound = bounds(xn, w, "F32")
    off = 8 * 2.0 ** -24 * (((1 + np.abs(z)) * np.abs(g) + np.abs(b)) @ np.abs(w).astype(np.float64))
    assert (np.abs(got - (s + bias)) <= bound + off + 2.0 ** -23 * np.abs(bias)).all()


# f32 sums over tiles of 16 columns are those of 16 waves whatever the waves: rows by themselves (16 waves of two requests, 8 of four) and among 12 (8 of one, 16 of one)
@pytest.mark.parametrize("k,n", [(1040, 8190), (1040, 12304), (2064, 8192)])
def test_f32_sums_do_not_depend_on_the_waves(hip, k, n):
    rng = np.random.default_rng(n)
    x, w = rng.standard_normal((12, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    run = lambda rows: hip_run(hip, program([("F32", list(rows.shape)), ("F32", [k, n])], lambda a, b: [F.linear(a, b)]), [rows, w])[0]
    assert np.array_equal(run(x)[:6], run(x[:6]))


@pytest.mark.parametrize("scheme", ["w8", "w4g128"])
@pytest.mark.parametrize("m,k,n", [(2, 128, 16), (7, 3072, 40), (16, 1664, 700), (8, 9216, 304), (5, 384, 4096), (16, 640, 4112), (9, 256, 12304)])
def test_codes(hip, scheme, m, k, n):
    from test_gpu_quant import code_spec, dequantize_host, quantize, scale_dims
    rng = np.random.default_rng(m + k + n)
    x = bf16(rng.standard_normal((m, k), dtype=np.float32))
    (q, s), (q2, s2) = (quantize(rng.standard_normal((k, n), dtype=np.float32) * np.float32(k ** -0.5), scheme) for _ in range(2))
    rows, cs, ss = ("Bf16", [m, k]), code_spec(scheme, k, n), ("Bf16", scale_dims(scheme, k, n))
    plain = program([rows, cs, ss], lambda a, b, c: [F.linear_quantized(a, b, c)])
    pair = program([rows, cs, ss, cs, ss], lambda a, b, bs, c, cs_: [F.swiglu(F.linear_quantized(a, b, bs), F.linear_quantized(a, c, cs_))])
    w, w2 = dequantize_host(q, s, scheme), dequantize_host(q2, s2, scheme)
    (a, ba), (b, bb) = (bounds(x, v, "Bf16") for v in (w, w2))
    # the kernels multiply by the codes and by the scale afterwards, where the dequantised matrix is rounded to bf16 first: half an
    # ulp of each weight, so 2^-9 of the magnitudes at most and a sixth of a random walk of them over k >= 128
    slack = [2.0 ** -9 * np.sqrt((x.astype(np.float64) ** 2) @ (v.astype(np.float64) ** 2)) * 6 for v in (w, w2)]
    ba, bb = ba + slack[0], bb + slack[1]
    got = hip_run(hip, plain, [x, q, s])[0]
    assert (np.abs(got - a) <= ba).all()
    g = a / (1 + np.exp(-a))
    got = hip_run(hip, pair, [x, q, s, q2, s2])[0]
    assert (np.abs(got - g * b) <= 1.1 * ba * np.abs(b) + bb * np.abs(g) + 2.0 ** -7 * np.abs(g * b) + 1.1 * ba * bb + 1e-6).all()


@pytest.mark.parametrize("quant", [1, 2])
def test_pairs_of_codes_share_a_cu(hip, quant):
    assert backend.load_library()._ZN5gptrs1k22skinny_pair_workgroupsEi(quant) >= 3
