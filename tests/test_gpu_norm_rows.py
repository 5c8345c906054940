"""Rows normalised with their gains held in registers: lengths at the edges of a thread's eight values, of a wave and of a workgroup,
the first length that is read again instead, lengths that are no multiple of eight.  Against float64."""
import numpy as np
import pytest

from parity import hip_run, po
from test_gpu_gemm_tiles import program
from gptrs_amd import functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8, 248, 264, 512, 520, 1027, 3070, 3072, 4096, 4104, 8192, 8200, 16392])
def test_rows(hip, n):
    rng = np.random.default_rng(n)
    x, g, b = (rng.standard_normal(s, dtype=np.float32) for s in ((3, n), (n,), (n,)))
    f32 = lambda *d: ("F32", list(d))   # noqa: E731
    rms16 = hip_run(hip, program([f32(3, n), f32(n)], lambda a, c: [F.rms_norm(a, c, 1e-5)[0].cast("Bf16")]), [x, g])[0]
    ln = hip_run(hip, program([f32(3, n), f32(n), f32(n)], lambda a, c, d: [F.layer_norm(a, c, d, 1e-5)[0]]), [x, g, b])[0]
    x64 = x.astype(np.float64)
    want = x64 / np.sqrt((x64 ** 2).mean(axis=1, keepdims=True) + 1e-5) * g
    # the sum of n squares in f32: 2 sqrt(n) roundings of it, halved by the root; the result rounded to bf16
    rel = np.sqrt(n) * 2.0 ** -24 + 2.0 ** -21
    assert (np.abs(np.asarray(rms16, np.float32) - want) <= (2.0 ** -8 + rel) * np.abs(want)).all()
    c = x64 - x64.mean(axis=1, keepdims=True)
    want = c / np.sqrt((c ** 2).mean(axis=1, keepdims=True) + 1e-5) * g + b
    # ... and a mean that is off by its own roundings
    assert (np.abs(ln - want) <= 2 * rel * (np.abs(want) + np.abs(b) + 4 * np.abs(g)) + 1e-6).all()


@pytest.mark.parametrize("n", [4, 252, 256, 260, 764, 768, 772, 1024, 1028, 3072, 3076, 4096, 4100])
@pytest.mark.parametrize("rows", [1, 255, 257])
def test_layer_norm_of_many_rows(hip, rows, n):
    """Rows that waves take 16 bytes at a time, on both sides of each line between the kernels and the last workgroup partly filled; f32 results and
    bf16 ones; some rows far from zero."""
    rng = np.random.default_rng(rows + n)
    x, g, b = (rng.standard_normal(s, dtype=np.float32) for s in ((rows, n), (n,), (n,)))
    x += (np.arange(rows) % 3)[:, None].astype(np.float32)
    f32 = lambda *d: ("F32", list(d))   # noqa: E731
    norm = lambda a, c, d: F.layer_norm(a, c, d, 1e-5)[0]   # noqa: E731
    y = hip_run(hip, program([f32(rows, n), f32(n), f32(n)], lambda a, c, d: [norm(a, c, d)]), [x, g, b])[0]
    y16 = hip_run(hip, program([f32(rows, n), f32(n), f32(n)], lambda a, c, d: [norm(a, c, d).cast("Bf16")]), [x, g, b])[0]
    x64 = x.astype(np.float64)
    c = x64 - x64.mean(axis=1, keepdims=True)
    want = c / np.sqrt((c ** 2).mean(axis=1, keepdims=True) + 1e-5) * g + b
    # as in test_rows; the mean's own roundings are those of values up to 2 + 4 in size, of rows whose spread is 1 (four values: down to a tenth)
    tol = 2 * (np.sqrt(n) * 2.0 ** -24 + 2.0 ** -21) * (np.abs(want) + np.abs(b) + 4 * np.abs(g) * np.maximum(1, 3 / np.sqrt((c ** 2).mean(axis=1, keepdims=True) + 1e-5))) + 1e-6
    assert (np.abs(y - want) <= tol).all()
    assert (np.abs(np.asarray(y16, np.float32) - want) <= tol + 2.0 ** -8 * np.abs(want)).all()


@pytest.mark.parametrize("n", [772, 900, 1024])
def test_layer_norm_of_772_to_1024_values_takes_one_way(hip, n):
    """However many rows there are: bit for bit what each gives in a program of few rows (sums in the same order)."""
    rng = np.random.default_rng(n)
    x, g, b = (rng.standard_normal(s, dtype=np.float32) for s in ((300, n), (n,), (n,)))
    f32 = lambda *d: ("F32", list(d))   # noqa: E731
    run = lambda a: hip_run(hip, program([f32(*a.shape), f32(n), f32(n)], lambda a, c, d: [F.layer_norm(a, c, d, 1e-5)[0]]), [a, g, b])[0]   # noqa: E731
    assert np.array_equal(run(x), np.concatenate([run(x[i:i + 100]) for i in range(0, 300, 100)]))


@pytest.mark.parametrize("ln", [False, True])
@pytest.mark.parametrize("m,k,n", [(2, 64, 48), (8, 3072, 576), (16, 512, 2304)])
def test_one_norm_of_several_layers(hip, ln, m, k, n):
    """Layers of a few rows under one norm read rows that were normed once: bit for bit what each gives in a program of its own, and a norm
    with other gains, or of other rows, is another one."""
    rng = np.random.default_rng(m + k + n)
    x = rng.standard_normal((m, k), dtype=np.float32)
    gs = [(1 + 0.1 * rng.standard_normal(k)).astype(np.float32) for _ in range(2)]
    b = (0.1 * rng.standard_normal(k)).astype(np.float32)
    ws = [rng.standard_normal((k, n), dtype=np.float32) * np.float32(k ** -0.5) for _ in range(4)]
    norm = lambda a, g, c: (F.layer_norm(a, g, c, 1e-5) if ln else F.rms_norm(a, g, 1e-5))[0].cast("Bf16")   # noqa: E731
    bodies = [lambda h, h2, w, a, g, c: F.linear(h, w[0], out_dtype="F32"),
              lambda h, h2, w, a, g, c: F.linear(h2, w[1], out_dtype="F32"),
              lambda h, h2, w, a, g, c: F.swiglu(F.linear(h, w[2]), F.linear(h, w[3])),
              lambda h, h2, w, a, g, c: F.linear(norm(a + a, g, c), w[1], out_dtype="F32"),
              lambda h, h2, w, a, g, c: F.linear(h, w[1], out_dtype="F32")]
    specs = [("F32", [m, k]), ("F32", [k]), ("F32", [k]), ("F32", [k])] + [("Bf16", [k, n])] * 4
    args = [x, *gs, b, *ws]

    def run(which):
        got = hip_run(hip, program(specs, lambda a, g, g2, c, *w: [bodies[i](norm(a, g, c), norm(a, g2, c), w, a, g, c) for i in which]), args)
        launches.append(hip.counter("last_program_launches"))
        return got

    launches = []
    together = run(range(5))
    for i, got in enumerate(together):
        assert np.array_equal(np.asarray(got, np.float32), np.asarray(run([i])[0], np.float32)), i
    assert launches[0] == sum(launches[1:]) - 2, launches   # three layers under one norm
    h64 = x.astype(np.float64) - (x.astype(np.float64).mean(1, keepdims=True) if ln else 0)
    h64 = h64 / np.sqrt((h64 ** 2).mean(1, keepdims=True) + 1e-5) * gs[0] + (b if ln else 0)
    want = h64 @ ws[0].astype(np.float64)
    # the normed row and the weights rounded to bf16: 2^-9 each, of the products' root mean square in the mean; ten times that
    assert np.abs(together[0] - want).max() <= 10 * 2.0 ** -8.5 * np.sqrt((h64 ** 2).mean() * (ws[0] ** 2).mean() * k)


@pytest.mark.parametrize("scheme,ln", [("bf16", False), ("bf16", True), ("w8", False), ("w4g128", False)])   # (a layer of codes takes no layer norm in)
@pytest.mark.parametrize("m,k,n", [(2, 128, 48), (8, 1024, 576), (16, 512, 2304)])
def test_one_norm_of_layers_with_operands(hip, scheme, ln, m, k, n):
    """The same of layers that have a bias, a residual, both or neither, between their weights and the norm's gains, and of int8 and int4 codes with their
    scales; a layer under other gains stands between them."""
    rng = np.random.default_rng(m + k + n)
    x, r = (rng.standard_normal((m, d), dtype=np.float32) for d in (k, n))
    gs = [(1 + 0.1 * rng.standard_normal(k)).astype(np.float32) for _ in range(2)]
    b = (0.1 * rng.standard_normal(k)).astype(np.float32)
    bias = rng.standard_normal(n, dtype=np.float32)
    ws = [rng.standard_normal((k, n), dtype=np.float32) * np.float32(k ** -0.5) for _ in range(5)]
    norm = lambda a, g, c: (F.layer_norm(a, g, c, 1e-5) if ln else F.rms_norm(a, g, 1e-5))[0].cast("Bf16")   # noqa: E731
    if scheme == "bf16":
        weights, per, wspecs = ws, 1, [("Bf16", [k, n])] * 5
        layer = lambda h, w, *more: F.linear(h, *w, *more)   # noqa: E731
    else:
        weights = [t for w in ws for t in (po.quantize_int8_per_channel if scheme == "w8" else po.quantize_int4_g128)(w)]
        per, wspecs = 2, ([("Si8", [k, n]), ("Bf16", [n])] if scheme == "w8" else [("Ui8", [k // 2, n]), ("Bf16", [k // 128, n])]) * 5
        layer = lambda h, w, *more: F.linear_quantized(h, *w, *more)   # noqa: E731
    bodies = [lambda h, h2, w, d, e: layer(h, w[0], d),
              lambda h, h2, w, d, e: layer(h, w[1]) + e,
              lambda h, h2, w, d, e: layer(h2, w[2], d),
              lambda h, h2, w, d, e: layer(h, w[3], d) + e,
              lambda h, h2, w, d, e: layer(h, w[4])]
    specs = [("F32", [m, k]), ("F32", [k]), ("F32", [k]), ("F32", [k]), ("Bf16", [n]), ("Bf16", [m, n])] + wspecs
    args = [x, *gs, b, bias, r, *weights]

    def run(which):
        got = hip_run(hip, program(specs, lambda a, g, g2, c, d, e, *w: [bodies[i](norm(a, g, c), norm(a, g2, c), [w[per * j:per * j + per] for j in range(5)], d, e) for i in which]), args)
        launches.append(hip.counter("last_program_launches"))
        return got

    launches = []
    together = run(range(5))
    for i, got in enumerate(together):
        assert np.array_equal(np.asarray(got, np.float32), np.asarray(run([i])[0], np.float32)), i
    assert launches[0] == sum(launches[1:]) - 3, launches   # four layers under one norm
