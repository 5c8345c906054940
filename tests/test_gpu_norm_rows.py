"""Rows normalised with their gains held in registers: lengths at the edges of a thread's eight values, of a wave and of a workgroup,
the first length that is read again instead, lengths that are no multiple of eight.  Against float64."""
import numpy as np
import pytest

from parity import hip_run
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
