"""A prompt's attention fused with the rotation of its rows and the updates of the caches (Fuser::pass_prefill_caches): one sequence
and stacked batches, against the oracle and against float64."""
import numpy as np
import pytest

from parity import assert_close, check_program, hip_run, oracle_run
from gptrs_amd import functional as F
from gptrs_amd.backend import fusion_report
from gptrs_amd.ptir import FunctionBuilder, Program, Tensor, bf16_bits_to_f32, f32_to_bf16_bits

CASES = [  # sequences, rows, query heads, key heads, head size, rotated, cache rows, first row that the update names
    (1, 2, 2, 2, 32, True, 2, 0), (1, 33, 4, 1, 32, True, 64, 5), (2, 32, 2, 2, 64, False, 32, 0), (3, 31, 8, 2, 64, True, 40, 100),
    (16, 3, 4, 4, 32, False, 8, -2), (2, 129, 8, 1, 128, True, 160, 7), (1, 200, 4, 2, 128, False, 256, 0), (2, 65, 6, 3, 64, True, 65, 0),
    # one row tile, whose workgroups fill the caches: 32, 64 and 128 rows by query heads to a key head, two workgroups to a key head, and one row more
    (2, 32, 8, 1, 128, True, 33, 1), (1, 64, 4, 2, 128, True, 64, 0), (2, 128, 2, 2, 64, False, 130, 2), (1, 127, 2, 2, 32, True, 128, 0), (1, 65, 4, 2, 64, False, 70, 3),
    (3, 5, 3, 1, 32, False, 6, 1),     # three query heads to a key head: the unfused series
]


def program(dt, B, T, hq, hkv, dh, rot, cap, base=None):
    fb = FunctionBuilder("main", dt)
    cfg = F.AttentionConfig(hq * dh, hq, hkv, dh)
    qkv = fb.param(dt, [B * T, (hq + 2 * hkv) * dh])
    tabs = [fb.param(dt, [T, dh // 2]) for _ in range(2)] if rot else []
    starts = fb.param("Si32", [3])
    caches = [fb.param(dt, base or [hkv, cap, dh]) for _ in range(2 * B)]
    ctxs, outs = [], []
    for b in range(B):
        rows = qkv if B == 1 else qkv.slice([b * T, 0], [T, qkv.dims[1]])
        if rot:
            rows = F.apply_rope_qkv_packed(cfg, rows, *tabs)
        ctx, k, v = F.attention(cfg, rows, None)
        ctxs.append(ctx)
        outs += [F.dynamic_update_slice_into(caches[2 * b], k, starts), F.dynamic_update_slice_into(caches[2 * b + 1], v, starts)]
    fb.set_results([ctxs[0] if B == 1 else Tensor.concat(0, ctxs)] + outs)
    return Program(fb)


def inputs(B, T, hq, hkv, dh, rot, cap, first, seed):
    rng = np.random.default_rng(seed)
    out = [rng.standard_normal((B * T, (hq + 2 * hkv) * dh), dtype=np.float32)]
    if rot:
        ang = np.arange(T)[:, None] * 100.0 ** (-np.arange(dh // 2) / (dh // 2))
        out += [np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)]
    return out + [np.array([0, first, 0], np.int32)] + [rng.standard_normal((hkv, cap, dh), dtype=np.float32) for _ in range(2 * B)]


@pytest.mark.parametrize("case", CASES)
def test_is_one_instruction(case):
    B, T, hq, hkv, dh, rot, cap, _ = case
    rep = fusion_report(program("F32", B, T, hq, hkv, dh, rot, cap))
    if hq // hkv == 3:
        assert "DynamicUpdateSlice" in rep
    else:
        assert rep == ["fused.attention_prefill_caches" + ("+rope" if rot else "")]


def test_a_cache_that_the_program_computes_stays_apart():
    """The update's base depends on the attention: taking both up in one instruction would make a cycle."""
    fb = FunctionBuilder("main", "F32")
    qkv, starts = fb.param("F32", [8, 96]), fb.param("Si32", [3])
    cfg = F.AttentionConfig(32, 1, 1, 32)
    ctx, k, v = F.attention(cfg, qkv, None)
    base = ctx.reshape([1, 8, 32])
    fb.set_results([ctx, F.dynamic_update_slice_into(base, k, starts), F.dynamic_update_slice_into(base, v, starts)])
    assert fusion_report(Program(fb)).count("DynamicUpdateSlice") == 2


def tables_of_values(B):
    """The rotation's tables are read back from the values that one of the updates has stored."""
    T, hd, cap = 8, 32, 16
    fb = FunctionBuilder("main", "F32")
    cfg = F.AttentionConfig(hd, 1, 1, hd)
    qkv, starts, sin = fb.param("F32", [B * T, 3 * hd]), fb.param("Si32", [3]), fb.param("F32", [T, hd // 2])
    caches = [fb.param("F32", [1, cap, hd]) for _ in range(2 * B)]
    parts = [qkv if B == 1 else qkv.slice([b * T, 0], [T, 3 * hd]) for b in range(B)]
    new_v = [F.dynamic_update_slice_into(caches[2 * b + 1], parts[b].slice([0, 2 * hd], [T, hd]).reshape([T, 1, hd]).transpose([1, 0, 2]), starts) for b in range(B)]
    cos = new_v[-1].reshape([cap, hd]).slice([0, 0], [T, hd // 2])
    ctxs, outs = [], []
    for b in range(B):
        ctx, k, _ = F.attention(cfg, F.apply_rope_qkv_packed(cfg, parts[b], cos, sin), None)
        ctxs.append(ctx)
        outs += [F.dynamic_update_slice_into(caches[2 * b], k, starts), new_v[b]]
    fb.set_results([ctxs[0] if B == 1 else Tensor.concat(0, ctxs)] + outs)
    return Program(fb)


@pytest.mark.parametrize("B", [1, 2])
def test_tables_made_of_stored_values_stay_apart(B):
    """The tables depend on the update of the values: taking both up in one instruction would make a cycle."""
    assert sum("DynamicUpdateSlice" in line for line in fusion_report(tables_of_values(B))) >= 2


@pytest.mark.gpu
@pytest.mark.parametrize("B", [1, 2])
def test_tables_made_of_stored_values(hip, B):
    rng = np.random.default_rng(8)
    args = [rng.standard_normal((8 * B, 96), dtype=np.float32), np.array([0, 3, 0], np.int32), rng.standard_normal((8, 16), dtype=np.float32)]
    args += [rng.standard_normal((1, 16, 32), dtype=np.float32) for _ in range(2 * B)]
    check_program(hip, tables_of_values(B), args, what=f"{B} sequences")


# tensors that hold more than the keys (or values) of one layer: more heads, wider rows, both; where the update goes
BASES = [((1, 8, 4, 2, 32, False), [6, 16, 32], (4, 3, 0)), ((1, 33, 2, 2, 32, True), [2, 64, 64], (0, 5, 32)), ((2, 9, 4, 2, 64, True), [4, 12, 72], (1, 2, 8)),
         ((3, 5, 2, 1, 32, False), [2, 5, 33], (7, -1, 1)), ((1, 17, 4, 4, 64, False), [5, 17, 64], (1, 0, 0))]


def test_wider_and_taller_bases_keep_their_updates():
    for (B, T, hq, hkv, dh, rot), base, _ in BASES:
        for dt in ("F32", "Bf16"):
            rep = fusion_report(program(dt, B, T, hq, hkv, dh, rot, 1, base))
            assert sum("DynamicUpdateSlice" in line for line in rep) == 2 * B, (base, rep)
            assert not any("prefill_caches" in line for line in rep), (base, rep)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ["F32", "Bf16"])
def test_wider_and_taller_bases(hip, dt):
    """Heads, rows and columns of the start all count; what the update does not name stays."""
    for (B, T, hq, hkv, dh, rot), base, at in BASES:
        args = inputs(B, T, hq, hkv, dh, rot, 1, 0, 5)[:3 if rot else 1] + [np.array(at, np.int32)]
        rng = np.random.default_rng(6)
        args += [rng.standard_normal(base, dtype=np.float32) for _ in range(2 * B)]
        if dt == "F32":
            check_program(hip, program(dt, B, T, hq, hkv, dh, rot, 1, base), args, what=f"{base} at {at}")
            continue
        args = [a if a.dtype == np.int32 else bf16_bits_to_f32(f32_to_bf16_bits(a)) for a in args]
        got = hip_run(hip, program(dt, B, T, hq, hkv, dh, rot, 1, base), args)
        want = oracle_run(program("F32", B, T, hq, hkv, dh, rot, 1, base), args)
        assert_close(got[0], want[0], atol=3e-2, rtol=2.0 ** -7, what=f"context {base}")      # as in test_bf16
        for i, (g, w) in enumerate(zip(got[1:], want[1:])):
            if i % 2 == 0 and rot:
                assert_close(g, w, atol=1e-6, rtol=2.0 ** -8, what=f"keys {base}")
            else:
                assert np.array_equal(g, w), f"cache {i} {base}"


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES)
def test_f32(hip, case):
    B, T, hq, hkv, dh, rot, cap, first = case
    check_program(hip, program("F32", B, T, hq, hkv, dh, rot, cap), inputs(B, T, hq, hkv, dh, rot, cap, first, 3), what=str(case))


@pytest.mark.gpu
@pytest.mark.parametrize("case", [(1, 7, 12, 12, 64, False, 16, 0), (3, 16, 4, 2, 64, False, 20, 3), (2, 15, 4, 1, 128, False, 15, 0), (16, 2, 2, 2, 128, False, 9, -1),
                                  (1, 16, 8, 8, 128, False, 16, 5), (1, 17, 12, 12, 64, False, 17, 0), (2, 16, 8, 2, 64, True, 16, 0)])
def test_f32_of_few_rows(hip, case):
    """Up to 16 rows without rotation a wave takes each row by itself; one row more, and rotated rows, go another way."""
    B, T, hq, hkv, dh, rot, cap, first = case
    check_program(hip, program("F32", B, T, hq, hkv, dh, rot, cap), inputs(B, T, hq, hkv, dh, rot, cap, first, 11), what=str(case))


@pytest.mark.gpu
@pytest.mark.parametrize("case,launches", [((1, 65, 4, 4, 64, True, 70, 0), 1), ((2, 100, 2, 2, 128, False, 100, 0), 1), ((1, 127, 12, 12, 32, True, 128, 1), 1),
                                           ((1, 128, 4, 4, 64, True, 130, 0), 2), ((1, 65, 4, 2, 64, True, 70, 0), 2), ((1, 64, 4, 2, 64, True, 70, 0), 1)])
def test_one_row_tile_fills_the_caches_itself(hip, case, launches):
    """Where a workgroup sees every row of its key head the caches are filled on the way: no launch for them, and no key groups, of which each sees a part."""
    B, T, hq, hkv, dh, rot, cap, first = case
    p, args = program("Bf16", B, T, hq, hkv, dh, rot, cap), inputs(B, T, hq, hkv, dh, rot, cap, first, 12)
    got = hip_run(hip, p, args, [False] * (len(args) - 2 * B) + [True] * 2 * B)
    assert hip.counter("last_program_launches") == launches
    want = oracle_run(program("F32", B, T, hq, hkv, dh, rot, cap), [a if a.dtype == np.int32 else bf16_bits_to_f32(f32_to_bf16_bits(a)).reshape(a.shape) for a in args])
    for i, (g, w) in enumerate(zip(got, want)):   # rotated rows and the attention's output are rounded once or twice
        assert_close(g, w, atol=2e-2, rtol=2e-2, what=f"{case} result {i}")


@pytest.mark.gpu
@pytest.mark.parametrize("donate", [False, True])
@pytest.mark.parametrize("case", CASES[:-1])
def test_bf16(hip, case, donate):
    B, T, hq, hkv, dh, rot, cap, first = case
    args = [a if a.dtype == np.int32 else bf16_bits_to_f32(f32_to_bf16_bits(a)) for a in inputs(B, T, hq, hkv, dh, rot, cap, first, 4)]
    n_in = 4 if rot else 2
    got = hip_run(hip, program("Bf16", B, T, hq, hkv, dh, rot, cap), args, [False] * n_in + [donate] * (2 * B))
    want = oracle_run(program("F32", B, T, hq, hkv, dh, rot, cap), args)
    # values between -5 and 5: rotated rows rounded once (2^-9 of up to 7), probabilities and the context once more
    assert_close(got[0], want[0], atol=3e-2, rtol=2.0 ** -7, what=f"context {case}")
    for i, (g, w) in enumerate(zip(got[1:], want[1:])):
        if i % 2 == 0 and rot:
            assert_close(g, w, atol=1e-6, rtol=2.0 ** -8, what=f"keys {case}")
        else:
            assert np.array_equal(g, w), f"cache {i} {case}"
