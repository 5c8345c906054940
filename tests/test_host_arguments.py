"""What the models prepare on the host ahead of a program: tokens and positions as arrays, rotation tables kept with the model, inputs of a
program whose parameters have been found."""
import numpy as np
import pytest

from oracle_backend import OracleBackend
from gptrs_amd import functional as F
from gptrs_amd import models


@pytest.mark.parametrize("rows", [[[0]], [[5, 99, 0]], [[1, 2], [3, 4]], [[np.int64(7), True], [np.int32(98)]], [[3.0, 4.5]], [(1, 2)], [np.array([8, 9])]])
def test_tokens(rows):
    got = np.asarray(models._checked_tokens(rows, 100), np.int32)
    np.testing.assert_array_equal(got, np.asarray([t for r in rows for t in r], np.int32))


@pytest.mark.parametrize("rows", [[[100]], [[-1]], [[0, 1], [2, 100]], [[1 << 40]], [[-(1 << 70)]], [[float("nan")]], [[-0.5]]])
def test_tokens_outside(rows):
    with pytest.raises(ValueError, match="out of range"):
        models._checked_tokens(rows, 100)


@pytest.mark.parametrize("dtype", ["F32", "Bf16"])
@pytest.mark.parametrize("scaling", [None, ("linear", 4.0)])
def test_rotation_rows_are_those_of_their_positions(dtype, scaling):
    cfg = models.MinistralConfig(vocab_size=32, context_length=96, embed_dim=32, num_layers=1, num_heads=4, num_kv_heads=2, head_dim=8, ffn_dim=32,
                                 rotary_dim=8, rope_scaling=scaling)
    m = models.Ministral(cfg, OracleBackend(), dtype)

    def rows(start, end):
        return tuple(models._np_to_bytes(x, dtype) for x in F.rotary_cos_sin_cache_slice(start, end - start, m.rope))

    for start, end in ((0, 7), (7, 8), (8, 9), (0, 33), (95, 96), (0, 96), (-2, 3)):
        assert m._rope_rows(start, end) == rows(start, end)
    m.rope.theta = 500.0
    assert m._rope_rows(3, 9) == rows(3, 9)


def test_rotation_rows_formed_by_a_call_are_those_it_asks_for(monkeypatch):
    """A prompt forms its own rows and no more, a step at the end of the kept rows those of the next steps too, and rows behind a gap (caches of an earlier
    program, say) are formed alone: position 100000 does not bring 100000 rows with it."""
    cfg = models.MinistralConfig(vocab_size=32, context_length=1 << 18, embed_dim=32, num_layers=1, num_heads=4, num_kv_heads=2, head_dim=8, ffn_dim=32, rotary_dim=8)
    m = models.Ministral(cfg, OracleBackend(), "Bf16")
    formed = []

    def slice_(start, length, rope, plain=F.rotary_cos_sin_cache_slice):
        formed.append((start, length))
        return plain(start, length, rope)

    def rows(start, end, plain=F.rotary_cos_sin_cache_slice):
        return tuple(models._np_to_bytes(x, "Bf16") for x in plain(start, end - start, m.rope))

    monkeypatch.setattr(F, "rotary_cos_sin_cache_slice", slice_)
    for (start, end), new in (((100000, 100001), [(100000, 1)]), ((0, 333), [(0, 333)]), ((0, 200), []), ((0, 700), [(333, 367)]), ((700, 701), [(700, 64)]), ((701, 702), []),
                              ((763, 764), []), ((764, 765), [(764, 64)]), ((5000, 5001), [(5000, 1)])):
        formed.clear()
        assert m._rope_rows(start, end) == rows(start, end)
        assert formed == new, (start, end)


def test_runs_behind_the_first_see_new_arguments_and_new_parameters():
    cfg = models.GptConfig(vocab_size=24, context_length=16, embed_dim=16, num_layers=1, num_heads=2, mlp_ratio=2)
    be = OracleBackend()
    m = models.Gpt.random(cfg, be, seed=3)

    def logits(tokens):
        return be.to_numpy(m.forward_with_decode_cache(tokens, 0, [None]))

    first, other, again = logits([1, 2, 3]), logits([4, 5, 6]), logits([1, 2, 3])
    np.testing.assert_array_equal(first, again)
    assert not np.array_equal(first, other)
    head = np.random.default_rng(1).standard_normal((16, 24)).astype(np.float32)
    m.set_param("lm_head", head)
    assert not np.array_equal(logits([1, 2, 3]), first)
    fresh = models.Gpt.random(cfg, OracleBackend(), seed=3)
    fresh.set_param("lm_head", head)
    np.testing.assert_array_equal(logits([1, 2, 3]), fresh.backend.to_numpy(fresh.forward_with_decode_cache([1, 2, 3], 0, [None])))


@pytest.mark.parametrize("layers,budget,runs", [(3, 1 << 28, [6]), (5, 2 * 2 * 2 * 32 * 8 * 4, [4, 4, 2]), (3, 1, [2, 2, 2]), (40, 1 << 28, [64, 16])])
def test_growing_caches_hold_little_beside_them(monkeypatch, layers, budget, runs):
    """Caches grow a program at a time, and a program holds no more new bytes than it is allowed, or one layer's."""
    cfg = models.GptConfig(vocab_size=24, context_length=64, embed_dim=16, num_layers=layers, num_heads=2, mlp_ratio=2)
    be = OracleBackend()
    m = models.Gpt.random(cfg, be, seed=3)
    caches = [None] * layers
    m.forward_with_decode_cache([1, 2, 3], 0, caches)
    before = [be.to_numpy(h) for s in caches for h in (s.keys, s.values)]
    monkeypatch.setattr(models, "GROW_BYTES", budget)
    grown, plain = [], m._grow_many
    monkeypatch.setattr(m, "_grow_many", lambda handles, *a: grown.append(len(handles)) or plain(handles, *a))
    rows = [caches]
    m._grow_caches(rows, 32)
    assert grown == runs
    for s, h, old in zip([s for s in caches for _ in (0, 1)], [h for s in caches for h in (s.keys, s.values)], before):
        new = be.to_numpy(h)
        assert s.capacity == 32 and new.shape[1] == 32
        np.testing.assert_array_equal(new[:, :old.shape[1]], old)
        assert not new[:, old.shape[1]:].any()


def test_a_seed_that_is_none_is_refused_before_the_prompt_is_read():
    cfg = models.GptConfig(vocab_size=24, context_length=16, embed_dim=16, num_layers=1, num_heads=2, mlp_ratio=2)
    m = models.Gpt.random(cfg, OracleBackend(), seed=3)
    read = []
    forward, m.forward_with_decode_cache = m.forward_with_decode_cache, lambda *a, **k: read.append(a) or forward(*a, **k)
    for seed, error in ((-1, ValueError), ("seven", TypeError), (1.5, TypeError)):
        with pytest.raises(error):
            models.Generator(m, [1, 2, 3], seed=seed)
        assert not read
    for seed in (0, 7, np.int64(7), [1, 2], np.random.SeedSequence(5)):
        gen = models.Generator(m, [1, 2, 3], seed=seed)
        assert gen._rng.random() == np.random.default_rng(seed if not isinstance(seed, np.random.SeedSequence) else np.random.SeedSequence(5)).random()
