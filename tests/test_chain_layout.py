"""The decode chain's packed copies (kernels_chain.hip) as the host lays them out, without a device (256 workgroups)."""
import ctypes

import numpy as np
import pytest

import __graft_entry__ as entry

entry.load_package()
from gptrs_amd import backend  # noqa: E402

KPW = (2, 4, 8, 1)   # k of a column in 16 / 4 bytes of a word, by format: bf16, int8, int4, f32
GRID, WAVES, STEP = 256, 8, 3


def lib():
    lib = backend.load_library()
    size, word = lib._ZN5gptrs1k18chain_weight_bytesEllbi, lib._ZN5gptrs1k17chain_weight_wordEllbill   # chain_weight_bytes, chain_weight_word
    size.argtypes, size.restype = [ctypes.c_int64] * 2 + [ctypes.c_bool, ctypes.c_int], ctypes.c_size_t
    word.argtypes, word.restype = [ctypes.c_int64] * 2 + [ctypes.c_bool, ctypes.c_int] + [ctypes.c_int64] * 2, ctypes.c_int64
    asked = lib._ZN5gptrs1k16chain_wave_wordsEllbiiiPli   # chain_wave_words: the walk that a wave makes
    asked.argtypes, asked.restype = [ctypes.c_int64] * 2 + [ctypes.c_bool] + [ctypes.c_int] * 3 + [ctypes.c_void_p, ctypes.c_int], ctypes.c_int
    return size, word, asked


@pytest.mark.parametrize("fmt,k,n,dual", [(0, 3072, 64, False), (0, 9216, 64, False), (0, 24576, 8, False), (0, 4, 4, False), (0, 132, 1020, False), (0, 132, 1028, False),
                                          (0, 9216, 1536, False), (0, 3072, 6176, False), (0, 1156, 7172, False), (0, 260, 8204, False), (0, 256, 320, True), (1, 3072, 3072, False),
                                          (1, 9216, 3072, False), (1, 640, 1028, True), (2, 2176, 8204, False), (3, 768, 768, False), (3, 768, 2304, False), (3, 768, 3073, False),
                                          (3, 3072, 768, False), (3, 4608, 2052, False),
                                          (2, 3072, 32768, False), (0, 1536, 1000, True), (3, 1536, 4608, False)])
def test_a_copy_holds_every_word_once(fmt, k, n, dual):
    """No larger than the matrix in whole words, and in the order in which waves ask for it: whole steps at one distance, the rest one word behind the other."""
    size, word, asked = lib()
    tiles, chunks = -(-(2 * n if dual else n) // 4), -(-k // (64 * KPW[fmt]))
    assert size(k, n, dual, fmt) == tiles * chunks * 1024
    at = np.array([[word(k, n, dual, fmt, t, c) for c in range(chunks)] for t in range(tiles)])
    assert np.array_equal(np.sort(at, axis=None), np.arange(tiles * chunks))
    lo, more = divmod(tiles, GRID)
    active = GRID if lo else more
    whole = max(lo, 1) * chunks // WAVES // STEP
    whole = whole if whole >= 2 else 0
    first = 0
    got = (ctypes.c_int64 * (tiles * chunks + 1))()
    for b in range(active, GRID):   # a workgroup without tiles asks for nothing
        assert all(asked(k, n, dual, fmt, b, w, got, len(got)) == 0 for w in range(WAVES))
    for b in range(active):
        mine = at[first:first + lo + (b < more)].reshape(-1)
        first += lo + (b < more)
        for w in range(WAVES):
            words = mine[len(mine) * w // WAVES:len(mine) * (w + 1) // WAVES]
            assert asked(k, n, dual, fmt, b, w, got, len(got)) == len(words) and list(got[:len(words)]) == list(words)
            i = np.arange(len(words))
            want = (i // STEP * active + b) * WAVES * STEP + w * STEP + i % STEP
            rest = i >= STEP * whole
            assert np.array_equal(words[~rest], want[~rest])
            assert rest.sum() == 0 or (words[rest][0] >= whole * active * WAVES * STEP and (np.diff(words[rest]) == 1).all())
            if whole and (more == 0 or lo == 0):
                assert rest.sum() <= STEP
    assert first == tiles
