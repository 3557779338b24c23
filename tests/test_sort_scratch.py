"""The radix sort's scratch: sized for a reserved capacity, it holds the digit counts of every smaller
sort too.  CPU only: the library's own size functions, no kernel runs."""
import ctypes as C

import pytest

import cnhip

DIGITS = 256


@pytest.fixture(scope="module")
def sort():
    lib = cnhip.load_library()
    words, rounds = lib._ZN2cn18sort_scratch_wordsEj, lib._ZN2cn11sort_roundsEj
    words.restype, words.argtypes = C.c_size_t, [C.c_uint32]
    rounds.restype, rounds.argtypes = C.c_uint32, [C.c_uint32]
    return words, rounds


def needed(n, rounds):
    """Words a sort of n pairs touches: counts of its tiles (256 x rounds pairs each), then the totals."""
    tile = 256 * rounds(n)
    return DIGITS * ((n + tile - 1) // tile) + DIGITS


def sizes():
    """Around every power of two and midway between them, where a rule on the size may change."""
    out = {1, 2, 3}
    for b in range(6, 25):
        for base in (1 << b, 3 << (b - 1)):
            out.update((base - 1, base, base + 1))
    return sorted(out | {4_000_000, 4_096_000, 5_000_000, 8_388_607, 8_813_865})


@pytest.mark.parametrize("capacity", [1, 4097, 131_072, 131_073, 262_143, 1 << 20, 4_194_304, 4_194_305, 5_000_000,
                                      8_388_608, 8_388_609, 16_777_216])
def test_scratch_of_a_capacity_holds_every_smaller_sort(sort, capacity):
    words, rounds = sort
    have = words(capacity)
    for n in sizes():
        if n <= capacity:
            assert have >= needed(n, rounds), (capacity, n)


def test_scratch_grows_with_the_capacity(sort):
    words, _ = sort
    got = [words(n) for n in sizes()]
    assert got == sorted(got)


def test_noalloc_scratch_holds_its_largest_sort(sort):
    from cnhip import abi
    words, _ = sort
    assert words(abi.CN_NOALLOC_MAX_PAIRS) <= DIGITS * (abi.CN_NOALLOC_MAX_PAIRS // 2048) + DIGITS
