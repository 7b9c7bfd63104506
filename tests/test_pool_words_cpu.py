"""The CFL words of a pool job share its items: of the blocks of a launch, each runs one item of the
work list; the items of a job, which follow one another there, take its words in turn on every XCD
that runs them (block b is on XCD b % 8), and blocks that start together take different words. (A
word with more than its share is a queue of atomics.)"""
import collections
import ctypes as C

import pytest

from euler_kokkos_amd import pool

WORDS = 32


@pytest.mark.parametrize("tiles", [[1], [7], [8], [16, 17, 15], [50 * k + 3 for k in range(1, 25)], [4] * 700, [3000, 1, 4000],
                                   [4096]])
def test_items_of_a_job_take_its_words_in_turn(tiles):
    L, n = pool._lib(), sum(tiles)
    item, word = C.c_uint(), C.c_uint()
    at = []
    for b in range(n):
        assert L.ek_pool_test_item(b, n, C.byref(item), C.byref(word)) == 0
        at.append((item.value, word.value))
    assert sorted(i for i, _ in at) == list(range(n))
    full = n // 8 * 8  # blocks in XCD order; the rest keep their place
    owner = [j for j, t in enumerate(tiles) for _ in range(t)]
    used = collections.defaultdict(collections.Counter)
    for b in range(full):
        used[owner[at[b][0]], b % 8][at[b][1]] += 1
    for c in used.values():
        count = sum(c.values())
        assert len(c) == min(count, WORDS) and max(c.values()) == -(-count // WORDS)
    for b in range(0, full - WORDS + 1, WORDS):
        assert len({w for _, w in at[b:b + WORDS]}) == WORDS
    assert L.ek_pool_test_item(n, n, C.byref(item), C.byref(word)) != 0
