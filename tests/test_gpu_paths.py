"""GPU tests of single paths of the sort, each at the sizes where it can go
wrong, bit-exact against the oracle."""
import numpy as np
import pytest

from strsets import pack, random_strings

pytestmark = pytest.mark.gpu


def check(ctx, oracle, arena, offs, with_lcp=True):
    perm, lcp = ctx.sort(arena, offs, with_lcp=with_lcp)
    r, msg = oracle.verify(arena, offs, perm, lcp) if with_lcp else oracle.verify(arena, offs, perm)
    assert r == 0, msg


@pytest.mark.parametrize("syncs", [1, 2, 3])
def test_new_context_ignores_recycled_sequence_words(ps5, oracle, syncs):
    """a context created after another one's pinned memory was returned sorts
    from its own staged counters, whatever number the memory still holds"""
    small = pack(random_strings(5000, 0, 12, b"abcdefgh", 11))
    large = pack(random_strings(60000, 0, 40, b"ab", 12))
    first = ps5.Context(0)
    first.set_planning(1)
    for _ in range(syncs):
        first.sort(*small)
    first.close()
    second = ps5.Context(0)
    try:
        check(second, oracle, *large)
    finally:
        second.close()
