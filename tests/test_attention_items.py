"""The attention work item size (host rule, no GPU calls)."""
import random

import pytest

from ditserve_amd import _lib
from tests.helpers import attn_items

if not _lib.LIB_PATH.exists():
    pytest.skip("libditk.so not built (run python -m ditserve_amd.build)", allow_module_level=True)

CUS = 256  # of an MI355X, and what the library assumes without a GPU


def items(lens, heads, equal=False, joint=False):
    return attn_items(sum(lens), sum(lens), len(lens), heads, equal, joint)


@pytest.mark.parametrize("lens,heads,want", [
    ([1560], 12, 128), ([1280, 1280], 12, 128), ([300, 333, 90], 24, 128), ([600], 24, 128),
    # a round of 256-query items; 128-query ones would take two
    ([978, 985, 75, 157], 24, 256), ([5000, 64, 64, 64, 64, 64], 12, 256), ([3584], 12, 256),
    # 2 rounds for 3, 47 for 94
    ([5888], 12, 256), ([9000, 3000], 12, 256), ([1357, 1357], 24, 256), ([65520], 12, 256)])
def test_choice(lens, heads, want):
    assert items(lens, heads) == want


def test_equal_segments_compare_rounds():
    assert items([77] * 30, 12, equal=True) == 128       # 360 items of either size
    assert items([1300] * 2, 12, equal=True) == 256      # 264 for 144: two rounds for one
    assert items([1280] * 2, 12, equal=True) == 128


def test_ragged_small_items_always_fit_one_round():
    """Whatever the segment lengths behind the totals, 128-query items are only taken
    where all of them run at once (so that they cannot lose to 256-query ones)."""
    rng = random.Random(5)
    taken = 0
    for _ in range(3000):
        heads, n = rng.choice([3, 12, 24]), rng.randint(2, 12)
        lens = [rng.choice([rng.randint(0, 300), rng.randint(1, 3000), 128, 129]) for _ in range(n)]
        if items(lens, heads, joint=rng.random() < 0.5) == 128:
            taken += 1
            assert sum(-(-x // 128) for x in lens) * heads <= CUS, (heads, lens)
    assert taken > 200


def test_bad_sizes():
    lib = _lib.load()
    assert lib.ditk_attn_item_queries(10, 10, 0, 1, 0, 0) == 0 and lib.ditk_attn_item_queries(-1, 1, 1, 1, 0, 0) == 0
