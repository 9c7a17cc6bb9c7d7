"""The order in which an XCD walks the query tiles of causal attention (csrc/index_math.h)."""
import pytest

from kernl_amd.debugger import index_lib


@pytest.mark.parametrize("heads", [1, 2, 15, 16, 17, 33, 80])
@pytest.mark.parametrize("tiles", [1, 2, 9])
@pytest.mark.parametrize("group", [1, 3, 8, 16])
def test_every_item_once_and_the_longest_of_a_group_first(heads, tiles, group):
    items = [index_lib().ranked_item(at, heads, tiles, group) for at in range(heads * tiles)]
    assert sorted(items) == [(head, rank) for head in range(heads) for rank in range(tiles)]
    if tiles > 1:
        for first in range(0, heads, group):
            ranks = [rank for head, rank in items if first <= head < first + group]
            assert ranks == sorted(ranks)


# heads of an XCD, rows, keys, start, head size
@pytest.mark.parametrize("heads, rows, keys, start, size, most", [
    (17, 1071, 1071, 0, 128, 8), (17, 907, 907, 0, 64, 16), (33, 700, 800, 100, 64, 16), (3, 2000, 2000, 0, 128, 8),
    (79, 264, 7960, 7696, 64, 3), (32, 981, 5849, 4868, 128, 2), (8, 100, 600, 500, 64, 8), (5, 64, 1 << 20, (1 << 20) - 64, 128, 1)])
def test_groups_are_alike_and_fit_the_cache_of_an_xcd(heads, rows, keys, start, size, most):
    group = index_lib().rank_group(heads, rows, keys, start, size)
    groups = -(-heads // most)
    assert group == -(-heads // groups)
    last = heads - (-(-heads // group) - 1) * group
    assert 1 <= last <= group <= most
    if 2 * start >= rows and group > 1:  # new rows over a cache
        assert group * keys * size * 4 <= 6 << 20
