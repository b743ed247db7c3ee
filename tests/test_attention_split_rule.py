"""The rule that cuts the last, partial round of attention items into key ranges,
asked on the host for a device of 256 CUs."""

import pytest

from taomate_hd_amd import _native

WS = 1 << 40


def _ranges(items, tiles, dim, i8, ws=WS, cus=256):
    return _native.load().tmhd_attn_last_round_ranges(items, tiles, dim, i8, ws, cus)


# items, key tiles, head_dim, INT8-QK, range counts within 10% of the fastest one measured
# (whole, they took 1.2 to 1.4 times as long; the last four, cut into more, 1.1 to 1.2 times)
@pytest.mark.parametrize(
    "items,tiles,dim,i8,good",
    [
        (5, 8, 128, 0, (3, 4)), (8, 9, 128, 0, (3, 4)), (8, 10, 128, 1, (3, 4, 5)), (4, 8, 128, 1, (4,)),
        (21, 12, 128, 1, (3, 4)), (5, 10, 64, 0, (4, 5)), (6, 11, 64, 1, (4, 5)), (22, 12, 64, 1, (4, 5)),
        (8, 27, 128, 0, range(4, 11)), (8, 34, 128, 1, range(5, 14)), (28, 17, 64, 0, range(3, 7)),
        (32, 15, 64, 0, range(3, 6)),
    ],
)
def test_small_calls(items, tiles, dim, i8, good):
    assert _ranges(items, tiles, dim, i8) in good


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("i8", [0, 1])
def test_limits(dim, i8):
    slots = 256 * (2 if i8 else 1)
    assert _ranges(slots, 100, dim, i8) == _ranges(3 * slots, 100, dim, i8) == 1  # whole rounds
    assert _ranges(5, 1, dim, i8) == _ranges(5, 3, dim, i8) == 1  # two tiles to a range
    assert _ranges(5, 100, dim, i8, ws=0) == 1
    for items in (1, 3, 40, 300, 700):
        for tiles in (4, 8, 33, 250):
            n = _ranges(items, tiles, dim, i8)
            assert 1 <= n <= 16 and 2 * n <= tiles
            # with a workspace for two workgroups' parts: whole, or what fits them
            few = _ranges(items, tiles, dim, i8, ws=4 * 256 * (dim + 1) * 4)
            assert few == 1 or few * (items % slots) <= 2
    assert _ranges(0, 8, dim, i8) == _ranges(8, 0, dim, i8) == _ranges(8, 8, 96, i8) == -1
