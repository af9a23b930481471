"""The rule that cuts a z range into the chunks of the z-marching kernels (csrc/common.h chunk_depth), on the host."""
import pytest

import chunk_rule as C

INT_MAX = 2**31 - 1


@pytest.mark.parametrize("nz,tiles", [(1, 1), (64, 8), (300, 17), (512, 512), (5, 100000)])
def test_any_cap(nz, tiles):
    """Every cap that a caller may pass as zblock gives a depth of 1 .. min(cap, nz); a cap past the range (the largest
    int as "no limit") is the same as the range."""
    for warm in (4.0, 12.5):
        for cap in (1, 2, 7, nz, INT_MAX - nz, INT_MAX):
            assert 1 <= C.depth(nz, tiles, 256, warm, cap) <= min(cap, nz)
        assert C.depth(nz, tiles, 256, warm, INT_MAX) == C.depth(nz, tiles, 256, warm, nz)


def test_full_rounds_keep_the_deepest_chunk():
    """A tile count that is a whole number of rounds gains nothing by cutting z."""
    for slots in (256, 512, 1024):
        for nz in (2, 48, 200):
            assert C.depth(nz, 1024, slots, 9.0, 256) == nz
