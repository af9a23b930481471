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


def test_depths_of_the_shapes_that_parity_tests_take():
    """The oracle comparisons cover the long march as well as the shortest chunks: what they say of their shapes' chunks
    is so."""
    one = {s: s[2] for s in C.DEEP_TYPE2 + C.DEEP_TYPE1 + [C.DEEP_ETTI, C.DEEP_ETTI_MIXED, C.DEEP_ORDER16]}
    for s in C.DEEP_TYPE2:
        for name, rows in (("FWD_DRV", 16), ("FWD_UPDATE", 8), ("ADJ_DRV", 8), ("ADJ_UPDATE", 16), ("RHO_GRAD", 8)):
            assert C.stencil_depth(s, name + "_CHUNK", rows) == one[s], name
    for s in C.DEEP_TYPE1:
        assert C.stencil_depth(s, "T1_CHUNK", 8) == one[s]
    for name, rows in (("FWD_DRV16", 16), ("FWD_UPDATE16", 8), ("ADJ_DRV16", 8), ("ADJ_UPDATE16", 8)):
        assert C.stencil_depth(C.DEEP_ORDER16, name + "_CHUNK", rows) == one[C.DEEP_ORDER16], name
    for name, s in (("VELOCITY", C.DEEP_ETTI), ("STRAIN", C.DEEP_ETTI), ("MIXED", C.DEEP_ETTI_MIXED)):
        assert C.stencil_depth(s, name + "_CHUNK", 8) == one[s], name
    s = C.THREE_QUARTERS_ETTI_MIXED
    assert C.stencil_depth(s, "MIXED_CHUNK", 8) == 100 > C.depth(100, 768, 1024, 9.0, 256)
    small = (70, 19, 67)
    assert all(C.stencil_depth(small, n, r) <= 4 for n in C.chunks() for r in (8, 16))
    for p in (0, 1):
        assert C.fused_depth(C.DEEP_FUSED, p, 64) == 60 and C.fused_depth(C.DEEP_FUSED, p, 16) == 15
        assert C.fused_depth(C.TWO_CHUNKS_FUSED, p, 64) == 35
        assert C.fused_depth(small, p, 64) == 2


def test_deepest_chunk_that_fills_a_round():
    """`full`: the deepest chunk is taken where its blocks fill that share of one round, no more than one; else the rounds
    decide."""
    for tiles, nz, deep in ((768, 200, True), (684, 200, True), (640, 200, False), (1025, 200, False), (384, 400, True)):
        cut = C.depth(nz, tiles, 1024, 9.0, 256)
        assert C.depth(nz, tiles, 1024, 9.0, 256, full=0.667) == (200 if deep else cut)
