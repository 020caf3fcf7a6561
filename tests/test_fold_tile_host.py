"""Tile shapes of the folded plan form on trees near and beyond the reach of
its kernel's 32-bit byte offsets (host only)."""

import numpy as np
import pytest

from volumential_amd import _capi


def _tile(dim, q, cplx, nb, n_rhs):
    out = np.full(5, -1, dtype=np.int64)
    _capi.check(_capi.lib().vl1_plan_fold_tile_host(dim, q, int(cplx), nb, nb, n_rhs,
                                                    out.ctypes.data), "vl1_plan_fold_tile_host")
    return dict(zip(("folded", "columns", "rhs", "boxes", "box_bytes"), out.tolist()))


# uniform level-10 quadtrees and level-6 octrees, the largest that fit at 8
# densities per tile and one box more, and the same at one density per tile
# (the densities of a box take 32 bytes per K group and density: 56 groups in
# 3D q = 6, 16 in 2D q = 8 and 32 there for complex data)
CASES = [(2, 8, False, 1 << 20, 8), (2, 8, True, 1 << 20, 4), (3, 6, True, 1 << 18, 8),
         (3, 8, False, 1 << 18, 8)]
for dim, q, cplx, kg in ((3, 6, False, 56), (2, 8, False, 16), (2, 8, True, 32)):
    for rc in (8, 4, 1):
        most = (1 << 32) // (32 * kg * rc) - 2
        CASES += [(dim, q, cplx, most, 8), (dim, q, cplx, most + 1, 8)]


@pytest.mark.parametrize("dim,q,cplx,nb,n_rhs", CASES)
@pytest.mark.parametrize("factor", [1, 8])
def test_offsets_reach_every_box(dim, q, cplx, nb, n_rhs, factor):
    """Box offsets up to the zero box (index nb), and a lane's share of one
    more box, stay below 2^32; plans beyond that at one density per tile do
    not fold."""
    t = _tile(dim, q, cplx, nb, n_rhs * factor)
    one = 32 * {(2, 8, False): 16, (2, 8, True): 32, (3, 6, False): 56, (3, 6, True): 112,
                (3, 8, False): 128}[dim, q, cplx]
    assert t["folded"] == ((nb + 2) * one <= 1 << 32)
    if t["folded"]:
        assert t["box_bytes"] == t["rhs"] * one
        assert (nb + 2) * t["box_bytes"] <= 1 << 32
        assert t["rhs"] >= 1 and t["boxes"] * t["rhs"] <= t["columns"]
        # no fewer densities than the offsets ask for
        if t["rhs"] < min(8, n_rhs * factor):
            assert (nb + 2) * one * 2 * t["rhs"] > 1 << 32


def test_small_trees_keep_eight_densities():
    assert _tile(3, 6, False, 32768, 64)["rhs"] == 8
    assert _tile(2, 8, True, 4096, 24)["rhs"] == 8


@pytest.mark.parametrize("n_rhs", [7, 11, 13, 17, 19, 23, 29, 31, 37, 41, 43, 47, 53, 59, 61])
def test_prime_counts_share_tiles(n_rhs):
    """Prime density counts take tiles of several densities with a few columns
    idle, not one density per tile."""
    t = _tile(3, 4, False, 4096, n_rhs)
    groups = -(-n_rhs // t["rhs"])
    assert t["rhs"] >= 2
    assert n_rhs * t["boxes"] >= 0.85 * groups * t["columns"]
