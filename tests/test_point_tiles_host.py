"""Host layout of the point tiles (p = 1 in 2D and 3D), built by dry-run plans."""
import pytest

import gen_inputs as gi


# Unbalanced 2D clouds whose tiles end at their 32nd reader, often inside a sibling
# group: such a tile's successor counts the rest of the group as its first, and stays
# within the 64 groups that a chain word can name.
# (seed, points, depth, components, sigma)
CLOUDS = [(243, 2555, 15, 3, 0.2), (17, 2000, 13, 4, 0.05), (18, 3750, 14, 4, 0.05)]


@pytest.mark.parametrize("tile", [0, 64, 128, 256])
@pytest.mark.parametrize("seed,n,maxd,ncomp,sigma", CLOUDS)
def test_unbalanced_clouds_build(dkt, tile, seed, n, maxd, ncomp, sigma):
    pts = dkt.Octs.from_array(gi.gauss_points(2, n, ncomp, sigma, seed, maxd), 2, maxd, dkt.CURVE_HILBERT)
    da = dkt.DA(dkt.construct_tree(pts, 1), 1)
    info = dkt.Plan(da, tile_leaves=tile, dry_run=True).info()
    assert info["readers_max"] == 32 and info["groups_mean"] > 1


# Default leaves per tile: 256, or 128 where readers end the tiles well before that.
@pytest.mark.parametrize("dim,maxd", [(2, 12), (3, 9)])
def test_default_tile_follows_the_readers(dkt, dim, maxd):
    def das(n, ncomp):
        pts = dkt.Octs.from_array(gi.gauss_points(dim, n, ncomp, 0.05, 7, maxd), dim, maxd, dkt.CURVE_HILBERT)
        return dkt.DA(dkt.balance_tree(pts, 1), 1), dkt.DA(dkt.construct_tree(pts, 1), 1)

    def info(da, tile=0):
        return dkt.Plan(da, tile_leaves=tile, dry_run=True).info()

    for n in (20, 200, 1500, 6000):
        for da in das(n, 4):
            wide = info(da, 256)
            poor = wide["leaves"] < 240 * (wide["tiles"] - 1)
            assert wide["tile_leaves"] == 256 and info(da)["tile_leaves"] == (128 if poor else 256)
    balanced, unbalanced = das(6000, 4)
    assert info(balanced)["tile_leaves"] == 256 and info(unbalanced)["tile_leaves"] == 128
