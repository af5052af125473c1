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
