"""Point tiles (p = 1 in 2D and 3D) against the per-leaf kernels, which take the
traversal as it is, over what the tiled layout can get wrong: meshes of one and
a few leaves, uniform ones (no hanging points), spheres (points shared between
parents and several row levels) and point clouds (stale-buffer readers), every
tile size, masking mode, operator and precision, one column, several and more
than one launch holds.

Tolerances: a node sums at most a few hundred products of O(1) factors, each
rounded once, so the relative L2 difference of two orders of summation stays
under 1e3 * 2^-53 in FP64; FP32 is held to the 2e-6 of the other FP32 tests."""
import numpy as np
import pytest

import gen_inputs as gi

pytestmark = pytest.mark.gpu

MESHES = {
    "one2d": (2, 10, lambda: np.array([[0, 0, 0]], np.uint32)),
    "uniform2d": (2, 10, lambda: np.array([[x << 6, y << 6, 4] for y in range(16) for x in range(16)], np.uint32)),
    "cloud2d": (2, 10, lambda: gi.gauss_points(2, 900, 3, 0.05, 5, 10)),
    "one3d": (3, 10, lambda: np.array([[0, 0, 0, 0]], np.uint32)),
    "cloud3d": (3, 9, lambda: gi.gauss_points(3, 1500, 4, 0.05, 7, 9)),
    "sphere3d": (3, 30, lambda: gi.sphere_tree(3, 30, 2, 5, (0.45, 0.5, 0.55), 0.28)),
}


@pytest.mark.parametrize("name", sorted(MESHES))
@pytest.mark.parametrize("tile", [0, 64, 128])
def test_point_tiles_match_leaf_kernels(dkt, name, tile):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    dim, maxd, cells = MESHES[name]
    da = dkt.DA(dkt.balance_tree(dkt.Octs.from_array(cells(), dim, maxd, dkt.CURVE_HILBERT), 1), 1)
    gen = torch.Generator().manual_seed(3)
    for op in (dkt.OP_STIFFNESS, dkt.OP_MASS, dkt.OP_IDENTITY):
        simple = dkt.Plan(da, op, simple=True)
        plan = dkt.Plan(da, op, tile_leaves=tile)
        for nrhs in (1, 3, 11):
            x = (torch.rand((da.n_nodes, nrhs) if nrhs > 1 else da.n_nodes, generator=gen, dtype=torch.float64) * 2 - 1).cuda()
            for masked in (0, 1, 2):
                want, got = torch.empty_like(x), torch.full_like(x, float("nan"))
                simple.matvec_torch(x, want, masked=masked)
                plan.matvec_torch(x, got, masked=masked)
                x32 = x.float()
                got32 = torch.full_like(x32, float("nan"))
                plan.matvec_torch(x32, got32, masked=masked)
                scale = float(want.norm())
                assert float((got - want).norm()) <= 1.2e-13 * scale, (op, nrhs, masked)
                assert float((got32.double() - want).norm()) <= 2e-6 * scale, (op, nrhs, masked)
