"""Several right-hand sides through the tile kernels (4D and p = 2 traversal,
p = 2 conforming): a column's workgroups do the work of the single-column
matvec in the same order, so every column equals it to the last bit, over
column counts below, at and past what one launch holds."""
import pytest

import gen_inputs as gi

pytestmark = pytest.mark.gpu

MESHES = {
    "cloud4d": (4, 9, 1, lambda: gi.gauss_points(4, 600, 3, 0.05, 5, 9)),
    "sphere2d_p2": (2, 30, 2, lambda: gi.sphere_tree(2, 30, 2, 7, (0.45, 0.5, 0.55), 0.28)),
    "sphere3d_p2": (3, 30, 2, lambda: gi.sphere_tree(3, 30, 2, 4, (0.45, 0.5, 0.55), 0.28)),
}


@pytest.mark.parametrize("name", sorted(MESHES))
@pytest.mark.parametrize("conforming", [False, True])
@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_columns_equal_single_matvecs(dkt, name, conforming, dtype):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    dim, maxd, order, cells = MESHES[name]
    da = dkt.DA(dkt.balance_tree(dkt.Octs.from_array(cells(), dim, maxd, dkt.CURVE_HILBERT), 1), order)
    plan = dkt.Plan(da, dkt.OP_STIFFNESS, conforming=conforming)
    gen = torch.Generator().manual_seed(4)
    for nrhs in (2, 7, 8, 9, 19):
        x = (torch.rand((da.n_nodes, nrhs), generator=gen, dtype=torch.float64) * 2 - 1).to(getattr(torch, dtype)).cuda()
        for masked in (0, 1, 2):
            y = torch.full_like(x, float("nan"))
            plan.matvec_torch(x, y, masked=masked)
            for q in range(nrhs):
                xq = x[:, q].contiguous()
                yq = torch.full_like(xq, float("nan"))
                plan.matvec_torch(xq, yq, masked=masked)
                assert torch.equal(y[:, q], yq), (nrhs, masked, q)
