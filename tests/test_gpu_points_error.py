"""FP32 matvecs over point tiles are as accurate as with every leaf interpolating for
itself, although a leaf's own part is subtracted again from one node.

Mass on the level-7 sphere (55,639 nodes), inputs uniform in [1, 2), where every sum
that the subtraction enters has one sign, against the FP64 per-leaf kernels on the
same inputs.  With per-leaf interpolation in the same kernel the relative L2 error
averaged 4.99e-8 over 16 inputs (4.57e-8 to 5.35e-8); with the point tiles' node sums
in FP32 it was 5.24e-8.  The bound is the former."""
import pytest

pytestmark = pytest.mark.gpu


def test_fp32_error_of_point_tiles(dkt):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    da = dkt.DA(dkt.balance_tree(dkt.sphere_tree(3, 30, 3, 7, (0.5, 0.5, 0.5), 0.3), 1), 1)
    exact, plan = dkt.Plan(da, dkt.OP_MASS, simple=True), dkt.Plan(da, dkt.OP_MASS)
    gen = torch.Generator().manual_seed(11)
    errors = []
    for _ in range(16):
        x = (torch.rand(da.n_nodes, generator=gen, dtype=torch.float64) + 1).float().cuda()
        y, want = torch.empty_like(x), torch.empty(da.n_nodes, dtype=torch.float64, device="cuda")
        plan.matvec_torch(x, y)
        exact.matvec_torch(x.double(), want)
        errors.append(float((y.double() - want).norm() / want.norm()))
    assert sum(errors) / len(errors) <= 4.99e-8, errors
