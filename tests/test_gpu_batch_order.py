"""Graph replays of a batch whose groups differ in work: the heaviest group's
launch is recorded first, each group on a branch, and large FP32 batches stay on
one stream.  Whichever group is the heaviest, and on both sides of that line (1e8
leaf ranks), every replay is bitwise each plan's own matvec."""
import pytest

pytestmark = pytest.mark.gpu


def _da(dkt, dim, p, level):
    return dkt.DA(dkt.balance_tree(dkt.sphere_tree(dim, 30, 2, level, (0.5,) * dim, 0.3), 1), p)


# (dim, p, level) per plan, columns, leaf ranks above the line
BATCHES = {
    "p1_heaviest": ([(3, 1, 6), (3, 2, 3), (2, 1, 4)], 2, False),
    "p2_heaviest": ([(3, 1, 3), (3, 2, 5), (2, 1, 4)], 2, False),
    "2d_heaviest": ([(3, 1, 3), (3, 2, 2), (2, 1, 9)], 2, False),
    "one_stream": ([(3, 2, 7), (3, 1, 5)], 64, True),
}


@pytest.mark.parametrize("name", sorted(BATCHES))
def test_replays_equal_own_matvecs(dkt, name):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    specs, nrhs, large = BATCHES[name]
    das = [_da(dkt, *s) for s in specs]
    assert (sum(d.n_elements * d.npe for d in das) * nrhs > 1e8) == large
    plans = [dkt.Plan(da) for da in das]
    gen = torch.Generator(device="cuda").manual_seed(6)
    xs = [torch.rand((da.n_nodes, nrhs), generator=gen, device="cuda", dtype=torch.float32) for da in das]
    ys = [torch.empty_like(x) for x in xs]
    s = torch.cuda.Stream()
    b = dkt.Batch(plans, xs, ys, graph=True)
    for rep in range(3):
        for x in xs:
            x.mul_(-0.5)
        refs = [torch.empty_like(x) for x in xs]
        for p, x, r in zip(plans, xs, refs):
            p.matvec_torch(x, r)
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            for y in ys:
                y.fill_(float("nan"))
            b.run(s.cuda_stream)
        s.synchronize()
        for y, r in zip(ys, refs):
            assert torch.equal(y, r), rep
