"""Stale-buffer replay of the point tiles (p = 1 in 2D and 3D) on meshes that reach
it in every tile size: unbalanced 2D and 3D point clouds, where most tiles end at
their 32nd reader, and a balanced 3D one.  Each case checks on the plan that it
has readers and carry terms.

A plan's matvec against the per-leaf kernels: a node sums at most a few hundred
products of O(1) factors, each rounded once, a carry slot at most a few hundred
more, so the relative L2 difference of two orders of summation stays under
1e3 * 2^-53 in FP64; FP32 is held to the 2e-6 of the other FP32 tests.  A batch of
plans with different tile sizes, whose launch has the work-items of the largest:
bitwise each plan's own matvec."""
import pytest

import gen_inputs as gi

MESHES = {
    "unbalanced2d": (2, 12, 3000, 9, False),
    "unbalanced3d": (3, 9, 1500, 7, False),
    "balanced3d": (3, 9, 1500, 7, True),
}
TILES = (64, 128, 256)


def _da(dkt, name):
    dim, maxd, n, seed, balanced = MESHES[name]
    pts = dkt.Octs.from_array(gi.gauss_points(dim, n, 4, 0.05, seed, maxd), dim, maxd, dkt.CURVE_HILBERT)
    return dkt.DA(dkt.balance_tree(pts, 1) if balanced else dkt.construct_tree(pts, 1), 1)


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


@pytest.mark.parametrize("name", sorted(MESHES))
def test_meshes_reach_the_replay(dkt, name):
    da = _da(dkt, name)
    for tile in TILES:
        info = dkt.Plan(da, tile_leaves=tile, dry_run=True).info()
        assert info["tiles"] > 16 and info["readers_max"] > 16 and info["carry_terms_max"] > 16


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(MESHES))
@pytest.mark.parametrize("tile", TILES)
def test_replay_matches_leaf_kernels(dkt, torch, name, tile):
    da = _da(dkt, name)
    gen = torch.Generator().manual_seed(3)
    for op in (dkt.OP_STIFFNESS, dkt.OP_MASS, dkt.OP_IDENTITY):
        simple, plan = dkt.Plan(da, op, simple=True), dkt.Plan(da, op, tile_leaves=tile)
        for nrhs in (1, 3):
            x = (torch.rand((da.n_nodes, nrhs) if nrhs > 1 else da.n_nodes, generator=gen, dtype=torch.float64) * 2 - 1).cuda()
            for masked in (0, 1, 2):
                want, got = torch.empty_like(x), torch.full_like(x, float("nan"))
                simple.matvec_torch(x, want, masked=masked)
                plan.matvec_torch(x, got, masked=masked)
                got32 = torch.full_like(x.float(), float("nan"))
                plan.matvec_torch(x.float(), got32, masked=masked)
                scale = float(want.norm())
                assert float((got - want).norm()) <= 1.2e-13 * scale, (op, nrhs, masked)
                assert float((got32.double() - want).norm()) <= 2e-6 * scale, (op, nrhs, masked)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("column_major", [False, True])
def test_batch_of_tile_sizes_equals_own_matvecs(dkt, torch, dtype, column_major):
    das = [_da(dkt, name) for name in sorted(MESHES)]
    plans = [dkt.Plan(da, tile_leaves=tile) for da in das for tile in TILES]
    gen = torch.Generator().manual_seed(8)
    for nrhs in (1, 3):
        xs = [(torch.rand((p.n_nodes, nrhs), generator=gen, dtype=torch.float64) * 2 - 1).to(getattr(torch, dtype)).cuda()
              for p in plans]
        refs = [torch.full_like(x, float("nan")) for x in xs]
        for p, x, r in zip(plans, xs, refs):
            p.matvec_torch(x, r, masked=1)
        if column_major:
            xs, refs = [x.t().contiguous() for x in xs], [r.t().contiguous() for r in refs]
        ys = [torch.full_like(x, float("nan")) for x in xs]
        dkt.Batch(plans, xs, ys, masked=1, column_major=column_major).run()
        torch.cuda.synchronize()
        for k, (y, r) in enumerate(zip(ys, refs)):
            assert torch.equal(y, r), (nrhs, k)
