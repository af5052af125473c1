"""p = 1 conforming plans at the limit of the point tiles' row levels (11).  A hanging
position may be the mean of positions that hang themselves one level up, and so
on: a cell beside an orthant that is refined towards their common face, along its
diagonal, reaches one level per axis of the face and per cell.  11 levels are the
most that point tiles take; 12 go to the conforming tile kernel, in every tile size.

Both against the per-leaf kernels: the weights of a row are products of halves and
exact, a node sums at most a few hundred products of O(1) factors, each rounded
once, so the relative L2 difference of two orders of summation stays under
1e3 * 2^-53 in FP64; FP32 is held to the 2e-6 of the other FP32 tests."""
import numpy as np
import pytest

MAXD = 16


def _cells(dim, depth, wide):
    """The low orthant refined to `depth` towards its upper face of the last axis (cells
    of level `wide` and finer only near the face's diagonal, in 2D near its low end), the
    others whole."""
    half = 1 << (MAXD - 1)
    leaves, todo = [], [(0,) * dim + (0,)]
    while todo:
        c = todo.pop()
        size, face = 1 << (MAXD - c[dim]), c[:dim - 1]
        near = c[dim] < wide or (c[0] <= 4 * size if dim == 2 else max(face) - min(face) <= size)
        if c[dim] == 0 or (c[dim] < depth and max(c[:dim]) < half and c[dim - 1] + size == half and near):
            todo += [tuple(c[d] + ((q >> d) & 1) * (size >> 1) for d in range(dim)) + (c[dim] + 1,)
                     for q in range(1 << dim)]
        else:
            leaves.append(c)
    return np.array(leaves, np.uint32)


# name: dim, depth, wide, whether point tiles take it
MESHES = {
    "11levels2d": (2, 12, 2, True),
    "12levels2d": (2, 13, 2, False),
    "10levels3d": (3, 6, 2, True),
    "12levels3d": (3, 7, 2, False),
    "9levels4d": (4, 4, 4, True),
    "12levels4d": (4, 5, 4, False),
}


def _da(dkt, name):
    dim, depth, wide, _ = MESHES[name]
    return dkt.DA(dkt.sort_tree(dkt.Octs.from_array(_cells(dim, depth, wide), dim, MAXD, dkt.CURVE_HILBERT)), 1)


def _matrices(dim):
    """Element matrices of every level, symmetric and of O(1), no two alike."""
    m = np.random.default_rng(dim).uniform(-1, 1, (MAXD + 1, 1 << dim, 1 << dim))
    return m + m.transpose(0, 2, 1)


@pytest.mark.parametrize("tile", [0, 64, 128, 256])
@pytest.mark.parametrize("name", sorted(MESHES))
def test_route(dkt, name, tile):
    info = dkt.Plan(_da(dkt, name), conforming=True, tile_leaves=tile, dry_run=True).info()
    assert (info["tile_nodes_mean"] > 0) == MESHES[name][3]  # point tiles report their mean
    assert info["tile_leaves"] == (tile or 256)


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [0, 64])
@pytest.mark.parametrize("name", sorted(MESHES))
def test_matches_leaf_kernels(dkt, torch, name, tile):
    da = _da(dkt, name)
    gen = torch.Generator().manual_seed(3)
    for op in (dkt.OP_STIFFNESS, dkt.OP_MASS, dkt.OP_IDENTITY, dkt.OP_CAPTURED):
        mats = _matrices(MESHES[name][0]) if op == dkt.OP_CAPTURED else None
        simple = dkt.Plan(da, op, mats, simple=True, conforming=True)
        plan = dkt.Plan(da, op, mats, conforming=True, tile_leaves=tile)
        for nrhs in (1, 3, 9):
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
def test_batch_of_both_routes_equals_own_matvecs(dkt, torch, dtype):
    plans = []
    for name in sorted(MESHES):
        da = _da(dkt, name)
        plans += [dkt.Plan(da, conforming=True), dkt.Plan(da, dkt.OP_CAPTURED, _matrices(MESHES[name][0]), conforming=True)]
    gen = torch.Generator().manual_seed(5)
    for nrhs in (1, 3):
        xs = [(torch.rand((p.n_nodes, nrhs), generator=gen, dtype=torch.float64) * 2 - 1).to(getattr(torch, dtype)).cuda()
              for p in plans]
        refs = [torch.full_like(x, float("nan")) for x in xs]
        ys = [torch.full_like(x, float("nan")) for x in xs]
        for p, x, r in zip(plans, xs, refs):
            p.matvec_torch(x, r, masked=1)
        dkt.Batch(plans, xs, ys, masked=1).run()
        torch.cuda.synchronize()
        for k, (y, r) in enumerate(zip(ys, refs)):
            assert torch.equal(y, r), (nrhs, k)
