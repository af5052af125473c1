"""The p = 2 conforming kernel adds several ranks of an element to their points between
two barriers (RankPhases in plan_common.h).  That is free of conflicts only if no
two ranks of a phase, of the same or of two leaves, lie at one position: checked
here on balanced and unbalanced trees, with the table built as the kernel's is."""
import itertools

import numpy as np
import pytest

import gen_inputs as gi


def phases(dim):
    out = []
    for size in range(dim):
        for c in range(1 << (dim - size)):
            ranks = []
            for axes in itertools.combinations(range(dim), size):
                free = c
                rank = []
                for d in range(dim):
                    if d in axes:
                        rank.append(1)
                    else:
                        rank.append(2 * (free & 1))
                        free >>= 1
                ranks.append(tuple(rank))
            out.append(ranks)
    out[-1].append((1,) * dim)
    return out


@pytest.mark.parametrize("dim,balanced", [(2, True), (2, False), (3, True), (3, False)])
def test_no_two_ranks_of_a_phase_meet(dkt, dim, balanced):
    maxd = 30
    tree = dkt.Octs.from_array(gi.sphere_tree(dim, maxd, 2, 6 if dim == 2 else 5, (0.45, 0.5, 0.55), 0.28), dim, maxd,
                               dkt.CURVE_HILBERT)
    if balanced:
        tree = dkt.balance_tree(tree, 1)
    leaves = tree.array().astype(np.int64)
    half = np.int64(1) << (maxd - leaves[:, dim] - 1)
    table = phases(dim)
    assert sorted(r for ph in table for r in ph) == sorted(itertools.product(range(3), repeat=dim))
    for ph in table:
        pos = np.concatenate([leaves[:, :dim] + half[:, None] * np.array(r) for r in ph])
        assert len(np.unique(pos, axis=0)) == len(pos), ph
