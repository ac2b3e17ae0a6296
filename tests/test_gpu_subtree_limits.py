"""Subtrees that do not fit: more nodes than a workgroup holds (the tree is then built level
by level), and more cells than a plan holds in hundreds of subtrees of one launch, whose
workgroups start before, while and after the first ones report it."""
import numpy as np
import pytest

import ic
import oracle
import photons_gpu as pg

pytestmark = pytest.mark.gpu

SUBTREE, SUBTREE_NODES = 1024, 512  # particles and nodes that one workgroup takes (leaves of 8 and more)
BOX = 2.0 ** 17


def points(n, copies, share, seed):
    """n points, `share` of them in groups of `copies` at one place (a split takes one of them
    off at a time), on a grid so that every mean is exact and the tree the oracle's"""
    r = np.random.Generator(np.random.PCG64(seed))
    k = int(n * share) // copies if copies else 0
    pos = np.concatenate([np.repeat(r.random((k, 3)), copies, 0), r.random((n - k * copies, 3))])
    return np.ascontiguousarray(np.floor(pos * 2 ** 20) * (BOX / 2 ** 20))


def largest_subtree(pos, prm):
    """the most nodes under a segment of at most SUBTREE particles, in the oracle's tree"""
    ex = oracle.Tree(pos, prm).export()
    son, size = ex["node_son"], ex["node_npart"]
    nodes = np.ones(len(son), np.int64)
    for v in range(len(son) - 1, -1, -1):  # pre-order: children have larger numbers
        nodes[v] += sum(nodes[c] for c in son[v] if c >= 0)
    return int(nodes[size <= SUBTREE].max())


def test_subtree_of_too_many_nodes():
    pos = points(60000, 60, 0.8, 3)
    prm = ic.force_params(len(pos), BOX, 128, rc_factor=4.5, maxleaf=8)
    assert largest_subtree(pos, prm) > SUBTREE_NODES
    ex = oracle.Tree(pos, prm).export()
    nl, leaf = len(ex["leaf_npart"]), np.repeat(np.arange(len(ex["leaf_npart"])), ex["leaf_npart"])

    def by_leaf(perm):  # the positions in every leaf (of particles at one place any may be in it)
        p = pos[perm]
        return p[np.lexsort((p[:, 2], p[:, 1], p[:, 0], leaf))]

    ctx = pg.Context(prm, pg.FP64)
    for again in range(2):  # ordinary, then planned
        ctx.force(pos)
        cells = ctx.cells()
        assert cells["nleaf"] == nl
        np.testing.assert_array_equal(cells["npart"], np.concatenate([ex["leaf_npart"], ex["node_npart"]]))
        np.testing.assert_array_equal(cells["ipart"][:nl], ex["leaf_ipart"])
        np.testing.assert_array_equal(cells["son"][nl:], np.where(ex["node_son"] < 0, -ex["node_son"] - 1,
                                                                  ex["node_son"] + nl))
        np.testing.assert_array_equal(by_leaf(ctx.perm(len(pos))), by_leaf(ex["perm"]))


@pytest.mark.parametrize("precision", [pg.FP64, pg.FP32_MIXED])
def test_subtrees_that_outgrow_the_plan(precision):
    """the same top of the tree, twice the cells below it: reported by a replayed graph, whose
    next replay is whole again, and measured anew by ordinary evaluations"""
    import torch
    n = 600000
    few, many = points(n, 0, 0.0, 11), points(n, 40, 0.25, 12)
    prm = ic.force_params(n, BOX, 256, rc_factor=4.5, maxleaf=8)
    want = []
    for pos in (few, many):
        fresh = pg.Context(prm, precision)
        want.append(fresh.force(pos))
        fresh.close()
    d_pos = torch.from_numpy(few).cuda()
    d_acc = torch.zeros_like(d_pos)
    ctx = pg.Context(prm, precision)
    ctx.graph_create(np.array([n]), np.array([BOX]), d_pos.data_ptr(), d_acc.data_ptr(), margin=0.0)
    for pos, k in ((many, 1), (few, 0), (many, 1), (few, 0)):
        print(f"precision {precision}: replay with cells of {'many' if k else 'few'}", flush=True)
        d_pos.copy_(torch.from_numpy(pos))
        torch.cuda.synchronize()
        ctx.graph_launch()
        ovf, _ = ctx.graph_check()
        assert (ovf != 0) == (k == 1)
        if k == 0:
            assert np.array_equal(d_acc.cpu().numpy(), want[0])
    ctx.close()
    ctx = pg.Context(prm, precision)
    for pos, k in ((few, 0), (few, 0), (many, 1), (many, 1), (few, 0)):
        assert np.array_equal(ctx.force(pos), want[k])
    ctx.close()
