"""Trees whose largest segment stays large for many levels (most particles in one small clump),
alone, in a forest of thousands of tiny boxes and under plans made for other positions: levels
by chunks and by a workgroup per segment, up to segments of more than 64 chunks in one."""
import numpy as np
import pytest

import ic
import photons_gpu as pg
from test_gpu_subtrees import check

pytestmark = pytest.mark.gpu


def clump(n, k, width, box, seed):
    """n particles, k of them in a Gaussian ball"""
    r = np.random.Generator(np.random.PCG64(seed))
    pos = r.random((n, 3))
    pos[:k] = 0.37 + width * r.normal(size=(k, 3))
    return np.ascontiguousarray(pos % 1.0 * box)


def box_of(n):
    return 500000.0 * (n / 256.0 ** 3) ** (1.0 / 3.0)


def fresh_force(prm, precision, pos):
    ctx = pg.Context(prm, precision)
    acc = ctx.force(pos)
    ctx.close()
    return acc


@pytest.mark.parametrize("n,k,width,maxleaf", [(24577, 24000, 1e-5, 32), (150001, 140000, 1e-4, 8), (200000, 180000, 1e-3, 32)])
def test_concentrated_tree_matches_oracle(n, k, width, maxleaf):
    pos = clump(n, k, width, box_of(n), n)
    check(pos, ic.force_params(n, box_of(n), 256, rc_factor=4.5, maxleaf=maxleaf))


@pytest.mark.parametrize("nsmall,nbig", [(2000, 200000), (5000, 2000003)])
def test_forest_of_tiny_boxes_and_a_concentrated_one(nsmall, nbig):
    counts = np.array([64] * (nsmall // 2) + [nbig] + [64] * (nsmall - nsmall // 2))
    lengths = box_of(counts.astype(np.float64))
    r = np.random.Generator(np.random.PCG64(nsmall))
    parts = [r.random((c, 3)) * L if c == 64 else clump(c, c * 7 // 10, 1e-3, L, nbig) for c, L in zip(counts, lengths)]
    prm = ic.force_params(nbig, box_of(nbig), 4 * round(nbig ** (1 / 3)), rc_factor=4.5, maxleaf=32, order=3, theta=0.6)
    ctx = pg.Context(prm, pg.FP64)
    off = np.concatenate([[0], np.cumsum(counts)])
    for again in range(2):  # ordinary, then planned
        print(f"{nsmall} boxes of 64 and one of {nbig}, evaluation {again}", flush=True)
        acc = ctx.force_boxes(counts, lengths, np.concatenate(parts))
        for b in (0, nsmall // 2, nsmall):
            alone = pg.Context(dict(prm.as_dict(), boxsize=float(lengths[b])), pg.FP64)
            assert np.array_equal(acc[off[b]:off[b + 1]], alone.force(parts[b])), b
            alone.close()
    ctx.close()


@pytest.mark.parametrize("n,before,after,margin", [
    (200000, (180000, 1e-3), (180000, 1e-3), 1.0),
    (600000, (12000, 1e-5), (540000, 1e-4), 16.0),  # a segment of 184,000 past the plan's levels by chunks
    (600000, (540000, 1e-4), (12000, 1e-5), 16.0)])
def test_plans_for_other_positions(n, before, after, margin):
    import torch
    box = box_of(n)
    # (a cutoff beyond all clumps, so that the lists of either set of positions fit the plan of the other)
    prm = ic.force_params(n, box, 16, rc_factor=4.5, maxleaf=32, order=3, theta=0.6)
    p0, p1 = clump(n, *before, box, 6), clump(n, *after, box, 7)
    want = [fresh_force(prm, pg.FP64, p) for p in (p0, p1)]
    d_pos = torch.from_numpy(p0).cuda()
    d_acc = torch.zeros_like(d_pos)
    ctx = pg.Context(prm, pg.FP64)
    ctx.graph_create(np.array([n]), np.array([box]), d_pos.data_ptr(), d_acc.data_ptr(), margin=margin)
    for k in (0, 1, 0, 1):
        print(f"replay {k}", flush=True)
        d_pos.copy_(torch.from_numpy(p1 if k else p0))
        d_acc.zero_()
        torch.cuda.synchronize()
        ctx.graph_launch()
        assert ctx.graph_check()[0] == 0
        assert np.array_equal(d_acc.cpu().numpy(), want[k]), k
    ctx.close()
