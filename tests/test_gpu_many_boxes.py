"""Forests of thousands of small boxes, whose trees go level by level, on both sides of the rule
(more than 2048 boxes of at most 16 leaves' worth of particles): the same forces bit for bit
as of the same boxes by subtrees and alone; odd box counts for the numbering of the roots."""
import numpy as np
import pytest

import ic
import photons_gpu as pg

pytestmark = pytest.mark.gpu


def boxes(nb, n, seed):
    """nb boxes of about n particles"""
    r = np.random.Generator(np.random.PCG64(seed))
    counts = np.where(np.arange(nb) % 7 == 3, n - n // 3, n)
    lengths = 500000.0 * (counts / 256.0 ** 3) ** (1.0 / 3.0)
    return counts, lengths, np.repeat(lengths, counts)[:, None] * r.random((int(counts.sum()), 3))


@pytest.mark.parametrize("precision", [pg.FP64, pg.FP32_MIXED])
@pytest.mark.parametrize("nb,n,maxleaf", [(2049, 40, 16), (2049, 128, 8), (2049, 129, 8), (5003, 64, 32), (3001, 500, 32)])
def test_same_forces_by_levels_and_by_subtrees(nb, n, maxleaf, precision):
    counts, lengths, pos = boxes(nb, n, nb + n)
    off = np.concatenate([[0], np.cumsum(counts)])
    prm = ic.force_params(n, float(lengths[0]), max(8, 2 * round(n ** (1 / 3) / 2)), rc_factor=4.5, maxleaf=maxleaf,
                          order=3)
    ctx = pg.Context(prm, precision)
    got = [ctx.force_boxes(counts, lengths, pos) for again in range(2)]  # ordinary, then planned
    assert np.array_equal(got[0], got[1])
    few = 2048  # by subtrees
    for b0 in range(0, nb, few):
        b1 = min(b0 + few, nb)
        print(f"boxes {b0} .. {b1} of {nb}", flush=True)
        part = ctx.force_boxes(counts[b0:b1], lengths[b0:b1], pos[off[b0]:off[b1]])
        assert np.array_equal(part, got[0][off[b0]:off[b1]])
    ctx.close()
    for b in (0, 3, nb - 1):
        alone = pg.Context(dict(prm.as_dict(), boxsize=float(lengths[b])), precision)
        assert np.array_equal(alone.force(pos[off[b]:off[b + 1]]), got[0][off[b]:off[b + 1]])
        alone.close()


def test_replayed_forest_by_levels():
    import torch
    counts, lengths, pos = boxes(3000, 100, 1)
    prm = ic.force_params(100, float(lengths[0]), 8, rc_factor=4.5, maxleaf=32, order=3)
    want = pg.Context(prm, pg.FP64).force_boxes(counts, lengths, pos)
    d_pos = torch.from_numpy(pos).cuda()
    d_acc = torch.zeros_like(d_pos)
    ctx = pg.Context(prm, pg.FP64)
    ctx.graph_create(counts, lengths, d_pos.data_ptr(), d_acc.data_ptr())
    for rep in range(3):
        d_acc.zero_()
        torch.cuda.synchronize()
        ctx.graph_launch()
        assert ctx.graph_check()[0] == 0
        assert np.array_equal(d_acc.cpu().numpy(), want), rep
    ctx.close()
