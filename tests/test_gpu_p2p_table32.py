"""The single-precision P2P kernel that reads its pair factor from the table over r^2 (FP32-mixed
boxes from 900,000 particles on), against the oracle's direct sum: leaf sizes at the edges of
its lane layout (pairs of targets, chunks of 64) and of its slices, softenings on both sides of
the split radius, the smallest and the largest order, images across the box's faces.

The opening angle is so small and the cutoff so long that every pair within 16 rs is a
particle pair."""
import numpy as np
import pytest

import ic
import oracle
import photons_gpu as pg

pytestmark = pytest.mark.gpu

N = 900001
EPS = 2.0 ** -24


@pytest.mark.parametrize("maxleaf,soft_rs,order,mesh", [(2, 0.024, 4, 512), (3, 0.024, 3, 512), (33, 0.0025, 3, 128),
                                                        (32, 0.6, 5, 128), (65, 6.0, 4, 128), (129, 0.024, 5, 128),
                                                        (256, 0.024, 3, 128)])
def test_forces_match_the_direct_sum(maxleaf, soft_rs, order, mesh):
    box = 500000.0 * (N / 256.0 ** 3) ** (1.0 / 3.0)
    pos, _ = ic.clustered(N, box, seed=8)
    prm = ic.force_params(N, box, mesh, rc_factor=16.0, theta=0.01, maxleaf=maxleaf, order=order)
    prm.soft = soft_rs * prm.rs
    ctx = pg.Context(prm, pg.FP32_MIXED)
    print(f"leaves of {maxleaf}, softening {soft_rs} rs, p = {order}", flush=True)
    acc = ctx.force(pos)
    assert np.array_equal(acc, ctx.force(pos))  # ordinary, then planned
    cells, perm = ctx.cells(), ctx.perm(N)
    ctx.close()
    rng = np.random.default_rng(2)
    edge = np.flatnonzero((pos < 0.01 * box).any(axis=1) | (pos > 0.99 * box).any(axis=1))
    sample = np.concatenate([rng.choice(N, 24, replace=False), rng.choice(edge, 8, replace=False)]).astype(np.int32)
    want = oracle.direct(pos, prm, sample, 19.0 * prm.rs)
    nl = cells["nleaf"]
    slot = np.empty(N, np.int64)
    slot[perm] = np.arange(N)
    leaf = np.searchsorted(cells["ipart"][:nl] + cells["npart"][:nl], slot[sample], side="right")
    half = 0.5 * np.linalg.norm(cells["width"][:nl][leaf], axis=1)
    for i, s in enumerate(sample):
        d = pos - pos[s]
        d -= box * np.round(d / box)
        r = np.linalg.norm(d, axis=1)
        r = r[(r > 0) & (r < 16.0 * prm.rs)]
        u, q = r / (2 * prm.rs), np.maximum(r, prm.soft)
        # sizes of the pair forces; G(u) <= (1 + 2u) exp(-u^2)
        f = prm.mass * r * np.minimum((1 + 2 * u) * np.exp(-u * u), 1.0) / q ** 3
        # the factor's row (its bound in u: 3e-7 and the cubic's (u^2 / 256)^4 / 6), the
        # coordinates of both particles about the leaf's centre, rounded, which move a factor
        # by up to four times their relative error, and the sums' roundings
        per_pair = 4e-7 + (np.minimum(u, 9.5) ** 2 / 256) ** 4 / 6 + 8 * EPS * (r + 2 * half[i]) / q
        bound = (f * per_pair).sum() + 4 * EPS * (np.sqrt(len(r)) + 64) * f.sum()
        err = np.linalg.norm(acc[s] - want[i])
        assert err <= bound, (i, err, bound, np.linalg.norm(want[i]))


def test_forest_of_boxes_by_both_kernels():
    """boxes on both sides of the limit in one evaluation: each as alone, bit for bit"""
    import torch
    counts = np.array([3000, N, 899999, 40000, 70])
    lengths = 500000.0 * (counts / 256.0 ** 3) ** (1.0 / 3.0)
    r = np.random.Generator(np.random.PCG64(7))
    parts = [r.random((c, 3)) * L for c, L in zip(counts, lengths)]
    prm = ic.force_params(256 ** 3, 500000.0, 256, rc_factor=6.0, theta=0.5, order=3).as_dict()
    alone = []
    for p, L in zip(parts, lengths):
        ctx = pg.Context(dict(prm, boxsize=float(L)), pg.FP32_MIXED)
        alone.append(ctx.force(p))
        ctx.close()
    want = np.concatenate(alone)
    d_pos = torch.from_numpy(np.concatenate(parts)).cuda()
    d_acc = torch.zeros_like(d_pos)
    ctx = pg.Context(prm, pg.FP32_MIXED)
    for again in range(2):  # ordinary, then planned
        assert np.array_equal(ctx.force_boxes(counts, lengths, np.concatenate(parts)), want)
    ctx.graph_create(counts, lengths, d_pos.data_ptr(), d_acc.data_ptr())
    for rep in range(3):
        d_acc.zero_()
        torch.cuda.synchronize()
        ctx.graph_launch()
        assert ctx.graph_check()[0] == 0
        assert np.array_equal(d_acc.cpu().numpy(), want), rep
    ctx.close()
