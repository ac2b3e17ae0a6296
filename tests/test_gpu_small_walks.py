"""Walks from a given pair of cells at any depth, which end where nothing is passed down, against
the oracle's list of the same walk, and the forces of few and of many pairs by the drop-in
entry points, sliced lists and unsliced."""
import ctypes as C

import numpy as np
import pytest

import ic
import oracle
import photons_gpu as pg

pytestmark = pytest.mark.gpu


def dp(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


def walked(ctx, a, b, lo, hi, n):
    acc, n_p2p, n_m2l = np.zeros((n, 3)), C.c_int64(), C.c_int64()
    rc = pg.lib().photons_walk_eval(ctx.h, a, b, lo, hi, 1, 0, dp(acc), C.byref(n_p2p), C.byref(n_m2l))
    assert rc == 0, pg.lib().photons_last_error().decode()
    out = []
    for t, s, sh in (ctx.p2p_list(), ctx.m2l_list()):
        out.append(np.stack([t, s, sh.astype(np.int32)], axis=1))
    assert (n_p2p.value, n_m2l.value) == (len(out[0]), len(out[1]))
    return acc, out


@pytest.mark.parametrize("precision", [pg.FP64, pg.FP32_MIXED])
@pytest.mark.parametrize("n,maxleaf", [(4096, 32), (40000, 16)])
def test_walks_add_up(n, maxleaf, precision):
    """the walk of a node with itself emits what the walks of its children's four pairs emit:
    from the root down, along either child in turn, to a leaf"""
    box = 500000.0 * (n / 256.0 ** 3) ** (1.0 / 3.0)
    pos, _ = ic.clustered(n, box, seed=n)
    prm = ic.force_params(n, box, 16, rc_factor=4.5, maxleaf=maxleaf, order=3)
    ctx = pg.Context(prm, precision)
    ctx.prepare(pos)
    cells = ctx.cells()
    nl, son = cells["nleaf"], cells["son"]
    A = nl  # the root
    for depth in range(40):
        acc, lists = walked(ctx, A, A, 0, 1, n)
        parts = [(a, b) for a in son[A] for b in son[A]]
        some = [walked(ctx, int(a), int(b), 0, 1, n) for a, b in parts]
        total = sum(p[0] for p in some)
        scale = max(np.abs(acc).max(), 1e-300)
        assert np.abs(total - acc).max() <= (1e-13 if precision == pg.FP64 else 2e-5) * scale
        for k in range(2):
            want = np.concatenate([p[1][k] for p in some])
            key = lambda x: x[np.lexsort((x[:, 2], x[:, 1], x[:, 0]))]
            np.testing.assert_array_equal(key(lists[k]), key(want))
        print(f"depth {depth}: {len(lists[0])} P2P and {len(lists[1])} M2L entries", flush=True)
        A = int(son[A][depth % 2])
        if A < nl:
            break
    # a leaf with itself, and with its neighbour
    for b in (A, A - 1 if A > 0 else A + 1):
        acc, lists = walked(ctx, A, b, 0, 1, n)
        np.testing.assert_array_equal(lists[0], [[A, b, 0]])
        assert len(lists[1]) == 0
    ctx.close()


def test_root_walk_is_the_oracles():
    n = 40000
    box = 500000.0 * (n / 256.0 ** 3) ** (1.0 / 3.0)
    pos, _ = ic.clustered(n, box, seed=n)
    prm = ic.force_params(n, box, 16, rc_factor=4.5, maxleaf=16, order=3)
    t = oracle.Tree(pos, prm)
    ctx = pg.Context(prm, pg.FP64)
    ctx.prepare(pos)
    root = ctx.cells()["nleaf"]
    got = [walked(ctx, root, root, *s, n)[1] for s in ((0, 1), (1, 27))]
    for k, w in enumerate((t.p2p_list(), t.m2l_list())):
        want = np.stack([w[0], w[1], w[2].astype(np.int32)], axis=1)
        want = want[np.argsort(want[:, 0], kind="stable")]
        for g, home in zip((got[0][k], got[1][k]), (True, False)):
            np.testing.assert_array_equal(g, want[(want[:, 2] == 0) == home])
    ctx.close()
