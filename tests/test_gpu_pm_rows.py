"""The deposit by rows where most rows of mesh points hold nothing: particles in one cell, in a
ball, on a line and in a few cells far apart (gaps of some rows and of most of the mesh),
against the numpy oracle."""
import numpy as np
import pytest

import photons_gpu as pg
import pm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nside", [34, 64])
@pytest.mark.parametrize("kind", ["first", "last", "ball", "line", "few"])
def test_matches_the_oracle(kind, nside):
    n, L = 100001, 1000.0
    r = np.random.Generator(np.random.PCG64(nside))
    u = r.random((n, 3))
    h = 1.0 / nside
    if kind == "first":  # clouds of the mesh's first corner alone: the empty rows come after
        u = 0.5 * h + u * 0.9 * h
    elif kind == "last":  # of its last one, across the box's corner
        u = (u * 0.4 + 0.05) * h
    elif kind == "ball":
        u = 0.37 + 0.1 * (u - 0.5)
    elif kind == "line":
        u[:, :2] = 0.41 + 0.2 * h * u[:, :2]
    else:  # rows 0, 3, 4, 9, 68, 69, 133 and one far on
        rows = np.array([0, 3, 4, 9, 68, 69, 133, nside * nside - 2 * nside])
        row = rows[r.integers(0, len(rows), n)]
        u[:, 0] = (row // nside + 0.5 + 0.1 * u[:, 0]) * h
        u[:, 1] = (row % nside + 0.5 + 0.1 * u[:, 1]) * h
    pos = np.ascontiguousarray(u % 1.0 * L)
    rs, mass = 1.25 * L / nside, 3.5
    want = pm.pm_force(pos, mass, nside, L, rs)
    p = pg.PM(nside, L, rs, mass)
    for again in range(2):  # a mesh that has been used
        got = p.force(pos)
        # the sums of n terms of one sign, and their transform: some n^(1/2) + log N roundings
        # of the potential, a gradient of which is formed
        phi = np.abs(want).max() * L / (2 * np.pi)
        assert np.abs(got - want).max() <= 1e-15 * (np.sqrt(n) + 100) * nside / L * phi * 10
    p.close()
