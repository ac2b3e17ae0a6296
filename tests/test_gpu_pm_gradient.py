"""The PM gradient is formed of differences of the potential: on a uniform lattice, whose potential
is one value everywhere, the force vanishes.  With the potential itself in the products it is
0.5 roundings of the potential per mesh width."""
import numpy as np
import pytest

import photons_gpu as pg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nside", [16, 32, 64])  # powers of two: the transforms keep the one value
def test_force_of_a_uniform_lattice(nside):
    L, mass = 1000.0, 3.5
    cell = np.stack(np.meshgrid(*[np.arange(nside)] * 3, indexing="ij"), -1).reshape(-1, 3)
    pos = np.ascontiguousarray((cell + np.array([0.137, 0.731, 0.589])) * (L / nside))
    p = pg.PM(nside, L, 1.25 * L / nside, mass)
    phi = nside ** 3 * mass / (np.pi * L)  # the zeroth mode's factor L^2 / (pi N^3) times the density
    for again in range(2):
        acc = p.force(pos)
        assert np.sqrt((acc ** 2).mean()) <= 0.05 * 2.0 ** -53 * phi * nside / L
    p.close()
