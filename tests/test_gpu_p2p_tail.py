"""Pairs beyond the end of the FP64 table over r^2 (u = r / 2 rs = 8.7 at most), whose factor is evaluated: relatively as exact
as erfc and exp are there, for softenings below and above the separation."""
import numpy as np
import pytest

import oracle
import photons_gpu as pg
from cases import case_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("soft_u", [0.012, 0.0156, 30.0])  # the second's octaves end at u = 11.3
@pytest.mark.parametrize("u", [8.75, 9.0, 11.2, 12.1, 17.0, 24.0])
def test_two_particles(u, soft_u):
    _, prm = case_inputs("clus16_pm32")
    p = prm.as_dict()
    p["periodic"] = 0
    d = u * 2 * p["rs"] / np.sqrt(3.0)
    p["boxsize"] = 2.5 * d
    p["rc"] = 10 * p["boxsize"]
    p["soft"] = soft_u * 2 * p["rs"]
    pos = np.array([[0.3 * d, 0.3 * d, 0.3 * d], [1.3 * d, 1.3 * d, 1.3 * d]])
    ref, _ = oracle.force(pos, p)
    acc = pg.Context(p, pg.FP64).force(pos)
    assert np.abs(ref).min() > 0.0
    # the erfcx fit's bound, and the rounding of u^2 in exp(-u^2) on both sides
    assert np.abs(acc - ref).max() <= (5e-14 + 8 * u * u * 2.0 ** -53) * np.abs(ref).max()
