"""A static evaluation with another softening or split radius than the context's ordinary
ones before and after it: each gives what a fresh context gives, bit for bit."""
import ctypes as C

import numpy as np
import pytest

import ic
import photons_gpu as pg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [pg.FP64, pg.FP32_MIXED])
@pytest.mark.parametrize("change", [{"soft": 3.0}, {"rs": 0.7}, {"soft": 1e-9}])  # times the context's own
def test_static_evaluation_between_ordinary_ones(precision, change):
    import torch
    n = 20 ** 3
    box = 500000.0 * (n / 256.0 ** 3) ** (1.0 / 3.0)
    pos, _ = ic.clustered(n, box, seed=6)
    a = ic.force_params(n, box, 20, rc_factor=6.0, order=4).as_dict()
    b = dict(a)
    for key, factor in change.items():
        b[key] *= factor
    want = []
    for p in (a, b):
        fresh = pg.Context(p, precision)
        want.append(fresh.force(pos))
        fresh.close()
    assert not np.array_equal(want[0], want[1])
    d_pos = torch.from_numpy(np.ascontiguousarray(pos)).cuda()
    d_acc = torch.zeros_like(d_pos)
    ctx = pg.Context(a, precision)
    for again in range(3):
        ctx.set_params(a, precision)
        assert np.array_equal(ctx.force(pos), want[0]), again
        ctx.set_params(b, precision)
        rc = pg.lib().photons_force_device_static(ctx.h, n, C.c_void_p(d_pos.data_ptr()), C.c_void_p(d_acc.data_ptr()))
        assert rc == 0, pg.lib().photons_last_error().decode()
        assert np.array_equal(d_acc.cpu().numpy(), want[1]), again
    assert np.array_equal(ctx.force(pos), want[1])
    ctx.close()
