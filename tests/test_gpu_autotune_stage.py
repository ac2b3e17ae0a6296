"""The autotuner times the staging size only where a box takes the kernel that has one."""
import numpy as np
import pytest

import ic
import photons_gpu as pg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,soft_rs,staged", [(900001, 0.024, False), (900001, 1e-9, True), (30000, 0.024, True)])
def test_staging_sizes_timed(n, soft_rs, staged):
    import torch
    box = 500000.0 * (n / 256.0 ** 3) ** (1.0 / 3.0)
    r = np.random.Generator(np.random.PCG64(4))
    d_pos = torch.from_numpy(r.random((n, 3)) * box).cuda()
    d_acc = torch.zeros_like(d_pos)
    prm = ic.force_params(n, box, 64, rc_factor=4.5, theta=0.6, order=3)
    prm.soft = soft_rs * prm.rs
    for stage in (256, 512):
        ctx = pg.Context(prm, pg.FP32_MIXED)
        ctx.set_p2p_stage(stage)
        leaf, best, table = ctx.autotune_boxes([n], [box], d_pos.data_ptr(), d_acc.data_ptr())
        assert set(table) == {(m, s) for m in (16, 32, 64) for s in ((256, 512) if staged else (stage,))}
        assert table[leaf, best] == min(table.values())
        ctx.close()
