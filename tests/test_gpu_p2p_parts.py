"""The space that the P2P slices' parts take: none without the pair table (no slices of a box
this large), at most 2^24 parts of 24 bytes with it, whatever the leaf size."""
import numpy as np
import pytest

import ic
import photons_gpu as pg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("maxleaf", [64, 256])
def test_parts_are_bounded(maxleaf):
    import torch
    n = 160 ** 3
    box = 500000.0 * (n / 256.0 ** 3) ** (1.0 / 3.0)
    r = np.random.Generator(np.random.PCG64(4))
    pos = r.random((n, 3)) * box
    base = ic.force_params(n, box, 160, rc_factor=4.5, theta=0.6, maxleaf=maxleaf, order=3).as_dict()
    held = []
    for soft in (1e-9 * base["rs"], base["soft"]):  # the first is not covered by the table
        ctx = pg.Context(dict(base, soft=soft), pg.FP64)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        ctx.set_plan_reuse(False)
        ctx.force(pos)
        held.append(free - torch.cuda.mem_get_info()[0])
        ctx.close()
    print(f"leaves of {maxleaf}: {held[0] / n:.0f} and {held[1] / n:.0f} bytes a particle", flush=True)
    # (buffers are allocated an eighth larger; allocations are in pages of 2 MiB)
    assert held[1] - held[0] <= 2 ** 24 * 24 * 1.125 + 2 ** 23
