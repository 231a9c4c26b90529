"""The back projection's layout of slices over lanes follows the size of the problem and of its batch; every
layout sums a column in the same order, so any limit on the slices per lane, any batch and any alignment give
bitwise the same dose."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# below, at and above the least numbers of wavefronts of two, three and four slices per lane
@pytest.mark.parametrize("n", [24, 100, 116, 132])
@pytest.mark.parametrize("nz", [64, 129, 200, 255, 300, 384])
@pytest.mark.parametrize("mu", [0.01, 0.0])
def test_every_layout_gives_the_same_dose(gpu, n, nz, mu):
    import torch
    from vamtoolbox_amd.batch import ParallelBatch
    from vamtoolbox_amd.parallel import ParallelPlan
    print(n, nz, mu, flush=True)
    ang = np.arange(0.0, 360.0, 20.0)
    plans = [ParallelPlan(n, nz, ang, mu=mu, device=gpu) for _ in range(6)]
    plan = plans[0]
    s = torch.rand(plan.sino_shape, device=gpu)
    shifted = torch.cat([torch.zeros(1, device=gpu), s.reshape(-1)])[1:].view(s.shape)
    plan.set_tuning(bp_zv=1)
    want = plan.backward(s)
    for zv in (2, 4):
        plan.set_tuning(bp_zv=zv)
        assert torch.equal(plan.backward(s), want) and torch.equal(plan.backward(shifted), want)
    flat = ParallelBatch(plans).backward(s.reshape(-1).repeat(6))
    assert torch.equal(flat.view(6, *want.shape), want.expand(6, *want.shape))
