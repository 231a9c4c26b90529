"""Infinite and NaN voxels stay on the rays that pass through them, as the per-lane kernels find them: forward
projections of pairs of opposite rays whose ends belong to one of the two only (even sizes)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _compare(gpu, n, nz, na, span=360.0, **kw):
    import torch
    from vamtoolbox_amd.parallel import ParallelPlan
    print(n, nz, na, span, kw, flush=True)
    ang = np.linspace(0.0, span, na, endpoint=False)
    plans = [ParallelPlan(n, nz, ang, device=gpu, per_lane_geometry=p, **kw) for p in (False, True)]
    vol = torch.rand(n, n, nz, device=gpu) - 0.25
    for row, col, z, x in ((0, n // 3, 0, np.inf), (n - 1, n // 2, nz // 2, -np.inf), (n // 2, 0, nz - 1, np.nan),
                           (n // 3, n - 1, nz // 3, np.inf), (n // 2, n // 2, nz // 4, np.nan)):
        vol[row, col, z] = float(x)
    got, ref = [torch.isfinite(p.forward(vol)) for p in plans]
    assert bool((got | ~ref).all()) and not bool(got.all())


# pairs in lane groups, in whole wavefronts and as eight rays side by side
@pytest.mark.parametrize("n, nz, na", [(70, 6, 120), (64, 24, 160), (80, 1, 120), (300, 1, 300)])
@pytest.mark.parametrize("mu", [0.0, 0.01])
def test_thin(gpu, n, nz, na, mu):
    _compare(gpu, n, nz, na, mu=mu, warp_clip=False)
