"""Infinite and NaN voxels stay on the rays that pass through them, as the per-lane kernels find them: forward
projections of pairs of opposite rays whose ends belong to one of the two only (even sizes), and of cells whose
second row or column has weight 0 (rays along the axes, the grid's border)."""

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


# one slice per lane, paired and not, clipped and not
@pytest.mark.parametrize("nz", [32, 40, 56, 63, 64])
@pytest.mark.parametrize("n, span", [(20, 360.0), (21, 360.0), (24, 180.0)])
@pytest.mark.parametrize("mu", [0.0, 0.01])
@pytest.mark.parametrize("positive", [False, True])
def test_wavefronts(gpu, n, nz, span, mu, positive):
    """Rays that meet no such voxel project to what the per-lane kernel projects them to, also where the range
    of the slice clips the samples (which turns a NaN into the range's end), alone and in a batch."""
    import torch
    from vamtoolbox_amd.batch import ParallelBatch
    from vamtoolbox_amd.parallel import ParallelPlan
    print(n, nz, span, mu, positive, flush=True)
    _compare(gpu, n, nz, 24, span, mu=mu, warp_clip=False)
    ang = np.linspace(0.0, span, 24, endpoint=False)
    plan, other, lane, linear = [ParallelPlan(m, nz, ang, mu=mu, device=gpu, warp_clip=c, per_lane_geometry=p)
                                 for m, c, p in ((n, True, False), (n + 1, True, False), (n, True, True), (n, False, True))]
    vol = torch.rand(n, n, nz, device=gpu) + (0.5 if positive else -0.5)
    vol[n // 3, 0, nz // 2] = vol[0, n // 2, 3] = float("inf")
    vol[n // 2, n - 1, 5] = float("nan")
    beside = torch.isfinite(linear.forward(vol))
    want = lane.forward(vol)
    one = plan.forward(vol)
    flat = ParallelBatch([plan, other]).forward(torch.cat([vol.reshape(-1), torch.ones((n + 1) ** 2 * nz, device=gpu)]))
    for got in (one, flat[: one.numel()].view(one.shape)):
        torch.testing.assert_close(got[beside], want[beside], rtol=1e-5, atol=1e-5)
    assert not bool(beside.all())
