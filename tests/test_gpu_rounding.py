"""The wavefront kernels' sums are no further from float64 than the per-lane kernels', which round the running
sum once per sample (forward) and once per angle (back).

On inputs of one sign the running sum's rounding is nearly all of the error.  It is rounded at most as often,
so the error is at most the per-lane kernels' up to the scatter of a relative L2 norm over more than 10^4
values (under 2 %) and the value's own few roundings at the size of one sample (under 1 %): 1.05."""

import numpy as np
import pytest

from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu

# thin back projections with and without the angles split, inclined ones with fixed slices and with rows per
# lane, unpaired forwards (angles over half a turn) of 32 slices and more (whose back projection multiplies
# row by row into the sum, two roundings per angle)
CASES = [(288, 28, 60, 0.0, 360.0, 0.0), (200, 24, 180, 0.0, 360.0, 0.0), (320, 1, 180, 0.01, 180.0, 0.0),
         (128, 96, 60, 0.005, 360.0, 12.0), (64, 128, 90, 0.01, 360.0, 20.0), (90, 40, 120, 0.0, 180.0, 4.0),
         (160, 48, 120, 0.01, 180.0, 0.0), (128, 32, 90, 0.02, 180.0, 0.0)]


@pytest.mark.parametrize("n, nz, na, mu, span, incl", CASES)
def test_no_further_from_float64(gpu, n, nz, na, mu, span, incl):
    import torch
    import oracle.d1 as d1
    from vamtoolbox_amd.parallel import ParallelPlan
    ang = np.linspace(0.0, span, na, endpoint=False)
    rng = np.random.default_rng(n + nz)
    kw = dict(mu=mu, incl_deg=incl)
    plan, lane = [ParallelPlan(n, nz, ang, warp_clip=False, per_lane_geometry=p, device=gpu, **kw) for p in (False, True)]
    at = np.unique(np.linspace(0, nz - 1, 6).astype(int))
    for name, shape in (("forward", (n, n, nz)), ("backward", (n, na, nz))):
        if name == "backward" and nz >= 32 and not incl:
            continue
        x = torch.tensor(rng.uniform(0.2, 1.0, shape), dtype=torch.float32, device=gpu)
        x64 = x.cpu().numpy().astype(np.float64)
        got, ref = [getattr(p, name)(x).cpu().numpy()[..., at] for p in (plan, lane)]
        exact = getattr(d1, name)(x64 if incl else x64[..., at], ang, **kw, **({"clip_output": False} if name == "forward" else {}))
        if incl:
            exact = exact[..., at]
        e, e_lane = rel_l2(got, exact), rel_l2(ref, exact)
        print("%s: %.3e, per lane %.3e, ratio %.2f" % (name, e, e_lane, e / e_lane), flush=True)
        assert e <= 1.05 * e_lane


@pytest.mark.parametrize("n, nz, na, span, incl", [(128, 96, 60, 360.0, 12.0), (96, 150, 48, 360.0, 5.0),
                                                   (128, 64, 75, 180.0, 0.0), (160, 40, 60, 180.0, 0.0)])
def test_equal_samples(gpu, n, nz, na, span, incl):
    """Equal samples round a running sum the same way every time, so the per-lane kernels' error grows with the
    ray.  Sums of at most 16 samples round at most at 16 / n of the ray's size, and the n / 16 additions of those
    sums at its size but not all alike: below 0.7 of the per-lane error for n >= 96."""
    import torch
    import oracle.d1 as d1
    from vamtoolbox_amd.parallel import ParallelPlan
    ang = np.linspace(0.0, span, na, endpoint=False) + 0.5
    plan, lane = [ParallelPlan(n, nz, ang, incl_deg=incl, warp_clip=False, per_lane_geometry=p, device=gpu)
                  for p in (False, True)]
    x = torch.full((n, n, nz), 0.7, device=gpu)
    at = np.linspace(nz // 3, 2 * nz // 3, 5).astype(int)
    x64 = x.cpu().numpy().astype(np.float64)
    exact = d1.forward(x64 if incl else x64[..., at], ang, incl_deg=incl, clip_output=False)
    if incl:
        exact = exact[..., at]
    e, e_lane = [rel_l2(p.forward(x).cpu().numpy()[..., at], exact) for p in (plan, lane)]
    print("%.3e, per lane %.3e, ratio %.2f" % (e, e_lane, e / e_lane), flush=True)
    assert e <= 0.7 * e_lane
