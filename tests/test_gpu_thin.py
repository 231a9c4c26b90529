"""Thin problems (fewer than 32 slices) on lane groups against the float64 oracle, at the edges of
the group widths (1, 2, 4, 8, 16, 32 lanes of one or four slices) and of the angle split, with the
warp clip inactive and active, paired and unpaired, aligned and misaligned buffers.

Tolerance: a value sums at most 2 n (forward) or 2 n_angles (back) float32 terms, each with about
4 roundings of 2^-24: relative L2 <= sqrt(2 * 700) * 4 * 2^-24 = 9e-6 <= 1e-5."""

import numpy as np
import pytest

from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu

CASES = [(2, 1, 3), (21, 1, 1), (40, 1, 64), (200, 1, 90), (20, 2, 7), (23, 3, 40), (22, 4, 30), (19, 5, 17),
         (24, 8, 33), (17, 9, 16), (20, 12, 24), (25, 16, 15), (18, 17, 48), (33, 20, 36), (21, 28, 20), (20, 31, 12)]


@pytest.mark.parametrize("n, nz, na", CASES)
@pytest.mark.parametrize("mu, off, positive", [(0.0, 0.0, False), (0.02, 1.5, False), (0.01, 0.3, True)])
def test_thin_parity(gpu, n, nz, na, mu, off, positive):
    import torch
    import oracle.d1 as d1
    from vamtoolbox_amd.parallel import ParallelPlan
    ang = np.linspace(0.0, 360.0, na, endpoint=False)
    rng = np.random.default_rng(n * 100 + nz)
    vol = rng.uniform(0.2, 1.0, (n, n, nz)) if positive else rng.uniform(-1, 1, (n, n, nz))
    sino = rng.uniform(0, 1, (n, na, nz))
    kw = dict(mu=mu, det_offset=off)
    print("n %d nz %d na %d %s positive %s" % (n, nz, na, kw, positive), flush=True)
    rf, rb = d1.forward(vol, ang, **kw), d1.backward(sino, ang, **kw)
    tv, ts = [torch.tensor(a, dtype=torch.float32, device=gpu) for a in (vol, sino)]
    plan = ParallelPlan(n, nz, ang, device=gpu, **kw)
    shifted = [torch.cat([torch.zeros(1, device=gpu), t.reshape(-1)])[1:].view(t.shape) for t in (tv, ts)]
    for pair, (v, s) in ((1, (tv, ts)), (0, (tv, ts)), (1, shifted)):
        plan.set_tuning(fp_pair=pair)
        e1, e2 = rel_l2(plan.forward(v).cpu().numpy(), rf), rel_l2(plan.backward(s).cpu().numpy(), rb)
        print("pair %d rel L2 forward %.2e backward %.2e" % (pair, e1, e2))
        assert e1 <= 1e-5 and e2 <= 1e-5


@pytest.mark.parametrize("nz", [1, 6, 24])
def test_thin_non_finite_values_stay_on_their_rays(gpu, nz):
    """Infinite voxels and samples change only what the per-lane kernels find changed."""
    import torch
    from vamtoolbox_amd.parallel import ParallelPlan
    n, ang = 20, np.arange(0.0, 360.0, 30.0)
    plans = [ParallelPlan(n, nz, ang, device=gpu, warp_clip=False, per_lane_geometry=p) for p in (False, True)]
    vol, sino = torch.rand(n, n, nz, device=gpu), torch.rand(n, len(ang), nz, device=gpu)
    vol[0, 0, 0] = vol[9, 10, nz // 2] = float("inf")
    sino[0, 0, 0] = sino[11, 5, nz // 2] = float("inf")
    for name, x in (("forward", vol), ("backward", sino)):
        got, ref = [torch.isfinite(getattr(p, name)(x)) for p in plans]
        assert bool((got | ~ref).all()) and not bool(got.all())


@pytest.mark.parametrize("n, nz", [(10, 1), (40, 1), (130, 1), (300, 1), (20, 30), (33, 700), (7, 1100)])
def test_slice_range_clips_every_slice(gpu, n, nz):
    """Slices whose range excludes zero clip their samples to it: a constant slice projects to the count
    of its samples' coverage, exactly as the oracle's (one and several blocks of the range pass)."""
    import torch
    import oracle.d1 as d1
    from vamtoolbox_amd.parallel import ParallelPlan
    rng = np.random.default_rng(n + nz)
    vol = np.ones((n, n, nz)) * rng.uniform(0.5, 1.5, (1, 1, nz))
    ang = np.array([0.0, 33.0, 213.0])
    plan = ParallelPlan(n, nz, ang, device=gpu)
    got = plan.forward(torch.tensor(vol, dtype=torch.float32, device=gpu)).cpu().numpy()
    e = rel_l2(got, d1.forward(vol.astype(np.float32).astype(np.float64), ang))
    assert e <= 1e-5, e
