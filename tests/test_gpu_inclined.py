"""Inclined projections on wavefronts against the float64 oracle, at the edges of their z layouts
(row groups of 8, 16, 32 lanes; 1, 2, 3 slabs of 64 rows; several chunks) and of the 64-sample and
64-angle tables; batched and fused-BCLP calls take the same kernels.

Tolerance: float32 data, float64 geometry.  A value sums at most 2 n taps (forward) or 4 n_angles
(back) of rounding 2^-24 each plus the weights' own 3 roundings, so relative L2 stays below
sqrt(4 * 200) * 2^-24 * 4 = 7e-6 <= 1e-5, the bound of the other projection tests."""

import numpy as np
import pytest

from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu

CASES = [(24, 1, 20, 9.0), (21, 7, 65, -7.0), (22, 8, 64, 12.0), (17, 15, 30, 25.0), (20, 16, 33, -3.0),
         (19, 31, 12, 8.0), (18, 32, 16, -20.0), (65, 63, 10, 5.0), (23, 64, 20, 15.0), (20, 127, 18, -11.0),
         (16, 128, 12, 10.0), (14, 192, 10, 6.0), (12, 260, 9, -8.0), (2, 40, 7, 30.0)]


@pytest.mark.parametrize("n, nz, na, incl", CASES)
@pytest.mark.parametrize("mu, off", [(0.0, 0.0), (0.03, 1.5)])
def test_inclined_parity(gpu, n, nz, na, incl, mu, off):
    import torch
    import oracle.d1 as d1
    from vamtoolbox_amd.parallel import ParallelPlan
    ang = np.linspace(0.0, 360.0, na, endpoint=False)
    rng = np.random.default_rng(n * 1000 + nz)
    vol, sino = rng.uniform(-1, 1, (n, n, nz)), rng.uniform(0, 1, (n, na, nz))
    kw = dict(mu=mu, det_offset=off, incl_deg=incl)
    print("n %d nz %d na %d %s" % (n, nz, na, kw), flush=True)
    plan = ParallelPlan(n, nz, ang, device=gpu, **kw)
    f = plan.forward(torch.tensor(vol, dtype=torch.float32, device=gpu)).cpu().numpy()
    b = plan.backward(torch.tensor(sino, dtype=torch.float32, device=gpu)).cpu().numpy()
    e1, e2 = rel_l2(f, d1.forward(vol, ang, **kw)), rel_l2(b, d1.backward(sino, ang, **kw))
    print("rel L2 forward %.2e backward %.2e" % (e1, e2))
    assert e1 <= 1e-5 and e2 <= 1e-5


@pytest.mark.parametrize("nz", [6, 70])
def test_inclined_non_finite_voxel_stays_on_its_rays(gpu, nz):
    """One infinite voxel (sinogram sample) changes only the rays (voxels) that the per-lane kernels,
    which read no weightless tap, find changed."""
    import torch
    from vamtoolbox_amd.parallel import ParallelPlan
    n, ang = 20, np.arange(0.0, 360.0, 30.0)
    plans = [ParallelPlan(n, nz, ang, incl_deg=10.0, device=gpu, per_lane_geometry=p) for p in (False, True)]
    vol, sino = torch.rand(n, n, nz, device=gpu), torch.rand(n, len(ang), nz, device=gpu)
    vol[0, 0, 0] = float("inf")
    vol[9, 10, nz // 2] = float("inf")
    sino[0, 0, 0] = float("inf")
    sino[11, 5, nz // 2] = float("inf")
    for name, x in (("forward", vol), ("backward", sino)):
        got, ref = [torch.isfinite(getattr(p, name)(x)) for p in plans]
        print(name, int((~got).sum()), int((~ref).sum()))
        assert bool((got | ~ref).all()) and not bool(got.all())


def test_inclined_batched_and_fused(gpu):
    """The batched call is bitwise the single calls; the fused BCLP step equals its unfused loop to rounding."""
    import torch
    import vamtoolbox_amd as vam
    from vamtoolbox_amd.batch import ParallelBatch
    from vamtoolbox_amd.parallel import ParallelPlan
    plans = [ParallelPlan(n, nz, np.linspace(0, 360, na, endpoint=False), mu=0.01, incl_deg=inc, device=gpu)
             for n, nz, na, inc in [(20, 12, 30, 8.0), (24, 70, 20, -5.0), (18, 40, 16, 0.0)]]
    B = ParallelBatch(plans)
    v, s = torch.rand(B.n_vol, device=gpu), torch.rand(B.n_sino, device=gpu)
    f, b = B.forward(v), B.backward(s)
    for p, vi, si, fi, bi in zip(plans, B.vol_views(v), B.sino_views(s), B.sino_views(f), B.vol_views(b)):
        assert torch.equal(p.forward(vi.clone()), fi) and torch.equal(p.backward(si.clone()), bi)
    n, nz = 24, 20
    t = np.zeros((n, n, nz))
    t[8:16, 9:15, 4:16] = 1.0
    pg = vam.geometry.ProjectionGeometry(np.linspace(0, 360, 40, endpoint=False), "parallel", CUDA=True,
                                         inclination_angle=10.0)
    g0 = torch.rand(n, 40, nz, device=gpu) * 0.05
    out = []
    for fused in (True, False):
        rm = vam.response.ResponseModel(type="analytical", B=20, M=0.6)
        o = vam.optimize.Options(method="BCLP", n_iter=3, response_model=rm, eps=0.05, learning_rate=1e-3, g0=g0,
                                 fused=fused)
        out.append(vam.optimize.optimize(vam.geometry.TargetGeometry(target=t), pg, o, output="components"))
    e = rel_l2(out[0][0], out[1][0])
    print("fused vs unfused rel L2 %.2e" % e)
    assert e <= 1e-6
    np.testing.assert_allclose(out[0][3].loss, out[1][3].loss, rtol=1e-9)
