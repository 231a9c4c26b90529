"""The back projection's patches (matrix products of rows and column weights) against the float64
oracle, at the edges of the slice layouts (1 to 4 slices per lane, contiguous or 64 apart), of the patch
tiles (n not a multiple of 2, 4 or the tile) and of the pairs of opposite angles.

At most 2 n_angles float32 terms with about 4 roundings of 2^-24 each: relative L2 <= sqrt(2 * 61) * 4 *
2^-24 = 2.7e-6 <= 5e-6.  In a batch the same sums run in the same order: bitwise equal."""

import numpy as np
import pytest

from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu

CASES = [(2, 32, 5), (3, 33, 16), (5, 64, 17), (9, 65, 1), (21, 96, 32), (16, 128, 12), (17, 129, 60), (33, 192, 20),
         (20, 193, 8), (18, 256, 24), (35, 257, 48), (7, 320, 61), (70, 40, 36)]


@pytest.mark.parametrize("n, nz, na", CASES)
@pytest.mark.parametrize("mu, off", [(0.02, 0.0), (0.01, 1.5), (0.0, 0.0), (0.0, 1.5), (0.0, -2.0), (0.0, 0.3)])
@pytest.mark.parametrize("clip", [True, False])
def test_patch_parity(gpu, n, nz, na, mu, off, clip):
    import torch
    import oracle.d1 as d1
    from vamtoolbox_amd.batch import ParallelBatch
    from vamtoolbox_amd.parallel import ParallelPlan
    print("n %d nz %d na %d mu %g off %g clip %s" % (n, nz, na, mu, off, clip), flush=True)
    ang = np.linspace(0.0, 360.0, na, endpoint=False)
    kw = dict(mu=mu, det_offset=off)
    plan, plan2 = [ParallelPlan(m, nz, ang, circle_clip=clip, device=gpu, **kw) for m in (n, n + 1)]
    rng = np.random.default_rng(n * 1000 + nz)
    s = torch.tensor(rng.uniform(-1, 1, (n, na, nz)), dtype=torch.float32, device=gpu)
    shifted = torch.cat([torch.zeros(1, device=gpu), s.reshape(-1)])[1:].view(s.shape)
    ref = d1.backward(s.cpu().numpy().astype(np.float64), ang, clip=clip, **kw)
    for x in (s, shifted):
        e = rel_l2(plan.backward(x).cpu().numpy(), ref)
        assert e <= 5e-6, e
    batch = ParallelBatch([plan, plan2])
    flat = batch.backward(torch.cat([s.reshape(-1), torch.zeros((n + 1) * na * nz, device=gpu)]))
    assert torch.equal(flat[: n * n * nz].view(ref.shape), plan.backward(s))


@pytest.mark.parametrize("mu", [0.0, 0.02])
@pytest.mark.parametrize("nz", [40, 128, 256])
def test_patches_keep_non_finite_and_largest_values(gpu, mu, nz):
    """Infinite samples reach the columns that the per-lane kernels find them in, and samples whose sum
    over two opposite angles would overflow but whose weighted values do not stay finite."""
    import torch
    from vamtoolbox_amd.parallel import ParallelPlan
    n, ang = 20, np.arange(0.0, 360.0, 30.0)
    plan, lanes = [ParallelPlan(n, nz, ang, mu=mu, device=gpu, per_lane_geometry=p) for p in (False, True)]
    s = torch.rand(n, len(ang), nz, device=gpu)
    s[0, 0, 0] = s[11, 5, nz // 2] = float("inf")
    s[6, 3, 5] = float("nan")
    got, ref = plan.backward(s), lanes.backward(s)
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(torch.isinf(got), torch.isinf(ref))
    big = torch.zeros_like(s)
    big[9, 1] = 3.0e38
    big[11, 7] = 3.0e38   # the mirrored bin of the opposite angle
    got, ref = plan.backward(big), lanes.backward(big)
    assert torch.equal(torch.isfinite(got), torch.isfinite(ref)) and bool(torch.isfinite(ref).any())
