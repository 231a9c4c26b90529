"""Back projection with detectors shifted until the two angles of an opposite pair share one bin (n = 2
centred, half a width either way), and one step inside and outside that, against the float64 oracle, alone and
in a batch.

At most 2 n_angles float32 terms with about 4 roundings of 2^-24 each: relative L2 <= sqrt(2 * 36) * 4 *
2^-24 = 2.0e-6 <= 5e-6."""

import numpy as np
import pytest

from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu

CASES = [(2, 0.0), (2, 0.5), (2, -0.5), (3, -1.0), (3, 1.0), (4, 1.0), (4, 0.5), (16, 7.0), (16, 6.5), (16, 7.5),
         (16, -8.0), (33, -16.0), (33, -15.5), (33, -16.5), (33, 16.0), (33, 15.5), (33, 16.5)]


@pytest.mark.parametrize("n, off", CASES)
@pytest.mark.parametrize("nz, na", [(32, 4), (100, 36), (192, 12)])
def test_single_shared_bin(gpu, n, off, nz, na):
    import torch
    import oracle.d1 as d1
    from vamtoolbox_amd.batch import ParallelBatch
    from vamtoolbox_amd.parallel import ParallelPlan
    print("n %d off %g nz %d na %d" % (n, off, nz, na), flush=True)
    ang = np.linspace(0.0, 360.0, na, endpoint=False)
    plan = ParallelPlan(n, nz, ang, det_offset=off, circle_clip=False, device=gpu)
    other = ParallelPlan(5, nz, ang, device=gpu)
    rng = np.random.default_rng(n * 1000 + nz)
    s = torch.tensor(rng.uniform(0.1, 1, (n, na, nz)), dtype=torch.float32, device=gpu)
    ref = d1.backward(s.cpu().numpy().astype(np.float64), ang, clip=False, det_offset=off)
    got = plan.backward(s)
    e = rel_l2(got.cpu().numpy(), ref)
    assert e <= 5e-6, e
    flat = ParallelBatch([plan, other]).backward(torch.cat([s.reshape(-1), torch.zeros(5 * na * nz, device=gpu)]))
    assert torch.equal(flat[: n * n * nz].view(ref.shape), got)


@pytest.mark.parametrize("n, nz", [(20, 40), (33, 128), (24, 256)])
def test_unpaired_plan_sums_angle_by_angle(gpu, n, nz):
    """fp_pair = 0 keeps the back projection unpaired too: without absorption the sums are bitwise those of a
    plan with an absorption so small that every weight is 1, which never combines angles."""
    import torch
    from vamtoolbox_amd.parallel import ParallelPlan
    ang = np.arange(0.0, 360.0, 15.0)
    plain, weak = [ParallelPlan(n, nz, ang, mu=mu, radius=1e6, device=gpu) for mu in (0.0, 1e-300)]
    s = torch.rand(plain.sino_shape, device=gpu)
    paired = plain.backward(s)
    plain.set_tuning(fp_pair=0)
    assert torch.equal(plain.backward(s), weak.backward(s))
    assert not torch.equal(paired, weak.backward(s))   # the two orders can be told apart here
    plain.set_tuning(fp_pair=1)
    assert torch.equal(plain.backward(s), paired)
