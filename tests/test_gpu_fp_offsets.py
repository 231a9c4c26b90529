"""Forward projection where a voxel column's byte offset from the first row of 64 samples passes 32 bits
(few columns, many slices: offsets from each sample's own cell), just below that, and ordinary sizes with
gaps between a ray's samples (absorption that underflows along a chord's middle), against the float64
oracle on some slices.

At most 2 n samples of about 6 roundings of 2^-24 each, 4 voxels a sample: relative L2 <= 4 * 2^-24 *
sqrt(6) = 6e-7 for independent errors, bounded here by 5e-6."""

import numpy as np
import pytest

from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, nz, mu", [(2, 8400000, 0.0), (3, 5500001, 0.01), (2, 8000000, 0.01), (33, 130, 60.0),
                                       (20, 64, 25.0), (97, 192, 0.01), (64, 77, 0.0)])
@pytest.mark.parametrize("pair", [1, 0])
def test_tap_offsets(gpu, n, nz, mu, pair):
    import torch
    import oracle.d1 as d1
    from vamtoolbox_amd.parallel import ParallelPlan
    print(n, nz, mu, pair, flush=True)
    ang = np.array([0.0, 30.0, 45.0, 180.0, 210.0, 225.0]) if n > 3 else np.array([20.0, 200.0])
    vol = torch.randn((n, n, nz), device=gpu, generator=torch.Generator(gpu).manual_seed(n))
    vol[0, 0], vol[-1, -1] = 1.0, -1.0   # every slice's range holds zero: no sample is clipped
    plan = ParallelPlan(n, nz, ang, mu=mu, device=gpu)
    plan.set_tuning(fp_pair=pair)
    got = plan.forward(vol)
    at = sorted({0, 1, nz // 2, nz - 2, nz - 1})
    ref = d1.forward(vol[:, :, at].cpu().numpy().astype(np.float64), ang, mu=mu)
    e = rel_l2(got[:, :, at].cpu().numpy(), ref)
    print("rel L2 %.2e" % e)
    assert e <= 5e-6
