"""Forward projection in every layout of slices over lanes, and where a voxel column's byte offset from the
first row of 64 samples passes 32 bits (few columns, many slices: offsets from each sample's own cell),
just below that, and at ordinary sizes with gaps between a ray's samples (absorption that underflows along
a chord's middle), against the float64 oracle.

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


@pytest.mark.parametrize("nz", [32, 40, 56, 63, 64, 65, 100, 127, 128, 129, 180, 191, 192, 193, 255, 256, 257, 300])
@pytest.mark.parametrize("positive", [False, True])
def test_slice_layouts(gpu, nz, positive):
    """One to four slices per lane, 64 apart or consecutive, in one or more chunks: single, in a batch and with
    the BCLP update, clipped and not, aligned and not, under every limit on the slices per lane."""
    import torch
    import oracle.d1 as d1
    from vamtoolbox_amd.batch import ParallelBatch
    from vamtoolbox_amd.parallel import ParallelPlan
    print(nz, positive, flush=True)
    n, ang = 19, np.arange(0.0, 360.0, 24.0 if nz % 2 else 30.0)
    rng = np.random.default_rng(nz)
    vol = torch.tensor(rng.uniform(0.2 if positive else -1.0, 1.0, (n, n, nz)), dtype=torch.float32, device=gpu)
    shifted = torch.cat([torch.zeros(1, device=gpu), vol.reshape(-1)])[1:].view(vol.shape)
    ref = d1.forward(vol.cpu().numpy().astype(np.float64), ang, mu=0.01)
    plans = [ParallelPlan(m, nz, ang, mu=0.01, device=gpu) for m in (n, n + 1)]
    for tuning in (dict(), dict(fp_zv=2), dict(fp_zv=1), dict(z_split=0), dict(fp_pair=0), dict(fp_reuse=0)):
        plans[0].set_tuning(**dict(dict(fp_zv=4, z_split=1, fp_pair=1, fp_reuse=1), **tuning))
        for x in (vol, shifted):
            e = rel_l2(plans[0].forward(x).cpu().numpy(), ref)
            assert e <= 5e-6, (tuning, e)
    plans[0].set_tuning(fp_zv=4, z_split=1, fp_pair=1, fp_reuse=1)
    one = plans[0].forward(vol)
    flat = ParallelBatch(plans).forward(torch.cat([vol.reshape(-1), torch.ones((n + 1) ** 2 * nz, device=gpu)]))
    assert rel_l2(flat[: one.numel()].view(one.shape).cpu().numpy(), ref) <= 5e-6
