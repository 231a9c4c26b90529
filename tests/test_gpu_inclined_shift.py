"""Inclined forward projection with slices fixed to lanes: one to four slices per lane, one and several
chunks of rows, shifts of both signs up to several slices per sample, samples on whole columns (taps of
weight 0), and column offsets past 32 bits, against the float64 oracle.

Tolerance: a value sums at most 2 n taps of a few roundings of 2^-24: relative L2 <= sqrt(2 * 130) * 4 *
2^-24 = 4e-6 <= 1e-5, the bound of the other inclined tests."""

import numpy as np
import pytest

from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, nz, incl", [(40, 64, 3.0), (40, 64, -3.0), (60, 96, 12.0), (130, 96, -12.0), (64, 97, 20.0),
                                         (30, 180, 25.0), (31, 255, -9.0), (24, 300, 14.0), (20, 520, 6.0),
                                         (12, 100, 70.0), (12, 100, -75.0), (2, 200, 45.0)])
@pytest.mark.parametrize("mu, off", [(0.0, 0.0), (0.03, 1.5), (12.0, 0.3)])
def test_fixed_slices(gpu, n, nz, incl, mu, off):
    import torch
    import oracle.d1 as d1
    from vamtoolbox_amd.parallel import ParallelPlan
    ang = np.array([0.0, 20.0, 45.0, 90.0, 137.0, 180.0, 250.0, 270.0])
    vol = np.random.default_rng(n * 1000 + nz).uniform(-1, 1, (n, n, nz)).astype(np.float32)
    kw = dict(mu=mu, det_offset=off, incl_deg=incl)
    print("n %d nz %d %s" % (n, nz, kw), flush=True)
    got = ParallelPlan(n, nz, ang, device=gpu, **kw).forward(torch.tensor(vol, device=gpu)).cpu().numpy()
    e = rel_l2(got, d1.forward(vol.astype(np.float64), ang, **kw))
    assert e <= 1e-5, e


@pytest.mark.parametrize("n, nz", [(2, 5500000), (3, 2500001)])
def test_fixed_slices_far_offsets(gpu, n, nz):
    import torch
    import oracle.d1 as d1
    from vamtoolbox_amd.parallel import ParallelPlan
    ang, kw = np.array([20.0, 100.0]), dict(mu=0.01, incl_deg=15.0)
    print(n, nz, flush=True)
    vol = torch.randn((n, n, nz), device=gpu, generator=torch.Generator(gpu).manual_seed(n))
    got = ParallelPlan(n, nz, ang, device=gpu, **kw).forward(vol)
    for j in (4, nz // 2, nz - 5):
        part = vol[:, :, j - 4:j + 5].cpu().numpy().astype(np.float64)
        e = rel_l2(got[:, :, j].cpu().numpy(), d1.forward(part, ang, **kw)[:, :, 4])
        assert e <= 1e-5, (j, e)
