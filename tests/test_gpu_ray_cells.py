"""Ray tracer against the float64 oracle where rays of a wavefront share, leave and re-enter cells: rows of
z below, at and past a wavefront, rays of zero energy among the others (lanes that trace nothing between
lanes that pass their taps on), inclined rays that leave through z, one slice.

Tolerance: an interaction's float32 weight has about 8 roundings of 2^-24, and the float32 slopes move a
position by at most 3 n half-voxel steps of 2^-24, 3e-6 voxels at n = 14: relative L2 <= 5e-6.  No
attenuation, so that no step's attenuation depends on which side of a boundary it starts."""

import numpy as np
import pytest

from tests.conftest import rel_l2
from tests.test_gpu_raytrace import _oracle, _setup

pytestmark = pytest.mark.gpu

CASES = [(14, 1, 0.0), (14, 2, 0.0), (12, 3, 5.0), (9, 63, 0.0), (8, 64, 4.0), (8, 65, 0.0), (6, 130, -7.0)]


@pytest.mark.parametrize("n, nz, incl", CASES)
@pytest.mark.parametrize("solver, param", [("rk4", "canonical"), ("rk4", "physical_path_length"),
                                           ("forward_symplectic_euler", "canonical"), ("leapfrog", "canonical")])
def test_cells_parity(gpu, n, nz, incl, solver, param):
    import torch
    from vamtoolbox_amd.projector.pyTorchRayTrace import PyTorchRayTracingPropagator
    print(n, nz, incl, solver, param, flush=True)
    ang = np.array([0.0, 33.0, 90.0, 135.0, 250.0])
    tg, pg, cv, nf, im, am, ab = _setup(n, nz, ang, solver, param, incl, att=False, seed=nz)
    P = PyTorchRayTracingPropagator(tg, pg, output_torch_tensor=True)
    tr, x0, v0, shape, e0 = _oracle(tg, pg, cv, nf, am, ab, solver, param, incl)
    rng = np.random.default_rng(n + nz)
    f = rng.random((n, n, nz))
    g = rng.random(int(np.prod(shape))) * (rng.random(int(np.prod(shape))) < 0.8)
    Wf = P.forward(torch.tensor(f, dtype=torch.float32, device=gpu)).cpu().numpy()
    WTg = P.backward(torch.tensor(g, dtype=torch.float32, device=gpu)).cpu().numpy()
    e1, e2 = rel_l2(Wf, tr.run(x0, v0, e0, f=f)), rel_l2(WTg, tr.run(x0, v0, e0, g=g))
    print("rel L2 integrate %.2e deposit %.2e" % (e1, e2))
    assert e1 <= 5e-6 and e2 <= 5e-6
