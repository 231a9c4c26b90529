"""Ray tracer's integral of a volume that is zero but for its outermost voxels, whose cells reach one voxel past
the grid on every side, after a deposit (which uses the same scratch memory); against the float64 oracle.

Tolerance: that of the interaction's float32 weights and positions, relative L2 <= 5e-6 of the same rays'
integral of a volume of ones (an integral of outer voxels alone is a few of its terms)."""

import numpy as np
import pytest

from tests.test_gpu_raytrace import _oracle, _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, nz, incl", [(2, 1, 0.0), (9, 1, 0.0), (2, 2, 0.0), (8, 3, 6.0), (9, 13, -5.0), (16, 20, 0.0)])
@pytest.mark.parametrize("solver", ["rk4", "leapfrog"])
def test_outer_voxels(gpu, n, nz, incl, solver):
    import torch
    from vamtoolbox_amd.projector.pyTorchRayTrace import PyTorchRayTracingPropagator
    print(n, nz, incl, solver, flush=True)
    ang = np.array([0.0, 27.0, 90.0, 180.0, 211.0])
    tg, pg, cv, nf, im, am, ab = _setup(n, nz, ang, solver, "canonical", incl, att=False, absorb=False,
                                        seed=nz)
    P = PyTorchRayTracingPropagator(tg, pg, output_torch_tensor=True)
    tr, x0, v0, shape, e0 = _oracle(tg, pg, cv, nf, am, ab, solver, "canonical", incl)
    f = np.random.default_rng(n + nz).random((n, n, nz)) + 1.0
    f[1:-1, 1:-1, 1 if nz > 2 else 0:nz - 1 if nz > 2 else nz] = 0.0
    P.backward(torch.full((int(np.prod(shape)),), 3.0, device=gpu))
    got = P.forward(torch.tensor(f, dtype=torch.float32, device=gpu)).cpu().numpy().reshape(-1)
    want = np.asarray(tr.run(x0, v0, e0, f=f)).reshape(-1)
    err = np.linalg.norm(got - want) / np.linalg.norm(np.asarray(tr.run(x0, v0, e0, f=np.ones_like(f))))
    print("error %.2e" % err)
    assert err <= 5e-6
