"""Problems of a batch that share launches, by class of kernel and lanes (thin, inclined, and forward ones): bitwise the single
calls, over sizes on both sides of an own launch, uneven mixtures, misaligned buffers, more problems than a launch
holds, the warp clip on and off, and with the first call under capture (where no table can be built)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _plans(gpu, mix, warp_clip):
    from vamtoolbox_amd.parallel import ParallelPlan
    if mix == "slices":
        sizes = [(20, 1, 12, 0.0)] * 70
    elif mix == "one":
        sizes = [(20, 3, 12, 0.0)]
    elif mix == "thin":
        sizes = [(n, nz, na, 0.0) for n, nz, na in [(16, 1, 9), (33, 2, 40), (24, 3, 16), (21, 4, 24), (40, 8, 64), (17, 7, 33),
                                                    (30, 16, 20), (18, 17, 18), (25, 28, 30), (20, 31, 200), (128, 1, 180)]]
    elif mix == "inclined":
        sizes = [(20, 5, 20, 4.0), (18, 12, 30, -8.0), (22, 31, 18, 15.0), (16, 40, 20, 10.0), (16, 100, 12, -20.0),
                 (24, 260, 12, 6.0), (12, 5, 20, 40.0), (60, 96, 60, 12.0)]
    elif mix == "slabs":
        sizes = [(24, 40, 24, 0.0), (20, 33, 16, 0.0), (33, 100, 9, 0.0), (17, 200, 20, 0.0), (18, 257, 12, 0.0),
                 (24, 40, 24, 0.0), (21, 64, 30, 0.0), (16, 150, 16, 0.0), (22, 128, 40, 0.0), (80, 64, 120, 0.0)]
    else:
        sizes = [(20, 1, 20, 0.0), (24, 40, 20, 0.0), (18, 9, 16, 7.0), (33, 77, 24, 0.0), (16, 20, 30, 0.0), (20, 50, 16, -5.0)]
    return [ParallelPlan(n, nz, np.linspace(0.0, 360.0, na, endpoint=False), mu=0.01 * (i % 2), incl_deg=inc,
                         warp_clip=warp_clip, device=gpu) for i, (n, nz, na, inc) in enumerate(sizes)]


def _alike(view):
    """A buffer of the view's shape and alignment (the problems' parts of the flat buffers lie at any offset, and
    the alignment decides the lanes' layout)."""
    import torch
    at = view.data_ptr() // 4 % 4
    return torch.zeros(view.numel() + 4, device=view.device)[at:at + view.numel()].view(view.shape)


def _check(plans, B, v, s, f, b):
    import torch
    for p, vi, si, fi, bi in zip(plans, B.vol_views(v), B.sino_views(s), B.sino_views(f), B.vol_views(b)):
        assert torch.equal(p.forward(vi, out=_alike(fi)), fi) and torch.equal(p.backward(si, out=_alike(bi)), bi)


@pytest.mark.parametrize("mix", ["slices", "one", "thin", "inclined", "mixed", "slabs"])
@pytest.mark.parametrize("warp_clip", [True, False])
@pytest.mark.parametrize("positive", [True, False])
def test_shared_launches(gpu, mix, warp_clip, positive):
    import torch
    from vamtoolbox_amd.batch import ParallelBatch
    print(mix, warp_clip, positive, flush=True)
    plans = _plans(gpu, mix, warp_clip)
    B = ParallelBatch(plans)
    v, s = torch.rand(B.n_vol, device=gpu) + (0.1 if positive else -0.5), torch.rand(B.n_sino, device=gpu)
    f, b = B.forward(v), B.backward(s)
    for _ in range(2):
        _check(plans, B, v, s, f, b)
        f.zero_(), b.zero_()
        B.forward(v, out=f), B.backward(s, out=b)   # the tables are there now


@pytest.mark.parametrize("mix", ["thin", "inclined"])
@pytest.mark.parametrize("warm", [True, False])
def test_capture(gpu, mix, warm):
    import torch
    from vamtoolbox_amd.batch import ParallelBatch
    plans = _plans(gpu, mix, True)
    B = ParallelBatch(plans)
    v, s = torch.rand(B.n_vol, device=gpu), torch.rand(B.n_sino, device=gpu)
    f, b = torch.zeros(B.n_sino, device=gpu), torch.zeros(B.n_vol, device=gpu)
    if warm:
        B.forward(v, out=f), B.backward(s, out=b)
        torch.cuda.synchronize()
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream(device=gpu)
    with torch.cuda.graph(graph, stream=stream):
        B.forward(v, out=f)
        B.backward(s, out=b)
    for k in range(3):
        v.mul_(0.5 + k)
        s.add_(0.25)
        graph.replay()
        torch.cuda.synchronize()
        _check(plans, B, v, s, f, b)
        f.zero_(), b.zero_()


def test_many_alignments(gpu):
    """Each problem's buffers aligned and not: more combinations than a batch keeps tables of."""
    import ctypes
    import torch
    from vamtoolbox_amd import _lib
    from vamtoolbox_amd.parallel import ParallelPlan
    lib = _lib.load()
    plans = [ParallelPlan(n, 4, np.linspace(0.0, 360.0, na, endpoint=False), mu=0.01, device=gpu)
             for n, na in [(12, 9), (16, 12), (18, 20), (21, 16)]]
    handle = ctypes.c_void_p()
    arr = (ctypes.c_void_p * 4)(*[p.handle for p in plans])
    _lib.check(lib.vamx_batch_create(arr, 4, ctypes.byref(handle)), "vamx_batch_create")

    def buffers(shapes, bits):
        out = []
        for j, sh in enumerate(shapes):
            m = int(np.prod(sh))
            out.append(torch.rand(m + 4, device=gpu)[bits >> j & 1:][:m].view(sh))
        return out

    try:
        for bits in list(range(12)) + [0, 11]:
            v = buffers([p.vol_shape for p in plans], bits)
            s, f, b = (buffers([x.shape for x in y], bits) for y in ([torch.empty(p.sino_shape) for p in plans],
                                                                     [torch.empty(p.sino_shape) for p in plans], v))
            pv, ps, pf, pb = ((ctypes.c_void_p * 4)(*[x.data_ptr() for x in y]) for y in (v, s, f, b))
            _lib.check(lib.vamx_batch_forward(handle, pv, pf, _lib.stream_ptr(gpu)), "vamx_batch_forward")
            _lib.check(lib.vamx_batch_backward(handle, ps, pb, _lib.stream_ptr(gpu)), "vamx_batch_backward")
            for p, vi, si, fi, bi in zip(plans, v, s, f, b):
                assert torch.equal(p.forward(vi, out=_alike(fi)), fi) and torch.equal(p.backward(si, out=_alike(bi)), bi)
    finally:
        torch.cuda.synchronize()
        lib.vamx_batch_destroy(handle)
