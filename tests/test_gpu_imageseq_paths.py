"""Order statistics and frames at the edges of their paths: arrays that the list of candidates holds as a
whole and just not, buckets of equal values larger than the list, candidates in few blocks, odd lengths and
misaligned arrays; frames whose rows are and are not multiples of 16 bytes, image tiles with remainders,
overlapping copies.  Values and bytes are equal to NumPy's, without tolerance."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _data(kind, n, rng):
    x = rng.standard_normal(n)
    if kind == "ties":        # more equal values than the list holds, and few above them
        x = np.where(rng.random(n) < 0.9, 0.25, x)
    elif kind == "near":      # all candidates in one 24-bit bucket until the last digits
        x = 1.0 + rng.integers(0, 1 << 20, n) * 2.0 ** -52
    elif kind == "block":     # the candidates lie together in the array
        x = np.sort(x)
    elif kind == "signs":
        x = np.where(rng.random(n) < 0.5, 0.0, -0.0) + np.where(rng.random(n) < 0.3, np.inf * np.sign(x), 0.0)
    elif kind == "nan":
        x[rng.integers(0, n)] = np.nan
    return x


@pytest.mark.parametrize("n", [1, 2, 1023, 32767, 32768, 32769, 100001, 3000001])
@pytest.mark.parametrize("kind", ["normal", "ties", "near", "block", "signs", "nan"])
def test_order_statistics_paths(gpu, n, kind):
    import torch
    from vamtoolbox_amd.imagesequence import _order_stats
    print(n, kind, flush=True)
    x = _data(kind, n, np.random.default_rng(n))
    s = np.sort(x)
    t = torch.tensor(x, dtype=torch.float64, device=gpu)
    shifted = torch.cat([torch.zeros(1, dtype=torch.float64, device=gpu), t])[1:]
    for r in sorted({0, n // 7, n // 2, int(0.95 * (n - 1)), max(n - 2, 0), n - 1}):
        for a in (t, shifted):
            got = _order_stats(a, r)
            if kind == "nan":
                assert np.isnan(got).all()
            else:
                assert got[0] == s[r] and got[1] == s[min(r + 1, n - 1)], (r, got)


@pytest.mark.parametrize("nu, nv, n_u, n_v, offset", [(1, 1, 16, 16, 4), (64, 64, 64, 160, 64), (65, 63, 80, 200, 70),
                                                      (37, 130, 100, 300, 50), (130, 20, 148, 64, 16)])
@pytest.mark.parametrize("flips", [(False, False), (True, True)])
def test_frames_at_tile_edges(gpu, nu, nv, n_u, n_v, offset, flips):
    import ctypes
    import torch
    from vamtoolbox_amd import _lib
    lib = _lib.load()
    na = 3
    print(nu, nv, n_u, n_v, offset, flips, flush=True)
    rng = np.random.default_rng(nu * nv)
    x = rng.uniform(-20.0, 300.0, (nu, na, nv))
    u1, v1 = (n_u - nu) // 2, [3 % (n_v - nv + 1), min(3 + offset, n_v - nv)]   # copies overlap where offset < nv
    ref = np.zeros((na, n_v, n_u), dtype=np.uint8)
    y = x[::-1] if flips[0] else x
    y = y[:, :, ::-1] if flips[1] else y
    img = np.clip(y, 0.0, 255.0).astype(np.uint8).transpose(1, 2, 0)
    for v in v1:
        ref[:, v:v + nv, u1:u1 + nu] = img
    prm = _lib.ImgSeqParams()
    prm.n_u, prm.n_v, prm.u1, prm.n_copies, prm.bit_depth, prm.normalize = n_u, n_v, u1, 2, 8, 0
    prm.flip_u, prm.flip_v, prm.norm_value, prm.intensity_scale = int(flips[0]), int(flips[1]), 1.0, 1.0
    prm.v1[0], prm.v1[1] = v1
    t = torch.tensor(x, dtype=torch.float64, device=gpu)
    for shift in (0, 4):
        buf = torch.full((ref.size + 16,), 7, dtype=torch.uint8, device=gpu)
        out = buf[shift:shift + ref.size]
        _lib.check(lib.vamx_imgseq_compose(t.data_ptr(), nu, na, nv, ctypes.byref(prm), out.data_ptr(),
                                           _lib.stream_ptr(gpu)), "vamx_imgseq_compose")
        assert np.array_equal(out.cpu().numpy().reshape(ref.shape), ref)
        assert bool((buf[shift + ref.size:] == 7).all()) and bool((buf[:shift] == 7).all())
