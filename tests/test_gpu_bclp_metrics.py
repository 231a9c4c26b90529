"""The one-pass final evaluation of a dose against NumPy's float64, for every response and exponent branch,
sizes of one element to several blocks, scalar and array tolerances and weights, non-finite doses.

Sums of up to 10^6 float64 terms in another order and a last-bit difference per exponential or power:
relative 10^6 * 2^-53 = 1.1e-10 at most, 1e-10 here; counts and the mapped dose's non-finite places equal."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RESPONSES = [dict(type="analytical", form="gen_log_fun", B=25, M=0.5), dict(type="analytical", form="identity"),
             dict(type="analytical", form="gen_log_fun", B=10, M=0.4, nu=0.7), dict(type="interpolation", form="gen_log_fun")]


@pytest.mark.parametrize("n", [1, 255, 257, 300007])
@pytest.mark.parametrize("p, arrays, special", [(2.0, False, False), (2.0, True, True), (3.0, True, False),
                                                (1.5, False, True)])
@pytest.mark.parametrize("resp", range(len(RESPONSES)))
def test_bclp_metrics(gpu, n, p, arrays, special, resp):
    import torch
    from vamtoolbox_amd import _lib
    from vamtoolbox_amd.response import ResponseModel
    model = ResponseModel(**RESPONSES[resp])
    rng = np.random.default_rng(n)
    d = rng.uniform(0, 1.5, n).astype(np.float32)
    if special:
        d[n // 2] = np.inf
        d[n // 3] = np.nan
    t = (rng.random(n) < 0.4).astype(np.float32)
    eps, w = [np.full(n, v, np.float32) for v in (0.1, 0.5)]
    if arrays:
        eps, w = rng.uniform(0, 0.3, n).astype(np.float32), rng.uniform(0, 2, n).astype(np.float32)
    dev = [torch.tensor(x, device=gpu) for x in (d, t, eps, w)]
    st, tabs = model.vamx_struct(gpu)
    prm = _lib.BclpParams(p=p, q=1.0, eps=float(eps[0]), weight=float(w[0]), learning_rate=1.0, glb=-np.inf, gub=np.inf,
                          dvol=1.0, grad_op=0)
    mapped = torch.empty(n, dtype=torch.float64, device=gpu)
    out = torch.empty(_lib.BCLP_METRICS * (1 + _lib.BCLP_METRIC_BLOCKS), dtype=torch.float64, device=gpu)
    _lib.check(_lib.load().vamx_bclp_metrics(
        ctypes.byref(st), ctypes.byref(prm), dev[0].data_ptr(), dev[1].data_ptr(), dev[2].data_ptr() if arrays else 0,
        dev[3].data_ptr() if arrays else 0, n, mapped.data_ptr(), out.data_ptr(), _lib.stream_ptr(gpu)), "metrics")
    with np.errstate(all="ignore"):
        m = model.map(d.astype(np.float64))
        e = m - t
        ae = np.abs(e)
        b = ae - eps.astype(np.float64)
        v, u, ab = (b > 0) * 1.0, (ae > 0) * 1.0, np.abs(b)
        ref = [np.sum(v * w * ab ** p), v.sum(), u.sum(), np.sum(v * ab), ae.sum(), np.sum(v * b * b), np.sum(e * e),
               np.max(v * ab), np.max(u * ae)]
    got = out[:9].cpu().numpy()
    np.testing.assert_allclose(mapped.cpu().numpy(), m, rtol=1e-12, atol=1e-15)
    np.testing.assert_allclose(got, ref, rtol=1e-10, atol=1e-15)
    assert got[1] == ref[1] and got[2] == ref[2]
