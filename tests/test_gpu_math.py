"""The shared elementary functions (brian2_amd/csrc/hb_math.h): the device's results are the
host's, bit for bit, and the host's are within an ulp of libm's, at the edges of every range."""
import ctypes
import math

import numpy as np
import pytest

EDGES = [0.0, 1.0, 2.0, 3.0, 4.0, 0.5, math.sqrt(2.0), math.sqrt(0.5), math.inf, 709.782712893384, 709.8, 710.0,
         745.1332191019412, 745.2, 708.396418532264, 700.0, 701.0, 717.0, 718.0, 40.0, 1e-16, 1e-17, 2.0**-60, 2.0**-61,
         5e-324, 2.2250738585072014e-308, 1e-310, 1.7976931348623157e308, 2.0**53, 2.0**53 + 2, 1e300, 1 / 18, 0.025]


def _arguments():
    rng = np.random.default_rng(7)
    e = np.array(EDGES)
    e = np.concatenate([e, np.nextafter(e, np.inf), np.nextafter(e, -np.inf)])
    e = np.concatenate([e, -e, [np.nan]])
    x = np.concatenate([e, rng.uniform(-760, 760, 4000), rng.uniform(-2, 2, 4000), np.exp(rng.uniform(-700, 700, 4000))])
    px, py = np.meshgrid(e, e)
    px = np.concatenate([px.ravel(), rng.uniform(0, 3, 8000), np.exp(rng.uniform(-740, 700, 8000))])
    py = np.concatenate([py.ravel(), rng.uniform(-40, 40, 8000), rng.choice([1 / 18, 0.025, 3.0, 4.0, -2.0], 8000)])
    return x, px, py


def _host():
    from brian2_amd import _lib

    L = _lib.lib
    x, px, py = _arguments()
    out = [np.array([f(float(v)) for v in x]) for f in (L.hb_host_exp, L.hb_host_expm1, L.hb_host_log, L.hb_host_exprel)]
    return x, px, py, out + [np.array([L.hb_host_pow(float(a), float(b)) for a, b in zip(px, py)])]


def test_host_functions_at_the_edges():
    x, px, py, (ex, em, lg, er, pw) = _host()

    def close(got, want):
        ok = (got == want) | (np.isnan(got) & np.isnan(want))
        with np.errstate(all="ignore"):
            return ok | (np.abs(got - want) <= np.spacing(np.abs(want)))

    with np.errstate(all="ignore"):
        assert close(ex, np.exp(x)).all() and close(em, np.expm1(x)).all() and close(lg, np.log(x)).all()
        want = np.where(np.abs(x) < 1e-16, 1.0, np.where(x > 717, np.inf, em / x))
        assert close(er, want).all()
        want = np.power(px, py)
        # a negative base, infinite too, has powers of finite whole numbers only, and of nan 0
        want[(px < 0) & ~(np.isfinite(py) & (py == np.floor(py)))] = np.nan
    # (a negative zero's sign is not followed)
    assert close(np.abs(pw), np.abs(want))[px != 0].all() and ((pw < 0) == (want < 0))[px != 0].all()


@pytest.mark.gpu
def test_device_functions_are_the_hosts():
    import torch

    from brian2_amd import _lib
    from brian2_amd.codegen import source_header
    from brian2_amd.runtime import Device

    x, px, py, want = _host()
    src = source_header(256) + """
struct args { const double *x, *px, *py; double *o[5]; int n, m; };
extern "C" __global__ void __launch_bounds__(256) math_edges(const args p) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < p.n) {
        p.o[0][i] = hb_exp(p.x[i]); p.o[1][i] = hb_expm1(p.x[i]); p.o[2][i] = hb_log(p.x[i]); p.o[3][i] = hb_exprel(p.x[i]);
    }
    if (i < p.m) p.o[4][i] = hb_pow(p.px[i], p.py[i]);
}
"""
    D = Device.get()
    fn = D.function(src, "math_edges")
    t = [torch.from_numpy(np.ascontiguousarray(a)).to("cuda") for a in (x, px, py)]
    out = [torch.zeros(len(w), dtype=torch.float64, device="cuda") for w in want]

    class Args(ctypes.Structure):
        _fields_ = [(f"p{i}", ctypes.c_void_p) for i in range(8)] + [("n", ctypes.c_int), ("m", ctypes.c_int)]

    buf = bytes(Args(*[a.data_ptr() for a in t + out], len(x), len(px)))
    _lib.check(_lib.lib.hb_launch(fn, -(-max(len(x), len(px)) // 256), 256, 0, D.stream, buf, len(buf)), "math edges")
    for got, w in zip(out, want):
        got = got.cpu().numpy()
        same = (got.view(np.int64) == w.view(np.int64)) | (np.isnan(got) & np.isnan(w))
        assert same.all()
