"""sin and cos of the device kernels (sxh_sincos_reduced in sx_ops.h): on the
host (the same IEEE operations) against 64-bit-significand arithmetic, on the
GPU against the host's bits through both engines.

Bound, at |r| = pi/4, where it is largest (the sine there lies in [0.5, 1), in
units of its ulp, 2^-53): half for the last subtraction; r^2 is rounded by half
and r^3 by a quarter of a unit, which reach r^3 / 6 as 0.065 and 0.042; the
subtracted r^3 / 6 - ... lies below 1/8 and is rounded by 1/16, its inner terms
add 0.01; the polynomial with rounded coefficients is within 2^-56.5 of the
sine, 0.06.  0.74 in all."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
DRIVER = r"""
#include "sx_ops.h"
extern "C" void run(const double* x, double* s, double* c, long n) {
  for (long i = 0; i < n; ++i) sxh::sxh_sincos_reduced(x[i], s + i, c + i);
}
"""


@pytest.fixture(scope="module")
def reduced(tmp_path_factory):
    d = tmp_path_factory.mktemp("sincos")
    cpp, so = d / "sc.cpp", d / "sc.so"
    cpp.write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-O2", "-mfma", "-ffp-contract=off", "-shared", "-fPIC",
                    "-I", os.path.join(HERE, "..", "casadi_amd", "csrc"), str(cpp), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))

    def run(x):
        x = np.ascontiguousarray(x, np.float64)
        s, c = np.empty_like(x), np.empty_like(x)
        p = lambda a: a.ctypes.data_as(C.c_void_p)
        lib.run(p(x), p(s), p(c), C.c_long(x.size))
        return s, c
    return run


# the arguments nearest to multiples of pi/2, by continued fractions (2^-54 to 2^-60 away)
NEAREST = np.array([float.fromhex(h) for h in ("0x1.921fb54442d18p+0", "0x1.6c6cbc45dc8dep+5", "0x1.6c6cbc45dc8dep+9",
                                               "0x1.39c6fd67805a7p+18", "0x1.9eb7148f354d6p+20", "0x1.b951f1572eba5p+23",
                                               "0x1.b951f1572eba5p+25")])


def _arguments(seed, n=40000):
    rng = np.random.default_rng(seed)
    near = rng.integers(-600000, 600001, n) * 2.0 ** rng.choice([0, 5], n) * (np.pi / 2) * (1 + rng.standard_normal(n) * 2.0 ** rng.integers(-52, -3, n))
    return np.concatenate([rng.uniform(-r, r, n) for r in (0.8, 10.0, 1e3, 3e4, 2.0 ** 20, 2.0 ** 26)] +
                          [near, 10.0 ** rng.uniform(-300, 0, n), [np.pi / 4, np.pi / 2, np.pi, 2.0 ** 20, -2.0 ** 20, 2.0 ** 26, -2.0 ** 26],
                           NEAREST, np.nextafter(NEAREST, 0.0), np.nextafter(NEAREST, np.inf)])


def test_reduced_sincos_error(reduced):
    if np.finfo(np.longdouble).nmant < 63:
        pytest.skip("no extended precision here")
    x = _arguments(3)
    s, c = reduced(x)
    xl = x.astype(np.longdouble)
    for got, ref in ((s, np.sin(xl)), (c, np.cos(xl))):
        ulp = np.spacing(np.abs(ref.astype(np.float64))).astype(np.longdouble)
        err = np.abs(got.astype(np.longdouble) - ref) / ulp
        assert err.max() <= 0.75 and err.mean() <= 0.26


def test_reduced_sincos_zeros(reduced):
    s, c = reduced(np.array([0.0, -0.0, 5e-324, -5e-324, 1e-300]))
    assert np.array_equal(s, [0.0, -0.0, 5e-324, -5e-324, 1e-300]) and not np.signbit(s[0]) and np.signbit(s[1])
    assert np.all(c == 1.0)


@pytest.mark.gpu
def test_device_sincos_has_the_host_bits(cuda, reduced):
    """The pair, either of the two alone and the partials, on both engines;
    past 2^26 and for infinities and NaN the library's values."""
    import torch
    import casadi_amd as ca
    from casadi_amd.hip import HipTape
    x = ca.SX.sym("x")
    fs = {"pair": [ca.sin(x), ca.cos(x)], "sin": [ca.sin(x)], "cos": [ca.cos(x)]}
    v = _arguments(4, 5000)
    hs, hc = reduced(v)
    big = np.array([2.0 ** 26 * 1.5, -1e12, 1e300, np.inf, -np.inf, np.nan])
    X = torch.tensor(np.concatenate([v, big])[None, :], device="cuda")
    one = torch.ones_like(X)
    print(f"[case] sincos n={X.shape[1]}", flush=True)
    for name, ex in fs.items():
        f = ca.Function(name, [x], ex)
        for engine in ("interp", "jit"):
            t = HipTape(f, engine=engine)
            outs = [o.cpu().numpy()[0] for o in t.eval([X])]
            want = {"pair": [hs, hc], "sin": [hs], "cos": [hc]}[name]
            for o, w in zip(outs, want):
                assert np.array_equal(o[:v.size], w), (name, engine)
            for o, w in zip(outs, {"pair": [np.sin, np.cos], "sin": [np.sin], "cos": [np.cos]}[name]):
                with np.errstate(invalid="ignore"):
                    assert np.allclose(o[v.size:], w(big), rtol=0, atol=1e-13, equal_nan=True)
            if len(ex) == 1:
                _, (g,) = t.fwd_adj([X], [one])
                d = hc if name == "sin" else -hs
                assert np.array_equal(g.cpu().numpy()[0, :v.size], d), (name, engine)
