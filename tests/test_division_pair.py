"""Division by a constant in two operations, q = RN(x yh + RN(x yl)), which the
specialised kernels take for the divisors that the generator has checked
(div_pair in jit.hip): the correctly rounded quotient, so every comparison is
bit for bit with IEEE division."""
import ctypes as C
import os
import random
import re
import subprocess

import numpy as np
import pytest

import casadi_amd as ca
from casadi_amd.hip import HipTape, jit_compile_check
from test_division import DIVISORS, near_midpoint_dividends

HERE = os.path.dirname(os.path.abspath(__file__))
SPECIAL = [0.0, -0.0, np.inf, -np.inf, np.nan, 5e-324, -5e-324, 1e-310, 2.0 ** -1022, 2.0 ** -901, -2.0 ** -900,
           1.7976931348623157e308, -1.7976931348623157e308, 3.0, -1.1]


def _quotients(divisors):
    x = ca.SX.sym("x", len(divisors))
    return ca.Function("q", [x], [ca.vertcat(*[x[i] / c for i, c in enumerate(divisors)])])


def _pairs(divisors):
    """The (c, yh, yl) that the generated source divides by in two operations."""
    src = HipTape(_quotients(divisors), engine="jit").jit_source()[0]
    num = r"(-?0x[0-9a-f.]+p[+-]\d+)"
    return [tuple(map(float.fromhex, m)) for m in re.findall(rf"sxh_div_c\(v\d+, {num}, {num}, {num}, wide\)", src)]


def test_accepted_divisors_round_correctly(tmp_path):
    rng = random.Random(11)
    some = [np.ldexp(1 + rng.getrandbits(52) * 2.0 ** -52, rng.randrange(-64, 64)) for _ in range(44)]
    divs = [c for c in DIVISORS if abs(np.frexp(c)[0]) != 0.5] + some
    pairs = [p for i in range(0, len(divs), 20) for p in _pairs(divs[i:i + 20])]
    assert len(divs) * 0.8 < len(pairs) < len(divs)     # most, and not all (one in fourteen is refused)
    cpp, so = tmp_path / "q.cpp", tmp_path / "q.so"
    cpp.write_text('#include "sx_ops.h"\nextern "C" int run(const double* x, double c, double h, double l, double* q, long n)'
                   "{ bool w = false; for (long i = 0; i < n; ++i) q[i] = sxh::sxh_div_c(x[i], c, h, l, w); return w; }\n")
    subprocess.run(["g++", "-std=c++17", "-O2", "-mfma", "-ffp-contract=off", "-shared", "-fPIC", "-I",
                    os.path.join(HERE, "..", "casadi_amd", "csrc"), str(cpp), "-o", str(so)], check=True)
    run = C.CDLL(str(so)).run
    run.argtypes = [C.c_void_p, C.c_double, C.c_double, C.c_double, C.c_void_p, C.c_long]
    def quotient(x, p):
        q = np.empty_like(x)
        return q, run(x.ctypes.data, *p, q.ctypes.data, x.size)
    for p in pairs:
        m = np.ldexp(1 + np.random.default_rng(3).integers(0, 2 ** 52, 20000) * 2.0 ** -52, 0)
        x = np.concatenate([near_midpoint_dividends(p[0], 2000, rng), m, -m * 2.0 ** 900, m * 2.0 ** -899, SPECIAL[:5],
                            SPECIAL[10:]])
        q, wide = quotient(x, p)
        with np.errstate(all="ignore"):
            assert np.array_equal(q.view(np.int64), (x / p[0]).view(np.int64)) and not wide
        assert all(quotient(np.array([t]), p)[1] for t in SPECIAL[5:10])


def test_refused_and_unlimited_forms():
    """A refused divisor keeps the corrected reciprocal; powers of two, more
    outputs than a body holds back and the switch keep IEEE division."""
    src = HipTape(_quotients([1.7]), engine="jit").jit_source()[0]
    assert "sxh_div_c(v0, 0x1.b333333333333p+0, 0x" in src and not _pairs([1.7])
    jit_compile_check(src)
    call = "= sxh::sxh_div_c("
    assert call not in HipTape(_quotients([2.0, -0.25]), engine="jit").jit_source()[0]
    assert call in HipTape(_quotients([3.0] * 8), engine="jit").jit_source(reverse=True)[0]
    assert call not in HipTape(_quotients([3.0] * 9), engine="jit").jit_source(reverse=True)[0]
    assert call not in HipTape(_quotients([3.0] * 33), engine="jit").jit_source()[0]


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 63, 1000])
def test_device_quotients_special_dividends(cuda, n):
    """Evaluation (also in place and on strided columns), the reverse sweep and
    a batch: special dividends in some wavefronts and not in others."""
    import torch
    from casadi_amd.hip import HipBatch
    divs = [1.1, -3.0, 0.3, 1.7, 9.81]
    x = ca.SX.sym("x", 5)
    f = ca.Function("f", [x], [ca.vertcat(*[x[i] / c for i, c in enumerate(divs)])])
    g = ca.Function("g", [x], [ca.sumsqr(ca.sin(ca.vertcat(*[x[i] / c for i, c in enumerate(divs)])))])
    rng = np.random.default_rng(n)
    v = rng.standard_normal((5, n)) * 10.0 ** rng.integers(-5, 5, (5, n))
    for k in range(0, n, 130):
        v[rng.integers(0, 5), k] = SPECIAL[(k // 130) % len(SPECIAL)]
    X = torch.tensor(v, device="cuda")
    with np.errstate(all="ignore"):
        ref = v / np.array(divs)[:, None]
    t = HipTape(f, engine="jit")
    same = lambda a, b: np.array_equal(a, b, equal_nan=True) and np.array_equal(np.signbit(a)[~np.isnan(b)],
                                                                                np.signbit(b)[~np.isnan(b)])
    assert same(t.eval([X], n)[0].cpu().numpy(), ref)
    wide = torch.zeros(5, n + 7, dtype=torch.float64, device="cuda")
    wide[:, :n] = X
    out = torch.empty_like(wide)[:, :n]
    assert same(t.eval([wide[:, :n]], n, out=[out])[0].cpu().numpy(), ref)
    Y = X.clone()
    assert same(t.eval([Y], n, out=[Y])[0].cpu().numpy(), ref)
    S = torch.tensor(rng.standard_normal((1, n)), device="cuda")
    (o,), (a,) = HipTape(g, engine="jit").fwd_adj([X], [S], n)
    (oi,), (ai,) = HipTape(g, engine="interp").fwd_adj([X], [S], n)
    # the sign of a zero adjoint is left open between the engines
    assert same(o.cpu().numpy(), oi.cpu().numpy()) and np.array_equal(a.cpu().numpy(), ai.cpu().numpy(), equal_nan=True)
    b = HipBatch([g, g], [n, n])
    bound = [b.bind(i, [X], [S]) for i in range(2)]
    b.launch()
    for (ob,), (ab,) in bound:
        assert same(ob.cpu().numpy(), o.cpu().numpy()) and same(ab.cpu().numpy(), a.cpu().numpy())
