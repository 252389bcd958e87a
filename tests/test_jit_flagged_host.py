"""The flagged straight-line bodies on the host: divisions by constants in two
operations and sin/cos without a branch, every store held back, and the whole
instance evaluated again exactly where an operand lies outside their ranges.
Single-segment forward, reverse and batch bodies, bit for bit against the
oracle, with outputs placed over inputs and sensitivities over seeds."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import oracle_ref as O
from test_jit_host_exec import NO_SINCOS_FUSION, CxjArgs, _table

QUALIFIERS = ("#define __device__\n#define __forceinline__ inline\n#define CXJ_KEEP(x) ((void)0)\n"
              "#define CXJ_KEEP_PTR(x) ((void)0)\n#define CXJ_AFTER(p, x) ((void)0)\n#define CXJ_GLOBAL\n"
              "#define CXJ_OPAQUE(p) ((void)0)\n#define CXJ_OPAQUE_AFTER(p, x) ((void)0)\n#define CXJ_ANY(b) (b)\n"
              "static long long cxj_reruns = 0;\n")


def _build(src, name, tmp):
    """run(args, n) of body `name`, returning how many instances ran again."""
    again = f"    {name}_x(A, k2);\n"
    assert src.count(again) == 1 and "sxh::sxh_div_c(" in src
    src = src[:src.index('extern "C" __global__')].replace(again, "    ++cxj_reruns;\n" + again)
    cpp, so = tmp / f"{name}.cpp", tmp / f"{name}.so"
    cpp.write_text(QUALIFIERS + src + 'extern "C" long long run(const CxjArgs* A, long long n) {\n  cxj_reruns = 0;\n'
                   f"  for (long long k = 0; k < n; ++k) {name}(*A, k);\n  return cxj_reruns;\n}}\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-mfma", "-ffp-contract=off", *NO_SINCOS_FUSION, "-shared", "-fPIC", "-w",
                    str(cpp), "-o", str(so)], check=True)
    run = C.CDLL(str(so)).run
    run.argtypes, run.restype = [C.POINTER(CxjArgs), C.c_longlong], C.c_longlong
    return run


def _states(n, seed):
    """Cart-pole states and forces; of every ten instances one has angles past
    2^26, one a speed whose tenth is below 2^-900 (and a zero angle)."""
    rng = np.random.default_rng(seed)
    x, u = rng.uniform(-1, 1, (4, n)), rng.uniform(-10, 10, (1, n))
    x[:, 3::10] = np.copysign(2e8, x[:, 3::10])
    x[:, 7::10] *= 1e-300
    u[:, 7::10] *= 1e-300
    return x, u, np.isin(np.arange(n) % 10, (3, 7))


def _args(n, **tables):
    A = CxjArgs()
    A.n, A.lds = n, n
    for k, v in tables.items():
        setattr(A, k, _table(v, n))
    return A


@pytest.mark.parametrize("form", ["fwd", "rev", "batch"])
@pytest.mark.parametrize("in_place", [False, True])
def test_flagged_bodies(tmp_path, form, in_place):
    from casadi_amd import workloads as W
    from casadi_amd.hip import HipTape, batch_source
    f = W.cartpole_step()
    tape = HipTape(f, engine="jit")
    src = batch_source([tape]) if form == "batch" else tape.jit_source(reverse=form == "rev")[0]
    run = _build(src, "cxj_f0" if form == "batch" else "cxj_body", tmp_path)
    n = 60
    x, u, flagged = _states(n, 5)
    seed = np.random.default_rng(6).standard_normal((4, n))
    (y,), (gx, gu) = O.adj_map(f, n, [x.T, u.T], [seed.T])
    x, u = x.copy(), u.copy()
    out = x if in_place else np.zeros((4, n))
    if form == "fwd":
        again = run(C.byref(_args(n, arg=[x, u], res=[out])), n)
    else:
        hx, hu = (seed, u) if in_place else (np.zeros((4, n)), np.zeros((1, n)))
        again = run(C.byref(_args(n, arg=[x, u], res=[out], aseed=[seed], asens=[hx, hu])), n)
        assert np.array_equal(hx, gx.T) and np.array_equal(hu, gu.T)
    assert np.array_equal(out, y.T)
    assert again == flagged.sum()
