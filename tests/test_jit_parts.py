"""Jacobian and Hessian sweeps over the independent parts of a tape: the
generated kernel on the host at the driver's launch geometry (bounds- and
race-checked, tests/jit_launch_emu.h) against the oracle, and on the GPU
against the whole-tape kernels and the interpreter, bit for bit."""
import ctypes as C
import os
import re
import subprocess

import numpy as np
import pytest

import oracle_ref as O
from test_jit_host_exec import NO_SINCOS_FUSION, CxjArgs, _table

HERE = os.path.dirname(os.path.abspath(__file__))
_MEM = re.compile(r"^#(define|undef) CXJ_(AT|IN|OUT|SEED|SENS|ST_IN|ST_OUT|ADJ_IN|ADJ_OUT|SNAP)\b.*$", re.M)


def _stages(n_stage, irregular=False, aux=False):
    """f: per stage k a nonlinear map of its slice of x and p (Jacobian wanted
    with respect to x); `irregular` takes the slices of x in a shuffled order
    (rows that advance by no fixed step), `aux` adds terms of their own."""
    import casadi_amd as ca
    x, p = ca.SX.sym("x", 3 * n_stage), ca.SX.sym("p", 2 * n_stage)
    order = np.random.default_rng(3).permutation(n_stage) if irregular else np.arange(n_stage)
    out = []
    for k in range(n_stage):
        a, b, c = (x[3 * int(order[k]) + i] for i in range(3))
        u, v = p[2 * k], p[2 * k + 1]
        for _ in range(6):
            a, b, c = ca.sin(a) * u + b / (2.0 + ca.cos(c)), b * c - 1.1 * a, ca.exp(-a * a) + c * v + a / 3.0
        out += [a, b * c]
    if aux:
        out += [x[0], 2.5 * p[0], ca.SX(4.0), x[1] * x[4]]
    return ca.Function("stages", [x, p], [ca.vertcat(*out)])


def _dense(n_part, width):
    """f: per part a map of `width` inputs to as many outputs, each depending on all of them."""
    import casadi_amd as ca
    x = ca.SX.sym("x", n_part * width)
    out = []
    for p in range(n_part):
        v = [x[width * p + i] for i in range(width)]
        h = [ca.sin(v[i]) * v[(i + 1) % width] for i in range(width)]
        s = sum(0.7 * e for e in h)
        out += [ca.cos(s + v[i]) * h[i] + v[i] / 1.1 for i in range(width)]
    return ca.Function("dense", [x], [ca.vertcat(*out)])


def _plan(kind):
    import casadi_amd as ca
    from casadi_amd import workloads as W
    from casadi_amd.hip import HipJacobian
    if kind.startswith("ocp"):
        w, lam, lag = W.quadrotor_ocp_lagrangian(N=int(kind[3:]))
        f = ca.Function("grad_lag", [w, lam], [ca.gradient(lag, w)])
        return f, lambda **k: HipJacobian(f, symmetric=True, first_block=True, **k)
    if kind.startswith("dense"):
        f = _dense(12, int(kind[5:]))
        return f, lambda **k: HipJacobian(f, **k)
    f = _stages(40 if kind == "regular" else 41, kind == "irregular", kind != "regular")
    return f, lambda **k: HipJacobian(f, first_block=True, **k)


def _reference(f, plan, n, args):
    """Values and, per nonzero, the Jacobian from the symbolic derivative."""
    (y,) = O.map_eval(f, n, [a.T for a in args])
    J = f.jacobian()
    blocks = O.map_eval(J, n, [a.T for a in args] + [None])
    sp = J.sparsity_out(0)
    at = {(int(r), int(c)): k for k, (r, c) in enumerate(zip(sp.row, sp.get_col()))}
    pick = [at[(int(r), int(c))] for r, c in zip(plan["jsp"].row, plan["jsp"].get_col())]
    return y.T, blocks[0].T[pick]


@pytest.mark.parametrize("kind,regs,soa32", [("ocp4", "200", False), ("ocp4", "24", False), ("ocp4", "60", True),
                                             ("regular", "200", True), ("irregular", "16", False)])
def test_parts_kernel_on_host(monkeypatch, tmp_path, kind, regs, soa32):
    monkeypatch.setenv("CXH_JIT_TANREGS", regs)
    f, make = _plan(kind)
    h = make(engine="jit")
    src, rows, units, spill = h.parts_source(soa32)
    m = re.search(r"__shared__ double cxj_lds\[(\d+)\];\n", src)
    srows = int(m.group(1)) // 64 if m else spill
    assert regs == "200" or srows > 0          # the small budgets spill: to LDS, or (24) to device memory
    n = 130
    gx = (n + 63) // 64
    src = _MEM.sub("", src)
    src = re.sub(r"__shared__ double cxj_lds\[\d+\];\n", "", src)
    src = re.sub(r"#define CXJ_SPILL_BASE\(u\) .*\n", "#define CXJ_SPILL_BASE(u) (cxj_emu::Ptr<double>(A.spill) + "
                 f"(((long long)blockIdx.y * {gx} + blockIdx.x) * {srows * 64} + threadIdx.x))\n", src)
    for q in ("CXJ_GLOBAL", "CXJ_SPILL"):
        src = src.replace(q + " const double*", "cxj_emu::Ptr<const double>").replace(q + " double*", "cxj_emu::Ptr<double>")
    cpp, so = tmp_path / "parts.cpp", tmp_path / "parts.so"
    cpp.write_text('#include "jit_launch_emu.h"\n#define CXJ_TABLE\n' + src +
                   '\nextern "C" void emu_launch(const CxjArgs* A, unsigned gx, unsigned gy, unsigned bx) '
                   "{\n  CXJ_EMU_LAUNCH_LOOP(cxj_parts(*A));\n}\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", *NO_SINCOS_FUSION, "-shared", "-fPIC", "-w", "-I", HERE,
                    str(cpp), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))
    lib.emu_add_region.argtypes = [C.c_void_p, C.c_longlong, C.c_int]
    lib.emu_errors.restype = C.c_longlong
    rng = np.random.default_rng(9)
    args = [rng.uniform(-1, 1, (f.nnz_in(i), n)) for i in range(2)]
    out, jac = np.full((f.nnz_out(0), n), np.nan), np.full((h.nnz_jac, n), np.nan)
    sp = np.zeros(max(1, units * gx * srows * 64))
    for i, b in enumerate([*args, out, jac, sp]):
        lib.emu_add_region(b.ctypes.data, b.nbytes, i)
    A = CxjArgs()
    A.n, A.lds = n, 64 * gx
    A.arg, A.res, A.asens = _table(args, n), _table([out], n), _table([jac], n)
    A.spill, A.adj_in = sp.ctypes.data, rows.ctypes.data
    lib.emu_launch(C.byref(A), gx, units, 64)
    assert lib.emu_errors() == 0
    y, j = _reference(f, h.plan, n, args)
    assert O.rel_err(out, y) <= 1e-13 and O.rel_err(jac, j) <= 1e-12


def test_tapes_that_do_not_split():
    """One part, or parts with nothing in common: the whole-tape kernels."""
    import casadi_amd as ca
    from casadi_amd import workloads as W
    from casadi_amd.hip import HipJacobian
    assert HipJacobian(W.cartpole_step(), engine="jit").parts_source() is None
    x = ca.SX.sym("x", 8)
    chain = x[0]
    for k in range(400):
        chain = ca.sin(chain) * x[k % 8] + 0.25 * k
    assert HipJacobian(ca.Function("chain", [x], [ca.vertcat(*[chain * x[i] for i in range(8)])]), engine="jit").parts_source() is None


def _chains(ops, n_part=3, n_param=40):
    """n_part chains of `ops` operations on a differentiated input and n_param parameters each."""
    import casadi_amd as ca
    x, p = ca.SX.sym("x", n_part), ca.SX.sym("p", n_part * n_param)
    out = []
    for k in range(n_part):
        c = x[k]
        for i in range(ops):
            c = ca.sin(c) if i % 2 == 0 else c * p[n_param * k + (i // 2) % n_param]
        out.append(c)
    return ca.Function("chains", [x, p], [ca.vertcat(*out)])


def test_longest_part_counts_its_inputs():
    """A part's program loads 41 inputs and stores one output beside its
    operations: 4096 instructions are one kernel, 4097 leave the whole-tape
    kernels to serve the call."""
    from casadi_amd.hip import HipJacobian
    plan = lambda ops: HipJacobian(_chains(ops), first_block=True, engine="jit")
    assert plan(4096 - 42).parts_source() is not None
    assert plan(4097 - 42).parts_source() is None


def test_direction_groups_hold_at_most_64(monkeypatch):
    """A group's directions are bits of a 64-bit mask, whatever the setting asks for."""
    import casadi_amd as ca
    from casadi_amd.hip import HipJacobian
    monkeypatch.setenv("CXH_JIT_DIRGROUP", "80")
    x = ca.SX.sym("x", 3 * 80)
    out = []
    for k in range(3):
        s = sum(ca.sin(x[80 * k + i]) * x[80 * k + (i + 1) % 80] for i in range(80))
        out += [s * x[80 * k + i % 80] for i in range(90)]
    h = HipJacobian(ca.Function("wide", [x], [ca.vertcat(*out)]), engine="jit")
    src, _, units, _ = h.parts_source()
    groups = len(re.findall(r"case \d+: cxj_body_c\d+_g\d+", src))
    assert h.plan["ndir"] == 80 and groups == 2 and units == 3 * groups


def test_an_output_written_twice_keeps_the_order():
    """The last of several writes to one output nonzero counts; parts run in no
    order, so such a tape stays whole."""
    from casadi_amd.hip import HipJacobian, HipTape
    from casadi_amd.ops import OP
    f = _chains(600)
    prog = np.array(f.instructions())
    tape = lambda p: HipTape.nested(p, int(p["i0"].max()) + 1, [3, 120], [3], [], engine="jit")
    assert HipJacobian(f, tape=tape(prog), first_block=True).parts_source() is not None
    outs = np.flatnonzero(prog["op"] == OP.OUTPUT)
    prog["i2"][outs[-1]] = prog["i2"][outs[0]]
    assert HipJacobian(f, tape=tape(prog), first_block=True).parts_source() is None


@pytest.mark.parametrize("size", ["5", "12"])
def test_larger_direction_groups_on_host(monkeypatch, tmp_path, size):
    """The group sizes that larger batches run, through the setting."""
    monkeypatch.setenv("CXH_JIT_DIRGROUP", size)
    test_parts_kernel_on_host(monkeypatch, tmp_path, "ocp4", "200", True)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2000, 5000, 20001])
def test_group_sizes_keep_the_bits(cuda, monkeypatch, n):
    """Batches of 12 parts dense in 14 directions that take groups of 3, of 5 and
    (past the number of wavefronts that fills the device) of all 14."""
    import torch
    f, make = _plan("dense14")
    x = torch.tensor(np.random.default_rng(n).uniform(-1, 1, (f.nnz_in(0), n)), device="cuda")
    print(f"[case] parts groups n={n}", flush=True)
    h = make(engine="jit")
    assert h.parts_source() is not None
    (y,), j = h([x])
    (yi,), ji = make()([x])
    assert torch.equal(y, yi) and torch.equal(j, ji)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n", [("ocp2", 1), ("ocp4", 65), ("ocp4", 1001), ("regular", 63), ("irregular", 200)])
def test_parts_keep_the_bits(cuda, monkeypatch, kind, n):
    import torch
    f, make = _plan(kind)
    rng = np.random.default_rng(n)
    args = [torch.tensor(rng.uniform(-1, 1, (f.nnz_in(i), n)), device="cuda") for i in range(2)]
    print(f"[case] parts {kind} n={n}", flush=True)
    h = make(engine="jit")
    (y,), j = h(args)
    assert kind == "ocp2" or h.parts_source() is not None
    (yi,), ji = make()(args)
    monkeypatch.setenv("CXH_JIT_PARTS", "0")
    (yw,), jw = make(engine="jit")(args)
    for a, b in ((y, yi), (j, ji), (y, yw), (j, jw)):
        assert torch.equal(a, b)
    monkeypatch.delenv("CXH_JIT_PARTS")
    for regs in ("24", "60"):                   # spill rows in device memory, in LDS
        monkeypatch.setenv("CXH_JIT_TANREGS", regs)
        (ys,), js = make(engine="jit")(args)
        assert torch.equal(ys, y) and torch.equal(js, j)
    monkeypatch.delenv("CXH_JIT_TANREGS")
    none, jo = make(engine="jit")(args, res=False)   # no outputs; an absent second input reads zeros
    assert none == [None] and torch.equal(jo, j)
    zeros = [args[0], torch.zeros_like(args[1])]
    assert torch.equal(h([args[0], None])[1], h(zeros)[1])


@pytest.mark.gpu
def test_parts_spill_memory_is_bounded(cuda, monkeypatch):
    """Spill rows of a batch that would need more than half a GiB: several
    launches over slices of the batch, the same bits."""
    import torch
    f, make = _plan("ocp4")
    n = 40001
    args = [torch.tensor(np.random.default_rng(n).uniform(-1, 1, (f.nnz_in(i), n)), device="cuda") for i in range(2)]
    print(f"[case] parts spill n={n}", flush=True)
    (y,), j = make(engine="jit")(args)
    monkeypatch.setenv("CXH_JIT_TANREGS", "24")
    h = make(engine="jit")
    _, _, units, spill = h.parts_source()
    assert units * spill * n * 8 > 2 << 29
    y2, j2 = torch.empty_like(y), torch.empty_like(j)   # leaves torch two blocks of the results' sizes
    del y2, j2
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    (ys,), js = h(args)
    torch.cuda.synchronize()
    assert before - torch.cuda.mem_get_info()[0] < 600 << 20
    assert torch.equal(ys, y) and torch.equal(js, j)
