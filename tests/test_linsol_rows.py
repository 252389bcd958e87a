"""The sixteen-lanes-per-instance LDL / QR programs: on the host, lane by lane
(tests/rows_emu.h), against the oracle's casadi_ldl / casadi_qr bit for bit
with every access checked; on the GPU against the generic kernel's bits."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import oracle_ref as O

HERE = os.path.dirname(os.path.abspath(__file__))


class RowsArgs(C.Structure):
    _fields_ = [(k, C.c_void_p) for k in ("a", "x", "f", "d", "z", "w", "tab", "status")] + \
        [("a_t", C.c_longlong), ("x_t", C.c_longlong)] + \
        [(k, C.c_uint) for k in ("a_s", "x_s", "ld", "w_t")] + [("eps", C.c_double), ("n", C.c_longlong)]


class Host:
    """A program compiled for the host and the buffers it may touch."""

    def __init__(self, source, tab, tmp):
        cpp, so = os.path.join(tmp, "rows.cpp"), os.path.join(tmp, "rows.so")
        with open(cpp, "w") as fh:
            fh.write('#include "rows_emu.h"\n' + source +
                     '\nextern "C" void rows_run(const CxrArgs* A) { for (long long i = 0; i < A->n; ++i) cxr_body(*A, i); }\n')
        subprocess.run(["g++", "-std=c++17", "-O0", "-ffp-contract=off", "-shared", "-fPIC", "-w", "-I", HERE, cpp, "-o", so],
                       check=True)
        self.lib = C.CDLL(so)
        self.lib.rows_errors.restype = C.c_longlong
        self.lib.rows_region.argtypes = [C.c_void_p, C.c_longlong]
        self.tab = np.ascontiguousarray(tab, np.int32)

    def run(self, n, layout="soa", ld=64, eps=0.0, status=None, **buf):
        A = RowsArgs()
        self.lib.rows_clear()
        for k, b in buf.items():
            setattr(A, k, b.ctypes.data)
            self.lib.rows_region(b.ctypes.data, b.nbytes)
        for k in ("a", "x"):
            if k in buf:
                m = buf[k].size // n
                setattr(A, k + "_s", 8 * (n if layout == "soa" else 1))
                setattr(A, k + "_t", 8 * (1 if layout == "soa" else m))
        if "w" in buf:
            A.w_t = buf["w"].nbytes // n
        A.ld, A.eps, A.n, A.tab = 8 * ld, eps, n, self.tab.ctypes.data
        A.status = None if status is None else status.ctypes.data
        self.lib.rows_run(C.byref(A))
        return self.lib.rows_errors()


def _pattern(kind):
    """A symmetric pattern and the AMD switch."""
    from casadi_amd import workloads as W
    from casadi_amd.sx import Sparsity
    if kind == "kkt":
        return W.ocp_kkt_sparsity(N=5)[0]
    if kind == "kkt63":                 # fifteen rows of L active at once; too wide for the QR
        return W.ocp_kkt_sparsity(3, 6, 3)[0]
    if kind == "diagonal":
        return Sparsity.triplet(5, 5, np.arange(5), np.arange(5))
    if kind == "one":
        return Sparsity.triplet(1, 1, [0], [0])
    if kind == "dense16":               # sixteen rows: the widest LDL
        r, c = np.divmod(np.arange(256), 16)
        return Sparsity.triplet(16, 16, r, c)
    if kind == "arrow":
        i = np.arange(1, 14)
        z = np.zeros(13, int)
        d = np.arange(14)
        return Sparsity.triplet(14, 14, np.concatenate([d, i, z]), np.concatenate([d, z, i]))
    rng = np.random.default_rng(5)      # random, some diagonal entries missing
    n = 30
    r, c = rng.integers(0, n, 26), rng.integers(0, n, 26)
    d = np.arange(0, n, 1 if kind == "random" else 3)
    return Sparsity.triplet(n, n, np.concatenate([d, r, c]), np.concatenate([d, c, r]))


def _values(sp, n, seed):
    """Symmetric values: random, one instance all zero, one with an infinity and a NaN."""
    rng = np.random.default_rng(seed)
    row, col = np.asarray(sp.row), np.asarray(sp.get_col())
    at = {(int(r), int(c)): k for k, (r, c) in enumerate(zip(row, col))}
    a = rng.standard_normal((sp.nnz(), n))
    a[row == col] += 4.0
    for (r, c), k in at.items():
        if r > c:
            a[k] = a[at[(c, r)]]
    a[:, n - 1] = 0.0
    a[0, n - 2] = np.inf
    a[sp.nnz() // 2, n - 3] = np.nan
    return a


KINDS = ["kkt", "kkt63", "diagonal", "one", "dense16", "arrow", "random", "gaps"]


@pytest.mark.parametrize("kind,opts,layout", [(k, {}, "soa") for k in KINDS] + [
    ("kkt", {}, "aos"), ("random", {"amd": False}, "aos"), ("arrow", {"amd": False}, "soa"),
    ("kkt", {"incomplete": True}, "soa"), ("random", {"incomplete": True, "amd": False}, "soa")])
def test_ldl_rows_on_host(tmp_path, kind, opts, layout):
    from casadi_amd.linsol import Linsol
    sp = _pattern(kind)
    ls = Linsol("l", "ldl", sp, opts)
    prog = ls.rows_source(0)
    if prog is None:
        pytest.skip("the pattern does not fit sixteen lanes")
    nn, n, ltc = sp.size1(), 6, ls.sp_lt.compressed()
    nlt = ls.sp_lt.nnz()
    a = _values(sp, n, 3)
    b = np.random.default_rng(4).standard_normal((nn, n))
    lay = (lambda m: np.ascontiguousarray(m)) if layout == "soa" else (lambda m: np.ascontiguousarray(m.T))
    back = (lambda m: m) if layout == "soa" else (lambda m: m.T)
    ld = 64
    new = lambda rows: np.zeros((max(rows, 1), ld))
    x, st = lay(b).copy(), np.full(n, -1, np.int32)
    (tmp_path / "a").mkdir(), (tmp_path / "b").mkdir(), (tmp_path / "c").mkdir()
    assert Host(*prog, str(tmp_path / "a")).run(n, layout, ld, status=st, a=lay(a), x=x, w=np.zeros((n, nlt + nn))) == 0
    f, d, st2 = new(nlt), new(nn), np.full(n, -1, np.int32)
    assert Host(*ls.rows_source(1), str(tmp_path / "b")).run(n, layout, ld, status=st2, a=lay(a), f=f, d=d) == 0
    x2 = lay(b).copy()
    assert Host(*ls.rows_source(2), str(tmp_path / "c")).run(n, layout, ld, x=x2, f=f, d=d, w=np.zeros((n, nlt + nn))) == 0
    for k in range(n):
        with np.errstate(all="ignore"):
            lt, dd = O.ldl(sp.compressed(), a[:, k], ltc, ls.p)
            xr = O.ldl_solve(b[:, k], ltc, lt, dd, ls.p)
        bad = int(np.sum(~((dd != 0) & np.isfinite(dd))))
        assert np.array_equal(f[:nlt, k], lt, equal_nan=True) and np.array_equal(d[:, k], dd, equal_nan=True), k
        assert np.array_equal(back(x)[:, k], xr, equal_nan=True) and np.array_equal(back(x2)[:, k], xr, equal_nan=True), k
        assert np.array_equal(np.signbit(back(x)[:, k][xr == 0]), np.signbit(xr[xr == 0])), k
        assert st[k] == st2[k] == bad


@pytest.mark.parametrize("kind,amd,layout", [(k, True, "soa") for k in KINDS] + [
    ("kkt", True, "aos"), ("random", False, "aos"), ("arrow", False, "soa")])
def test_qr_rows_on_host(tmp_path, kind, amd, layout):
    from casadi_amd.linsol import Linsol
    sp = _pattern(kind)
    ls = Linsol("q", "qr", sp, {"amd": amd})
    svc, src = ls.sp_v.compressed(), ls.sp_r.compressed()
    nn, n, ld = sp.size1(), 6, 64
    a = _values(sp, n, 7)
    b = np.random.default_rng(8).standard_normal((nn, n))
    lay = (lambda m: np.ascontiguousarray(m)) if layout == "soa" else (lambda m: np.ascontiguousarray(m.T))
    back = (lambda m: m) if layout == "soa" else (lambda m: m.T)
    fused, fact = ls.rows_source(0), ls.rows_source(1)
    if fact is None:
        assert fused is None
        pytest.skip("the pattern does not fit sixteen lanes")
    nr, nv = ls.sp_r.nnz(), ls.sp_v.nnz()
    new = lambda rows: np.zeros((max(rows, 1), ld))
    (tmp_path / "a").mkdir(), (tmp_path / "b").mkdir()
    x, st, st2 = lay(b).copy(), np.full(n, -1, np.int32), np.full(n, -1, np.int32)
    if fused is not None:
        assert Host(*fused, str(tmp_path / "a")).run(n, layout, ld, ls.eps, st, a=lay(a), x=x, w=np.zeros((n, nr + nn))) == 0
    z, f, d = new(nv), new(nr), new(nn)
    assert Host(*fact, str(tmp_path / "b")).run(n, layout, ld, ls.eps, st2, a=lay(a), f=f, d=d, z=z) == 0
    for k in range(n):
        with np.errstate(all="ignore"):
            v, r, beta = O.qr(sp.compressed(), a[:, k], svc, src, ls.prinv, ls.pc)
            xr = O.qr_solve(b[:, k], 0, svc, v, src, r, beta, ls.prinv, ls.pc)
        for got, ref in ((z[:nv, k], v), (f[:nr, k], r), (d[:, k], beta)):
            assert np.array_equal(got, ref, equal_nan=True), k
        diag = r[np.asarray(ls.sp_r.colind)[1:] - 1]
        assert st2[k] == int(np.sum(~(np.abs(diag) >= ls.eps))), k
        if fused is not None:
            assert np.array_equal(back(x)[:, k], xr, equal_nan=True) and st[k] == st2[k], k


def test_wide_patterns_keep_the_one_lane_program():
    """More than sixteen active rows or columns: no sixteen-lane program."""
    from casadi_amd import workloads as W
    from casadi_amd.linsol import Linsol
    from casadi_amd.sx import Sparsity
    r, c = np.divmod(np.arange(17 * 17), 17)
    dense = Sparsity.triplet(17, 17, r, c)
    assert all(Linsol("l", "ldl", dense).rows_source(p) is None for p in (0, 1))
    assert all(Linsol("q", "qr", dense).rows_source(p) is None for p in (0, 1))
    assert Linsol("q", "qr", W.ocp_kkt_sparsity(3, 6, 3)[0]).rows_source(0) is None


def test_batch_limit_follows_the_width():
    """A pattern whose pivots hold few values leaves the sixteen lanes at a
    smaller batch: 4096 instances per value, all 32768 from 6 (LDL) or 8 (QR)
    values, the LDL's solve alone at most 12288."""
    from casadi_amd import workloads as W
    from casadi_amd.linsol import Linsol
    from casadi_amd.sx import Sparsity
    i = np.arange(39)
    d = np.arange(40)
    tri = Sparsity.triplet(40, 40, np.concatenate([d, i, i + 1]), np.concatenate([d, i + 1, i]))
    kkt = W.ocp_kkt_sparsity(30)[0]
    limit = lambda solver, sp, part: int(Linsol("l", solver, sp, {"amd": sp is kkt}).rows_source(part)[0].split("\n")[0].split()[-1])
    assert [limit("ldl", tri, p) for p in (0, 1, 2)] == [4096 * 79 // 40] * 3
    assert [limit("qr", tri, p) for p in (0, 1)] == [4096 * (3 * 40 - 3 + 40) // 40] * 2
    assert [limit("ldl", kkt, p) for p in (0, 1, 2)] == [32768, 32768, 12288]
    assert [limit("qr", kkt, p) for p in (0, 1)] == [32768, 32768]


@pytest.mark.gpu
@pytest.mark.parametrize("solver", ["ldl", "qr"])
@pytest.mark.parametrize("n_inst", [1, 15, 16, 17, 63, 65, 1000])
def test_rows_programs_match_the_generic_kernel(cuda, monkeypatch, solver, n_inst):
    import torch
    from casadi_amd import workloads as W
    from casadi_amd.linsol import Linsol
    sp, a = W.ocp_kkt_batch(np.random.default_rng(n_inst), n_inst, 5)
    if n_inst > 2:
        a[:, 2] = 0.0
    A = torch.tensor(a, device="cuda")
    B = torch.tensor(np.random.default_rng(1).standard_normal((sp.size1(), n_inst)), device="cuda")
    print(f"[case] rows {solver} instances={n_inst}", flush=True)
    rows, gen = Linsol("j", solver, sp), Linsol("i", solver, sp, {"engine": "interp"})
    assert rows.rows_source(0) is not None
    (xr, sr), (xg, sg) = rows.solve_batch(A, B), gen.solve_batch(A, B)
    assert torch.equal(sr, sg) and np.array_equal(xr.cpu().numpy(), xg.cpu().numpy(), equal_nan=True)
    if n_inst <= 2 or solver == "ldl":
        for s in (rows, gen):
            s.nfact(A)
        for rhs in (B, B * 2.0):
            assert np.array_equal(rows.solve(rhs).cpu().numpy(), gen.solve(rhs).cpu().numpy(), equal_nan=True)
    # and the one-lane programs, which larger batches run
    monkeypatch.setenv("CXH_LINSOL_ROWS_MAX", "0")
    xo, so = Linsol("o", solver, sp).solve_batch(A, B)
    assert torch.equal(so, sr) and np.array_equal(xo.cpu().numpy(), xr.cpu().numpy(), equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize("solver", ["ldl", "qr"])
def test_one_lane_programs_match_the_generic_kernel(cuda, monkeypatch, solver):
    """The horizon-30 system through the programs that batches above the
    sixteen-lane limit run (several segments for the QR): fused, factor alone
    and solve alone."""
    import torch
    from casadi_amd import workloads as W
    from casadi_amd.linsol import Linsol
    monkeypatch.setenv("CXH_LINSOL_ROWS_MAX", "0")
    n_inst = 193
    sp, a = W.ocp_kkt_batch(np.random.default_rng(30), n_inst, 30)
    A = torch.tensor(a, device="cuda")
    B = torch.tensor(np.random.default_rng(31).standard_normal((sp.size1(), n_inst)), device="cuda")
    one, gen = Linsol("o", solver, sp), Linsol("i", solver, sp, {"engine": "interp"})
    for s in (one, gen):
        s.nfact(A)
    print(f"[case] one-lane {solver} factor", flush=True)
    assert torch.equal(one.solve(B), gen.solve(B))
    print(f"[case] one-lane {solver} solve", flush=True)
    for name in ("l", "again"):
        (x, st), (xg, sg) = one.solve_batch(A, B), gen.solve_batch(A, B)
        assert torch.equal(x, xg) and torch.equal(st, sg), name
