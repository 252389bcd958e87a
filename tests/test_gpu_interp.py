"""The interpreter's evaluation and adjoint on random programs whose
instructions overwrite their own operands, take one slot twice and end in
partly filled chunks of 64: the bits of the specialised kernels, which are
generated from the same tape without its re-encoding (equal zeros may differ in
sign, NaN where NaN)."""
import numpy as np
import pytest

from conftest import seed_of

pytestmark = pytest.mark.gpu
ASSIGN, ADD, SUB, MUL, DIV, NEG, SQRT, SQ, TWICE, SIN, COS = 0, 1, 2, 3, 4, 5, 10, 11, 12, 13, 14
LT, FABS, IF_ELSE_ZERO, FMIN, FMAX, ATAN2, CONST, INPUT, OUTPUT = 19, 29, 32, 34, 35, 43, 44, 45, 46
BINARY = [ADD, SUB, MUL, DIV, LT, IF_ELSE_ZERO, FMIN, FMAX, ATAN2]
UNARY = [ASSIGN, NEG, SQ, TWICE, SIN, COS, FABS]


def _program(rng, length, ws):
    from casadi_amd.function import INSTR_DTYPE
    a = np.zeros(length, INSTR_DTYPE)
    for k in range(length):
        i0, i1, i2 = rng.integers(0, ws, 3)
        if k < ws:                      # every slot defined first
            op, i0 = (INPUT, k) if k < 5 else (CONST, k)
        else:
            op = int(rng.choice([ADD, SUB, MUL, SUB, MUL] + BINARY + UNARY + [CONST, INPUT, OUTPUT]))
            if rng.random() < 0.3:
                i1 = i0
            if rng.random() < 0.3:
                i2 = i1
        if k >= length - 3:
            op = OUTPUT
        a["op"][k], a["i0"][k] = op, i0
        if op == CONST:
            a["i1"][k], a["i2"][k] = np.array([rng.choice([0.0, -0.0, 1.5, -0.75, 1e-300])]).view(np.int32)
        elif op == INPUT:
            a["i1"][k], a["i2"][k] = 0, k if k < 5 else rng.integers(0, 5)
        elif op == OUTPUT:
            a["i0"][k], a["i1"][k], a["i2"][k] = 0, i1, rng.integers(0, 4) if k < length - 3 else length - 1 - k
        else:
            a["i1"][k], a["i2"][k] = i1, i2 if op in BINARY else i1
    return a


@pytest.mark.parametrize("length, ws, every, ipw, lds", [
    (70, 9, 0, 64, True), (64, 5, 0, 64, True), (129, 12, 64, 16, True), (300, 20, 37, 64, True), (300, 20, 100, 8, False)])
def test_random_programs_match_the_specialised_kernels(cuda, length, ws, every, ipw, lds):
    import torch
    from casadi_amd.hip import HipTape
    rng = np.random.default_rng(seed_of(length + every) + ws)
    for rep in range(3):
        prog = _program(rng, length, ws)
        n = 193
        x = rng.standard_normal((5, n)) * 0.5
        x[:, 7] = [0.0, -0.0, np.inf, np.nan, 1.0]
        X, S = torch.tensor(x, device="cuda"), torch.tensor(rng.standard_normal((4, n)), device="cuda")
        got = {}
        for engine in ("interp", "jit"):
            t = HipTape.nested(prog, ws, [5], [4], [], engine=engine, w_in_lds=lds)
            if engine == "interp":
                t.config(ipw=ipw)
            print(f"[case] {engine} length {length} every {every} rep {rep}", flush=True)
            y = [torch.zeros(4, n, dtype=torch.float64, device="cuda")]
            t.eval([X], n, out=y)
            # the specialised sweep in one segment: across segments it hands zero adjoints of dead values on
            o, g = t.fwd_adj([X], [S], n, checkpoint_every=every if engine == "interp" else 0)
            written = sorted({int(i) for i in prog["i2"][prog["op"] == OUTPUT]})
            got[engine] = [y[0].cpu().numpy(), o[0].cpu().numpy()[written], g[0].cpu().numpy()]
        for a, b in zip(got["interp"], got["jit"]):
            assert np.array_equal(a, b, equal_nan=True)
