"""A map on host arrays whose blocks are dense columns goes to the device as it
is: the bits of the instance-major path, for every form an argument may take."""
import numpy as np
import pytest

import casadi_amd as ca
from casadi_amd.map import MapFunction

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 1000])
@pytest.mark.parametrize("engine", ["jit", "interp"])
def test_dense_columns_match_the_instance_major_path(cuda, n, engine):
    x, u = ca.SX.sym("x", 3), ca.SX.sym("u")
    f = ca.Function("f", [x, u], [ca.vertcat(x[0] * u / 1.1, ca.sin(x[1]) + u), x[2] - u])
    m = MapFunction(f, n, "hip", opts={"engine": engine})
    rng = np.random.default_rng(n)
    X, U = rng.standard_normal((3, n)), rng.standard_normal((1, n))
    wide = np.zeros((3, 2 * n))
    wide[:, ::2] = X
    for a, b in [(X, U), (np.asfortranarray(X), U.reshape(-1) if n > 1 else U), (wide[:, ::2], 0.25),
                 (X[:, :1], U), (None, U), (X.astype(np.float32), U.tolist())]:
        got = m.call([a, b])
        aos = [m._aos(i, v) for i, v in enumerate((a, b))]
        ref = m.tape.eval_host([None if v is None else v.reshape(-1) for v in aos], n)
        for j, (g, r) in enumerate(zip(got, ref)):
            assert g.flags.c_contiguous and g.flags.writeable and np.array_equal(g, m._dense_out(j, r))
    with pytest.raises(ValueError):
        m.call([np.zeros((3, n + 1)), U]) if n > 1 else m.call([np.zeros((2, 1)), U])
