"""GMRES-IR on operators of extreme scale and with a deep inner solve.

Multiplying the operator and the right-hand side by a power of two leaves the
solution as it is and, as long as no FP32 value leaves the normal range, every
rounding too.  The preconditioner's right-hand side stays near one in every
iteration, whatever the scale and however far the inner solve goes, so
z = M^-1 u stays in range up to the largest operators FP32 holds: the largest
entry here, 11,264 times 2^112, is 0.17 of FP32's largest value.

Both solves reach rtol 1e-10; as solutions of one system they agree far better
than 1e-6 (condition number some 10^3 at this size), and the iteration takes
the same V-cycles."""
import numpy as np
import pytest

import oracle as O
from stzpp_amd import multigrid as MG

pytestmark = pytest.mark.gpu

T_XZ = np.array([[1.0, 0.0, 0.5], [0.0, 1.0, 0.0], [0.0, 0.0, 1.0]])


def solve(kind, power, **kw):
    n = 32
    s = 2.0 ** power
    if kind == "shear":
        prd, o = (1, 1, 0), n + 1
        st, fix = MG.shear_stencil(1.0, 1.5, 1.0 / n, 1.0 / n, 1.0 / n, 1.0)
    else:
        prd, o = (1, 1, 1), n
        st, fix = MG.trans_stencil(T_XZ, 1.0, 1.5, 1.0 / n, 1.0 / n, 1.0 / n, 1.0), None
    N = n * n * o
    b = np.array(O.det_field(N, 71)).reshape(N, 3)
    b -= b.mean(axis=0)
    mg = MG.Multigrid(n, n, o, prd)
    mg.setup_matrices_const(s * st, None if fix is None else s * fix)
    mg.setup_fields(np.zeros((N, 3)), s * b)
    st = mg.solve(MG.SOLVE_FP32_GMRES_IR, rtol=1e-10, max_cycles=60, **kw)
    x = mg.x(0)
    return st, x - (x.mean(axis=0) if prd[2] else 0.0)


@pytest.mark.parametrize("kind", ["shear", "trans"])
@pytest.mark.parametrize("power", [-104, 104, 112])
@pytest.mark.parametrize("kw", [{}, {"restart": 16, "inner_rtol": 1e-6}, {"restart": 16, "inner_rtol": 1e-12}])
def test_gmres_ir_of_a_scaled_operator(kind, power, kw):
    st0, x0 = solve(kind, 0, **kw)
    st, x = solve(kind, power, **kw)
    print(kind, power, kw, st0["cycles"], st["cycles"], st0["outer"], st["outer"],
          np.abs(x - x0).max() / np.abs(x0).max(), flush=True)
    assert st["cycles"] == st0["cycles"] and st["outer"] == st0["outer"]
    assert np.abs(x - x0).max() < 1e-6 * np.abs(x0).max()
