"""The 16-lane colour pass of per-point operators (k_gs_points) and the sweeps
of the coarsest level, in the V-cycle and tabulated as x = Q r, against the
oracle.

Points: every kind of boundary (walls all around, periodic, an odd periodic
size with its third colour), sizes whose colour passes end inside a row of
lanes and inside a workgroup, and the smallest grid.  Bottom sweeps: without
the map they run from the tables in the V-cycle; the map's form with tables and
indices in registers takes levels of up to 64 points of a colour (16 x 16 x 16,
16 x 16 x 8, 16 x 16 x 15, 20 x 12 x 9 and 12 x 20 x 12 here, the first and
third at 64), its other form the rest (80, 72 and 96 points).  FP64 rounding of a 27-block sum stays far below 1e-12 of the
largest value over a few sweeps, FP32 below 2e-6 in one.
"""
import numpy as np
import pytest

import oracle as O
from stzpp_amd import multigrid as MG

pytestmark = pytest.mark.gpu


def relerr(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


def f32(a):
    return np.asarray(a, dtype=np.float32).astype(np.float64)


def operator(m, n, o, prd, seed):
    """An operator of its own at every point: the shear stencil scaled and
    perturbed."""
    st, fix = MG.shear_stencil(1.0, 1.5, 1.0 / m, 1.0 / n, 1.0 / o, 1.0)
    pts = O.point_operator((m, n, o), prd, st, fix)[1].reshape(-1, 27, 9)
    rng = np.random.default_rng(seed)
    return np.ascontiguousarray(pts * rng.uniform(0.8, 1.2, pts.shape))


@pytest.mark.parametrize("m,n,o,prd", [(3, 3, 3, (0, 0, 0)), (9, 7, 5, (0, 0, 0)), (8, 6, 7, (1, 1, 0)),
                                       (10, 9, 8, (1, 0, 1)), (5, 7, 6, (1, 1, 1)), (20, 22, 11, (1, 1, 0)),
                                       (17, 16, 16, (0, 1, 1))])
def test_point_sweep(m, n, o, prd):
    N = m * n * o
    pts = operator(m, n, o, prd, N)
    x, r = O.det_field(N, 31), O.det_field(N, 32)
    mg = MG.Multigrid(m, n, o, prd, op_mode=MG.POINT, coarsest_total=N)
    mg.setup_matrices_points(pts)
    orc = O.OracleMG(m, n, o, prd, mode=O.POINT, coarsest_total=N)
    orc.set_ops(0, pts)
    orc.params(smoother=1)
    mg.setup_fields(x, r)
    orc.set_fields(0, x, r)
    mg.gauss_seidel(0, 2)
    orc.gs(0, 2)
    assert relerr(mg.x(0), orc.fields(0)[0]) < 1e-12
    mg.setup_fields(x, r)
    orc.set_fields(0, f32(x), f32(r))
    mg.gauss_seidel_fp32(0, 1)
    orc.gs(0, 1)
    assert relerr(mg.x(0), orc.fields(0)[0]) < 2e-6


@pytest.mark.parametrize("m,n,o,pz", [(16, 16, 16, 1), (16, 16, 8, 1), (16, 16, 15, 0), (16, 16, 17, 0), (20, 12, 9, 0),
                                      (24, 16, 9, 0), (12, 20, 12, 1), (32, 16, 12, 1)])
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("bottom_map", [0, 1])
def test_bottom_sweeps(m, n, o, pz, fp32, bottom_map):
    """Two-level V-cycles whose coarsest level runs its 24 sweeps in one
    workgroup, at every cycle or once for each column of the map, against the
    oracle's."""
    prd = (1, 1, pz)
    T = np.array([[1.05, 0.0, 0.2], [0.0, 1.0, 0.0], [0.0, 0.0, 0.95]])
    st = MG.trans_stencil(T, 1.0, 1.5, 1.0 / m, 1.0 / n, 1.0 / o, 1.0)
    fix = MG.shear_stencil(1.0, 1.5, 1.0 / m, 1.0 / n, 1.0 / o, 1.0)[1]
    mg = MG.Multigrid(m, n, o, prd)
    mg.set_option(MG.OPT_BOTTOM_MAP, bottom_map)
    mg.setup_matrices_const(st, None if pz else fix)
    assert mg.nlevels == 2
    orc = O.OracleMG(m, n, o, prd, mode=O.PLANE)
    orc.set_ops(0, O.plane_operator(o, pz, st, None if pz else fix))
    orc.rat()
    orc.params(smoother=1)
    N = m * n * o
    x, r = O.det_field(N, 41), O.det_field(N, 42)
    if not fp32:
        mg.setup_fields(x, r)
        orc.set_fields(0, x, r)
        mg.v_cycle(2)
        orc.vcycle(2)
        assert relerr(mg.x(0), orc.fields(0)[0]) < 1e-11
    else:
        # one FP32 refinement cycle from zero leaves the FP64 V-cycle's
        # solution up to FP32 rounding
        mg.setup_fields(np.zeros((N, 3)), r)
        with pytest.raises(MG.MultigridError):  # max_cycles reached
            mg.solve(MG.SOLVE_FP32_IR, rtol=1e-14, max_cycles=1, inner_cycles=1)
        orc.set_fields(0, np.zeros((N, 3)), r)
        orc.vcycle(1)
        assert relerr(mg.x(0), orc.fields(0)[0]) < 2e-5
