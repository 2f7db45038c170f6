"""The one-launch sweep (k_gs_halo) against the oracle's 8-colour sweep.

Sizes where it can go wrong: the smallest planes (8, 10 and 12 points wide:
the 24-point window wraps up to three times), tiles that stick out of the
plane (sides not multiples of 8), the fewest planes, an even number of
periodic planes against an odd number between walls, the largest level it
takes while a marching tile divides the plane (512 workgroups) and the first
one beyond, and sides that only it sweeps fused.  Each zero pattern, plain
and centrosymmetric.

Bounds: a sweep forms each value from 27 x 9 products, so FP64 rounding
stays below a few hundred ulp of the largest value over three sweeps
(1e-12), and FP32 below 2e-6 for one sweep on FP32-rounded inputs.
"""
import numpy as np
import pytest

import oracle as O
from stzpp_amd import multigrid as MG

pytestmark = pytest.mark.gpu

T_XZ = np.array([[1.0, 0.0, 0.5], [0.0, 1.0, 0.0], [0.0, 0.0, 1.0]])
T_FULL = np.array([[1.1, 0.2, 0.3], [0.0, 0.9, 0.1], [0.0, 0.0, 1.0]])


def relerr(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


def f32(a):
    return np.asarray(a, dtype=np.float32).astype(np.float64)


def planes_of(kind, m, n, o, pz, outward=False):
    hx, hy, hz = 1.0 / m, 1.0 / n, 1.0 / o
    st, fix = MG.shear_stencil(1.0, 1.5, hx, hy, hz, 1.0)
    if kind in ("trans", "full"):
        st = MG.trans_stencil(T_XZ if kind == "trans" else T_FULL, 1.0, 1.5, hx, hy, hz, 1.0)
    elif kind == "dense":
        # centrosymmetric dense blocks: a Galerkin level of a periodic problem
        big = MG.Multigrid(64, 64, 64, (1, 1, 1))
        big.setup_matrices_const(MG.trans_stencil(T_XZ, 1.0, 1.5, hx, hy, hz, 1.0), None)
        st = big.level_operator(1)[0]
    planes = O.plane_operator(o, pz, st, None if pz else fix)
    if kind == "plain":
        # not centrosymmetric: a perturbed dense stencil, another one per plane
        rng = np.random.default_rng(5)
        planes = np.array(planes).reshape(o, 27, 3, 3)
        planes += 0.02 * np.abs(planes).max() * rng.uniform(-1, 1, planes.shape) * (planes.any(axis=(1, 2, 3)))[
            :, None, None, None]
        if not pz and not outward:
            planes[0, :9] = 0
            planes[-1, 18:] = 0
    return np.ascontiguousarray(planes)


SIZES = [(8, 16, 16, 1), (10, 14, 9, 0), (12, 12, 13, 0), (12, 10, 10, 1), (16, 20, 4, 1), (20, 28, 5, 0),
         (18, 22, 13, 0), (32, 24, 16, 1), (64, 64, 16, 1), (64, 64, 17, 0), (36, 44, 25, 0), (72, 72, 17, 0)]


@pytest.mark.parametrize("m,n,o,pz", SIZES)
@pytest.mark.parametrize("kind", ["shear", "trans", "full", "dense", "plain"])
def test_one_launch_sweep(kind, m, n, o, pz):
    prd = (1, 1, pz)
    planes = planes_of(kind, m, n, o, pz)
    N = m * n * o
    x, r = O.det_field(N, 11), O.det_field(N, 12)
    mg = MG.Multigrid(m, n, o, prd, coarsest_total=N)  # this level alone
    mg.setup_matrices_planes(planes)
    orc = O.OracleMG(m, n, o, prd, mode=O.PLANE, coarsest_total=N)
    orc.set_ops(0, planes)
    orc.params(smoother=1)
    mg.setup_fields(x, r)
    orc.set_fields(0, x, r)
    mg.gauss_seidel(0, 3)
    orc.gs(0, 3)
    assert relerr(mg.x(0), orc.fields(0)[0]) < 1e-12
    mg.setup_fields(x, r)
    orc.set_fields(0, f32(x), f32(r))
    mg.gauss_seidel_fp32(0, 1)
    orc.gs(0, 1)
    assert relerr(mg.x(0), orc.fields(0)[0]) < 2e-6


@pytest.mark.parametrize("m,n,o", [(20, 28, 4), (16, 16, 10), (20, 28, 6), (12, 10, 18), (8, 16, 12), (64, 64, 16),
                                   (16, 16, 9)])
@pytest.mark.parametrize("kind", ["shear", "full", "plain"])
def test_walls_with_blocks_that_point_outward(kind, m, n, o):
    """Walls with an even number of planes, whose last pair has no plane above
    it, and with blocks of the two outermost planes that point across the
    wall: nothing lies there, so they add nothing.  Such a level is the
    coarsest one (only odd numbers of walled planes are coarsened).  Rounding
    as above."""
    planes = planes_of(kind, m, n, o, 0, outward=True)
    if kind != "plain":
        planes[0], planes[-1] = planes[1], planes[1]
    assert planes.reshape(o, 27, 9)[-1, 18:].any() and planes.reshape(o, 27, 9)[0, :9].any()
    N = m * n * o
    x, r = O.det_field(N, 61), O.det_field(N, 62)
    mg = MG.Multigrid(m, n, o, (1, 1, 0), coarsest_total=N)
    mg.setup_matrices_planes(planes)
    orc = O.OracleMG(m, n, o, (1, 1, 0), mode=O.PLANE, coarsest_total=N)
    orc.set_ops(0, planes)
    orc.params(smoother=1)
    mg.setup_fields(x, r)
    orc.set_fields(0, x, r)
    mg.gauss_seidel(0, 3)
    orc.gs(0, 3)
    assert relerr(mg.x(0), orc.fields(0)[0]) < 1e-12
    mg.setup_fields(x, r)
    orc.set_fields(0, f32(x), f32(r))
    mg.gauss_seidel_fp32(0, 1)
    orc.gs(0, 1)
    assert relerr(mg.x(0), orc.fields(0)[0]) < 2e-6


@pytest.mark.parametrize("m,n,o,pz", [(20, 28, 17, 0), (24, 32, 16, 1), (16, 16, 17, 0)])
def test_vcycle_from_zero(m, n, o, pz):
    """V-cycles through one-launch levels, whose first sweep starts from
    x = 0 without reading it, against the oracle's."""
    prd = (1, 1, pz)
    st, fix = MG.shear_stencil(1.0, 1.5, 1.0 / m, 1.0 / n, 1.0 / o, 1.0)
    mg = MG.Multigrid(m, n, o, prd)
    mg.setup_matrices_const(st, None if pz else fix)
    orc = O.OracleMG(m, n, o, prd, mode=O.PLANE)
    orc.set_ops(0, O.plane_operator(o, pz, st, None if pz else fix))
    orc.rat()
    orc.params(smoother=1)
    x, r = O.det_field(m * n * o, 21), O.det_field(m * n * o, 22)
    mg.setup_fields(x, r)
    orc.set_fields(0, x, r)
    mg.v_cycle(2)
    orc.vcycle(2)
    assert relerr(mg.x(0), orc.fields(0)[0]) < 1e-11


@pytest.mark.parametrize("m,n,o,pz", [(8, 16, 16, 1), (12, 20, 9, 0), (16, 16, 17, 0), (18, 22, 13, 0), (32, 24, 16, 1),
                                      (36, 44, 25, 0), (64, 64, 33, 0)])
@pytest.mark.parametrize("kind", ["shear", "trans", "full", "dense", "plain"])
def test_residual_and_restriction_in_one_launch(kind, m, n, o, pz):
    """Tiles that stick out of the coarse plane, one and several tiles, walls
    and periodic z; the residual is a 27-block sum and the restriction 27
    weights, so FP64 rounding stays below 1e-12 of the largest value."""
    prd = (1, 1, pz)
    planes = planes_of(kind, m, n, o, pz)
    N = m * n * o
    x, r = O.det_field(N, 51), O.det_field(N, 52)
    mg = MG.Multigrid(m, n, o, prd, coarsest_total=N - 1)
    mg.setup_matrices_planes(planes)
    orc = O.OracleMG(m, n, o, prd, mode=O.PLANE, coarsest_total=N - 1)
    orc.set_ops(0, planes)
    assert mg.nlevels == 2
    mg.setup_fields(x, r)
    mg.setup_fields(O.det_field(mg.npts(1), 53), None, 1)
    orc.set_fields(0, x, r)
    mg.restriction(1)
    orc.restrict(1)
    xc, rc = mg.fields(1)
    assert not xc.any()
    assert relerr(rc, orc.fields(1)[1]) < 1e-12


@pytest.mark.parametrize("kind", ["shear", "trans", "full"])
@pytest.mark.parametrize("timed", [0, 2])  # FP64 sweep, FP32 sweep
def test_patterns_without_symmetry_cost_no_more_than_dense(kind, timed):
    """A zero pattern only takes entries out of the dense stencil's sums, so
    its sweep is no slower than the dense one, also where no two opposite
    blocks are equal.  Half as much again is left for the clock; the fault this
    guards against took 2.3 times as long."""
    m, n, o = 32, 32, 33
    us = {}
    for k in ("plain", kind):
        planes = planes_of(k, m, n, o, 0)
        rng = np.random.default_rng(8)
        planes = planes * (1 + 1e-3 * rng.uniform(-1, 1, planes.shape))
        mg = MG.Multigrid(m, n, o, (1, 1, 0), coarsest_total=m * n * o)
        mg.setup_matrices_planes(planes)
        mg.setup_fields(O.det_field(m * n * o, 81), O.det_field(m * n * o, 82))
        mg.time_kernel(timed, 0, 50)
        us[k] = 1e3 * min(mg.time_kernel(timed, 0, 50) for _ in range(5))
    print(us, flush=True)
    assert us[kind] < 1.5 * us["plain"]


@pytest.mark.parametrize("kind,o,fused", [("plain", 47, True), ("plain", 49, False), ("full", 71, True),
                                          ("full", 73, False), ("trans", 95, True), ("trans", 97, False),
                                          ("shear", 95, True), ("shear", 97, False), ("plain", 161, False)])
def test_large_level_that_no_tile_divides(kind, o, fused):
    """76 x 76 points, 100 workgroups a plane pair: up to 2400 (dense), 3600 (no
    corners) and 4800 (transformed, shear) workgroups sweep in one launch, more
    in eight colour launches, which beat it there (100 x 100 x 100 dense 115 us
    against 210).  Both compute the same sweep (rounding as above)."""
    N = 76 * 76 * o
    mg = MG.Multigrid(76, 76, o, (1, 1, 0), coarsest_total=N)
    mg.setup_matrices_planes(planes_of(kind, 76, 76, o, 0))
    x, r = O.det_field(N, 91), O.det_field(N, 92)
    mg.setup_fields(x, r)
    mg.gauss_seidel(0, 1)
    got = mg.x(0)
    if fused:
        assert mg.time_kernel(4, 0, 1) > 0  # one launch of the fused sweep
    else:
        with pytest.raises(MG.MultigridError):
            mg.time_kernel(4, 0, 1)
    mg.set_option(MG.OPT_FUSED_SMOOTHER, 0)
    mg.setup_fields(x, r)
    mg.gauss_seidel(0, 1)
    assert relerr(got, mg.x(0)) < 1e-12
