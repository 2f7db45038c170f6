"""The marching kernels of the direct step.

They cut z into as many chunks as the device keeps workgroups of 64 x 4 tiles
resident.  Small grids, where every chunk is one plane, have the tile's edges:
grids smaller than a tile, four points short of and past its edges, the
smallest allowed, odd counts of planes, walled and periodic z.  MARCHING are
grids wide enough that a chunk holds several planes on 256 CUs with two
workgroups each (512 resident): 256 x 192 x 16 has 192 tiles and two chunks of
8 planes (the 17 vertex planes 9 and 8), 256 x 160 x 16 160 tiles and chunks of
6, 6 and 4 planes (vertices 6, 6, 5), 128 x 128 x 32 64 tiles and chunks of 4,
160 x 96 x 32 72 tiles, six chunks of 5 planes and one of 2.

Without yielding no transcendental function enters and every operation is
rounded in the reference's order, so two steps equal the oracle's bit for bit
(tolerance zero).

With yielding the STZ rate goes through exp, whose last bit the GPU's library
may round otherwise than glibc.  The rate's relative change is some 50 times
that of stress or chi, over two steps with a few ulp each: ad_Dpl is held to
1e-11 of its largest value, the other fields, which it changes by at most their
own size, to 1e-12 of the larger of theirs and one.  Half of the cells yield, at
random, and the diffusion of chi moves it by 1e-4 to 1e-2 at most, so a wrong
neighbour or a wrong step's ad_Dpl shows at 10^8 times the bound.  ad_Dpl's
neighbours are this step's at -x/-y/-z and last step's at +x/+y/+z and at
periodic images; the second step has both."""
import numpy as np
import pytest

import oracle as O
from stzpp_amd import shear_sim as SS

pytestmark = pytest.mark.gpu

EDGES = [(4, 4, 4), (5, 9, 7), (60, 8, 8), (68, 8, 8), (56, 12, 8), (72, 12, 8), (136, 12, 12), (12, 40, 28)]
MARCHING = [((256, 192, 16), 0), ((256, 160, 16), 0), ((128, 128, 32), 1), ((160, 96, 32), 1)]


def pair(N, pz, params, sig, u, chi):
    """A simulation and the oracle's with the same state, and both their
    states (with the reference map) after steps of dt."""
    P = {**SS.config0_params(N[0]), **params}
    prd = (1, 1, pz)
    rho, kappa = 1.0, 0.35
    sim = SS.ShearSim(*N, params={**P, "rho": rho, "kappa": kappa, "tmult": 0.5}, prd=prd)
    orc = O.OracleShear(N, {k: float(sim.params[k]) for k in O.STEP_PARAM_ORDER}, prd=prd)
    orc.set_direct(rho, kappa)
    sim.set_initial_conditions(chi, u=u, sig=sig, t=0.25)
    sim.init_ref()
    orc.set_state(0.25, u, sig, chi)
    orc.init_ref()

    def step(dt, n):
        sim.step_forward(dt, n)
        orc.step_direct(dt, n)
        got, want = sim.state(), orc.state()
        got["xi"], want["xi"] = sim.ref_map(), orc.ref_map()
        return got, want

    return sim, step


def counts(N, pz):
    return N[0] * N[1] * N[2], N[0] * N[1] * (N[2] + 1 - pz)


def elastic(N, pz):
    nc, nv = counts(N, pz)
    rng = np.random.default_rng(sum(N) + pz)
    u = 0.01 * rng.standard_normal((nv, 3))
    sig = 0.1 * rng.standard_normal((nc, 6))
    chi = 0.08 + 0.01 * rng.random(nc)
    sim, step = pair(N, pz, {"sy": 1e6}, sig, u, chi)
    got, want = step(sim.direct_dt(), 2)
    assert sim.last_stats["yielded_cells"] == 0
    for key in ("u", "sig", "chi", "dpl", "xi"):
        assert np.all(np.isfinite(want[key])), key
        assert np.array_equal(got[key], want[key]), (key, np.abs(got[key] - want[key]).max())


@pytest.mark.parametrize("pz", [0, 1])
@pytest.mark.parametrize("N", EDGES)
def test_gpu_direct_elastic_steps_at_tile_edges(N, pz):
    elastic(N, pz)


@pytest.mark.parametrize("N,pz", MARCHING)
def test_gpu_direct_elastic_steps_in_chunks(N, pz):
    elastic(N, pz)


@pytest.mark.parametrize("N,pz", [(N, pz) for N in EDGES for pz in (0, 1)] + MARCHING)
def test_gpu_direct_yielding_steps(N, pz):
    nc, nv = counts(N, pz)
    rng = np.random.default_rng(sum(N) + pz)
    u = 0.01 * rng.standard_normal((nv, 3))
    sig = 0.05 * rng.standard_normal((nc, 6))
    sig[:, 1] += np.where(rng.random(nc) < 0.5, 1.1, 0.3)
    chi = 0.09 + 0.005 * rng.standard_normal(nc)
    h = min(2 / N[0], 2 / N[1], 1 / N[2])
    sim, step = pair(N, pz, {"eps0": 0.2, "diff_l": 3 * h}, sig, u, chi)
    got, want = step(1e-4, 2)
    assert nc / 5 < sim.last_stats["yielded_cells"] < 4 * nc / 5
    assert np.abs(want["dpl"]).max() > 0.1
    for key in ("u", "sig", "chi", "dpl", "xi"):
        assert np.all(np.isfinite(want[key])), key
        big = np.abs(want[key]).max()
        bound = 1e-11 * big if key == "dpl" else 1e-12 * max(1.0, big)
        assert np.abs(got[key] - want[key]).max() < bound, (key, np.abs(got[key] - want[key]).max(), big)
