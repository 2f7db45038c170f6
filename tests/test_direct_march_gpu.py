"""The marching kernels of the direct step at the sizes where a tile of 64 x 4
points and a chunk of planes can go wrong: grids smaller than a tile, four points
short of and past its edges, the smallest allowed, odd counts of planes, walled
and periodic z.

Without yielding no transcendental function enters and every operation is
rounded in the reference's order, so two steps equal the oracle's bit for bit
(tolerance zero)."""
import numpy as np
import pytest

import oracle as O
from stzpp_amd import shear_sim as SS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pz", [0, 1])
@pytest.mark.parametrize("N", [(4, 4, 4), (5, 9, 7), (60, 8, 8), (68, 8, 8), (56, 12, 8), (72, 12, 8),
                               (136, 12, 12), (12, 40, 28)])
def test_gpu_direct_elastic_steps_at_tile_edges(N, pz):
    P = {**SS.config0_params(N[0]), "sy": 1e6}
    prd = (1, 1, pz)
    rho, kappa = 1.0, 0.35
    sim = SS.ShearSim(*N, params={**P, "rho": rho, "kappa": kappa, "tmult": 0.5}, prd=prd)
    orc = O.OracleShear(N, {k: float(sim.params[k]) for k in O.STEP_PARAM_ORDER}, prd=prd)
    orc.set_direct(rho, kappa)
    rng = np.random.default_rng(sum(N) + pz)
    nc = N[0] * N[1] * N[2]
    nv = N[0] * N[1] * (N[2] + 1 - pz)
    u = 0.01 * rng.standard_normal((nv, 3))
    sig = 0.1 * rng.standard_normal((nc, 6))
    chi = 0.08 + 0.01 * rng.random(nc)
    sim.set_initial_conditions(chi, u=u, sig=sig, t=0.25)
    sim.init_ref()
    orc.set_state(0.25, u, sig, chi)
    orc.init_ref()
    dt = sim.direct_dt()
    sim.step_forward(dt, 2)
    orc.step_direct(dt, 2)
    assert sim.last_stats["yielded_cells"] == 0
    got, want = sim.state(), orc.state()
    got["xi"], want["xi"] = sim.ref_map(), orc.ref_map()
    for key in ("u", "sig", "chi", "dpl", "xi"):
        assert np.all(np.isfinite(want[key])), key
        assert np.array_equal(got[key], want[key]), (key, np.abs(got[key] - want[key]).max())
