"""Whole fields through the pinned ring (host_copy.hpp) equal the field read
back by the other path, at sizes around the ring's thresholds and chunk."""
import numpy as np
import pytest

from stzpp_amd import shear_sim as SS

pytestmark = pytest.mark.gpu


# cubes of 11.8 MB (runtime path), 12.6 MB, 14.2 MB (last chunk short) and
# 16.8 MB (whole chunks); reference maps of 36.6 to 101 MB
@pytest.mark.parametrize("N", [(192, 160, 96), (256, 192, 64), (192, 192, 96), (256, 128, 128)])
def test_cubes_and_reference_map(N):
    sim = SS.ShearSim(*N, params=SS.config0_params(N[0]))
    rng = np.random.default_rng(N[0])
    nc, nv = sim.ncells, sim.nverts
    chi = rng.uniform(0.05, 0.12, nc)
    sig = rng.standard_normal((nc, 6))
    u = rng.standard_normal((nv, 3))
    sim.set_initial_conditions(chi, u=u, sig=sig)
    for mode, src in ((11, chi), (3, sig[:, 0]), (8, sig[:, 5])):
        want = src.reshape(N[2], N[1], N[0]).transpose(2, 1, 0).astype(np.float32).ravel()
        assert np.array_equal(sim.output_cube(mode), want)
    xi = rng.standard_normal((nv, 3))
    sim.set_ref_map(xi)
    assert np.array_equal(sim.ref_map(), xi)
