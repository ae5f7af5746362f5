"""The halo of a step: cells whose proxy is a bulk cell (copied in the delta-phi launch) and cells whose proxy is an interface
cell (updated once more as an image), with interfaces across every side and corner, and with the two fields' sides
different, so that an image may belong to one field only. FP64: the whole halo-inclusive state equals the oracle's."""
import os
import tempfile

import numpy as np
import pytest

from gp_testlib import model_step_c32, oracle_step
from microsim_amd import _abi, configs, host
from microsim_amd.solver import GPSolver

pytestmark = pytest.mark.gpu


def _case(mx, my, phi_sides, mu_sides):
    """Seeds on the sides and corners; the maps of mu taken from a second set of sides."""
    def load(sides):
        inp, _, _ = configs.config_ternary(max(mx, my), 0, seed=1234)
        inp.mesh_x, inp.mesh_y, inp.bc_phi = mx, my, sides
        fills = [configs.Fill("cylinder", 0, (0, 0, 4.0)), configs.Fill("cylinder", 1, (mx - 1, my // 2, 5.0)),
                 configs.Fill("cylinder", 1, (mx // 2, my - 1, 4.0)), configs.Fill("cylinder", 0, (mx - 1, my - 1, 3.0))]
        with tempfile.TemporaryDirectory() as d:
            configs.write_case(d, inp, fills)
            return host.load_case(os.path.join(d, "Input.in"), os.path.join(d, "Filling.in"))
    c, other = load(phi_sides), load(mu_sides)
    for k in range(6):
        c.params.halo_src_x[1][k] = other.params.halo_src_x[0][k]
        c.params.halo_src_y[1][k] = other.params.halo_src_y[0][k]
    return c


@pytest.mark.parametrize("mesh", [(24, 20), (37, 131), (260, 41)])
@pytest.mark.parametrize("sides", [((3, 3, 3, 3), (3, 3, 3, 3)), ((1, 1, 1, 1), (3, 3, 3, 3)), ((3, 3, 1, 1), (1, 1, 1, 1))])
def test_halo_equals_the_oracle(mesh, sides):
    c = _case(*mesh, *sides)
    phi, mu = c.phi.copy(), c.mu.copy()
    oracle_step(c.params, phi, mu, 12)
    print("[gpu] halo", mesh, sides, flush=True)
    for stats in (False, True):
        with GPSolver(c.params, _abi.GP_FP64) as s:
            s.upload(c.phi, c.mu)
            s.step(5, stats=stats)
            s.step(7, stats=stats)
            gp, gm = s.download()
        assert np.array_equal(gp, phi) and np.array_equal(gm, mu)


@pytest.mark.parametrize("sides", [((3, 3, 3, 3), (3, 3, 3, 3)), ((1, 1, 1, 1), (3, 3, 3, 3))])
def test_halo_compensated_equals_the_host_build(sides):
    c = _case(37, 131, *sides)
    phi, mu = model_step_c32(c.params, c.phi, c.mu, 9)
    with GPSolver(c.params, _abi.GP_FP32C) as s:
        s.upload(c.phi, c.mu)
        s.step(9)
        gp, gm = s.download()
    i = (slice(None), slice(3, -3), slice(3, -3))
    assert np.array_equal(gp[i], phi[i]) and np.array_equal(gm[i], mu[i])
