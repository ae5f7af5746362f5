"""The sums of squared increments: rounding in single precision, and what a sum is taken over."""
import os
import tempfile

import numpy as np
import pytest

from microsim_amd import _abi, configs, host
from microsim_amd.solver import GPSolver

pytestmark = pytest.mark.gpu


def _liquid(mx, my):
    """A binary liquid with mirror sides whose mu increment is 2^-9 lap(mu), exactly."""
    inp, _ = configs.config_c0(mx, 1, 1)
    inp.mesh_x, inp.mesh_y, inp.restart, inp.bc_phi, inp.dt = mx, my, 0, (1, 1, 1, 1), 2.0 ** -6
    with tempfile.TemporaryDirectory() as d:
        configs.write_case(d, inp, [configs.Fill("cylinder", 0, (mx // 2, my // 2, 3.0))])
        c = host.load_case(os.path.join(d, "Input.in"), os.path.join(d, "Filling.in"))
    k = (c.N - 1) * _abi.NCM * _abi.NCM
    c.params.dx = c.params.dy = 1.0
    c.params.A[k], c.params.cmu[k], c.params.diffusivity[k] = 1.0, 0.5, 0.125
    c.phi[:] = 0.0
    c.phi[-1] = 1.0
    return c


@pytest.mark.parametrize("precision", [_abi.GP_FP32, _abi.GP_FP32C])
@pytest.mark.parametrize("seg", ["4", "16"])
def test_no_single_precision_sum_of_more_than_sixteen_terms(precision, seg, monkeypatch):
    """Rows of alternating sign: every increment is 1023 2^-19, its square has 20 significant bits, so sums of up to 16
    of them are exact in 24 bits and the first odd multiple past 16 is not. The result is exact."""
    c = _liquid(64, 248)
    c.mu[0] = (1023.0 / 4096.0) * (1.0 - 2.0 * (np.arange(70) % 2))[:, None]
    monkeypatch.setenv("GP_CELL_SEG", seg)
    print("[gpu] sums of squares, precision", precision, "segment", seg, flush=True)
    with GPSolver(c.params, precision) as s:
        s.upload(c.phi, c.mu)
        st = s.step(1, stats=True)
    assert st["rel_change_mu"][0] == 64 * 248 * 1023.0 ** 2 * 2.0 ** -38
