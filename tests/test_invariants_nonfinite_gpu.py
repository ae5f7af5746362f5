"""Solute and energy of states with non-finite values: NaN and infinities come out as from the sums over all phases
(the oracle), also where a phase is absent and its terms are zeros times the value."""
import ctypes as C

import numpy as np
import pytest

from gp_testlib import load_golden, oracle
from microsim_amd import _abi
from microsim_amd.solver import GPSolver

pytestmark = pytest.mark.gpu


def _class(v):
    return np.where(np.isnan(v), 2, np.isinf(v) * np.sign(v)).tolist()


@pytest.mark.parametrize("precision", [_abi.GP_FP64, _abi.GP_FP32])
@pytest.mark.parametrize("phase", ["liquid", "none"])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_nonfinite_mu(value, phase, precision):
    case, _ = load_golden("tern_c1_mini")
    phi, mu = np.zeros_like(case.phi), np.full_like(case.mu, 0.25)
    if phase == "liquid":
        phi[-1] = 1.0
    mu[0, 40, 50] = value
    sol, en = (C.c_double * 4)(), C.c_double()
    oracle().oracle_invariants(C.byref(case.params), _abi.dptr(phi), _abi.dptr(mu), sol, C.byref(en))
    print("[gpu] invariants of mu =", value, phase, precision, flush=True)
    with GPSolver(case.params, precision) as s:
        s.upload(phi, mu)
        st = s.stats()
    got = np.append(st["solute"], st["energy"])
    assert _class(got) == _class(np.append(sol[:case.NC], en.value))
    assert np.isnan(got).any()
