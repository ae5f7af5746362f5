"""States at the ends of the range, up and down again: the device encodes and decodes as the host forms do (gp_model.h, numpy),
bit for bit: zeros of both signs, subnormal values in either precision, values that overflow single precision, halfway
values, infinities and NaN."""
import ctypes as C

import numpy as np
import pytest

from gp_testlib import load_golden, model_lib
from microsim_amd import _abi
from microsim_amd.solver import GPSolver

pytestmark = pytest.mark.gpu

VALUES = np.array([0.0, -0.0, 5e-324, -5e-324, 1e-310, 1e-46, 1.4e-45, -1e-41, 1e-39, 1.1754943e-38, -2.0 ** -126, 1e-30,
                   1.0 + 2.0 ** -24, -(1.0 + 2.0 ** -24), 1.0 - 2.0 ** -25, 1.0 + 2.0 ** -31, 0.3, -7.1e9, 3.4028234e38,
                   3.4028235677973366e38, -3.5e38, 1e300, np.inf, -np.inf, np.nan])


def _host(v, field, precision):
    """v as stored and read back, with the host build of the codecs."""
    if precision == _abi.GP_FP64:
        return v
    if precision == _abi.GP_FP32:
        with np.errstate(over="ignore"):
            return v.astype(np.float32).astype(np.float64)
    out, hi, n = np.empty(v.size), np.empty(v.size, dtype=np.float32), v.size
    second = np.empty(n, dtype=np.float32 if field == 0 else np.int8)
    f = model_lib().df_roundtrip if field == 0 else model_lib().c32_roundtrip
    f(_abi.dptr(np.ascontiguousarray(v)), n, hi.ctypes.data_as(C.c_void_p), second.ctypes.data_as(C.c_void_p), _abi.dptr(out))
    return out


@pytest.mark.parametrize("precision", [_abi.GP_FP64, _abi.GP_FP32, _abi.GP_FP32C])
def test_extreme_values_round_trip(precision):
    case, _ = load_golden("tern_c1_mini")
    phi, mu = case.phi.copy(), case.mu.copy()
    row = slice(20, 20 + VALUES.size)
    phi[0, 30, row] = VALUES
    mu[1, 40, row] = VALUES
    print("[gpu] extreme values, precision", precision, flush=True)
    with GPSolver(case.params, precision) as s:
        s.upload(phi, mu)
        p, m = s.download()
    for got, want in ((p[0, 30, row], _host(VALUES, 0, precision)), (m[1, 40, row], _host(VALUES, 1, precision))):
        nan = np.isnan(want)
        assert np.array_equal(np.isnan(got), nan)
        assert np.array_equal(got[~nan].view(np.int64), want[~nan].view(np.int64))
