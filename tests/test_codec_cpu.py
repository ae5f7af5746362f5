"""The compensated form of mu (gp_model.h c32_encode / c32_decode) at the ends of its range: both zeros, subnormal and
non-finite values, and values halfway between two FP32 numbers come back as stored, with their sign."""
import numpy as np

import gp_testlib
from microsim_amd import _abi


def _roundtrip(v):
    v = np.ascontiguousarray(v, dtype=np.float64)
    hi, q, out = np.empty(v.size, np.float32), np.empty(v.size, np.int8), np.empty_like(v)
    gp_testlib.model_lib().c32_roundtrip(_abi.dptr(v), v.size, hi.ctypes.data, q.ctypes.data, _abi.dptr(out))
    return hi, q, out


def test_single_precision_values_keep_their_bits():
    f = np.array([0.0, -0.0, 1e-45, -1e-45, 1e-39, -1e-39, 2.0 ** -126, -2.0 ** -126, 3.4e38, -3.4e38, np.inf, -np.inf],
                 dtype=np.float32).astype(np.float64)
    hi, q, out = _roundtrip(f)
    assert np.array_equal(out.view(np.int64), f.view(np.int64)) and not q.any()


def test_halfway_values():
    """|v - hi| = ulp / 2 is the largest extension, 64 units, and exact; both signs."""
    v = np.ldexp([1.0 + 2.0 ** -24, 1.0 + 3.0 * 2.0 ** -24, 1.0 - 2.0 ** -25, 2.0 - 2.0 ** -24], [[0], [-100], [90]]).ravel()
    hi, q, out = _roundtrip(np.concatenate([v, -v]))
    assert np.array_equal(out, np.concatenate([v, -v]))
    assert np.abs(q.astype(int)).max() == 64 and (np.abs(q) >= 32).all()
