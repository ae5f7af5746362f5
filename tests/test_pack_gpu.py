"""States to the device and back (gp_pack.h): a downloaded state is the uploaded one with its boundary copies, rounded to
the stored precision, bit for bit: the smallest grid, odd sides, and a state of more rows than one staging run holds (its
runs cross from one component to the next). The two state buffers agree (a step reads one and keeps cells of the other)."""
import ctypes as C

import numpy as np
import pytest

from gp_testlib import model_lib
from microsim_amd import _abi, configs, host
from microsim_amd.solver import GPSolver

pytestmark = pytest.mark.gpu


def _params(tmp_path, mx, my, sides):
    inp = configs.GPInput(mesh_x=mx, mesh_y=my, nphases=4, ncomp=3, dt=0.02, gamma=configs.upper(4, 1.0),
                          tau_ab=configs.upper(4, 0.3), dab=configs.upper(4, 0.02), gamma_abc=[1.5, 0.5, 1.0, 2.0],
                          components=["Al", "Cu", "Ni"], phases=["alpha", "beta", "gamma", "liquid"], epsilon=4.0, tau=0.3)
    configs.ternary_material(inp, np.random.default_rng(31))
    inp.bc_phi = sides
    configs.write_case(str(tmp_path), inp, [configs.Fill("cylinder", 0, (mx // 2, my // 2, 2.0))])
    return host.load_case(str(tmp_path / "Input.in"), str(tmp_path / "Filling.in")).params


def _stored(v, field, precision):
    if precision == _abi.GP_FP64:
        return v
    if precision == _abi.GP_FP32:
        return v.astype(np.float32).astype(np.float64)
    out, n = np.empty(v.size), v.size
    hi = np.empty(n, dtype=np.float32)
    second = np.empty(n, dtype=np.float32 if field == 0 else np.int8)
    f = model_lib().df_roundtrip if field == 0 else model_lib().c32_roundtrip
    f(_abi.dptr(np.ascontiguousarray(v.ravel())), n, hi.ctypes.data_as(C.c_void_p), second.ctypes.data_as(C.c_void_p),
      _abi.dptr(out))
    return out.reshape(v.shape)


def _with_halo(v, p, field):
    v = v.copy()
    rx, ry = v.shape[1:]
    hx, hy = (0, 1, 2, rx - 3, rx - 2, rx - 1), (0, 1, 2, ry - 3, ry - 2, ry - 1)
    for k in range(6):
        v[:, hx[k], :] = v[:, p.halo_src_x[field][k], :]
    for k in range(6):
        v[:, :, hy[k]] = v[:, :, p.halo_src_y[field][k]]
    return v


@pytest.mark.parametrize("precision", [_abi.GP_FP64, _abi.GP_FP32, _abi.GP_FP32C])
@pytest.mark.parametrize("mesh,sides", [((4, 5), (1, 1, 1, 1)), ((61, 131), (3, 3, 1, 1)), ((1100, 1025), (3, 3, 3, 3))])
def test_state_round_trip(tmp_path, mesh, sides, precision):
    p = _params(tmp_path, *mesh, sides)
    rng = np.random.default_rng(7)
    phi = rng.uniform(0.0, 1.0, (4, mesh[0] + 6, mesh[1] + 6))
    mu = rng.normal(0.0, 1.0, (2, mesh[0] + 6, mesh[1] + 6)) * 10.0 ** rng.integers(-9, 3, (2, 1, 1))
    phi[0, 5, 5], phi[1, 5, 5] = 0.0, 1.0
    want = [_with_halo(_stored(v, f, precision), p, f) for f, v in enumerate((phi, mu))]
    print("[gpu] round trip", mesh, sides, precision, flush=True)
    with GPSolver(p, precision) as s:
        for _ in range(2):
            s.upload(phi, mu)
            got = s.download()
            for g, w in zip(got, want):
                assert np.array_equal(g, w)
