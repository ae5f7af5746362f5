"""k_cbulk's tiles at their edges: strips of 124 cells (full, one short, one over), segments of 16 and of 4 rows, uniform
and mixed tiles, against the FP64 oracle (bit for bit), the host build of the compensated mode (bit for bit) and, for
FP32, one segment length against the other (the arithmetic of a cell does not depend on its tile)."""
import os
import tempfile

import numpy as np
import pytest

from gp_testlib import model_step_c32, oracle_step
from microsim_amd import _abi, configs, host

pytestmark = pytest.mark.gpu

MESHES = [(16, 124), (15, 125), (17, 123), (36, 249), (33, 372), (5, 260), (64, 40)]


def _case(mx, my, bc=(3, 3, 1, 1)):
    inp, _, _ = configs.config_ternary(max(mx, my), 0, seed=1234)
    inp.mesh_x, inp.mesh_y, inp.bc_phi = mx, my, bc
    fills = [configs.Fill("cylinder", 0, (mx // 2, 9, 5.0)), configs.Fill("cylinder", 1, (mx // 3, my - 14, 6.0))]
    with tempfile.TemporaryDirectory() as d:
        configs.write_case(d, inp, fills)
        return host.load_case(os.path.join(d, "Input.in"), os.path.join(d, "Filling.in"))


def _run(case, precision, seg, monkeypatch, steps, stats):
    from microsim_amd.solver import GPSolver
    print("[gpu] mesh", case.params.mesh_x, case.params.mesh_y, "precision", precision, "segment", seg, "stats", stats,
          flush=True)
    monkeypatch.setenv("GP_CELL_SEG", str(seg))
    with GPSolver(case.params, precision) as s:
        s.upload(case.phi, case.mu)
        s.step(1)
        st = s.step(steps - 1, stats=stats)
        return s.download() + (st,)


@pytest.mark.parametrize("seg", [4, 16])
@pytest.mark.parametrize("mesh", MESHES)
def test_tiles_fp64_equal_the_oracle(mesh, seg, monkeypatch):
    case = _case(*mesh)
    phi, mu = case.phi.copy(), case.mu.copy()
    oracle_step(case.params, phi, mu, 8)
    p0, m0 = phi.copy(), mu.copy()
    oracle_step(case.params, phi, mu, 1)
    gp, gm, st = _run(case, _abi.GP_FP64, seg, monkeypatch, 9, True)
    i = (slice(None), slice(3, -3), slice(3, -3))
    assert np.array_equal(gp[i], phi[i]) and np.array_equal(gm[i], mu[i])
    assert st["nonfinite"] == 0
    # the sums of the last step (a sum of mesh_x mesh_y terms: relative rounding far below 1e-10); grids whose rows are
    # not a multiple of four add the padding rows' terms to those of mu
    np.testing.assert_allclose(st["rel_change_phi"], ((phi - p0)[i] ** 2).sum((1, 2)), rtol=1e-10)
    if mesh[0] % 4 == 0:
        np.testing.assert_allclose(st["rel_change_mu"], ((mu - m0)[i] ** 2).sum((1, 2)), rtol=1e-10)


@pytest.mark.parametrize("mesh", MESHES[:4])
def test_tiles_fp32c_equal_the_host_build(mesh, monkeypatch):
    case = _case(*mesh)
    phi, mu = model_step_c32(case.params, case.phi, case.mu, 6)
    for seg in (4, 16):
        gp, gm, _ = _run(case, _abi.GP_FP32C, seg, monkeypatch, 6, seg == 4)
        i = (slice(None), slice(3, -3), slice(3, -3))
        assert np.array_equal(gp[i], phi[i]) and np.array_equal(gm[i], mu[i])


@pytest.mark.parametrize("mesh", MESHES)
def test_tiles_fp32_do_not_depend_on_the_segment(mesh, monkeypatch):
    case = _case(*mesh)
    a = _run(case, _abi.GP_FP32, 4, monkeypatch, 7, True)
    b = _run(case, _abi.GP_FP32, 16, monkeypatch, 7, False)
    c = _run(case, _abi.GP_FP32, 16, monkeypatch, 7, True)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    for k in ("phi_max", "phi_min", "mu_max", "mu_min", "nonfinite"):
        assert a[2][k] == c[2][k]
    # per-lane partial sums in FP32 over at most 32 cells each
    np.testing.assert_allclose(a[2]["rel_change_mu"], c[2]["rel_change_mu"], rtol=1e-5)
