"""Halo maps in which three halo rows and columns share one source: a step copies to the first two only, and the third keeps
what the upload left there, in both state buffers. Sweeps over such a run cannot step from one stored state into another
(its halo would be missing there) and go through the handle's buffers instead."""
import os
import tempfile

import numpy as np
import pytest

from microsim_amd import _abi, configs, host
from microsim_amd.solver import GPSolver

pytestmark = pytest.mark.gpu


def _case(mx=40, my=36):
    inp, _, _ = configs.config_ternary(max(mx, my), 0, seed=1234)
    inp.mesh_x, inp.mesh_y, inp.bc_phi = mx, my, (1, 1, 1, 1)
    fills = [configs.Fill("cylinder", 0, (2, my // 2, 6.0)), configs.Fill("cylinder", 1, (mx // 2, my - 3, 6.0)),
             configs.Fill("cylinder", 1, (mx - 4, 2, 5.0))]
    with tempfile.TemporaryDirectory() as d:
        configs.write_case(d, inp, fills)
        c = host.load_case(os.path.join(d, "Input.in"), os.path.join(d, "Filling.in"))
    p = c.params
    for f in range(2):
        p.halo_src_x[f][:] = [4, 4, 4, mx + 1, mx + 1, mx + 1]
        p.halo_src_y[f][:] = [4, 4, 4, my + 1, my + 1, my + 1]
    return c


@pytest.mark.parametrize("precision", [_abi.GP_FP64, _abi.GP_FP32, _abi.GP_FP32C])
def test_a_halo_cell_without_proxy_keeps_the_upload(precision):
    c = _case()
    rx, ry = c.phi.shape[1:]
    kept = np.zeros((rx, ry), dtype=bool)   # the third row and column of each side, where the other index has a proxy
    kept[[2, rx - 1], :] = kept[:, [2, ry - 1]] = True
    inner = (slice(None), slice(3, -3), slice(3, -3))
    print("[gpu] halo without proxies, precision", precision, flush=True)
    with GPSolver(c.params, precision) as s:
        s.upload(c.phi, c.mu)
        first = s.download()
        for n in range(4):
            s.step(1, stats=n % 2 == 1)
            got = s.download()
            for g, f in zip(got, first):
                assert np.array_equal(g[:, kept], f[:, kept])
                # the others are copies of this step's interior
                assert np.array_equal(g[:, 0, 3:-3], g[:, 4, 3:-3]) and np.array_equal(g[:, 1, 3:-3], g[:, 4, 3:-3])
                assert np.array_equal(g[:, rx - 3, 3:-3], g[:, rx - 5, 3:-3])
                assert np.array_equal(g[:, 3:-3, ry - 2], g[:, 3:-3, ry - 5])
    assert not np.array_equal(got[0][inner], first[0][inner]) and not np.array_equal(got[1][inner], first[1][inner])


@pytest.mark.parametrize("precision", [_abi.GP_FP64, _abi.GP_FP32C])
def test_sweep_through_the_handles_buffers(precision):
    """A sweep of one segment (recomputed states) gives the gradient of one with every state kept. Both sum the same terms
    in the order of atomic additions; a term is one of some twenty of a cell and step, so 1e-11 of the largest entry."""
    c = _case()
    rng = np.random.default_rng(5)
    w, out = (rng.standard_normal(c.phi.shape), rng.standard_normal(c.mu.shape)), []
    for every in (1, 4, 9):
        print("[gpu] sweep without proxies, interval", every, "precision", precision, flush=True)
        with GPSolver(c.params, precision) as s:
            s.upload(c.phi, c.mu)
            s.adjoint_forward(9, every)
            last = s.download()
            out.append(s.adjoint_backward(*w) + last)
    for o in out[1:]:
        for got, want in zip(o[:3], out[0][:3]):
            assert np.abs(got - want).max() <= 1e-11 * np.abs(want).max()
        assert np.array_equal(o[3], out[0][3]) and np.array_equal(o[4], out[0][4])
