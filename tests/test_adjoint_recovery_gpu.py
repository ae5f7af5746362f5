"""The adjoint after a call that failed: every later call is refused or gives what a fresh handle gives."""
import os
import tempfile

import numpy as np
import pytest

from microsim_amd import _abi, configs, host
from microsim_amd.solver import GPError, GPSolver

pytestmark = pytest.mark.gpu


def _case(mx, my):
    inp, _, _ = configs.config_ternary(max(mx, my), 0, seed=1234)
    inp.mesh_x, inp.mesh_y = mx, my
    fills = [configs.Fill("cylinder", 0, (mx // 2, 9, 5.0)), configs.Fill("cylinder", 1, (mx // 3, my - 14, 6.0))]
    with tempfile.TemporaryDirectory() as d:
        configs.write_case(d, inp, fills)
        return host.load_case(os.path.join(d, "Input.in"), os.path.join(d, "Filling.in"))


def _weights(case):
    rng = np.random.default_rng(3)
    return rng.standard_normal(case.phi.shape), rng.standard_normal(case.mu.shape)


def _same(a, b):
    """Gradients of one trajectory: sums in the order of atomic additions."""
    for x, y in zip(a, b):
        assert np.abs(x - y).max() <= 1e-11 * np.abs(y).max()


def test_no_sweep_over_checkpoints_that_do_not_fit():
    """4096 checkpoints of 2048^2 are more than the card holds: the recording fails, there is none afterwards (the earlier
    one is gone as well), and a sweep is refused before it launches anything."""
    case = _case(2048, 2048)
    w = _weights(case)
    with GPSolver(case.params) as s:
        s.upload(case.phi, case.mu)
        for before in (0, 2):
            if before:
                s.adjoint_forward(before, 1)
            print("[gpu] recording that does not fit, after", before, "steps", flush=True)
            with pytest.raises(GPError) as e:
                s.adjoint_forward(4096, 1)
            assert e.value.code == _abi.GP_E_OOM
            with pytest.raises(GPError) as e:
                s.adjoint_backward(*w)
            assert e.value.code == _abi.GP_E_ARG
        s.upload(case.phi, case.mu)
        s.adjoint_forward(3, 2)
        got = s.adjoint_backward(*w)
    with GPSolver(case.params) as s:
        s.upload(case.phi, case.mu)
        s.adjoint_forward(3, 2)
        _same(got, s.adjoint_backward(*w))


def test_one_checkpoint_of_the_largest_interval():
    case = _case(40, 36)
    w, got = _weights(case), []
    for every in (3, (1 << 63) - 1):
        print("[gpu] checkpoint interval", every, flush=True)
        with GPSolver(case.params) as s:
            s.upload(case.phi, case.mu)
            s.adjoint_forward(3, every)
            got.append(s.adjoint_backward(*w))
    _same(*got)


@pytest.mark.parametrize("nsteps", [1 << 40, (1 << 62) + 1])
def test_recording_of_more_checkpoints_than_the_host_could_list(nsteps):
    case = _case(40, 36)
    with GPSolver(case.params) as s:
        s.upload(case.phi, case.mu)
        print("[gpu] recording", nsteps, "checkpoints", flush=True)
        with pytest.raises(GPError) as e:
            s.adjoint_forward(nsteps, 1)
        assert e.value.code == _abi.GP_E_OOM
        phi, mu = s.download()
        assert np.array_equal(phi, case.phi) and np.array_equal(mu, case.mu)


@pytest.mark.parametrize("precision", [_abi.GP_FP64, _abi.GP_FP32C])
@pytest.mark.parametrize("nsteps", [3, 4, 5])
def test_steps_after_a_sweep_that_failed(precision, nsteps, monkeypatch):
    """A sweep that ends in the middle of a segment leaves the handle with one of its own two states, the last of the
    trajectory or the one before, and steps from there as an undisturbed run does (the cell classes are those of the state
    that it holds, not those of the segment)."""
    case = _case(60, 52)
    wphi, wmu = _weights(case)
    wmu[0, 30, 20] = np.nan
    with GPSolver(case.params, precision) as s:
        s.upload(case.phi, case.mu)
        s.adjoint_forward(nsteps, nsteps)
        monkeypatch.setenv("GP_ADJOINT_CHECK", "1000")
        print("[gpu] sweep that fails,", nsteps, "steps, precision", precision, flush=True)
        with pytest.raises(GPError) as e:
            s.adjoint_backward(wphi, wmu)
        assert e.value.code == _abi.GP_E_NAN
        held = s.download()
        s.step(7)
        got = s.download()
    equal = lambda u, v: np.array_equal(u[0], v[0]) and np.array_equal(u[1], v[1])
    for n in (nsteps - 1, nsteps):
        with GPSolver(case.params, precision) as s:
            s.upload(case.phi, case.mu)
            s.step(n)
            if equal(held, s.download()):
                s.step(7)
                assert equal(got, s.download())
                return
    raise AssertionError("the state is none of the trajectory's last two")
