"""delta-phi and the face currents by present pairs and solids (microsim_amd/csrc/gp_pairs.h) equal the full loops over
ordered pairs and solids (gp_model.h) bit for bit: cells with one to four phases, absent phases, zero gradients, negative
and clamped phi, both potentials, with and without anisotropy, symmetric and unsymmetric coefficients, and non-finite
values."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from gp_testlib import REPO, golden_cases, load_golden
from microsim_amd import _abi


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("pairs") / "libpairs.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off",
                    "-I" + os.path.join(REPO, "include"), "-I" + os.path.join(REPO, "microsim_amd", "csrc"),
                    "-o", out, os.path.join(REPO, "tests", "cpu_model", "pairs_check.cpp")], check=True)
    lib = C.CDLL(out)
    lib.pairs_check.argtypes = [C.POINTER(_abi.GPParams), C.c_int, _abi._dp, _abi._dp]
    lib.pairs_check_vjp.argtypes = [C.POINTER(_abi.GPParams), _abi._dp, _abi._dp]
    return lib


def _params(rng, N, NC):
    """Random finite parameters of N phases and NC mu fields (dx, dy powers of two)."""
    p = _abi.GPParams.from_buffer_copy(load_golden(golden_cases()[0])[0].params)
    P, NCM = _abi.P, _abi.NCM
    p.nphases, p.ncomp, p.dx, p.dy, p.dt, p.epsilon = N, NC + 1, 1.0, 2.0, 0.01, 4.0
    p.tau = 0.3
    p.solve, p.fn_aniso, p.fn_w = 0, int(rng.integers(0, 2)), int(rng.integers(1, 3))
    for a in range(N):
        for b in range(a + 1, N):
            t, g = rng.uniform(0, 6.28), rng.uniform(0.5, 2.0)
            rot = [np.cos(t), -np.sin(t), np.sin(t), np.cos(t)]
            for i, j in ((a, b), (b, a)):
                p.gamma[i * P + j], p.dab[i * P + j], p.tau_ab[i * P + j] = g, 0.02 * g, 0.3 * g
                for q in range(4):
                    p.rot[(i * P + j) * 4 + q], p.rot_inv[(i * P + j) * 4 + q] = rot[q], rot[(0, 2, 1, 3)[q]]
        for k in range(NC):
            p.B[a * NCM + k], p.Beq[a * NCM + k] = rng.normal(), rng.normal()
            for q in range(NC):
                p.diffusivity[(a * NCM + k) * NCM + q] = rng.uniform(0.1, 1.0) if k == q else 0.0
                p.A[(a * NCM + k) * NCM + q] = rng.uniform(0.5, 1.0)
                p.cmu[(a * NCM + k) * NCM + q] = rng.uniform(0.2, 1.0) if k == q else rng.uniform(-0.1, 0.1)
    for i in range(P ** 3):
        p.gamma_abc[i] = rng.uniform(0.0, 2.0)
    return p


def _cell(rng, N, NC, kind):
    """phi [N, 9], mu [NC, 5], delta-phi [N, 5] and y of one cell in which a random number of phases is present."""
    live = rng.permutation(N)[:rng.integers(1, N + 1)]
    phi = np.zeros((N, 9))
    phi[live] = rng.uniform(0.0, 1.0, (len(live), 9)) ** 2
    if kind == "sharp":
        phi[live] = np.where(rng.uniform(size=(len(live), 9)) < 0.5, np.round(phi[live]), phi[live])
    phi[live[0]] += 1.0 - phi.sum(0)
    if kind == "flat":
        phi[:] = phi[:, 4:5]
    if kind == "wild":
        phi[live] = rng.normal(0.3, 0.7, (len(live), 9))
    mu = rng.normal(0.0, 0.3, (NC, 5))
    d = np.zeros((N, 5))
    d[live] = np.where(rng.uniform(size=(len(live), 5)) < 0.3, 0.0, rng.normal(0.0, 0.01, (len(live), 5)))
    if kind == "nonfinite":
        phi[rng.integers(N), rng.integers(9)] = rng.choice([np.inf, -np.inf, np.nan])
    return np.concatenate([phi.ravel(), mu.ravel(), d.ravel(), [float(rng.integers(0, 30))]])


@pytest.mark.parametrize("form", [0, 1, 2, 3])
@pytest.mark.parametrize("shape", [(2, 1), (3, 2), (4, 2), (3, 3)])
@pytest.mark.parametrize("sym", [True, False])
def test_pairs_equal_the_full_loops(lib, shape, form, sym):
    rng = np.random.default_rng(100 * form + 10 * shape[0] + shape[1])
    out = np.zeros(64)
    for _ in range(40):
        p = _params(rng, *shape)
        if not sym:
            p.rot[_abi.P * 4] += 0.25
            p.gamma[1] *= 1.5
        p.jat_skip_row = int(rng.integers(0, 30))
        for kind in ("smooth", "sharp", "flat", "wild", "nonfinite"):
            for _ in range(6):
                n = lib.pairs_check(C.byref(p), form, _abi.dptr(_cell(rng, *shape, kind)), _abi.dptr(out))
                assert n == 2 * (shape[0] + 4 * shape[1])
                r = out[:n].reshape(-1, 2)
                if kind == "nonfinite":
                    assert np.array_equal(np.isfinite(r[:, 0]), np.isfinite(r[:, 1]))
                    r = r[np.isfinite(r[:, 0])]
                assert np.array_equal(r[:, 0], r[:, 1]), (kind, r)


@pytest.mark.parametrize("shape", [(2, 1), (3, 2), (4, 2), (3, 3)])
@pytest.mark.parametrize("sym", [True, False])
def test_transposed_pairs_match_the_full_loops(lib, shape, sym):
    """The joined terms of (a, b) and (b, a) are sums of the same products in another order: a few hundred roundings of
    terms that may cancel, so 1e-11 of the largest entry of the group (stencil and mu, or theta)."""
    rng = np.random.default_rng(7 + 10 * shape[0] + shape[1])
    N, NC = shape
    out, compared = np.zeros(256), 0
    for _ in range(40):
        p = _params(rng, N, NC)
        if not sym:
            p.rot[_abi.P * 4] += 0.25
            p.gamma[1] *= 1.5
        for kind in ("smooth", "sharp", "flat", "wild"):
            for _ in range(6):
                cell = np.concatenate([_cell(rng, N, NC, kind), rng.normal(0.0, 1.0, N)])
                n = lib.pairs_check_vjp(C.byref(p), _abi.dptr(cell), _abi.dptr(out))
                r = out[:n].reshape(-1, 2)
                # a non-finite derivative (tau = 0 / 0, a projection over a zero sum) shows in both forms
                assert np.isfinite(r[:, 0]).all() == np.isfinite(r[:, 1]).all()
                if not np.isfinite(r).all():
                    continue
                compared += 1
                for part in (r[:9 * N + NC], r[9 * N + NC:]):
                    scale = np.abs(part).max()
                    assert np.abs(part[:, 0] - part[:, 1]).max() <= 1e-11 * scale, (kind, part)
    assert compared > 800
