"""The Poisson solve away from the reference's settings: Anderson steps farther
apart than the host looks at the solve, none at all, and a start that is already
converged."""
import ctypes as C
import time

import numpy as np
import pytest

import helpers as H
import oracle as O
from sqdft_amd import _lib as L
from sqdft_amd.scf import SCF

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def al():
    S = H.test_al()[0]
    scf = SCF(S)
    pc = S.pseudocharge()
    yield S, scf, pc["b"] + pc["rho"]
    scf.close()


def solve(scf, rhs, guess, tol, maxiter, beta, m, p):
    phi, it, rr = np.zeros_like(rhs), C.c_int(), C.c_double()
    code = scf._lib.sqg_poisson_aaj(scf.sq._ctx, L.dptr(rhs), L.dptr(guess), tol, maxiter, beta, m, p, L.dptr(phi),
                                    C.byref(it), C.byref(rr))
    return code, phi, it.value, rr.value


def relative_residual(info, phi, rhs):
    """||phi's Jacobi residual|| / (4 pi ||rhs|| / |3 lap0|) in FP64, x fastest."""
    n, lap = info["n"], info["coeff_lap"]
    f = phi.reshape(n, n, n)
    lp = 3 * lap[0] * f
    for a in range(1, info["FDn"] + 1):
        for ax in range(3):
            lp = lp + lap[a] * (np.roll(f, a, ax) + np.roll(f, -a, ax))
    r = 4 * np.pi * rhs.reshape(n, n, n) + lp
    return np.linalg.norm(r) / np.linalg.norm(4 * np.pi * rhs)


@pytest.mark.parametrize("m,p", [(7, 16), (7, 17), (3, 40)])
def test_sparse_anderson_steps(al, m, p):
    """The oracle's count, and a phi whose residual is the one reported, below
    the tolerance: 1e-6 of it, a residual of 1e-6 being the difference of terms of
    order one that rounding leaves to 1e-14.  (The iterates themselves are not
    compared: Anderson steps over nearly dependent differences amplify rounding.)"""
    print("poisson", m, p, flush=True)
    S, scf, rhs = al
    pp, info = S.poisson_params(), S.info
    lap = info["coeff_lap"][: info["FDn"] + 1]
    _, oit, _ = O.poisson_aaj(info["n"], info["FDn"], lap, rhs, np.ones(S.nn), 1e-6, 400, pp["beta"], m, p)
    code, phi, it, rr = solve(scf, rhs, np.ones(S.nn), 1e-6, 400, pp["beta"], m, p)
    assert code == 0 and it == oit and rr <= 1e-6
    assert abs(relative_residual(info, phi, rhs) - rr) <= 1e-6 * rr


@pytest.mark.parametrize("maxiter", [1, 15, 16, 17, 33])
def test_plain_relaxation_matches_oracle(al, maxiter):
    """No Anderson step at all: same count, residual to 1e-6 and phi to 1e-10 (the
    suite's bounds for this solver)."""
    print("plain relaxation", maxiter, flush=True)
    S, scf, rhs = al
    info = S.info
    lap = info["coeff_lap"][: info["FDn"] + 1]
    ref, oit, orr = O.poisson_aaj(info["n"], info["FDn"], lap, rhs, np.ones(S.nn), 1e-6, maxiter, 0.6, 2, 1000)
    code, phi, it, rr = solve(scf, rhs, np.ones(S.nn), 1e-6, maxiter, 0.6, 2, 1000)
    assert code == 0 and it == oit and abs(rr - orr) <= 1e-6 * orr
    assert H.rel(phi, ref) < 1e-10


def test_converged_start_does_not_pay_for_maxiter(al):
    """With no Anderson step due, a start that meets the tolerance returns after
    one iteration: 100,000 enqueued ones would take more than 0.3 s."""
    S, scf, rhs = al
    pp = S.poisson_params()
    code, phi, _, _ = solve(scf, rhs, np.ones(S.nn), 1e-8, 2000, pp["beta"], pp["m"], pp["p"])
    assert code == 0
    for _ in range(2):
        t = time.perf_counter()
        code, _, it, _ = solve(scf, rhs, phi, 1e-6, 100000, pp["beta"], pp["m"], 10 ** 6)
        t = time.perf_counter() - t
        print("converged start", t, flush=True)
        assert code == 0 and it == 1
    assert t < 0.1


@pytest.mark.parametrize("tol", [0.0, -1.0, float("nan"), float("inf"), 1e17])
def test_tolerances_that_ask_for_no_iteration_are_refused(al, tol):
    S, scf, rhs = al
    for maxiter in (1, 100):
        code, phi, it, _ = solve(scf, rhs, np.ones(S.nn), tol, maxiter, 0.6, 7, 6)
        assert code == -1 and it == 0 and not phi.any()   # SQG_E_ARG, nothing written
