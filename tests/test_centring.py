"""Centring (HDSDPCenter) of starts that are close to the boundary of S(y) > 0 or far from
the centre, on the CPU oracle and on the GPU, checked with numpy: the centre's residual
b - mu A(S^-1) is what the call promises to make small."""
import numpy as np
import pytest

from hdsdp_amd import instances as I
from hdsdp_amd.solver import Solver


@pytest.fixture(params=["oracle", pytest.param("gpu_lib", marks=pytest.mark.gpu)])
def lib(request):
    return request.getfixturevalue(request.param)


def _residual(inst, mu, y):
    """||b - mu A(S^-1)|| / (1 + ||b||) of S = C - sum y_i A_i."""
    A = [inst.dense_coeff(k) for k in range(inst.m + 1)]
    S = A[0] - sum(yk * Ak for yk, Ak in zip(y, A[1:]))
    W = np.linalg.inv(S)
    g = inst.b - mu * np.array([np.sum(Ak * W) for Ak in A[1:]])
    return np.linalg.norm(g) / (1.0 + np.linalg.norm(inst.b))


def _start(family):
    if family == "theta":
        inst = I.lovasz_theta(22, 0.3, 0)
        y = np.zeros(inst.m)
        y[0] = -inst.n * 1.001
        return inst, y, 1e-5
    inst = I.maxcut(40, 0.3, 0, "unif")
    return inst, 2.0 * np.diag(inst.dense_coeff(0)) - 1.0, 1e-6


@pytest.mark.parametrize("family", ["theta", "maxcut"])
def test_far_starts_reach_the_centre(lib, family):
    """The guaranteed step 1 / (1 + delta) centres these starts in 57 and 38 Newton systems; a
    longer step must not run out of the 60 allowed.  The call succeeds with a residual of
    at most 1e-5, its own limit; numpy's S^-1 (cond S below 1e8) adds less than 1e-6 to it."""
    inst, y0, mu = _start(family)
    with Solver(lib, inst, relopt=1e-8, absopt=1e30) as s:
        s.setup()
        y, steps, res = s.center(mu, y0, tol=1e-10)
    assert steps <= 60 and res <= 1e-5
    assert _residual(inst, mu, y) <= 1.1e-5


def test_centred_start_is_returned_as_it_is(lib):
    """A start whose residual is half the tolerance takes no Newton step and comes back unchanged."""
    inst, y0, mu = _start("maxcut")
    with Solver(lib, inst, relopt=1e-8, absopt=1e30) as s:
        s.setup()
        y, _, _ = s.center(mu, y0, tol=1e-10)
        near = y * (1.0 + 1e-10)
        tol = 2.0 * _residual(inst, mu, near)
        assert 1e-10 < tol < 1e-2  # far above rounding
        again, steps, res = s.center(mu, near, tol=tol)
    assert steps == 0 and res <= tol
    assert np.array_equal(again, near)


@pytest.mark.parametrize("n,seed,mu,tol", [(24, 3, 1e-4, 1e-12), (26, 4, 1e-5, 1e-11)])
def test_one_step_below_the_tolerance_at_most(oracle, capfd, monkeypatch, n, seed, mu, tol):
    """After longer steps one more full step follows the first residual below tol and no other,
    also where rounding lifts the residual above tol again (tolerances at rounding level)."""
    monkeypatch.setenv("HDSDP_TRACE_CENTER", "1")
    inst = I.maxcut(n, 0.3, seed, "unif")
    with Solver(oracle, inst, relopt=1e-8, absopt=1e30) as s:
        s.setup()
        _, steps, res = s.center(mu, 2.0 * np.diag(inst.dense_coeff(0)) - 1.0, tol=tol)
    start = [float(line.split("residual")[1].split()[0]) for line in capfd.readouterr().err.splitlines()
             if line.startswith("[hdsdp] centre step")]
    assert len(start) == steps and res <= tol
    assert all(r > tol for r in start[:-1])  # residuals the steps but the last were taken from
