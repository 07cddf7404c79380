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
