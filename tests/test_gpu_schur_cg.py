"""The Schur CG by its own counts: which of its ends a solve reached (convergence, the iteration
limit, no progress, not a number), after how many iterations and with which preconditioner,
against the same recurrences in numpy.  A wrong end would be repaired by the factorisation that
follows it and not show in the solution."""
import numpy as np
import pytest

import devtools as dt
from hdsdp_amd import _capi

pytestmark = pytest.mark.gpu

ONE = np.ones(1)


def _stats(d):
    s = np.zeros(7)
    assert d.lib.hdsdp_dev_stats(d.h, _capi.dptr(s), 7) == 0
    return {"cg": int(s[2]), "factored": int(s[4]), "last": int(s[5])}


def _system(lib, m, n, S, rng, precision=0, diag=1.0):
    """A device with the Schur matrix of m single-entry constraints, M_pq = <A_p, W A_q W> with
    W = S^-1, plus diag on its diagonal; and that matrix by numpy."""
    r, c = np.tril_indices(n)
    pick = np.sort(rng.choice(len(r), size=m, replace=False))
    C = dt.Coeff(dt.DENSE, n, val=np.concatenate([S[j:, j] for j in range(n)]))
    d = dt.Dev(lib, [C] + [dt.Coeff(dt.SPARSE, n, row=[r[k]], col=[c[k]], val=ONE) for k in pick], precision)
    d.update(1.0, 0.0, np.zeros(m), 0.0, 0)
    assert d.factorize(0) == 1
    d.schur(0, 0.0)
    d.add_diag(diag * np.ones(m))
    W = np.linalg.inv(S)
    ri, ci = r[pick], c[pick]
    w = np.where(ri == ci, 1.0, 2.0)
    M = (W[np.ix_(ri, ri)] * W[np.ix_(ci, ci)] + W[np.ix_(ri, ci)] * W[np.ix_(ci, ri)]) * np.outer(w, w) / 2.0
    M[np.diag_indices(m)] += diag
    return d, M


def _mild(n, rng):
    G = rng.standard_normal((n, n)) / np.sqrt(n)
    return 4.0 * np.eye(n) + 0.6 * (G + G.T) / np.sqrt(2.0)


def _spread(n, rng, decades):
    """Eigenvalues over so many decades."""
    Q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    S = (Q * np.logspace(0, -decades, n)) @ Q.T
    return 0.5 * (S + S.T)


def _jacobi_cg(M, b, rel, absol, maxit):
    """(end, iterations) of Jacobi CG with a restart from the true residual at iter % 20 == 5."""
    jac, r, x = np.diag(M).copy(), b.copy(), np.zeros(len(b))
    bnorm = np.linalg.norm(b)
    tol = max(min(absol, bnorm * rel), 0.1 * absol)
    z = r / jac
    p = z.copy()
    Mp = M @ p
    for it in range(maxit):
        rz = z @ r
        alpha = rz / (p @ Mp)
        x += alpha * p
        if it % 20 == 5:
            r = b - M @ x
            z = r / jac
            p = z.copy()
            Mp = M @ p
            continue
        r = r - alpha * Mp
        z = r / jac
        p = z + (r @ z) / rz * p
        Mp = M @ p
        nrm = np.linalg.norm(r)
        if it > 20 and nrm > 0.01 * bnorm:
            return "stalled", it + 1
        if nrm < tol:
            return "converged", it + 1
    return "limit", maxit


# one workgroup (m <= 256: 64 rows per lane and register, columns in LDS from 193), vector
# steps in registers (1024 entries each, up to 6144) and the loops beyond; queued batches change
# at 2048, 4096 and 8192
@pytest.mark.parametrize("m", [1, 2, 63, 64, 65, 128, 129, 192, 193, 255, 256, 257, 1024, 1025, 2048, 2049, 3073, 4097,
                               6144, 6145, 8193])
def test_converges_as_numpy_does(gpu_lib, m):
    """|r| < 1e-11 |b| after numpy's number of iterations, one more or less where rounding
    decides, past a restart, without a factorisation; the solution is checked to 1e-10 |b|
    (recurrence drift of a few m u, cond < 3)."""
    rng = np.random.default_rng(m)
    n = max(2, int(np.ceil(np.sqrt(2.2 * m))))
    d, M = _system(gpu_lib, m, n, _mild(n, rng), rng)
    b = rng.standard_normal(m)
    absol = 1e-11 * np.linalg.norm(b)
    d.kkt_params(1e-11, absol, 200, -1)
    assert d.kkt_factorize() == 0
    before = _stats(d)
    x = d.kkt_solve(b)
    got, ldl = _stats(d), d.uses_ldl()
    d.close()
    end, steps = _jacobi_cg(M, b, 1e-11, absol, 200)
    assert end == "converged" and (steps > 6 or m <= 2)
    assert abs(got["cg"] - before["cg"] - steps) <= 1 and got["factored"] == before["factored"] and ldl == 0
    assert np.linalg.norm(M @ x - b) <= 1e-10 * np.linalg.norm(b)


# limits before, at and after the restarts (iterations 5 and 25), within and at the ends of the
# queued batches
@pytest.mark.parametrize("limit", [1, 3, 5, 6, 7, 10, 12, 25, 26, 27])
@pytest.mark.parametrize("m", [65, 256, 257, 3000, 7000])
def test_iteration_limit_switches_to_the_factor(gpu_lib, m, limit):
    """A Jacobi CG that runs out of its iterations: all of them counted, then one factorisation
    and a step or two with it, for this right-hand side and the next one alike.  cond M is
    about 100: the factor's steps and numpy's M leave a few hundred m u of |b|."""
    rng = np.random.default_rng(m)
    n = int(np.ceil(np.sqrt(2.2 * m)))
    d, M = _system(gpu_lib, m, n, _spread(n, rng, 1), rng, diag=0.0)
    b = rng.standard_normal(m)
    rel = 1e-11
    absol = rel * np.linalg.norm(b)
    assert _jacobi_cg(M, b, rel, absol, limit) == ("limit", limit)
    d.kkt_params(rel, absol, limit, -1)
    assert d.kkt_factorize() == 0
    before = _stats(d)
    sols = []
    for rhs in (b, -2.0 * b):
        sols.append(d.kkt_solve(rhs))
    got, ldl = _stats(d), d.uses_ldl()
    d.close()
    # one step of the factor's CG is enough, so limit 1 leaves it one as well
    assert ldl == 0 and got["factored"] == before["factored"] + 1
    assert limit + 2 <= got["cg"] - before["cg"] <= limit + 4
    for rhs, x in zip((b, -2.0 * b), sols):
        assert np.linalg.norm(M @ x - rhs) <= 1e-10 * np.linalg.norm(rhs)


@pytest.mark.parametrize("m", [150, 256, 300, 2500])
def test_no_progress_switches_to_the_factor(gpu_lib, m):
    """Above a hundredth of the start after 21 iterations: 22 iterations, then the factor.  W has
    eigenvalues from 1 to 1e5, which Jacobi scaling does not mend; the factor solves to the
    tolerance, and numpy's M carries W's rounding, n u cond S = 1e-9, on top."""
    rng = np.random.default_rng(m)
    n = int(np.ceil(np.sqrt(2.2 * m)))
    d, M = _system(gpu_lib, m, n, _spread(n, rng, 5), rng, diag=0.0)
    b = rng.standard_normal(m)
    absol = 1e-9 * np.linalg.norm(b)
    assert _jacobi_cg(M, b, 1e-9, absol, 400) == ("stalled", 22)
    d.kkt_params(1e-9, absol, 400, -1)
    assert d.kkt_factorize() == 0
    before = _stats(d)
    x = d.kkt_solve(b)
    got, ldl, Md = _stats(d), d.uses_ldl(), d.get_schur()
    d.close()
    assert ldl == 0 and got["factored"] == before["factored"] + 1
    assert got["cg"] - before["cg"] - 22 <= 20 and got["last"] < 20
    assert np.linalg.norm(Md @ x - b) <= 1e-8 * np.linalg.norm(b)


@pytest.mark.parametrize("m", [100, 256, 300, 2500, 7000])
def test_not_a_number_switches_to_the_direct_solver(gpu_lib, m):
    """A zero on M's diagonal makes the Jacobi preconditioner infinite and the residual NaN: the
    indefinite solver takes the system over and solves this right-hand side."""
    rng = np.random.default_rng(m)
    n = int(np.ceil(np.sqrt(2.2 * m)))
    d, M = _system(gpu_lib, m, n, _mild(n, rng), rng)
    delta = np.zeros(m)
    delta[m // 3] = -d.get_schur()[m // 3, m // 3]
    d.add_diag(delta)
    M[m // 3, m // 3] = 0.0
    b = rng.standard_normal(m)
    d.kkt_params(1e-11, 1e-11, 100, -1)
    assert d.kkt_factorize() == 0 and d.uses_ldl() == 0
    x = d.kkt_solve(b)
    ldl = d.uses_ldl()
    d.close()
    assert ldl == 1
    assert np.linalg.norm(M @ x - b) <= 1e-9 * np.linalg.norm(b)


# diagonal blocks of 2048 rows and of 4096 (m = 10241), outer blocks of the FP32 Cholesky
@pytest.mark.parametrize("m", [2048, 2049, 3073, 4097, 10241])
def test_fp32_factor_by_blocks(gpu_lib, monkeypatch, m):
    """Mixed precision with the FP32 factor of an FP64-built M (from m = 65536 by itself): the
    factor's CG takes more than one iteration, which the FP64 factor never does, so the last
    solve was not the fallback's; the residual is confirmed in FP64, 1e-11 |b|, to which numpy's
    M adds 12 m u as above."""
    monkeypatch.setenv("HDSDP_MIXED_CHOL32_MIN", "1")
    rng = np.random.default_rng(m)
    n = int(np.ceil(np.sqrt(2.2 * m)))
    d, M = _system(gpu_lib, m, n, _mild(n, rng), rng, precision=1)
    b = rng.standard_normal(m)
    rel = 1e-11
    d.kkt_params(rel, rel * np.linalg.norm(b), 5, -1)
    assert _jacobi_cg(M, b, rel, rel * np.linalg.norm(b), 5)[0] == "limit"
    assert d.kkt_factorize() == 0
    before = _stats(d)
    sols = []
    for rhs in (b, -2.0 * b):
        sols.append(d.kkt_solve(rhs))
        got = _stats(d)
        assert got["factored"] == before["factored"] + 1 and d.uses_ldl() == 0
        assert 1 <= got["last"] < 5
    d.close()
    for rhs, x in zip((b, -2.0 * b), sols):
        assert np.linalg.norm(M @ x - rhs) <= (rel + 12.0 * m * 1.1e-16) * np.linalg.norm(rhs)


def test_fp32_factor_by_blocks_of_a_bf16_schur_matrix(gpu_lib):
    """The same factor of a dense Schur matrix from the bf16 products at m > 2048, where mixed
    precision takes it by itself: solves refined against the exact operator, to 1e-11 |b| here."""
    n, m = 70, 2100
    rng = np.random.default_rng(7)
    S = _mild(n, rng)
    C = dt.Coeff(dt.DENSE, n, val=np.concatenate([S[j:, j] for j in range(n)]))
    d = dt.Dev(gpu_lib, [C] + [dt.rand_dense(rng, n) for _ in range(m)], 1)
    d.update(1.0, 0.0, np.zeros(m), 0.0, 0)
    assert d.factorize(0) == 1
    d.schur(0, 0.0)
    d.add_diag(0.1 * np.ones(m))
    W = np.linalg.inv(S)
    L = np.linalg.cholesky(0.5 * (W + W.T))
    T = np.array([(L.T @ c.dense() @ L).ravel() for c in d.coeffs[1:]])
    M = T @ T.T + 0.1 * np.eye(m)
    b = rng.standard_normal(m)
    rel = 1e-11
    d.kkt_params(rel, rel * np.linalg.norm(b), 8, -1)
    assert _jacobi_cg(M, b, rel, rel * np.linalg.norm(b), 8)[0] == "limit"
    assert d.kkt_factorize() == 0
    before = _stats(d)
    x = d.kkt_solve(b)
    got, ldl = _stats(d), d.uses_ldl()
    d.close()
    assert got["factored"] == before["factored"] + 1 and ldl == 0
    assert np.linalg.norm(M @ x - b) <= (rel + 12.0 * m * 1.1e-16) * np.linalg.norm(b)


# first size in blocks, ragged last pairs of the whole inverse's levels, the wider span
@pytest.mark.parametrize("m", [2048, 2049, 2500, 4097, 6200, 10241])
def test_repeated_exact_solves(gpu_lib, m):
    """kkt_solve_exact again and again with one factor, past the point (m / 400) where the inverse
    of the factor is completed, then the CG with that factor, then a new factor: 12 m u of
    |b| for the refined solves as in test_schur_solve_by_blocks, the tolerance for the CG."""
    rng = np.random.default_rng(m)
    n = int(np.ceil(np.sqrt(2.2 * m)))
    d, M = _system(gpu_lib, m, n, _mild(n, rng), rng)
    x = np.zeros(m)

    def exact(b):
        assert gpu_lib.hdsdp_dev_kkt_solve_exact(d.h, _capi.dptr(b), _capi.dptr(x)) == 0
        return np.linalg.norm(M @ x - b) / np.linalg.norm(b)

    for _ in range(m // 400 + 3):
        assert exact(rng.standard_normal(m)) <= 12.0 * m * 1.1e-16
    rel = 1e-11
    b = rng.standard_normal(m)
    # a Jacobi CG of one iteration, then the factor of the same M
    d.kkt_params(rel, rel * np.linalg.norm(b), 1, -1)
    assert d.kkt_factorize() == 0
    y = d.kkt_solve(b)
    assert np.linalg.norm(M @ y - b) <= (rel + 12.0 * m * 1.1e-16) * np.linalg.norm(b)
    d.add_diag(np.ones(m))
    M[np.diag_indices(m)] += 1.0
    for _ in range(2):
        assert exact(rng.standard_normal(m)) <= 12.0 * m * 1.1e-16
    assert d.uses_ldl() == 0
    d.close()
