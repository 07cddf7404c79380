"""Device ABI parity: the HIP library against the CPU oracle and numpy closed
forms on identical inputs (buffers, Cholesky/PSD check, log-det, Schur
assembly, CG, Lanczos step length, primal recovery).  Tolerances: FP64 results
within 1e-10 relative of the oracle; Lanczos step lengths within 1e-8."""
import numpy as np
import pytest

import devtools as dt

pytestmark = pytest.mark.gpu

CASES = {
    # name: (n, m, kinds)
    "spr1_unit": (37, 45, [dt.SPR1]),
    "sparse_small": (41, 70, [dt.SPARSE]),
    "mixed_sparse": (66, 90, [dt.SPARSE, dt.SPR1, "SPARSE_BIG", "SPR1_BIG"]),
    "dense": (30, 40, [dt.DENSE]),
    "dsr1": (35, 50, [dt.DSR1]),
    "all_kinds_blocks": (130, 150, [dt.SPARSE, dt.SPR1, dt.DENSE, dt.DSR1, "SPARSE_BIG", dt.ZERO]),
    # single-entry constraints (edges, diagonal entries): the LDS pair kernel, with a
    # ragged last block of Schur columns (m not a multiple of 8) and, in the second
    # case, heavy rows and empty constraints among them
    "single_entry": (45, 121, ["SPARSE_ONE"]),
    "single_entry_heavy": (50, 150, ["SPARSE_ONE", "SPARSE_ONE", "SPARSE_BIG", dt.ZERO]),
}


def make_pair(gpu_lib, oracle, name, seed=0):
    n, m, kinds = CASES[name]
    rng = np.random.default_rng(seed)
    coeffs = dt.rand_coeffs(rng, n, m, kinds)
    return coeffs, dt.Dev(gpu_lib, coeffs), dt.Dev(oracle, coeffs), rng


def rel(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)


@pytest.mark.parametrize("name", list(CASES))
def test_buffer_factor_logdet(gpu_lib, oracle, name):
    coeffs, g, o, rng = make_pair(gpu_lib, oracle, name)
    y, eye = dt.interior_point(coeffs, rng)
    for d in (g, o):
        d.update(1.0, -1.0, y, eye, 0)
        assert d.factorize(0) == 1
    S = dt.dense_buffer(coeffs, 1.0, -1.0, y, eye)
    ld = np.linalg.slogdet(S)[1]
    assert abs(g.logdet(0) - ld) <= 1e-10 * max(1.0, abs(ld))
    assert abs(g.logdet(0) - o.logdet(0)) <= 1e-11 * max(1.0, abs(ld))
    # not positive definite: shift far below the smallest eigenvalue
    lam = np.linalg.eigvalsh(S).min()
    for d in (g, o):
        d.update(1.0, -1.0, y, eye - lam - 1.0, 1)
        assert d.factorize(1) == 0


@pytest.mark.parametrize("name", list(CASES))
def test_schur_matches_oracle_and_closed_form(gpu_lib, oracle, name):
    coeffs, g, o, rng = make_pair(gpu_lib, oracle, name, seed=1)
    y, eye = dt.interior_point(coeffs, rng)
    Rd = -0.37
    res = []
    for d in (g, o):
        d.update(1.0, -1.0, y, eye, 0)
        assert d.factorize(0) == 1
        a, b, t = d.schur(0, Rd)
        res.append((a, b, t, d.get_schur()))
    (ga, gb, gt, gM), (oa, ob, ot, oM) = res
    S = dt.dense_buffer(coeffs, 1.0, -1.0, y, eye)
    W = np.linalg.inv(S)
    A = [c.dense() for c in coeffs[1:]]
    M = np.array([[np.trace(Ai @ W @ Aj @ W) for Aj in A] for Ai in A])
    asinv = np.array([np.sum(Ai * W) for Ai in A])
    asrd = Rd * np.array([np.sum(Ai * (W @ W)) for Ai in A])
    assert rel(gM, M) < 1e-9
    assert rel(gM, oM) < 1e-10
    assert rel(ga, asinv) < 1e-9 and rel(ga, oa) < 1e-10
    assert rel(gb, asrd) < 1e-9 and rel(gb, ob) < 1e-10
    assert abs(gt - np.trace(W)) <= 1e-10 * abs(np.trace(W))
    # corrector: vectors only, M untouched
    for d in (g, o):
        a2, b2, t2 = d.schur(1, Rd)
        assert t2 == 0.0
    assert rel(g.get_schur(), gM) == 0.0


@pytest.mark.parametrize("name", list(CASES))
def test_hsd_terms_match_oracle_and_closed_form(gpu_lib, oracle, name):
    """The self-dual embedding's terms of a HOMOGENEOUS build (B = W C W):
    <A_i, B>, <C, W>, <C, B> and Rd tr(B) against numpy and the oracle."""
    coeffs, g, o, rng = make_pair(gpu_lib, oracle, name, seed=5)
    y, eye = dt.interior_point(coeffs, rng)
    Rd = -0.37
    res = []
    for d in (g, o):
        d.update(1.0, -1.0, y, eye, 0)
        assert d.factorize(0) == 1
        d.schur(2, Rd)
        res.append(d.hsd(Rd))
    (ga, gcs, gcsc, grd), (oa, ocs, ocsc, ord_) = res
    W = np.linalg.inv(dt.dense_buffer(coeffs, 1.0, -1.0, y, eye))
    Cm = coeffs[0].dense()
    B = W @ Cm @ W
    A = [c.dense() for c in coeffs[1:]]
    assert rel(ga, [np.sum(Ai * B) for Ai in A]) < 1e-9 and rel(ga, oa) < 1e-10
    for got, orc, ref in ((gcs, ocs, np.sum(Cm * W)), (gcsc, ocsc, np.sum(Cm * B)), (grd, ord_, Rd * np.trace(B))):
        scale = max(1.0, abs(ref), np.abs(Cm).max() * np.abs(W).sum())
        assert abs(got - ref) <= 1e-10 * scale and abs(got - orc) <= 1e-11 * scale


# (a zero constraint leaves M a zero row: "zero_diag" runs on the dense case only)
@pytest.mark.parametrize("name,mode", [("dense", "shift"), ("dense", "zero_diag"), ("all_kinds_blocks", "shift")])
def test_indefinite_schur_switches_to_lu(gpu_lib, oracle, name, mode):
    """The indefinite fallback: after the Cholesky switch fails on an indefinite M the
    device solves by LU with partial pivoting, the oracle by Bunch-Kaufman LDL^T; both
    match numpy's solve of that M, and each other."""
    coeffs, g, o, rng = make_pair(gpu_lib, oracle, name, seed=7)
    y, eye = dt.interior_point(coeffs, rng)
    res = []
    for d in (g, o):
        r = np.random.default_rng(11)
        res.append(dt.indefinite_fallback_run(d, coeffs, y, eye, r, mode))
    (gs, gm, gf0, gf1, _), (os_, om, of0, of1, _) = res
    assert (gf0, gf1) == (0, 1) and (of0, of1) == (0, 1)
    for (gx, rhs), (ox, _), A in zip(gs, os_, gm):
        ref = np.linalg.solve(A, rhs)
        bound = 1e-15 * np.linalg.cond(A) * 100
        assert np.linalg.norm(gx - ref) / np.linalg.norm(ref) <= bound
        assert np.linalg.norm(gx - ox) / np.linalg.norm(ox) <= 2 * bound


def test_indefinite_schur_switch_in_mixed_precision(gpu_lib):
    """The same switch on a mixed-precision device (dense constraints, whose Schur
    blocks come from bf16 split products): the LU solve runs on the FP64 M."""
    n, m, kinds = CASES["dense"]
    rng = np.random.default_rng(7)
    coeffs = dt.rand_coeffs(rng, n, m, kinds)
    d = dt.Dev(gpu_lib, coeffs, precision=1)
    y, eye = dt.interior_point(coeffs, rng)
    sols, mats, f0, f1, Mread = dt.indefinite_fallback_run(d, coeffs, y, eye, np.random.default_rng(11), "shift")
    assert (f0, f1) == (0, 1)
    d64 = dt.Dev(gpu_lib, coeffs, precision=0)
    d64.update(1.0, -1.0, y, eye, 0)
    assert d64.factorize(0) == 1
    d64.schur(0, 0.0)
    M64 = d64.get_schur()
    M64 = np.tril(M64) + np.tril(M64, -1).T
    for (x, rhs), A in zip(sols, mats):
        A = A - Mread + M64  # the same diagonal changes on the FP64 Schur matrix
        ref = np.linalg.solve(A, rhs)
        assert np.linalg.norm(x - ref) / np.linalg.norm(ref) <= 1e-15 * np.linalg.cond(A) * 100


@pytest.mark.parametrize("name", ["spr1_unit", "mixed_sparse", "all_kinds_blocks"])
def test_cg_solve(gpu_lib, oracle, name):
    coeffs, g, o, rng = make_pair(gpu_lib, oracle, name, seed=2)
    y, eye = dt.interior_point(coeffs, rng)
    m = len(coeffs) - 1
    diag = rng.uniform(0.1, 1.0, m)
    rhs = rng.standard_normal(m)
    sols = []
    for d in (g, o):
        d.update(1.0, -1.0, y, eye, 0)
        assert d.factorize(0) == 1
        d.schur(0, 0.0)
        d.add_diag(diag)
        d.regularize(1e-6)
        d.kkt_params(5e-12, 1e-12)
        assert d.kkt_factorize() == 0
        sols.append(d.kkt_solve(rhs))
    M = g.get_schur()
    x = np.linalg.solve(M, rhs)
    assert rel(sols[0], x) < 1e-7
    assert rel(sols[0], sols[1]) < 1e-7


@pytest.mark.parametrize("name", list(CASES))
def test_ratio_test_lanczos(gpu_lib, oracle, name):
    coeffs, g, o, rng = make_pair(gpu_lib, oracle, name, seed=3)
    y, eye = dt.interior_point(coeffs, rng)
    dy = rng.standard_normal(len(coeffs) - 1)
    steps = []
    for d in (g, o):
        d.update(1.0, -1.0, y, eye, 0)
        assert d.factorize(0) == 1
        d.update(0.0, -1.0, dy, 0.3, 2)
        steps.append([d.ratio(0), d.ratio(0)])  # second call warm-starts
    assert rel(steps[0], steps[1]) < 1e-8
    S = dt.dense_buffer(coeffs, 1.0, -1.0, y, eye)
    dS = dt.dense_buffer(coeffs, 0.0, -1.0, dy, 0.3)
    L = np.linalg.cholesky(S)
    Li = np.linalg.inv(L)
    lam = np.linalg.eigvalsh(Li @ (-dS) @ Li.T).max()
    if lam > 0:
        # the safeguarded Lanczos bound never oversteps the boundary S + a dS = 0
        assert steps[0][0] <= 1.0 / lam * (1 + 1e-8)
        assert np.linalg.eigvalsh(S + 0.999 * steps[0][0] * dS).min() > 0


@pytest.mark.parametrize("name", ["spr1_unit", "all_kinds_blocks"])
def test_axpy_and_primal_recovery(gpu_lib, oracle, name):
    coeffs, g, o, rng = make_pair(gpu_lib, oracle, name, seed=4)
    y, eye = dt.interior_point(coeffs, rng)
    m = len(coeffs) - 1
    dy = 0.01 * rng.standard_normal(m)
    out = []
    for d in (g, o):
        d.update(1.0, -1.0, y, eye, 0)
        assert d.factorize(0) == 1
        d.update(0.0, -1.0, dy, 0.0, 2)
        ok = d.axpy_check(0.5, 1)
        ld = d.logdet(1)
        d.update(1.0, -1.0, y, eye, 1)  # checker = S for the recovery
        assert d.primal(0.7, y, dy) == 1
        out.append((ok, ld, d.get_primal(), d.primal_stats()))
    (gok, gld, gX, gst), (ook, old, oX, ost) = out
    assert gok == ook == 1
    assert abs(gld - old) <= 1e-11 * max(1.0, abs(old))
    S = dt.dense_buffer(coeffs, 1.0, -1.0, y, eye)
    W = np.linalg.inv(S)
    dS = dt.dense_buffer(coeffs, 0.0, 1.0, dy, 0.0)
    X = 0.7 * (W + W @ dS @ W)
    assert rel(gX, X) < 1e-9 and rel(gX, oX) < 1e-10
    AX = np.array([np.sum(c.dense() * X) for c in coeffs[1:]])
    assert rel(gst[0], AX) < 1e-9
    assert abs(gst[1] - np.sum(coeffs[0].dense() * X)) <= 1e-9 * max(1.0, np.abs(X).sum())
    assert abs(gst[3] - np.trace(X)) <= 1e-10 * max(1.0, abs(np.trace(X)))


@pytest.mark.parametrize("name", ["dense", "dsr1"])
def test_schur_mixed_precision_gram(gpu_lib, name, monkeypatch):
    """Mixed precision builds the dense and rank-one Schur matrices from bf16 split
    products (three terms per operand, FP32-equivalent): within 1e-6 relative of the
    FP64 closed form (the two-term split reaches only ~3e-6); the right-hand sides
    stay FP64.  (Rank-one Gram blocks take the bf16 path only for r >= 32 n unless
    forced, as here.)"""
    monkeypatch.setenv("HDSDP_GRAM_BF16", "1")
    n, m, kinds = CASES[name]
    rng = np.random.default_rng(5)
    coeffs = dt.rand_coeffs(rng, n, m, kinds)
    y, eye = dt.interior_point(coeffs, rng)
    d = dt.Dev(gpu_lib, coeffs, precision=1)
    d.update(1.0, -1.0, y, eye, 0)
    assert d.factorize(0) == 1
    a, b, t = d.schur(0, -0.5)
    M = d.get_schur()
    W = np.linalg.inv(dt.dense_buffer(coeffs, 1.0, -1.0, y, eye))
    A = [c.dense() for c in coeffs[1:]]
    Mref = np.array([[np.sum(Ai * (W @ Aj @ W)) for Aj in A] for Ai in A])
    assert rel(M, Mref) < 1e-6
    assert rel(a, [np.sum(Ai * W) for Ai in A]) < 1e-10


@pytest.mark.parametrize("planes", ["1", "0"])
@pytest.mark.parametrize("n,m", [(260, 300), (130, 700), (37, 90)])
def test_dense_schur_mixed_planes(gpu_lib, n, m, planes, monkeypatch):
    """The mixed-precision dense Schur matrix from bf16 planes (L^-T and A_p split by the
    producing kernels, V_p = A_p L^-T written as planes by the product's epilogue, the
    packed T_p padded to a multiple of 32 with zeros): several 128-wide tiles with ragged
    edges (n = 260), the split-K Gram in parts plus a ragged last part (m = 700), and n not
    a multiple of 8 (n = 37, padded planes).  Within 1e-6 relative of the FP64 closed form
    and within 1e-6 of the FP64 device build.  Both mixed kernels: the planes (split once by
    the producers) and the products that split their FP32 operands in the loop."""
    monkeypatch.setenv("HDSDP_BF16_PLANES", planes)
    rng = np.random.default_rng(19)
    coeffs = dt.rand_coeffs(rng, n, m, [dt.DENSE])
    y, eye = dt.interior_point(coeffs, rng)
    out = []
    for prec in (1, 0):
        d = dt.Dev(gpu_lib, coeffs, precision=prec)
        d.update(1.0, -1.0, y, eye, 0)
        assert d.factorize(0) == 1
        d.schur(0, 0.0)
        out.append(d.get_schur())
        d.close()
    Mx, M64 = out
    W = np.linalg.inv(dt.dense_buffer(coeffs, 1.0, -1.0, y, eye))
    L = np.linalg.cholesky(W)
    T = np.stack([(L.T @ c.dense() @ L).ravel() for c in coeffs[1:]])
    Mref = T @ T.T
    print(n, m, "mixed vs closed form", rel(Mx, Mref), "vs fp64", rel(Mx, M64), flush=True)
    assert rel(Mx, Mref) < 1e-6
    assert rel(Mx, M64) < 1e-6


@pytest.mark.parametrize("n,m", [(260, 300), (130, 700)])
def test_dense_schur_large_tiles(gpu_lib, n, m):
    """Dense Schur matrices large enough for the 128-wide product kernels: the
    triangular T = L^-1 A L^-T products (16-byte loads, skipped zero k ranges, edge
    tiles) at n = 260, and the split-K Gram over lower tiles only (XCD-balanced
    launch) at m = 700.  Against the closed form within 1e-9 relative."""
    rng = np.random.default_rng(9)
    coeffs = dt.rand_coeffs(rng, n, m, [dt.DENSE])
    y, eye = dt.interior_point(coeffs, rng)
    g = dt.Dev(gpu_lib, coeffs)
    g.update(1.0, -1.0, y, eye, 0)
    assert g.factorize(0) == 1
    a, b, t = g.schur(0, 0.0)
    M = g.get_schur()
    W = np.linalg.inv(dt.dense_buffer(coeffs, 1.0, -1.0, y, eye))
    L = np.linalg.cholesky(W)
    T = np.stack([(L.T @ c.dense() @ L).ravel() for c in coeffs[1:]])
    Mref = T @ T.T
    assert rel(M, Mref) < 1e-9
    assert rel(a, [np.sum(c.dense() * W) for c in coeffs[1:]]) < 1e-9


def test_rank_one_buffer_split_k(gpu_lib):
    """The rank-m buffer update F diag(w) F^T of m = 4000 dense rank-one constraints at
    n = 300 runs as a k-split product (three k parts of 1344, 1344 and 1312 in one
    launch) and an in-order reduction of the partials: S = C - A^T y + eye I against
    the dense sum within 1e-11 relative."""
    rng = np.random.default_rng(12)
    coeffs = dt.rand_coeffs(rng, 300, 4000, [dt.DSR1])
    y = 0.1 * rng.standard_normal(4000)
    g = dt.Dev(gpu_lib, coeffs)
    try:
        g.update(1.0, -1.0, y, 0.7, 0)
        S = g.get_dual()
    finally:
        g.close()
    Sref = dt.dense_buffer(coeffs, 1.0, -1.0, y, 0.7)
    assert rel(S, Sref) < 1e-11


@pytest.mark.parametrize("m", [150, 700])
def test_cg_solve_lower_triangle_product(gpu_lib, oracle, m, monkeypatch):
    """CG on the one-pass product with M that reads only its lower triangle (the path
    of m >= 16384, forced here for every size): 256-row by 128-column tiles, ragged at
    both edges at m = 700, their partials added in a fixed order.  The solution against
    numpy's solve of the same M and against the oracle's CG, within 1e-7."""
    monkeypatch.setenv("HDSDP_SYMV_LOWER_MIN", "1")
    rng = np.random.default_rng(13)
    coeffs = dt.rand_coeffs(rng, 50, m, [dt.SPARSE, dt.SPR1, dt.DSR1])
    y, eye = dt.interior_point(coeffs, rng)
    diag = rng.uniform(0.1, 1.0, m)
    rhs = rng.standard_normal(m)
    g, o = dt.Dev(gpu_lib, coeffs), dt.Dev(oracle, coeffs)
    sols = []
    try:
        for d in (g, o):
            d.update(1.0, -1.0, y, eye, 0)
            assert d.factorize(0) == 1
            d.schur(0, 0.0)
            d.add_diag(diag)
            d.regularize(1e-6)
            d.kkt_params(5e-12, 1e-12)
            assert d.kkt_factorize() == 0
            sols.append(d.kkt_solve(rhs))
        M = g.get_schur()
    finally:
        g.close()
        o.close()
    x = np.linalg.solve(M, rhs)
    assert rel(sols[0], x) < 1e-7
    assert rel(sols[0], sols[1]) < 1e-7


# (these sizes take the step-by-step form; trailing updates on the second stream begin at 3073
# rows, in test_cholesky_block_edges)
@pytest.mark.parametrize("n", [257, 300, 520, 777])
def test_blocked_cholesky_look_ahead(gpu_lib, n):
    """The blocked Cholesky with look-ahead (n > 4 panels of 64): trailing updates of
    two panels per pass, odd and even panel counts, a ragged last panel.  log det S
    against numpy's slogdet within 1e-10 relative, and a matrix shifted below its
    smallest eigenvalue reported not positive definite."""
    rng = np.random.default_rng(n)
    coeffs = dt.rand_coeffs(rng, n, 12, [dt.DENSE])
    y, eye = dt.interior_point(coeffs, rng)
    g = dt.Dev(gpu_lib, coeffs)
    try:
        g.update(1.0, -1.0, y, eye, 0)
        assert g.factorize(0) == 1
        S = dt.dense_buffer(coeffs, 1.0, -1.0, y, eye)
        ld = np.linalg.slogdet(S)[1]
        assert abs(g.logdet(0) - ld) <= 1e-10 * max(1.0, abs(ld))
        lam = np.linalg.eigvalsh(S).min()
        g.update(1.0, -1.0, y, eye - lam - 1.0, 1)
        assert g.factorize(1) == 0
    finally:
        g.close()


def _spd_coeffs(n, rng, flip=None):
    """C = 4 I + a symmetric part of norm below 2.5 (condition below 5), two diagonal
    constraints; flip: index of a diagonal entry made negative."""
    G = rng.standard_normal((n, n)) / np.sqrt(n)
    S = 4.0 * np.eye(n) + 0.6 * (G + G.T) / np.sqrt(2.0)
    if flip is not None:
        S[flip, flip] = -1.0
    packed = np.concatenate([S[j:, j] for j in range(n)])
    one = np.ones(1)
    con = [dt.Coeff(dt.SPARSE, n, row=[k], col=[k], val=one) for k in (0, n - 1)]
    return S, [dt.Coeff(dt.DENSE, n, val=packed)] + con


# block (16), tile (64) and launch (48 tiles) edges of the blocked Cholesky
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 64, 65, 80, 127, 129, 500, 3072, 3073, 3140])
def test_cholesky_block_edges(gpu_lib, n):
    """Factor, log det and inverse entries of S at the edges of the blocked Cholesky.
    Bounds: n-term sums with unit roundoff u = 1.1e-16 and condition kappa < 5 give a
    relative error of the factor of n u, so |log det| moves by at most 2 n (n u kappa) and
    entries of S^-1 by (3 n u kappa) |S^-1|."""
    rng = np.random.default_rng(n)
    S, coeffs = _spd_coeffs(n, rng)
    d = dt.Dev(gpu_lib, coeffs)
    d.update(1.0, 0.0, np.zeros(2), 0.0, 0)
    assert d.factorize(0) == 1
    u = 1.1e-16
    assert abs(d.logdet(0) - np.linalg.slogdet(S)[1]) <= 10.0 * n * n * u + 1e-15
    a, _, _ = d.schur(1, 0.0)
    W = np.linalg.inv(S)
    assert np.max(np.abs(a - np.array([W[0, 0], W[-1, -1]]))) <= (15.0 * n + 20.0) * u
    d.close()


@pytest.mark.parametrize("n,flip", [(1, 0), (16, 15), (64, 0), (64, 16), (64, 63), (65, 64), (200, 137), (3100, 3080)])
def test_cholesky_flags_a_negative_pivot(gpu_lib, n, flip):
    """A negative diagonal entry in any 16-column block, tile or outer block of the Cholesky."""
    _, coeffs = _spd_coeffs(n, np.random.default_rng(n), flip)
    d = dt.Dev(gpu_lib, coeffs)
    d.update(1.0, 0.0, np.zeros(2), 0.0, 1)
    assert d.factorize(1) == 0
    d.update(1.0, 0.0, np.zeros(2), 8.0, 1)  # the shifted matrix is positive definite
    assert d.factorize(1) == 1
    d.close()


# one diagonal block, the first sizes with two, a ragged last block, and the wider span
@pytest.mark.parametrize("m", [2048, 2049, 2200, 4097, 10241])
def test_schur_solve_by_blocks(gpu_lib, m):
    """kkt_solve_exact (FP64 Cholesky of M, block substitution, two refinement steps) across
    the block edges of the substitution.  M = (S^-1)_ij^2 for single diagonal constraints
    plus a diagonal of 1: with S = 2 I + a rank-one part, cond(M) < 3, and a refined solve
    is accurate to a few m u cond (u = 1.1e-16)."""
    rng = np.random.default_rng(m)
    n = 160
    v = rng.standard_normal(n) / np.sqrt(n)
    S = 2.0 * np.eye(n) + np.outer(v, v)
    C = dt.Coeff(dt.DENSE, n, val=np.concatenate([S[j:, j] for j in range(n)]))
    r, c = np.tril_indices(n)
    pick = np.sort(rng.choice(len(r), size=m, replace=False))
    one = np.ones(1)
    d = dt.Dev(gpu_lib, [C] + [dt.Coeff(dt.SPARSE, n, row=[r[k]], col=[c[k]], val=one) for k in pick])
    d.update(1.0, 0.0, np.zeros(m), 0.0, 0)
    assert d.factorize(0) == 1
    d.schur(0, 0.0)
    d.add_diag(np.ones(m))
    W = np.linalg.inv(S)
    ri, ci = r[pick], c[pick]
    w = np.where(ri == ci, 1.0, 2.0)
    M = (W[np.ix_(ri, ri)] * W[np.ix_(ci, ci)] + W[np.ix_(ri, ci)] * W[np.ix_(ci, ri)]) * np.outer(w, w) / 2.0
    M[np.diag_indices(m)] += 1.0
    b = rng.standard_normal(m)
    x = np.zeros(m)
    assert gpu_lib.hdsdp_dev_kkt_solve_exact(d.h, dt._capi.dptr(b), dt._capi.dptr(x)) == 0
    d.close()
    res = np.linalg.norm(M @ x - b) / np.linalg.norm(b)
    assert res <= 12.0 * m * 1.1e-16


# FP64 dense Gram: the largest n of the old order, then the lower-triangle products with the
# T_p one after the other (few tiles) and in k panels, at ragged and whole tiles
@pytest.mark.parametrize("n,m", [(511, 20), (512, 20), (515, 530), (640, 513), (513, 1)])
def test_dense_gram_build(gpu_lib, n, m):
    """M(p, q) = <A_p, W A_q W> and <A_p, W> of dense constraints against numpy.  With
    condition kappa < 5 of S, products of n terms and Gram sums of n^2 / 2 terms round to
    (4 n + n^2 / 2) u kappa^2 |M| at worst (u = 1.1e-16); rounding errors add up as their
    root, and 25 n u |M| leaves a factor of ten over that."""
    rng = np.random.default_rng(n + m)
    S, (C, _, _) = _spd_coeffs(n, rng)
    d = dt.Dev(gpu_lib, [C] + [dt.rand_dense(rng, n) for _ in range(m)])
    d.update(1.0, 0.0, np.zeros(m), 0.0, 0)
    assert d.factorize(0) == 1
    a, _, _ = d.schur(0, 0.0)
    M = d.get_schur()
    W = np.linalg.inv(S)
    W = 0.5 * (W + W.T)
    L = np.linalg.cholesky(W)
    A = np.empty((m, n, n))
    T = np.empty((m, n * n))
    for k, c in enumerate(d.coeffs[1:]):
        A[k] = c.dense()
        T[k] = (L.T @ A[k] @ L).ravel()
    ref = T @ T.T
    d.close()
    u = 1.1e-16
    assert np.max(np.abs(M - ref)) <= 25.0 * n * u * np.max(np.abs(ref))
    assert np.max(np.abs(a - np.einsum("kij,ij->k", A, W))) <= 25.0 * n * u * np.sqrt(n) * np.max(np.abs(W))


# the one-workgroup forms of the Schur CG (m <= 256) and of Lanczos (n <= 160) and the first
# sizes past them; rows per lane change at multiples of 64
@pytest.mark.parametrize("n,m", [(2, 1), (63, 64), (64, 65), (128, 129), (129, 256), (160, 257), (161, 192)])
def test_small_cg_and_lanczos_edges(gpu_lib, oracle, n, m):
    """Jacobi CG solutions and two ratio tests (the second from the warm start) against the
    oracle's loops.  CG stops at a residual below 1e-11 |rhs| on both sides, so solutions
    agree to 2e-11 cond(M) < 1e-9 (the added diagonal keeps cond(M) below 10).  The two
    Lanczos runs of at most 30 steps differ by their rounding, held to 1e-6 here: the diagonal
    dS makes the spectrum's end well separated."""
    rng = np.random.default_rng(1000 * n + m)
    # single-entry constraints on distinct positions, the first ones on the diagonal
    r, c = np.tril_indices(n)
    pick = rng.permutation(len(r))[:m]
    one = np.ones(1)
    con = [dt.Coeff(dt.SPARSE, n, row=[r[k]], col=[c[k]], val=one) for k in pick]
    S, (C, _, _) = _spd_coeffs(n, rng)
    rhs = rng.standard_normal(len(con))
    dy = rng.standard_normal(len(con)) / np.sqrt(n)
    res = []
    for lib in (gpu_lib, oracle):
        d = dt.Dev(lib, [C] + con)
        d.kkt_params(1e-11, 1e-11, 200, -1)
        d.update(1.0, 0.0, np.zeros(len(con)), 0.0, 0)
        assert d.factorize(0) == 1
        d.schur(0, 0.0)
        d.add_diag(np.ones(len(con)))
        assert d.kkt_factorize() == 0
        x = d.kkt_solve(rhs)
        tiny = d.kkt_solve(1e-14 * rhs)  # below the tolerance: the solution stays as it was
        d.update(0.0, 1.0, dy, 0.0, 2)
        steps = [d.ratio(0), d.ratio(0)]
        res.append((x, tiny, steps))
        d.close()
    (gx, gt, gs), (ox, ot, os_) = res
    assert rel(gx, ox) < 1e-9
    assert np.all(gt == 0.0) and np.all(ot == 0.0)
    assert rel(gs, os_) < 1e-6


# edges of the 32-wide tiles and their slabs of 64 k, full and shorter last pairs of the
# triangular inverse's levels, and the first size whose S^-1 is formed in its lower half
@pytest.mark.parametrize("n", [2, 31, 32, 33, 64, 65, 96, 97, 129, 193, 257, 321, 449, 1280, 1281])
def test_products_on_small_tiles(gpu_lib, n):
    """S^-1 (through the Schur matrix of off-diagonal entries, which reads both triangles) and the
    primal recovery X = mu S^-1 (S + dS) S^-1 against numpy.  With condition kappa < 5 of S,
    the inverse and four products of n terms round to 30 n u kappa (u = 1.1e-16) relative to
    the largest entry at worst."""
    rng = np.random.default_rng(n)
    S, (C, _, _) = _spd_coeffs(n, rng)
    r, c = np.tril_indices(n)
    pick = rng.permutation(len(r))[:min(len(r), 40)]
    r, c, m = r[pick], c[pick], len(pick)
    one = np.ones(1)
    d = dt.Dev(gpu_lib, [C] + [dt.Coeff(dt.SPARSE, n, row=[r[k]], col=[c[k]], val=one) for k in range(m)])
    for which in (0, 1):
        d.update(1.0, 0.0, np.zeros(m), 0.0, which)
        assert d.factorize(which) == 1
    d.schur(0, 0.0)
    M = d.get_schur()
    W = np.linalg.inv(S)
    w = np.where(r == c, 1.0, 2.0)
    ref = (W[np.ix_(r, r)] * W[np.ix_(c, c)] + W[np.ix_(r, c)] * W[np.ix_(c, r)]) * np.outer(w, w) / 2.0
    tol = 150.0 * n * 1.1e-16
    assert np.max(np.abs(M - ref)) <= tol * np.max(np.abs(ref))
    dy = rng.standard_normal(m)
    dS = np.zeros((n, n))
    dS[r, c] = dy
    dS[c, r] = dy
    d.primal(0.5, np.zeros(m), dy)
    X = d.get_primal()
    d.close()
    want = 0.5 * (W + W @ dS @ W)
    assert np.max(np.abs(X - want)) <= tol * np.max(np.abs(want)) * max(1.0, np.linalg.norm(dS, 2))
    assert np.array_equal(X, X.T)


# rank-m updates of few tiles: one part, two, a shorter last part, whole and ragged tiles
@pytest.mark.parametrize("n,m", [(32, 1000), (33, 2049), (64, 3001), (101, 2050), (130, 5000)])
def test_rank_one_buffer_on_small_tiles(gpu_lib, n, m):
    """S = C - sum y_i s_i f_i f_i^T over dense rank-one constraints against numpy: sums of m
    terms, rounding to m u sum_i |y_i s_i f_i f_i^T| at worst (u = 1.1e-16)."""
    rng = np.random.default_rng(n + m)
    _, (C, _, _) = _spd_coeffs(n, rng)
    cons = [dt.rand_dsr1(rng, n) for _ in range(m)]
    y = rng.standard_normal(m)
    d = dt.Dev(gpu_lib, [C] + cons)
    d.update(1.0, -1.0, y, 0.0, 0)
    S = d.get_dual()
    d.close()
    F = np.array([c.val for c in cons])
    w = y * np.array([c.sign for c in cons])
    want = C.dense() - F.T @ (F * w[:, None])
    bound = np.abs(F).T @ (np.abs(F) * np.abs(w)[:, None])
    assert np.all(np.abs(S - want) <= 2.0 * m * 1.1e-16 * (bound + np.abs(want)))


# the T_p of small blocks, stored packed by 32- and 64-wide tiles: one tile, ragged tiles, many
@pytest.mark.parametrize("n,m", [(2, 3), (31, 2), (33, 40), (65, 70), (130, 200), (257, 90), (300, 450)])
def test_dense_gram_packed_tiles(gpu_lib, n, m):
    """The dense Gram build as above (same bounds) at the edges of the narrower tiles."""
    test_dense_gram_build(gpu_lib, n, m)


# the step with the next product in one launch (n <= 2048) and the separate launches past it
@pytest.mark.parametrize("n", [161, 255, 1023, 1025, 2048, 2049])
def test_lanczos_step_with_product(gpu_lib, n):
    """Two ratio tests (the second from the warm start) for dS = -e_0 e_0^T, where the largest
    step is 1 / (S^-1)_00.  The iteration stops once its bound on the eigenvalue is within
    1e-3 of the estimate and takes the larger one, so the step is at most the true one (up to
    rounding, n u kappa) and short of it by 1e-3 (1 / lambda) of it."""
    rng = np.random.default_rng(n)
    S, coeffs = _spd_coeffs(n, rng)
    d = dt.Dev(gpu_lib, coeffs)
    d.update(1.0, 0.0, np.zeros(2), 0.0, 0)
    assert d.factorize(0) == 1
    e0 = np.zeros(n)
    e0[0] = 1.0
    lam = np.linalg.solve(S, e0)[0]
    for _ in range(2):
        d.update(0.0, 1.0, np.array([-1.0, 0.0]), 0.0, 2)
        step = d.ratio(0)
        assert step <= (1.0 / lam) * (1.0 + 10.0 * n * 1.1e-16)
        assert step >= 1.0 / (lam + 1e-3) * (1.0 - 1e-9)
    d.close()


# entries per thread of the Jacobi CG's vector step, and the first size past them
@pytest.mark.parametrize("m", [1024, 1025, 2049, 3072, 4096, 4097, 6144, 6145])
def test_jacobi_cg_vector_step_edges(gpu_lib, m):
    """Jacobi CG to |r| < 1e-11 |b| on M + I of single-entry constraints against numpy's M x: cond
    < 3 and the recursive residual's drift of a few m u leave 1e-10 of |b|."""
    rng = np.random.default_rng(m)
    n = 120
    S, (C, _, _) = _spd_coeffs(n, rng)
    r, c = np.tril_indices(n)
    pick = np.sort(rng.choice(len(r), size=m, replace=False))
    one = np.ones(1)
    d = dt.Dev(gpu_lib, [C] + [dt.Coeff(dt.SPARSE, n, row=[r[k]], col=[c[k]], val=one) for k in pick])
    d.kkt_params(1e-11, 1e-11, 200, -1)
    d.update(1.0, 0.0, np.zeros(m), 0.0, 0)
    assert d.factorize(0) == 1
    d.schur(0, 0.0)
    d.add_diag(np.ones(m))
    assert d.kkt_factorize() == 0
    b = rng.standard_normal(m)
    x = d.kkt_solve(b)
    M = d.get_schur()
    d.close()
    assert np.linalg.norm(M @ x - b) <= 1e-10 * np.linalg.norm(b)


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 600])
def test_primal_dot_products(gpu_lib, n):
    """<X, S> and tr(X) of the recovered X against sums of its entries in numpy: n^2 terms in
    at most n + 300 additions each, relative to the sum of absolute values."""
    rng = np.random.default_rng(n)
    S, coeffs = _spd_coeffs(n, rng)
    d = dt.Dev(gpu_lib, coeffs)
    for which in (0, 1):
        d.update(1.0, 0.0, np.zeros(2), 0.0, which)
        assert d.factorize(which) == 1
    d.primal(0.5, np.zeros(2), np.zeros(2))
    X = d.get_primal()
    _, _, xs, tx = d.primal_stats()
    d.close()
    u = 1.1e-16
    assert abs(xs - np.sum(X * S)) <= (2.0 * n + 600.0) * u * np.sum(np.abs(X * S))
    assert abs(tx - np.trace(X)) <= (n + 300.0) * u * np.sum(np.abs(np.diag(X)))


# the edge of the one-workgroup sums (64 rows) and sizes of one to four passes
@pytest.mark.parametrize("n", [3, 31, 32, 33, 45, 46, 56, 63, 64, 65])
def test_primal_dot_products_of_small_blocks(gpu_lib, n):
    """The same sums as above (same bounds) where one workgroup takes them whole."""
    test_primal_dot_products(gpu_lib, n)
