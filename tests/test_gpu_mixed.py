"""Mixed precision against the plain FP64 GPU path on the same instances, solved
to a 1e-6 relative gap.

Two kinds of instance:
  * sparse constraints (MaxCut, theta), and rank-one constraints with r < 32 n:
    M is built in FP64 and only its preconditioner may be FP32 (equilibrated
    Cholesky; from m = 65536 by itself, below where HDSDP_MIXED_CHOL32_MIN says
    so, otherwise the run is the FP64 one); the CG stops on FP64 residuals at
    the reference's tolerances, so the iterates agree to the solve tolerance:
    same status and iteration count;
  * dense constraints (and rank-one ones when forced onto the bf16 Gram
    path): the Gram blocks of M come from bf16 split products (three terms per
    operand, FP32-equivalent, FP64 accumulation); once the factor preconditioner
    is in use each Newton system is refined against the exact FP64 Schur operator
    applied matrix-free (corrections from CG on the bf16-built M), so the
    directions carry FP64 accuracy; when such an M cannot be factored, or the
    refinement stalls above 1e-13 of ||b||, the library rebuilds M in FP64 and
    stays there.  The trajectory may still differ from FP64 by an iteration.
All must end optimal with objectives within 1e-8 relative of the FP64 run and
y* within 1e-7, except on two rank-one instances, bound 1e-6:
  * rankone_n60_m500, whose y* at a 1e-6 gap is determined only to ~1e-7: the
    FP64 GPU run and the reference HDSDP differ by 2.2e-7 on it, and its
    trajectory is ulp-sensitive (a last-bit change in the factorisation moves
    the mixed-vs-FP64 distance between 1.5e-8 and 2.5e-7);
  * the rank-one instance forced onto the bf16 Gram path: there the solves are
    refined against the exact operator from the first iteration, where the FP64 path starts with
    Jacobi-CG solves accurate to 1e-6, and the two end 5e-7 apart in y
    (measured: FP64 GPU vs reference HDSDP 3.8e-8, forced bf16 vs reference
    5.1e-7)."""
import numpy as np
import pytest

import devtools as dt
from hdsdp_amd import instances as I
from hdsdp_amd.solver import run_solver

pytestmark = pytest.mark.gpu

# name -> (instance, Gram-built Schur matrix, HDSDP_GRAM_BF16 override or None, y tolerance)
CASES = {
    "maxcut_n200": (lambda: I.maxcut(200, 0.05, 1, "pm1"), False, None, 1e-7),
    "theta_n50": (lambda: I.lovasz_theta(50, 0.3, 21), False, None, 1e-7),
    "dense_n40_m60": (lambda: I.dense_random(40, 60, 24), True, None, 1e-7),
    "dense_n120_m240": (lambda: I.dense_random(120, 240, 33), True, None, 1e-7),
    "rankone_n60_m500": (lambda: I.rank_one(60, 500, 5, 45), False, None, 1e-6),
    "rankone_n200_m2000": (lambda: I.rank_one(200, 2000, 20, 4), False, None, 1e-7),
    "rankone_n200_m2000_bf16": (lambda: I.rank_one(200, 2000, 20, 4), True, "1", 1e-6),
}


@pytest.mark.parametrize("name", list(CASES))
def test_mixed_matches_fp64(gpu_lib, name, monkeypatch):
    make, gram, force, ytol = CASES[name]
    if force is not None:
        monkeypatch.setenv("HDSDP_GRAM_BF16", force)
    inst = make()
    opts = dict(relopt=1e-6, absopt=1e30)
    r64 = run_solver(gpu_lib, inst, precision=0, **opts)
    rmx = run_solver(gpu_lib, inst, precision=1, **opts)
    rel_y = np.linalg.norm(rmx.y - r64.y) / np.linalg.norm(r64.y)
    print(name, r64.status, r64.iters, rmx.status, rmx.iters, rel_y, rmx.rel_gap, flush=True)
    assert rmx.status == r64.status == 3
    assert rmx.rel_gap <= 1e-6
    if gram:
        assert abs(rmx.iters - r64.iters) <= 2
    else:
        assert rmx.iters == r64.iters
    assert abs(rmx.dobj - r64.dobj) <= 1e-8 * max(1.0, abs(r64.dobj))
    assert abs(rmx.pobj - r64.pobj) <= 1e-8 * max(1.0, abs(r64.pobj))
    assert rel_y <= ytol


# The two mixed-precision workloads at their own sizes: the dense random SDP n = 1000,
# m = 2000 (every Gram block from bf16 planes) and the rank-one SDP n = 2000, m = 20000
# in factor form (FP64 Gram, lower-triangle CG products; its Cholesky preconditioner is FP64
# by itself and FP32 in test_mixed_full_size_fp32_factor).
FULL = {
    "dense_n1000_m2000": (lambda: I.dense_random(1000, 2000, 3), True),
    "rankone_n2000_m20000": (lambda: I.rank_one(2000, 20000, 20, 4), False),
}


@pytest.mark.parametrize("name", list(FULL))
def test_mixed_full_size(gpu_lib, name):
    """Mixed against FP64 at full size, 1e-6 gap: same status, dual objective within 1e-8
    and y* within 1e-7 relative.

    The rank-one instance (FP64 Gram, FP32 preconditioner) takes the FP64 path's
    iterations, and its objectives agree to 1e-8.  On the dense instance the Gram blocks
    are bf16 products; the path there is sensitive to rounding at the level of FP64
    alone: the FP64 GPU solve itself takes 38 or 43 iterations depending on the
    summation order inside the Cholesky panel of S (both orders measured), so the
    iteration counts are held within 6 of each other.  Its final primal objective comes
    from the recovered X, whose own gap to the dual objective is 3.5e-4 relative in
    the FP64 solve (the DIMACS gap error): the two primal objectives must agree to
    that gap."""
    make, gram = FULL[name]
    inst = make()
    opts = dict(relopt=1e-6, absopt=1e30)
    print(f"[mixed-full] {name}: fp64 solve", flush=True)
    r64 = run_solver(gpu_lib, inst, precision=0, **opts)
    print(f"[mixed-full] {name}: mixed solve", flush=True)
    rmx = run_solver(gpu_lib, inst, precision=1, **opts)
    rel_y = np.linalg.norm(rmx.y - r64.y) / np.linalg.norm(r64.y)
    print(name, "fp64", r64.status, r64.iters, f"{r64.seconds:.2f}s", "mixed", rmx.status, rmx.iters,
          f"{rmx.seconds:.2f}s", "y", rel_y, "gap", rmx.rel_gap, flush=True)
    assert rmx.status == r64.status == 3
    assert abs(rmx.dobj - r64.dobj) <= 1e-8 * max(1.0, abs(r64.dobj))
    assert rel_y <= 1e-7
    if gram:
        assert abs(rmx.iters - r64.iters) <= 6
        primal_gap = abs(r64.pobj - r64.dobj)
        assert abs(rmx.pobj - r64.pobj) <= max(1e-8 * max(1.0, abs(r64.pobj)), primal_gap)
    else:
        assert rmx.iters == r64.iters
        assert abs(rmx.pobj - r64.pobj) <= 1e-8 * max(1.0, abs(r64.pobj))


def test_mixed_full_size_fp32_factor(gpu_lib, monkeypatch):
    """The rank-one instance of test_mixed_full_size, same bounds, with the FP32 Cholesky
    preconditioner that larger systems take by themselves."""
    monkeypatch.setenv("HDSDP_MIXED_CHOL32_MIN", "16384")
    test_mixed_full_size(gpu_lib, "rankone_n2000_m20000")


@pytest.mark.parametrize("name", ["dense_n120_m240", "rankone_n60_m500"])
def test_mixed_against_reference(gpu_lib, name, monkeypatch):
    """The mixed path (bf16 planes for every dense / rank-one Gram block, forced for
    rank-one) against the reference HDSDP's FP64 result on the same instance: same status,
    at most two iterations apart, objectives within 1e-8 or the reference's own spread,
    y* within 1e-7 or that spread."""
    monkeypatch.setenv("HDSDP_GRAM_BF16", "1")
    inst, fix = dt.load_golden(name)
    res = run_solver(gpu_lib, inst, psdp=0, precision=1, **fix["options"])
    rep = dt.parity_report(fix, res)
    tol = dt.golden_tolerances(fix)
    print(name, rep, tol, flush=True)
    assert res.status == fix["status"]
    assert abs(res.iters - fix["iters"]) <= 2
    assert rep["dobj_rel"] <= tol["dobj"] and rep["pobj_rel"] <= tol["pobj"]
    assert rep["y_rel"] <= max(1e-7, tol["y"])
