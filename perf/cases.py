"""Timed workloads of the solver's device path and of its differentiation.

Every case goes through a public entry point: the device ABI of ``include/hdsdp_gpu.h``
(what an interior-point host calls, on host vectors, with the block's state resident in
HBM) or ``hdsdp_amd.solver.Solver``.  Whole ``optimize`` calls are left to ``bench.py``:
the interior-point path turns rounding into another (equally valid) sequence of
iterates, so its outputs cannot be compared value by value; one iteration's can.

Paths (``case["path"]``):

``step``    one iteration of the dual method: S(y) assembled and factored, the Schur
            system built, preconditioned and solved for every right-hand side, the step
            length from the Lanczos ratio test, the trial point's S assembled and
            factored, and the corrector's right-hand side and solve on the same M.
``embed``   one iteration of the self-dual embedding (the HOMOGENEOUS build with C's terms).
``primal``  primal recovery and one step of the primal method (on by default, as in HDSDP).
``centre``  ``Solver.center`` and ``Solver.adjoint``: the forward and backward pass of the
            differentiable solve.

Families (``case["family"]``) are the constraint structures of the repository's own
configurations: ``theta`` (Lovasz theta: an identity row and single-entry edges),
``maxcut`` (single diagonal entries, sparse C), ``dense`` (dense symmetric A_i) and
``rankone`` (dense rank-one A_i in factor form).  ``late`` is the second half of a solve:
the Schur CG has given up its Jacobi preconditioner for the Cholesky factor of M, and the
dual iterate is feasible (Rd = 0); otherwise the iterate is infeasible (Rd != 0) and CG
runs with the Jacobi preconditioner.  ``precision`` is the solver's own option.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from hdsdp_amd import _capi, instances
from hdsdp_amd.solver import Solver, load_library

DEV = "cuda"
F64 = torch.float64
SPARSE, DENSE, SPR1, DSR1 = 1, 2, 3, 4
VIEW = np.dtype([("type", "<i4"), ("nnz", "<i4"), ("row", "<u8"), ("col", "<u8"), ("val", "<u8"), ("sign", "<f8")])


# ---- the cases ---------------------------------------------------------------------


def _case(name, path, family, n, m, late=False, precision="fp64"):
    c = {"path": path, "family": family, "n": n, "m": m, "late": late, "precision": precision}
    return {"name": name, **c} if name else c


def listed():
    return [
        # smallest solves (a theta number of a 50-vertex graph): launches and round trips
        _case("step theta 50", "step", "theta", 50, 368),
        # MaxCut on 200 vertices, the repository's first configuration, early phase
        _case("step maxcut 200", "step", "maxcut", 200, 200),
        # a small dense SDP with odd sizes, early phase
        _case("step dense 121", "step", "dense", 121, 243),
        # Lovasz theta on 400 vertices: the Schur system (m = 8084) dominates
        _case("step theta 400 late", "step", "theta", 400, 8084, late=True),
        # MaxCut on 2000 vertices: S itself is the large matrix
        _case("step maxcut 2000 late", "step", "maxcut", 2000, 2000, late=True),
        # dense SDP in FP64 at the headline's n: the Gram products of the Schur build
        _case("step dense 1000 late", "step", "dense", 1000, 1000, late=True),
        # the headline workload's iteration in mixed precision (n = 1000, m = 2000)
        _case("step dense 1000 mixed", "step", "dense", 1000, 2000, late=True, precision="mixed"),
        # rank-one SDP with m >> n (n = 2000, m = 20000): the largest Schur system
        _case("step rankone 2000 late", "step", "rankone", 2000, 20000, late=True),
        # an ordinary rank-one SDP, ragged sizes, early phase
        _case("step rankone 301", "step", "rankone", 301, 3001),
        # the self-dual embedding on a dense block of ordinary size
        _case("embed dense 300", "embed", "dense", 300, 450, late=True),
        # primal recovery and the primal method on an ordinary theta SDP
        _case("primal theta 250", "primal", "theta", 250, 2001, late=True),
        # forward and backward of the differentiable solve on an ordinary MaxCut SDP
        _case("centre maxcut 500", "centre", "maxcut", 500, 500),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["step"] * 6 + ["embed", "primal", "centre"])
    if path == "centre":
        n = _log_int(rng, 60, 800)
        return _case(None, path, "maxcut", n, n)
    late = rng.random() < 0.5
    if path == "primal":
        family = rng.choice(["theta", "maxcut"])
        late = True
    else:
        family = rng.choice(["theta", "maxcut", "dense", "rankone"])
    precision = "fp64"
    if family == "theta":
        n = _log_int(rng, 40, 400)
        m = 1 + int(round(rng.uniform(0.08, 0.3) * n * (n - 1) / 2))
        m = min(m, 8001)
    elif family == "maxcut":
        n = _log_int(rng, 60, 2000)
        m = n
    elif family == "dense":
        n = _log_int(rng, 40, 900)
        m = max(30, int(n * rng.uniform(0.5, 2.0)))
        m = min(m, int(6e8 / (n * (n + 1) / 2)))
        if late and path == "step" and rng.random() < 0.5:
            precision = "mixed"
    else:
        n = _log_int(rng, 60, 1500)
        m = min(int(n * rng.uniform(3.0, 10.0)), n * (n + 1) // 4, 12000)
    return _case(None, path, family, n, m, late, precision)


# ---- problem data ------------------------------------------------------------------


class Data:
    """One problem and one iterate, on the GPU in 64 bits, made from the seed alone."""

    def __init__(self, case, seed):
        self.case = case
        self.n, self.m = n, m = case["n"], case["m"]
        self.family = case["family"]
        rng = np.random.default_rng([seed, 17])
        gen = torch.Generator(device=DEV)
        gen.manual_seed(1000003 * (seed % 1000000) + 29)
        self.eye = 0.0
        if self.family == "theta":
            pairs = np.sort(rng.choice(n * (n - 1) // 2, size=m - 1, replace=False))
            i = ((1.0 + np.sqrt(8.0 * pairs + 1.0)) / 2.0).astype(np.int64)  # i (i - 1) / 2 <= pair, i > j
            i = np.where(i * (i - 1) // 2 > pairs, i - 1, i)
            i = np.where((i + 1) * i // 2 <= pairs, i + 1, i)
            self.ei, self.ej = i.astype(np.int32), (pairs - i * (i - 1) // 2).astype(np.int32)
            y = 0.3 * rng.standard_normal(m)
            y[0] = -1.4 * n if case["late"] else -0.2 * n
            self.eye = 0.0 if case["late"] else 1.6 * n
            self.b = np.zeros(m)
            self.b[0] = 1.0
        elif self.family == "maxcut":
            cnt = max(n, int(round(min(0.05, 20.0 / n) * n * (n - 1) / 2)))
            pairs = np.sort(rng.choice(n * (n - 1) // 2, size=min(cnt, n * (n - 1) // 2), replace=False))
            i = ((1.0 + np.sqrt(8.0 * pairs + 1.0)) / 2.0).astype(np.int64)
            i = np.where(i * (i - 1) // 2 > pairs, i - 1, i)
            i = np.where((i + 1) * i // 2 <= pairs, i + 1, i)
            j = pairs - i * (i - 1) // 2
            w = rng.random(i.shape[0]) + 0.05
            deg = np.bincount(i, w, n) + np.bincount(j, w, n)
            self.ei, self.ej, self.w = i.astype(np.int32), j.astype(np.int32), w
            self.cdiag = -deg / 4.0  # C = -L / 4
            # S = C - diag(y) is diagonally dominant for y < -deg / 2
            y = -0.5 * deg * (1.0 + 0.5 * rng.random(n)) - 0.05
            if not case["late"] and case["path"] != "centre":
                y *= 0.5
                self.eye = 0.3 * float(deg.max()) + 1.0
            self.b = np.ones(m)
        elif self.family == "dense":
            npk = n * (n + 1) // 2
            self.A = torch.empty((m + 1, npk), dtype=F64, device=DEV)  # packed lower columns, C last
            for q0 in range(0, m, 256):
                q1 = min(m, q0 + 256)
                self.A[q0:q1] = torch.randn((q1 - q0, npk), generator=gen, dtype=F64, device=DEV) / math.sqrt(n)
            dpos = torch.arange(n, device=DEV)
            self.dpos = dpos * n - dpos * (dpos - 1) // 2
            y0 = rng.standard_normal(m)
            self.A[m] = torch.as_tensor(y0, device=DEV) @ self.A[:m]
            self.A[m, self.dpos] += 1.0
            dy = rng.standard_normal(m)
            y = y0 + (0.38 if case["late"] else 0.9) / np.linalg.norm(dy) * dy
            self.eye = 0.0 if case["late"] else 1.5
            self.b = self.A[:m, self.dpos].sum(1).cpu().numpy()
        else:
            f = torch.randn((m, n), generator=gen, dtype=F64, device=DEV) / math.sqrt(n)
            nrm = torch.linalg.vector_norm(f, dim=1)
            self.F = f / nrm[:, None]
            self.sgn = (nrm * nrm).cpu().numpy()
            y = (0.4 if case["late"] else 0.8) * n / m * (rng.random(m) - 0.6)
            self.eye = 0.0 if case["late"] else 0.7
            self.b = self.sgn.copy()
        self.y = y
        # shape of the trial step and of the losses: generic vectors
        self.dual = 1e-2 * rng.standard_normal(m)

    # -- host form: presolved coefficients as the device ABI takes them

    def views(self):
        n, m = self.n, self.m
        v = np.zeros(m + 1, dtype=VIEW)
        keep = []

        def ptr(a):
            keep.append(a)
            return a.ctypes.data

        if self.family == "theta":
            ones = np.ones(max(n, m))
            v["type"][0], v["nnz"][0], v["sign"][0] = DSR1, n, -float(n)
            v["val"][0] = ptr(np.full(n, 1.0 / math.sqrt(n)))
            d = np.arange(n, dtype=np.int32)
            v["type"][1:], v["nnz"][1:], v["nnz"][1] = SPARSE, 1, n
            v["row"][1] = v["col"][1] = ptr(d)
            v["val"][1:] = ptr(ones)
            at = 4 * np.arange(m - 1, dtype=np.uint64)
            v["row"][2:] = np.uint64(ptr(self.ei)) + at
            v["col"][2:] = np.uint64(ptr(self.ej)) + at
        elif self.family == "maxcut":
            rows = np.concatenate([np.arange(n, dtype=np.int32), self.ei])
            cols = np.concatenate([np.arange(n, dtype=np.int32), self.ej])
            vals = np.concatenate([self.cdiag, self.w / 4.0])
            order = np.lexsort((rows, cols))
            rows, cols, vals = (np.ascontiguousarray(a[order]) for a in (rows, cols, vals))
            v["type"][0], v["nnz"][0] = SPARSE, len(vals)
            v["row"][0], v["col"][0], v["val"][0] = ptr(rows), ptr(cols), ptr(vals)
            v["type"][1:], v["nnz"][1:], v["sign"][1:] = SPR1, 1, 1.0
            v["row"][1:] = np.uint64(ptr(np.arange(n, dtype=np.int32))) + 4 * np.arange(m, dtype=np.uint64)
            v["val"][1:] = ptr(np.ones(1))
        elif self.family == "dense":
            host = _staging(self.A.numel()).view(self.A.shape)
            host.copy_(self.A)
            npk = self.A.shape[1]
            v["type"] = DENSE
            base = np.uint64(host.data_ptr())
            v["val"][1:] = base + np.uint64(8 * npk) * np.arange(m, dtype=np.uint64)
            v["val"][0] = base + np.uint64(8 * npk * m)
            keep.append(host)
        else:
            host = self.F.cpu().numpy()
            d = np.arange(n, dtype=np.int32)
            v["type"][0], v["nnz"][0] = SPARSE, n
            v["row"][0] = v["col"][0] = ptr(d)
            v["val"][0] = ptr(np.ones(n))
            v["type"][1:], v["nnz"][1:], v["sign"][1:] = DSR1, n, self.sgn
            v["val"][1:] = np.uint64(ptr(host)) + np.uint64(8 * n) * np.arange(m, dtype=np.uint64)
        return v, keep

    # -- 64-bit restatements

    def full(self, k0, k1):
        """Dense symmetric A_k for k0 <= k < k1 (k = m: C), dense family."""
        n = self.n
        i, j = torch.tril_indices(n, n, device=DEV)
        pos = j * n - j * (j - 1) // 2 + (i - j)
        out = torch.empty((k1 - k0, n, n), dtype=F64, device=DEV)
        out[:, i, j] = self.A[k0:k1, pos]
        out[:, j, i] = self.A[k0:k1, pos]
        return out

    def c_matrix(self):
        n = self.n
        if self.family == "theta":
            return -torch.ones((n, n), dtype=F64, device=DEV)
        if self.family == "maxcut":
            S = torch.diag(torch.as_tensor(self.cdiag, device=DEV))
            i, j = self._edges()
            w = torch.as_tensor(self.w / 4.0, device=DEV)
            S[i, j] = w
            S[j, i] = w
            return S
        if self.family == "dense":
            return self.full(self.m, self.m + 1)[0]
        return torch.eye(n, dtype=F64, device=DEV)

    def _edges(self):
        return torch.as_tensor(self.ei, device=DEV).long(), torch.as_tensor(self.ej, device=DEV).long()

    def a_transpose(self, y):
        """sum_i y_i A_i."""
        n, m = self.n, self.m
        y = torch.as_tensor(y, device=DEV)
        if self.family == "theta":
            S = y[0] * torch.eye(n, dtype=F64, device=DEV)
            i, j = self._edges()
            S[i, j] = y[1:]
            S[j, i] = y[1:]
            return S
        if self.family == "maxcut":
            return torch.diag(y)
        if self.family == "dense":
            i, j = torch.tril_indices(n, n, device=DEV)
            pk = (y @ self.A[:m])[j * n - j * (j - 1) // 2 + (i - j)]
            S = torch.zeros((n, n), dtype=F64, device=DEV)
            S[i, j] = pk
            S[j, i] = pk
            return S
        w = y * torch.as_tensor(self.sgn, device=DEV)
        return self.F.T @ (self.F * w[:, None])

    def a_of(self, B):
        """<A_i, B> for symmetric B."""
        n, m = self.n, self.m
        if self.family == "theta":
            i, j = self._edges()
            return torch.cat([torch.trace(B)[None], 2.0 * B[i, j]])
        if self.family == "maxcut":
            return torch.diagonal(B).clone()
        if self.family == "dense":
            i, j = torch.tril_indices(n, n, device=DEV)
            w = torch.empty(n * (n + 1) // 2, dtype=F64, device=DEV)
            w[j * n - j * (j - 1) // 2 + (i - j)] = torch.where(i == j, 1.0, 2.0) * B[i, j]
            return self.A[:m] @ w
        return torch.as_tensor(self.sgn, device=DEV) * (self.F * (self.F @ B)).sum(1)

    def schur(self, W):
        """<A_i, W A_j W>."""
        n, m = self.n, self.m
        if self.family == "theta":
            i, j = self._edges()
            M = torch.empty((m, m), dtype=F64, device=DEV)
            M[1:, 1:] = 2.0 * (W[i][:, i] * W[j][:, j] + W[i][:, j] * W[j][:, i])
            row = self.a_of(W @ W)
            M[0, :] = row
            M[:, 0] = row
            return M
        if self.family == "maxcut":
            return W * W
        if self.family == "dense":
            L = torch.linalg.cholesky(W)  # <A_p, W A_q W> = <L^T A_p L, L^T A_q L>
            T = torch.empty((m, n * n), dtype=F64, device=DEV)
            for k in range(0, m, 64):
                k1 = min(m, k + 64)
                T[k:k1] = (L.T.contiguous() @ (self.full(k, k1) @ L)).reshape(k1 - k, n * n)
            return T @ T.T
        s = torch.as_tensor(self.sgn, device=DEV)
        K = self.F @ W @ self.F.T
        return s[:, None] * K * K * s[None, :]


_pinned = None


def _staging(count):
    """Host buffer the dense coefficients are handed over in (the library copies them)."""
    global _pinned
    if _pinned is None or _pinned.numel() < count:
        _pinned = None
        _pinned = torch.empty(count, dtype=F64, pin_memory=True)
    return _pinned[:count]


# ---- one device block ----------------------------------------------------------------


class Block:
    """A loaded ``hdsdp_dev`` with the calls an interior-point host makes on it."""

    def __init__(self, data):
        self.lib, self.n, self.m = load_library(), data.n, data.m
        self.h = C.c_void_p()
        precision = 1 if data.case["precision"] == "mixed" else 0
        self._do(self.lib.hdsdp_dev_create(C.byref(self.h), self.m, self.n, precision))
        views, keep = data.views()
        self._do(self.lib.hdsdp_dev_load(self.h, views.ctypes.data))
        del keep
        # the solver's CG accuracy and iteration limit by size of the Schur system
        m = self.m
        self.acc, self.maxit = 1e-12, max(50, m // 20)
        if m > 15000:
            self.acc, self.maxit = 50e-12, 450
        elif m > 5000:
            self.acc, self.maxit = 5e-12, 120
        self.set_cg(5.0 * self.acc, self.acc, self.maxit)

    def __del__(self):
        if self.h:
            self.lib.hdsdp_dev_destroy(C.byref(self.h))

    @staticmethod
    def _do(rc):
        if rc:
            raise RuntimeError(f"device call failed ({rc})")

    def set_cg(self, rel, absolute, maxit):
        self._do(self.lib.hdsdp_dev_kkt_params(self.h, rel, absolute, maxit, -1))

    def assemble(self, c, a, y, eye, which):
        self._do(self.lib.hdsdp_dev_update_buffer(self.h, c, a, _capi.dptr(y), eye, which))

    def factor(self, which):
        ok = C.c_int()
        self._do(self.lib.hdsdp_dev_factorize(self.h, which, C.byref(ok)))
        return ok.value

    def logdet(self, which):
        v = C.c_double()
        self._do(self.lib.hdsdp_dev_logdet(self.h, which, C.byref(v)))
        return v.value

    def ratio(self, which):
        v = C.c_double()
        self._do(self.lib.hdsdp_dev_ratio_test(self.h, which, C.byref(v)))
        return v.value

    def schur(self, kind, Rd):
        a, b, t = np.zeros(self.m), np.zeros(self.m), C.c_double()
        self._do(self.lib.hdsdp_dev_schur(self.h, kind, Rd, _capi.dptr(a), _capi.dptr(b), C.byref(t)))
        return a, b, t.value

    def add_diag(self, d):
        self._do(self.lib.hdsdp_dev_kkt_add_diag(self.h, _capi.dptr(d)))

    def precondition(self):
        self._do(self.lib.hdsdp_dev_kkt_factorize(self.h))

    def solve(self, rhs):
        x = np.zeros(self.m)
        self._do(self.lib.hdsdp_dev_kkt_solve(self.h, _capi.dptr(rhs), _capi.dptr(x)))
        return x


BOUND = 1e-3  # the dual box's share of the Schur diagonal


def prepare(case, seed):
    d = Data(case, seed)
    if case["path"] == "centre":
        inst = instances.maxcut_graph(d.n, d.ej.astype(np.int64), d.ei.astype(np.int64), d.w)
        sv = Solver(load_library(), inst, relopt=1e-8, absopt=1e30)
        sv.setup()
        return {"case": case, "solver": sv, "mu": 0.05, "y": d.y, "grad": d.dual}
    dev = Block(d)
    st = {"case": case, "dev": dev, "y": d.y, "b": d.b, "eye": d.eye, "Rd": -d.eye, "dual": d.dual,
          "diag": np.full(d.m, BOUND), "mu": _mu(d)}
    if case["late"]:
        # the state a solve is in once its Jacobi CG has run into the iteration limit:
        # the Schur CG keeps the Cholesky preconditioner from then on
        dev.assemble(1.0, -1.0, d.y, d.eye, 0)
        dev.factor(0)
        dev.schur(0, 0.0)
        dev.precondition()
        rhs = np.random.default_rng(seed).standard_normal(d.m)
        dev.set_cg(1e-9, 1e-9 * float(np.linalg.norm(rhs)), 4)
        dev.solve(rhs)
        dev.set_cg(5.0 * dev.acc, dev.acc, dev.maxit)
        factored = np.zeros(5)
        dev._do(dev.lib.hdsdp_dev_stats(dev.h, _capi.dptr(factored), 5))
        if factored[4] < 1 or dev.lib.hdsdp_dev_kkt_uses_ldl(dev.h):
            raise RuntimeError("the Schur CG has not taken up its Cholesky preconditioner")
    return st


def _mu(d):
    """The barrier parameter of the iterate's own scale, X = I against mu S^-1."""
    s = float(torch.trace(d.c_matrix())) - float(torch.trace(d.a_transpose(d.y))) + d.n * d.eye
    return 0.5 * s / d.n


# ---- one pass ------------------------------------------------------------------------


def run(st):
    return {"step": _step, "embed": _embed, "primal": _primal, "centre": _centre}[st["case"]["path"]](st)


def _step(st):
    dev, y, Rd, mu = st["dev"], st["y"], st["Rd"], st["mu"]
    dev.assemble(1.0, -1.0, y, st["eye"], 0)
    psd = dev.factor(0)
    logdet = dev.logdet(0)
    asinv, asinvrd, trace = dev.schur(0, Rd)
    dev.add_diag(st["diag"])
    dev.precondition()
    xb = dev.solve(st["b"])
    xa = dev.solve(asinv)
    dy = xb / mu - xa
    out = {"psd": psd, "logdet": logdet, "asinv": asinv, "xb": xb, "xa": xa}
    if Rd != 0.0:
        xr = dev.solve(asinvrd)
        dy = dy + xr
        out |= {"asinvrd": asinvrd, "trace": trace, "xr": xr}
    # step length and trial point (Rd shrinks with the step)
    dev.assemble(0.0, -1.0, dy, 0.0, 2)
    bound = dev.ratio(0)
    step = min(0.7 * bound, 1.0)
    yt = y + step * dy
    dev.assemble(1.0, -1.0, yt, st["eye"], 0)
    out |= {"bound": bound, "trial psd": dev.factor(0), "trial logdet": dev.logdet(0)}
    # corrector: the right-hand side at the new point, the Schur matrix of the old one
    asinv2, _, _ = dev.schur(1, 0.0)
    xc = dev.solve(asinv2)
    dev.assemble(0.0, -1.0, xb / mu - xc, 0.0, 2)
    return out | {"corrector asinv": asinv2, "corrector x": xc, "corrector bound": dev.ratio(0)}


def _embed(st):
    dev, Rd = st["dev"], -0.25
    dev.assemble(1.0, -1.0, st["y"], st["eye"] - Rd, 0)
    psd = dev.factor(0)
    asinv, asinvrd, trace = dev.schur(2, Rd)
    acs = np.zeros(dev.m)
    cs, csc, csr = C.c_double(), C.c_double(), C.c_double()
    dev._do(dev.lib.hdsdp_dev_hsd(dev.h, Rd, _capi.dptr(acs), C.byref(cs), C.byref(csc), C.byref(csr)))
    dev.precondition()
    out = {"psd": psd, "asinv": asinv, "asinvrd": asinvrd, "trace": trace, "acs": acs,
           "c": np.array([cs.value, csc.value, csr.value])}
    for name, rhs in (("xb", st["b"]), ("xa", asinv), ("xr", asinvrd), ("xc", acs)):
        out[name] = dev.solve(rhs)
    return out


def _primal(st):
    dev, y, mu, dy = st["dev"], st["y"], st["mu"], st["dual"]
    dev.assemble(1.0, -1.0, y, 0.0, 0)
    dev.factor(0)
    dev.assemble(1.0, -1.0, y, 0.0, 1)
    ok = C.c_int()
    dev._do(dev.lib.hdsdp_dev_primal(dev.h, mu, _capi.dptr(y), _capi.dptr(dy), C.byref(ok)))
    ax = np.zeros(dev.m)
    cx, xs, tx = C.c_double(), C.c_double(), C.c_double()
    dev._do(dev.lib.hdsdp_dev_primal_stats(dev.h, _capi.dptr(ax), C.byref(cx), C.byref(xs), C.byref(tx)))
    X = np.zeros((dev.n, dev.n), order="F")
    dev._do(dev.lib.hdsdp_dev_get_primal(dev.h, X.ctypes.data_as(_capi.P_DBL)))
    out = {"ok": ok.value, "ax": ax, "stats": np.array([cx.value, xs.value, tx.value]), "X": X}
    # the primal method: W = X for the Schur matrix, then one step
    dev._do(dev.lib.hdsdp_dev_psdp_init(dev.h))
    dev.schur(3, 0.0)
    dev.precondition()
    ax2, rhs = np.zeros(dev.m), np.zeros(dev.m)
    dev._do(dev.lib.hdsdp_dev_psdp_rhs(dev.h, 0.5 * mu, _capi.dptr(ax2), _capi.dptr(rhs)))
    x = dev.solve(rhs)
    dev.assemble(0.0, -1.0, x, 0.0, 2)
    dual_bound = dev.ratio(0)
    bound, psd = C.c_double(), C.c_int()
    dev._do(dev.lib.hdsdp_dev_psdp_direction(dev.h, 0.5 * mu, 1, C.byref(bound)))
    alpha = min(0.95 * bound.value, 1.0)
    dev._do(dev.lib.hdsdp_dev_psdp_step(dev.h, alpha, C.byref(psd), C.byref(cx), C.byref(xs)))
    return out | {"rhs": rhs, "x": x, "dual bound": dual_bound, "primal bound": bound.value, "psd": psd.value,
                  "after": np.array([cx.value, xs.value])}


def _centre(st):
    y, _, _ = st["solver"].center(st["mu"], st["y"], tol=1e-11)
    db, dC = st["solver"].adjoint(st["mu"], y, st["grad"])
    return {"y": y, "db": db, "dC": dC}


# ---- 64-bit values -------------------------------------------------------------------


def _solve64(M, *rhs):
    """M x = rhs by Cholesky with one step of refinement."""
    L = torch.linalg.cholesky(M)
    out = []
    for r in rhs:
        r = torch.as_tensor(r, device=DEV)[:, None]
        x = torch.cholesky_solve(r, L)
        x = x + torch.cholesky_solve(r - M @ x, L)
        out.append(x[:, 0].cpu().numpy())
    return out


def _sym(A):
    return 0.5 * (A + A.T)


def exact(case, seed):
    d = Data(case, seed)
    n, m, path = d.n, d.m, case["path"]
    Cm = d.c_matrix()
    I = torch.eye(n, dtype=F64, device=DEV)
    if path == "centre":
        return _exact_centre(d, Cm)
    eye = d.eye + (0.25 if path == "embed" else 0.0)
    S = _sym(Cm - d.a_transpose(d.y) + eye * I)
    W = _sym(torch.cholesky_inverse(torch.linalg.cholesky(S)))
    if path == "step":
        M = d.schur(W)
        M.diagonal().add_(BOUND)
        asinv = d.a_of(W)
        out = {"psd": None, "logdet": float(torch.linalg.slogdet(S)[1]), "asinv": asinv.cpu().numpy()}
        # the step bound is the Lanczos iteration's own estimate, and what follows depends on it
        for k in ("bound", "trial psd", "trial logdet", "corrector asinv", "corrector x", "corrector bound"):
            out[k] = None
        if d.eye != 0.0:
            ard = -d.eye * d.a_of(W @ W)
            out |= {"asinvrd": ard.cpu().numpy(), "trace": float(torch.trace(W))}
            out["xb"], out["xa"], out["xr"] = _solve64(M, d.b, asinv, ard)
        else:
            out["xb"], out["xa"] = _solve64(M, d.b, asinv)
        return out
    if path == "embed":
        Rd = -0.25
        M, B = d.schur(W), _sym(W @ Cm @ W)
        asinv, ard, acs = d.a_of(W), Rd * d.a_of(_sym(W @ W)), d.a_of(B)
        out = {"psd": None, "asinv": asinv.cpu().numpy(), "asinvrd": ard.cpu().numpy(),
               "trace": float(torch.trace(W)), "acs": acs.cpu().numpy(),
               "c": np.array([float((Cm * W).sum()), float((Cm * B).sum()), Rd * float(torch.trace(B))])}
        out["xb"], out["xa"], out["xr"], out["xc"] = _solve64(M, d.b, asinv, ard, acs)
        return out
    mu = _mu(d)
    X = _sym(mu * (W + W @ d.a_transpose(d.dual) @ W))
    ax = d.a_of(X)
    XSX = _sym(X @ S @ X)
    rhs = d.a_of(XSX) - 0.5 * mu * ax
    return {"ok": None, "ax": ax.cpu().numpy(),
            "stats": np.array([float((Cm * X).sum()), float((X * S).sum()), float(torch.trace(X))]),
            "X": X.cpu().numpy(), "rhs": rhs.cpu().numpy(), "x": _solve64(d.schur(X), rhs)[0],
            "dual bound": None, "primal bound": None, "psd": None, "after": None}


def _exact_centre(d, Cm):
    """Newton on b = mu A(S^-1) for diag constraints, then the implicit-function gradients."""
    mu, y = 0.05, torch.as_tensor(d.y, device=DEV)
    b = torch.as_tensor(d.b, device=DEV)

    def at(y):
        L, info = torch.linalg.cholesky_ex(Cm - torch.diag(y))
        return None if int(info) else _sym(torch.cholesky_inverse(L))

    W = at(y)
    for _ in range(200):
        g = b - mu * torch.diagonal(W)
        dy = torch.cholesky_solve(g[:, None] / mu, torch.linalg.cholesky(W * W))[:, 0]
        delta = float(torch.sqrt((dy @ g / mu).clamp(min=0.0)))
        a = 1.0 / (1.0 + delta) if delta > 0.25 else 1.0
        while (Wn := at(y + a * dy)) is None:
            a *= 0.5
        y, W = y + a * dy, Wn
        if delta < 1e-13:
            break
    lam = torch.cholesky_solve(torch.as_tensor(d.dual, device=DEV)[:, None], torch.linalg.cholesky(W * W))[:, 0]
    return {"y": y.cpu().numpy(), "db": (lam / mu).cpu().numpy(), "dC": _sym(W @ torch.diag(lam) @ W).cpu().numpy()}


# ---- what a pass cannot do without ---------------------------------------------------


def work(case):
    """Coefficients read, vectors in and out, the Schur matrix written once (and its
    factor, where one is formed); flops of the factorisations, inverses and products."""
    n, m, fam, path = float(case["n"]), float(case["m"]), case["family"], case["path"]
    coef = {"theta": 16.0 * m, "maxcut": 16.0 * m + 12.0 * 10.0 * n, "dense": 4.0 * m * n * n, "rankone": 8.0 * m * n}[fam]
    schur = 4.0 * m * m
    gram = {"theta": 7.0 * m * m / 2.0, "maxcut": 2.0 * m * m, "dense": m * n**3 + 0.5 * m * m * n * n,
            "rankone": m * n * n + m * m * n}[fam]
    s_factor, s_inverse = n**3 / 3.0, 2.0 * n**3 / 3.0
    late = case["late"] or path == "centre"
    solve = m**3 / 3.0 if late else 10.0 * 2.0 * m * m
    flops = gram + solve + s_factor + s_inverse
    if path == "step":
        flops += s_factor + s_inverse
    elif path == "primal":
        flops += 2.0 * s_factor + 8.0 * n**3
    elif path == "embed":
        flops += 4.0 * n**3
    else:
        flops = 8.0 * flops + 4.0 * n**3  # about eight Newton steps, one adjoint
    return {"bytes": coef + schur * (2.0 if late else 1.0) + 8.0 * 10.0 * m + 8.0 * 2.0 * n * n, "flops": flops}
