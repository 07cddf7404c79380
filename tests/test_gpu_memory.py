"""Problems that fit the device by little: what the faster layouts and factors take beyond the
plain ones must not cost a problem its place.  The rest of the card is held by a tensor."""
import numpy as np
import pytest
import torch

import devtools as dt
from hdsdp_amd import _capi

pytestmark = pytest.mark.gpu

GB = 1 << 30


@pytest.fixture
def leave():
    """leave(bytes): allocate all but so many bytes of the device until the test ends."""
    held = []

    def hold(free):
        torch.cuda.empty_cache()
        while (rest := torch.cuda.mem_get_info()[0] - free) > 64 << 20:
            held.append(torch.empty(min(rest, 32 * GB), dtype=torch.uint8, device="cuda"))

    yield hold
    held.clear()
    torch.cuda.empty_cache()


def _mild(n, rng):
    G = rng.standard_normal((n, n)) / np.sqrt(n)
    return 4.0 * np.eye(n) + 0.6 * (G + G.T) / np.sqrt(2.0)


def test_mixed_factor_in_fp32_where_fp64_does_not_fit(gpu_lib, leave):
    """m = 16500: M takes 2.2 GB, the FP64 factor and its inverses 6.5, the FP32 ones 3.3.  With 5
    GB beside M the FP32 factor is taken, as for every such m before the FP64 one was
    preferred; it needs more than one iteration, to 1e-11 |b|, and the residual is taken with
    M x = A(W A*(x) W) + x in numpy (rounding below 1e-11 |b| again)."""
    m, n = 16500, 190
    rng = np.random.default_rng(1)
    S = _mild(n, rng)
    r, c = np.tril_indices(n)
    pick = np.sort(rng.choice(len(r), size=m, replace=False))
    one = np.ones(1)
    co = [dt.Coeff(dt.DENSE, n, val=np.concatenate([S[j:, j] for j in range(n)]))]
    co += [dt.Coeff(dt.SPARSE, n, row=[r[k]], col=[c[k]], val=one) for k in pick]
    d = dt.Dev(gpu_lib, co, 1)
    leave(5 * GB)
    d.update(1.0, 0.0, np.zeros(m), 0.0, 0)
    assert d.factorize(0) == 1
    d.schur(0, 0.0)
    d.add_diag(np.ones(m))
    b = rng.standard_normal(m)
    rel = 1e-11
    d.kkt_params(rel, rel * np.linalg.norm(b), 5, -1)
    assert d.kkt_factorize() == 0
    x = d.kkt_solve(b)
    s = np.zeros(7)
    assert gpu_lib.hdsdp_dev_stats(d.h, _capi.dptr(s), 7) == 0
    ldl = d.uses_ldl()
    d.close()
    assert ldl == 0 and s[4] == 1 and 1 <= s[5] < 5
    W = np.linalg.inv(S)
    X = np.zeros((n, n))
    X[r[pick], c[pick]] = x
    X = X + np.tril(X, -1).T
    Y = W @ X @ W
    Mx = np.where(r == c, 1.0, 2.0)[pick] * Y[r[pick], c[pick]] + x
    assert np.linalg.norm(Mx - b) <= 2.0 * rel * np.linalg.norm(b)


def test_dense_build_without_panels_where_they_do_not_fit(gpu_lib, leave):
    """513 dense constraints at n = 900: 1.7 GB of coefficients, then 1.7 GB of T_p and two batches
    of 0.5 GB laid out plainly, 2.1 GB and two of 1 GB in panels padded to 640 constraints.
    With 5.2 GB in all the problem loads, and M is that of the panels (25 n u as in
    test_dense_gram_build)."""
    n, m = 900, 513
    rng = np.random.default_rng(2)
    S = _mild(n, rng)
    co = [dt.Coeff(dt.DENSE, n, val=np.concatenate([S[j:, j] for j in range(n)]))]
    co += [dt.rand_dense(rng, n) for _ in range(m)]
    got = []
    for free in (None, 5.2 * GB):
        if free:
            leave(int(free))
        d = dt.Dev(gpu_lib, co)
        d.update(1.0, 0.0, np.zeros(m), 0.0, 0)
        assert d.factorize(0) == 1
        d.schur(0, 0.0)
        got.append(d.get_schur())
        d.close()
    assert not np.array_equal(got[0], got[1])  # the two layouts sum in another order
    assert np.max(np.abs(got[0] - got[1])) <= 25.0 * n * 1.1e-16 * np.max(np.abs(got[0]))
