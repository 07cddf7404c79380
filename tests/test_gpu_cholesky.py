"""The blocked Cholesky (hdk::potrf) called by itself, on the GPU, against numpy."""
import ctypes as C
import subprocess

import numpy as np
import pytest
import torch

from hdsdp_amd.solver import LIB_PATH

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def potrf(gpu_lib):
    """potrf(A) -> (L, info) of the lower triangle of a float64 or float32 array."""
    syms = [x.split()[-1] for x in subprocess.run(["nm", "-D", LIB_PATH], capture_output=True, text=True,
                                                  check=True).stdout.splitlines()]
    syms = [x for x in syms if "3hdk" in x]
    plain = subprocess.run(["c++filt"], input="\n".join(syms), capture_output=True, text=True, check=True).stdout
    table = {p.split("(")[0].split()[-1]: s for s, p in zip(syms, plain.splitlines()) if "lambda" not in p}

    def call(A):
        n = len(A)
        a = torch.as_tensor(np.ascontiguousarray(A.T), device="cuda")  # column-major
        L, info = torch.zeros_like(a), torch.full((1,), 7, dtype=torch.int32, device="cuda")
        dinv = torch.zeros((n + 63) // 64 * 4096, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        fn = getattr(gpu_lib, table["hdk::potrf<%s>" % ("double" if A.dtype == np.float64 else "float")])
        p = lambda t: C.c_void_p(t.data_ptr())
        fn(C.c_void_p(0), C.c_int(n), p(a), C.c_int(n), p(L), C.c_int(n), p(dinv), p(info), C.c_void_p(0))
        torch.cuda.synchronize()
        return L.cpu().numpy().T, int(info.cpu()[0])

    return call


def _spd(n, rng, flips=()):
    G = rng.standard_normal((n, n)) / np.sqrt(n)
    S = 4.0 * np.eye(n) + 0.6 * (G + G.T) / np.sqrt(2.0)
    for i in flips:
        S[i, i] = -1.0
    return S


# a single tile, launches of several tiles, more tiles than CUs, outer blocks of 768 (from 3073
# rows on): a failure in an earlier one, alone and with another in the first tile of a later one
@pytest.mark.parametrize("n,flips", [(40, ()), (64, (17,)), (65, (64,)), (200, (137, 150)), (1500, (700, 1400)),
                                     (3000, (64,)), (3200, ()), (3200, (2309,)), (3200, (3199,)), (3200, (100,)),
                                     (3200, (100, 2309)), (3200, (800, 1536))])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_info_is_the_first_failing_column(potrf, dtype, n, flips):
    """info: the first column whose pivot is not positive, from 1, or 0."""
    _, info = potrf(_spd(n, np.random.default_rng(n), flips).astype(dtype))
    assert info == (min(flips) + 1 if flips else 0)


# one block of 16 columns, one tile, several tiles; a subnormal, a normal and a huge scale
@pytest.mark.parametrize("n", [1, 10, 16, 17, 40, 64])
@pytest.mark.parametrize("scale", [2.0**-1040, 2.0**-1030, 2.0**-1000, 2.0**1018])
def test_factor_at_the_ends_of_the_range(potrf, n, scale):
    """S = scale B B^T for a small-integer B: its factor is sqrt(scale) B.  Every sum of the
    elimination is a small multiple of scale, exact down to the smallest subnormal (2^-1074);
    quotients by pivots of 25 scale round to u = 1.1e-16 and sums of n of them to n u of the
    largest entry, 6, with n steps on the way: 50 n u.  Subnormal sums round to 2^-1074 / scale
    more per step."""
    rng = np.random.default_rng(n)
    B = np.tril(rng.integers(-1, 2, (n, n)).astype(float), -1)
    B[np.abs(np.subtract.outer(np.arange(n), np.arange(n))) > 3] = 0.0
    B += 5.0 * np.eye(n)
    L, info = potrf((B @ B.T) * scale)
    assert info == 0
    root = scale**0.5
    tol = 50.0 * n * (1.1e-16 + 2.0**-1074 / scale)
    assert np.max(np.abs(np.tril(L) / root - B)) <= tol
