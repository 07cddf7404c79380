"""Launch grids of the host side of the kernels, without a GPU: a preloaded stand-in for the
call that sets a launch's grid records it and leaves the launch out, and the launchers run with sizes and addresses
alone.  HIP promises 65535 workgroups in y and z (x: 2^31 - 1), so matrix rows and columns
belong on x: Schur systems run to m = 94000 or so, where four m x m matrices fill the card."""
import os
import subprocess
import sys

import pytest

from hdsdp_amd.solver import LIB_PATH

STUB = r"""
#include <stdio.h>
typedef struct { unsigned x, y, z; } dim3_;
int __hipPushCallConfiguration(dim3_ g, dim3_ b, unsigned long s, void *t) {
    printf("%u %u %u\n", g.x, g.y, g.z);
    fflush(stdout);
    return 1; /* not 0: the caller leaves the launch out */
}
int hipMemcpyAsync(void *d, const void *s, unsigned long n, int k, void *t) { return 0; }
"""

CALL = r"""
import ctypes as C, subprocess, sys
lib = C.CDLL(sys.argv[1])
names = {}
for line in subprocess.run(["nm", "-D", sys.argv[1]], capture_output=True, text=True, check=True).stdout.splitlines():
    sym = line.split()[-1]
    if "3hdk" in sym:
        names[sym] = None
plain = subprocess.run(["c++filt"], input="\n".join(names), capture_output=True, text=True, check=True).stdout
table = {p.replace("void ", "").split("(")[0]: s for s, p in zip(names, plain.splitlines()) if "lambda" not in p}
n, p, i = int(sys.argv[3]), lambda k: C.c_void_p(256 * (k + 1)), C.c_int
null = C.c_void_p(0)
calls = {
    "trtri": lambda T: (null, i(n), p(0), i(n), p(1), p(2), i(n), p(3), i(4096)),
    "solve_prepare": lambda T: (null, i(n), p(0), i(n), p(1), p(2), p(3)),
    "solve_apply": lambda T: (null, i(n), p(0), i(n), p(1), p(2), p(3), p(4), p(5)),
    "potrf": lambda T: (null, i(n), p(0), i(n), p(1), i(n), p(2), p(3), null),
    "mirror_lower": lambda T: (null, i(n), p(0), i(n)),
}
for T in ("double", "float"):
    getattr(lib, table[f"hdk::{sys.argv[2]}<{T}>"])(*calls[sys.argv[2]](T))
"""


@pytest.mark.parametrize("launcher", ["trtri", "solve_prepare", "solve_apply", "potrf", "mirror_lower"])
def test_rows_and_columns_stay_off_grid_y(tmp_path, launcher):
    stub = str(tmp_path / "stub.so")
    version = tmp_path / "version.map"
    version.write_text("hip_4.2 { global: *; };")
    subprocess.run(["gcc", "-shared", "-fPIC", f"-Wl,--version-script={version}", "-x", "c", "-o", stub, "-"],
                   input=STUB, text=True, check=True)
    out = subprocess.run([sys.executable, "-c", CALL, LIB_PATH, launcher, "70000"], capture_output=True, text=True,
                         env={**os.environ, "LD_PRELOAD": stub}, timeout=100)
    assert out.returncode == 0, out.stderr
    grids = [tuple(map(int, line.split())) for line in out.stdout.splitlines()]
    assert grids
    assert all(1 <= x < 2**31 and 1 <= y <= 65535 and 1 <= z <= 65535 for x, y, z in grids)
