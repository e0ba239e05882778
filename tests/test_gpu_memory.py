"""Contexts where device memory is short: padded rows are given up before the context is.

A child process puts its own hipMalloc before the runtime's, which refuses blocks above a limit.
"""
import os
import subprocess
import sys

import pytest

from conftest import PKG

pytestmark = pytest.mark.gpu

HIP_MALLOC = """
#include <dlfcn.h>
#include <stddef.h>
static size_t limit = (size_t)-1;
static int refused = 0;
void set_limit(size_t n) { limit = n; }
int refusals(void) { return refused; }
int hipMalloc(void** p, size_t n) {
    static int (*next)(void**, size_t);
    if (n > limit) { ++refused; return 2; }   /* hipErrorOutOfMemory */
    if (!next) next = (int (*)(void**, size_t))dlsym(dlopen("libamdhip64.so", RTLD_NOW), "hipMalloc");
    return next(p, n);
}
"""

CHILD = """
import ctypes, sys
import numpy as np
short = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
import mcb
nx, ny, nz, storage, tau_g = (float(v) if "." in v else int(v) for v in sys.argv[3:])
p = mcb.make_params(nx, ny, nz, storage=storage, tau_f=0.6, tau_g=tau_g)
bubble = [(0.4 * nx, 0.5 * ny, 0.5 * nz, 0.3 * min(nx, ny, nz))]
plain = 19 * (nx * ny + 63) // 64 * 64 * nz * (2 if storage else 4)
short.set_limit(ctypes.c_size_t(plain + plain // 8))
lat = mcb.Lattice(p)
lat.init_bubbles(bubble, 3.0)
assert short.refusals() > 0, "nothing was refused"
short.set_limit(ctypes.c_size_t(-1))
with mcb.Batch(storage) as b:
    cid = b.add(p, bubble, 3.0)
    lat.step(5)
    b.step(5)
    for k in ("phi", "f"):
        assert np.array_equal(lat.read(k), b.read(cid, k)), k
lat.close()
print("same")
"""


@pytest.mark.parametrize("storage,tau_g", [(0, 0.8), (0, 1.0), (1, 1.0)])
def test_context_takes_plain_rows_where_padded_ones_do_not_fit(gpu_lib, tmp_path, storage, tau_g):
    src, so = tmp_path / "short.c", tmp_path / "libshort.so"
    src.write_text(HIP_MALLOC)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", str(src), "-o", str(so), "-ldl"], check=True)
    got = subprocess.run([sys.executable, "-c", CHILD, str(so), os.path.abspath(PKG), "65", "40", "40", str(storage), str(tau_g)],
                         capture_output=True, text=True, timeout=100)
    assert got.returncode == 0 and got.stdout.strip().endswith("same"), got.stdout + got.stderr
