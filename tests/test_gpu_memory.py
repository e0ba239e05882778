"""Where the runtime refuses: padded rows are given up before the context is, the ring of large reads before the read.

A child process puts its own hipMalloc and hipEventCreateWithFlags before the runtime's, which refuse on request.
"""
import os
import subprocess
import sys

import pytest

from conftest import PKG

pytestmark = pytest.mark.gpu

HIP = """
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
static int no_events = 0;
void refuse_events(int on) { no_events = on; }
int hipEventCreateWithFlags(void** e, unsigned flags) {
    static int (*next)(void**, unsigned);
    if (no_events && no_events-- == 1) { no_events = 1; ++refused; return 2; }   /* after no_events - 1 more */
    if (!next) next = (int (*)(void**, unsigned))dlsym(dlopen("libamdhip64.so", RTLD_NOW), "hipEventCreateWithFlags");
    return next(e, flags);
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

READ_CHILD = """
import ctypes, sys
import numpy as np
short = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
import mcb
phi = np.random.default_rng(1).random((128, 96, 130), dtype=np.float32)
lat = mcb.Lattice(mcb.make_params(130, 96, 128))
lat.init_phi(phi)
for left in (1, 3):      # the first or the third event is refused
    short.refuse_events(left)
    got = lat.read("phi")
    assert short.refusals() > 0, "nothing was refused"
    short.refuse_events(0)
    assert np.array_equal(got, phi)
assert np.array_equal(lat.read("phi"), phi)
lat.close()
print("same")
"""


def run_child(tmp_path, code, *args):
    src, so = tmp_path / "short.c", tmp_path / "libshort.so"
    src.write_text(HIP)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", str(src), "-o", str(so), "-ldl"], check=True)
    got = subprocess.run([sys.executable, "-c", code, str(so), os.path.abspath(PKG), *args], capture_output=True, text=True,
                         timeout=100)
    assert got.returncode == 0 and got.stdout.strip().endswith("same"), got.stdout + got.stderr


@pytest.mark.parametrize("storage,tau_g", [(0, 0.8), (0, 1.0), (1, 1.0)])
def test_context_takes_plain_rows_where_padded_ones_do_not_fit(gpu_lib, tmp_path, storage, tau_g):
    run_child(tmp_path, CHILD, "65", "40", "40", str(storage), str(tau_g))


def test_large_read_without_the_ring_where_events_are_refused(gpu_lib, tmp_path):
    run_child(tmp_path, READ_CHILD)
