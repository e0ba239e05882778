"""Reads of large fields pass through a ring of pinned memory in chunks, moved by several threads: the sizes around its
chunk and thread rules, into memory the library does not know, against a copy of the same device memory."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# Cells (4 bytes each): below the ring's least size, at it, a ragged last chunk and slice, a little past four chunks, the
# larger chunk's least size and a ragged size above it.
SHAPES = [(64, 64, 255), (64, 64, 256), (128, 96, 101), (1049, 4, 500), (256, 128, 128), (250, 149, 131)]


@pytest.mark.parametrize("nx,ny,nz", SHAPES)
@pytest.mark.parametrize("storage", [0, 1])
def test_large_reads_return_every_cell(gpu_lib, nx, ny, nz, storage):
    mcb = gpu_lib
    phi = np.random.default_rng(nx).random(nx * ny * nz, dtype=np.float32)
    with mcb.Lattice(mcb.make_params(nx, ny, nz, storage=storage)) as lat:
        lat.init_phi(phi)
        for _ in range(3):
            assert np.array_equal(np.asarray(lat.read("phi")).ravel(), phi)


def test_reads_of_two_threads_at_once(gpu_lib):
    mcb = gpu_lib
    n = 128
    fields = [np.random.default_rng(i).random(n ** 3, dtype=np.float32) for i in range(2)]
    lats = [mcb.Lattice(mcb.make_params(n, n, n)) for _ in fields]
    for lat, phi in zip(lats, fields):
        lat.init_phi(phi)
    same = [[], []]

    def read(i):
        for _ in range(8):
            same[i].append(np.array_equal(np.asarray(lats[i].read("phi")).ravel(), fields[i]))

    threads = [threading.Thread(target=read, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert same == [[True] * 8] * 2
    for lat in lats:
        lat.close()


@pytest.mark.parametrize("nx,ny,nz", [(9, 7, 5), (16, 16, 31), (16, 16, 32), (17, 31, 16), (128, 64, 128)])
@pytest.mark.parametrize("storage", [0, 1])
def test_populations_read_as_rows_of_any_size(gpu_lib, nx, ny, nz, storage):
    """f and g, whose 19 rows share one wait below 32 KiB, wait one by one above and pass through the ring from 4 MiB on:
    a context's reads against a batch case's, and phi as the sum of g."""
    mcb = gpu_lib
    p = mcb.make_params(nx, ny, nz, storage=storage, tau_f=0.6, tau_g=0.8)
    bubble = [(0.5 * nx, 0.5 * ny, 0.5 * nz, 0.3 * min(nx, ny, nz))]
    with mcb.Lattice(p) as lat, mcb.Batch(storage) as b:
        lat.init_bubbles(bubble, 3.0)
        cid = b.add(p, bubble, 3.0)
        lat.step(2)
        b.step(2)
        f, g = lat.read("f"), lat.read("g")
        assert np.array_equal(f, b.read(cid, "f")) and np.array_equal(g, b.read(cid, "g"))
        lat.compute_macros()
        tol = 19 * 2.0 ** -23 if storage == 0 else 2.0 ** -10     # sums in another order; 16 bits: the mass correction
        assert np.abs(g.sum(axis=0, dtype=np.float64) - lat.read("phi")).max() <= tol
        if storage == 0:
            assert np.abs(f.sum(axis=0, dtype=np.float64) - lat.read("rho")).max() <= tol
