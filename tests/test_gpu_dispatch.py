"""The step at the sizes where its tiles, chunks and launches change.

FP32: bit for bit against the oracle, on lattices whose phase pass runs single
planes, partial tiles, chunks that do not divide the lattice, and one or more
full rounds of workgroups.
"""
import ctypes

import numpy as np
import pytest

from conftest import f32_bubbles, oracle_for

pytestmark = pytest.mark.gpu

FIELDS = ("phi", "rho", "ux", "uy", "uz")


def fp32_matches_oracle(mcb, steps, nx, ny, nz, **kw):
    p = mcb.make_params(nx, ny, nz, tau_f=0.6, sigma=0.08, **kw)
    bub = f32_bubbles([(0.43 * nx, 0.55 * ny, 0.48 * nz, 0.3 * min(nx, ny, nz))])
    lat = mcb.Lattice(p)
    lat.init_bubbles(bub, 3.0)
    lat.step(steps)
    got = lat.observables()
    lat.close()
    o = oracle_for(p)
    o.init(bub, 3.0)
    o.step(steps)
    o.macros()
    for k in FIELDS:
        assert np.array_equal(got[k], o.field(k)), (k, int(np.count_nonzero(got[k] != o.field(k))))
    o.close()


@pytest.mark.parametrize("normals", [1, 2])
@pytest.mark.parametrize("nx,ny,nz", [(64, 9, 3), (65, 17, 5), (70, 16, 67), (33, 31, 130), (16, 10, 40), (130, 24, 21)])
def test_phase_pass_chunks(gpu_lib, nx, ny, nz, normals):
    fp32_matches_oracle(gpu_lib, 5, nx, ny, nz, tau_g=1.0, normals=normals)


def test_phase_pass_ghost_layers(gpu_lib):
    fp32_matches_oracle(gpu_lib, 6, 66, 19, 70, tau_g=1.0, bc_mode=gpu_lib.BC_REFERENCE, weights=gpu_lib.WEIGHTS_LITERAL)


@pytest.mark.parametrize("nx,ny,nz,tau_g", [(64, 64, 5, 0.8), (64, 70, 64, 1.0), (40, 33, 29, 1.0), (96, 20, 40, 0.8),
                                            (16, 24, 18, 1.0)])
def test_small_lattice_tiles(gpu_lib, nx, ny, nz, tau_g):
    fp32_matches_oracle(gpu_lib, 4, nx, ny, nz, tau_g=tau_g)


def alone(mcb, p, bubble, steps):
    lat = mcb.Lattice(p)
    lat.init_bubbles([bubble], 3.0)
    lat.step(steps)
    phi = lat.read("phi")
    lat.close()
    return phi


@pytest.mark.parametrize("storage", [0, 1])
def test_batch_groups_side_by_side(gpu_lib, storage):
    """Cases of several tile shapes, one shape large enough to be split over two lanes: every case as if alone, across
    steps, a join at odd parity and a leave."""
    mcb = gpu_lib
    sides = [(192, 160, 150), (192, 160, 150), (48, 40, 20), (96, 33, 17), (32, 32, 32), (70, 21, 30)]
    with mcb.Batch(storage) as b:
        ids = []
        for i, (nx, ny, nz) in enumerate(sides):
            p = mcb.make_params(nx, ny, nz, storage=storage, tau_f=0.55 + 0.02 * i)
            bub = (0.4 * nx, 0.5 * ny, 0.6 * nz, 0.28 * min(nx, ny, nz))
            if i == 4:
                b.step(3)
            ids.append((b.add(p, [bub], 3.0), p, bub, 7 if i < 4 else 4))
        b.step(1)
        gone = ids.pop(3)
        b.remove(gone[0])
        b.step(3)
        for cid, p, bub, steps in ids:
            got, want = b.read(cid, "phi"), alone(mcb, p, bub, steps)
            assert np.array_equal(got, want), (p.nx, p.ny, p.nz, int(np.count_nonzero(got != want)))


@pytest.mark.parametrize("nx,ny,nz", [(33, 5, 7), (50, 9, 6), (64, 5, 9), (65, 11, 5), (100, 4, 6), (31, 13, 20)])
@pytest.mark.parametrize("storage,tau_g", [(0, 1.0), (0, 0.8), (1, 1.0), (1, 0.8), (2, 1.0)])
def test_population_rows_of_any_length(gpu_lib, storage, tau_g, nx, ny, nz):
    """Populations written and read in the reference layout, through the padded rows and partial blocks of a context, and
    a state image taken to a batch case, whose rows are not padded."""
    mcb = gpu_lib
    p = mcb.make_params(nx, ny, nz, storage=storage, tau_f=0.7, tau_g=tau_g)
    w = np.array([1 / 3] + [1 / 18] * 6 + [1 / 36] * 12).reshape(19, 1, 1, 1)
    rng = np.random.default_rng(nx)
    f = (w * (1.0 + rng.normal(0.0, 1e-2, (19, nz, ny, nx)))).astype(np.float32)
    lat = mcb.Lattice(p)
    lat.init_bubbles([(0.5 * nx, 0.5 * ny, 0.5 * nz, 0.3 * min(nx, ny, nz))], 3.0)
    lat.step(1)
    lat.write("f", f)
    back = lat.read("f")
    if storage == 0:
        assert np.array_equal(back, f)
    else:   # one 16-bit rounding of the offset from w_l per link, folded into the rest link
        assert np.abs(back - f).max() < (2.0 ** -11 if storage == 1 else 2.0 ** -8) * 0.2 * w.max() * 2
    image = lat.save_state()
    lat.step(3)
    with mcb.Batch(storage) as b:
        cid = b.add_state(image)
        b.step(3)
        assert np.array_equal(b.read(cid, "phi"), lat.read("phi"))
        assert np.array_equal(b.read(cid, "f"), lat.read("f"))
    other = mcb.Lattice(p)
    other.load_state(image)
    other.step(3)
    assert np.array_equal(other.read("f"), lat.read("f"))
    lat.close()
    other.close()


def test_16bit_image_with_written_g_moves_between_context_and_batch(gpu_lib):
    """A moment-form case whose g was written keeps populations and their FP64 mass sums, tile by tile: the same tiles in a
    context, whose moment form uses others, and in a batch."""
    mcb = gpu_lib
    nx, ny, nz = 60, 24, 40
    p = mcb.make_params(nx, ny, nz, storage=1, tau_f=0.7, tau_g=1.0)
    lat = mcb.Lattice(p)
    lat.init_bubbles([(30.0, 12.0, 20.0, 7.0)], 3.0)
    lat.step(2)
    lat.write("g", lat.read("g"))
    lat.step(1)
    image = lat.save_state()
    lat.step(4)
    with mcb.Batch(1) as b:
        cid = b.add_state(image)
        b.step(4)
        assert np.array_equal(b.read(cid, "phi"), lat.read("phi"))
    with mcb.Lattice(p) as other:
        other.load_state(image)
        other.step(4)
        assert np.array_equal(other.read("phi"), lat.read("phi"))
    lat.close()


@pytest.mark.parametrize("storage,tau_g,nx,ny,nz", [
    (0, 1.0, 33, 24, 60), (0, 0.8, 72, 33, 20), (0, 0.8, 48, 16, 9), (0, 1.0, 160, 64, 40), (0, 0.8, 130, 70, 33),
    (1, 1.0, 96, 40, 24), (1, 1.0, 144, 36, 30), (1, 1.0, 112, 20, 50), (1, 1.0, 40, 30, 20), (2, 1.0, 200, 90, 70)])
def test_tiles_of_a_lattice_alone(gpu_lib, storage, tau_g, nx, ny, nz):
    """The tile that a context picks against tiles of 16x16x3: no cell's arithmetic depends on its tile."""
    mcb = gpu_lib
    p = mcb.make_params(nx, ny, nz, storage=storage, tau_f=0.7, tau_g=tau_g)
    got = []
    for tiling in (None, (16, 16, 3)):
        lat = mcb.Lattice(p)
        if tiling:
            lat.set_tiling(*tiling)
        lat.init_bubbles([(0.4 * nx, 0.5 * ny, 0.5 * nz, 0.3 * min(nx, ny, nz))], 3.0)
        lat.step(6)
        got.append((lat.read("phi"), lat.read("f")))
        lat.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("storage", [1, 2])
@pytest.mark.parametrize("nx,ny,nz", [(33, 13, 70), (64, 64, 33), (80, 9, 40), (112, 10, 17), (130, 66, 35), (20, 18, 50)])
def test_mass_sum_of_stored_g_alone(gpu_lib, storage, nx, ny, nz):
    """A context sums phi on a batch case's tiles whatever tiles it steps on: the bits of the correction are the same."""
    mcb = gpu_lib
    p = mcb.make_params(nx, ny, nz, storage=storage, tau_f=0.6, tau_g=0.8)
    bubble = [(0.4 * nx, 0.5 * ny, 0.5 * nz, 0.3 * min(nx, ny, nz))]
    with mcb.Lattice(p) as lat, mcb.Batch(storage) as b:
        lat.init_bubbles(bubble, 3.0)
        lat.step(8)
        phi0 = lat.read("phi")
        cid = b.add_state(lat.save_state())
        lat.step(8)
        b.step(8)
        assert np.array_equal(b.read(cid, "phi"), lat.read("phi"))
        assert abs(float(lat.read("phi").sum(dtype=np.float64)) - float(phi0.sum(dtype=np.float64))) <= 1e-3


@pytest.mark.parametrize("storage,nx,ny,nz", [(1, 64, 8, 33), (2, 65, 9, 20), (1, 130, 31, 17), (2, 64, 7, 24), (1, 256, 200, 130),
                                              (2, 128, 64, 48)])
def test_phase_tiles_of_16_bit_cases(gpu_lib, storage, nx, ny, nz):
    """The phase pass of a large lattice alone on 8-row tiles with longer chunks (256x200x130), against 4 rows and a batch."""
    mcb = gpu_lib
    p = mcb.make_params(nx, ny, nz, storage=storage, tau_f=0.6)
    bubble = [(0.4 * nx, 0.5 * ny, 0.5 * nz, 0.3 * min(nx, ny, nz))]
    got = []
    for tiling in (None, (64, 4, 16)):
        with mcb.Lattice(p) as lat, mcb.Batch(storage) as b:
            cid = b.add(p, bubble, 3.0)
            lat.init_bubbles(bubble, 3.0)
            if tiling:
                lat.set_tiling(*tiling)
                b.set_tiling(cid, *tiling)
            lat.step(6)
            b.step(6)
            got += [lat.read("phi"), lat.read("f"), b.read(cid, "phi"), b.read(cid, "f")]
    for a, b in zip(got[:4], got[4:]):
        assert np.array_equal(a, b)
    assert np.array_equal(got[0], got[2])


@pytest.mark.parametrize("storage,nx,ny,nz", [(1, 256, 200, 130), (2, 200, 200, 150), (1, 64, 8, 33)])
def test_macros_of_a_case_with_phase_tiles_of_its_own(gpu_lib, storage, nx, ny, nz):
    """The macro pass runs its phase pass on the case's phase tiles, each cell once (200x200x150 and 256x200x130 have tiles
    of their own, 64x8x33 has not): the fields, and the steps and mass corrections after it, are those of 64x4 tiles."""
    mcb = gpu_lib
    p = mcb.make_params(nx, ny, nz, storage=storage, tau_f=0.6)
    bubble = [(0.4 * nx, 0.5 * ny, 0.5 * nz, 0.3 * min(nx, ny, nz))]
    got = []
    for tiling in (None, (64, 4, 16)):
        with mcb.Lattice(p) as lat:
            if tiling:
                lat.set_tiling(*tiling)
            lat.init_bubbles(bubble, 3.0)
            out = [lat.observables()]     # before the first step: phi from the initial populations
            for steps in (1, 4, 3):
                lat.step(steps)
                out.append(lat.observables())
            out.append({"f": lat.read("f")})
            got.append(out)
    for a, b in zip(*got):
        for k in a:
            assert np.array_equal(a[k], b[k]), (k, int(np.count_nonzero(a[k] != b[k])))


@pytest.mark.parametrize("nx", [15, 17, 29, 30, 34, 63, 64, 66, 97, 128])
@pytest.mark.parametrize("storage,tau_g", [(0, 1.0), (0, 0.8), (1, 0.8), (2, 1.0)])
def test_rows_around_the_padding_rule(gpu_lib, storage, tau_g, nx):
    """Contexts with padded rows and with plain ones against a batch case, whose rows are plain, and its own tiles."""
    mcb = gpu_lib
    p = mcb.make_params(nx, 11, 19, storage=storage, tau_f=0.65, tau_g=tau_g)
    bubble = [(0.4 * nx, 5.0, 9.0, 3.3)]
    with mcb.Lattice(p) as lat, mcb.Batch(storage) as b:
        lat.init_bubbles(bubble, 3.0)
        cid = b.add(p, bubble, 3.0)
        lat.step(7)
        b.step(7)
        for k in ("phi", "f", "g"):
            assert np.array_equal(lat.read(k), b.read(cid, k)), k
        got, want = lat.observables(), b.observables(cid)
        for k in FIELDS:
            assert np.array_equal(got[k], want[k]), k


@pytest.mark.parametrize("tau_g", [1.0, 0.8])
@pytest.mark.parametrize("sides,other", [((32, 32), 48), ((80, 80), 33), ((48, 144), 176), ((24, 24), 96), ((112, 112), 16)])
def test_fp32_batch_shapes_change_as_cases_join_and_leave(gpu_lib, sides, other, tau_g):
    """A batch of one tile shape, with a case of another shape for some steps, and one whose tile the caller sets."""
    mcb = gpu_lib

    def case(n):
        return mcb.make_params(n, 20, 18, tau_f=0.6, tau_g=tau_g), (0.4 * n, 10.0, 9.0, 5.0)

    with mcb.Batch(0) as b:
        ids = [b.add(case(n)[0], [case(n)[1]], 3.0) for n in sides]
        b.step(3)
        extra = b.add(case(other)[0], [case(other)[1]], 3.0)
        b.step(2)
        b.set_tiling(ids[0], 16, 16, 5)
        b.step(2)
        got = {"extra": b.read(extra, "phi")}
        want = {"extra": alone(mcb, case(other)[0], case(other)[1], 4)}
        b.remove(extra)
        b.step(4)
        for i, n in zip(ids, sides):
            got[i], want[i] = b.read(i, "phi"), alone(mcb, case(n)[0], case(n)[1], 11)
        for k in got:
            assert np.array_equal(got[k], want[k]), k


@pytest.mark.parametrize("storage,sides", [(1, [(192, 160, 150)] * 2), (0, [(192, 160, 150), (160, 150, 200)]),
                                           (0, [(192, 160, 150)] * 6)])
def test_large_batch_as_halves_and_whole(gpu_lib, storage, sides):
    """Calls of one step run the batch whole, longer ones as two halves side by side (the last is too large for that)."""
    mcb = gpu_lib
    with mcb.Batch(storage) as b:
        cases = []
        for i, (nx, ny, nz) in enumerate(sides):
            p = mcb.make_params(nx, ny, nz, storage=storage, tau_f=0.55 + 0.02 * i)
            bub = ((0.4 + 0.05 * i) * nx, 0.5 * ny, 0.6 * nz, 0.28 * min(nx, ny, nz))
            cases.append((b.add(p, [bub], 3.0), p, bub))
        for steps in (2, 1, 3, 1, 1, 4):
            b.step(steps)
        for cid, p, bub in cases:
            assert np.array_equal(b.read(cid, "phi"), alone(mcb, p, bub, 12)), cid


@pytest.mark.parametrize("storage,sides", [(1, [32, 48, 33, 64, 80]), (1, [(192, 160, 150)] * 2), (0, [32, 48, 70])])
def test_batch_steps_inside_a_caller_graph(gpu_lib, storage, sides):
    """A caller that captures the batch's stream gets every group and every half recorded there; replays, with the batch's
    own steps and reads between them, advance it like the same steps launched directly."""
    mcb = gpu_lib
    hip = ctypes.CDLL("libamdhip64.so")
    vp = ctypes.c_void_p
    stream, graph, exe = vp(), vp(), vp()
    assert hip.hipStreamCreate(ctypes.byref(stream)) == 0
    with mcb.Batch(storage, stream=stream) as g, mcb.Batch(storage) as e:
        ids = []
        for i, n in enumerate(sides):
            nx, ny, nz = (n, 20, 18) if isinstance(n, int) else n
            p = mcb.make_params(nx, ny, nz, storage=storage, tau_f=0.6, tau_g=0.8 if i % 2 else 1.0)
            bub = [(0.4 * nx, 0.5 * ny, 0.5 * nz, 0.3 * min(nx, ny, nz))]
            ids.append((g.add(p, bub, 3.0), e.add(p, bub, 3.0)))
        g.step(1)
        e.step(1)
        g.synchronize()
        assert hip.hipStreamBeginCapture(stream, 1) == 0          # thread-local mode
        g.step(2)                                                 # recorded, not run
        assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
        assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
        for replay in range(4):
            assert hip.hipGraphLaunch(exe, stream) == 0
            g.step(2)
            e.step(4)
            for a, b in ids:
                x, y = g.read(a, "phi"), e.read(b, "phi")
                assert np.array_equal(x, y), (replay, a, int(np.count_nonzero(x != y)))
        hip.hipGraphExecDestroy(exe)
        hip.hipGraphDestroy(graph)
    hip.hipStreamDestroy(stream)


@pytest.mark.parametrize("storage,tau_g,nx,ny,nz", [(0, 1.0, 40, 36, 44), (0, 0.8, 40, 36, 44), (1, 1.0, 66, 20, 50), (1, 0.8, 48, 30, 20)])
def test_autotuned_context(gpu_lib, storage, tau_g, nx, ny, nz):
    """The tuner measures what a context runs, the rule's tile among the rest: contexts of the same form of g take its
    choice, others keep the rule's, and no choice changes a result."""
    mcb = gpu_lib
    p = mcb.make_params(nx, ny, nz, storage=storage, tau_f=0.6, tau_g=tau_g)
    q = mcb.make_params(nx, ny, nz, storage=storage, tau_f=0.6, tau_g=1.8 - tau_g)
    bub = (0.4 * nx, 0.5 * ny, 0.5 * nz, 0.3 * min(nx, ny, nz))

    def tiling(params):
        with mcb.Lattice(params) as lat:
            return lat.tiling()

    rule, other = tiling(p), tiling(q)
    want = alone(mcb, p, bub, 6)
    tx, ty, zc, ms = mcb.autotune(p)
    assert ms > 0 and tiling(p) == (tx, ty, zc) and tiling(q) == other
    assert np.array_equal(alone(mcb, p, bub, 6), want)
    with mcb.Lattice(p) as lat, mcb.Batch(storage) as b:
        lat.init_bubbles([bub], 3.0)
        lat.step(3)
        cid = b.add_state(lat.save_state())
        lat.step(3)
        b.step(3)
        assert np.array_equal(lat.read("phi"), b.read(cid, "phi"))
    # From the tuned state the rule's tile is still a candidate.
    assert mcb.autotune(p)[:2] in mcb.tilings() and rule[:2] in mcb.tilings()


@pytest.mark.parametrize("tau_gs", [(1.0,), (0.8, 1.0)])
@pytest.mark.parametrize("sides", [[(48, 40, 40), (64, 40, 40), (32, 40, 50)] * 6, [(192, 160, 80), (32, 40, 40)] * 5])
def test_fp32_batch_shape_by_shape(gpu_lib, sides, tau_gs):
    """Enough cases of each shape: longer calls step shape by shape (the second batch with its largest one in two), calls
    of one step all together; with a case that leaves, which changes the order."""
    mcb = gpu_lib
    with mcb.Batch(0) as b:
        cases = []
        for i, (nx, ny, nz) in enumerate(sides):
            p = mcb.make_params(nx, ny, nz, tau_f=0.55 + 0.01 * i, tau_g=tau_gs[i % len(tau_gs)])
            bub = ((0.3 + 0.02 * i) * nx, 0.5 * ny, 0.6 * nz, 0.28 * min(nx, ny, nz))
            cases.append((b.add(p, [bub], 3.0), p, bub))
        for steps in (3, 1, 2):
            b.step(steps)
        b.remove(cases.pop(1)[0])
        for steps in (1, 4):
            b.step(steps)
        for cid, p, bub in cases:
            assert np.array_equal(b.read(cid, "phi"), alone(mcb, p, bub, 11)), cid
