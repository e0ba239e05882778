"""The short reciprocal, root and division of the step (lattice.hpp) are correctly rounded.

Arguments are set through written populations and fields so that a result shows the reciprocal or root itself; numpy's
float32 division and root, both correctly rounded, are the reference. Bit for bit, hence no tolerance.
"""
import numpy as np
import pytest

from conftest import oracle_for
from test_gpu_ops import SIGNATURES, random_state

pytestmark = pytest.mark.gpu

F32 = np.float32


def velocity_of(mcb, shape, rho0, f1):
    """ux of cells that hold rho0 in f_0 and f1 in f_1 at rest in a uniform phase: f1 / (rho0 + f1), formed as the
    reciprocal of the density times f1."""
    nx, ny, nz = shape
    p = mcb.make_params(nx, ny, nz, tau_f=0.6, path=mcb.PATH_FUSED)
    f = np.zeros((19, nz * ny * nx), dtype=F32)
    f[0], f[1] = rho0, f1
    with mcb.Lattice(p) as lat:
        lat.init_phi(np.zeros(nz * ny * nx, dtype=F32))
        lat.write("f", f)
        lat.compute_macros()
        return lat.read("ux").ravel(), lat.read("rho").ravel()


def test_reciprocal_of_every_mantissa(gpu_lib):
    rho = np.arange(2 ** 23, dtype=np.uint32) + np.uint32(0x3F800000)      # every float of [1, 2)
    rho = rho.view(F32)
    ux, got = velocity_of(gpu_lib, (256, 256, 128), rho - F32(1), np.ones_like(rho))
    assert np.array_equal(got, rho)
    want = F32(1) / rho
    assert np.array_equal(ux, want), rho[ux != want][:8]


def test_reciprocal_across_exponents(gpu_lib):
    rng = np.random.default_rng(3)
    n = 64 ** 3
    scale = np.exp2(rng.integers(-100, 101, n)).astype(F32)
    m = (rng.integers(0, 2 ** 23, n).astype(np.uint32) + np.uint32(0x3F800000)).view(F32)
    ux, rho = velocity_of(gpu_lib, (64, 64, 64), (m - F32(1)) * scale, scale)
    assert np.array_equal(rho, m * scale)
    assert np.array_equal(ux, F32(1) / m)


def normals_of(mcb, gx, gy):
    """gradCalc at sites that see gx at x + 1, gy at y + 1 and zeros: one site per 3 x 3 x 2 cells, unit face weights."""
    sx, sy, sz = 64, 64, gx.size // 4096
    phi = np.zeros((2 * sz, 3 * sy, 3 * sx), dtype=F32)
    phi[::2, ::3, 1::3] = gx.reshape(sz, sy, sx)
    phi[::2, 1::3, ::3] = gy.reshape(sz, sy, sx)
    nz, ny, nx = phi.shape
    consts = mcb.op_consts(mcb.make_params(nx, ny, nz, bc_mode=0))
    consts.w[1] = F32(1) / F32(3)
    assert F32(3) * F32(consts.w[1]) == F32(1)
    dev = [mcb.DeviceArray.from_numpy(phi)] + [mcb.DeviceArray(phi.nbytes) for _ in range(4)]
    mcb.op("gradCalc", *dev, nx, ny, nz, consts)
    out = [d.to_numpy(phi.shape)[::2, ::3, ::3].ravel() for d in (dev[1], dev[2], dev[4])]
    for d in dev:
        d.free()
    return out


def check_normals(mcb, gx, gy):
    m = gx * gx + gy * gy
    factor = F32(1) / np.sqrt(np.maximum(m, F32(1e-9)))
    for got, want in zip(normals_of(mcb, gx, gy), (gx * factor, gy * factor, m * factor)):
        bad = got != want
        assert not bad.any(), (m[bad][:8], got[bad][:8], want[bad][:8])
    return m


def test_root_of_every_mantissa(gpu_lib):
    """Every float of [1, 4) as the squared gradient: gx carries its root, gy what the rounding of gx^2 leaves."""
    step = 2 ** 19
    for lo in range(0x3F800000, 0x40800000, step):
        want = (np.arange(step, dtype=np.uint32) + np.uint32(lo)).view(F32)
        gx = np.sqrt(want.astype(np.float64)).astype(F32)
        over = gx * gx > want
        gx[over] = np.nextafter(gx[over], F32(0))
        gy = np.sqrt(want.astype(np.float64) - (gx * gx)).astype(F32)
        assert np.array_equal(check_normals(gpu_lib, gx, gy), want)


def test_root_across_exponents(gpu_lib):
    rng = np.random.default_rng(4)
    n = 2 ** 19
    scale = np.exp2(rng.integers(-20, 63, n)).astype(F32)
    m = check_normals(gpu_lib, (rng.uniform(1, 2, n).astype(F32)) * scale, np.zeros(n, dtype=F32))
    assert m.min() < 1e-9 and m.max() > 2.0 ** 124


@pytest.mark.parametrize("exponents", [(-30, 30), (-50, -25), (50, 90)])
def test_step_with_densities_of_any_size(gpu_lib, exponents):
    """One step of written populations of size 2^e, e by plane, through the short forms: the oracle's bits."""
    mcb = gpu_lib
    nx, ny, nz = 40, 12, 24
    p = mcb.make_params(nx, ny, nz, tau_f=0.6, sigma=0.08, path=mcb.PATH_FUSED)
    bubble = [(20.0, 6.0, 12.0, 5.0)]
    scale = np.exp2(np.linspace(*exponents, nz).round()).astype(F32).reshape(1, nz, 1, 1)
    f = random_state((nz, ny, nx), seed=9)["f"] * scale
    o = oracle_for(p)
    with mcb.Lattice(p) as lat:
        lat.init_bubbles(bubble, 3.0)
        o.init(bubble, 3.0)
        lat.write("f", f)
        o.field("f")[...] = f.reshape(o.field("f").shape)
        got = lat.observables()
        o.macros()
        for k in ("rho", "ux", "uy", "uz"):
            assert np.array_equal(got[k], o.field(k), equal_nan=True), k
        lat.step(1)
        o.step(1)
        a, b = lat.read("f").reshape(19, -1), o.field("f").reshape(19, -1)     # NaN where a force meets a tiny density
        same = (a == b) | (np.isnan(a) & np.isnan(b))
        assert same.all(), (int(np.count_nonzero(~same)), a[~same][:6], b[~same][:6])
    o.close()


@pytest.mark.parametrize("name", ["momentiCalc", "collisionFluid"])
def test_operators_take_every_density(gpu_lib, name):
    """A caller's densities and populations from subnormals to near the largest float, forces of their size."""
    mcb = gpu_lib
    nx, ny, nz = 40, 10, 70
    p = mcb.make_params(nx, ny, nz, bc_mode=0, weights=mcb.WEIGHTS_LITERAL, tau_f=0.55, sigma=0.1)
    s = random_state((nz, ny, nx), seed=5)
    e = np.linspace(-147, 127, nz).round()
    for k in ("rho", "ffx", "ffy", "ffz", "f", "pxx", "pyy", "pzz", "pxy", "pxz", "pyz"):
        s[k] = (s[k].astype(np.float64) * np.exp2(e).reshape(nz, 1, 1)).astype(F32)
    for k in ("ux", "uy", "uz"):
        s[k][:, 0] = s[k][:, 0].astype(np.float64) * np.exp2(-e).reshape(nz, 1).clip(2.0 ** -120, 2.0 ** 120)
    o = oracle_for(p)
    for k, v in s.items():
        o.field(k)[...] = v
    dev = {k: mcb.DeviceArray.from_numpy(v) for k, v in s.items()}
    mcb.op(name, *[dev[k] for k in SIGNATURES[name]], nx, ny, nz, mcb.op_consts(p))
    o.stage(name)
    for k in SIGNATURES[name]:
        got, want = dev[k].to_numpy(s[k].shape), o.field(k)
        same = (got == want) | (np.isnan(got) & np.isnan(want))
        assert same.all(), (k, int(np.count_nonzero(~same)), np.argwhere(~same)[:4])
    for d in dev.values():
        d.free()
    o.close()
