"""The step at the sizes where its tiles, chunks and launches change.

FP32: bit for bit against the oracle, on lattices whose phase pass runs single
planes, partial tiles, chunks that do not divide the lattice, and one or more
full rounds of workgroups.
"""
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
