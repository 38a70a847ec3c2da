"""The fermion force runs on packed real spinors (D and eta are real); public solves with a
complex right-hand side keep the complex form.  Both against the oracle where the packing
could go wrong: lattices without a tile, the smallest extents, r != 1, several chains and
noise vectors.  Fixed iteration counts, so the iterates agree to rounding: 1e-12."""
import numpy as np
import pytest

import oracle as O
from test_gpu_parity import RTOL, mk, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nt,Nx,r,vectors", [(2, 2, 1.0, 1), (3, 5, 1.0, 2), (7, 32, 0.0, 1), (8, 64, 0.7, 3),
                                             (16, 16, 1.0, 1)])
def test_packed_force(gpu, Nt, Nx, r, vectors):
    Y = gpu
    # few iterations: on the smallest lattices CG reaches rounding level after that
    p, orc = mk(Y, Nt=Nt, Nx=Nx, r=r, nNoise=vectors, cgTol=0.0, cgTolMode=0, cgMaxIter=4 if Nt * Nx < 16 else 12)
    phi = 1.0 + O.hot_start(Nt + Nx, Nt, Nx)
    with Y.Context(p) as c:
        c.set_field(phi)
        d, st = c.fermion_force(3)
    dr, sr = O.fermion_drift(orc, phi, 3)
    assert vectors * st["iters"] == sr["iters"]   # the oracle adds up its solves
    assert rel(d, dr) < RTOL


def test_complex_solve_after_packed_force(gpu):
    """A complex right-hand side on a context whose buffers a packed solve has just used."""
    Y = gpu
    Nt, Nx = 16, 32
    p, orc = mk(Y, Nt=Nt, Nx=Nx, cgTol=0.0, cgTolMode=0, cgMaxIter=15)
    phi = 1.0 + O.hot_start(4, Nt, Nx)
    rng = np.random.default_rng(1)
    b = rng.standard_normal((Nt * Nx, 4)) + 1j * rng.standard_normal((Nt * Nx, 4))
    with Y.Context(p) as c:
        c.set_field(phi)
        c.fermion_force(0)
        x, _ = c.cg_solve(b)
    xr, _ = O.cg(orc, phi, b, Y.YCN_DAGGER)
    assert rel(x, xr) < RTOL
