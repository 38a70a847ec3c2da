"""The coloured-noise filter where its FFT plan and its launches turn: every radix, odd
primes beyond them, odd extents, the longest line, lattices on both sides of the one-block
form, and a column count that is no multiple of a block's, against the oracle's FFT (1e-12 of
the largest value, the bar of the other filter tests)."""
import numpy as np
import pytest

import oracle as O
from test_gpu_parity import RTOL, mk, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nt,Nx,s,chains", [(2, 2, 1.0, 1), (3, 7, 1.0, 1), (8, 16, 0.5, 3), (128, 32, 0.25, 1),
                                            (22, 26, 1.0, 2), (45, 50, 0.25, 4), (63, 75, 0.7, 1), (68, 66, 1.0, 1),
                                            (17, 2048, 0.5, 1), (2048, 6, 1.0, 1), (210, 128, 0.3, 2),
                                            (31, 1021, 0.5, 1), (256, 512, 0.0, 1)])
def test_filter_plans(gpu, Nt, Nx, s, chains):
    Y = gpu
    p, _ = mk(Y, Nt=Nt, Nx=Nx, cutFraction=s, nReplicas=chains)
    xi = np.random.default_rng(Nt * 10 + Nx).standard_normal((chains, Nt, Nx))
    with Y.Context(p) as c:
        got = c.coloured_filter(xi).reshape(chains, Nt, Nx)
    for k in range(chains):
        assert rel(got[k], O.coloured_filter(xi[k], s)) < RTOL, k


@pytest.mark.parametrize("Nt,Nx", [(5, 9), (6, 10), (70, 64), (64, 81)])
def test_generated_field(gpu, Nt, Nx):
    """The generated field at odd and even row lengths (one or two sites per Philox call)."""
    Y = gpu
    p, orc = mk(Y, Nt=Nt, Nx=Nx, seed=2 ** 40 + 5, cutFraction=0.5)
    with Y.Context(p) as c:
        got = c.coloured_noise(2 ** 33 + 1)
    assert rel(got, O.coloured_noise(orc, 2 ** 33 + 1)) < RTOL


@pytest.mark.parametrize("Nt,Nx,s,chains", [(40, 48, 1.0, 1), (96, 160, 0.7, 2), (128, 256, 0.5, 1), (512, 64, 1.0, 1),
                                            (6, 1024, 0.4, 3), (320, 2048, 0.3, 1), (1536, 34, 1.0, 1)])
def test_powers_of_two(gpu, Nt, Nx, s, chains):
    """Every split of a power of two 2^3 ... 2^11 into radix-8 and radix-4 passes, alone and with an
    odd factor, with blocks of 64 to 512 threads."""
    test_filter_plans(gpu, Nt, Nx, s, chains)
