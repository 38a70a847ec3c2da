"""Where a solve of the pipelined FP64 iterations goes on after a stop, and which tile and finalize
the pipelined iterations of a context run: the cases that only a deliberate choice reaches, each
with an assertion that it was reached."""
import pytest

import oracle as O
from test_gpu_parity import mk, rel
from test_gpu_pipelined import EO_TILES, RC_TILES, TILES, extents

pytestmark = pytest.mark.gpu

FIN = {"fused": "prologue", "separate": "separate"}


@pytest.mark.parametrize("fin", list(FIN))
@pytest.mark.parametrize("precision,tile", [("fp32", t) for t in range(len(TILES))]
                         + [("fp64", t) for t in range(len(TILES) + len(RC_TILES))])
def test_forced_plain_tile_is_reported(gpu, monkeypatch, precision, tile, fin):
    """the tile and finalize that the environment names are the ones the tuning report says run, on
    every lattice that the tests of the tiles use"""
    monkeypatch.setenv("YCN_TILE_PL", str(tile))
    monkeypatch.setenv("YCN_PL_FIN", fin)
    monkeypatch.setenv("YCN_ONCHIP", "0")
    Y = gpu
    name = "%dx%d" % (TILES + RC_TILES)[tile] + ("r" if tile >= len(TILES) else "")
    for scale in (0, 1, 2, 4):
        Nt, Nx = extents(tile, scale)
        p, _ = mk(Y, Nt=Nt, Nx=Nx, nNoise=2)
        p.cgPrecision = Y.YCN_CG_MIXED if precision == "fp32" else Y.YCN_CG_FP64
        with Y.Context(p) as c:
            assert c.tuning_report().endswith(f"{precision} pipelined iteration: {name}, {FIN[fin]} finalize")


@pytest.mark.parametrize("fin", list(FIN))
@pytest.mark.parametrize("tile", range(len(EO_TILES)))
def test_forced_even_odd_tile_is_reported(gpu, monkeypatch, tile, fin):
    monkeypatch.setenv("YCN_TILE_PL", str(tile))
    monkeypatch.setenv("YCN_EO_FIN", fin)
    Y = gpu
    for scale in (1, 2, 3):
        Nt, Nx = scale * EO_TILES[tile][0], scale * EO_TILES[tile][1]
        if Nx % 32 and Nt % 16:
            Nx *= 2
        p, _ = mk(Y, Nt=Nt, Nx=Nx, nNoise=2)
        p.evenOdd = 1
        with Y.Context(p) as c:
            assert "fp64 pipelined iteration: %dx%d, %s finalize" % (*EO_TILES[tile], FIN[fin]) in c.tuning_report()


@pytest.mark.parametrize("fin", list(FIN))
def test_even_odd_solve_goes_on_from_its_stop(gpu, monkeypatch, fin):
    """A context's first solve starts from tol |r_0|, here too loose a threshold: it stops above the
    tolerance and goes on with a lower one from the residual and the direction that the close
    brought up.  The same solve again starts from the threshold that the first one needed, and takes
    one phase.  Both are one CG, so their iteration counts differ by what the thresholds leave: a
    factor of 2 in the residual, five iterations at the rate of this system, and two of parity.  One
    that began anew from x would need tens more."""
    monkeypatch.setenv("YCN_EO_FIN", fin)
    Y = gpu
    Nt, Nx = 48, 64
    p, orc = mk(Y, Nt=Nt, Nx=Nx, M=0.05, g=0.5, cgTol=1e-10, cgTolMode=1, cgMaxIter=20000)
    p.evenOdd = 1
    phi = O.hot_start(9, Nt, Nx)
    dr, _ = O.fermion_drift(orc, phi, 3)
    with Y.Context(p) as c:
        assert FIN[fin] + " finalize" in c.tuning_report().split("fp64 pipelined iteration:")[1]
        c.set_field(phi)
        (d1, first), (d2, second) = c.fermion_force(3), c.fermion_force(3)
    print(f"# first {first}, second {second}", flush=True)
    for d, st in ((d1, first), (d2, second)):
        assert st["converged"] == 1 and st["true_rel_resid"] <= 1e-10
        assert rel(d, dr) < 1e-8
    assert first["restarts"] > 0 and second["restarts"] == 0
    assert abs(first["iters"] - second["iters"]) <= 7


@pytest.mark.parametrize("fin", list(FIN))
@pytest.mark.parametrize("tile", [1, len(TILES)])
def test_plain_solve_restarts_from_its_true_residual(gpu, monkeypatch, tile, fin):
    """A tolerance below what rounding leaves between the recursive residual and the true one (about
    1.5e-15 of |b| on such lattices): the solve restarts, a second phase beginning with the first launch's
    form, and gets there."""
    monkeypatch.setenv("YCN_TILE_PL", str(tile))
    monkeypatch.setenv("YCN_PL_FIN", fin)
    monkeypatch.setenv("YCN_ONCHIP", "0")
    Y = gpu
    p, orc = mk(Y, Nt=45, Nx=50, cgTol=1e-15, cgTolMode=1, cgMaxIter=20000)
    phi = 1.0 + O.hot_start(8, 45, 50)
    with Y.Context(p) as c:
        c.set_field(phi)
        d, st = c.fermion_force(3)
    print(f"# {st}", flush=True)
    assert st["restarts"] > 0
    assert st["converged"] == 1 and st["true_rel_resid"] <= 1e-15
    orc.cgTol = 1e-13
    assert rel(d, O.fermion_drift(orc, phi, 3)[0]) < 1e-10
