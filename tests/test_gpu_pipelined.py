"""The plain solvers' pipelined iterations, FP32 (mixed precision) and FP64: every tile with either
finalize, on several systems at once, on the smallest lattice each tile takes and on lattices that
it does not divide; odd iteration caps, which end after an even launch whose x update is still to
be added; caps on both sides of a captured chunk's end; restarts from the true residual."""
import numpy as np
import pytest

import oracle as O
from test_gpu_parity import RTOL, mk, rel

pytestmark = pytest.mark.gpu

TILES = [(4, 16), (8, 32), (16, 16), (16, 32), (32, 32), (8, 64), (16, 64)]


def extents(tile, scale):
    """scale tiles each way; scale 0: two tiles and a part in time, one and a small part in space."""
    TT, TX = (TILES + RC_TILES)[tile]
    return (scale * TT, scale * TX) if scale else (2 * TT + 3, TX + (1 if tile < len(TILES) else 3))


@pytest.mark.parametrize("fin", ["fused", "separate"])
@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("scale,r", [(1, 1.0), (4, 0.7), (0, 1.0)])
def test_every_tile(gpu, monkeypatch, tile, fin, scale, r):
    """One tile (its halo is the tile itself), 4 x 4 of them and cut-off ones: converged drifts of
    two noise vectors against the oracle's FP64 drift, to what the tolerance leaves (1e-8, as for
    the other mixed solvers)."""
    monkeypatch.setenv("YCN_TILE_PL", str(tile))
    monkeypatch.setenv("YCN_PL_FIN", fin)
    monkeypatch.setenv("YCN_ONCHIP", "0")
    Y = gpu
    Nt, Nx = extents(tile, scale)
    p, orc = mk(Y, Nt=Nt, Nx=Nx, r=r, nNoise=2, cgTol=1e-10, cgTolMode=1, cgMaxIter=20000)
    p.cgPrecision = Y.YCN_CG_MIXED
    phi = 1.0 + O.hot_start(Nt + Nx, Nt, Nx)
    with Y.Context(p) as c:
        c.set_field(phi)
        d, st = c.fermion_force(3)
    dr, _ = O.fermion_drift(orc, phi, 3)
    assert st["converged"] == 1 and st["true_rel_resid"] <= 1e-10
    assert rel(d, dr) < 1e-8


@pytest.mark.parametrize("cap", [61, 62])
def test_odd_cap(gpu, monkeypatch, cap):
    Y = gpu
    res = {}
    phi = O.hot_start(11, 32, 64)
    monkeypatch.setenv("YCN_ONCHIP", "0")
    for n in (cap - 1, cap, cap + 1):
        p, _ = mk(Y, Nt=32, Nx=64, M=0.3, g=0.5, cgTol=1e-30, cgTolMode=1, cgMaxIter=n)
        p.cgPrecision = Y.YCN_CG_MIXED
        with Y.Context(p) as c:
            c.set_field(phi)
            d, st = c.fermion_force(5)
        assert st["converged"] == 0 and st["iters"] == n
        res[n] = d
    # the drifts converge: a dropped update would leave the odd cap where the one before it is
    step = np.linalg.norm(res[cap] - res[cap - 1])
    assert step > 0.2 * np.linalg.norm(res[cap + 1] - res[cap - 1]) > 0


def test_measured_correlator(gpu, monkeypatch):
    """D D^dag, the operator of the measurement's propagator, through the same iteration."""
    monkeypatch.setenv("YCN_ONCHIP", "0")
    Y = gpu
    p, orc = mk(Y, Nt=32, Nx=48, cgTol=1e-11, cgTolMode=1, cgMaxIter=20000)
    p.cgPrecision = Y.YCN_CG_MIXED
    phi = 1.0 + O.hot_start(5, 32, 48)
    with Y.Context(p) as c:
        c.set_field(phi)
        _, _, corr = c.measure(0, 3)
    assert rel(corr, O.correlator(orc, phi)[0]) < 1e-9


# the FP64 tiles that compute A p again instead of storing it
RC_TILES = [(16, 32), (32, 32), (16, 64)]


@pytest.mark.parametrize("fin", ["fused", "separate"])
@pytest.mark.parametrize("tile", range(len(TILES) + len(RC_TILES)))
@pytest.mark.parametrize("scale,r,cap", [(1, 0.7, 13), (0, 1.0, 12), (0, 0.7, 1), (2, 1.0, 26)])
def test_fp64_every_tile(gpu, monkeypatch, tile, fin, scale, r, cap):
    """Fixed iteration counts: the oracle's count, and its iterate to rounding."""
    monkeypatch.setenv("YCN_TILE_PL", str(tile))
    monkeypatch.setenv("YCN_PL_FIN", fin)
    monkeypatch.setenv("YCN_ONCHIP", "0")
    Y = gpu
    Nt, Nx = extents(tile, scale)
    p, orc = mk(Y, Nt=Nt, Nx=Nx, r=r, nNoise=2, cgTol=0.0, cgTolMode=0, cgMaxIter=cap)
    phi = 1.0 + O.hot_start(Nt + Nx, Nt, Nx)
    with Y.Context(p) as c:
        name = "%dx%d%s " % ((TILES + RC_TILES)[tile] + ("r" if tile >= len(TILES) else "",))
        assert name in c.tuning_report().split("fp64 pipelined tiles")[1]
        c.set_field(phi)
        d, st = c.fermion_force(3)
    dr, sr = O.fermion_drift(orc, phi, 3)
    assert 2 * st["iters"] == sr["iters"]   # the oracle adds up its solves
    assert rel(d, dr) < RTOL


@pytest.mark.parametrize("mode,tol", [(0, 1e-9), (1, 1e-10), (1, 3e-15)])
def test_fp64_stop(gpu, monkeypatch, mode, tol):
    """Both tolerance modes; 3e-15 is near where rounding holds the true residual above the
    recursive one, so that the solve restarts from it."""
    monkeypatch.setenv("YCN_ONCHIP", "0")
    Y = gpu
    Nt, Nx = 45, 50
    p, orc = mk(Y, Nt=Nt, Nx=Nx, cgTol=tol, cgTolMode=mode, cgMaxIter=20000)
    phi = 1.0 + O.hot_start(8, Nt, Nx)
    with Y.Context(p) as c:
        c.set_field(phi)
        d, st = c.fermion_force(3)
    dr, sr = O.fermion_drift(orc, phi, 3)
    print(f"# {tol}: {st} oracle {sr}", flush=True)
    if tol > 1e-12:
        assert st["converged"] == 1 and st["iters"] == sr["iters"]
    assert rel(d, dr) < 1e-8


EO_TILES = [(8, 32), (16, 32), (16, 16), (4, 32), (2, 32), (4, 16), (32, 32)]


@pytest.mark.parametrize("fin", ["fused", "separate"])
@pytest.mark.parametrize("tile", range(len(EO_TILES)))
@pytest.mark.parametrize("scale,r,cap", [(1, 0.7, 12), (2, 1.0, 13), (3, 0.7, 1), (2, 1.0, 26)])
def test_fp64_even_odd_every_tile(gpu, monkeypatch, tile, fin, scale, r, cap):
    """The even-odd FP64 iteration at fixed iteration counts: the oracle's iterate to rounding."""
    monkeypatch.setenv("YCN_TILE_PL", str(tile))
    monkeypatch.setenv("YCN_EO_FIN", fin)
    Y = gpu
    Nt, Nx = scale * EO_TILES[tile][0], scale * EO_TILES[tile][1]
    if Nx % 32 and Nt % 16:
        Nx *= 2   # even-odd lattices need 32 | Nx or 16 | Nt, Nx
    p, orc = mk(Y, Nt=Nt, Nx=Nx, r=r, nNoise=2, cgTol=0.0, cgTolMode=0, cgMaxIter=cap)
    p.evenOdd = 1
    orc.evenOdd = 1
    phi = 1.0 + O.hot_start(Nt + Nx, Nt, Nx)
    with Y.Context(p) as c:
        c.set_field(phi)
        d, st = c.fermion_force(3)
    dr, _ = O.fermion_drift(orc, phi, 3)
    assert st["iters"] == cap
    assert rel(d, dr) < RTOL


@pytest.mark.parametrize("mode,tol", [(0, 1e-9), (1, 1e-10), (1, 1e-13)])
def test_fp64_even_odd_stop(gpu, monkeypatch, mode, tol):
    """Both tolerance modes, one after the other solve: in the relative mode the second starts from
    the first's learned threshold and may have to go on from where it stopped."""
    monkeypatch.setenv("YCN_ONCHIP", "0")
    Y = gpu
    Nt, Nx = 48, 64
    p, orc = mk(Y, Nt=Nt, Nx=Nx, M=0.1, cgTol=tol, cgTolMode=mode, cgMaxIter=20000)
    p.evenOdd = 1
    with Y.Context(p) as c:
        for k in range(3):
            phi = 0.3 * k + O.hot_start(8 + k, Nt, Nx)
            c.set_field(phi)
            d, st = c.fermion_force(3)
            dr, sr = O.fermion_drift(orc, phi, 3)
            print(f"# {tol}: {st}", flush=True)
            assert st["converged"] == 1 and st["iters"] % 2 == 0
            assert mode == 0 or st["true_rel_resid"] <= tol
            assert rel(d, dr) < 1e-8


@pytest.mark.parametrize("fin", ["fused", "separate"])
@pytest.mark.parametrize("tile,Nt,Nx,r", [(12, 64, 64, 1.0), (12, 128, 192, 0.7), (13, 32, 128, 0.7), (13, 96, 256, 1.0)])
def test_large_even_odd_fp32_tiles(gpu, monkeypatch, tile, Nt, Nx, r, fin):
    """The 64x64 and 32x128 tiles: one tile, whose halo is itself, and several; converged drifts of
    two noise vectors as in test_every_tile."""
    monkeypatch.setenv("YCN_TILE_EO32", str(tile))
    monkeypatch.setenv("YCN_EO_FIN", fin)
    Y = gpu
    p, orc = mk(Y, Nt=Nt, Nx=Nx, r=r, nNoise=2, cgTol=1e-10, cgTolMode=1, cgMaxIter=20000)
    p.evenOdd = 1
    p.cgPrecision = Y.YCN_CG_MIXED
    phi = 1.0 + O.hot_start(Nt + Nx, Nt, Nx)
    with Y.Context(p) as c:
        c.set_field(phi)
        d, st = c.fermion_force(3)
    dr, _ = O.fermion_drift(orc, phi, 3)
    assert st["converged"] == 1 and st["true_rel_resid"] <= 1e-10
    assert rel(d, dr) < 1e-8


@pytest.mark.parametrize("Nt,Nx,r,vectors,scale", [(16, 16, 1.0, 1, 0.02), (32, 48, 0.7, 3, 0.0), (48, 16, 1.0, 2, 0.02),
                                                   (64, 64, 1.0, 2, 5.0)])
def test_flexible_iteration(gpu, Nt, Nx, r, vectors, scale):
    """The flexible solver's two launches per iteration: a zero network (plain CG), random ones and
    one so bad that it is switched off; chunks of 10 iterations; converged drifts of several noise
    vectors as in test_every_tile.  An odd iteration cap is kept."""
    Y = gpu
    kw = dict(Nt=Nt, Nx=Nx, r=r, nNoise=vectors, cgTol=1e-10, cgTolMode=1)
    phi = 1.0 + O.hot_start(Nt + Nx, Nt, Nx)
    w = (scale * np.random.default_rng(3).standard_normal(4896)).astype(np.float32)
    for cap in (20000, 13):
        p, orc = mk(Y, cgMaxIter=cap, **kw)
        p.cgPrecision = Y.YCN_CG_MIXED
        p.precond = Y.YCN_PRECOND_CNN
        p.reliableEvery = 10
        with Y.Context(p) as c:
            c.precond_set_weights(w)
            c.set_field(phi)
            d, st = c.fermion_force(3)
        print(f"# {Nt}x{Nx} {scale} {cap}: {st}", flush=True)
        if cap == 13:
            assert st["iters"] == 13 and st["converged"] == 0 and np.all(np.isfinite(d))
            continue
        dr, _ = O.fermion_drift(orc, phi, 3)
        assert st["converged"] == 1 and st["true_rel_resid"] <= 1e-10
        assert rel(d, dr) < 1e-8
