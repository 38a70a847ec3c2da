"""Kernel timing (ycn_profile_begin / ycn_profile_end) and forced tiles on the plain solvers'
contexts whose iterations are pipelined: a named kernel is timed where the solver has one to time,
and a forced normal-operator tile is the one that runs."""
import pytest

import oracle as O
from test_gpu_parity import mk, rel

pytestmark = pytest.mark.gpu

NT, NX = 64, 96   # larger than a one-workgroup solve
TILES32 = [(8, 32), (4, 64), (16, 16), (8, 64), (16, 32), (4, 16)]


def context(Y, mixed, **kw):
    p, orc = mk(Y, Nt=NT, Nx=NX, cgTol=1e-10, cgTolMode=1, cgMaxIter=20000, **kw)
    p.cgPrecision = Y.YCN_CG_MIXED if mixed else Y.YCN_CG_FP64
    return Y.Context(p), orc


@pytest.mark.parametrize("mixed", [True, False])
def test_update_kernel_is_timed(gpu, mixed):
    """"cg_update": the solve under it runs the iteration that has an update kernel, reads x, r, p
    and Ap and writes x and r (packed spinors, two planes), and gives the same drift."""
    Y = gpu
    phi = 1.0 + O.hot_start(4, NT, NX)
    c, orc = context(Y, mixed)
    with c:
        c.set_field(phi)
        d0, _ = c.fermion_force(2)
        c.profile_begin("cg_update")
        d, st = c.fermion_force(2)
        ms, n, b = c.profile_end()
        d1, _ = c.fermion_force(2)
    print(f"# {n} launches for {st['iters']} iterations, {b} bytes", flush=True)
    assert n >= st["iters"] and ms > 0.0
    assert b == NT * NX * 6 * 2 * (8 if mixed else 16)
    dr, _ = O.fermion_drift(orc, phi, 2)
    assert st["converged"] == 1 and max(rel(x, dr) for x in (d0, d, d1)) < 1e-8


def test_measured_dirac_application_is_timed(gpu):
    """"dirac": the propagator of a measurement ends with one application, D^dag on a packed spinor."""
    Y = gpu
    c, _ = context(Y, False)
    with c:
        c.set_field(1.0 + O.hot_start(4, NT, NX))
        c.profile_begin("dirac")
        c.measure(0, 1)
        ms, n, b = c.profile_end()
    assert n == 1 and ms > 0.0
    assert b == NT * NX * (2 * 2 * 16 + 8)


@pytest.mark.parametrize("tile", [0, 2, 5])
def test_forced_fp32_tile_runs(gpu, monkeypatch, tile):
    """YCN_TILE32: the fused normal operator, which reads r, p and phi and writes p and Ap, runs in
    place of the pipelined iteration (5 to 7 vectors and phi per launch)."""
    monkeypatch.setenv("YCN_TILE32", str(tile))
    Y = gpu
    phi = 1.0 + O.hot_start(5, NT, NX)
    c, orc = context(Y, True)
    with c:
        c.set_field(phi)
        c.profile_begin("cg_normal_op")
        d, st = c.fermion_force(2)
        _, n, b = c.profile_end()
    assert n >= st["iters"]
    assert b == NT * NX * (4 * 2 * 8 + 4), TILES32[tile]
    dr, _ = O.fermion_drift(orc, phi, 2)
    assert st["converged"] == 1 and rel(d, dr) < 1e-8
