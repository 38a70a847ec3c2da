"""Fermion-force solves held by one workgroup, where their sizes turn: one site per thread
and two, a full and a partly filled last wave, several noise vectors, each stopping rule.
Against the oracle at a fixed iteration count (1e-12) and against the launched iterations
(YCN_ONCHIP=0) where the stopping and restart rules decide."""
import numpy as np
import pytest

import oracle as O
from test_gpu_parity import RTOL, mk, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nt,Nx,r,vectors", [(32, 32, 1.0, 1), (25, 41, 0.7, 1), (32, 64, 1.0, 2), (33, 62, 0.0, 1),
                                             (2, 33, 1.0, 3)])
def test_onchip_force(gpu, Nt, Nx, r, vectors):
    Y = gpu
    p, orc = mk(Y, Nt=Nt, Nx=Nx, r=r, nNoise=vectors, driftMode=1, cgTol=0.0, cgTolMode=0, cgMaxIter=20)
    phi = 1.0 + O.hot_start(Nt + Nx, Nt, Nx)
    with Y.Context(p) as c:
        c.set_field(phi)
        d, st = c.fermion_force(3)
    dr, sr = O.fermion_drift(orc, phi, 3)
    assert vectors * st["iters"] == sr["iters"]
    assert rel(d, dr) < RTOL


@pytest.mark.parametrize("mode,tol,cap", [(0, 1e-8, 1000), (1, 1e-10, 1000), (1, 1e-17, 300), (1, 1e-10, 0)])
def test_onchip_stopping(gpu, monkeypatch, mode, tol, cap):
    """Both stopping rules, a tolerance below rounding (restarts, then not converged) and a
    zero cap: the same verdict as the launched iterations, and the same drift to what the
    tolerance leaves open."""
    Y = gpu
    p, _ = mk(Y, Nt=22, Nx=32, cgTol=tol, cgTolMode=mode, cgMaxIter=cap)
    phi = 1.0 + O.hot_start(9, 22, 32)
    out = {}
    for on in ("1", "0"):
        monkeypatch.setenv("YCN_ONCHIP", on)
        with Y.Context(p) as c:
            c.set_field(phi)
            out[on] = c.fermion_force(1)
    (d1, s1), (d0, s0) = out["1"], out["0"]
    assert s1["converged"] == s0["converged"] == (0 if tol < 1e-16 or cap == 0 else 1)
    assert (s1["restarts"] > 0) == (s0["restarts"] > 0)
    assert abs(s1["iters"] - s0["iters"]) <= (1 if tol > 1e-16 else cap)
    if cap:
        assert rel(d1, d0) < 1e-9
    else:
        assert not np.any(d1) and not np.any(d0)


@pytest.mark.parametrize("Nt,Nx,r,vectors", [(2, 32, 1.0, 1), (32, 64, 1.0, 2), (34, 64, 0.7, 1), (64, 64, 1.0, 1),
                                             (16, 256, 1.0, 3), (6, 32, 0.5, 1)])
def test_onchip_even_odd_force(gpu, Nt, Nx, r, vectors):
    """Even-odd solves by one workgroup: one entry per thread up to 1024 of them and two
    beyond, idle threads in the last wave, an odd number of row pairs."""
    Y = gpu
    p, orc = mk(Y, Nt=Nt, Nx=Nx, r=r, nNoise=vectors, driftMode=1, cgTol=0.0, cgTolMode=0, cgMaxIter=15)
    p.evenOdd = orc.evenOdd = 1
    phi = 1.0 + O.hot_start(Nt + Nx, Nt, Nx)
    with Y.Context(p) as c:
        c.set_field(phi)
        d, st = c.fermion_force(3)
    dr, sr = O.fermion_drift(orc, phi, 3)
    assert vectors * st["iters"] == sr["iters"]
    assert rel(d, dr) < RTOL


@pytest.mark.parametrize("mode,tol,cap", [(0, 1e-8, 1000), (1, 1e-10, 1000), (1, 1e-17, 100), (1, 1e-10, 0)])
def test_onchip_even_odd_stopping(gpu, monkeypatch, mode, tol, cap):
    Y = gpu
    p, _ = mk(Y, Nt=34, Nx=64, cgTol=tol, cgTolMode=mode, cgMaxIter=cap)
    p.evenOdd = 1
    phi = 1.0 + O.hot_start(9, 34, 64)
    out = {}
    for on in ("1", "0"):
        monkeypatch.setenv("YCN_ONCHIP", on)
        with Y.Context(p) as c:
            c.set_field(phi)
            c.fermion_force(0)                   # the second solve starts from a learned threshold
            out[on] = c.fermion_force(1) + (c.measure(0, 5)[2],)
    (d1, s1, c1), (d0, s0, c0) = out["1"], out["0"]
    assert s1["converged"] == s0["converged"] == (0 if tol < 1e-16 or cap == 0 else 1)
    assert (s1["restarts"] > 0) == (s0["restarts"] > 0)
    if cap == 0:
        assert rel(d1, d0) < RTOL and rel(c1, c0) < RTOL
    else:
        # the launched solver pauses after even numbers of iterations only
        assert abs(s1["iters"] - s0["iters"]) <= (2 if tol > 1e-16 else cap)
        assert rel(d1, d0) < 1e-7 and rel(c1, c0) < 1e-7


@pytest.mark.parametrize("Nt,Nx,chains,eo,steps", [(8, 16, 1, 0, 70), (7, 32, 3, 0, 17), (32, 32, 2, 1, 33)])
def test_run_equals_steps(gpu, Nt, Nx, chains, eo, steps):
    """A run makes the noise of several steps in one launch (16 at most) and waits for up to 64:
    the same fields as step by step, bit for bit (plain solver) or to the solver's tolerance
    (even-odd: the starting thresholds are learned on the device or on the host)."""
    Y = gpu
    p, _ = mk(Y, Nt=Nt, Nx=Nx, nReplicas=chains, cgTol=1e-10, cgTolMode=1)
    p.evenOdd = eo
    out = []
    for run in (True, False):
        with Y.Context(p) as c:
            c.hot_start(4)
            if run:
                c.langevin_run(5, steps)
            else:
                for k in range(steps):
                    c.langevin_step(5 + k)
            out.append(c.get_field())
    assert np.array_equal(*out) if not eo else rel(*out) < 1e-7
