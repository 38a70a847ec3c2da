"""The launched solvers on lattices that one workgroup would hold (YCN_ONCHIP=0): the checks of the
force, the step, the sweep's lattices, the measurement and the trajectories, whose lattices are
small, run on the launched iterations too; and which of these iterations runs is asserted."""
import numpy as np
import pytest

import oracle as O
import test_gpu_evenodd as eo
import test_gpu_packed as packed
import test_gpu_parity as parity
import test_gpu_statistics as stat
import test_gpu_trajectories as traj
from test_gpu_parity import mk, rel

pytestmark = pytest.mark.gpu


@pytest.fixture
def launched(monkeypatch):
    monkeypatch.setenv("YCN_ONCHIP", "0")


def again(test, *args):
    """(test, arguments) with a readable id"""
    return pytest.param(test, args, id="-".join([test.__name__] + [str(a) for a in args]))


UNTILED = [(3, 32), (7, 32), (6, 32), (22, 32), (10, 12), (13, 18)]


@pytest.mark.parametrize("test,args", [again(parity.test_langevin_step, a, *s) for a in (0, 1)
                                       for s in ((16, 16), (32, 32), (6, 32))]
                         + [again(parity.test_sweep_configuration, n) for n in (2, 10, 22)]
                         + [again(parity.test_mixed_precision_on_untiled_lattices, *s) for s in UNTILED]
                         + [again(parity.test_langevin_step_converged, a) for a in (0, 1)]
                         + [again(parity.test_measure, m) for m in ("plain", "eo-fp64", "eo-mixed")]
                         + [again(parity.test_measure_batched_replica, e) for e in (0, 1)]
                         + [again(t) for t in (parity.test_batched_replicas, parity.test_multi_rhs_noise,
                                               parity.test_mixed_langevin_step, packed.test_complex_solve_after_packed_force)]
                         + [again(packed.test_packed_force, *a) for a in ((2, 2, 1.0, 1), (3, 5, 1.0, 2), (7, 32, 0.0, 1),
                                                                          (8, 64, 0.7, 3), (16, 16, 1.0, 1))])
def test_plain(gpu, launched, test, args):
    test(gpu, *args)


@pytest.mark.parametrize("test,args", [again(eo.test_eo_force_converged, p, n, n) for p in ("fp64", "mixed") for n in (32, 64)]
                         + [again(eo.test_eo_second_solve_starts_from_learned_threshold, p) for p in ("fp64", "mixed")]
                         + [again(eo.test_eo_mixed_wilson_parameter, r) for r in (0.7, 1.0)]
                         + [again(eo.test_eo_mixed_small_time_extents, n) for n in (2, 6, 10)]
                         + [again(eo.test_eo_small_time_extents, n) for n in (2, 10, 22)]
                         + [again(eo.test_eo_force_fixed_iterations, *s) for s in ((16, 16), (32, 32), (6, 32), (8, 64))]
                         + [again(eo.test_eo_langevin_steps_fixed_iterations, a) for a in (0, 1)]
                         + [again(t) for t in (eo.test_eo_batched_replicas_and_noise,
                                               eo.test_eo_mixed_iteration_cap_with_prediction)])
def test_even_odd(gpu, launched, test, args):
    test(gpu, *args)


@pytest.mark.parametrize("method,adaptive", [("mixed", 0), ("eo-mixed", 0), ("eo-mixed", 1)])
def test_32_trajectory(gpu, launched, method, adaptive):
    """2000 steps of the FP32 solvers against the oracle's"""
    traj._trajectory_32(gpu, method, adaptive)


def test_statistics_chains(gpu, monkeypatch):
    """The 32 replicas of the statistical comparison with the oracle, whose even-odd solves one
    workgroup holds: with launched mixed-precision solves the same chains (to 1e-9, what the solver's
    tolerance leaves, as for the trajectories), so the comparison holds for them too."""
    Y = gpu
    out = {}
    for on in ("1", "0"):
        monkeypatch.setenv("YCN_ONCHIP", on)
        p = Y.default_params(Nt=stat.NT, Nx=stat.NX, nReplicas=stat.R, **stat.PHYS)
        p.cgPrecision, p.evenOdd = Y.YCN_CG_MIXED, 1
        with Y.Context(p) as c:
            c.set_replicas(np.full(stat.R, stat.PHYS["m2"]), np.arange(200, 200 + stat.R, dtype=np.uint64))
            c.hot_start(200)
            st = c.langevin_run(0, 1000)
            assert st["converged"] == 1 and st["true_rel_resid"] <= 1e-10, st
            out[on] = c.get_field()
    assert rel(out["0"], out["1"]) < 1e-9


@pytest.mark.parametrize("mixed,evenOdd", [(0, 0), (1, 0), (0, 1)])
@pytest.mark.parametrize("on", [1, 0])
def test_switch_is_what_decides(gpu, monkeypatch, mixed, evenOdd, on):
    """One workgroup per system: a run waits once for all its steps.  Launched: at least once a step."""
    monkeypatch.setenv("YCN_ONCHIP", str(on))
    Y = gpu
    p, _ = mk(Y, Nt=16, Nx=32, cgTol=1e-10, cgTolMode=1)
    p.cgPrecision, p.evenOdd = mixed, evenOdd
    with Y.Context(p) as c:
        c.hot_start(2)
        before = c.host_syncs()[0]
        c.langevin_run(0, 8)
        waits = c.host_syncs()[0] - before
    assert waits == 1 if on else waits >= 8


# bytes per site and launch of the FP32 operator (packed spinors): the two-stencil pair passes seven
# vectors and the field twice; a pipelined launch five or seven and the field
PAIR, PIPELINED = 7 * 16 + 8, (5 * 16 + 4, 7 * 16 + 4)


@pytest.mark.parametrize("Nt,Nx,pair", [(3, 32, True), (10, 12, True), (7, 32, False), (6, 32, False), (22, 32, False),
                                        (13, 18, False), (3, 1024, True), (2, 1500, True), (5, 1024, False)])
def test_mixed_operator_without_a_tile(gpu, monkeypatch, Nt, Nx, pair):
    """Which FP32 operator a lattice that no fused tile divides runs: the pipelined iteration where a
    tile can be cut off, else the two-stencil pair, also by default on lattices of more than 2048
    sites.  The force, with several noise vectors, and a solve with a complex right-hand side (the
    same pair on four planes) against the oracle's, as for the other mixed solvers."""
    if Nt * Nx <= 2048:
        monkeypatch.setenv("YCN_ONCHIP", "0")
    Y = gpu
    p, orc = mk(Y, Nt=Nt, Nx=Nx, nNoise=2, cgTol=1e-10, cgTolMode=1, cgMaxIter=20000)
    p.cgPrecision = Y.YCN_CG_MIXED
    phi = 1.0 + O.hot_start(Nt + Nx, Nt, Nx)
    rng = np.random.default_rng(Nt + Nx)
    rhs = rng.standard_normal((Nt * Nx, 4)) + 1j * rng.standard_normal((Nt * Nx, 4))
    dr, _ = O.fermion_drift(orc, phi, 3)
    with Y.Context(p) as c:
        assert ("pipelined iteration" in c.tuning_report()) == (not pair)
        c.set_field(phi)
        d, st = c.fermion_force(3)
        assert st["converged"] == 1 and st["true_rel_resid"] <= 1e-10 and rel(d, dr) < 1e-8
        c.profile_begin("cg_normal_op")
        d, st = c.fermion_force(3)
        _, n, b = c.profile_end()
        x, sx = c.cg_solve(rhs)
    assert st["converged"] == 1 and rel(d, dr) < 1e-8
    per_site = b / (2 * Nt * Nx)
    assert per_site == PAIR if pair else PIPELINED[0] <= per_site <= PIPELINED[1], per_site
    assert sx["converged"] == 1 and sx["true_rel_resid"] <= 1e-10
    assert rel(x, O.cg(orc, phi, rhs, Y.YCN_DAGGER)[0]) < 1e-7


@pytest.mark.parametrize("Nt,Nx,evenOdd", [(32, 64, 0), (32, 64, 1), (45, 50, 0)])
def test_cap_with_prediction(gpu, launched, Nt, Nx, evenOdd):
    """A mixed solve that cannot reach its tolerance stops at the iteration cap and says so, also when
    the solve before it lets the host enqueue chunks without polling between them: 120 iterations in
    chunks of 50 are polled three times or more at first, once the count is known not after the first."""
    Y = gpu
    cap = 120
    p, _ = mk(Y, Nt=Nt, Nx=Nx, M=0.05, g=0.5, cgTol=1e-30, cgTolMode=1, cgMaxIter=cap)
    p.cgPrecision, p.evenOdd = Y.YCN_CG_MIXED, evenOdd
    waits = []
    with Y.Context(p) as c:
        c.set_field(0.3 + O.hot_start(11, Nt, Nx))
        for k in range(3):
            before = c.host_syncs()[0]
            d, st = c.fermion_force(5 + k)
            waits.append(c.host_syncs()[0] - before)
            print(f"# solve {k}: {st}, {waits[-1]} waits", flush=True)
            assert st["converged"] == 0 and st["iters"] == cap, st
            assert np.all(np.isfinite(d)) and np.isfinite(st["true_rel_resid"])
    assert waits[1] < waits[0] and waits[2] < waits[0], waits
