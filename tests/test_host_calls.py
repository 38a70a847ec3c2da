"""What the library's host side asks of the HIP runtime, without a GPU: each test runs a child
process in which tests/host/hip_stub.cpp stands in for the runtime (device memory is host memory,
launches do nothing), drives the C-ABI through the Python binding and looks at the recorded calls."""
import ctypes as C
import json
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    d = tmp_path_factory.mktemp("hip_stub")
    lib = str(d / "libamdhip64.so.7")
    # libycn.so asks for the runtime's symbol versions
    versions = d / "versions"
    versions.write_text("hip_4.2 { global: hip*; __hip*; stub*; local: *; };\n"
                        "hip_4.3 { global: hipGraph*; hipStreamBeginCapture; hipStreamEndCapture; } hip_4.2;\n")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wl,-soname,libamdhip64.so.7",
                    f"-Wl,--version-script={versions}", "-o", lib,
                    os.path.join(ROOT, "tests", "host", "hip_stub.cpp")], check=True)
    return lib


def child(stub, what, **kw):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), stub, what, json.dumps(kw)], capture_output=True,
                       text=True, timeout=120, cwd=ROOT)
    assert r.returncode == 0, r.stdout[-4000:] + r.stderr[-4000:]
    return json.loads(r.stdout.splitlines()[-1])


def open_stub(path):
    lib = C.CDLL(path, mode=C.RTLD_GLOBAL)
    lib.stub_record.restype = C.c_char_p
    return lib


# ---- every entry point works on its context's device, whichever is current ---------------------
CONTEXTS = [dict(Nt=16, Nx=16), dict(Nt=64, Nx=64, evenOdd=1, cgPrecision=1), dict(Nt=64, Nx=96, cgPrecision=1),
            dict(Nt=64, Nx=96), dict(Nt=96, Nx=96, evenOdd=1, cgPrecision=1, cgTolMode=1), dict(Nt=32, Nx=32, precond=1)]


def entry_points(hip, params):
    """[entry point, calls made while another device than the context's was current, whether the
    caller's device was current again afterwards]"""
    import yukawacolourednoise_amd as Y
    p = Y.default_params(device=1, **params)
    V, out = p.Nt * p.Nx, []
    b = np.ones((V, 4), dtype=complex)

    def used(c, name, call):
        hip.hipSetDevice(0)
        hip.stub_clear()
        try:
            call()
        except Y.YcnError as e:   # nothing ran: no solve converges and no step reports
            if e.code not in (Y.abi.YCN_ERR_NOT_CONVERGED, Y.abi.YCN_ERR_HIP):
                raise
        lines = hip.stub_record().decode().splitlines()
        dev = C.c_int()
        hip.hipGetDevice(C.byref(dev))
        out.append([name, [x for x in lines if x.split()[1] != "1"], dev.value == 0])

    for k, calls in enumerate((
            [("langevin_step", lambda c: c.langevin_step(0)), ("langevin_run", lambda c: c.langevin_run(1, 3))],
            [("langevin_run", lambda c: c.langevin_run(1, 3)), ("langevin_step", lambda c: c.langevin_step(0))],
            [("set_replicas", lambda c: c.set_replicas(np.array([0.1]), np.array([3], dtype=np.uint64))),
             ("hot_start", lambda c: c.hot_start(3)), ("coloured_noise", lambda c: c.coloured_noise(2)),
             ("coloured_filter", lambda c: c.coloured_filter(np.ones((p.Nt, p.Nx)))),
             ("dirac_apply", lambda c: c.dirac_apply(b, phi=np.ones((p.Nt, p.Nx)))),
             ("cg_solve", lambda c: c.cg_solve(b)), ("fermion_force", lambda c: c.fermion_force(1)),
             ("measure", lambda c: c.measure(0, 1)), ("profile", lambda c: c.profile_begin("cg_normal_op")),
             ("profiled step", lambda c: c.langevin_step(4)), ("profile_end", lambda c: c.profile_end())]
            + ([("precond_apply", lambda c: c.precond_apply(b)),
                ("precond_train", lambda c: c.precond_train(0, 1, pairs_per_solve=1))] if params.get("precond") else []))):
        with Y.Context(p) as c:
            for name, call in calls:
                used(c, f"{k} {name}", lambda: call(c))
    return out


@pytest.mark.parametrize("params", CONTEXTS)
def test_entry_points_use_the_contexts_device(stub, params):
    for name, wrong, restored in child(stub, "entry_points", **params):
        assert not wrong, (name, wrong[:5])
        assert restored, name


# ---- the one-workgroup even-odd solve: no two of its buffers are the same memory ---------------
def onchip_buffers(hip, params):
    """the buffers of every such launch of a force and of a measurement's propagator"""
    import yukawacolourednoise_amd as Y
    hip.stub_watch(b"k_onchip_eo", 13)
    # k_onchip_eo's arguments after its structure
    names = ["phi", "seeds", "streamBase", "step", "eta", "b", "drift", "out", "st", "ratioIn", "ratioOut", "nsys"]
    with Y.Context(Y.default_params(evenOdd=1, **params)) as c:
        hip.stub_clear()
        for call in (lambda: c.fermion_force(0), lambda: c.measure(0, 1)):
            try:
                call()
            except Y.YcnError as e:   # nothing ran: no solve converges
                assert e.code == Y.abi.YCN_ERR_NOT_CONVERGED
        launches = [x.split()[3:] for x in hip.stub_record().decode().splitlines() if "k_onchip_eo" in x]
    return [dict(zip(names, map(int, x))) for x in launches]


@pytest.mark.parametrize("params", [dict(Nt=16, Nx=16), dict(Nt=64, Nx=64, nReplicas=2, nNoise=3)])
def test_onchip_even_odd_buffers_are_distinct(stub, params):
    launches = child(stub, "onchip_buffers", **params)
    assert sum(x["out"] != 0 for x in launches) == 1   # the propagator's
    assert len(launches) > 1
    for x in launches:
        buffers = [x[k] for k in ("phi", "eta", "b", "drift", "out", "st") if x[k]]
        assert len(set(buffers)) == len(buffers), x


if __name__ == "__main__":
    sys.path.insert(0, ROOT)
    print(json.dumps(globals()[sys.argv[2]](open_stub(sys.argv[1]), json.loads(sys.argv[3]))))
