"""The engine's host side when the runtime refuses something: nb_engine.cpp with
a stand-in for the HIP runtime and the kernels (tests/host_runtime.cpp), whose
memory has limits and whose launches fail on request."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "gpu-nbody_amd", "csrc")


@pytest.fixture(scope="module")
def host_lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host") / "libnbody_host.so")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-shared", "-fPIC", "-pthread", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-D__align__(x)=__attribute__((aligned(x)))", "-DHIP_SYMBOL(x)=&x", f"-I{rocm}/include",
                    f"-I{CSRC}", f"-I{ROOT}/include", os.path.join(CSRC, "nb_engine.cpp"),
                    os.path.join(ROOT, "tests", "host_runtime.cpp"), "-Wl,-Bsymbolic", "-o", out], check=True)
    return out


@pytest.fixture
def host(host_lib, monkeypatch):
    """The package on the stand-in; the library comes along for its switches."""
    from nbody_amd import _lib

    monkeypatch.setattr(_lib, "LIB_PATH", host_lib)
    monkeypatch.setattr(_lib, "_lib", None)
    lib = _lib.load()
    lib.host_device_room.argtypes = lib.host_pinned_room.argtypes = [C.c_longlong]
    lib.host_device_used.restype = lib.host_pinned_used.restype = C.c_longlong
    yield lib
    for room in (lib.host_device_room, lib.host_pinned_room):
        room(-1)
    lib.host_fail_state_launch(0)


def _state(n, seed=1):
    g = np.random.default_rng(seed)
    return tuple(g.normal(size=n).astype(np.float32) for _ in range(7))


def _sim(st, **kw):
    from helpers import make_sim

    return make_sim(st, theta=0.5, softening=0.05, dt=1e-3, vote_width=64, **kw)


@pytest.mark.parametrize("nth", [1, 2, 3])
def test_failed_state_is_no_state(host, nth):
    """A set_state whose nth piece (of three) fails: sorted[] is neither the old
    order nor the identity, so nothing may start from it."""
    from nbody_amd import NbError, _lib

    st = _state(20_000)
    sim = _sim(st)
    sim.steps(2)
    host.host_fail_state_launch(nth)
    with pytest.raises(NbError) as e:
        sim.set_state(*_state(20_000, 2))
    assert e.value.code == _lib.NB_E_HIP
    for call in (sim.step, sim.probe_accel, lambda: sim.run_stage(1)):
        with pytest.raises(NbError) as e:
            call()
        assert e.value.code == _lib.NB_E_STATE
    sim.set_state(*st)
    sim.steps(1)
    for got, put in zip(sim.state(), st):
        assert np.array_equal(got, put)
    sim.close()
    assert host.host_device_used() == 0 and host.host_pinned_used() == 0
