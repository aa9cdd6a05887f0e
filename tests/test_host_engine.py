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


_ROWS = 4096
_CALLS = {
    # what leaves scratch with the handle, then what needs room
    "direct": ("gradient", lambda sim: sim.direct_accel(np.arange(1024, dtype=np.int32))),
    "paths": ("gradient", lambda sim: sim.paths()),
    "features": ("diagnostics", lambda sim: sim.coarse_features()),
    "model": ("diagnostics", lambda sim: sim.set_model(_model())),
    "gradient": ("forward", lambda sim: sim.mlp_loss_grad(*_pairs(20 * _ROWS))),
}


def _model():
    from helpers import random_model

    return random_model(3)


def _pairs(rows):
    g = np.random.default_rng(rows)
    return g.normal(size=(rows, 24)).astype(np.float32), g.normal(size=(rows, 3)).astype(np.float32)


def _before(sim, kind):
    """What the call that leaves scratch also takes for good."""
    if kind == "diagnostics":
        sim.direct_accel(np.arange(16, dtype=np.int32))  # the check buffers
    else:
        sim.set_model(_model())


def _leave_scratch(sim, kind):
    if kind == "diagnostics":
        sim.diagnostics(pe_samples=16)
    elif kind == "gradient":
        sim.mlp_loss_grad(*_pairs(_ROWS))
    else:
        sim.mlp_forward(_pairs(_ROWS)[0])


@pytest.mark.parametrize("what", list(_CALLS))
def test_kept_scratch_makes_room(host, what):
    """What one call left with the handle goes back when another finds no room: a
    call fits wherever it would fit if nothing had been kept, and the launches
    after it do not see the failed attempt."""
    from nbody_amd import NbError, _lib

    kind, call = _CALLS[what]
    lo, hi = 0, 1 << 28  # by halves, the least room that the call needs with nothing kept
    while hi - lo > 64:
        room = (lo + hi) // 2
        fresh = _sim(_state(20_000))
        _before(fresh, kind)
        host.host_device_room(room)
        try:
            call(fresh)
            hi = room
        except NbError as e:
            assert e.code == _lib.NB_E_HIP
            lo = room
        host.host_device_room(-1)
        fresh.close()
    sim = _sim(_state(20_000))
    _before(sim, kind)
    fixed = host.host_device_used()
    _leave_scratch(sim, kind)
    left = host.host_device_used() - fixed
    assert left > 0
    host.host_device_room(hi - left)
    call(sim)
    host.host_device_room(-1)
    sim.steps(1)
    sim.close()
    assert host.host_device_used() == 0


@pytest.mark.parametrize("call", ["state", "accel", "masses", "positions64", "vertices", "set_state", "step", "root"])
def test_an_earlier_failure_is_not_this_calls(host, call):
    """A handle that could not be created leaves an error with the runtime; calls
    on another handle do not report it as theirs."""
    from nbody_amd import NbError, _lib

    st = _state(1000)
    sim = _sim(st, flags=_lib.NB_FP64_POSITIONS)
    host.host_device_room(1 << 20)
    with pytest.raises(NbError) as e:
        _sim(_state(100_000))
    assert e.value.code == _lib.NB_E_HIP
    host.host_device_room(-1)
    out = np.zeros((1000, 4), np.float32)
    {"state": sim.state, "accel": sim.accel, "masses": sim.masses, "positions64": sim.positions64,
     "vertices": lambda: sim.copy_vertices(out, None), "set_state": lambda: sim.set_state(*st),
     "step": sim.step, "root": sim.root}[call]()
    sim.close()


@pytest.mark.parametrize("n", [1, 8193, 20_000, 70_001, 600_001])
@pytest.mark.parametrize("pinned", [0, 1 << 13])
def test_a_handle_without_pinned_memory(host, n, pinned):
    """No pinned memory at all, or too little for the slots: the handle is created
    and its copies (pieces of 256 KiB, 512 KiB and 1 MiB) are the same."""
    from nbody_amd import _lib

    st = _state(n)
    host.host_pinned_room(pinned)
    sim = _sim(_state(n, 2), flags=_lib.NB_FP64_POSITIONS)
    sim.steps(1)
    sim.set_state(*st)
    assert sim.counters().step == -1
    for got, put in zip(sim.state(), st):
        assert np.array_equal(got, put)
    assert np.array_equal(sim.positions64(), np.stack(st[:3], 1).astype(np.float64))
    assert np.array_equal(sim.masses(), st[6]) and not sim.accel().any()
    pos, vel = np.full((n, 4), 7, np.float32), np.full((n, 4), 7, np.float32)
    sim.copy_vertices(pos, vel)
    one = np.ones(n, np.float32)
    assert np.array_equal(pos, np.stack([*st[:3], one], 1)) and np.array_equal(vel, np.stack([*st[3:6], one], 1))
    sim.steps(2)
    assert host.host_pinned_used() == 0
    sim.close()
    assert host.host_device_used() == 0
