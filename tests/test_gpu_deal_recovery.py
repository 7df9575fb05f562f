"""The deal of window launches after a call that reported an error, and after a
captured launch was replayed, which files its units twice: every simulation is
still stepped exactly once.  Through the C-ABI, as a host
that captures its steps calls it; against the phase kernels."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

import carl_amd
from abi import CAR_NAMES, SIM_NAMES, enum_values
from carl_amd import build, workloads
from gpu_harness import describe_mismatch, dev, gpu_state

pytestmark = pytest.mark.gpu

CODES = enum_values("CARL_")
TICKS = 4
RELAXED = 2            # hipStreamCaptureModeRelaxed


@pytest.fixture(scope="module")
def libs():
    engine = C.CDLL(str(build.engine_path()))
    engine.carl_env_stream.restype = C.c_void_p
    engine.carl_last_error.restype = C.c_char_p
    return engine, C.CDLL("libamdhip64.so")


class Dealt:
    """An environment of the C-ABI whose launches are dealt, beside one of the
    same state on the phase kernels."""

    def __init__(self, libs, n, n_blue, n_orange):
        self.engine, self.hip = libs
        rng = np.random.default_rng(n)
        self.phased = carl_amd.Env(n, n_blue, n_orange, 5, TICKS, True, False, False)
        self.phased.tick_window = 0
        state = workloads.clustered_reset_state(rng, n, n_blue + n_orange)
        self.phased.apply_reset_state(**{k: dev(v) for k, v in state.items()})
        self.actions = dev(workloads.random_continuous_actions(rng, n, n_blue + n_orange)).reshape(-1)
        torch.cuda.synchronize()
        self.env = C.c_void_p()
        flags = CODES["CARL_FLAG_INVERT_ORANGE"]
        assert self.engine.carl_env_create(n, n_blue, n_orange, 5, TICKS, flags, C.byref(self.env)) == 0
        car, sim, tick = gpu_state(self.phased)
        car, sim = np.ascontiguousarray(car), np.ascontiguousarray(sim)
        assert self.engine.carl_env_import_state(self.env, C.c_void_p(car.ctypes.data), C.c_void_p(sim.ctypes.data), tick) == 0
        self.planes = car.shape, sim.shape
        dealt = C.c_int()
        assert self.engine.carl_env_get_param(self.env, CODES["CARL_PARAM_TICK_BALANCED_LAUNCH"], C.byref(dealt)) == 0
        assert dealt.value == 1
        self.stream = C.c_void_p(self.engine.carl_env_stream(self.env))

    def tick(self):
        return self.engine.carl_env_tick(self.env, CODES["CARL_ACTIONS_CONTINUOUS"], C.c_void_p(self.actions.data_ptr()),
                                         TICKS)

    def tick_phased(self, again=False):
        """The same ticks on the phase kernels; `again`: with the tick numbers
        of the call before."""
        if again:
            car, sim, tick = self.phased.export_state()
            self.phased.import_state(car, sim, tick - TICKS)
        self.phased.tick(self.actions, CODES["CARL_ACTIONS_CONTINUOUS"], TICKS)

    def assert_same(self, context):
        car, sim = (np.zeros(s, dtype=np.uint32) for s in self.planes)
        tick = C.c_int()
        assert self.engine.carl_env_export_state(self.env, C.c_void_p(car.ctypes.data), C.c_void_p(sim.ctypes.data),
                                                 C.byref(tick)) == 0
        want_car, want_sim, _ = gpu_state(self.phased)
        report = describe_mismatch(CAR_NAMES, car, want_car) + describe_mismatch(SIM_NAMES, sim, want_sim)
        assert not report, f"{context}:\n  " + "\n  ".join(report)

    def close(self):
        assert self.engine.carl_env_synchronize(self.env) == 0
        self.engine.carl_env_destroy(self.env)


SIZES = [(3000, 1, 1), (10_007, 2, 2), (4099, 3, 2)]


@pytest.mark.parametrize("n,n_blue,n_orange", SIZES)
def test_replayed_launches(gpu, libs, n, n_blue, n_orange):
    d = Dealt(libs, n, n_blue, n_orange)
    for step in range(3):
        assert d.tick() == 0
        d.tick_phased()
    d.assert_same("before the capture")
    graph, run = C.c_void_p(), C.c_void_p()
    assert d.hip.hipStreamBeginCapture(d.stream, RELAXED) == 0
    rc = d.tick()
    assert d.hip.hipStreamEndCapture(d.stream, C.byref(graph)) == 0 and rc == 0
    assert d.hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
    for replay in range(3):
        assert d.hip.hipGraphLaunch(run, d.stream) == 0
        d.tick_phased(again=replay > 0)
        d.assert_same(f"replay {replay}")
    for step in range(4):
        assert d.tick() == 0
        d.tick_phased()
        d.assert_same(f"step {step} after the replays")
    assert d.hip.hipGraphExecDestroy(run) == 0 and d.hip.hipGraphDestroy(graph) == 0
    d.close()


@pytest.mark.parametrize("n,n_blue,n_orange", SIZES)
def test_call_that_reports_an_error(gpu, libs, n, n_blue, n_orange):
    """A tick that reports an error (here one that an unrelated HIP call left
    behind, so its launch has run) has counted no ticks and the next one
    starts the deal over."""
    d = Dealt(libs, n, n_blue, n_orange)
    for step in range(3):
        assert d.tick() == 0
        d.tick_phased()
    d.assert_same("before the error")
    assert d.hip.hipSetDevice(1 << 20) != 0
    assert d.tick() == CODES["CARL_ERR_RUNTIME"]
    d.tick_phased()
    d.assert_same("with the error")
    for step in range(4):
        assert d.tick() == 0, d.engine.carl_last_error()
        d.tick_phased(again=step == 0)
        d.assert_same(f"step {step} after the error")
    d.close()
