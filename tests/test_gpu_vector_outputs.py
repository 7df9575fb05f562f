"""The vector environment's step written by one kernel equals the same step
through separate torch operations (which a reward function selects) over
steps in which episodes end, by goals for either team and by timeouts: odd
sizes, both action kinds, deferred and immediate reports, side streams,
returns and lengths carried in, and the sizes at which the report is read in two parts."""
from __future__ import annotations

import ctypes as C
from contextlib import contextmanager

import numpy as np
import pytest
import torch

from carl_amd import build
from carl_amd.gymnasium import torch as vec

pytestmark = pytest.mark.gpu


def make(n_sim, blue, orange, discrete, deferred, max_ticks):
    return vec.CARLTorchVectorEnv(n_sim, blue, orange, seed=5, frameskip=4, max_ticks=max_ticks,
                                  overtime_timeout_ticks=8, no_touch_timeout_ticks=24, discrete_actions=discrete,
                                  defer_episode_reporting=deferred)


def team_reward(env):
    """The engine's own reward as a reward function."""
    return lambda context: context.events.score_delta[:, None] * env._team_sign


def actions(gen, env, discrete):
    u = torch.rand((env.n_envs, 7), generator=gen, device="cuda")
    return (u * torch.tensor([3, 3, 3, 2, 2, 3, 2], device="cuda")).int() if discrete else u * 2 - 1


def place_balls(envs, gen, shift=0):
    """Balls beyond either goal line and in the field, the same in every
    environment: a third of the matches ends with a goal for each team."""
    n = envs[0].n_sim
    third = (torch.randperm(n, generator=gen, device="cuda") + shift) % 3
    position = torch.zeros((n, 3), dtype=torch.float32, device="cuda")
    position[:, 1] = (third == 1) * 5300.0 - (third == 2) * 5300.0
    position[:, 2] = 100.0
    still = torch.zeros_like(position)
    for env in envs:
        env.set_ball(position, still, still)


@contextmanager
def default_dtype(dtype):
    before = torch.get_default_dtype()
    torch.set_default_dtype(dtype)
    try:
        yield
    finally:
        torch.set_default_dtype(before)


@pytest.mark.parametrize("deferred", [False, True])
@pytest.mark.parametrize("made,stepped", [
    (torch.float64, torch.float64), (torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
    (torch.float32, torch.float64), (torch.float32, torch.bfloat16), (torch.float64, torch.bfloat16),
    (torch.bfloat16, torch.float64),
])
def test_steps_do_not_depend_on_the_default_dtype(made, stepped, deferred):
    """A program's default dtype, set before the environment is made or
    between its steps, changes no value.  The observations stay the engine's
    float32; rewards are float32, or float64 where the environment was made
    under that."""
    want = make(33, 2, 1, False, deferred, 16)
    with default_dtype(made):
        ours = make(33, 2, 1, False, deferred, 16)
        first = ours.reset()
    torch.testing.assert_close(first, want.reset(), rtol=0, atol=0)
    gen = torch.Generator(device="cuda").manual_seed(3)
    signs = set()
    for step in range(12):
        if step % 5 == 2:
            place_balls((ours, want), gen)
        a = actions(gen, want, False)
        ref = want.step(a)
        with default_dtype(stepped):
            got = ours.step(a)
        assert got[0].dtype == torch.float32 and got[1].dtype == torch.promote_types(torch.float32, made)
        for g, w in zip(got[:4], ref[:4]):
            torch.testing.assert_close(g.to(w.dtype), w, rtol=0, atol=0)
        assert got[4].keys() == ref[4].keys()
        if not deferred:
            assert got[4]["reward"] == ref[4]["reward"] and got[4]["length"] == ref[4]["length"]
        signs |= set(ref[1].tolist())
    assert signs == {-1.0, 0.0, 1.0}
    assert ours.drain_episode_reports() == want.drain_episode_reports()
    torch.testing.assert_close(ours._ledger.returns.float(), want._ledger.returns, rtol=0, atol=0)


# 1 agent; a row length and agent count of every remainder; more ended agents
# at once than one read of the report holds; several rows per thread
@pytest.mark.parametrize("n_sim,blue,orange,discrete,deferred,side", [
    (1, 1, 0, False, False, False),
    (17, 1, 1, True, False, True),
    (33, 2, 1, False, True, False),
    (127, 1, 1, False, False, False),
    (128, 1, 1, True, True, True),
    (301, 4, 4, False, False, False),
    (70_001, 1, 1, False, False, False),
])
def test_one_kernel_equals_separate_operations(n_sim, blue, orange, discrete, deferred, side):
    ours = make(n_sim, blue, orange, discrete, deferred, 16)
    want = make(n_sim, blue, orange, discrete, deferred, 16)
    want.register_reward(team_reward(want))
    gen = torch.Generator(device="cuda").manual_seed(n_sim)
    stream = torch.cuda.Stream() if side else torch.cuda.current_stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        torch.testing.assert_close(ours.reset(), want.reset(), rtol=0, atol=0)
        # totals from before, as after many steps: both words of a length
        agent = torch.arange(ours.n_envs, device="cuda")
        for env in (ours, want):
            env._ledger.returns.copy_(agent % 7 - 2.75)
            env._ledger.lengths.copy_((agent % 3) * (1 << 33) + agent % 11)
        ended = 0
        signs, flags = set(), set()
        for step in range(14):
            if step in (1, 6, 11):
                place_balls((ours, want), gen, shift=step // 5)
            a = actions(gen, ours, discrete)
            got, ref = ours.step(a), want.step(a)
            for g, w in zip(got[:4], ref[:4]):
                assert type(g) is type(w) and g.dtype == w.dtype and g.shape == w.shape
                torch.testing.assert_close(g, w, rtol=0, atol=0)
            assert got[4].keys() == ref[4].keys()
            for k, w in ref[4].items():
                if k == "final_obs" :   # rows of episodes that ended
                    rows = ref[4]["_final_obs"]
                    torch.testing.assert_close(got[4][k][rows], w[rows], rtol=0, atol=0)
                elif isinstance(w, torch.Tensor):
                    torch.testing.assert_close(got[4][k], w, rtol=0, atol=0)
                else:
                    assert got[4][k] == w
            for name in ("_score_difference", "_episode_ticks", "_overtime"):
                torch.testing.assert_close(getattr(ours, name), getattr(want, name), rtol=0, atol=0)
            ended += int((got[2] | got[3]).sum())
            signs |= set(got[1].tolist())
            flags |= set(zip(got[2].tolist(), got[3].tolist()))
        assert ended >= ours.n_envs
        assert signs == {-1.0, 0.0, 1.0} and flags == {(False, False), (True, False), (False, True)}
        if deferred:
            assert ours.drain_episode_reports() == want.drain_episode_reports()
        torch.testing.assert_close(ours._ledger.returns, want._ledger.returns, rtol=0, atol=0)
        torch.testing.assert_close(ours._ledger.lengths, want._ledger.lengths, rtol=0, atol=0)
    torch.cuda.synchronize()


@pytest.mark.parametrize("count", [0, 1, 255, 256, 400])
def test_report_order_and_parts(count):
    """The native list holds agents in no order; lengths use both words."""
    rng = np.random.default_rng(count)
    agents = rng.permutation(500)[:count]
    returns = rng.integers(-9, 9, count).astype(np.float32)
    lengths = rng.integers(0, 1 << 40, count)
    rows = np.zeros((501, 4), dtype=np.int32)
    rows[0, 0] = count
    rows[1:count + 1, 0] = agents
    rows[1:count + 1, 1] = returns.view(np.int32)
    rows[1:count + 1].view(np.int64)[:, 1] = lengths
    ledger = vec._EpisodeLedger(500, torch.device("cuda"), False)
    report = ledger.report(torch.from_numpy(rows.reshape(-1)).cuda())
    order = np.argsort(agents)
    want = {"reward": returns[order].tolist(), "length": lengths[order].tolist()} if count else None
    assert report == want


def test_null_outputs_are_refused():
    env = make(3, 1, 1, False, False, 16)
    with pytest.raises(ValueError, match="null vector output"):
        env._env._vector_outputs(*[0] * 14)
    t = env._ledger.returns.data_ptr()
    with pytest.raises(ValueError, match="given together"):
        env._env._vector_outputs(*[t] * 10, t, 0, 0, 0)


class VectorIo(C.Structure):
    """carl_vector_io"""
    _fields_ = [(name, C.c_void_p) for name in (
        "obs", "reward", "terminated", "truncated", "done", "returns", "lengths", "score_difference",
        "episode_ticks", "overtime", "step_returns", "step_lengths", "step_done", "ended")]


# addresses of every alignment a float may have; numbers of words that leave a
# remainder of the copy's four, and more of them than one pass of the threads takes
@pytest.mark.parametrize("n_sim,blue,orange", [(1, 1, 0), (7, 1, 0), (3, 2, 1), (20_001, 2, 2)])
@pytest.mark.parametrize("offset", [0, 1, 2, 3])
def test_observations_are_copied_to_any_address(n_sim, blue, orange, offset):
    """A C caller's observation array may lie at any float's address; the
    words around it stay as they were."""
    engine = C.CDLL(str(build.engine_path()))
    engine.carl_last_error.restype = C.c_char_p
    agents = n_sim * (blue + orange)
    env = C.c_void_p()
    assert engine.carl_env_create(n_sim, blue, orange, 3, 1, 1, C.byref(env)) == 0, engine.carl_last_error()
    dim = engine.carl_observation_dim(blue + orange, 0)
    words = agents * dim
    buffer = torch.full((words + 8,), 7.25, dtype=torch.float32, device="cuda")
    assert buffer.data_ptr() % 16 == 0
    sizes = {"lengths": torch.int64, "returns": torch.float32, "reward": torch.float32, "score_difference": torch.int32,
             "episode_ticks": torch.int32}
    rest = {name: torch.zeros(agents, dtype=sizes.get(name, torch.bool), device="cuda") for name, _ in VectorIo._fields_[1:10]}
    torch.cuda.synchronize()
    io = VectorIo(buffer.data_ptr() + 4 * offset, *(x.data_ptr() for x in rest.values()), None, None, None, None)
    assert engine.carl_env_vector_outputs(env, C.byref(io)) == 0, engine.carl_last_error()
    assert engine.carl_env_synchronize(env) == 0
    data, shape, ndim, dtype = C.c_void_p(), (C.c_int64 * 3)(), C.c_int(), C.c_int()
    assert engine.carl_env_buffer(env, 0, C.byref(data), shape, C.byref(ndim), C.byref(dtype)) == 0
    assert list(shape)[:2] == [n_sim, blue + orange] and shape[2] == dim
    want = np.empty(words, dtype=np.float32)
    assert hip_to_host(want, data) == 0
    got = buffer.cpu().numpy()
    assert np.array_equal(got[offset:offset + words].view(np.uint32), want.view(np.uint32))
    assert (got[:offset] == 7.25).all() and (got[offset + words:] == 7.25).all()
    assert (rest["lengths"] == 1).all()
    engine.carl_env_destroy(env)


def hip_to_host(out, data):
    hip = C.CDLL("libamdhip64.so")
    return hip.hipMemcpy(C.c_void_p(out.ctypes.data), data, C.c_size_t(out.nbytes), 2)
