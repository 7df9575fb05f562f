"""Launch shapes chosen by the run's size.

A run too small to fill the GPU is spread over more workgroups: the packing
kernel takes fewer simulations per workgroup (64 down to 32 observation rows'
worth), each wave of the window kernel as few as one.  Window launches whose
waves are all resident deal their simulations to the waves in units.  The sizes
here are the smallest, ones that fill no workgroup evenly, and ones past the
size at which the workgroups are full.
"""
import numpy as np
import pytest
import torch

import carl_amd
from carl_amd import workloads
from abi import CAR_NAMES, SIM_NAMES
from gpu_harness import OUTPUTS, Pair, describe_mismatch, dev, gpu_state, pad_reset_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n_blue,n_orange", [
    (1, 1, 1),      # one simulation: one packing workgroup, one wave with cars
    (17, 1, 1),     # a packing workgroup of 16 and one of 1
    (33, 1, 0),     # one car each: 32 rows and 1
    (19, 2, 1),     # an odd number of cars per workgroup, 16 simulations each
    (9, 4, 4),      # packing workgroups of 4, 4 and 1
])
def test_small_runs_match_the_oracle(gpu, n, n_blue, n_orange):
    """Short episodes, so that resets and transition rows run on most steps."""
    rng = np.random.default_rng(n + 10 * n_blue)
    nc = n_blue + n_orange
    p = Pair(n, n_blue, n_orange, seed=3, frameskip=4)
    assert p.gpu.tick_window_launch == 2        # one simulation per wave
    p.set_param("max_ticks", 13)
    p.set_param("overtime_timeout_ticks", 8)
    p.apply_reset_state(workloads.clustered_reset_state(rng, n, nc))
    for step in range(12):
        p.step_continuous(workloads.random_continuous_actions(rng, n, nc))
        report = p.state_mismatches() + p.output_mismatches()
        assert not report, f"after step {step}:\n  " + "\n  ".join(report)
    p.close()


@pytest.mark.parametrize("n,n_blue,n_orange", [(33000, 1, 1), (4099, 4, 4), (5003, 2, 2)])
def test_large_run_equals_a_small_one(gpu, n, n_blue, n_orange):
    """The first simulations of a large run, whose packing workgroups are full
    (33,000) and whose window workgroups hold several simulations, against the
    same simulations on their own."""
    rng = np.random.default_rng(n)
    nc, few = n_blue + n_orange, 37
    envs = [carl_amd.Env(k, n_blue, n_orange, 3, 4, True, False, True) for k in (n, few)]
    assert envs[0].tick_window_launch > 2 == envs[1].tick_window_launch
    state = workloads.clustered_reset_state(rng, n, nc)
    for env in envs:
        env.max_ticks = 13
        env.overtime_timeout_ticks = 8
        env.apply_reset_state(**{k: dev(v[:env.n_sim]) for k, v in state.items()})
    for step in range(8):
        actions = workloads.random_continuous_actions(rng, n, nc)
        for env in envs:
            env.step_continuous(dev(actions[:env.n_sim]))
            env.synchronize()
        for name in OUTPUTS:
            a, b = (torch.from_dlpack(getattr(env, "get_" + name)())[:few].cpu().numpy() for env in envs)
            assert a.tobytes() == b.tobytes(), (name, step)


def _pair_of_envs(n, n_blue, n_orange, frameskip, make_state, rng):
    """The same environment twice, the second on the phase kernels."""
    envs = [carl_amd.Env(n, n_blue, n_orange, 5, frameskip, True, False, True) for _ in range(2)]
    envs[1].tick_window = 0
    state = {k: dev(v) for k, v in make_state(rng, n, n_blue + n_orange).items()}
    for env in envs:
        env.max_ticks = 40 * frameskip
        env.apply_reset_state(**state)
    return envs


def _assert_same_state(envs, context):
    a, b = gpu_state(envs[0]), gpu_state(envs[1])
    report = describe_mismatch(CAR_NAMES, a[0], b[0]) + describe_mismatch(SIM_NAMES, a[1], b[1])
    assert not report, f"{context}:\n  " + "\n  ".join(report)


@pytest.mark.parametrize("n,n_blue,n_orange", [
    (1, 1, 1),        # one unit: most waves have none
    (7, 2, 2),        # fewer workgroups than XCDs
    (1000, 1, 1),     # one simulation per unit and wave
    (4099, 4, 4),     # two or three units per wave
    (4097, 3, 2),     # the instance for any team size
    (10007, 2, 2),    # the last unit not full, groups of unequal size
    (30011, 1, 0),    # one car per simulation
    (9001, 3, 3),
    (50001, 1, 1),    # units of whole cache lines that do not go round
    (65536 + 64, 1, 1),   # more workgroups than are resident, dealt as one group
    (65536 + 32, 1, 1),   # the same with a workgroup that is not full: not dealt
])
def test_dealt_launches_match_the_phase_kernels(gpu, n, n_blue, n_orange):
    """Launches of a size's own shape (no tick_window set), dealt from the
    second step on, against the phase kernels: clustered scenes, masked resets
    in between, and a launch too short to be dealt."""
    rng = np.random.default_rng(n)
    nc = n_blue + n_orange
    envs = _pair_of_envs(n, n_blue, n_orange, 4, workloads.clustered_reset_state, rng)
    assert envs[0].tick_balanced_launch == (n != 65536 + 32)
    for step in range(10):
        if step == 4:
            mask = dev(rng.uniform(size=n) < 0.25)
            fresh = {k: dev(v) for k, v in workloads.random_reset_state(rng, n, nc).items()}
            for env in envs:
                env.apply_reset_state(**fresh, reset_mask=mask)
        actions = dev(workloads.random_continuous_actions(rng, n, nc))
        for env in envs:
            if step == 7:
                env.tick(actions.reshape(-1), 1, 2)
            else:
                env.step_continuous(actions)
        _assert_same_state(envs, f"step {step}")


@pytest.mark.parametrize("n,n_blue,n_orange,ticks", [
    (40, 1, 1, 63), (40, 1, 1, 64), (41, 1, 1, 65), (19, 3, 3, 130), (70, 1, 0, 200), (9, 4, 4, 530)])
def test_pads_over_long_launches(gpu, n, n_blue, n_orange, ticks):
    """The window kernel counts the pads' cooldowns down once for up to 64
    ticks of a launch: cars parked on pads (some sharing one), small pads that
    recover within a launch (480 ticks), cooldowns left over from the launch
    before, against the phase kernels."""
    rng = np.random.default_rng(n + ticks)
    nc = n_blue + n_orange
    envs = _pair_of_envs(n, n_blue, n_orange, 4, pad_reset_state, rng)
    for launch in range(4):
        actions = workloads.random_continuous_actions(rng, n, nc) * (0.0 if launch % 2 else 1.0)
        for env in envs:
            env.tick(dev(actions.astype(np.float32)).reshape(-1), 1, ticks if launch != 2 else 5)
        _assert_same_state(envs, f"launch {launch}")
