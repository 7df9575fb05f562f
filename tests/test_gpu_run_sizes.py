"""Launch shapes chosen by the run's size.

A run too small to fill the GPU is spread over more workgroups: the packing
kernel takes fewer simulations per workgroup (64 down to 32 observation rows'
worth), the window kernel as few as one, its cars split between the two waves.
The sizes here are the smallest, ones that fill no workgroup evenly, and one
past the size at which the packing workgroups are full.
"""
import numpy as np
import pytest
import torch

import carl_amd
from carl_amd import workloads
from gpu_harness import OUTPUTS, Pair, dev

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
    assert p.gpu.tick_window_launch == 1
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
    assert envs[0].tick_window_launch > 1 == envs[1].tick_window_launch
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
