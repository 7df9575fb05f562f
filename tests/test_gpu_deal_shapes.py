"""A tick_window set between dealt launches changes the workgroups the units
are parted over, and with them which units a group's lists hold: the deal
starts over.  The sizes are ones whose launches keep the unit and the number
of groups, but whose groups get other units (769 workgroups of 64 simulations
after 985 of 50)."""
from __future__ import annotations

import numpy as np
import pytest

from carl_amd import workloads
from gpu_harness import dev
from test_gpu_run_sizes import _assert_same_state, _pair_of_envs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,team,window", [(49216, 1, 64), (24608, 2, 32)])
def test_deal_starts_over_with_other_workgroups(gpu, n, team, window):
    rng = np.random.default_rng(n)
    envs = _pair_of_envs(n, team, team, 4, workloads.random_reset_state, rng)
    assert envs[0].tick_balanced_launch and envs[0].tick_window_launch != window
    for step in range(6):
        if step == 3:
            envs[0].tick_window = window
            assert envs[0].tick_balanced_launch and envs[0].tick_window_launch == window
        actions = dev(workloads.random_continuous_actions(rng, n, 2 * team))
        for env in envs:
            env.step_continuous(actions)
        _assert_same_state(envs, f"step {step}")
