"""The window kernel's suspension shares a wave's wheels in contact out to its
lanes, 64 a round, while they are at most 128; with more, every lane computes
its own car's.  Waves of 64 cars with the numbers of wheels on the floor around
those limits, cars on some of their wheels only among them, against the oracle.
"""
import numpy as np
import pytest

from carl_amd import workloads
from gpu_harness import Pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grounded", [(1, 15), (16, 17), (31, 32), (33, 64), (0, 24)])
def test_wheels_in_contact_match_the_oracle(gpu, grounded):
    """Two waves of 64 cars: `grounded` cars of each stand on the floor, most
    on four wheels and every fifth tilted onto two or three."""
    rng = np.random.default_rng(grounded)
    n = 128
    state = workloads.random_reset_state(rng, n, 1)
    state["car_position"][:, 0] = np.stack([rng.uniform(-3000, 3000, n), rng.uniform(-4000, 4000, n), np.full(n, 900.0)], 1)
    tilt = 0
    for wave, count in enumerate(grounded):
        for car in 64 * wave + rng.permutation(64)[:count]:
            state["car_position"][car, 0, 2] = 17.0
            tilt += 1
            if tilt % 5 == 0:      # rolled or pitched: one side's or end's wheels leave the floor
                roll, pitch = rng.choice([(0.25, 0.0), (0.0, 0.2), (0.12, 0.1), (-0.25, 0.05)])
                state["car_position"][car, 0, 2] = 22.0
                q = np.array([np.sin(roll / 2), np.sin(pitch / 2), 0.0, 1.0])
                state["car_rotation"][car, 0] = q / np.linalg.norm(q)
    p = Pair(n, 1, 0, seed=5, frameskip=1)
    p.gpu.tick_window = 128         # one workgroup: 64 cars in each wave
    assert p.gpu.tick_window_launch == 128
    p.apply_reset_state(state)
    for launch in range(6):
        p.tick(workloads.random_continuous_actions(rng, n, 1), 1, 1 if launch < 3 else 4)
        report = p.state_mismatches()
        assert not report, f"after launch {launch}:\n  " + "\n  ".join(report)
    p.close()
