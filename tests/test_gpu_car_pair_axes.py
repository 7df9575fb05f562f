"""Car pairs whose boxes meet at every kind of edge axis.

The pair test leaves out an edge axis that provably cannot replace the
shallowest overlap found so far; the clip of the incident face returns a
polygon that no plane cuts as it is.  Pairs at random orientations, at almost
parallel ones (edge axes near zero length), at right angles (edge axes that tie
with face axes) and far from the field's centre (where the projections round
most) against the oracle, every result bit for bit.
"""
import numpy as np
import pytest

from carl_amd import workloads
from gpu_harness import Pair

pytestmark = pytest.mark.gpu


def _rotations(rng, n, kind):
    if kind == "random":
        q = rng.normal(size=(n, 4))
    elif kind == "near_parallel":
        # a common random rotation, one car turned by up to 1e-7 .. 1e-1 rad about each axis
        q = np.concatenate([rng.normal(size=(n, 3)) * 10.0 ** rng.uniform(-7, -1, (n, 1)), np.ones((n, 1))], axis=1)
    else:
        # quarter turns about a random axis of the car, most of them exact
        axis = np.eye(3)[rng.integers(0, 3, n)]
        half = rng.integers(0, 4, n) * (np.pi / 4) + rng.choice([0.0, 0.0, 1e-6, 1e-3], n)
        q = np.concatenate([axis * np.sin(half)[:, None], np.cos(half)[:, None]], axis=1)
    return q / np.linalg.norm(q, axis=1, keepdims=True)


@pytest.mark.parametrize("kind", ["random", "near_parallel", "quarter_turns"])
@pytest.mark.parametrize("corner", [False, True])
def test_pairs_match_the_oracle(gpu, kind, corner):
    rng = np.random.default_rng([len(kind), corner])
    n = 4000
    state = workloads.random_reset_state(rng, n, 2)
    at = np.stack([rng.uniform(-2500, 2500, n), rng.uniform(-3500, 3500, n), rng.uniform(400, 1500, n)], axis=1)
    if corner:
        at = np.array([3300.0, 4300.0, 1700.0]) + rng.uniform(-100, 100, (n, 3))
    # centres from deep inside each other to just apart
    away = rng.normal(size=(n, 3))
    away *= rng.uniform(5, 130, (n, 1)) / np.linalg.norm(away, axis=1, keepdims=True)
    state["car_position"] = np.stack([at, at + away], axis=1).astype(np.float32)
    state["car_rotation"] = np.stack([_rotations(rng, n, "quarter_turns" if kind != "random" else kind),
                                      _rotations(rng, n, kind)], axis=1).astype(np.float32)
    state["car_velocity"] = (rng.normal(size=(n, 2, 3)) * 400).astype(np.float32)
    state["ball_position"][:] = [0.0, 0.0, 1900.0]
    p = Pair(n, 1, 1, seed=5, frameskip=1)
    p.apply_reset_state(state)
    for tick in range(3):
        p.tick(workloads.random_continuous_actions(rng, n, 2), 1)
        report = p.state_mismatches()
        assert not report, f"after tick {tick}:\n  " + "\n  ".join(report)
    p.close()
