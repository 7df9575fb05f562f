"""The cars' and balls' candidate lists leave out no triangle that a test
accepts: poses that touch the mesh at the lists' reach.

A grid cell lists the triangles that come within the car's (or ball's) reach
of it, by the triangle's own distance.  A car's box corners are the points
farthest from its centre, so each car here is put where one corner just
reaches a point of a random triangle (inside it, on an edge or at a vertex,
slivers included), and each ball where its surface just reaches one; the
oracle tests every triangle of the broadphase cell."""
from pathlib import Path

import numpy as np
import pytest

import carl_amd
from carl_amd import workloads
from gpu_harness import Pair

pytestmark = pytest.mark.gpu

HALF = np.array([60.186455, 43.282655, 19.262505])   # the car's half extents
HITBOX = np.array([13.87566, 0.0, 20.755])           # its box's centre in the car's frame
BALL_RADIUS = 91.25


def _mesh():
    v, t = [], []
    for line in (Path(carl_amd.__file__).parent / "assets" / "arena.obj").read_text().splitlines():
        f = line.split()
        if f and f[0] == "v":
            v.append((float(f[2]), float(f[1]), float(f[3])))   # the file swaps the horizontal axes
        elif f and f[0] == "f":
            t.append([int(x.split("/")[0]) - 1 for x in f[1:4]])
    return np.array(v)[np.array(t)]


def _points(rng, tri):
    """A random point of each triangle: a third inside, on an edge, at a vertex."""
    w = rng.dirichlet((1.0, 1.0, 1.0), len(tri))
    kind = rng.integers(0, 3, len(tri))
    w[kind == 1, 2] = 0.0
    w[kind == 2, 1:] = 0.0
    w /= w.sum(1, keepdims=True)
    return np.einsum("tk,tkc->tc", w, tri)


def _rotate(q, v):
    u = q[:, :3]
    t = 2.0 * np.cross(u, v)
    return v + q[:, 3:] * t + np.cross(u, t)


@pytest.mark.parametrize("depth", [-0.5, 0.05, 3.0])
def test_contacts_at_the_lists_reach(gpu, depth):
    """depth: how far past the triangle's point the corner (and the ball's
    surface) reaches; below 0 it stays short of it."""
    rng = np.random.default_rng(int(100 + 10 * depth))
    mesh = _mesh()
    n = 4096
    state = workloads.random_reset_state(rng, n, 1)
    p = _points(rng, mesh[rng.integers(0, len(mesh), n)])
    q = rng.normal(size=(n, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    corner = HALF * rng.choice([-1.0, 1.0], (n, 3))
    reach = np.linalg.norm(HALF)
    centre = p - _rotate(q, corner * (1.0 - depth / reach))
    ball_at = _points(rng, mesh[rng.integers(0, len(mesh), n)])
    away = rng.normal(size=(n, 3))
    away /= np.linalg.norm(away, axis=1, keepdims=True)
    f32 = lambda x: np.ascontiguousarray(x, dtype=np.float32)  # noqa: E731
    state.update(car_position=f32(centre - _rotate(q, np.broadcast_to(HITBOX, (n, 3))))[:, None, :],
                 car_rotation=f32(q)[:, None, :], car_velocity=f32(rng.normal(size=(n, 1, 3)) * 300.0),
                 car_angular_velocity=f32(rng.normal(size=(n, 1, 3))),
                 ball_position=f32(ball_at + away * (BALL_RADIUS - depth)))
    pair = Pair(n, 1, 0, seed=5, frameskip=2)
    pair.apply_reset_state(state)
    pair.step_continuous(workloads.random_continuous_actions(rng, n, 1))
    report = pair.state_mismatches() + pair.output_mismatches()
    pair.close()
    assert not report, "\n  ".join(report)
