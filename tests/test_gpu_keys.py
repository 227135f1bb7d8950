"""Tie keys of evaluate and its form for robots beyond the staged one's limits
(GPU; C ABI): values within 5e-6 m, rows within 1e-4 of FP64 central
differences, ties to the smallest (group, primitive, sphere)."""

import numpy as np
import pytest

from cabi_robot import CUTOFF, PRISMATIC, REVOLUTE, Balls, Context, Robot, central

pytestmark = pytest.mark.gpu

ROOT = (-1, 0, -1, (0, 0, 0), (0, 0, 0))


def _values(robot, scene, Q):
    """FP64 external and self values and whether the winners are clear."""
    c, r = robot.centres(Q), robot.radii()
    group = np.array([s[3] for s in robot.spheres])
    out, clear = [], []
    ext = [g not in robot.only_self for g in group]
    tables = [np.concatenate([np.linalg.norm(c[:, ext] - m, axis=2) - r[ext] - b for m, b in scene.balls], 1)]
    for a, b in robot.pairs:
        ia, ib = np.flatnonzero(group == a), np.flatnonzero(group == b)
        d = np.linalg.norm(c[:, ia, None] - c[:, None, ib], axis=3) - (r[ia][:, None] + r[ib])
        tables.append(d.reshape(len(Q), -1))
    for d in [tables[0]] + ([np.concatenate(tables[1:], 1)] if robot.pairs else []):
        top = np.partition(d, 1, axis=1)[:, :2]
        out.append(np.minimum(top[:, 0], CUTOFF))
        clear.append(top[:, 1] - top[:, 0] > 1e-5)
    return np.stack(out, 1), np.stack(clear, 1)


def _check(robot, scene, Q):
    v, j = Context(robot, scene).evaluate(Q)
    ref, clear = _values(robot, scene, Q)
    assert np.abs(v - ref).max() <= 5e-6
    sel = clear & (np.abs(ref - CUTOFF) > 1e-4)
    assert len(Q) == 1 or sel.mean() > 0.5
    # a step of 1e-7 moves no distance by the 1e-5 that sets the winner apart
    assert np.abs(j - central(lambda x: _values(robot, scene, x)[0], Q, 1e-7))[sel].max() <= 1e-4


def _balls(n, seed):
    rng = np.random.default_rng(seed)
    return Balls([(p, 0.02) for p in rng.uniform([-1, -1, 0], [1, 1, 1], (n, 3))])


@pytest.mark.parametrize("B", [65, 3000])
def test_group_ids_far_beyond_the_sphere_count(B):
    """Empty groups between the used ones: ids whose products with the primitive
    and sphere counts pass 2^32."""
    nodes = [ROOT, (0, REVOLUTE, 0, (0, 0, 0.3), (0, 0, 1)), (1, REVOLUTE, 1, (0.3, 0, 0.1), (0, 1, 0)),
             (2, REVOLUTE, 2, (0.3, 0, 0), (0, 1, 0))]
    spheres = [(i, (0.2, 0.02 * i, 0), 0.05, g) for i, g in ((1, 5), (2, 2796202), (3, 2796203))]
    Q = np.random.default_rng(B).uniform(-1.5, 1.5, (B, 3))
    _check(Robot(nodes, spheres, 2796204), _balls(512, 2), Q)


def test_tie_goes_to_the_smaller_group():
    """Two spheres of a sliding link as far from a ball each, on both sides."""
    ids = (2796202, 2796203)  # times 512 primitives times 3 spheres: below and above 2^32
    nodes = [ROOT, (0, PRISMATIC, 0, (0, 0, 0.25), (1, 0, 0))]
    far = [((0.0, 5.0 + i, 5.0), 0.01) for i in range(510)]
    spheres = [(1, (0.25, 0, 0), 0.0625, ids[0]), (1, (-0.25, 0, 0), 0.0625, ids[1]), (1, (0, 3.0, 0), 0.01, ids[1])]
    near = [((0.5, 0, 0.25), 0.125), ((-0.5, 0, 0.25), 0.125)]
    for balls in (near, near[::-1]):
        v, j = Context(Robot(nodes, spheres, ids[1] + 1), Balls(balls + far)).evaluate(np.zeros((70, 1)))
        assert np.array_equal(v[:, 0], np.full(70, 0.0625, np.float32))
        assert np.abs(j[:, 0, 0] + 1.0).max() <= 1e-6  # the sphere of the first group nears its ball


@pytest.mark.parametrize("B", [1, 70, 600])
def test_a_self_group_beyond_the_staged_keys(B):
    """A group of more than 2,048 spheres in a self pair: the lane-per-configuration form."""
    rng = np.random.default_rng(7)
    nodes = [ROOT, (0, REVOLUTE, 0, (0, 0, 0.3), (0, 0, 1)), (1, REVOLUTE, 1, (0.4, 0, 0), (0, 1, 0)),
             (2, PRISMATIC, 2, (0.1, 0, 0.1), (1, 0, 0))]
    spheres = [(1, c, 0.01, 0) for c in rng.uniform([0, -0.1, -0.1], [0.3, 0.1, 0.1], (2049, 3))]
    spheres += [(3, (0.05 * i, 0, 0), 0.03, 1) for i in range(3)]
    Q = rng.uniform([-1.5, 2.2, -0.1], [1.5, 3.8, 0.1], (B, 3))
    _check(Robot(nodes, spheres, 2, pairs=[(0, 1)], only_self=[0]), _balls(400, 3), Q)


def test_more_keys_than_32_bits():
    """2,900 spheres against 512 primitives: the same form, by its key range."""
    rng = np.random.default_rng(8)
    nodes = [ROOT, (0, REVOLUTE, 0, (0, 0, 0.3), (0, 0, 1)), (1, REVOLUTE, 1, (0.3, 0, 0), (0, 1, 0))]
    spheres = [(1 + k // 1450, c, 0.01, k) for k, c in enumerate(rng.uniform(-0.3, 0.3, (2900, 3)))]
    Q = rng.uniform(-1.5, 1.5, (4, 2))
    _check(Robot(nodes, spheres, 2900), _balls(512, 4), Q)
