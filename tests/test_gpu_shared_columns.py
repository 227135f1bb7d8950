"""Robots with q columns that drive several joints (GPU; C ABI only: the URDF
path gives every joint its own column): the derivative of a column is the sum
over its joints at or above the sphere's link.  Bars as in test_gpu_staged:
distances within 5e-6 m, gradients within 1e-4 of FP64 central differences."""

import numpy as np
import pytest

from cabi_robot import CUTOFF, FIXED, PRISMATIC, REVOLUTE, Balls, Context, Robot, central

pytestmark = pytest.mark.gpu


def _gripper(planar):
    """An arm joint (column 0), two opposed fingers on column 1 whose tips come
    after both in node order, and a chain of two coupled joints on column 2."""
    nodes = [(-1, 0, -1, (0, 0, 0), (0, 0, 0)),
             (0, REVOLUTE, 0, (0, 0, 0.3), (0, 0, 1)),
             (1, FIXED, -1, (0.2, 0, 0), (0, 0, 0)),
             (2, PRISMATIC, 1, (0.05, 0.02, 0), (0, 1, 0)),
             (2, PRISMATIC, 1, (0.05, -0.02, 0), (0, -1, 0)),
             (3, FIXED, -1, (0.06, 0, 0.01), (0, 0, 0)),
             (4, FIXED, -1, (0.06, 0, -0.01), (0, 0, 0)),
             (0, REVOLUTE, 2, (0, 0.1, 0.2), (0, 1, 0)),
             (7, REVOLUTE, 2, (0.15, 0, 0), (0, 1, 0))]
    spheres = [(1, (0.1, 0, 0), 0.04, 0), (2, (0, 0, 0.01), 0.05, 1), (3, (0.01, 0, 0), 0.02, 2),
               (4, (0.01, 0, 0), 0.02, 3), (5, (0, 0.01, 0), 0.015, 4), (6, (0, -0.01, 0), 0.015, 5),
               (6, (0.02, 0, 0), 0.01, 5), (7, (0.08, 0, 0), 0.03, 6), (8, (0.1, 0, 0.02), 0.03, 7)]
    return Robot(nodes, spheres, 8, pairs=[(4, 5), (0, 7), (4, 7)], planar=planar)


BALLS = Balls([((0.3, 0.1, 0.35), 0.05), ((0.25, -0.2, 0.3), 0.08), ((0.2, 0.1, 0.05), 0.1), ((-0.2, 0.1, 0.4), 0.06),
               ((0.05, 0.3, 0.25), 0.05)])


def _configs(robot, B, seed=1):
    rng = np.random.default_rng([B, seed])
    Q = rng.uniform(-1.5, 1.5, (B, robot.D))
    Q[:, 1] = rng.uniform(0, 0.05, B)
    if robot.planar:
        Q[:, robot.n_q:robot.n_q + 2] *= 0.1
    return Q


def _sample(B, k=200):
    return np.arange(B) if B <= k else np.unique(np.concatenate([np.random.default_rng(B).choice(B, k), [0, B - 1]]))


@pytest.mark.parametrize("planar", [False, True])
@pytest.mark.parametrize("B", [1, 70, 4100])
def test_pair_gradients_and_adjoint(planar, B):
    robot = _gripper(planar)
    Q, ctx = _configs(robot, B), Context(robot, BALLS)
    dist, grad = ctx.pairs(Q)
    at = _sample(B)
    assert np.abs(dist[at] - BALLS.distances(robot, Q[at])).max() <= 5e-6
    assert np.abs(grad[at] - central(lambda x: BALLS.distances(robot, x), Q[at])).max() <= 1e-4
    w = np.random.default_rng(2).uniform(size=dist.shape).astype(np.float32)
    ref = np.einsum("bsp,bspj->bj", w.astype(float), grad.astype(float))
    scale = np.einsum("bsp,bspj->bj", w.astype(float), np.abs(grad).astype(float)).max()
    # FP32 sums of S * P terms: a few roundings of the largest partial sum
    assert np.abs(ctx.vjp(Q, w) - ref).max() <= 64 * 6e-8 * max(scale, 1.0)


def _values(robot, Q):
    """FP64 external and self values and whether the winner is clear."""
    d = BALLS.distances(robot, Q).reshape(len(Q), -1)
    c, r = robot.centres(Q), robot.radii()
    group = np.array([s[3] for s in robot.spheres])
    s = np.concatenate([(np.linalg.norm(c[:, group == a][:, :, None] - c[:, group == b][:, None], axis=3)
                         - (r[group == a][:, None] + r[group == b][None])[None]).reshape(len(Q), -1)
                        for a, b in robot.pairs], 1)
    top = [np.sort(x, axis=1) for x in (d, s)]
    return (np.stack([np.minimum(x[:, 0], CUTOFF) for x in top], 1),
            np.stack([x[:, 1] - x[:, 0] > 1e-5 for x in top], 1))


@pytest.mark.parametrize("planar", [False, True])
@pytest.mark.parametrize("B", [1, 70, 2049, 20001])
def test_evaluate_rows(planar, B):
    robot = _gripper(planar)
    Q = _configs(robot, B, 3)
    v, j = Context(robot, BALLS).evaluate(Q)
    at = _sample(B, 400)
    ref, clear = _values(robot, Q[at])
    assert np.abs(v[at] - ref).max() <= 5e-6
    rows = central(lambda x: _values(robot, x)[0], Q[at])
    far = np.abs(ref - CUTOFF) > 1e-4  # not where a difference steps over the cutoff
    sel = clear & far
    assert B < 70 or sel.mean() > 0.8
    assert np.abs(j[at] - rows)[sel].max(initial=0.0) <= 1e-4
    assert np.array_equal(j[at][ref >= CUTOFF], np.zeros_like(j[at][ref >= CUTOFF]))


@pytest.mark.parametrize("planar", [False, True])
@pytest.mark.parametrize("node", [2, 5, 6, 8])
def test_link_jacobian(planar, node):
    robot = _gripper(planar)
    Q, point = _configs(robot, 70, 4), (0.02, -0.01, 0.03)
    probe = Robot(robot.nodes, [(node, point, 0.01, 0)], 1, planar=planar)
    ref = central(lambda x: probe.centres(x)[:, 0], Q)
    assert np.abs(Context(robot, BALLS).link_jacobian(Q, node, point) - ref).max() <= 1e-4
