"""Pair distances and gradients far out and where no direction is defined (GPU).

The distance is that of the primitives' formulas in FP32: infinite beyond the
square root of the largest float, and a NaN coordinate's terms count as 0 (every
comparison with them is false)."""

import numpy as np
import pytest

from cabi_robot import Balls, Context, Robot
from plainmp_amd import synth
from support import product_cst

pytestmark = pytest.mark.gpu

_R = synth._rot_rpy(0.3, -0.5, 0.9)
_AT = np.array([0.5, 0.1, 0.4])
_BOX = {"type": "box", "width": np.array([0.2, 0.3, 0.4]), "position": _AT}
_CYL = {"type": "cylinder", "radius": 0.1, "height": 0.8, "position": _AT}
PRIMS = {
    "box": {**_BOX, "rotation": np.eye(3)},
    "box_rot": {**_BOX, "rotation": _R},
    "cylinder": {**_CYL, "rotation": np.eye(3)},
    "cylinder_rot": {**_CYL, "rotation": _R},
    "sphere": {"type": "sphere", "radius": 0.1, "position": _AT, "rotation": np.eye(3)},
    "ground": {"type": "ground", "height": 0.1},
}
VALUES = [0.3, 1e3, 1e15, 3e19, -3e19, 1e30, -1e30, np.inf, -np.inf, np.nan]


def _distance(p, c):
    """The formula in FP32 (c [..., 3] FP32 centres)."""
    f = np.float32
    pos = lambda x: np.where(x > 0, x, f(0))
    neg = lambda x: np.where(x < 0, x, f(0))
    if p["type"] == "ground":
        return c[..., 2] + f(p["height"])
    d = c - np.asarray(p["position"], f)
    if p["type"] == "sphere":
        return np.sqrt((d * d).sum(-1)) - f(p["radius"])
    if not np.array_equal(p["rotation"], np.eye(3)):
        R = np.asarray(p["rotation"], f)
        d = d[..., 0, None] * R[0] + d[..., 1, None] * R[1] + d[..., 2, None] * R[2]
    if p["type"] == "box":
        s = np.abs(d) - np.asarray(p["width"], f) / 2
    else:
        rho = np.sqrt(d[..., 0] ** 2 + d[..., 1] ** 2)
        s = np.stack([rho - f(p["radius"]), np.abs(d[..., 2]) - f(p["height"] / 2)], -1)
    return np.sqrt((pos(s) ** 2).sum(-1)) + neg(s).max(-1)


@pytest.mark.parametrize("kind", sorted(PRIMS))
def test_far_and_nan_bases(kind):
    from plainmp_amd.kinematics import BaseType

    r, prim = synth.panda_like(0), PRIMS[kind]
    Q = np.zeros((2 * len(VALUES) + 1, r.dof + 3))
    Q[:, : r.dof] = synth.uniform_configs(r, len(Q), 1)
    for i, v in enumerate(VALUES):
        Q[i, r.dof] = v
        Q[len(VALUES) + i, r.dof + 1] = v
    Q[-1, r.dof:r.dof + 2] = 3e19, -3e19
    pc = product_cst(synth.Workload("far", r, [prim]), base_type=BaseType.PLANAR)
    dist, grad = pc.pair_clearance_batch(Q, True)
    radii = _distance(prim, pc.sphere_centers_batch(Q[:1], True)[0]) - dist[0, :, 0]
    with np.errstate(all="ignore"):
        ref = _distance(prim, pc.sphere_centers_batch(Q, True)) - radii
    got = dist[..., 0]
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.isinf(got), np.isinf(ref))
    ok = np.isfinite(ref)
    # a few roundings of the largest of the numbers involved
    assert (np.abs(got[ok] - ref[ok]) <= 1e-6 * np.maximum(1.0, np.abs(ref[ok]))).all()
    # a translation of the base changes a distance by at most as much, also where
    # the distance is infinite (a cylinder's radial part is then inf / inf)
    finite = np.isfinite(Q).all(axis=1)
    if prim["type"] == "cylinder":
        finite &= np.isfinite(got).all(axis=1)
    assert (np.abs(grad[finite][..., r.dof:r.dof + 2]) <= 1 + 1e-5).all()


@pytest.mark.parametrize("B", [21, 700])
@pytest.mark.parametrize("kind", sorted(PRIMS))
def test_far_and_nan_bases_distances_alone(kind, B):
    """The kernel without gradients, which leaves workgroups with such a base to
    the formulas; those without one keep the bits they have beside gradients."""
    from plainmp_amd.kinematics import BaseType

    r, prim = synth.panda_like(0), PRIMS[kind]
    Q = np.zeros((B, r.dof + 3))
    Q[:, : r.dof] = synth.uniform_configs(r, B, 1)
    odd = np.r_[0, np.arange(1, len(VALUES) + 1) * (B // 32 or 1)][: len(VALUES)]
    Q[odd, r.dof + np.arange(len(odd)) % 2] = VALUES
    pc = product_cst(synth.Workload("far", r, [prim]), base_type=BaseType.PLANAR)
    got, beside = pc.pair_clearance_batch(Q, False)[0][..., 0], pc.pair_clearance_batch(Q, True)[0][..., 0]
    assert np.array_equal(np.isnan(got), np.isnan(beside)) and np.array_equal(np.isinf(got), np.isinf(beside))
    ok = np.isfinite(got)
    assert (np.abs(got[ok] - beside[ok]) <= 1e-6 * np.maximum(1.0, np.abs(beside[ok]))).all()
    clean = np.ones(B, bool)  # configurations more than a workgroup's 64 from an odd one
    for i in odd:
        clean[max(0, i - 64): i + 65] = False
    assert np.array_equal(got[clean], beside[clean]) and (B < 100 or clean.any())


@pytest.mark.parametrize("at", [2e14, 1e16, 3e19])
def test_far_primitives_and_links(at):
    robot = Robot([(-1, 0, -1, (0, 0, 0), (0, 0, 0)), (0, 2, 0, (0, 0, 0.5), (0, 0, 1))], [(1, (0.1, 0, 0), 0.1, 0)], 1)
    long = Robot([(-1, 0, -1, (0, 0, 0), (0, 0, 0)), (0, 2, 0, (at, 0, 0.5), (0, 0, 1))], [(1, (0.1, 0, 0), 0.1, 0)], 1)
    near, far = ((0, 0.3, 0.5), 0.2), ((at, 0, 0), 0.2)
    with np.errstate(over="ignore"):
        d = np.float32(np.sqrt(np.float32(at) * np.float32(at)))
    for ctx, ref in ((Context(robot, Balls([near, far])), d), (Context(long, Balls([near])), d)):
        for grad in (False, True):
            dist = ctx.pairs(np.zeros((3, 1)), grad)[0][:, 0, -1]
            assert np.array_equal(np.isinf(dist), np.full(3, np.isinf(ref)))
            assert np.isinf(ref) or np.abs(dist - ref).max() <= 1e-6 * ref


def test_centre_on_centre():
    """A sphere at a ball's very centre: the distance is minus both radii and no
    direction is preferred."""
    robot = Robot([(-1, 0, -1, (0, 0, 0), (0, 0, 0)), (0, 2, 0, (0, 0, 0.5), (0, 0, 1))], [(1, (0, 0, 0), 0.1, 0)], 1)
    dist, grad = Context(robot, Balls([((0, 0, 0.5), 0.2)])).pairs(np.array([[0.0], [0.7]]))
    assert np.abs(dist - -0.3).max() <= 1e-7
    assert np.array_equal(grad, np.zeros_like(grad))
