"""Pair distances and gradients against point clouds (GPU): robots of 7 to 60
columns, scenes with and without solids and with several clouds, and q columns
that drive several joints.  Distances within 5e-6 m (1e-5 for 60 compositions),
gradients within 1e-4 of central differences where those meet no kink."""

import numpy as np
import pytest

from cabi_robot import Balls, Context, central
from plainmp_amd import synth
from support import oracle_cst, product_cst
from test_gpu_shared_columns import _configs, _gripper
from test_gpu_staged import _comb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("robot,B,n_prims", [("panda", 1, 0), ("panda", 70, 9), ("panda", 3000, 3), ("humanoid", 70, 0),
                                             ("humanoid", 600, 11), ("comb", 70, 0), ("comb", 300, 9)])
def test_distances_and_gradients(robot, B, n_prims):
    from oracle import _oracle
    from plainmp_amd.kinematics import BaseType

    r = {"panda": synth.panda_like, "humanoid": synth.humanoid31, "comb": lambda _: _comb()}[robot](0)
    extra, base = (6, "FLOATING") if robot == "humanoid" else (0, "FIXED")
    Q = np.concatenate([synth.uniform_configs(r, B, 4), np.random.default_rng(4).normal(0, 0.3, (B, extra))], 1)
    wl = synth.Workload("clouds", r, synth.mixed_primitives(n_prims, 6), cloud=synth.shelf_cloud(1500, 6))
    oc = oracle_cst(wl, base_type=getattr(_oracle.BaseType, base))
    pc = product_cst(wl, base_type=getattr(BaseType, base))
    dist, grad = pc.pair_clearance_batch(Q, True)
    assert np.array_equal(dist, pc.pair_clearance_batch(Q, False)[0])
    at = np.unique(np.r_[0, B - 1, np.random.default_rng(B).choice(B, min(B, 10))])
    S = Q[at]
    ref = oc.pair_clearance_batch(S, True, 8)
    assert np.abs(dist[at] - ref).max() <= (1e-5 if robot == "comb" else 5e-6)
    h = 1e-5
    for j in range(0, Q.shape[1], 1 if robot == "panda" else 4):
        e = np.zeros(Q.shape[1])
        e[j] = h
        up, dn = (oc.pair_clearance_batch(S + k * e, True, 8) for k in (1, -1))
        smooth = np.abs(up - 2 * ref + dn) < 1e-8
        assert smooth.mean() > 0.9
        assert np.abs(grad[at][..., j] - (up - dn) / (2 * h))[smooth].max() <= 1e-4


@pytest.mark.parametrize("planar", [False, True])
@pytest.mark.parametrize("B", [70, 2100])
def test_several_clouds_and_shared_columns(planar, B):
    rng = np.random.default_rng(3)
    scene = Balls([((0.3, 0.1, 0.35), 0.05)], [(rng.uniform([-0.5, -0.5, 0], [0.5, 0.5, 0.6], (n, 3)), 0.01)
                                               for n in (70, 300, 1)])
    robot = _gripper(planar)
    Q, ctx = _configs(robot, B), Context(robot, scene)
    dist, grad = ctx.pairs(Q)
    assert np.array_equal(dist, ctx.pairs(Q, False)[0])
    at = np.arange(B)[:: max(1, B // 70)]
    f = lambda x: scene.distances(robot, x)
    assert np.abs(dist[at] - f(Q[at])).max() <= 5e-6
    # a step of 1e-6 crosses a change of the nearest point at most where the
    # second difference shows it
    h = 1e-6
    ref = central(f, Q[at], h)
    kink = np.zeros(ref.shape[:3], bool)
    for j in range(robot.D):
        e = np.zeros(robot.D)
        e[j] = h
        kink |= np.abs(f(Q[at] + e) - 2 * f(Q[at]) + f(Q[at] - e)) > 1e-9
    assert kink.mean() < 0.05
    assert np.abs(grad[at] - ref).max(-1)[~kink].max() <= 1e-4
    w = rng.uniform(size=dist.shape).astype(np.float32)
    total = np.einsum("bsp,bspj->bj", w.astype(float), grad.astype(float))
    scale = np.einsum("bsp,bspj->bj", w.astype(float), np.abs(grad).astype(float)).max()
    # FP32 sums of S * P terms: a few roundings of the largest partial sum
    assert np.abs(ctx.vjp(Q, w) - total).max() <= 64 * 6e-8 * max(scale, 1.0)
