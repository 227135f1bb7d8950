"""Motion checks, validity and evaluate on both sides of the bounds where a
robot's table size decides the form and the waves of a workgroup (GPU), against
the FP64 oracle on samples."""

import numpy as np
import pytest

from plainmp_amd import synth
from support import oracle_cst, product_cst
from test_gpu_staged import _comb, _sample

pytestmark = pytest.mark.gpu


def _setup(name):
    """Robot, base type name, extra columns, scene."""
    solids = dict(prims=synth.mixed_primitives(8, 2))
    cloud = dict(prims=synth.mixed_primitives(3, 2), cloud=synth.shelf_cloud(2000, 2))
    kind, scene = (name[:-6], cloud) if name.endswith("_cloud") else (name, solids)
    if kind == "humanoid":
        return synth.humanoid31(0), "FLOATING", 6, scene
    return {"panda": synth.panda_like, "dual_arm": synth.dual_arm, "fetch": synth.fetch_like,
            "comb": lambda _: _comb()}[kind](0), "FIXED", 0, scene


def _configs(r, extra, n, seed):
    return np.concatenate([synth.uniform_configs(r, n, seed),
                           np.random.default_rng(seed).normal(0, 0.3, (n, extra))], 1)


def _constraints(wl, base):
    from oracle import _oracle
    from plainmp_amd.kinematics import BaseType

    return (oracle_cst(wl, base_type=getattr(_oracle.BaseType, base)),
            product_cst(wl, base_type=getattr(BaseType, base)))


@pytest.mark.parametrize("name,E", [
    ("panda_cloud", 8192), ("panda_cloud", 8193), ("dual_arm", 4096), ("dual_arm", 4097), ("dual_arm_cloud", 8193),
    ("fetch", 8192), ("fetch", 8193), ("humanoid", 1024), ("humanoid", 1025), ("humanoid_cloud", 3000), ("comb", 1024),
    ("comb", 1025)])
def test_motions(name, E):
    from plainmp_amd.ompl import BoxMotionValidator

    r, base, extra, scene = _setup(name)
    wl = synth.Workload("shapes", r, **scene)
    oc, pc = _constraints(wl, base)
    a, b = _configs(r, extra, E, 1), _configs(r, extra, E, 2)
    b = a + np.resize([0.02, 0.2, 1.0], E)[:, None] * (b - a)
    got, n_got = BoxMotionValidator(pc, [0.05] * a.shape[1]).check_motions(a, b)
    at = _sample(E, 250)
    ref, n_ref = oc.check_motions(a[at], b[at], True, [0.05] * a.shape[1], 0.0, 8)
    assert np.array_equal(got[at], ref.astype(bool))
    assert np.array_equal(n_got[at], n_ref)


@pytest.mark.parametrize("name", ["humanoid", "humanoid_cloud", "dual_arm_cloud"])
@pytest.mark.parametrize("B", [9000, 20000, 40000])
def test_configurations(name, B):
    r, base, extra, scene = _setup(name)
    Q = _configs(r, extra, B, 3)
    wl = synth.Workload("shapes", r, Q=Q, **scene)
    oc, pc = _constraints(wl, base)
    at = _sample(B, 100)
    assert np.array_equal(pc.is_valid_batch(Q)[at], oc.is_valid_batch(Q[at], 8).astype(bool))
    # 31 compositions: five times the roundings of a 7-joint arm
    assert np.abs(pc.evaluate_batch(Q)[0][at] - oc.evaluate_batch(Q[at], 8)[0]).max() <= 2.5e-5
