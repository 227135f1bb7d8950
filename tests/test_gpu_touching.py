"""Configurations that touch a cylinder exactly, decided without a band (GPU).

A sphere slides along x up to cylinders stacked on one axis.  Radii and positions
are FP32 numbers whose differences are exact and the root of a correctly rounded
square is the number itself, so the test's margin is 0, which counts as in the
band however narrow, and the FP64 test decides as it does with the default
band."""

import numpy as np
import pytest

from plainmp_amd import synth
from support import product_cst

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tilted", [False, True])
def test_touching_cylinders(tilted):
    n, r = 480, 2.0**-8
    radius = np.random.default_rng(1).integers(1 << 18, 1 << 22, n) / 2.0**23  # 0.03 to 0.5 m
    at = (np.arange(n) - n / 2) / 32  # along the axis, within 8 m
    # a quarter turn about x: the axis lies along y
    R = np.array([[1.0, 0, 0], [0, 0, -1], [0, 1, 0]]) if tilted else np.eye(3)
    axis = (0, 1, 0) if tilted else (0, 0, 1)
    prims = [{"type": "cylinder", "radius": a, "height": 2.0**-7, "position": c * np.array(axis), "rotation": R}
             for c, a in zip(at, radius)]
    urdf = ('<?xml version="1.0"?>\n<robot name="slider">\n'
            + "".join(synth._link(x) for x in ("base", "lift", "slide"))
            + synth._joint("j0", "prismatic", "base", "lift", (0, 0, 0), (0, 0, 0), axis=axis, lower=-9, upper=9)
            + synth._joint("j1", "prismatic", "lift", "slide", (0, 0, 0), (0, 0, 0), axis=(1, 0, 0), lower=-9, upper=9)
            + "</robot>\n")
    robot = synth.Robot(urdf, ["j0", "j1"], [("slide", np.zeros((1, 3)), np.array([r]), False)], [], np.full(2, -9.0),
                        np.full(2, 9.0))
    pc = product_cst(synth.Workload("touch", robot, prims))
    for side in (1, -1):
        for off in (0.0, 2.0**-12, -(2.0**-12)):  # touching, outside, inside
            Q = np.stack([at, side * (radius + r + off)], 1)
            assert np.array_equal(Q, Q.astype(np.float32))
            pc.set_band(1e-5)
            ref = pc.is_valid_batch(Q)
            pc.set_band(0.0)
            assert np.array_equal(pc.is_valid_batch(Q), ref)
            if off != 0.0:
                assert ref.all() == (off > 0) and ref.any() == (off > 0)
