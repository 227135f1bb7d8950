"""A robot of 60 columns and 80 poses (GPU): its tables do not fit LDS with as
many configurations as a workgroup takes at the larger batch sizes, so
validity and evaluate give each configuration more lanes than its batch size
asks for.  Against the FP64 oracle on samples; 60 compositions: ten times the
roundings of a 7-joint arm."""

import numpy as np
import pytest

from plainmp_amd import synth
from support import oracle_cst, product_cst, rows_agree
from test_gpu_staged import _comb, _sample

pytestmark = pytest.mark.gpu


def _scene():
    """Balls, boxes and cylinders beside the upper half of the chain."""
    rng = np.random.default_rng(6)
    prims = []
    for k in range(18):
        a, z = rng.uniform(0, 2 * np.pi), rng.uniform(1.0, 2.6)
        at = np.array([0.8 * np.cos(a), 0.8 * np.sin(a), z])
        shape = [{"type": "sphere", "radius": 0.1}, {"type": "box", "width": np.full(3, 0.15)},
                 {"type": "cylinder", "radius": 0.08, "height": 0.2}][k % 3]
        prims.append({**shape, "position": at, "rotation": np.eye(3)})
    return prims


@pytest.mark.parametrize("B", [70, 3000, 6000, 9000, 20000, 40000])
def test_validity_and_rows(B):
    r = _comb()
    Q = synth.uniform_configs(r, B, 8)
    wl = synth.Workload("comb", r, _scene(), Q=Q)
    oc, pc = oracle_cst(wl), product_cst(wl)
    at = _sample(B, 64)
    S = Q[at]
    assert np.array_equal(pc.is_valid_batch(Q)[at], oc.is_valid_batch(S, 8).astype(bool))
    vref, jref = oc.evaluate_batch(S, 8)
    v, j = pc.evaluate_batch(Q)
    assert np.abs(v[at] - vref).max() <= 1e-5
    # rows of clear winners; within 1e-4 of the cutoff a difference may step over it
    d = np.sort(oc.pair_clearance_batch(S, True, 8).reshape(len(S), -1), axis=1)
    ext = (d[:, 1] - d[:, 0] > 1e-4) & (vref[:, 0] < 0.1 - 1e-4)
    assert ext.sum() >= 5
    rows_agree(oc, S, j[at], jref, ext, 0)
    for row in range(vref.shape[1]):
        none = vref[:, row] >= 0.1
        assert np.array_equal(j[at][none, row], np.zeros_like(jref[none, row]))
