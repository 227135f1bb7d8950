"""Batches whose every configuration is decided in FP64 whole (GPU): a joint
eight turns out of the FP32 walk's range, at the batch sizes where the lanes and
waves that share a configuration change, against the FP64 oracle."""

import numpy as np
import pytest

from plainmp_amd import synth
from support import oracle_cst, product_cst
from test_gpu_staged import _comb, _sample

pytestmark = pytest.mark.gpu

CASES = {
    "panda": lambda: (synth.panda_like(0), dict(prims=synth.mixed_primitives(70, 3))),  # over 64 candidates a block
    "fetch_cloud": lambda: (synth.fetch_like(0), dict(prims=synth.mixed_primitives(5, 8),
                                                      cloud=synth.shelf_cloud(3000, 8))),
    "dual_arm": lambda: (synth.dual_arm(0), dict(prims=synth.mixed_primitives(12, 3))),
    "no_scene": lambda: (synth.dual_arm(0), dict(prims=[])),
    "comb": lambda: (_comb(), dict(prims=synth.mixed_primitives(12, 3))),
}


@pytest.mark.parametrize("case", sorted(CASES))
@pytest.mark.parametrize("B", [1, 70, 3000, 6000, 20000, 70000])
def test_validity(case, B):
    r, scene = CASES[case]()
    Q = synth.uniform_configs(r, B, 5)
    Q[:, -1] += 16 * np.pi
    wl = synth.Workload("whole", r, scene.pop("prims"), Q=Q, **scene)
    got, n = product_cst(wl).is_valid_batch_stats(Q)
    at = _sample(B, 300)
    ref = oracle_cst(wl).is_valid_batch(Q[at], 8).astype(bool)
    assert np.array_equal(got[at], ref)
    assert n == B  # every configuration is counted once, whoever shared it
    Q[::2, -1] -= 16 * np.pi  # among configurations in range
    got, n = product_cst(wl).is_valid_batch_stats(Q)
    ref = oracle_cst(wl).is_valid_batch(Q[at], 8).astype(bool)
    assert np.array_equal(got[at], ref)
    assert B // 2 <= n <= B
