"""Staged workgroups (several waves per group of configurations) at the batch
sizes where their launch shape changes, against the FP64 oracle (GPU).

Bars as in test_gpu_parity: booleans exact, values within 5e-6 m, rows within
1e-4 relative wherever the winning pair is unambiguous.  Large batches are
compared on their first and last configurations and a random sample.
"""

import numpy as np
import pytest

from plainmp_amd import synth
from support import oracle_cst, product_cst, rows_agree

pytestmark = pytest.mark.gpu

ROBOTS = {"panda": synth.panda_like, "fetch": synth.fetch_like, "dual_arm": synth.dual_arm}


def _sample(n, k=96, seed=0):
    idx = np.random.default_rng(seed).choice(n, min(n, k), replace=False)
    return np.unique(np.concatenate([idx, np.arange(min(n, 4)), np.arange(max(0, n - 4), n)]))


def _workload(robot, B, n_prims=24, seed=3):
    r = ROBOTS[robot](0)
    return synth.Workload("staged", r, synth.mixed_primitives(n_prims, seed), Q=synth.uniform_configs(r, B, seed))


@pytest.mark.parametrize("robot", sorted(ROBOTS))
@pytest.mark.parametrize("B", [1, 63, 4096, 4097, 8193, 16385, 32769])
def test_evaluate_batch_sizes(robot, B):
    wl = _workload(robot, B)
    oc, pc = oracle_cst(wl), product_cst(wl)
    idx = _sample(B)
    Q = wl.Q[idx]
    vref, jref = oc.evaluate_batch(Q, 8)
    v, j = pc.evaluate_batch(wl.Q)
    assert np.abs(v[idx] - vref).max() <= 5e-6
    # central differences settle a row at a kink; ties of the winner are left out
    d = np.sort(oc.pair_clearance_batch(Q, True, 8).reshape(len(Q), -1), axis=1)
    if not any(s[3] for s in wl.robot.sphere_specs):  # only-self spheres are not among the external pairs
        rows_agree(oc, Q, j[idx], jref, (d[:, 1] - d[:, 0] > 1e-5) & (vref[:, 0] < 0.1), 0)
    for row in range(vref.shape[1]):
        none = vref[:, row] >= 0.1  # no pair within the cutoff: a zero row
        assert np.array_equal(j[idx][none, row], np.zeros_like(jref[none, row]))


@pytest.mark.parametrize("lengths", [[0, 1, 2, 0, 3, 64, 65, 0], [100] * 400])
def test_trajectory_costs_in_the_evaluate_launch(lengths):
    """Empty and shortest trajectories, and enough for whole-block launches."""
    r = synth.dual_arm(0)
    off = np.concatenate([[0], np.cumsum(lengths)]).astype(int)
    X = synth.uniform_configs(r, int(off[-1]), 5)
    wl = synth.Workload("traj", r, synth.mixed_primitives(8, 5))
    _, _, cost, grad = product_cst(wl).traj_cost_grad_batch(X, list(off))
    for i, (a, b) in enumerate(zip(off[:-1], off[1:])):
        x = X[a:b]
        acc = np.zeros_like(x)
        acc[1:-1] = x[:-2] - 2 * x[1:-1] + x[2:] if len(x) > 2 else acc[1:-1]
        g = -4 * acc
        g[1:] += 2 * acc[:-1]
        g[:-1] += 2 * acc[1:]
        # one rounding of the FP64 sum; the gradient's terms likewise
        assert abs(cost[i] - (acc ** 2).sum()) <= 1e-6 * (acc ** 2).sum()
        assert np.abs(grad[a:b] - g).max(initial=0.0) <= 1e-6 * max(1.0, np.abs(g).max(initial=0.0))


@pytest.mark.parametrize("robot", sorted(ROBOTS))
@pytest.mark.parametrize("B", [1, 65, 2049, 4097, 8193, 16385, 32769])
def test_validity_batch_sizes(robot, B):
    wl = _workload(robot, B, n_prims=6)
    got = product_cst(wl).is_valid_batch(wl.Q)
    idx = _sample(B, 2048)
    assert np.array_equal(got[idx], oracle_cst(wl).is_valid_batch(wl.Q[idx], 8).astype(bool))


@pytest.mark.parametrize("band", [0.0, 1e-5, 2e-3, 0.2])
@pytest.mark.parametrize("B", [37, 3000])
def test_validity_pending_pairs(band, B):
    """Solid, cloud and self pairs on the pending list, from none to far more
    than it holds (then whole configurations are re-decided): the answer is
    that of the FP64 tests at every band."""
    r = synth.fetch_like(0)
    Q = synth.uniform_configs(r, B, 8)
    wl = synth.Workload("pending", r, synth.mixed_primitives(5, 8), cloud=synth.shelf_cloud(3000, 8), Q=Q)
    oc, pc = oracle_cst(wl), product_cst(wl)
    pc.set_band(band)
    got, n = pc.is_valid_batch_stats(Q)
    ref = oc.is_valid_batch(Q, 8).astype(bool)
    assert 0.02 < ref.mean() < 0.98 or B < 100
    if band > 0:  # with no band the FP32 decisions stand, a few ulps of the distances off
        assert np.array_equal(got, ref)
    assert 0 <= n <= B and (band < 0.1 or n > 0)
