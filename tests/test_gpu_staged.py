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


def _pair_case(robot, B, n_prims):
    wl = _workload(robot, B, n_prims=n_prims)
    return wl, oracle_cst(wl), product_cst(wl)


@pytest.mark.parametrize("robot,B,n_prims", [("panda", 1, 1), ("panda", 65, 3), ("panda", 2049, 9), ("panda", 2080, 8),
                                             ("fetch", 97, 33), ("dual_arm", 64, 5), ("dual_arm", 1001, 2)])
def test_pair_distances_gradients_and_adjoint(robot, B, n_prims):
    """Whole and odd rows, primitive counts that leave a slice short; gradients
    by central differences of the oracle's distances away from kinks, the
    adjoint as the weighted sum of the gradients."""
    import torch

    wl, oc, pc = _pair_case(robot, B, n_prims)
    dist, grad = pc.pair_clearance_batch(wl.Q, True)
    dist_only = pc.pair_clearance_batch(wl.Q, False)
    assert np.array_equal(dist, dist_only[0] if isinstance(dist_only, tuple) else dist_only)
    idx = _sample(B, 24)
    Q = wl.Q[idx]
    assert np.abs(dist[idx] - oc.pair_clearance_batch(Q, True, 8)).max() <= 5e-6
    D, h = wl.robot.dof, 1e-5
    fd = np.empty((len(Q),) + dist.shape[1:] + (D,))
    sd = np.empty_like(fd)
    for j in range(D):
        e = np.zeros(D)
        e[j] = h
        up, mid, dn = (oc.pair_clearance_batch(Q + k * e, True, 8) for k in (1, 0, -1))
        fd[..., j], sd[..., j] = (up - dn) / (2 * h), np.abs(up - 2 * mid + dn)
    # central differences are off by about h^2 / 6 times the third derivative
    # (below 1e-6 here) unless a kink lies in between, which the second
    # difference shows (a smooth one is about h^2 times the curvature)
    smooth = sd.max(axis=-1) < 1e-8
    assert smooth.mean() > 0.95
    err = np.abs(grad[idx] - fd).max(axis=-1)
    assert err[smooth].max() <= 1e-4
    w = np.random.default_rng(1).uniform(size=dist.shape).astype(np.float32)
    q = torch.from_numpy(np.ascontiguousarray(wl.Q.T)).to("cuda")
    wt = torch.from_numpy(np.ascontiguousarray(w.transpose(1, 2, 0))).to("cuda")
    out = torch.empty((D, B), device="cuda")
    torch.cuda.synchronize()
    pc._dev_pair_clearance_vjp(q.data_ptr(), B, B, wt.data_ptr(), out.data_ptr(), 0)
    torch.cuda.synchronize()
    ref = np.einsum("bsp,bspj->bj", w.astype(np.float64), grad.astype(np.float64))
    scale = np.einsum("bsp,bspj->bj", w.astype(np.float64), np.abs(grad).astype(np.float64)).max()
    # FP32 sums of S * P terms: a few roundings of the largest partial sum
    assert np.abs(out.T.cpu().numpy() - ref).max() <= 64 * 6e-8 * max(scale, 1.0)


def _motions(robot, E, spans, seed=9):
    """Motions whose lengths run through `spans` (of the joint range) in turn,
    some of no length and some with a joint eight turns out of range."""
    r = ROBOTS[robot](0)
    rng = np.random.default_rng(seed)
    a, b = (rng.uniform(r.lower, r.upper, size=(E, r.dof)) for _ in range(2))
    b = a + np.resize(spans, E)[:, None] * (b - a)
    b[5::23] = a[5::23]
    a[7::31, -1] += 16 * np.pi
    b[7::31, -1] += 16 * np.pi
    return r, a, b


@pytest.mark.parametrize("robot,E", [("panda", 1), ("panda", 1024), ("panda", 1025), ("fetch", 257), ("dual_arm", 300)])
@pytest.mark.parametrize("schedule", [(0, 0), (64, 1), (256, 2)])
@pytest.mark.parametrize("band", [None, 0.02])
def test_motions_by_workgroups(robot, E, schedule, band):
    """Motions of 1 to over 128 states (1, 2, 4 and 8 lanes a state, several
    chunks), a workgroup each or a few workgroups for all, on both sides of the
    form's bound; the wide band sends states to the FP64 decisions and more of
    them than a pending list holds."""
    from plainmp_amd.ompl import BoxMotionValidator

    r, a, b = _motions(robot, E, [1.0, 0.02, 0.1, 0.2, 0.4, 3.0])
    wl = synth.Workload("motions", r, synth.mixed_primitives(12, 2))
    oc, pc = oracle_cst(wl), product_cst(wl)
    pc._dev_set_schedule(*schedule, 0, 0)
    if band is not None:
        pc.set_band(band)
    w = [0.05] * r.dof
    ref, n_ref = oc.check_motions(a, b, True, w, 0.0, 8)
    mv = BoxMotionValidator(pc, w)
    for _ in range(2):  # the second call's count starts from zero again
        got, n_got = mv.check_motions(a, b)
        assert np.array_equal(got, ref.astype(bool))
        assert np.array_equal(n_got, n_ref)
        assert 0 <= mv.last_recheck_count() <= E
    if band is not None and E > 1:
        assert mv.last_recheck_count() > 0


@pytest.mark.parametrize("n", [64, 2048, 2049, 4096, 524288, 524289])
def test_cloud_build_sizes(n):
    """One workgroup's keys, the first that take several, and both sides of the
    bound from which the digit counts are summed by a launch of their own; every
    table bit-exact, with runs of equal codes across wave and workgroup borders."""
    from oracle import _oracle
    from plainmp_amd import kdtree as kd

    P = np.random.default_rng(n).uniform(-1, 1, (n, 3))
    P[n // 3 : n // 3 + min(n // 2, 5000)] = P[7]
    got, ref = dict(kd.build_cloud_tiles(P)), dict(_oracle.cloud_tiles(P))
    for d in (got, ref):  # the 8 padding bytes of each 48-byte tile record carry no value
        d["tiles"] = np.frombuffer(d["tiles"], np.uint8).reshape(-1, 48)[:, :40].tobytes()
    for k in ref:
        assert got[k] == ref[k], k


def _comb(n=60):
    """A chain of n joints whose links each carry a sphere, every third one a side
    link with another: more poses than 64 configurations' tables fit LDS with, and more
    path entries than are staged."""
    rng = np.random.default_rng(4)
    links, joints, urdf, specs = ["base"], [], "", []
    for i in range(n):
        prev, ln, side = "base" if i == 0 else f"l{i - 1}", f"l{i}", f"s{i}"
        axis = ((0, 0, 1), (0, 1, 0), (1, 0, 0))[i % 3]
        urdf += synth._joint(f"j{i}", "revolute", prev, ln, (0, 0, 0.05), (0, 0, 0), axis=axis, lower=-0.3, upper=0.3)
        links.append(ln)
        joints.append(f"j{i}")
        specs.append((ln, np.zeros((1, 3)), np.array([0.03]), False))
        if i % 3 == 2:
            urdf += synth._joint(f"f{i}", "fixed", ln, side, (0.04, 0, 0), (0.1, 0.2, 0.3))
            links.append(side)
            specs.append((side, rng.normal(0, 0.01, (1, 3)), np.array([0.02]), False))
    urdf = '<?xml version="1.0"?>\n<robot name="comb">\n' + "".join(synth._link(x) for x in links) + urdf + "</robot>\n"
    return synth.Robot(urdf, joints, specs, [("l0", f"s{n - 1}")], np.full(n, -0.3), np.full(n, 0.3))


def test_a_robot_whose_tables_do_not_fit_64_configurations():
    from plainmp_amd.ompl import BoxMotionValidator

    r = _comb()
    Q = synth.uniform_configs(r, 70, 8)
    wl = synth.Workload("comb", r, synth.mixed_primitives(6, 3), Q=Q)
    oc, pc = oracle_cst(wl), product_cst(wl)
    assert np.array_equal(pc.is_valid_batch(Q), oc.is_valid_batch(Q, 8).astype(bool))
    assert np.abs(pc.evaluate_batch(Q)[0] - oc.evaluate_batch(Q, 8)[0]).max() <= 1e-5
    dist, grad = pc.pair_clearance_batch(Q, True)
    ref = oc.pair_clearance_batch(Q, True, 8)
    assert np.abs(dist - ref).max() <= 1e-5  # 60 compositions: ten times the roundings of a 7-joint arm
    assert np.array_equal(dist, pc.pair_clearance_batch(Q, False)[0])
    h = 1e-5
    for j in (0, 31, 59):
        e = np.zeros(r.dof)
        e[j] = h
        up, dn = (oc.pair_clearance_batch(Q + k * e, True, 8) for k in (1, -1))
        smooth = np.abs(up - 2 * ref + dn) < 1e-8
        assert smooth.mean() > 0.95
        assert np.abs(grad[..., j] - (up - dn) / (2 * h))[smooth].max() <= 1e-4
    w = [0.05] * r.dof
    ok, n_ok = oc.check_motions(Q[:-1], Q[1:], True, w, 0.0, 8)
    got, n_got = BoxMotionValidator(pc, w).check_motions(Q[:-1], Q[1:])
    assert np.array_equal(got, ok.astype(bool)) and np.array_equal(n_got, n_ok)
