"""Performance cases: the work a motion planner or trajectory optimiser has
the framework do, through the entry points such a program calls.

A case names its path (``kind``), robot, scene and size.  The kinds and the
ranges that ``draw`` spreads over:

    valid      validity of a batch of sampled configurations        64 .. 131,072
    edges      motions between sampled states, resident on the GPU  32 .. 4,096
    path       the segments of one planner path, host arrays        16 .. 2,048 states
    pair       every sphere-primitive distance with its gradient    64 .. 8,192
    autograd   distances forward and their adjoint backward         64 .. 8,192
    evaluate   constraint values with Jacobian rows                 64 .. 16,384
    traj       evaluate rows + smoothness of uneven trajectories    1 .. 2,048
    build      spatial structure of a point cloud from the GPU      1,000 .. 1,048,576 points

Robots and scenes are the seeded ones of ``plainmp_amd.synth``: a Panda-class
arm, the same arm on a lift, a Fetch-like robot with self pairs and a dual
arm, among two bars, mixed primitives or a scanned shelf.  The scene,
configurations and motions follow the seed; the robot does not.  All results
a kind returns are whole; ``exact`` gives them in FP64 wherever they are
computed numbers (booleans, counts and packed tables have no such value).
"""

from __future__ import annotations

import math
import xml.etree.ElementTree as ET

import numpy as np
import torch

from plainmp_amd import roofline, synth

CUTOFF = 0.1  # the largest value SphereCollisionCst.evaluate returns
ROBOTS = ("panda_like", "mobile_torso", "fetch_like", "dual_arm")
EDGE_STATES = 50  # states a motion across the joint range has checked, on average


def listed():
    return [
        # a sampler's rejection test, the smallest device batch: launches and latency count
        {"name": "valid_bars_1024", "kind": "valid", "robot": "panda_like", "scene": "bars", "size": 1024},
        # a roadmap's samples, more than one round of lane-per-configuration waves, ragged, with self pairs
        {"name": "valid_fetch_100003", "kind": "valid", "robot": "fetch_like", "scene": "mixed", "prims": 16,
         "size": 100003},
        # the same test against a scanned scene
        {"name": "valid_cloud_16384", "kind": "valid", "robot": "mobile_torso", "scene": "cloud", "points": 65536,
         "size": 16384},
        # path simplification: one planner path checked from host arrays, a call per path
        {"name": "path_mixed_65", "kind": "path", "robot": "panda_like", "scene": "mixed", "prims": 16, "span": 0.15,
         "size": 65},
        # roadmap edges across the joint range: the batched motion check
        {"name": "edges_mixed_4096", "kind": "edges", "robot": "panda_like", "scene": "mixed", "prims": 16,
         "span": 1.0, "size": 4096},
        # the same against a scanned scene
        {"name": "edges_cloud_4096", "kind": "edges", "robot": "mobile_torso", "scene": "cloud", "points": 65536,
         "span": 1.0, "size": 4096},
        # gradient-based planning that wants every distance and its derivative
        {"name": "pair_mixed_8192", "kind": "pair", "robot": "panda_like", "scene": "mixed", "prims": 32, "size": 8192},
        # a learned or optimised cost through torch.autograd: distances forward, adjoint backward
        {"name": "autograd_mixed_8191", "kind": "autograd", "robot": "panda_like", "scene": "mixed", "prims": 32,
         "size": 8191},
        # the collision rows of a batch of IK restarts
        {"name": "evaluate_bars_256", "kind": "evaluate", "robot": "panda_like", "scene": "bars", "size": 256},
        # the collision rows of many solver instances
        {"name": "evaluate_mixed_8192", "kind": "evaluate", "robot": "panda_like", "scene": "mixed", "prims": 32,
         "size": 8192},
        # a batch of trajectories of uneven length: rows of every waypoint, smoothness cost and gradient
        {"name": "traj_dual_arm_2048", "kind": "traj", "robot": "dual_arm", "scene": "mixed", "prims": 24,
         "size": 2048},
        # a depth frame (640 x 480) made into the structure the cloud checks walk
        {"name": "build_307200", "kind": "build", "points": 307200, "size": 307200},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["valid", "edges", "path", "pair", "autograd", "evaluate", "traj", "build"])
    if kind == "build":
        n = _log_int(rng, 1000, 1 << 20)
        return {"kind": kind, "points": n, "size": n}
    case = {"kind": kind, "robot": rng.choice(ROBOTS)}
    scenes = ["bars", "mixed", "mixed"] + (["cloud"] if kind in ("valid", "edges", "path") else [])
    case["scene"] = rng.choice(scenes)
    if case["scene"] == "mixed":
        case["prims"] = rng.randint(3, 32 if kind in ("pair", "autograd") else 48)
    if case["scene"] == "cloud":
        case["robot"] = rng.choice(["panda_like", "mobile_torso"])
        case["points"] = _log_int(rng, 1000, 65536)
    if kind in ("edges", "path"):
        # from a planner's extension step to the whole joint range
        case["span"] = round(math.exp(rng.uniform(math.log(0.05), 0.0)), 3) if kind == "edges" else \
            round(rng.uniform(0.02, 0.3), 3)
    size = {"valid": (64, 131072), "edges": (32, 4096), "path": (16, 2048), "pair": (64, 8192),
            "autograd": (64, 8192), "evaluate": (64, 16384), "traj": (1, 2048)}[kind]
    case["size"] = _log_int(rng, *size)
    if case["scene"] == "cloud" and kind == "valid":
        case["size"] = min(case["size"], 16384)
    if kind in ("pair", "autograd") and case["robot"] == "dual_arm":
        case["size"] = max(64, case["size"] // 6)  # 160 spheres x 14 columns: the same memory
    return case


# ------------------------------------------------------------------ inputs
def _robot(case):
    return getattr(synth, case["robot"])(0)


def _prims(case, seed):
    if case["scene"] == "bars":
        return synth.two_bars(seed)
    if case["scene"] == "mixed":
        return synth.mixed_primitives(case["prims"], seed)
    return []


def _configs(robot, n, seed):
    return synth.uniform_configs(robot, n, [seed, 1])


def _ends(case, robot, seed):
    """Start states over the joint range and end states `span` of it away
    (1: anywhere), inside the limits."""
    rng = np.random.default_rng([seed, 2])
    a = rng.uniform(robot.lower, robot.upper, size=(case["size"], robot.dof))
    b = rng.uniform(robot.lower, robot.upper, size=(case["size"], robot.dof))
    return a, a + case["span"] * (b - a)


def _path(case, robot, seed):
    rng = np.random.default_rng([seed, 3])
    step = rng.normal(scale=case["span"], size=(case["size"], robot.dof))
    step[0] = rng.uniform(robot.lower, robot.upper)
    return np.clip(np.cumsum(step, axis=0), robot.lower, robot.upper)


def _trajectories(case, robot, seed):
    """Lines between two states with a small wiggle, 20 to 100 waypoints (the
    lengths belong to the case, not to the seed)."""
    rng = np.random.default_rng([seed, 4])
    lens = np.random.default_rng(case["size"]).integers(20, 101, size=case["size"])
    off = np.zeros(case["size"] + 1, dtype=np.int64)
    off[1:] = np.cumsum(lens)
    which = np.repeat(np.arange(case["size"]), lens)
    t = (np.arange(off[-1]) - off[which]) / (lens[which] - 1)
    a = rng.uniform(robot.lower, robot.upper, size=(case["size"], robot.dof))
    b = rng.uniform(robot.lower, robot.upper, size=(case["size"], robot.dof))
    X = a[which] + t[:, None] * (b - a)[which] + rng.normal(0.0, 0.02, size=(int(off[-1]), robot.dof))
    return off, X


def _frame(n, seed):
    """Points of a scanned scene: a table and two shelf planes."""
    return synth.shelf_cloud(n, seed)


def _soa(x):
    return torch.from_numpy(np.ascontiguousarray(x.T)).to("cuda")


def _weights(case, robot, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.rand((robot.n_spheres, len(_prims(case, seed)), case["size"]), device="cuda", generator=g)


def _empty(shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device="cuda")


def prepare(case, seed):
    from plainmp_amd.ompl import BoxMotionValidator

    s = {"case": case}
    if case["kind"] == "build":
        from plainmp_amd._native import kdtree

        n = case["points"]
        nt, ns, scratch = kdtree.cloud_tile_sizes(n)
        s["points"] = torch.from_numpy(_frame(n, seed)).to("cuda")
        # cleared once: the records' padding is never written
        s["tables"] = [_empty(int(b), torch.uint8).zero_() for b in (48 * nt, 48 * nt, 1024 * nt, 2048 * nt, 32 * ns)]
        s["scratch"] = _empty(int(scratch), torch.uint8)
        return s
    robot, n = _robot(case), case["size"]
    cloud = _frame(case["points"], seed) if case["scene"] == "cloud" else None
    wl = synth.Workload("case", robot, _prims(case, seed), cloud=cloud)
    # the spheres keep the order given, so that results are in the order of the specs
    cst = s["cst"] = synth.build_constraint(wl, reorder=False)
    S, P, D, C = cst.n_spheres(), cst.n_prims(), cst.q_dim(), cst.cst_dim()
    kind = case["kind"]
    if kind in ("edges", "path"):
        s["mv"] = BoxMotionValidator(cst, [0.05] * D)
    if kind == "path":
        s["P"] = _path(case, robot, seed)
    elif kind == "edges":
        a, b = _ends(case, robot, seed)
        s["s1"], s["s2"] = _soa(a), _soa(b)
        s["out"] = (_empty(n, torch.uint8), _empty(n, torch.int32))
    elif kind == "autograd":
        s["q"] = torch.from_numpy(_configs(robot, n, seed)).to("cuda").requires_grad_()
        # upstream weights as elementwise losses of the distances leave them
        s["w"] = _weights(case, robot, seed).permute(2, 0, 1)
    elif kind == "traj":
        off, X = _trajectories(case, robot, seed)
        s["x"], s["off"] = _soa(X), [int(v) for v in off]
        s["out"] = (_empty((C, len(X))), _empty((C, D, len(X))), _empty(n), _empty((D, len(X))))
    else:
        s["q"] = _soa(_configs(robot, n, seed))
        if kind == "valid":
            s["out"] = (_empty(n, torch.uint8),)
        elif kind == "pair":
            s["out"] = (_empty((S, P, n)), _empty((S, P, D, n)))
        else:
            s["out"] = (_empty((C, n)), _empty((C, D, n)))
    return s


def run(s):
    case = s["case"]
    kind, n = case["kind"], case["size"]
    st = torch.cuda.current_stream().cuda_stream
    if kind == "valid":
        s["cst"]._dev_is_valid(s["q"].data_ptr(), n, n, s["out"][0].data_ptr(), 0, st)
    elif kind == "edges":
        s["mv"]._dev_check_motions(s["s1"].data_ptr(), s["s2"].data_ptr(), n, n, s["out"][0].data_ptr(),
                                   s["out"][1].data_ptr(), st)
    elif kind == "path":
        return s["mv"].check_path(s["P"])
    elif kind == "pair":
        s["cst"]._dev_pair_clearance(s["q"].data_ptr(), n, n, s["out"][0].data_ptr(), s["out"][1].data_ptr(), st)
    elif kind == "autograd":
        from plainmp_amd.autograd import pair_clearance

        d = pair_clearance(s["cst"], s["q"])
        (g,) = torch.autograd.grad(d, s["q"], grad_outputs=s["w"])
        return d.detach(), g
    elif kind == "evaluate":
        s["cst"]._dev_evaluate(s["q"].data_ptr(), n, n, s["out"][0].data_ptr(), s["out"][1].data_ptr(), st)
    elif kind == "traj":
        N = s["off"][-1]
        s["cst"]._dev_traj_cost_grad(s["x"].data_ptr(), N, N, s["off"], [], *(o.data_ptr() for o in s["out"]), st)
    else:
        from plainmp_amd._native import kdtree

        kdtree._dev_cloud_build_tiles(s["points"].data_ptr(), n, *(t.data_ptr() for t in s["tables"]),
                                      s["scratch"].data_ptr(), st)
        return list(s["tables"])
    return s["out"]


# -------------------------------------------------------------------- work
def work(case):
    kind, n = case["kind"], case["size"]
    if kind == "build":  # points in; tables of 64-point tiles out
        return {"bytes": n * 24 + math.ceil(n / 64) * 3168, "flops": n * 20}
    robot, D = _robot(case), _robot(case).dof
    prims = _prims(case, 0)
    S, P, pairs = robot.n_spheres, len(prims), synth.self_pair_count(robot)
    C = (1 if P else 0) + (1 if pairs else 0)
    check = roofline.config_flops(robot, prims, pairs)
    if kind == "valid":
        return {"bytes": n * (8 * D + 1), "flops": n * check}
    if kind in ("edges", "path"):
        states = max(1.0, EDGE_STATES * case["span"]) if kind == "edges" else max(1.0, 2.0 * case["span"] / 0.05)
        return {"bytes": n * (16 * D + 5), "flops": n * states * (check + 3 * D)}
    if kind == "pair":
        return {"bytes": n * (8 * D + 4 * S * P * (1 + D)), "flops": n * (check + S * P * (12 + 17 * D / 2))}
    if kind == "autograd":
        return {"bytes": n * (16 * D + 8 * S * P), "flops": n * (2 * check + S * P * 18)}
    if kind == "evaluate":
        return {"bytes": n * (8 * D + 4 * C * (1 + D)), "flops": n * roofline.evaluate_flops(robot, prims, pairs)}
    N = 60 * n
    return {"bytes": N * (8 * D + 4 * C * (1 + D) + 4 * D), "flops": N * roofline.traj_waypoint_flops(robot, prims, pairs)}


# ---------------------------------------------------------- FP64 results
def _rpy(r, p, y):
    cr, sr, cp, sp, cy, sy = math.cos(r), math.sin(r), math.cos(p), math.sin(p), math.cos(y), math.sin(y)
    rx = np.array([[1, 0, 0], [0, cr, -sr], [0, sr, cr]])
    ry = np.array([[cp, 0, sp], [0, 1, 0], [-sp, 0, cp]])
    rz = np.array([[cy, -sy, 0], [sy, cy, 0], [0, 0, 1]])
    return rz @ ry @ rx


class _Fk:
    """Forward kinematics of a robot's URDF in FP64 for a batch q (B, D):
    centres (B, 3) of a link's spheres and the (axis, origin, rotates) of the
    controlled joints above each link."""

    def __init__(self, robot, q):
        self.B, self.dev = q.shape[0], q.device
        eye = torch.eye(3, dtype=torch.float64, device=self.dev).expand(self.B, 3, 3)
        zero = torch.zeros((self.B, 3), dtype=torch.float64, device=self.dev)
        root = ET.fromstring(robot.urdf)
        joints = root.findall("joint")
        children = {j.find("child").get("link") for j in joints}
        self.pose, self.cols = {}, {}
        for link in root.findall("link"):
            if link.get("name") not in children:
                self.pose[link.get("name")], self.cols[link.get("name")] = (eye, zero), {}
        todo = list(joints)
        while todo:
            j = next(j for j in todo if j.find("parent").get("link") in self.pose)
            todo.remove(j)
            parent, child = j.find("parent").get("link"), j.find("child").get("link")
            R, t = self.pose[parent]
            o = j.find("origin")
            xyz = self._vec(o.get("xyz", "0 0 0"))
            R0 = torch.tensor(_rpy(*map(float, o.get("rpy", "0 0 0").split())), dtype=torch.float64, device=self.dev)
            cols = dict(self.cols[parent])
            t = t + R @ xyz
            R = R @ R0
            if j.get("type") in ("revolute", "continuous", "prismatic") and j.get("name") in robot.joint_names:
                k = robot.joint_names.index(j.get("name"))
                a = self._vec(j.find("axis").get("xyz"))
                rev = j.get("type") != "prismatic"
                if rev:
                    K = torch.tensor([[0, -a[2], a[1]], [a[2], 0, -a[0]], [-a[1], a[0], 0]], dtype=torch.float64,
                                     device=self.dev)
                    th = q[:, k, None, None]
                    R = R @ (torch.eye(3, dtype=torch.float64, device=self.dev) + torch.sin(th) * K
                             + (1 - torch.cos(th)) * (K @ K))
                else:
                    t = t + q[:, k, None] * (R @ a)
                cols[k] = (R @ a, t, rev)
            self.pose[child], self.cols[child] = (R, t), cols

    def _vec(self, text):
        return torch.tensor([float(v) for v in text.split()], dtype=torch.float64, device=self.dev)

    def centre(self, link, p):
        R, t = self.pose[link]
        return t + R @ torch.as_tensor(p, dtype=torch.float64, device=self.dev)

    def column(self, link, k, c):
        """d c / d q_k (B, 3) of a point c on a link, or None."""
        if k not in self.cols[link]:
            return None
        a, o, rev = self.cols[link][k]
        return torch.linalg.cross(a, c - o) if rev else a


def _sdf(p, c):
    """Signed distance and its gradient of a primitive at points c (B, 3)."""
    R = torch.as_tensor(np.asarray(p["rotation"], float), device=c.device)
    d = (c - torch.as_tensor(np.asarray(p["position"], float), device=c.device)) @ R
    if p["type"] == "sphere":
        n = d.norm(dim=1)
        return n - p["radius"], (d / n[:, None]) @ R.T
    if p["type"] == "box":
        u, e = torch.sign(d), d.abs() - torch.as_tensor(np.asarray(p["width"], float) / 2, device=c.device)
        directions = u[:, :, None] * torch.eye(3, dtype=c.dtype, device=c.device)
    else:
        rho = d[:, :2].norm(dim=1)
        e = torch.stack([rho - p["radius"], d[:, 2].abs() - p["height"] / 2], dim=1)
        radial = torch.cat([d[:, :2] / rho[:, None], torch.zeros_like(d[:, 2:])], dim=1)
        axial = torch.zeros_like(d)
        axial[:, 2] = torch.sign(d[:, 2])
        directions = torch.stack([radial, axial], dim=1)
    out = e.clamp(min=0.0)
    dist = out.norm(dim=1)
    inside = e.max(dim=1)
    weights = torch.where((dist > 0)[:, None], out / dist.clamp(min=1e-300)[:, None],
                          torch.nn.functional.one_hot(inside.indices, e.shape[1]).to(c.dtype))
    g = (weights[:, :, None] * directions).sum(dim=1)
    return dist + inside.values.clamp(max=0.0), g @ R.T


def _spheres(robot):
    return [(link, np.asarray(pos)[i], float(r[i]), bool(only)) for link, pos, r, only in robot.sphere_specs
            for i in range(len(r))]


def _exact_pairs(robot, prims, q, w=None):
    """dist (S, P, B) and its gradient (S, P, D, B), or with weights w
    (S, P, B) the adjoint (B, D)."""
    fk, sp = _Fk(robot, q), _spheres(robot)
    B, D = q.shape
    dist = torch.zeros((len(sp), len(prims), B), dtype=torch.float64, device=q.device)
    grad = torch.zeros((len(sp), len(prims), D, B) if w is None else (B, D), dtype=torch.float64, device=q.device)
    for s, (link, p, r, _) in enumerate(sp):
        c = fk.centre(link, p)
        cols = {k: fk.column(link, k, c) for k in fk.cols[link]}
        for i, prim in enumerate(prims):
            d, g = _sdf(prim, c)
            dist[s, i] = d - r
            for k, col in cols.items():
                if w is None:
                    grad[s, i, k] = (g * col).sum(dim=1)
                else:
                    grad[:, k] += w[s, i].double() * (g * col).sum(dim=1)
    return dist, grad


def _exact_rows(robot, prims, q):
    """Values (C, B) and rows (C, D, B): the smallest clearance to the
    primitives, then between the self pairs, each at most CUTOFF."""
    fk, sp = _Fk(robot, q), _spheres(robot)
    B, D = q.shape
    centres = [fk.centre(link, p) for link, p, _, _ in sp]

    def least():
        return (torch.full((B,), CUTOFF, dtype=torch.float64, device=q.device),
                torch.zeros((D, B), dtype=torch.float64, device=q.device))

    vals, rows = [], []
    if prims:
        best, row = least()
        for s, (link, _, r, only) in enumerate(sp):
            if only:
                continue
            cols = {k: fk.column(link, k, centres[s]) for k in fk.cols[link]}
            for prim in prims:
                d, g = _sdf(prim, centres[s])
                less = d - r < best
                best = torch.where(less, d - r, best)
                row = torch.where(less, 0.0, row)
                for k, col in cols.items():
                    row[k] = torch.where(less, (g * col).sum(dim=1), row[k])
        vals.append(best)
        rows.append(row)
    if robot.self_pairs:
        best, row = least()
        for a, b in robot.self_pairs:
            for s in (i for i, x in enumerate(sp) if x[0] == a):
                for t in (i for i, x in enumerate(sp) if x[0] == b):
                    d = centres[s] - centres[t]
                    n = d.norm(dim=1)
                    less = n - sp[s][2] - sp[t][2] < best
                    best = torch.where(less, n - sp[s][2] - sp[t][2], best)
                    row = torch.where(less, 0.0, row)
                    for k in set(fk.cols[a]) | set(fk.cols[b]):
                        ca, cb = fk.column(a, k, centres[s]), fk.column(b, k, centres[t])
                        move = (0.0 if ca is None else ca) - (0.0 if cb is None else cb)
                        row[k] = torch.where(less, (d / n[:, None] * move).sum(dim=1), row[k])
        vals.append(best)
        rows.append(row)
    return torch.stack(vals), torch.stack(rows)


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("pair", "autograd", "evaluate", "traj"):
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    robot, prims = _robot(case), _prims(case, seed)
    if kind == "traj":
        off, X = _trajectories(case, robot, seed)
        x = torch.from_numpy(X).to(dev)
        parts = [_exact_rows(robot, prims, part) for part in x.split(1 << 15)]
        vals, jac = (torch.cat([p[i] for p in parts], dim=-1) for i in (0, 1))
        # second differences inside each trajectory, and the gradient of their sum of squares
        acc = torch.zeros_like(x)
        acc[1:-1] = x[:-2] - 2 * x[1:-1] + x[2:]
        ends = torch.from_numpy(np.concatenate([off[:-1], off[1:] - 1])).to(dev)
        acc[ends] = 0.0
        grad = -4 * acc
        grad[1:] += 2 * acc[:-1]
        grad[:-1] += 2 * acc[1:]
        total = torch.cat([torch.zeros(1, dtype=x.dtype, device=dev), (acc ** 2).sum(dim=1).cumsum(dim=0)])
        o = torch.from_numpy(off).to(dev)
        return vals, jac, total[o[1:]] - total[o[:-1]], grad.T
    q = torch.from_numpy(_configs(robot, case["size"], seed)).to(dev)
    if kind == "pair":
        return _exact_pairs(robot, prims, q)
    if kind == "autograd":
        dist, grad = _exact_pairs(robot, prims, q, _weights(case, robot, seed))
        return dist.permute(2, 0, 1), grad
    return _exact_rows(robot, prims, q)
