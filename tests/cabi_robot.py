"""Robots given to the C ABI as plain node tables (ctypes), with their
kinematics in FP64 numpy: what the URDF path never builds, such as q columns
that drive several joints."""

import ctypes as ct

import numpy as np

import plainmp_amd

FIXED, REVOLUTE, PRISMATIC = 1, 2, 3
i32, i64, f64 = ct.c_int32, ct.c_int64, ct.c_double
CUTOFF = 0.1


class RobotDesc(ct.Structure):
    _fields_ = [("n_nodes", i32)] + [(n, ct.c_void_p) for n in (
        "node_parent", "node_kind", "node_q_col", "node_quat", "node_trans", "node_axis", "node_identity")] + [
        ("n_q_cols", i32), ("base_type", i32), ("base_pose", f64 * 7), ("n_spheres", i32)] + [
        (n, ct.c_void_p) for n in ("sphere_node", "sphere_local", "sphere_radius", "sphere_group")] + [
        ("n_groups", i32), ("group_only_self", ct.c_void_p), ("n_self_pairs", i32), ("self_pairs", ct.c_void_p)]


class PrimDesc(ct.Structure):
    _fields_ = [("type", i32), ("axis_aligned", ct.c_uint8), ("z_axis_aligned", ct.c_uint8), ("position", f64 * 3),
                ("rotation", f64 * 9), ("rotation_inv", f64 * 9), ("size", f64 * 3), ("lb", f64 * 3), ("ub", f64 * 3),
                ("points", ct.c_void_p), ("n_points", i64)]


class SceneDesc(ct.Structure):
    _fields_ = [("n_prims", i32), ("prims", ct.POINTER(PrimDesc))]


def library():
    lib = ct.CDLL(plainmp_amd.LIBRARY_PATH)
    lib.pmp_last_error.restype = ct.c_char_p
    return lib


class Robot:
    """nodes: (parent, kind, q_col, trans, axis) with node 0 the root;
    spheres: (node, centre, radius, group), in group order; fixed or planar
    base (columns x, y, yaw after the joints')."""

    def __init__(self, nodes, spheres, n_groups, pairs=(), planar=False, only_self=()):
        self.nodes, self.spheres, self.pairs, self.planar = nodes, spheres, list(pairs), planar
        self.n_q = 1 + max([n[2] for n in nodes] + [-1])
        self.D = self.n_q + (3 if planar else 0)
        self.only_self = set(only_self)
        N, S = len(nodes), len(spheres)
        a = self._arrays = {
            "node_parent": np.array([n[0] for n in nodes], np.int32),
            "node_kind": np.array([n[1] for n in nodes], np.int32),
            "node_q_col": np.array([n[2] for n in nodes], np.int32),
            "node_quat": np.tile([0.0, 0.0, 0.0, 1.0], (N, 1)),
            "node_trans": np.array([n[3] for n in nodes], float),
            "node_axis": np.array([n[4] for n in nodes], float),
            "node_identity": np.ones(N, np.uint8),
            "sphere_node": np.array([s[0] for s in spheres], np.int32),
            "sphere_local": np.array([s[1] for s in spheres], float),
            "sphere_radius": np.array([s[2] for s in spheres], float),
            "sphere_group": np.array([s[3] for s in spheres], np.int32),
            "group_only_self": np.isin(np.arange(n_groups), list(only_self)).astype(np.uint8),
            "self_pairs": np.array(self.pairs, np.int32).reshape(-1, 2)}
        self.desc = RobotDesc(n_nodes=N, n_q_cols=self.n_q, base_type=int(planar), n_spheres=S, n_groups=n_groups,
                              n_self_pairs=len(self.pairs), base_pose=(f64 * 7)(0, 0, 0, 0, 0, 0, 1),
                              **{k: v.ctypes.data for k, v in a.items()})

    def centres(self, Q):
        """World centres [B][S][3] in FP64."""
        B = len(Q)
        R, t = [None] * len(self.nodes), [None] * len(self.nodes)
        for i, (parent, kind, col, trans, axis) in enumerate(self.nodes):
            if i == 0:
                yaw = Q[:, self.n_q + 2] if self.planar else np.zeros(B)
                R[0] = _rot(np.array([0.0, 0.0, 1.0]), yaw)
                t[0] = np.zeros((B, 3))
                if self.planar:
                    t[0][:, :2] = Q[:, self.n_q:self.n_q + 2]
                continue
            move = np.asarray(trans, float)[None] + (Q[:, col:col + 1] * np.asarray(axis) if kind == PRISMATIC else 0.0)
            t[i] = t[parent] + np.einsum("bij,bj->bi", R[parent], np.broadcast_to(move, (B, 3)))
            R[i] = R[parent] @ _rot(np.asarray(axis, float), Q[:, col]) if kind == REVOLUTE else R[parent]
        return np.stack([t[n] + R[n] @ np.asarray(c, float) for n, c, _, _ in self.spheres], 1)

    def radii(self):
        return np.array([s[2] for s in self.spheres])


def _rot(axis, angle):
    x, y, z = axis
    K = np.array([[0, -z, y], [z, 0, -x], [-y, x, 0]])
    s, c = np.sin(angle)[:, None, None], np.cos(angle)[:, None, None]
    return np.eye(3)[None] + s * K + (1 - c) * (K @ K)


class Balls:
    """A scene of spheres (centre, radius), then point clouds (points, radius)."""

    def __init__(self, balls, clouds=()):
        self.balls = [(np.asarray(c, float), float(r)) for c, r in balls]
        self.clouds = [(np.ascontiguousarray(p, float), float(r)) for p, r in clouds]
        self._prims = (PrimDesc * max(1, len(balls) + len(clouds)))()
        for p, (c, r) in zip(self._prims, self.balls):
            p.type, p.axis_aligned, p.z_axis_aligned = 3, 1, 1
            p.position[:], p.size[:] = list(c), [r, 0.0, 0.0]
            p.rotation[:] = p.rotation_inv[:] = [1.0, 0, 0, 0, 1.0, 0, 0, 0, 1.0]
            p.lb[:], p.ub[:] = list(c - r), list(c + r)
        for p, (points, r) in zip(self._prims[len(balls):], self.clouds):
            p.type, p.axis_aligned, p.z_axis_aligned = 5, 1, 1
            p.rotation[:] = p.rotation_inv[:] = [1.0, 0, 0, 0, 1.0, 0, 0, 0, 1.0]
            p.size[:] = [r, 0.0, 0.0]
            p.lb[:], p.ub[:] = list(points.min(0) - r), list(points.max(0) + r)
            p.points, p.n_points = points.ctypes.data, len(points)
        self.n_prims = len(balls) + len(clouds)
        self.desc = SceneDesc(self.n_prims, self._prims)

    def distances(self, robot, Q):
        """[B][S][P] signed distances in FP64."""
        c = robot.centres(Q)
        d = [np.linalg.norm(c - m, axis=2) - r for m, r in self.balls]
        d += [np.linalg.norm(c[:, :, None] - p, axis=3).min(2) - r for p, r in self.clouds]
        return np.stack(d, 2) - robot.radii()[None, :, None]


def central(f, Q, h=1e-5):
    """Central differences of f(Q) along every column, last axis."""
    out = []
    for j in range(Q.shape[1]):
        e = np.zeros(Q.shape[1])
        e[j] = h
        out.append((f(Q + e) - f(Q - e)) / (2 * h))
    return np.stack(out, -1)


class Context:
    """A context with the robot and scene uploaded; arrays go in as [B][D]
    rows and come back batch first."""

    def __init__(self, robot, scene):
        self.lib, self.robot, self.scene, self.ctx = library(), robot, scene, ct.c_void_p()
        self.ok(self.lib.pmp_create(i32(0), ct.byref(self.ctx)))
        self.ok(self.lib.pmp_upload_robot(self.ctx, ct.byref(robot.desc)))
        self.ok(self.lib.pmp_upload_scene(self.ctx, ct.byref(scene.desc)))

    def __del__(self):
        if self.ctx:
            self.lib.pmp_destroy(self.ctx)

    def ok(self, status):
        if status != 0:
            raise RuntimeError(self.lib.pmp_last_error().decode())

    def _q(self, Q):
        import torch

        q = torch.from_numpy(np.ascontiguousarray(Q.T)).to("cuda")
        torch.cuda.synchronize()
        return q

    @staticmethod
    def _out(*shape, dtype="float32"):
        import torch

        return torch.full(shape, 77, device="cuda", dtype=getattr(torch, dtype))

    @staticmethod
    def _ptr(t):
        return ct.c_void_p(t.data_ptr())

    @staticmethod
    def _host(t):
        import torch

        torch.cuda.synchronize()
        return np.moveaxis(t.cpu().numpy(), -1, 0)

    def pairs(self, Q, grad=True):
        B, S, P = len(Q), len(self.robot.spheres), self.scene.n_prims
        q, dist, g = self._q(Q), self._out(S, P, B), self._out(S, P, self.robot.D, B)
        self.ok(self.lib.pmp_pair_clearance_batch(self.ctx, self._ptr(q), i64(B), i64(B), self._ptr(dist),
                                                  self._ptr(g) if grad else None))
        return self._host(dist), self._host(g)

    def vjp(self, Q, w):
        import torch

        B = len(Q)
        q, out = self._q(Q), self._out(self.robot.D, B)
        wt = torch.from_numpy(np.ascontiguousarray(np.moveaxis(w, 0, -1))).to("cuda")
        torch.cuda.synchronize()
        self.ok(self.lib.pmp_pair_clearance_vjp(self.ctx, self._ptr(q), i64(B), i64(B), self._ptr(wt), self._ptr(out)))
        return self._host(out)

    def evaluate(self, Q):
        B, K = len(Q), 1 + bool(self.robot.pairs)
        q, v, j = self._q(Q), self._out(K, B), self._out(K, self.robot.D, B)
        self.ok(self.lib.pmp_evaluate_batch(self.ctx, self._ptr(q), i64(B), i64(B), self._ptr(v), self._ptr(j)))
        return self._host(v), self._host(j)

    def link_jacobian(self, Q, node, point):
        B = len(Q)
        q, j = self._q(Q), self._out(3, self.robot.D, B)
        self.ok(self.lib.pmp_link_jacobian_batch(self.ctx, self._ptr(q), i64(B), i64(B), i32(node),
                                                 (f64 * 3)(*point), self._ptr(j)))
        return self._host(j)
