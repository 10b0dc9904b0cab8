"""The framework's measured cases: what a program that uses it has it do.

Kinds of case:

  frame   frames of one scene through ``capi.World`` from a snapshot of the
          state (a planner's or trainer's reset, then its steps); ``blocking``
          steps read the frame's counts back, as the stress driver does,
          the others leave everything on the device.
  batch   frames of many independent scenes in one ``capi.Batch.step``.
  grad    a differentiable rollout: ``dy_diff_forward``, then
          ``dy_diff_backward`` of a given adjoint of the final state.
  rays    closest-hit ray queries over the tree of the scene's broadphase.
  sort    the compute layer's key sort.

State, adjoints, rays and keys live in tensors on the GPU whose addresses the
C ABI takes; outputs are those tensors.  The library's streams and torch's
share the one HIP runtime of the process (torch is imported first), so
``torch.cuda.synchronize()`` waits for both.

Frames, pairs, contacts and hits are deterministic to the bit, which is the
library's contract, so those cases compare exactly.

All states work on one stream: the library's grid-synchronised kernels expect
the device to run one stream's work at a time (see DYPHUR_COOP_LAUNCH).
"""
import ctypes as C
import math

import numpy as np
import torch

from dyphur_amd import capi, scenes

F32 = np.float32
N_STATE = 13  # pos, rot, vel, ang: the first fields of capi.BODY_FLOAT_FIELDS


def listed():
    return [
        # A robot-sized scene, each step's counts read back: launches and latency; reference-order solver.
        {"name": "frame_blocks_63", "kind": "frame", "scene": "blocks", "n": 63, "at": 30, "frames": 2,
         "blocking": True},
        # The reference's own demo scene, settling, stepped as its driver does.
        {"name": "frame_blocks_1024", "kind": "frame", "scene": "blocks", "n": 1024, "at": 150, "frames": 4,
         "blocking": True},
        # A game- or robotics-sized pile in mid-run.
        {"name": "frame_mixed_5000", "kind": "frame", "scene": "mixed", "n": 5000, "at": 240, "frames": 4,
         "blocking": False},
        # The 32 768-body workload near the settled end of its 600-frame run.
        {"name": "frame_mixed_32768", "kind": "frame", "scene": "mixed", "n": 32768, "at": 480, "frames": 4,
         "blocking": False},
        # A larger pile while it collapses (odd body count).
        {"name": "frame_mixed_98305", "kind": "frame", "scene": "mixed", "n": 98305, "at": 150, "frames": 2,
         "blocking": False},
        # Articulated chains: joints with limits and motors beside contacts.
        {"name": "frame_joints_8192", "kind": "frame", "scene": "chains", "n": 8192, "at": 60, "frames": 4,
         "blocking": False},
        # Many small environments stepped together: a training batch, and the full 4 096-pile workload.
        {"name": "batch_piles_300", "kind": "batch", "scenes": 300, "median": 48, "top": 256, "at": 60,
         "frames": 10},
        {"name": "batch_piles_4096", "kind": "batch", "scenes": 4096, "median": 64, "top": 512, "at": 60,
         "frames": 20},
        # Trajectory optimisation of thrown stacks: forward and backward, short horizon.
        {"name": "grad_stacks_256", "kind": "grad", "scene": "stack", "scenes": 256, "median": 64, "top": 64,
         "substeps": 1, "at": 0, "frames": 20, "every": 10},
        # The same over ragged mixed scenes with substeps (workgroup-sized scenes among them), a second into their
        # run, when the lower bodies have landed.
        {"name": "grad_mixed_200", "kind": "grad", "scene": "mixed", "scenes": 200, "median": 128, "top": 600,
         "substeps": 4, "at": 60, "frames": 10, "every": 5},
        # A lidar sweep over the 32 768-body pile.
        {"name": "rays_mixed_32768", "kind": "rays", "n": 32768, "at": 240, "rays": 65536},
        # Key sort of the compute layer: 63-bit keys with a payload, odd count.
        {"name": "sort_u64_1000003", "kind": "sort", "n": 1000003},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "batch", "grad", "rays", "sort"])
    if kind == "frame":
        what = rng.choice(["blocks", "mixed", "mixed", "chains"])
        n = _log(rng, 30, {"blocks": 4000, "mixed": 80000, "chains": 9000}[what])
        return {"kind": "frame", "scene": what, "n": n, "at": rng.randrange(0, 300 if n < 20000 else 180),
                "frames": rng.randrange(1, 4), "blocking": rng.random() < 0.5}
    if kind == "batch":
        return {"kind": "batch", "scenes": _log(rng, 16, 3000), "median": rng.randrange(20, 80),
                "top": rng.randrange(128, 512), "at": rng.randrange(0, 100), "frames": rng.randrange(1, 16)}
    if kind == "grad":
        what = rng.choice(["stack", "mixed"])
        return {"kind": "grad", "scene": what, "scenes": _log(rng, 8, 256 if what == "stack" else 160),
                "median": 64 if what == "stack" else rng.randrange(30, 150),
                "top": 64 if what == "stack" else rng.randrange(200, 600),
                "substeps": rng.choice([1, 2, 4]), "at": rng.randrange(0, 60), "frames": rng.randrange(4, 12),
                "every": rng.choice([3, 5, 10])}
    if kind == "rays":
        return {"kind": "rays", "n": _log(rng, 100, 40000), "at": rng.randrange(0, 200), "rays": _log(rng, 500, 200000)}
    return {"kind": "sort", "n": _log(rng, 1000, 3000000)}


# ---------------------------------------------------------------------------
# Scenes
# ---------------------------------------------------------------------------
def _random_mixed(n_dyn, rng, scale=1.0):
    """scenes.random_mixed's distribution (2/3 boxes, 1/3 spheres over a
    ground plate, one body per 1.1 m^3 of a 30:40:30 volume at scale 1), drawn
    with numpy so that large scenes are quick to make."""
    n = n_dyn + 1
    side = (n_dyn / 32768.0) ** (1.0 / 3.0) if scale == 1.0 else 1.0
    ex, ey, ez = 30.0 * side * scale, 40.0 * side * scale, 30.0 * side * scale
    box = rng.permutation(n_dyn) < (2 * n_dyn) // 3
    half = np.where(box[:, None], rng.uniform(0.1, 0.5, (n_dyn, 3)), rng.uniform(0.1, 0.4, (n_dyn, 1))) * scale
    half = half.astype(F32).astype(np.float64)
    mass = np.where(box, 8000.0 * half.prod(1), 4000.0 * math.pi / 3.0 * half[:, 0] ** 3)
    sq = half ** 2
    diag = np.where(box[:, None], mass[:, None] / 3.0 * (sq.sum(1, keepdims=True) - sq), 0.4 * mass[:, None] * sq)
    pos = np.zeros((n, 3), F32)
    pos[:-1, 0] = rng.uniform(-ex / 2, ex / 2, n_dyn)
    pos[:-1, 1] = rng.uniform(0, ey, n_dyn) + scale
    pos[:-1, 2] = rng.uniform(-ez / 2, ez / 2, n_dyn)
    q = rng.normal(size=(n, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    q[-1] = 1.0, 0.0, 0.0, 0.0
    inertia = np.zeros((n, 9), F32)
    inertia[:, [0, 4, 8]] = 1.0
    inertia[:-1, [0, 4, 8]] = diag
    ground = max(2.0, 20.0 * side * scale)
    top = ey + 5.0 + scale
    return scenes.Scene(
        name="random_mixed", shape_type=np.append(np.where(box, scenes.SHAPE_BOX, scenes.SHAPE_SPHERE),
                                                  scenes.SHAPE_BOX).astype(np.uint32),
        shape_half=np.vstack([half, [ground, 0.5, ground]]).astype(F32), pos=pos, rot=q.astype(F32),
        vel=np.zeros((n, 3), F32), ang=np.zeros((n, 3), F32), mass=np.append(mass, 0.0).astype(F32), inertia=inertia,
        shape=np.arange(n, dtype=np.uint32), flags=np.append(np.zeros(n_dyn), scenes.FLAG_STATIC).astype(np.uint32),
        bounds=np.array([-ground, -2.0, -ground, ground, top, ground], F32), max_pairs=48 * n, max_contacts=16 * n)


def _blocks(n_dyn, rng):
    """scenes.stress_blocks with about n_dyn boxes, each nudged by up to 2 cm."""
    nx = max(2, round((n_dyn / 2.0) ** (1.0 / 3.0)))
    sc = scenes.stress_blocks(nx, max(1, n_dyn // (nx * nx)), nx)
    sc.pos[:-1] += rng.uniform(-0.02, 0.02, (sc.n - 1, 3)).astype(F32)
    return sc


def _counts(n_scenes, median, lo, hi):
    """Bodies per scene, lognormal; the sizes belong to the case, so that every seed's outputs have one shape."""
    rng = np.random.default_rng([n_scenes, median, hi])
    return np.clip(np.round(median * np.exp(0.75 * rng.normal(size=n_scenes))), lo, hi).astype(int)


def _piles(counts, rng):
    """scenes.pile_scene for each count (jittered columns of up to 8 boxes with
    5 cm gaps and small initial velocities), drawn with numpy."""
    n_dyn = counts.astype(int)
    off = np.concatenate([[0], np.cumsum(n_dyn)])
    total = off[-1]
    scene = np.repeat(np.arange(len(n_dyn)), n_dyn)
    k = np.arange(total) - off[scene]
    cols = (n_dyn + 7) // 8
    side = np.maximum(1, np.ceil(np.sqrt(cols)).astype(int))[scene]
    c, level = k % cols[scene], k // cols[scene]
    h = rng.uniform(0.1, 0.4, (total, 3)).astype(F32).astype(np.float64)
    pos = np.empty((total, 3))
    pos[:, 0] = (c % side - (side - 1) / 2.0) * 1.1 + rng.uniform(-0.05, 0.05, total)
    pos[:, 2] = (c // side - (side - 1) / 2.0) * 1.1 + rng.uniform(-0.05, 0.05, total)
    column = np.lexsort((level, c, scene))
    step = (0.05 + 2.0 * h[:, 1])[column]
    below = np.cumsum(step) - step
    first = level[column] == 0
    below -= np.maximum.accumulate(np.where(first, below, 0.0))
    pos[column, 1] = 0.5 + below + 0.05 + h[column, 1]
    mass = 8000.0 * h.prod(1)
    sq = h ** 2
    diag = mass[:, None] / 3.0 * (sq.sum(1, keepdims=True) - sq)
    vel = 0.5 * rng.normal(size=(total, 3))
    out = []
    for s, m in enumerate(n_dyn):
        b = slice(off[s], off[s] + m)
        n = m + 1
        inertia = np.zeros((n, 9), F32)
        inertia[:, [0, 4, 8]] = 1.0
        inertia[:-1, [0, 4, 8]] = diag[b]
        rot = np.zeros((n, 4), F32)
        rot[:, 0] = 1.0
        tail = np.zeros((1, 3))
        out.append(scenes.Scene(
            name="pile", shape_type=np.full(n, scenes.SHAPE_BOX, np.uint32),
            shape_half=np.vstack([h[b], [10.0, 0.5, 10.0]]).astype(F32), pos=np.vstack([pos[b], tail]).astype(F32),
            rot=rot, vel=np.vstack([vel[b], tail]).astype(F32), ang=np.zeros((n, 3), F32),
            mass=np.append(mass[b], 0.0).astype(F32), inertia=inertia, shape=np.arange(n, dtype=np.uint32),
            flags=np.append(np.zeros(m), scenes.FLAG_STATIC).astype(np.uint32),
            bounds=np.array([-15, -2, -15, 15, 30, 15], F32), max_pairs=max(256, 48 * n), max_contacts=max(64, 16 * n)))
    return out


# ---------------------------------------------------------------------------
# State in tensors
# ---------------------------------------------------------------------------
_streams = []


def _stream():
    """The program's one stream."""
    if not _streams:
        _streams.append(capi.Stream())
    return _streams[0]


class TensorBodies:
    """Body arrays as rows of one tensor, in capi.BodyView's layout."""

    def __init__(self, scene):
        inv, inertia, flags = capi.body_dynamics(scene.mass, scene.inertia, scene.flags)
        rows = np.vstack([scene.pos.T, scene.rot.T, scene.vel.T, scene.ang.T, inv[None], inertia.T])
        self.n = scene.n
        self.fields = torch.from_numpy(np.ascontiguousarray(rows, F32)).cuda()
        self.ids = torch.from_numpy(np.stack([scene.shape, flags]).astype(np.int64)).to(torch.int32).cuda()
        self.start = None

    def view(self):
        v = capi.BodyView()
        for i, k in enumerate(capi.BODY_FLOAT_FIELDS):
            setattr(v, k, self.fields[i].data_ptr())
        v.shape, v.flags, v.n = self.ids[0].data_ptr(), self.ids[1].data_ptr(), self.n
        return v

    def state(self):
        return self.fields[:N_STATE]

    def snapshot(self):
        self.start = self.state().clone()

    def reset(self, s):
        """Back to the snapshot, in order on stream s."""
        _copy(self.fields, self.start, s)


def _copy(dst, src, s):
    capi.check(capi.lib().dy_memcpy_d2d_async(capi.vp(dst.data_ptr()), capi.vp(src.data_ptr()),
                                              src.numel() * src.element_size(), s.h), "dy_memcpy_d2d_async")


def _adjoint_view(rows, n):
    """A BodyView whose mutable fields and inverse mass are rows of a (14, n) tensor."""
    v = capi.BodyView()
    for i, k in enumerate(capi.BODY_FLOAT_FIELDS[:N_STATE + 1]):
        setattr(v, k, rows[i].data_ptr() if i < len(rows) else None)
    v.n = n
    return v


def _world(case, seed):
    rng = np.random.default_rng(seed)
    n = case["n"]
    if case.get("scene", "mixed") == "blocks":
        sc = _blocks(n, rng)
    elif case.get("scene") == "chains":
        links = 8 if n >= 64 else 4
        sc = scenes.joint_chains(max(1, n // links), links, seed=seed)
    else:
        sc = _random_mixed(n, rng)
    w = capi.World(sc, _stream())
    w.bodies = TensorBodies(sc)
    torch.cuda.synchronize()
    for _ in range(case["at"]):
        w.step_async()
    w.check()
    w.bodies.snapshot()
    return w, rng


def prepare(case, seed):
    kind = case["kind"]
    if kind == "frame":
        w, _ = _world(case, seed)
        return {"kind": kind, "world": w, "frames": case["frames"], "blocking": case["blocking"]}
    if kind == "rays":
        w, rng = _world(case, seed)
        n, m = w.scene.n, case["rays"]
        capi.integrate(w.s, w.bodies, w.scene.gravity, w.scene.dt, 1)
        w.bp.build_and_query(w.s, w.bodies, w.shapes, w.scene.bounds)
        lo, hi = w.scene.bounds[:3].astype(np.float64), w.scene.bounds[3:].astype(np.float64)
        # sensors on the walls of the scene's bounds, looking at points of the pile
        origin = rng.uniform(lo, hi, (m, 3))
        axis, face = rng.integers(0, 3, m), rng.random(m) < 0.5
        origin[np.arange(m), axis] = np.where(face, lo[axis], hi[axis])
        target = rng.uniform(lo, hi, (m, 3))
        target[:, 1] = rng.uniform(-1.0, 0.4 * hi[1], m)
        d = target - origin
        d /= np.linalg.norm(d, axis=1, keepdims=True)
        rays = np.hstack([origin, d, np.full((m, 1), 2.0 * np.linalg.norm(hi - lo))]).astype(F32)
        bvh = capi.BvhView()
        capi.check(capi.lib().dy_broadphase_bvh_view(w.bp.h, n, C.byref(bvh)), "dy_broadphase_bvh_view")
        w.s.wait()
        return {"kind": kind, "world": w, "bvh": bvh, "rays": torch.from_numpy(rays).cuda(),
                "hits": torch.zeros((m, 2), dtype=torch.int32, device="cuda")}
    if kind == "sort":
        rng = np.random.default_rng(seed)
        n = case["n"]
        keys = torch.from_numpy(rng.integers(0, 1 << 63, n, dtype=np.int64)).cuda()
        vals = torch.arange(n, dtype=torch.int32, device="cuda")
        return {"kind": kind, "s": _stream(), "from": (keys, vals), "to": (keys.clone(), vals.clone())}
    rng = np.random.default_rng(seed)
    if kind == "batch":
        b = capi.Batch(_piles(_counts(case["scenes"], case["median"], 8, case["top"]), rng), _stream())
    elif case["scene"] == "stack":
        g = scenes.Pcg32(seed)
        b = capi.Batch([scenes.diff_stack(g) for _ in range(case["scenes"])], _stream())
    else:
        b = capi.Batch([_random_mixed(int(c), rng, 0.5) for c in
                        _counts(case["scenes"], case["median"], 16, case["top"])], _stream())
    b.bodies = TensorBodies(b.merged)
    torch.cuda.synchronize()
    if case["at"]:
        b.step(case["at"], n_substeps=case.get("substeps", 1))
    b.s.wait()
    b.bodies.snapshot()
    if kind == "batch":
        return {"kind": kind, "batch": b, "frames": case["frames"]}
    d = capi.Diff(b, case["frames"], case["every"], n_substeps=case["substeps"], tape_contacts_per_body=6.0)
    n = b.n_bodies
    # d/dx of a squared distance to targets about half a metre away, and a small weight on the velocities
    final = torch.zeros((N_STATE, n), device="cuda")
    final[:3] = torch.from_numpy(rng.normal(size=(3, n)).astype(F32)).cuda()
    final[7:10] = torch.from_numpy(0.1 * rng.normal(size=(3, n)).astype(F32)).cuda()
    torch.cuda.synchronize()
    return {"kind": kind, "batch": b, "diff": d, "frames": case["frames"], "final": final,
            "initial": torch.zeros((N_STATE + 1, n), device="cuda")}


def run(state):
    kind = state["kind"]
    if kind == "frame":
        w = state["world"]
        w.bodies.reset(w.s)
        for _ in range(state["frames"]):
            if state["blocking"]:
                w.step()
            else:
                w.step_async()
        return w.bodies.state()
    if kind == "batch":
        b = state["batch"]
        b.bodies.reset(b.s)
        b.step(state["frames"])
        return b.bodies.state()
    if kind == "grad":
        b, d = state["batch"], state["diff"]
        b.bodies.reset(b.s)
        d.forward(state["frames"])
        n, g = b.n_bodies, b.scenes[0].gravity
        final, initial = _adjoint_view(state["final"], n), _adjoint_view(state["initial"], n)
        bv, sv = b.bodies.view(), b.shapes.view()
        capi.check(capi.lib().dy_diff_backward(d.h, b.s.h, C.byref(bv), C.byref(sv), g[0], g[1], g[2],
                                               b.scenes[0].dt, C.byref(final), C.byref(initial)), "dy_diff_backward")
        return b.bodies.state(), state["initial"]
    if kind == "rays":
        w, rays, hits = state["world"], state["rays"], state["hits"]
        bv, sv = w.bodies.view(), w.shapes.view()
        capi.check(capi.lib().dy_ray_query(w.s.h, C.byref(state["bvh"]), C.byref(bv), C.byref(sv),
                                           rays.data_ptr(), hits.data_ptr(), len(rays)), "dy_ray_query")
        return hits[:, 0].view(torch.float32), hits[:, 1]
    for dst, src in zip(state["to"], state["from"]):
        _copy(dst, src, state["s"])
    keys, vals = state["to"]
    capi.check(capi.lib().dy_sort_by_key_u64_u32(state["s"].h, keys.data_ptr(), vals.data_ptr(), len(keys)),
               "dy_sort_by_key_u64_u32")
    return state["to"]


def work(case):
    kind = case["kind"]
    if kind == "rays":  # the ray and its hit; the tree's boxes and links and the bodies once; ~40 box and ~4 body tests
        return {"bytes": case["rays"] * 36 + case["n"] * (2 * 32 + 60), "flops": case["rays"] * (40 * 20 + 4 * 120)}
    if kind == "sort":  # key and payload in and out
        return {"bytes": case["n"] * 24, "flops": 0}
    steps = case["frames"] * case.get("substeps", 1)
    bodies = case["n"] if kind == "frame" else case["scenes"] * (case["median"] * (1.3 if case["top"] != case["median"] else 1.0) + 1)
    # A settled pile has about 14 candidate pairs and 4 contacts a body; a pair's test takes about 400 operations
    # and a contact's projection about 500 (only its first does any work).
    flops = bodies * steps * (14 * 400 + 4 * 500 + 150)
    if kind == "grad":  # the record of the forward is not charged: state and adjoint in and out
        return {"bytes": bodies * (88 + 52 + 52 + 56), "flops": 3 * flops}
    # every frame's state exists: a frame of one scene reads a body's 88 bytes and writes 52; a batch's launch does so once
    return {"bytes": bodies * 140 * (case["frames"] if kind == "frame" else 1), "flops": flops}


def tolerance(case):
    if case["kind"] == "grad":
        # The trajectory is exact; the adjoint's sums may be formed in another order, and contact events amplify
        # their roundings: over 30 frames the reverse sweep is within 2.5e-5 of the same trajectory's forward mode.
        return {"rel": 1e-4, "max": 1e-2}
    return "exact"


def exact(case, seed):
    """Hit distances by brute force over all bodies in float64.  Frames and
    gradients have no 64-bit value: a contact that exists at one precision and
    not at the other renumbers the contacts, and with them the solver's order."""
    if case["kind"] != "rays":
        return None
    st = prepare(case, seed)
    w, rays = st["world"], st["rays"].double()
    f, sc = w.bodies.fields.double(), w.scene
    half = torch.from_numpy(sc.shape_half[sc.shape].astype(np.float64)).cuda()
    sphere = torch.from_numpy(sc.shape_type[sc.shape] == scenes.SHAPE_SPHERE).cuda()
    pos, q, u = f[0:3].T, f[3], -f[4:7].T

    def turn(v):  # by the conjugate of each body's orientation
        t = 2.0 * torch.cross(u.expand_as(v), v, dim=-1)
        return v + t * q[:, None] + torch.cross(u.expand_as(t), t, dim=-1)

    best = []
    step = max(1, 4_000_000 // sc.n)
    for k in range(0, len(rays), step):
        o, d, far = rays[k:k + step, None, 0:3], rays[k:k + step, None, 3:6], rays[k:k + step, 6]
        oc = o - pos
        a, b = (d * d).sum(-1), (d * oc).sum(-1)
        disc = b * b - a * ((oc * oc).sum(-1) - half[:, 0] ** 2)
        root = disc.clamp(min=0).sqrt()
        near = (-b - root) / a
        ts = torch.where(near < 0, (-b + root) / a, near)
        ts = torch.where((disc >= 0) & (ts >= 0), ts, torch.inf)
        lo, ld = turn(oc), turn(d.expand_as(oc))
        t1, t2 = (-half - lo) / ld, (half - lo) / ld
        tmin, tmax = torch.minimum(t1, t2).amax(-1), torch.maximum(t1, t2).amin(-1)
        tb = torch.where(tmin >= 0, tmin, tmax)
        tb = torch.where((tmax >= 0) & (tmin <= tmax), tb, torch.inf)
        t = torch.where(sphere, ts, tb).amin(-1)
        best.append(torch.where(t < far, t, far))
    return torch.cat(best), None
