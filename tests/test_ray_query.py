"""Ray queries over the LBVH (core/src/ray_query.cpp, core/include/core/ray_query.hpp).

CPU: the oracle against the reference's known answers
(core/tests/ray_query_test.cpp:44-181) and against a brute force over all
bodies (the closest exact hit among bodies whose binary16 leaf box the ray
enters); GPU: dy_ray_query bit for bit against the oracle.
"""
import ctypes
import dataclasses

import numpy as np
import pytest

from dyphur_amd import scenes

F32 = np.float32
NO_HIT = 0xFFFFFFFF


def _ray(o, d, t_max=1e9):
    return np.array(list(o) + list(d) + [t_max], F32)


def _two(shape, half, pa, pb, bounds):
    sc = scenes.two_body(shape, shape, half, half, pa, pb)
    sc.bounds = np.array(bounds, F32)
    return sc


KATS = [
    # (scene, rays, expected (body, t) per ray; t None for a miss)
    ("sphere_x", lambda: _two(1, (1, 1, 1), (0, 0, 0), (0, 50, 0), (-6, -6, -6, 56, 56, 56)),
     [_ray((-5, 0, 0), (1, 0, 0)), _ray((-5, 3, 0), (1, 0, 0))], [(0, 4.0), (NO_HIT, None)]),
    ("box_x", lambda: _two(0, (1, 1, 1), (0, 0, 0), (0, 50, 0), (-6, -6, -6, 56, 56, 56)),
     [_ray((-5, 0, 0), (1, 0, 0)), _ray((-5, 2, 0), (1, 0, 0))], [(0, 4.0), (NO_HIT, None)]),
    ("closest_of_two", lambda: _two(1, (1, 1, 1), (0, 0, 0), (10, 0, 0), (-6, -6, -6, 16, 6, 6)),
     [_ray((-5, 0, 0), (1, 0, 0))], [(0, 4.0)]),
    ("t_max", lambda: _two(1, (1, 1, 1), (0, 0, 0), (50, 0, 0), (-6, -6, -6, 56, 6, 6)),
     [_ray((-5, 0, 0), (1, 0, 0), 2.0)], [(NO_HIT, None)]),
]


def _oracle_query(oracle, sc, rays):
    b, s = oracle.Bodies(sc), oracle.Shapes(sc)
    w = oracle.World.for_scene(sc)
    w.build_and_query(b, s, sc.bounds)
    return w.ray_query(b, s, sc.n, np.stack(rays)), w, b, s


@pytest.mark.parametrize("case", [k[0] for k in KATS])
def test_oracle_ray_query_reference_answers(oracle, case):
    name, mk, rays, want = next(k for k in KATS if k[0] == case)
    (t, body), *_ = _oracle_query(oracle, mk(), rays)
    for i, (wb, wt) in enumerate(want):
        assert body[i] == wb
        if wt is not None:
            assert abs(t[i] - wt) <= 1e-3


def _slab(o, inv, mn, mx):
    t1, t2 = (mn - o) * inv, (mx - o) * inv
    lo, hi = np.minimum(t1, t2), np.maximum(t1, t2)
    return lo.max(-1), hi.min(-1)


def _brute(sc, st, aabb16, sorted_idx, ray):
    """Closest exact hit among all bodies whose binary16 leaf box the ray
    enters before t_max, in float32 with the reference's operation order."""
    n = sc.n
    o, d, t_max = ray[:3], ray[3:6], ray[6]
    with np.errstate(divide="ignore", invalid="ignore", over="ignore"):
        inv = F32(1) / d
        box = aabb16[n - 1:, :6].copy().view(np.float16).astype(F32)
        lo, hi = _slab(o, inv, box[:, :3], box[:, 3:])
        enter = (hi >= 0) & (hi >= lo) & (lo < t_max)
        best_t, best = t_max, NO_HIT
        for leaf in np.nonzero(enter)[0]:
            i = int(sorted_idx[leaf])
            shp = int(sc.shape[i])
            p = np.array([st["pos_x"][i], st["pos_y"][i], st["pos_z"][i]], F32)
            h = sc.shape_half[shp].astype(F32)
            if sc.shape_type[shp] == scenes.SHAPE_SPHERE:
                oc = o - p
                a = F32(d[0] * d[0] + d[1] * d[1] + d[2] * d[2])
                b = F32(d[0] * oc[0] + d[1] * oc[1] + d[2] * oc[2])
                c = F32(F32(oc[0] * oc[0] + oc[1] * oc[1] + oc[2] * oc[2]) - h[0] * h[0])
                disc = F32(b * b - a * c)
                if disc < 0:
                    continue
                sq = np.sqrt(disc)
                t = F32((-b - sq) / a)
                if t < 0:
                    t = F32((-b + sq) / a)
            else:
                qw, qx, qy, qz = (F32(st[k][i]) for k in ("rot_w", "rot_x", "rot_y", "rot_z"))
                u = np.array([-qx, -qy, -qz], F32)

                def rot(v):
                    tv = np.array([u[1] * v[2] - u[2] * v[1], u[2] * v[0] - u[0] * v[2],
                                   u[0] * v[1] - u[1] * v[0]], F32) * F32(2)
                    return (v + tv * qw) + np.array([u[1] * tv[2] - u[2] * tv[1], u[2] * tv[0] - u[0] * tv[2],
                                                     u[0] * tv[1] - u[1] * tv[0]], F32)

                lo_, ld = rot((o - p).astype(F32)), rot(d.astype(F32))
                il = F32(1) / ld
                t1, t2 = (-h - lo_) * il, (h - lo_) * il
                tmin, tmax = np.minimum(t1, t2).max(), np.maximum(t1, t2).min()
                if tmax < 0 or tmin > tmax:
                    continue
                t = tmin if tmin >= 0 else tmax
            if 0 <= t < best_t:
                best_t, best = F32(t), i
    return best_t, best


def test_oracle_ray_query_equals_brute_force(oracle):
    sc = scenes.random_mixed(800, seed=17, extent=(10, 6, 10))
    rng = np.random.default_rng(3)
    rays = []
    for _ in range(300):
        o = rng.uniform([-8, 0, -8], [8, 12, 8])
        tgt = rng.uniform([-5, 1, -5], [5, 7, 5])
        rays.append(_ray(o, (tgt - o) / np.linalg.norm(tgt - o), rng.uniform(3, 30)))
    (t, body), w, b, s = _oracle_query(oracle, sc, rays)
    bvh = w.bvh(sc.n)
    st = b.state()
    hits = 0
    for k, r in enumerate(rays):
        bt, bb = _brute(sc, st, bvh["aabb"], bvh["sorted_idx"], r)
        assert body[k] == bb, k
        assert t[k].view(np.uint32) == F32(bt).view(np.uint32), k
        hits += bb != NO_HIT
    assert hits > 100


@pytest.mark.gpu
@pytest.mark.parametrize("case", [k[0] for k in KATS] + ["mixed_3000"])
def test_gpu_ray_query_bitexact(gpu, oracle, case):
    if case == "mixed_3000":
        sc = scenes.random_mixed(3000, seed=11, extent=(12, 10, 12))
        rng = np.random.default_rng(8)
        rays = []
        for _ in range(20000):
            o = rng.uniform([-10, 0, -10], [10, 14, 10])
            tgt = rng.uniform([-6, 1, -6], [6, 10, 6])
            rays.append(_ray(o, tgt - o, rng.uniform(0.5, 3.0)))
    else:
        _, mk, rays, _ = next(k for k in KATS if k[0] == case)
        sc = mk()
    print(f"[ray] {case} n={sc.n} rays={len(rays)}", flush=True)
    (t_ref, b_ref), *_ = _oracle_query(oracle, sc, rays)
    s = gpu.Stream()
    db = gpu.DeviceBodies(sc, s)
    ds = gpu.DeviceShapes(sc, s)
    bp = gpu.Broadphase(s, sc.n, sc.max_pairs)
    bp.build_and_query(s, db, ds, sc.bounds)
    t, body = gpu.ray_query(s, bp, sc.n, db, ds, np.stack(rays))
    assert np.array_equal(body, b_ref)
    assert np.array_equal(t.view(np.uint32), t_ref.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("n,m,moved,axis", [(2, 40, False, False), (3, 4096, False, True), (300, 4095, True, False),
                                            (300, 4096, True, True), (1500, 20000, True, False),
                                            (20000, 1200, True, False), (2000, 5000, False, True)])
def test_gpu_ray_query_teams_bitexact(gpu, oracle, n, m, moved, axis):
    """Rays walked by teams, from the view's arrays and from records: bodies
    that moved since the tree was built (hits before their box), rays along the
    axes and from the boxes' own planes (slab distances that are no number),
    long rays through many bodies and every t_max."""
    rng = np.random.default_rng(n + m)
    side = 1.2 * n ** (1 / 3)
    sc = scenes.random_mixed(n - 1, seed=5, extent=(side, side, side))
    print(f"[ray teams] n={n} rays={m} moved={moved} axis={axis}", flush=True)
    o = rng.uniform(-side, side, (m, 3))
    d = rng.uniform(-side, side, (m, 3)) + [0, side / 2, 0] - o
    if axis:
        keep = rng.integers(0, 3, m)
        sign = np.where(rng.random(m) < 0.5, 1.0, -1.0)
        d = np.zeros((m, 3))
        d[np.arange(m), keep] = sign
        o[: m // 2] = np.round(o[: m // 2] * 4) / 4
    t_max = rng.choice([0.5, 3.0, 50.0, np.inf], m)
    rays = np.hstack([o, d, t_max[:, None]]).astype(F32)
    (_, _), w, b, osh = _oracle_query(oracle, sc, list(rays[:1]))
    s = gpu.Stream()
    db = gpu.DeviceBodies(sc, s)
    ds = gpu.DeviceShapes(sc, s)
    bp = gpu.Broadphase(s, sc.n, sc.max_pairs)
    bp.build_and_query(s, db, ds, sc.bounds)
    if moved:
        shift = rng.uniform(-0.3, 0.3, (3, sc.n)).astype(F32)
        for k, f in enumerate(("pos_x", "pos_y", "pos_z")):
            v = (db.download(s)[f] + shift[k]).astype(F32)
            db.f[f].upload(v, s)
            b.arr[f][:] = v
    t_ref, b_ref = w.ray_query(b, osh, sc.n, rays)
    t, body = gpu.ray_query(s, bp, sc.n, db, ds, rays)
    assert np.array_equal(body, b_ref)
    assert np.array_equal(t.view(np.uint32), t_ref.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("n,m,axis", [(1, 300, False), (4, 700, True), (5, 2749, False), (5, 2750, True),
                                      (119, 65450, True), (300, 93530, False), (300, 93531, False)])
def test_gpu_ray_query_lanes_bitexact(gpu, oracle, n, m, axis):
    """Many rays over few bodies go one a lane: both sides of the lines between
    lanes and teams, with and without rays along the axes."""
    rng = np.random.default_rng(n + m)
    side = 1.2 * n ** (1 / 3) + 1.0
    sc = scenes.random_mixed(max(n - 1, 1), seed=6, extent=(side, side, side))
    if n == 1:
        sc = dataclasses.replace(sc, **{k: getattr(sc, k)[:1] for k in ("pos", "rot", "vel", "ang", "mass", "inertia",
                                                                        "shape", "flags")})
    print(f"[ray lanes] n={sc.n} rays={m} axis={axis}", flush=True)
    o = rng.uniform(-side, side, (m, 3))
    d = rng.uniform(-side, side, (m, 3)) + [0, side / 2, 0] - o
    if axis:
        keep = rng.integers(0, 3, m)
        d = np.zeros((m, 3))
        d[np.arange(m), keep] = np.where(rng.random(m) < 0.5, 1.0, -1.0)
        o[: m // 2] = np.round(o[: m // 2] * 4) / 4
    t_max = rng.choice([0.5, 3.0, 50.0, np.inf], m)
    rays = np.hstack([o, d, t_max[:, None]]).astype(F32)
    (t_ref, b_ref), _, _, _ = _oracle_query(oracle, sc, list(rays))
    s = gpu.Stream()
    db = gpu.DeviceBodies(sc, s)
    ds = gpu.DeviceShapes(sc, s)
    bp = gpu.Broadphase(s, sc.n, sc.max_pairs)
    bp.build_and_query(s, db, ds, sc.bounds)
    t, body = gpu.ray_query(s, bp, sc.n, db, ds, rays)
    assert np.array_equal(body, b_ref)
    assert np.array_equal(t.view(np.uint32), t_ref.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("n,m", [(20000, 2**28 + 5), (40, 2**27 + 3)])
def test_gpu_ray_query_more_rays_than_one_grid(gpu, n, m):
    """More rays than one launch's grid can take (teams from 2^28 rays on, and
    the first run's end among the lanes): every ray has its own hit."""
    side = 1.2 * n ** (1 / 3)
    sc = scenes.random_mixed(n - 1, seed=5, extent=(side, side, side))
    print(f"[rays past one grid] n={sc.n} rays={m}", flush=True)
    s = gpu.Stream()
    db, ds = gpu.DeviceBodies(sc, s), gpu.DeviceShapes(sc, s)
    bp = gpu.Broadphase(s, sc.n, sc.max_pairs)
    bp.build_and_query(s, db, ds, sc.bounds)
    rng = np.random.default_rng(2)
    some = 4093
    o = rng.uniform(-side, side, (some, 3))
    d = rng.uniform(-side, side, (some, 3)) - o
    few = np.hstack([o, d, np.full((some, 1), 2.0)]).astype(F32)
    t, body = gpu.ray_query(s, bp, sc.n, db, ds, few)
    want = np.stack([t.view(np.uint32), body], 1)
    rays = gpu.DeviceArray(7 * m, F32)
    rays.upload(few.ravel(), s, 7 * some)
    have = some
    while have < m:  # the same rays again and again
        more = min(have, m - have)
        gpu.check(gpu.lib().dy_memcpy_d2d_async(gpu.vp(rays.ptr + 28 * have), gpu.vp(rays.ptr), 28 * more, s.h), "copy")
        have += more
    hits = gpu.DeviceArray(2 * m, np.uint32)
    bvh = gpu.BvhView()
    gpu.check(gpu.lib().dy_broadphase_bvh_view(bp.h, sc.n, ctypes.byref(bvh)), "view")
    bv, sv = db.view(), ds.view()
    gpu.check(gpu.lib().dy_ray_query(s.h, ctypes.byref(bvh), ctypes.byref(bv), ctypes.byref(sv), rays.ptr, hits.ptr, m),
              "dy_ray_query")
    for k in range(0, m, 4096 * some):
        part = min(4096 * some, m - k)
        got = gpu.download_ptr(hits.ptr + 8 * k, 2 * part, np.uint32, s).reshape(part, 2)
        whole = part // some * some
        assert np.all(got[:whole].reshape(-1, some, 2) == want), k
        assert np.array_equal(got[whole:], want[: part - whole]), k
    rays.free()
    hits.free()


@pytest.mark.gpu
@pytest.mark.parametrize("n,m", [(200, 4000), (2000, 20000), (4, 4000)])
def test_gpu_ray_query_not_finite(gpu, oracle, n, m):
    """Directions, origins and t_max that are infinite, zero or no number, and
    bodies whose binary16 boxes are infinite: teams from the view's arrays and
    from records, and lanes."""
    rng = np.random.default_rng(n + m)
    side = 1.2 * n ** (1 / 3) + 1.0
    sc = scenes.random_mixed(n - 1, seed=8, extent=(side, side, side))
    sc.pos[::3, 0] += F32(1e5)  # past 65 504
    sc.pos[1::7, 1] -= F32(2e5)
    print(f"[ray not finite] n={sc.n} rays={m}", flush=True)
    o = rng.uniform(-side, side, (m, 3))
    target = sc.pos[rng.integers(0, sc.n, m)].astype(np.float64)
    d = (target - o) * rng.choice([1.0, 1e-3], (m, 1))
    odd = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1e-40, 3e38])
    pick = rng.random((m, 3)) < 0.35
    d = np.where(pick, odd[rng.integers(0, len(odd), (m, 3))], d)
    far = np.array([np.inf, -np.inf, np.nan, 1e5, 3.4e38, 0.0])
    pick = rng.random((m, 3)) < 0.05
    o = np.where(pick, far[rng.integers(0, len(far), (m, 3))], o)
    t_max = rng.choice([0.0, -1.0, 1.0, 50.0, 3e38, np.inf, -np.inf, np.nan], m, p=[.05, .05, .1, .2, .2, .3, .05, .05])
    rays = np.hstack([o, d, t_max[:, None]]).astype(F32)
    (t_ref, b_ref), *_ = _oracle_query(oracle, sc, list(rays))
    s = gpu.Stream()
    db, ds = gpu.DeviceBodies(sc, s), gpu.DeviceShapes(sc, s)
    bp = gpu.Broadphase(s, sc.n, sc.max_pairs)
    bp.build_and_query(s, db, ds, sc.bounds)
    t, body = gpu.ray_query(s, bp, sc.n, db, ds, rays)
    assert np.array_equal(body, b_ref)
    same = t.view(np.uint32) == t_ref.view(np.uint32)
    assert np.all(same | (np.isnan(t) & np.isnan(t_ref)))


@pytest.mark.gpu
@pytest.mark.parametrize("n,m", [(2000, 5000), (90, 60000)])
def test_gpu_ray_query_captured(gpu, n, m):
    """A captured query (teams without records, lanes) replays to the eager
    result, with eager work and moved bodies between the replays."""
    rng = np.random.default_rng(n)
    side = 1.2 * n ** (1 / 3)
    sc = scenes.random_mixed(n - 1, seed=9, extent=(side, side, side))
    print(f"[ray captured] n={sc.n} rays={m}", flush=True)
    o = rng.uniform(-side, side, (m, 3))
    rays = np.hstack([o, rng.uniform(-side, side, (m, 3)) - o, np.full((m, 1), 3.0)]).astype(F32)
    s = gpu.Stream()
    db, ds = gpu.DeviceBodies(sc, s), gpu.DeviceShapes(sc, s)
    bp = gpu.Broadphase(s, sc.n, sc.max_pairs)
    bp.build_and_query(s, db, ds, sc.bounds)
    d_rays = gpu.DeviceArray.from_numpy(rays.ravel(), s)
    d_hits = gpu.DeviceArray(2 * m, np.uint32)
    bvh = gpu.BvhView()
    gpu.check(gpu.lib().dy_broadphase_bvh_view(bp.h, sc.n, ctypes.byref(bvh)), "view")
    bv, sv = db.view(), ds.view()
    with gpu.Graph.capture(s) as g:
        gpu.check(gpu.lib().dy_ray_query(s.h, ctypes.byref(bvh), ctypes.byref(bv), ctypes.byref(sv), d_rays.ptr,
                                         d_hits.ptr, m), "dy_ray_query")
    for _ in range(4):
        db.f["pos_x"].upload(sc.pos[:, 0] + rng.uniform(-0.2, 0.2, sc.n).astype(F32), s)
        t, body = gpu.ray_query(s, bp, sc.n, db, ds, rays)
        d_hits.upload(np.zeros(2 * m, np.uint32), s)
        g.launch(s)
        got = d_hits.download(s).reshape(m, 2)
        assert np.array_equal(got[:, 1], body) and np.array_equal(got[:, 0], t.view(np.uint32))


class _SmallPool:
    """The device's stream-ordered allocations from a pool of at most `size`
    bytes while it is open."""

    class Props(ctypes.Structure):  # hipMemPoolProps
        _fields_ = [("alloc_type", ctypes.c_int), ("handle_types", ctypes.c_int), ("location_type", ctypes.c_int),
                    ("location_id", ctypes.c_int), ("security", ctypes.c_void_p), ("max_size", ctypes.c_size_t),
                    ("reserved", ctypes.c_ubyte * 56)]

    def __init__(self, hip, size):
        self.hip = hip  # a library that the runtime's own entry points are found through
        self.size, self.pool, self.old = size, ctypes.c_void_p(), ctypes.c_void_p()

    def __enter__(self):
        p = self.Props(alloc_type=1, location_type=1, max_size=self.size)
        assert self.hip.hipDeviceGetMemPool(ctypes.byref(self.old), 0) == 0
        assert self.hip.hipMemPoolCreate(ctypes.byref(self.pool), ctypes.byref(p)) == 0
        assert self.hip.hipDeviceSetMemPool(0, self.pool) == 0
        return self

    def take(self, size, s):
        """What an allocation of `size` bytes on stream s returns."""
        q = ctypes.c_void_p()
        st = self.hip.hipMallocAsync(ctypes.byref(q), ctypes.c_size_t(size), s.h)
        if st == 0:
            assert self.hip.hipFreeAsync(q, s.h) == 0
        self.hip.hipGetLastError()
        return st

    def __exit__(self, *exc):
        assert self.hip.hipDeviceSetMemPool(0, self.old) == 0
        assert self.hip.hipDeviceSynchronize() == 0
        assert self.hip.hipMemPoolDestroy(self.pool) == 0


@pytest.mark.gpu
def test_gpu_ray_query_without_room_for_records(gpu, oracle):
    """A call whose scratch allocation fails walks the view's arrays instead."""
    n, m = 20000, 5000
    side = 1.2 * n ** (1 / 3)
    sc = scenes.random_mixed(n - 1, seed=5, extent=(side, side, side))
    print(f"[rays without records] n={sc.n} rays={m}", flush=True)
    rng = np.random.default_rng(4)
    o = rng.uniform(-side, side, (m, 3))
    rays = np.hstack([o, rng.uniform(-side, side, (m, 3)) - o, np.full((m, 1), 2.0)]).astype(F32)
    (t_ref, b_ref), *_ = _oracle_query(oracle, sc, list(rays))
    s = gpu.Stream()
    db, ds = gpu.DeviceBodies(sc, s), gpu.DeviceShapes(sc, s)
    bp = gpu.Broadphase(s, sc.n, sc.max_pairs)
    bp.build_and_query(s, db, ds, sc.bounds)
    s.wait()
    with _SmallPool(gpu.lib(), 1 << 16) as pool:
        assert pool.take(80 * n, s) != 0
        t, body = gpu.ray_query(s, bp, sc.n, db, ds, rays)
    assert np.array_equal(body, b_ref)
    assert np.array_equal(t.view(np.uint32), t_ref.view(np.uint32))
