"""Class assignment: every body's thread in lock step with its partners, on one
XCD (few bodies) and over the chip, with one body a thread and several."""
import numpy as np
import pytest

from dyphur_amd import scenes

pytestmark = pytest.mark.gpu


def _jp_order(n):
    """Contacts 0 .. n - 1 by falling priority."""
    k = np.arange(n, dtype=np.uint64)
    h = k.astype(np.uint32)
    h ^= h >> np.uint32(16)
    h *= np.uint32(0x85EBCA6B)
    h ^= h >> np.uint32(13)
    h *= np.uint32(0xC2B2AE35)
    h ^= h >> np.uint32(16)
    return np.argsort((h.astype(np.uint64) << np.uint64(32)) | k)[::-1]


def _greedy(a, b, static, serial):
    """Classes by definition: in priority order (JP) the lowest colour free on
    both bodies, in index order one more than the bodies' levels."""
    order = np.arange(len(a)) if serial else _jp_order(len(a))
    used = [0] * len(static)
    out = np.zeros(len(a), np.uint32)
    for c in order:
        ends = [x for x in (a[c], b[c]) if not static[x]]
        if serial:
            out[c] = max([used[x] for x in ends], default=0)
            for x in ends:
                used[x] = int(out[c]) + 1
        else:
            m = 0
            for x in ends:
                m |= used[x]
            out[c] = (~m & (m + 1)).bit_length() - 1
            for x in ends:
                used[x] |= 1 << int(out[c])
    return out


def _contacts(n, nc):
    """Random contacts over n bodies, a tenth of them static, grouped by the
    first body as the broadphase lists them."""
    rng = np.random.default_rng(n + nc)
    a = np.sort(rng.integers(0, n, nc)).astype(np.uint32)
    b = ((a + rng.integers(1, n, nc)) % n).astype(np.uint32)
    static = rng.random(n) < 0.1
    sc = scenes.random_mixed(n - 1, seed=1, extent=(40, 40, 40))
    sc.mass = np.where(static, 0.0, np.maximum(sc.mass, 1.0)).astype(np.float32)
    sc.flags = np.where(static, scenes.FLAG_STATIC, 0).astype(np.uint32)
    return a, b, static, sc


def _view(gpu, s, a, b, fields):
    names = ("body_a", "body_b", "pos_x", "pos_y", "pos_z", "norm_x", "norm_y", "norm_z", "depth")
    arrays = [gpu.DeviceArray.from_numpy(np.ascontiguousarray(v), s) for v in (a, b, *fields)]
    arrays.append(gpu.DeviceArray.from_numpy(np.array([len(a)], np.uint32), s))
    cv = gpu.ContactView()
    for name, arr in zip(names, arrays):
        setattr(cv, name, arr.ptr)
    cv.n, cv.capacity = arrays[-1].ptr, len(a)
    return cv, arrays


@pytest.mark.parametrize("n,nc,blocks,serial", [
    (64, 250, 0, False), (64, 257, 0, False), (1000, 3000, 0, False), (1000, 3000, 1, False), (1000, 900, 0, True),
    (16384, 40001, 0, False), (16385, 40001, 0, False), (16385, 20000, 3, False), (16385, 9000, 2, True),
])
def test_classes_match_greedy(gpu, monkeypatch, n, nc, blocks, serial):
    """Random contacts over n bodies (a tenth static; contacts between two
    static bodies among them): both sides of the one-XCD line, of the
    256-contact line, and with several bodies a thread."""
    if blocks:
        monkeypatch.setenv("DYPHUR_ASSIGN_BLOCKS", str(blocks))
    print(f"[assign] n={n} nc={nc} blocks={blocks} serial={serial}", flush=True)
    s = gpu.Stream()
    a, b, static, sc = _contacts(n, nc)
    db = gpu.DeviceBodies(sc, s)
    solver = gpu.XpbdSolver(s, 2, nc, 0.5)
    solver.set_force_serial(serial)
    z = np.zeros(nc, np.float32)
    cv, _keep = _view(gpu, s, a, b, [z] * 7)
    solver.solve(s, cv, db, sc.dt)
    st = solver.stats()
    used_serial = serial or nc <= 256
    ref = _greedy(a, b, static, used_serial)
    assert bool(st["used_serial"]) == used_serial
    assert st["n_constraints"] == nc and st["n_classes"] == ref.max() + 1
    assert np.array_equal(solver.classes(s, nc), ref)


@pytest.mark.parametrize("n,nc,blocks", [(1000, 3000, 0), (16385, 40001, 0), (16385, 20000, 3), (30000, 20000, 0)])
@pytest.mark.parametrize("kind", ["overflow", "deep"])
def test_fallback_to_reference_order(gpu, monkeypatch, n, nc, blocks, kind):
    """A body in more than 64 contacts that can see each other's colours, and a
    chain of 300 rounds: the assignment ranks its lists again in contact order
    inside the launch, on one XCD and over the chip, with one body a thread and
    several."""
    if blocks:
        monkeypatch.setenv("DYPHUR_ASSIGN_BLOCKS", str(blocks))
    print(f"[assign fallback] {kind} n={n} nc={nc} blocks={blocks}", flush=True)
    a, b, static, sc = _contacts(n, nc)
    free = np.nonzero(~static)[0]
    if kind == "overflow":
        hub = free[len(free) // 2]
        at = np.arange(0, nc, nc // 150)
        a[at], b[at] = hub, free[: len(at)]
        a[at[b[at] == hub]] = free[-1]
    else:
        at = _jp_order(nc)[:300]  # contact at[k] waits for at[k - 1]
        chain = free[-301:]
        used = np.isin(a, chain) | np.isin(b, chain)
        a[used], b[used] = free[0], free[1]
        a[at], b[at] = chain[:-1], chain[1:]
    s = gpu.Stream()
    db = gpu.DeviceBodies(sc, s)
    solver = gpu.XpbdSolver(s, 2, nc, 0.5)
    z = np.zeros(nc, np.float32)
    cv, _keep = _view(gpu, s, a, b, [z] * 7)
    ref = _greedy(a, b, static, True)
    for _ in range(2):
        solver.solve(s, cv, db, sc.dt)
        st = solver.stats()
        assert st["used_serial"] == 1 and st["overflow"] == (1 if kind == "overflow" else st["overflow"])
        assert st["n_constraints"] == nc and st["n_classes"] == ref.max() + 1
        assert np.array_equal(solver.classes(s, nc), ref)


@pytest.mark.parametrize("heavy", [False, True])
@pytest.mark.parametrize("n,nc,iters,blocks", [
    (40, 33, 10, 0), (300, 257, 1, 0), (300, 900, 10, 1), (16384, 40001, 3, 0), (16385, 40001, 3, 0), (16385, 40001, 2, 2),
    (24576, 60001, 3, 0), (24577, 60001, 3, 0), (24577, 40001, 2, 2),
])
def test_first_iteration_by_words_matches_records(gpu, monkeypatch, n, nc, iters, blocks, heavy):
    """The sweep that hands bodies on as tagged words against the sweep over
    acknowledged records, bit for bit.  Contacts between bodies of almost no
    inverse mass stay live after the first iteration, so the later ones run
    (test_later_iterations_by_words has such contacts move)."""
    if blocks:
        monkeypatch.setenv("DYPHUR_SWEEP_BLOCKS", str(blocks))
    rng = np.random.default_rng(7)
    a, b, static, sc = _contacts(n, nc)
    if heavy:
        big = (rng.random(n) < 0.3) & ~static
        sc.mass[big] = 1e13
        sc.inertia[np.ix_(big, [0, 4, 8])] = 1e13
    normal = rng.normal(size=(3, nc))
    normal /= np.linalg.norm(normal, axis=0)
    depth = rng.uniform(-0.01, 0.05, nc)
    at = sc.pos[a].T + rng.uniform(-0.3, 0.3, (3, nc))
    fields = [v.astype(np.float32) for v in (*at, *normal, depth)]
    got = []
    for pair in ("1", "0"):
        monkeypatch.setenv("DYPHUR_SWEEP_PAIR", pair)
        print(f"[words] n={n} nc={nc} iters={iters} blocks={blocks} heavy={heavy} pair={pair}", flush=True)
        s = gpu.Stream()
        db = gpu.DeviceBodies(sc, s)
        solver = gpu.XpbdSolver(s, iters, nc, 0.5)
        cv, _keep = _view(gpu, s, a, b, fields)
        for _ in range(2):
            solver.solve(s, cv, db, sc.dt)
        assert solver.stats()["n_constraints"] == nc
        got.append(db.download(s))
    for k in got[0]:
        assert np.array_equal(np.asarray(got[0][k]).view(np.uint32), np.asarray(got[1][k]).view(np.uint32)), k


def _plates(n):
    """n - 1 dynamic bodies over one static one, six contacts each with it, that
    stay live after the first iteration: their inertia about z and their mass
    are so large that a contact which pushes along their plane (a third of them)
    cannot move them until another one has turned the plane."""
    rng = np.random.default_rng(n)
    sc = scenes.random_mixed(n - 1, seed=2, extent=(40, 40, 40))
    sc.mass = np.where(np.arange(n) < n - 1, 1e13, 0.0).astype(np.float32)
    sc.flags = np.where(np.arange(n) < n - 1, 0, scenes.FLAG_STATIC).astype(np.uint32)
    sc.rot[:] = 1.0, 0.0, 0.0, 0.0
    sc.inertia[:] = 0.0
    sc.inertia[:, [0, 4, 8]] = 1.0, 1.0, 1e13
    a = np.repeat(np.arange(n - 1), 6)
    nc = len(a)
    b = np.full(nc, n - 1)
    turn = rng.random(nc) < 2 / 3
    angle = rng.uniform(0, 2 * np.pi, nc)
    normal = np.where(turn, [[0.0]] * 2 + [[1.0]], [np.cos(angle), np.sin(angle), 0.0 * angle])
    arm = rng.uniform(0.2, 0.5, (3, nc)) * [[1], [1], [0]]
    return sc, a, b, [v.astype(np.float32) for v in (*(sc.pos[a].T + arm), *normal, rng.uniform(0.01, 0.05, nc))]


def _solved(gpu, sc, a, b, fields, iters, solves=1):
    s = gpu.Stream()
    db = gpu.DeviceBodies(sc, s)
    solver = gpu.XpbdSolver(s, iters, len(a), 0.5)
    cv, _keep = _view(gpu, s, a.astype(np.uint32), b.astype(np.uint32), fields)
    for _ in range(solves):
        solver.solve(s, cv, db, sc.dt)
    assert solver.stats()["n_constraints"] == len(a)
    return db.download(s)


def _same_bits(x, y):
    return all(np.array_equal(np.asarray(x[k]).view(np.uint32), np.asarray(y[k]).view(np.uint32)) for k in x)


@pytest.mark.parametrize("n", [60, 3000, 24600])
@pytest.mark.parametrize("refuse", [1, 4, 8])
def test_refused_launches_change_nothing(gpu, monkeypatch, n, refuse):
    """A refused launch of the assignment (1), the first iteration (4) or the
    later ones (8), in the solve that meets it and in the next one, with
    contacts that only the later iterations move."""
    print(f"[refused] n={n} refuse={refuse}", flush=True)
    sc, a, b, fields = _plates(n)
    first = _solved(gpu, sc, a, b, fields, 1)
    want = _solved(gpu, sc, a, b, fields, 4, 2)
    once = _solved(gpu, sc, a, b, fields, 4)
    assert np.max(np.abs(first["rot_w"] - once["rot_w"])) > 1e-4  # the later iterations matter
    monkeypatch.setenv("DYPHUR_REFUSE_LAUNCH", str(refuse))
    assert _same_bits(_solved(gpu, sc, a, b, fields, 4), once)
    assert _same_bits(_solved(gpu, sc, a, b, fields, 4, 2), want)


@pytest.mark.parametrize("threads", [128, 256, 1024])
def test_pair_threads_launch_as_asked(gpu, monkeypatch, threads):
    """Every accepted DYPHUR_SWEEP_PAIR_THREADS launches: a refused one would
    leave the solver to launches per round and per class with the host between
    them, which take more than ten times as long."""
    n, nc = 5000, 15000
    a, b, _, sc = _contacts(n, nc)
    rng = np.random.default_rng(1)
    normal = rng.normal(size=(3, nc))
    normal /= np.linalg.norm(normal, axis=0)
    fields = [v.astype(np.float32) for v in (*sc.pos[a].T, *normal, rng.uniform(0.0, 0.01, nc))]
    ms = []
    for t in (512, threads):
        monkeypatch.setenv("DYPHUR_SWEEP_PAIR_THREADS", str(t))
        print(f"[pair threads] {t}", flush=True)
        s = gpu.Stream()
        db = gpu.DeviceBodies(sc, s)
        solver = gpu.XpbdSolver(s, 10, nc, 0.5)
        cv, _keep = _view(gpu, s, a, b, fields)
        solver.solve(s, cv, db, sc.dt)
        solver.set_timing(True)
        for _ in range(10):
            solver.solve(s, cv, db, sc.dt)
        tm = solver.timing(s)
        ms.append((tm["assign_ms"] + tm["sweep_ms"]) / tm["solves"])
    assert ms[1] < 4.0 * ms[0], ms


@pytest.mark.parametrize("n,nc,serial", [(50, 100, False), (1000, 3000, False), (1000, 3000, True), (16400, 30000, False)])
def test_contact_of_a_body_with_itself_is_an_error_at_once(gpu, n, nc, serial):
    """No list order lets such a contact go first; the solve reports it without
    waiting for the kernels' limits, and leaves the bodies where they were."""
    import time
    print(f"[self contact] n={n} nc={nc} serial={serial}", flush=True)
    a, b, static, sc = _contacts(n, nc)
    k = int(np.nonzero(~static[a])[0][nc // 3])
    b[k] = a[k]
    z = np.zeros(nc, np.float32)
    s = gpu.Stream()
    db = gpu.DeviceBodies(sc, s)
    solver = gpu.XpbdSolver(s, 3, nc, 0.5)
    solver.set_force_serial(serial)
    cv, _keep = _view(gpu, s, a, b, [z] * 6 + [z + np.float32(0.01)])
    before = db.download(s)
    t0 = time.perf_counter()
    solver.solve(s, cv, db, sc.dt)
    with pytest.raises(gpu.DyError):
        solver.stats()
    assert time.perf_counter() - t0 < 0.5
    after = db.download(s)
    for f in ("pos_x", "pos_y", "pos_z", "vel_x", "vel_y", "vel_z"):
        assert np.array_equal(before[f], after[f]), f


def test_two_large_worlds_on_two_streams(gpu):
    """Two worlds of 26 000 bodies step side by side, each on its own stream:
    the kernels whose workgroups wait for each other leave room for another
    world's, and both worlds go as they go alone."""
    scs = [scenes.random_mixed(26000, seed=k, extent=(26, 26, 26)) for k in (3, 4)]
    frames = 12
    alone = []
    for sc in scs:
        w = gpu.World(sc)
        for _ in range(frames):
            w.step_async()
        w.check()
        alone.append(w.fnv())
    print("[two worlds] side by side", flush=True)
    worlds = [gpu.World(sc) for sc in scs]
    for _ in range(frames):
        for w in worlds:
            w.step_async()
    for w in worlds:
        w.check()
    assert [w.fnv() for w in worlds] == alone


def test_solver_memory_per_contact(gpu):
    """A solver takes 156 bytes a contact; the launches per round take 36 more
    only when a solve needs them."""
    import ctypes
    free, total = ctypes.c_size_t(), ctypes.c_size_t()

    def left():
        assert gpu.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    s = gpu.Stream()
    gpu.XpbdSolver(s, 2, 1000, 0.5).close()
    n = 16 << 20
    before = left()
    solver = gpu.XpbdSolver(s, 2, n, 0.5)
    took = before - left()
    solver.close()
    print(f"[solver memory] {took / n:.1f} bytes a contact", flush=True)
    assert 150 * n < took < 162 * n


@pytest.mark.parametrize("n,iters", [(60, 2), (3000, 4), (24600, 3)])
def test_later_iterations_by_words(gpu, monkeypatch, n, iters):
    """Contacts that the first iteration leaves live and the later ones move:
    the records made from the words, against the sweep over records."""
    print(f"[later iterations] n={n} iters={iters}", flush=True)
    sc, a, b, fields = _plates(n)
    first = _solved(gpu, sc, a, b, fields, 1)
    got = _solved(gpu, sc, a, b, fields, iters, 2)
    once = _solved(gpu, sc, a, b, fields, iters)
    assert np.max(np.abs(first["rot_w"] - once["rot_w"])) > 1e-4
    monkeypatch.setenv("DYPHUR_SWEEP_PAIR", "0")
    assert _same_bits(_solved(gpu, sc, a, b, fields, iters, 2), got)


def test_timing_charges_the_iterations_that_ran(gpu):
    """Ten iterations of which nine have nothing to do count as one, and all
    count where contacts stay live."""
    for sc, a, b, fields, iters, ran in [
            (lambda c: (c[3], c[0], c[1], [np.zeros(900, np.float32)] * 7))(_contacts(300, 900)) + (10, 1),
            _plates(60) + (4, 4)]:
        print(f"[sweep bytes] nc={len(a)} iters={iters}", flush=True)
        s = gpu.Stream()
        db = gpu.DeviceBodies(sc, s)
        solver = gpu.XpbdSolver(s, iters, len(a), 0.5)
        cv, _keep = _view(gpu, s, np.asarray(a, np.uint32), np.asarray(b, np.uint32), fields)
        solver.set_timing(True)
        solver.solve(s, cv, db, sc.dt)
        tm, st = solver.timing(s), solver.stats()
        once = 44.0 * st["n_constraints"] + 132.0 * st["dyn_endpoints"] + 32.0 * sc.n
        assert tm["solves"] == 1 and tm["sweep_bytes"] == ran * once
