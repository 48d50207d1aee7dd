"""GPU tests of what the library refuses and what it may hold: scene depth,
bad geometry, device memory budgets and kept device blocks."""
import ctypes as C
import os
import threading

import numpy as np
import pytest

import orc
import vlb

pytestmark = pytest.mark.gpu


def _concentric(n):
    """n triangles of growing size around one centre, all of one Morton code:
    each one's least union is with its next smaller neighbour, so one pair
    merges per clustering pass and the tree is a chain of depth n - 1."""
    s = 1.0 + np.arange(n) * 1e-3
    z = np.zeros(n)
    v = np.stack([np.stack([-s, -s, z], 1), np.stack([s, -s, z], 1), np.stack([z, s, z], 1)], 1)
    return v.reshape(-1, 3).astype(np.float32), np.arange(3 * n, dtype=np.uint32).reshape(n, 3)


@pytest.mark.parametrize("n", [4096, 4097, 4098, 4099, 10_000])
def test_trees_beyond_the_depth_limit_are_refused(ctx, n):
    """Depth 4096 is the limit: at it a scene answers as the oracle does,
    beyond it the upload is refused, also where the tree is several times as
    deep, and the context goes on."""
    xyz, idx = _concentric(n)
    if n - 1 > 4096:
        with pytest.raises(vlb.VlbError) as e:
            ctx.upload_scene(xyz, idx)
        assert e.value.status == vlb.ERR_INVALID
        small, sidx = _concentric(100)
        sid = ctx.upload_scene(small, sidx)
        assert ctx.scene_info(sid)["depth"] == 99
        ctx.release_scene(sid)
        return
    sid = ctx.upload_scene(xyz, idx)
    assert ctx.scene_info(sid)["depth"] == n - 1
    rng = np.random.default_rng(n)
    m = 1000
    org = np.zeros((m, 3), np.float32)
    org[:, :2] = rng.uniform(-5, 5, (m, 2))
    org[:, 2] = rng.choice([-1.0, 1.0], m)
    d = np.zeros((m, 3), np.float32)
    d[:, :2] = rng.uniform(-0.3, 0.3, (m, 2))
    d[:, 2] = -org[:, 2]
    got = ctx.trace_closest(sid, org, d, 0.0, 10.0)
    ref = orc.Scene(xyz, idx, bvh=False).trace_closest(org, d, 0.0, 10.0, brute=True)
    assert (ref[0] >= 0).any() and (ref[0] < 0).any()
    assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1])
    ctx.release_scene(sid)


def _free_bytes():
    """Free memory of the device, as the driver sees it."""
    free, total = C.c_size_t(), C.c_size_t()
    assert vlb.lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _plans(c, sid, n, rays):
    """n plans that hold 12 * 1024 * rays bytes of radiance each."""
    probes = np.random.default_rng(1).uniform(-1, 1, (1024, 3)).astype(np.float32)
    p = vlb.Params(probes=probes, rays=rays)
    return [c.plan(sid, p) for _ in range(n)]


def _fill(c):
    """16 MiB blocks until the budget refuses one."""
    fill = []
    with pytest.raises(vlb.VlbError) as e:
        while True:
            fill.append(c.alloc(16 << 20))
    assert e.value.status == vlb.ERR_BUDGET
    return fill


def test_reused_blocks_stay_within_the_budget():
    """Blocks kept from larger buffers: a context filled to its budget through
    them is given as much as one that kept none, and holds no more of the
    device than the budget (and what hipMalloc rounds up to: at most 2 MiB for
    each buffer of a mebibyte or more)."""
    budget, room = 1200 << 20, []
    for kept in (False, True):
        with vlb.Context(hbm_budget=budget) as c:
            sid = c.upload_scene(np.zeros((0, 3), np.float32), np.zeros((0, 3), np.uint32))
            small = _plans(c, sid, 1, 64)
            small[0].execute()
            small[0].download()
            before = _free_bytes()
            for pl in _plans(c, sid, 8 if kept else 0, 8192):  # 8 x 96 MiB
                pl.destroy()
            plans = _plans(c, sid, 8, 6720)                    # 8 x 79 MiB
            fill = _fill(c)
            assert before - _free_bytes() <= budget + (48 << 20)
            room.append(len(fill))
            for d in fill:
                c.free(d)
            for pl in plans + small:
                pl.destroy()
    assert room[0] == room[1] > 0


def test_oldest_kept_blocks_go_first():
    """More freed than a context keeps (1/32 of the device): the blocks freed
    last stay, not only the one that went over."""
    total = C.c_size_t()
    assert vlb.lib.hipMemGetInfo(C.byref(C.c_size_t()), C.byref(total)) == 0
    limit = total.value // 32
    with vlb.Context() as c:
        sid = c.upload_scene(np.zeros((0, 3), np.float32), np.zeros((0, 3), np.uint32))
        size = []
        for share in (0.55, 0.25, 0.35):
            rays = int(share * limit) // (12 * 1024 * 64) * 64
            size.append(12 * 1024 * rays)
            _plans(c, sid, 1, rays)[0].destroy()
        held = _free_bytes()
    kept = _free_bytes() - held
    assert size[1] + size[2] <= kept <= limit + (64 << 20)


def test_kept_blocks_are_given_back():
    """What a context keeps is the device's again after trim(), and is no
    reason for another context of the process to run out of memory."""
    with vlb.Context() as c, vlb.Context(hbm_budget=1 << 50) as other:
        sid = c.upload_scene(np.zeros((0, 3), np.float32), np.zeros((0, 3), np.uint32))
        rays, p = 131072, vlb.Params(probes=np.zeros((8, 3), np.float32), rays=64)
        want = c.bake(sid, p)
        before = _free_bytes()
        _plans(c, sid, 1, rays)[0].destroy()                  # 1.5 GiB
        assert before - _free_bytes() >= 12 * 1024 * rays
        c.trim()
        assert before - _free_bytes() <= 64 << 20
        _plans(c, sid, 1, rays)[0].destroy()
        d = other.alloc(_free_bytes() + (512 << 20))          # a third of what is kept
        other.free(d)
        assert np.array_equal(c.bake(sid, p), want)


@pytest.mark.parametrize("size", [(1 << 64) - 1, (1 << 64) - 4096, (1 << 64) - (3 << 20), 1 << 63])
def test_requests_near_the_size_limit_are_refused(ctx, size):
    """Sizes whose rounding to a capacity, or sum with what is in use, wraps."""
    d = ctx.alloc(4096)
    with pytest.raises(vlb.VlbError) as e:
        ctx.alloc(size)
    assert e.value.status in (vlb.ERR_BUDGET, vlb.ERR_OOM)
    ctx.free(d)


def test_refused_uploads_leave_nothing_behind(ctx):
    """Uploads refused for a bad index: the process does not grow.  (An event
    of the HIP runtime, the smallest thing a call could leave, takes over 200
    bytes of host memory.)"""
    v, idx = np.zeros((3, 3), np.float32), np.array([[0, 1, 3]], np.uint32)

    def refused(n):
        for _ in range(n):
            with pytest.raises(vlb.VlbError):
                ctx.upload_scene(v, idx)
        with open("/proc/self/statm") as f:
            return int(f.read().split()[1]) * os.sysconf("SC_PAGESIZE")

    before = refused(1000)
    assert refused(5000) - before < 5000 * 200


def test_bad_geometry_is_named_where_it_does_not_fit():
    """Geometry beyond the budget: refused for its first bad index, else its
    first bad coordinate, else for the budget."""
    n = 100_000
    v = np.random.default_rng(0).uniform(-1, 1, (3 * n, 3)).astype(np.float32)
    idx = np.arange(3 * n, dtype=np.uint32).reshape(n, 3)
    with vlb.Context(hbm_budget=1 << 20) as c:
        with pytest.raises(vlb.VlbError) as e:
            c.upload_scene(v, idx)
        assert e.value.status == vlb.ERR_BUDGET
        v[70_000, 1] = np.nan
        with pytest.raises(vlb.VlbError, match="coordinate .* at 210001$") as e:
            c.upload_scene(v, idx)
        assert e.value.status == vlb.ERR_INVALID
        idx[50_000, 2] = 3 * n
        with pytest.raises(vlb.VlbError, match="index out of range at 150002$") as e:
            c.upload_scene(v, idx)
        assert e.value.status == vlb.ERR_INVALID


@pytest.mark.parametrize("prec,per_ray", [(vlb.PREC_FP32, 84), (vlb.PREC_BF16, 84), (vlb.PREC_BF16_FAST, 52)])
def test_served_direction_sets_fit_a_budget_of_their_tables(prec, per_ray):
    """A request with a new direction set, served with no more of the budget
    left than its tables take (16 bytes of direction, 4 of index and the basis
    row of each ray): it is served, with the coefficients of a bake."""
    R = 1 << 16                                   # whole slices: no padding rays
    s = vlb.generate_scene(vlb.SCENE_ROOM, 2)
    probes = np.random.default_rng(2).uniform([1, 0.5, 1], [9, 3.5, 9], (20, 3)).astype(np.float32)
    p = vlb.Params(probes=probes, rays=R, precision=prec, lights=[(vlb.LIGHT_DIRECTIONAL, (0.2, -1.0, 0.1), (3.0, 3.0, 3.0))])
    with vlb.Context() as c:
        srv = vlb.Server(c, state_budget=1 << 22, step_rays=1 << 16, max_active=4, precision=prec)
        want = srv.wait(srv.submit(c.upload_scene_dict(s), p))
        srv.destroy()
    with vlb.Context(hbm_budget=256 << 20) as c:
        sid = c.upload_scene_dict(s)
        srv = vlb.Server(c, state_budget=1 << 22, step_rays=1 << 16, max_active=4, precision=prec)
        tables = c.alloc(per_ray * R)
        fill = []
        for size in (16 << 20, 1 << 20, 1 << 16, 1 << 12):
            try:
                while True:
                    fill.append(c.alloc(size))
            except vlb.VlbError as e:
                assert e.status == vlb.ERR_BUDGET
        c.free(tables)                            # room for them and at most 4095 bytes
        got = srv.wait(srv.submit(sid, p))
        srv.destroy()
        for d in fill:
            c.free(d)
    assert np.array_equal(got[0], want[0])


def test_blocks_given_back_while_others_work():
    """trim() in a loop beside bakes, a server and another context's bakes:
    everyone's results are those of a quiet run."""
    s = vlb.generate_scene(vlb.SCENE_ROOM, 2)
    rng = np.random.default_rng(9)
    sets = [rng.uniform([1, 0.5, 1], [9, 3.5, 9], (n, 3)).astype(np.float32) for n in (30, 200, 500)]
    prm = [vlb.Params(probes=q, rays=640, rays_per_slice=640) for q in sets]
    with vlb.Context() as c, vlb.Context() as other:
        sid, oid = c.upload_scene_dict(s), other.upload_scene_dict(s)
        want = [c.bake(sid, p) for p in prm]
        errors, stop = [], threading.Event()

        def run(f):
            try:
                f()
            except BaseException as e:  # reported by the main thread
                errors.append(e)

        def bakes(ctx, sid):
            for _ in range(15):
                for p, w in zip(prm, want):
                    assert np.array_equal(ctx.bake(sid, p), w)

        def serves():
            for _ in range(3):
                srv = vlb.Server(c, step_rays=1 << 15, state_budget=1 << 24)
                ids = [srv.submit(sid, p) for p in prm * 3]
                got = [srv.wait(i)[0] for i in ids]
                srv.destroy()
                assert all(np.array_equal(g, w) for g, w in zip(got, want * 3))

        def trims():
            while not stop.is_set():
                c.trim()
                other.trim()

        work = [threading.Thread(target=run, args=(f,)) for f in
                (lambda: bakes(c, sid), lambda: bakes(other, oid), serves)]
        trimmer = threading.Thread(target=run, args=(trims,))
        for t in work + [trimmer]:
            t.start()
        for t in work:
            t.join()
        stop.set()
        trimmer.join()
    assert not errors, errors


def test_a_new_context_counts_kept_blocks_as_free():
    """The default budget is the device's free memory: what another context
    keeps of it is not missing there."""
    with vlb.Context() as c:
        sid = c.upload_scene(np.zeros((0, 3), np.float32), np.zeros((0, 3), np.uint32))
        _plans(c, sid, 1, 131072)[0].destroy()                # 1.5 GiB kept
        with vlb.Context() as other:
            other.free(other.alloc(_free_bytes() + (512 << 20)))
