"""GPU tests of the launch paths picked by size or option: each path against
the same work on the path it stands in for, or against the oracle."""
import threading

import numpy as np
import pytest

import orc
import vlb
from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def room(ctx):
    s = vlb.generate_scene(vlb.SCENE_ROOM, 2)
    sid = ctx.upload_scene_dict(s)
    yield s, sid, orc.Scene.from_dict(s)
    ctx.release_scene(sid)


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


@pytest.mark.parametrize("cnt", [(3, 2, 3), (1, 1, 1)])
def test_indirect_occupancy_bounds_agree(ctx, room, cnt):
    """The multi-bounce kernel at every occupancy bound (trace_variant 4: none,
    8: 6 waves/SIMD, 12: 8): the same coefficients bit for bit, and within 1e-5
    of the FP64 oracle (the bar of every FP32 bake)."""
    s, sid, o = room
    probes, step = vlb.probe_grid([1.5, 1.0, 1.5], [8.5, 3.0, 8.5], list(cnt))
    step = np.where(np.isfinite(step) & (step != 0), step, 1.0)
    g = vlb.grid_desc([1.5, 1.0, 1.5], step, cnt, num_coefs=9)
    sun = vlb.sun_direction(np.random.default_rng(7))
    lights = [(vlb.LIGHT_DIRECTIONAL, (-sun).tolist(), (3.0, 2.5, 2.0)),
              (vlb.LIGHT_POINT, (5.0, 2.0, 5.0), (20.0, 20.0, 20.0))]
    lp = vlb.lookup_params(vlb.LOOKUP_IRRADIANCE, True, 2e-3)
    src = np.random.default_rng(1).normal(size=(len(probes), 9, 3)).astype(np.float32)
    got = {}
    for v in (4, 8, 12):
        p = vlb.Params(probes=probes, rays=333, lights=lights, sun_dir=sun.tolist(), trace_variant=v)
        plan = ctx.plan(sid, p)
        plan.set_indirect(g, lp, 0.75, coeffs=src)
        plan.execute()
        got[v] = plan.download()
        plan.destroy()
    assert np.array_equal(_bits(got[4]), _bits(got[12])) and np.array_equal(_bits(got[4]), _bits(got[8]))
    ref = o.bake_indirect(p, g, src, lp, 0.75, mode64=True)["coeffs"]
    assert rel_err(got[12], ref).max() <= 1e-5


@pytest.mark.parametrize("scale", [1e-12, 1.0, 1e12])
@pytest.mark.parametrize("ntris", [1, 2, 3, 4, 5, 9, 64])
def test_small_trees_at_extreme_scales(ctx, ntris, scale):
    """Trees of every child count (unused slots, leaf-only and mixed nodes) at
    scales where the node unit is far from 1, with rays along the axes (zero
    direction components) and from far outside: hit ids and distances are the
    oracle's exactly, as for every scene."""
    rng = np.random.default_rng(ntris)
    tri = rng.uniform(-1, 1, (ntris, 1, 3)) + rng.uniform(-0.7, 0.7, (ntris, 3, 3))
    tri[::3, :, 1] = np.round(tri[::3, :1, 1])          # flat ones, some coplanar
    xyz = (tri.reshape(-1, 3) * scale).astype(np.float32)
    idx = np.arange(len(xyz), dtype=np.uint32).reshape(-1, 3)
    n = 3000
    target = rng.uniform(-1, 1, (n, 3))
    d = rng.normal(size=(n, 3))
    d[: n // 3] = np.eye(3)[rng.integers(0, 3, n // 3)] * rng.choice([-1.0, 1.0], (n // 3, 1))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    dist = np.where(np.arange(n) % 2, 0.7, 30.0)[:, None]
    org = ((target - d * dist) * scale).astype(np.float32)
    d = d.astype(np.float32)
    tmax = np.float32(100.0 * scale)
    alb = np.ones((ntris, 3), np.float32)
    sid = ctx.upload_scene(xyz, idx, None, alb)
    o = orc.Scene(xyz, idx, None, alb)
    got = ctx.trace_closest(sid, org, d, 0.0, tmax)
    ref = o.trace_closest(org, d, 0.0, tmax)
    assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1])
    assert (ref[0] >= 0).any()
    occ = ctx.trace_occluded(sid, org, d, tmax, 0.0)
    assert np.array_equal(occ, o.trace_occluded(org, d, np.full(n, tmax, np.float32), 0.0))
    ctx.release_scene(sid)


def test_probes_on_walls_agree_across_kernels(ctx, room):
    """Rays that run in the plane of a wall (probes on the scene bounds, an
    equirect grid with columns along the axes): the check that decides those
    hits gives the same bits in every kernel family, with point queries on the
    same rays in agreement."""
    s, sid, o = room
    probes, _ = vlb.probe_grid([0, 0, 0], [10, 4, 10], [3, 2, 3], vlb.ORDER_REFERENCE_BFS)
    p = vlb.Params(probes=probes, dir_mode=vlb.DIRS_EQUIRECT, equirect_w=157, equirect_h=50, sh_order=3,
                   sh_constants=vlb.SH_LITERAL, shade_mode=vlb.SHADE_REFERENCE)
    ref = None
    for v in (12, 4, 16, 20, 36):
        p.trace_variant = v
        got = ctx.bake(sid, p)
        ref = got if ref is None else ref
        assert np.array_equal(_bits(got), _bits(ref)), v
    p.trace_variant = 0
    _, hits = ctx.bake_radiance(sid, p, want_radiance=False)
    xyz, _ = vlb.directions(p.dir_mode, 0, 157, 50)
    for i in (0, 5, 17):
        prim = ctx.trace_closest(sid, np.repeat(probes[i:i + 1], len(xyz), 0), xyz)[0]
        assert np.array_equal(prim, hits[i])


@pytest.mark.parametrize("mode,n", [("fib", 1), ("fib", 63), ("fib", 1000), ("fib", 16384), ("eq", (7, 3)),
                                    ("eq", (64, 32)), ("eq", (157, 50))])
@pytest.mark.parametrize("prec", [vlb.PREC_FP32, vlb.PREC_BF16, vlb.PREC_FP16])
def test_device_ray_tables_project_like_the_oracle(ctx, mode, n, prec):
    """The direction and basis tables built on the device, through a sky-only
    bake: every ray's radiance is a function of its direction (so a wrong
    direction, order or weight shows), and the coefficients are the FP64
    oracle's within the bar of the precision (1e-5, split 16-bit forms 1e-4)."""
    sid = ctx.upload_scene(np.zeros((0, 3), np.float32), np.zeros((0, 3), np.uint32))
    o = orc.Scene(np.zeros((0, 3)), np.zeros((0, 3), np.uint32))
    probes = np.zeros((3, 3), np.float32)
    sun = vlb.sun_direction(np.random.default_rng(3)).tolist()
    if mode == "fib":
        p = vlb.Params(probes=probes, rays=n, sun_dir=sun, precision=prec, sh_order=3)
    else:
        p = vlb.Params(probes=probes, dir_mode=vlb.DIRS_EQUIRECT, equirect_w=n[0], equirect_h=n[1],
                       sun_dir=sun, precision=prec, sh_order=3, sh_constants=vlb.SH_LITERAL)
    rad, hit = ctx.bake_radiance(sid, p)
    assert (hit == -1).all()
    xyz, _ = vlb.directions(p.dir_mode, p.rays, p.equirect_w, p.equirect_h)
    d = xyz.astype(np.float64)
    want = 0.5 + 1.5 * np.maximum(d[:, 1], 0.0) + 50.0 * np.exp(200.0 * (d @ np.asarray(sun) - 1.0))
    np.testing.assert_allclose(rad[0, :, 0], want, rtol=3e-5)
    got = ctx.bake(sid, p)
    ref = o.bake(p, mode64=True)["coeffs"]
    assert rel_err(got, ref).max() <= (1e-5 if prec == vlb.PREC_FP32 else 1e-4)
    ctx.release_scene(sid)


@pytest.mark.parametrize("P", [1, 15, 16, 17, 1000, 20000])
def test_device_probe_order_keeps_every_probe(ctx, room, P):
    """Probes sorted on the device come back in the caller's order: each
    probe's coefficients are those of a bake of that probe alone."""
    s, sid, o = room
    rng = np.random.default_rng(P)
    probes = rng.uniform([1, 0.5, 1], [9, 3.5, 9], (P, 3)).astype(np.float32)
    if P > 16:
        probes[5:9] = probes[4]                        # equal keys: a stable order
    p = vlb.Params(probes=probes, rays=64, lights=[(vlb.LIGHT_DIRECTIONAL, (0.0, -1.0, 0.0), (3.0, 3.0, 3.0))])
    got = ctx.bake(sid, p)
    for i in rng.integers(0, P, 4):
        p.probes = probes[i:i + 1]
        assert rel_err(ctx.bake(sid, p), got[i:i + 1]).max() <= 1e-6


def _mixed_calls(c, sid, probes):
    """One-shot calls of different buffer sizes: their results in a fixed order."""
    sun = [(vlb.LIGHT_DIRECTIONAL, (0.2, -1.0, 0.1), (3.0, 3.0, 3.0))]
    rng = np.random.default_rng(len(probes))
    res = []
    for rays, order in ((48, 2), (700, 3), (129, 2)):
        res.append(c.bake(sid, vlb.Params(probes=probes, rays=rays, sh_order=order, lights=sun)))
    d = rng.normal(size=(777, 3)).astype(np.float32)
    o = np.tile(probes[:1], (777, 1))
    res += list(c.trace_closest(sid, o, d))
    res.append(c.project_equirect(rng.integers(0, 256, (40, 80, 4), dtype=np.uint8)))
    return res


@pytest.mark.parametrize("budget", [0, 64 << 20])
def test_reused_device_blocks_hold_nothing_over(budget):
    """Calls whose buffers are blocks freed by other calls (larger, smaller,
    from two threads at once; with a budget that some of the kept blocks have
    to make room for) return what the first call on a fresh context returns."""
    s = vlb.generate_scene(vlb.SCENE_ROOM, 2)
    rng = np.random.default_rng(5)
    sets = [rng.uniform([1, 0.5, 1], [9, 3.5, 9], (n, 3)).astype(np.float32) for n in (300, 37)]
    want = []
    for p in sets:
        with vlb.Context() as c:
            want.append(_mixed_calls(c, c.upload_scene_dict(s), p))
    with vlb.Context(hbm_budget=budget) as c:
        sid = c.upload_scene_dict(s)
        errors = []

        def work(k):
            try:
                for _ in range(3):
                    got = _mixed_calls(c, sid, sets[k])
                    assert all(np.array_equal(a, b) for a, b in zip(got, want[k]))
            except BaseException as e:  # reported by the main thread
                errors.append(e)

        ts = [threading.Thread(target=work, args=(k,)) for k in (0, 1)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert not errors, errors
        c.release_scene(sid)
        again = c.upload_scene_dict(s)  # a scene built in kept blocks
        got = _mixed_calls(c, again, sets[0])
        assert all(np.array_equal(a, b) for a, b in zip(got, want[0]))


@pytest.mark.parametrize("layout", ["scattered", "coincident", "line"])
@pytest.mark.parametrize("n", [1, 2, 255, 257, 960, 1024, 1025, 1920, 1921, 3000])
def test_exported_tree_is_whole_at_the_pass_boundaries(ctx, n, layout):
    """Triangle counts around the sizes where the clustering passes change
    (one launch to 256 clusters, 960 per block of the windowed passes, 1024):
    every leaf once, every box the exact union of its triangles, the depth
    that of the longest path."""
    rng = np.random.default_rng(n)
    v = rng.uniform(-1, 1, (n, 3, 3)).astype(np.float32)
    if layout == "coincident":
        v[:] = v[0]
    if layout == "line":
        v *= np.float32(0.01)
        v[..., 0] += np.arange(n, dtype=np.float32)[:, None]
    sid = ctx.upload_scene(v.reshape(-1, 3), np.arange(3 * n, dtype=np.uint32).reshape(n, 3))
    nodes, leaf = ctx.export_bvh(sid)
    info = ctx.scene_info(sid)
    ctx.release_scene(sid)
    assert sorted(leaf) == list(range(n))
    tlo, thi = v.min(1), v.max(1)
    kids = nodes.view(np.int32)[:, 12:14]
    boxes = [(nodes[:, 0:3], nodes[:, 3:6]), (nodes[:, 6:9], nodes[:, 9:12])]
    seen = np.zeros(n, int)
    ulo, uhi, height = {}, {}, {}
    order, stack = [], [0]
    while stack:                       # parents before children
        k = stack.pop()
        order.append(k)
        stack += [c for c in kids[k] if c >= 0]
    assert len(order) == len(set(order)) == len(nodes) == max(1, n - 1)
    for k in reversed(order):
        lo, hi, h = [], [], 0
        for side, c in enumerate(kids[k]):
            if c < 0:
                seen[~c] += 1
                l, u = tlo[leaf[~c]], thi[leaf[~c]]
            else:
                l, u, h = ulo[c], uhi[c], max(h, height[c])
            assert np.array_equal(boxes[side][0][k], l) and np.array_equal(boxes[side][1][k], u)
            lo.append(l)
            hi.append(u)
        ulo[k], uhi[k], height[k] = np.minimum(*lo), np.maximum(*hi), h + 1
    assert (seen == (2 if n == 1 else 1)).all()
    assert info["depth"] == height[0]


def test_exported_tree_of_many_blocks_is_whole(ctx):
    """1.6M triangles: more clustering blocks than one block adds up the counts
    of.  Every leaf and inner node is a child once, and every child's box is
    the union of its own two."""
    n = 1_600_000
    rng = np.random.default_rng(1)
    v = rng.uniform(-1, 1, (n, 1, 3)).astype(np.float32) + rng.uniform(-.01, .01, (n, 3, 3)).astype(np.float32)
    sid = ctx.upload_scene(v.reshape(-1, 3), np.arange(3 * n, dtype=np.uint32).reshape(n, 3))
    nodes, leaf = ctx.export_bvh(sid)
    ctx.release_scene(sid)
    kids = nodes.view(np.int32)[:, 12:14].T.reshape(-1).astype(np.int64)
    lo = np.concatenate([nodes[:, 0:3], nodes[:, 6:9]])
    hi = np.concatenate([nodes[:, 3:6], nodes[:, 9:12]])
    assert np.array_equal(np.sort(kids), np.r_[np.arange(-n, 0), np.arange(1, n - 1)])
    assert np.array_equal(np.sort(leaf), np.arange(n))
    inner = kids >= 0
    c = kids[inner]
    assert np.array_equal(lo[inner], np.minimum(nodes[c, 0:3], nodes[c, 6:9]))
    assert np.array_equal(hi[inner], np.maximum(nodes[c, 3:6], nodes[c, 9:12]))
    prim = leaf[~kids[~inner]]
    assert np.array_equal(lo[~inner], v.min(1)[prim]) and np.array_equal(hi[~inner], v.max(1)[prim])


@pytest.mark.parametrize("n", [1, 255, 257, 300_001])
def test_first_bad_index_or_coordinate_is_named(ctx, n):
    """Geometry checked on the device: the first bad index is reported, before
    any bad coordinate; coordinates of unused vertices count; 2^100 passes."""
    rng = np.random.default_rng(n)
    v = rng.uniform(-1, 1, (3 * n + 2, 3)).astype(np.float32)
    idx = np.arange(3 * n, dtype=np.uint32).reshape(n, 3)
    good = v.copy()
    good[-1] = 2.0 ** 100
    ctx.release_scene(ctx.upload_scene(good, idx))
    for bad in (np.nan, np.inf, np.float32(1.5) * np.float32(2.0 ** 100)):
        w = v.copy()
        w[-1, 1] = bad
        w[-1, 2] = np.nan
        with pytest.raises(vlb.VlbError, match=f"coordinate .* at {w.size - 2}$"):
            ctx.upload_scene(w, idx)
    w = v.copy()
    w[0, 0] = np.nan
    j = idx.copy()
    j[n // 2:, 1] = len(v)
    with pytest.raises(vlb.VlbError, match=f"index out of range at {3 * (n // 2) + 1}$"):
        ctx.upload_scene(w, j)
    assert ctx.scene_info(ctx.upload_scene(v, idx))["num_tris"] == n


@pytest.mark.parametrize("P,R", [(1, 1), (1, 33), (16, 32), (17, 95), (64, 1024), (64, 1056), (256, 1024), (257, 1024), (500, 2049), (1500, 4096)])
def test_work_fetch_covers_every_ray(ctx, room, P, R):
    """Launches from one trace tile to more rounds than waves, through the
    fused kernel (small launches with fewer workgroups) and the wavefront
    kernels (work taken by their own counters): the same bits."""
    s, sid, o = room
    probes = np.random.default_rng(P + R).uniform([1, 0.5, 1], [9, 3.5, 9], (P, 3)).astype(np.float32)
    lights = [(vlb.LIGHT_DIRECTIONAL, (0.3, -1.0, 0.2), (3.0, 2.0, 1.0))]
    got = [ctx.bake(sid, vlb.Params(probes=probes, rays=R, lights=lights, trace_variant=v))
           for v in (0, 4, 12, 36, 13)]
    for g in got[1:]:
        assert np.array_equal(_bits(g), _bits(got[0]))
