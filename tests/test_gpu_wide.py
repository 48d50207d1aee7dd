"""GPU tests of scenes of 2^26 triangles and more, whose nodes and triangles
need 64-bit byte offsets: kernels of their own, at every occupancy and shadow
order, alone and mixed with smaller scenes."""
import numpy as np
import pytest

import vlb

pytestmark = pytest.mark.gpu

FILL = (1 << 26) + (1 << 24)


@pytest.fixture(scope="module")
def scenes():
    """The room, and the room behind 2^26 + 2^24 triangles that no ray reaches
    (beyond every t_max): its own leaves lie past 4 GiB, and it bakes the same
    bits."""
    s = vlb.generate_scene(vlb.SCENE_ROOM, 2)
    xyz, idx = np.asarray(s["xyz"], np.float32).reshape(-1, 3), np.asarray(s["idx"], np.uint32).reshape(-1, 3)
    far = np.float32(-3e4) + np.float32([[0, 0, 0], [1, 0, 0], [0, 1, 0]])
    big = np.empty((FILL + len(idx), 3), np.uint32)
    big[:FILL] = [0, 1, 2]
    big[FILL:] = idx + 3
    with vlb.Context() as c:
        narrow = c.upload_scene(xyz, idx)
        wide = c.upload_scene(np.concatenate([far, xyz]), big)
        del big
        assert c.scene_info(wide)["num_tris"] > 1 << 26
        yield c, narrow, wide
        c.release_scene(wide)
        c.release_scene(narrow)


def _params(seed, P=70, R=500, **kw):
    probes = np.random.default_rng(seed).uniform([1, 0.5, 1], [9, 3.5, 9], (P, 3)).astype(np.float32)
    lights = [(vlb.LIGHT_DIRECTIONAL, (0.3, -1.0, 0.2), (3.0, 2.0, 1.0)), (vlb.LIGHT_POINT, (5.0, 3.0, 5.0), (9.0, 9.0, 9.0))]
    return vlb.Params(probes=probes, rays=R, lights=lights, rays_per_slice=256, **kw)


def _same(a, b):
    return np.array_equal(np.ascontiguousarray(a).view(np.uint32), np.ascontiguousarray(b).view(np.uint32))


@pytest.mark.parametrize("variant", [0, 4, 8, 12, 28, 32, 36, 16])
def test_bakes(scenes, variant):
    c, narrow, wide = scenes
    p = _params(1, trace_variant=variant)
    assert _same(c.bake(wide, p), c.bake(narrow, p))


@pytest.mark.parametrize("variant", [4, 8, 12])
def test_indirect(scenes, variant):
    c, narrow, wide = scenes
    probes, step = vlb.probe_grid([1.5, 1.0, 1.5], [8.5, 3.0, 8.5], [3, 2, 3])
    g = vlb.grid_desc([1.5, 1.0, 1.5], step, [3, 2, 3], num_coefs=9)
    lp = vlb.lookup_params(vlb.LOOKUP_IRRADIANCE, True, 2e-3)
    src = np.random.default_rng(1).normal(size=(len(probes), 9, 3)).astype(np.float32)
    p = _params(2, trace_variant=variant)
    p.probes = probes
    got = []
    for sid in (narrow, wide):
        pl = c.plan(sid, p)
        pl.set_indirect(g, lp, 0.75, coeffs=src)
        pl.execute()
        got.append(pl.download())
        pl.destroy()
    assert _same(got[0], got[1])


def test_queries_radiance_and_counts(scenes):
    c, narrow, wide = scenes
    rng = np.random.default_rng(3)
    org = rng.uniform([1, 0.5, 1], [9, 3.5, 9], (3000, 3)).astype(np.float32)
    d = rng.normal(size=(3000, 3)).astype(np.float32)
    a, b = c.trace_closest(narrow, org, d), c.trace_closest(wide, org, d)
    assert np.array_equal(np.where(a[0] >= 0, a[0] + FILL, -1), b[0]) and (b[0] >= 1 << 26).any()
    assert all(_same(x, y) for x, y in zip(a[1:], b[1:]))
    assert np.array_equal(c.trace_occluded(narrow, org, d, 5.0), c.trace_occluded(wide, org, d, 5.0))
    p = _params(3)
    ra, rb = c.bake_radiance(narrow, p), c.bake_radiance(wide, p)
    assert _same(ra[0], rb[0])
    assert np.array_equal(np.where(ra[1] >= 0, ra[1] + FILL, -1), rb[1])


@pytest.mark.parametrize("variant", [4, 8, 12, 28, 32, 36, 16])
def test_batches_mix_both(scenes, variant):
    """Rounds of one job each, and all jobs in one round."""
    c, narrow, wide = scenes
    jobs = [(narrow, 10), (wide, 11), (narrow, 12), (wide, 13)]
    want = [c.bake(narrow, _params(seed)) for _, seed in jobs]
    for rounds in (1 << 16, 1 << 28):
        b = c.batch([(sid, _params(seed)) for sid, seed in jobs], max_round_rays=rounds, trace_variant=variant)
        for _ in range(2):
            b.execute()
            b.sync()
            for j, w in enumerate(want):
                assert _same(b.download(j), w), (variant, rounds, j)
        b.destroy()


@pytest.mark.parametrize("variant", [0, 12, 16])
def test_server_serves_both(scenes, variant):
    """Small scenes alone, then with a large one (a step captured for it), then
    alone again."""
    c, narrow, wide = scenes
    want = {seed: c.bake(narrow, _params(seed)) for seed in range(20, 29)}
    srv = vlb.Server(c, step_rays=1 << 15, trace_variant=variant)
    for group in ([(narrow, 20), (narrow, 21)], [(narrow, 22), (wide, 23), (narrow, 24), (wide, 25)],
                  [(narrow, 26), (narrow, 27)], [(wide, 28)]):
        ids = [(srv.submit(sid, _params(seed)), seed) for sid, seed in group]
        for rid, seed in ids:
            assert _same(srv.wait(rid)[0], want[seed]), seed
    srv.destroy()
