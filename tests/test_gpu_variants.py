"""GPU tests of which trace kernel a plan runs: the variant the caller picked,
or, left to the library, a kernel for small launches below a size."""
import numpy as np
import pytest

import orc
import vlb
from conftest import rel_err

pytestmark = pytest.mark.gpu

# probes, rays: in units of a trace tile (16 x 32 rays)
SMALL = [(16, 32), (17, 33), (64, 1024), (65, 1024), (100, 1000), (128, 1024), (129, 1024), (256, 1024)]


@pytest.fixture(scope="module")
def room(ctx):
    s = vlb.generate_scene(vlb.SCENE_ROOM, 2)
    sid = ctx.upload_scene_dict(s)
    yield sid, orc.Scene.from_dict(s)
    ctx.release_scene(sid)


def _params(P, R, **kw):
    probes = np.random.default_rng(P * R).uniform([1, 0.5, 1], [9, 3.5, 9], (P, 3)).astype(np.float32)
    lights = [(vlb.LIGHT_DIRECTIONAL, (0.3, -1.0, 0.2), (3.0, 2.0, 1.0)), (vlb.LIGHT_POINT, (5.0, 3.0, 5.0), (9.0, 9.0, 9.0))]
    return vlb.Params(probes=probes, rays=R, lights=lights, **kw)


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


def _run(ctx, sid, p):
    pl = ctx.plan(sid, p)
    pl.execute()
    out, grid = pl.download(), pl.stats()["grid"]
    pl.destroy()
    return out, grid


def _tiles(P, R):
    return -(-P // 16) * -(-R // 64) * 2          # rays padded to slices of 64


@pytest.mark.parametrize("P,R", SMALL)
def test_a_picked_variant_runs_also_in_small_launches(ctx, room, P, R):
    """Every fused variant in its own kernel (two workgroups per trace tile,
    eight at least), the library's choice in the small one, the same bits."""
    sid, _ = room
    ref, grid0 = _run(ctx, sid, _params(P, R))
    t = _tiles(P, R)
    for v in list(range(1, 13)) + list(range(25, 37)):
        got, grid = _run(ctx, sid, _params(P, R, trace_variant=v))
        assert np.array_equal(_bits(got), _bits(ref)), v
        assert grid == max(8, -(-t * 2 // 8) * 8), v
    if t * 512 <= 1 << 16:                       # there with fewer rays per wave
        assert grid0 != grid


@pytest.mark.parametrize("mode", [vlb.SHADE_LAMBERT, vlb.SHADE_REFERENCE])
@pytest.mark.parametrize("variant", [0, 5, 8, 9, 12, 33, 36])
def test_shading_of_every_kernel_against_the_oracle(ctx, room, mode, variant):
    sid, o = room
    p = _params(40, 700, trace_variant=variant, shade_mode=mode, ref_light=(5.0, 3.5, 5.0))
    got, _ = _run(ctx, sid, p)
    assert rel_err(got, o.bake(p, mode64=True)["coeffs"]).max() <= 1e-5   # the bar of every FP32 bake


def test_deep_stacks_spill_the_same_in_every_kernel(ctx):
    """Concentric triangles, tilted (a chain of nodes): stacks run past their
    LDS entries into each kernel's overflow area."""
    n = 200
    s = 1.0 + np.arange(n) * 0.01
    h = 0.3 * s
    v = np.stack([np.stack([-s, -s, -h], 1), np.stack([s, -s, h], 1), np.stack([0 * s, s, 0 * h], 1)], 1)
    xyz, idx = v.reshape(-1, 3).astype(np.float32), np.arange(3 * n, dtype=np.uint32).reshape(n, 3)
    sid = ctx.upload_scene(xyz, idx)
    assert ctx.scene_info(sid)["depth"] >= 30
    o = orc.Scene(xyz, idx)
    probes = np.random.default_rng(1).uniform(-2, 2, (30, 3)).astype(np.float32)
    p = vlb.Params(probes=probes, rays=500, lights=[(vlb.LIGHT_DIRECTIONAL, (0.2, -0.3, -1.0), (3.0, 3.0, 3.0))])
    ref = o.bake(p, mode64=True)["coeffs"]
    got = []
    for v in (0, 4, 8, 12, 16, 36):
        p.trace_variant = v
        got.append(_run(ctx, sid, p)[0])
        assert np.array_equal(_bits(got[-1]), _bits(got[0])), v
    assert rel_err(got[0], ref).max() <= 1e-5
    ctx.release_scene(sid)


def test_autotuned_small_plans(ctx, room):
    """What the autotuner picks for a small plan is what later plans of that
    scene and ray count run, the library's small kernel among the candidates;
    a variant given to a later plan wins."""
    sid, _ = room
    p = _params(64, 1024)
    want, own = _run(ctx, sid, p)
    for _ in range(2):
        pl = ctx.plan(sid, p)
        v = pl.autotune(3)
        assert 1 <= v <= 36
        pl.execute()
        assert np.array_equal(_bits(pl.download()), _bits(want))
        grid = pl.stats()["grid"]
        pl.destroy()
        assert _run(ctx, sid, p)[1] == grid
        if grid == own:
            assert v == 12
    assert _run(ctx, sid, _params(64, 1024, trace_variant=12))[1] != own


@pytest.mark.parametrize("P,R", [(16, 64), (64, 1024), (65, 1024), (128, 1024), (129, 1024), (256, 1024), (257, 1024)])
def test_small_launches_by_their_size(ctx, P, R):
    """The library's choice around the sizes where its rays per wave change:
    16, 32 or 64, the fewest that make at most 16 waves per compute unit (4
    workgroups), then the ordinary kernel."""
    sid = ctx.upload_scene_dict(vlb.generate_scene(vlb.SCENE_ROOM, 2))   # a scene no autotuner has seen
    rays, cus = _tiles(P, R) * 512, ctx.device_info()["num_cus"]
    per = next((n for n in (16, 32, 64) if rays <= n * 16 * cus), None)
    got, grid = _run(ctx, sid, _params(P, R))
    ref, ordinary = _run(ctx, sid, _params(P, R, trace_variant=12))
    ctx.release_scene(sid)
    assert grid == (-(-rays // (4 * per)) if per else ordinary)
    assert np.array_equal(_bits(got), _bits(ref))
