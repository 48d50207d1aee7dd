"""GPU tests of the launch paths picked by size or option: each path against
the same work on the path it stands in for, or against the oracle."""
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
