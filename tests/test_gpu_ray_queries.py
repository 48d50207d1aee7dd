"""GPU tests of the point ray queries over the ranges their arguments may
have: directions of any length, origins far outside the scene, hits exactly
at t_min and t_max, equal distances.  The answer is the brute-force oracle's,
bit for bit: boxes decide which nodes are visited, never what is hit."""
import numpy as np
import pytest

import orc
import vlb

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def floor(ctx):
    """A flat floor whose triangles all come twice (equal distances), with
    random triangles around it."""
    n = 16
    x = np.linspace(-1, 1, n + 1)
    g = np.stack(np.meshgrid(x, x, indexing="ij"), -1)
    a, b, c, d = g[:-1, :-1], g[1:, :-1], g[:-1, 1:], g[1:, 1:]
    flat = np.concatenate([np.stack([a, b, c], -2), np.stack([b, d, c], -2)]).reshape(-1, 3, 2)
    tri = np.stack([flat[..., 0], np.full(flat.shape[:2], 0.25), flat[..., 1]], -1)
    rng = np.random.default_rng(2)
    loose = rng.uniform(-1, 1, (300, 1, 3)) + rng.uniform(-0.1, 0.1, (300, 3, 3))
    tri = np.concatenate([tri, loose, tri[::-1]]).astype(np.float32)
    xyz, idx = tri.reshape(-1, 3), np.arange(3 * len(tri), dtype=np.uint32).reshape(-1, 3)
    sid = ctx.upload_scene(xyz, idx)
    yield sid, orc.Scene(xyz, idx, bvh=False)
    ctx.release_scene(sid)


def _rays(dist, length, n=1500):
    rng = np.random.default_rng(7)
    target = rng.uniform(-1, 1, (n, 3))
    target[::3, 1] = 0.25
    d = rng.normal(size=(n, 3))
    d[::5, 1] *= 0.01                             # near grazing
    d[np.arange(0, n, 7), rng.integers(0, 3, len(range(0, n, 7)))] = 0.0
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return (target - d * dist).astype(np.float32), (d * length).astype(np.float32)


@pytest.mark.parametrize("length", [1e-7, 1e-5, 1e-3, 0.1, 1.0, 10.0, 1e3])
@pytest.mark.parametrize("dist", [1.0, 1e2, 1e3, 1e4, 3e4])
def test_any_direction_length_and_far_origins(ctx, floor, dist, length):
    sid, o = floor
    org, d = _rays(dist, length)
    tmax = np.float32(1e30)
    ref = o.trace_closest(org, d, 0.0, tmax, brute=True)
    hit = ref[0] >= 0
    assert hit.sum() > 100
    got = ctx.trace_closest(sid, org, d, 0.0, tmax)
    for g, r in zip(got, ref):
        assert np.array_equal(g, r)
    occ = ctx.trace_occluded(sid, org, d, np.full(len(org), tmax), 0.0)
    assert np.array_equal(occ, hit)
    # a hit exactly at t_max counts, here and with its lower prim id
    assert ctx.trace_occluded(sid, org[hit], d[hit], ref[1][hit], 0.0).all()
    # a hit exactly at t_min counts, and nothing before it
    for i in np.flatnonzero(hit)[:20]:
        t = ref[1][i]
        want = o.trace_closest(org[i], d[i], t, tmax, brute=True)
        assert want[0][0] >= 0 and want[1][0] == t
        got = ctx.trace_closest(sid, org[i], d[i], t, tmax)
        assert got[0][0] == want[0][0] and got[1][0] == t


@pytest.mark.parametrize("length", [1e-32, 1e-30, 1e-20, 1e20, 1e30])
def test_directions_at_the_ends_of_the_float_range(ctx, floor, length):
    """Distances up to 10^32 and down to 10^-30: the oracle's hits."""
    sid, o = floor
    org, d = _rays(2.0, length)
    tmax = np.float32(3e38)
    ref = o.trace_closest(org, d, 0.0, tmax, brute=True)
    assert (ref[0] >= 0).sum() > 100
    got = ctx.trace_closest(sid, org, d, 0.0, tmax)
    for g, r in zip(got, ref):
        assert np.array_equal(g, r)


def test_zero_directions_hit_nothing(ctx, floor):
    """... and take no longer than the rays of a usual call (a rejected box
    ends each at the root or a few nodes below)."""
    sid, o = floor
    org = np.random.default_rng(1).uniform(-1, 1, (100_000, 3)).astype(np.float32)
    org[:1000] = 0.0
    d = np.zeros_like(org)
    d[::2] = -0.0
    for tmax in (np.float32(1e30), np.float32(np.inf)):
        assert (ctx.trace_closest(sid, org, d, 0.0, tmax)[0] == -1).all()
        assert not ctx.trace_occluded(sid, org, d, np.full(len(org), tmax), 0.0).any()
