"""The four-wide traversal tree at its edges: scenes of one triangle up to a
few nodes, trees deep enough to leave the LDS part of the stack, flat boxes,
scenes away from the origin; rays along the axes, from far away, with
directions of other lengths and with a finite range.  Boxes only decide which
triangles are looked at, so the hit must be, bit for bit, the one that the FP32
triangle test and its bounds gate give over all triangles, as long as that test
places no hit in front of its triangle's padded box (tiny nested triangles seen
from far away: test_tiny_triangles_from_far_away)."""
import numpy as np
import pytest

import gyunity_amd as g
from gyunity_amd._lib import FAULT_LAUNCH, FAULT_SYNC, GY_ERR_INJECTED
from tests.scene_util import wide_levels

def soup(kind, n, rng):
    """n triangles, (n, 3, 3) float32."""
    if kind == "random":
        c = rng.uniform(0, 1, (n, 1, 3))
        return (c + rng.uniform(-0.1, 0.1, (n, 3, 3))).astype(np.float32)
    if kind == "chain":  # sizes and distances halve: one triangle leaves each level of the tree
        s = 0.8 ** np.arange(n)
        base = np.array([[0, 0, 0], [1, 0, 0.3], [0, 1, 0.1]])
        return (s[:, None, None] * (base + np.array([1.0, 1.0, 1.0]))).astype(np.float32)
    if kind == "overlap":  # every triangle crosses the cube: a ray leaves children behind on every level
        return rng.uniform(0, 1, (n, 3, 3)).astype(np.float32)
    if kind == "flat":  # all in one plane
        c = np.concatenate([rng.uniform(0, 1, (n, 1, 2)), np.full((n, 1, 1), 0.5)], axis=2)
        d = rng.uniform(-0.05, 0.05, (n, 3, 3))
        d[..., 2] = 0
        return (c + d).astype(np.float32)
    if kind == "wall":  # one triangle so large that the axes of the nodes above it take no part
        tri = soup("random", n, rng)
        tri[n // 2] = 1e12 * np.array([[-1, -1, -0.5], [3, -1, -0.5], [-1, 3, -0.5]])
        return tri
    assert kind == "far"  # 300 away from the origin
    return (soup("random", n, rng).astype(np.float64) + 300.0).astype(np.float32)


def scene(tri, lights=1):
    """The triangles as a Lambert scene; the first `lights` of them emit."""
    room, _, _ = g.generate_scene(g.GY_SCENE_CORNELL, 0, 64)
    n = tri.shape[0]
    fn = np.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0])
    fn = (fn / np.maximum(np.linalg.norm(fn, axis=1, keepdims=True), 1e-30)).astype(np.float32)
    light = np.full(n, -1, np.int32)
    light[:lights] = np.arange(lights)
    return g.SceneArrays(tri.reshape(n, 9), np.repeat(fn, 3, axis=0).reshape(n, 9), fn, np.zeros(n, np.uint32), light,
                         room.mats, np.arange(lights, dtype=np.int32), np.full((lights, 3), 5.0, np.float32))


def rays_for(tri, n, rng, far=40.0):
    tri = tri[np.abs(tri).max((1, 2)) < 1e9]  # rays around and to the triangles of ordinary size
    lo, hi = tri.reshape(-1, 3).min(0).astype(np.float64), tri.reshape(-1, 3).max(0).astype(np.float64)
    ext = np.maximum(hi - lo, 0.1)
    target = tri[rng.integers(0, tri.shape[0], n)].astype(np.float64)
    w = rng.dirichlet(np.ones(3), n)
    target = (w[:, :, None] * target).sum(1)
    org = lo + rng.uniform(-0.5, 1.5, (n, 3)) * ext
    kind = rng.integers(0, 6, n)
    org[kind == 1] = target[kind == 1] + (org[kind == 1] - target[kind == 1]) * far
    d = target - org
    axis = rng.integers(0, 3, n)
    par = kind == 2  # along an axis: two components +0 or -0
    d[par] = 0.0
    d[par, axis[par]] = rng.choice([-1.0, 1.0], par.sum())
    org[par] = target[par] - d[par] * 2.0
    flat = kind == 3  # one component zero
    d[flat, axis[flat]] = rng.choice([0.0, -0.0], flat.sum())
    d /= np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-30)
    scale = np.where(kind == 4, 10.0 ** rng.uniform(-6, 6, n), 1.0)
    rays = np.zeros(n, g.RAY_DTYPE)
    rays["org"], rays["dir"] = org, d * scale[:, None]
    rays["tmax"] = np.where(kind == 5, rng.uniform(0.1, 2.0, n) * np.linalg.norm(ext), np.inf)
    return rays


def brute_force(tri, rays):
    """Closest hit (t, prim, b1, b2) and any hit of every ray over every triangle:
    Triangle::Intersect (shape/Triangle.cpp:71-103) gated by the slab test on the
    triangle's own bounds (accelerator/BVHAccel.cpp:127-149), minimum of
    (t, -prim), in FP32 operation by operation."""
    f = np.float32
    o, d = rays["org"][:, None, :], rays["dir"][:, None, :]
    tmin, tmax = rays["tmin"][:, None], rays["tmax"][:, None]
    p0 = tri[None, :, 0]
    e1, e2 = tri[None, :, 1] - p0, tri[None, :, 2] - p0

    def cross(a, b):
        return np.stack([a[..., 1] * b[..., 2] - a[..., 2] * b[..., 1], a[..., 2] * b[..., 0] - a[..., 0] * b[..., 2],
                         a[..., 0] * b[..., 1] - a[..., 1] * b[..., 0]], -1)

    def dot(a, b):
        return (a[..., 0] * b[..., 0] + a[..., 1] * b[..., 1]) + (a[..., 2] * b[..., 2] + f(0))

    with np.errstate(all="ignore"):
        s1 = cross(d, e2)
        div = dot(s1, e1)
        inv = f(1) / div
        s = o - p0
        b1 = dot(s, s1) * inv
        s2 = cross(s, e1)
        b2 = dot(d, s2) * inv
        t = dot(e2, s2) * inv
        ok = ~(div == 0) & ~((b1 < 0) | (b1 > 1)) & ~((b2 < 0) | (b1 + b2 > 1)) & ~((t < tmin) | (t > tmax))
        mn, mx = tri.min(1)[None], tri.max(1)[None]
        di = f(1) / d
        lo = (np.where(di < 0, mx, mn) - o) * di
        hi = (np.where(di < 0, mn, mx) - o) * di
        n, x = lo[..., 0], hi[..., 0]
        gate = ~((n > hi[..., 1]) | (lo[..., 1] > x))
        n, x = np.where(lo[..., 1] > n, lo[..., 1], n), np.where(hi[..., 1] < x, hi[..., 1], x)
        gate &= ~((n > hi[..., 2]) | (lo[..., 2] > x))
        n, x = np.where(lo[..., 2] > n, lo[..., 2], n), np.where(hi[..., 2] < x, hi[..., 2], x)
        ok &= gate & (n < tmax) & (x > tmin)
    key = np.where(ok, t, np.inf)
    last = key.shape[1] - 1
    prim = last - np.argmin(key[:, ::-1], axis=1)  # the largest id among the nearest
    hit = ok.any(1)
    at = (np.arange(len(rays)), prim)
    return (np.where(hit, t[at], f(0)), np.where(hit, prim, -1).astype(np.int32), np.where(hit, b1[at], f(0)),
            np.where(hit, b2[at], f(0)), hit.astype(np.int32))


CASES = [("random", n) for n in (1, 2, 3, 4, 5, 16, 17, 129, 900)] + [("chain", 60), ("chain", 150), ("flat", 300), ("far", 300), ("wall", 300),
                                                                         ("overlap", 20000)]


@pytest.mark.gpu
@pytest.mark.parametrize("leaf", [1, 4])
@pytest.mark.parametrize("kind,n", CASES)
def test_hits_are_the_brute_force_hits(gpu_ctx, kind, n, leaf):
    rng = np.random.default_rng(n + leaf)
    tri = soup(kind, n, rng)
    sa = scene(tri)
    # the triangle test itself places a hit of the chain's small triangles
    # outside their padded boxes from farther away
    rays = rays_for(tri, 4000 if n < 1000 else 200, rng, 4.0 if kind == "chain" else 40.0)
    t, prim, b1, b2, occluded = (np.concatenate(p) for p in zip(*(brute_force(tri, r) for r in np.array_split(rays, 20))))
    assert 0.2 < occluded.mean()
    with g.Scene(gpu_ctx, sa, max_leaf_size=leaf) as sc:
        hits, any_hit = sc.trace_closest(rays), sc.trace_any(rays)
        assert sc.count_visits(rays)[0] >= len(rays)  # the root at least
    assert np.array_equal(hits["prim"], prim)
    assert np.array_equal(hits["t"], t) and np.array_equal(hits["b1"], b1) and np.array_equal(hits["b2"], b2)
    assert np.array_equal(any_hit, occluded)


@pytest.mark.gpu
@pytest.mark.parametrize("leaf", [1, 4])
@pytest.mark.parametrize("far", [4.0, 40.0, 400.0])
def test_tiny_triangles_from_far_away(gpu_ctx, far, leaf):
    # The triangle test's FP32 distance can be off by more than its box is
    # padded, so the traversal can find a triangle close behind first and then
    # pass the box by.  2 to 9 of about 4500 hits; the bound is four times
    # the largest.  What is found is a hit, behind the nearest, and whether there
    # is one does not depend on it.
    rng = np.random.default_rng(150 + leaf)
    tri = soup("chain", 150, rng)
    rays = rays_for(tri, 8000, rng, far)
    t, prim, _, _, occluded = (np.concatenate(p) for p in zip(*(brute_force(tri, r) for r in np.array_split(rays, 20))))
    with g.Scene(gpu_ctx, scene(tri), max_leaf_size=leaf) as sc:
        hits, any_hit = sc.trace_closest(rays), sc.trace_any(rays)
    assert np.array_equal(any_hit, occluded) and np.array_equal(hits["prim"] >= 0, prim >= 0)
    other = hits["prim"] != prim
    assert other.sum() <= 36 and (hits["t"][other] >= t[other]).all()
    assert np.array_equal(hits["t"][~other], t[~other])


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1e-9, 1.1e-10, 0.9e-10, 1e-12, 1e-20, 1e17, 0.9e18, 1.1e18, 1e20, 1e22])
def test_short_and_long_directions_keep_the_culling(gpu_ctx, scale):
    # directions beyond the slab test's reach of 1e-10 to 1e18: the hits of the
    # brute force, and no more nodes than for directions of length 1
    rng = np.random.default_rng(5)
    tri = soup("random", 900, rng)
    rays = rays_for(tri, 3000, rng)
    rays["dir"] /= np.abs(rays["dir"]).max(1, keepdims=True)
    scaled = rays.copy()
    with np.errstate(under="ignore"):
        scaled["dir"] = rays["dir"] * np.float32(scale)
        scaled["tmax"] = rays["tmax"] / np.float32(scale)
    t, prim, b1, b2, occluded = (np.concatenate(p) for p in zip(*(brute_force(tri, r) for r in np.array_split(scaled, 20))))
    assert 0.2 < occluded.mean()
    with g.Scene(gpu_ctx, scene(tri)) as sc:
        hits, any_hit = sc.trace_closest(scaled), sc.trace_any(scaled)
        visits, plain = sc.count_visits(scaled), sc.count_visits(rays)
    assert np.array_equal(hits["prim"], prim) and np.array_equal(hits["t"], t)
    assert np.array_equal(hits["b1"], b1) and np.array_equal(hits["b2"], b2) and np.array_equal(any_hit, occluded)
    assert visits[0] < 1.05 * plain[0] and visits[1] < 1.05 * plain[1]


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n", [("chain", 150), ("overlap", 20000)])
def test_deep_stacks_render_alike_in_both_forms(gpu_ctx, kind, n):
    # the stack's deep entries go to global memory in the wavefront's trace
    # kernels and to private memory in the megakernel: same film
    rng = np.random.default_rng(n)
    sa = scene(soup(kind, n, rng), lights=n // 2)
    cam = g.camera((1.0, 1.0, 4.0), (0.6, 0.6, 0.0), (0, 1, 0), 50.0, 72, 40)
    films = []
    with g.Scene(gpu_ctx, sa, max_leaf_size=1) as sc:
        assert 3 * wide_levels(sc.bvh()[0]) > 24  # entries of the LDS part
        for mode in (g.GY_RENDER_MEGAKERNEL, g.GY_RENDER_WAVEFRONT):
            films.append(sc.render(cam, g.render_params(4, 4, mode=mode)))
    assert np.array_equal(films[0][0], films[1][0], equal_nan=True) and films[0][0].sum() > 0
    assert np.array_equal(films[0][1], films[1][1])


@pytest.mark.gpu
@pytest.mark.parametrize("spp", [48, 49])  # 64 x 64: 3072 waves, the most of a small launch at 256 CUs, and 3136
@pytest.mark.parametrize("kind,n", [("random", 300), ("ico", 6), ("chain", 300)])  # tree within an L2, beyond it, deep
def test_megakernel_forms_render_alike(gpu_ctx, kind, n, spp):
    # every instantiation that the sizes of the launch and of the tree choose
    # between, and the explicit block sizes: the wavefront's film
    if kind == "ico":
        sa, _, _ = g.generate_scene(g.GY_SCENE_ICOSPHERE_GGX, 1, n)
        cam = g.camera((0.5, 0.5, 2.35), (0.5, 0.5, 0.0), (0, 1, 0), 40.0, 64, 64)
    else:
        sa = scene(soup(kind, n, np.random.default_rng(n)), lights=n // 2)
        cam = g.camera((1.0, 1.0, 4.0), (0.6, 0.6, 0.0), (0, 1, 0), 50.0, 64, 64)
    with g.Scene(gpu_ctx, sa, max_leaf_size=1) as sc:
        want = sc.render(cam, g.render_params(spp, 3, mode=g.GY_RENDER_WAVEFRONT))
        assert want[0].sum() > 0
        for block in (0, 64, 128, 256):
            got = sc.render(cam, g.render_params(spp, 3, mode=g.GY_RENDER_MEGAKERNEL, block_size=block))
            assert np.array_equal(got[0], want[0], equal_nan=True) and np.array_equal(got[1], want[1])


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n", [("random", 64), ("random", 3000), ("chain", 150)])  # tree within the L1 or beyond
def test_light_tracing_forms_splat_alike(gpu_ctx, kind, n):
    # both forms add the same splats in another order: at most 64 * 40 * 8 * 4
    # FP32 additions of one sign in a pixel
    sa = scene(soup(kind, n, np.random.default_rng(n)), lights=n // 2)
    cam = g.camera((1.0, 1.0, 4.0), (0.6, 0.6, 0.0), (0, 1, 0), 50.0, 64, 40)
    with g.Scene(gpu_ctx, sa, max_leaf_size=1) as sc:
        want = sc.render_light_tracing(cam, g.render_params(8, 4, mode=g.GY_RENDER_WAVEFRONT))
        assert want.sum() > 0
        for block in (0, 64, 128, 256):
            got = sc.render_light_tracing(cam, g.render_params(8, 4, mode=g.GY_RENDER_MEGAKERNEL, block_size=block))
            assert np.allclose(got, want, rtol=81920 * 2.0 ** -24, atol=0)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n", [("random", 64), ("random", 1500), ("random", 2500), ("random", 60000), ("random", 72000),
                                    ("chain", 150), ("wall", 300)])
def test_both_builders_trees_give_the_same_hits(gpu_ctx, kind, n):
    # the host collapses its own trees of up to 2048 binary nodes, one workgroup
    # trees of up to 65,536, a launch a level larger ones
    rng = np.random.default_rng(n)
    tri = soup(kind, n, rng)
    rays = rays_for(tri, 4000, rng, 4.0)
    found = []
    for builder in (0, 1):
        with g.Scene(gpu_ctx, scene(tri), builder=builder) as sc:
            found.append((sc.trace_closest(rays), sc.trace_any(rays)))
    assert found[0][0].tobytes() == found[1][0].tobytes()
    assert np.array_equal(found[0][1], found[1][1])


@pytest.mark.gpu
@pytest.mark.parametrize("level,builder,fault", [(6, 0, FAULT_SYNC), (6, 1, FAULT_SYNC), (5, 1, FAULT_LAUNCH), (6, 1, FAULT_LAUNCH)])
def test_a_tree_that_failed_on_the_device_makes_no_scene(gpu_ctx, level, builder, fault):
    # a large tree is copied out of the build's workspace last (the wait for it
    # fails); the first launch of the host's builds is the collapse.  Traversal
    # follows the tree's indices without bounds checks
    sa, _, _ = g.generate_scene(g.GY_SCENE_ICOSPHERE_GGX, 1, level)
    gpu_ctx.inject_fault(fault)
    with pytest.raises(g.GyError) as e:
        g.Scene(gpu_ctx, sa, builder=builder)
    assert e.value.code == GY_ERR_INJECTED
    rays = rays_for(sa.pos.reshape(-1, 3, 3), 1000, np.random.default_rng(0))
    with g.Scene(gpu_ctx, sa, builder=builder) as sc:
        assert (sc.trace_closest(rays)["prim"] >= 0).mean() > 0.2
