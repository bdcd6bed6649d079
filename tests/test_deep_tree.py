"""Trees so deep that the traversal stack of the large kernels is chosen, in
every integrator.  The tree is a chain of triangles whose sizes halve towards
the origin: from there a ray leaves three children of each level behind, more
than the stack's LDS part holds in any kernel.  The stack that a scene needs is
derived here from its binary tree, as scene creation does it."""
import numpy as np
import pytest

import gyunity_amd as g
from tests.scene_util import env_image, wide_levels
from tests.test_wide_bvh import scene, soup

pytestmark = pytest.mark.gpu
SMALL_STACK = 64
LDS_STACK = 24  # of the per-path kernels; 16 of the wavefront's
W, H = 40, 24


def chain(extra=0):
    """A chain that shines towards the origin, and `extra` triangles beside it."""
    rng = np.random.default_rng(7)
    tri = soup("chain", 300, rng)[:, ::-1]
    if extra:
        tri = np.concatenate([tri, soup("random", extra, rng) + np.float32([2.5, 0, 0])])
    return scene(np.ascontiguousarray(tri), lights=100)


EYE = (-0.02, -0.01, -0.015)


def cam(w=W, h=H):
    return g.camera(EYE, (1.33, 1.33, 1.13), (0, 1, 0), 30.0, w, h)


def deep_scene(ctx, sa):
    sc = g.Scene(ctx, sa, max_leaf_size=1)
    levels = wide_levels(sc.bvh()[0])
    assert 3 * levels > SMALL_STACK and 3 * levels > 2 * LDS_STACK, levels
    return sc


@pytest.mark.parametrize("builder", [0, 1])
def test_which_scenes_need_the_large_stack(gpu_ctx, builder):
    # the documented bound: three entries a level
    rng = np.random.default_rng(0)
    for kind, n, deep in (("chain", 300, True), ("chain", 60, False), ("random", 900, False), ("overlap", 20000, False)):
        with g.Scene(gpu_ctx, scene(soup(kind, n, rng)), max_leaf_size=1, builder=builder) as sc:
            levels = wide_levels(sc.bvh()[0])
            assert (3 * levels > SMALL_STACK) == deep and sc.stats().max_depth >= levels, (kind, levels)


@pytest.mark.parametrize("extra", [0, 800, 90000])  # the tree in the L1, in the L2, beyond it
def test_path_tracing(gpu_ctx, extra):
    with deep_scene(gpu_ctx, chain(extra)) as sc:
        want = sc.render(cam(), g.render_params(4, 5, mode=g.GY_RENDER_WAVEFRONT))
        assert want[0].sum() > 0
        for block in (0, 64, 128, 256):
            got = sc.render(cam(), g.render_params(4, 5, mode=g.GY_RENDER_MEGAKERNEL, block_size=block))
            assert np.array_equal(got[0], want[0], equal_nan=True) and np.array_equal(got[1], want[1])
        # past the small launches' instantiation
        big = [sc.render(cam(256, 200), g.render_params(5, 5, mode=m)) for m in (g.GY_RENDER_MEGAKERNEL, g.GY_RENDER_WAVEFRONT)]
        assert np.array_equal(big[0][0], big[1][0], equal_nan=True)


def test_samples_and_ray_queries(gpu_ctx):
    with deep_scene(gpu_ctx, chain()) as sc:
        prm = g.render_params(3, 5)
        color, weight = sc.render(cam(), prm)
        y, x, s = (a.ravel() for a in np.meshgrid(np.arange(H), np.arange(W), np.arange(3), indexing="ij"))
        L, raster, _ = sc.li_samples(cam(), prm, x, y, s)
        Lv, _, _ = sc.vpt_li_samples(cam(), prm, x, y, s, equiangular=False)
        vcolor, vweight = sc.render_vpt(cam(), prm, equiangular=False)
        rays = np.zeros(W * H, g.RAY_DTYPE)
        rng = np.random.default_rng(2)
        rays["org"] = EYE
        rays["dir"] = np.array([1.33, 1.33, 1.13]) + rng.uniform(-0.3, 0.3, (W * H, 3))
        rays["tmax"] = np.inf
        hits, occluded = sc.trace_closest(rays), sc.trace_any(rays)
    # pixels that only their own three samples reach
    for (c, w), l in (((color, weight), L), ((vcolor, vweight), Lv)):
        own = w == 3
        assert own.mean() > 0.5
        mine = l.reshape(H, W, 3, 3)
        total = mine[:, :, 0] + mine[:, :, 1] + mine[:, :, 2]
        assert np.array_equal(total[own], c[own])
    assert np.array_equal(hits["prim"] >= 0, occluded > 0) and 0.2 < occluded.mean()


@pytest.mark.parametrize("env", [False, True])
def test_environment_and_volume_forms(gpu_ctx, env):
    with deep_scene(gpu_ctx, chain()) as sc:
        if env:
            sc.set_environment(env_image())
        runs = [lambda p: sc.render(cam(), p), lambda p: sc.render_vpt(cam(), p, equiangular=False)]
        if not env:  # equi-angular sampling takes no environment light
            runs.append(lambda p: sc.render_vpt(cam(), p, equiangular=True))
        for run in runs:
            a, b = (run(g.render_params(4, 5, mode=m)) for m in (g.GY_RENDER_MEGAKERNEL, g.GY_RENDER_WAVEFRONT))
            assert np.array_equal(a[0], b[0], equal_nan=True) and np.array_equal(a[1], b[1]) and a[0].sum() > 0


@pytest.mark.parametrize("extra", [0, 800])
@pytest.mark.parametrize("env", [False, True])
def test_light_tracing(gpu_ctx, extra, env):
    # the same splats in another order: at most 40 * 24 * 8 * 5 additions of one sign
    with deep_scene(gpu_ctx, chain(extra)) as sc:
        if env:
            sc.set_environment(env_image())
        c = g.camera((3.0, 2.0, 4.0), (0.8, 0.8, 0.8), (0, 1, 0), 50.0, W, H)
        want = sc.render_light_tracing(c, g.render_params(8, 5, mode=g.GY_RENDER_WAVEFRONT))
        assert want.sum() > 0
        for block in (64, 128, 256):
            got = sc.render_light_tracing(c, g.render_params(8, 5, mode=g.GY_RENDER_MEGAKERNEL, block_size=block))
            assert np.allclose(got, want, rtol=38400 * 2.0 ** -24, atol=0)


def with_hidden_chain(sa):
    """The scene, a room open towards +z, and a chain behind its back wall, which
    no path reaches: one that leaves the room goes on towards +z."""
    add = scene(-soup("chain", 300, np.random.default_rng(7)))
    n = add.n_tri
    uv = sa.uv if sa.uv is not None else np.zeros((sa.n_tri, 6), np.float32)
    return g.SceneArrays(np.concatenate([sa.pos, add.pos]), np.concatenate([sa.nrm, add.nrm]), np.concatenate([sa.face_n, add.face_n]),
                         np.concatenate([sa.mat, np.zeros(n, np.uint32)]), np.concatenate([sa.light, np.full(n, -1, np.int32)]), sa.mats,
                         sa.light_tri, sa.light_le, uv=np.concatenate([uv, np.zeros((n, 6), np.float32)]), tex_info=sa.tex_info,
                         tex_data=sa.tex_data)


def room_and_both(ctx, kind, param):
    """The room (small stack) and the room with the chain (large stack)."""
    sa, _, _ = g.generate_scene(kind, 0, param)
    sa.pos += np.float32(SHIFT)  # the chain runs into the origin, the only place for its sizes
    assert sa.pos.min() > 0
    for arrays in (sa, with_hidden_chain(sa)):
        with g.Scene(ctx, arrays, max_leaf_size=1) as sc:
            assert (3 * wide_levels(sc.bvh()[0]) > SMALL_STACK) == (arrays is not sa)
            yield sc


SHIFT = 3.0
ROOM_CAM = ((SHIFT + 0.5, SHIFT + 0.5, SHIFT + 2.35), (SHIFT + 0.5, SHIFT + 0.5, SHIFT), (0, 1, 0), 40.0, W, H)


def test_photon_mapping_and_spheres(gpu_ctx):
    c = g.camera(*ROOM_CAM)
    sp = np.zeros(2, g.SPHERE_DTYPE)
    sp["center"] = SHIFT + np.array([(0.3, 0.18, 0.55), (0.5, 0.72, 0.45)])
    sp["radius"], sp["material"] = [0.15, 0.07], [0, 0]
    sp["emissive"], sp["le"] = [0, 1], [(0, 0, 0), (6, 6, 6)]
    rng = np.random.default_rng(3)
    rays = np.zeros(2000, g.RAY_DTYPE)
    rays["org"], rays["dir"], rays["tmax"] = SHIFT + rng.uniform(0.1, 0.9, (2000, 3)), rng.normal(size=(2000, 3)), np.inf
    out = []
    for sc in room_and_both(gpu_ctx, g.GY_SCENE_CORNELL, 64):
        got = list(sc.render_sppm(c, g.sppm_params(3, 20000, 6, 0.05, 0.7)))
        got += list(sc.render(c, g.render_params(4, 5)))
        sc.set_spheres(sp)
        got += list(sc.render(c, g.render_params(4, 5)))
        hits = sc.trace_closest(rays)
        hits["prim"][hits["prim"] >= sc.arrays.n_tri] -= sc.arrays.n_tri - 1000  # spheres follow the triangles
        got += [hits, sc.trace_any(rays)]
        out.append(got)
    assert out[0][2].sum() > 0 and out[0][3].sum() > 0
    for a, b in zip(*out):
        assert a.tobytes() == b.tobytes()


def test_adjoints(gpu_ctx):
    # the same terms, added by float atomics in another order: at most
    # 40 * 24 * 4 * 5 additions to a texel or a light, of both signs
    c = g.camera(*ROOM_CAM)
    prm = g.render_params(4, 5, mode=g.GY_RENDER_WAVEFRONT)
    dI = np.random.default_rng(1).uniform(-1.0, 1.0, (H, W, 3)).astype(np.float32)
    out = []
    for sc in room_and_both(gpu_ctx, g.GY_SCENE_ADJOINT, 16):
        image = sc.render(c, prm)
        one = sc.adjoint(c, prm, dI, emission=True)
        with g.Batch(gpu_ctx) as b:
            b.add(sc, c, prm)
            b.render()
            many = b.adjoint([dI], sc.texture_floats(), n_light=sc.n_light)
        out.append((image, one, many))
    (room, one, many), (image, *deep) = out
    assert np.array_equal(room[0], image[0]) and room[0].sum() > 0
    for k in (0, 1):  # texels, lights
        want = one[k]
        assert np.abs(want).max() > 0
        for got in (many[k], deep[0][k], deep[1][k]):
            assert np.abs(got - want).max() <= 19200 * 2.0 ** -24 * np.abs(want).max()


def test_batch_of_shallow_and_deep_scenes(gpu_ctx):
    # one launch sequence, its spill store as large as the deepest scene needs
    sa, _, _ = g.generate_scene(g.GY_SCENE_CORNELL, 0, 64)
    room = g.camera((0.5, 0.5, 2.35), (0.5, 0.5, 0.0), (0, 1, 0), 40.0, W, H)
    prm = g.render_params(4, 5, mode=g.GY_RENDER_WAVEFRONT)
    with g.Scene(gpu_ctx, sa) as shallow, deep_scene(gpu_ctx, chain()) as deep:
        want = [shallow.render(room, prm), deep.render(cam(), prm)]
        for order in ((0, 1), (1, 0), (0, 0, 1)):
            with g.Batch(gpu_ctx) as b:
                ids = [b.add((shallow, deep)[k], (room, cam())[k], prm) for k in order]
                for _ in range(2):
                    b.render()
                    for i, k in zip(ids, order):
                        got = b.film(i)
                        assert np.array_equal(got[0], want[k][0], equal_nan=True) and np.array_equal(got[1], want[k][1])
