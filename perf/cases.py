"""Performance cases of the renderer: what a program that uses this framework
has it do, through its public entry points (gyunity_amd and the C ABI).

A case is one call, or the forward and backward call of a gradient step, on a
scene that is already on the device.  Scenes are the repository's procedural
ones (Cornell room, displaced icosphere of 20 * 4^level triangles in that room,
batch members, textured rooms), sized from a 64 x 64 thumbnail to the
1024 x 1024, 64 samples per pixel, 1.31M-triangle render.

Kinds:
  render    Scene.render: path tracing, megakernel or wavefront, Sobol or
            Halton, area light or environment map, film downloaded
  batch     Batch.render: many scenes of uneven size in one launch sequence
  gradient  render_textures forward and backward (path-replay adjoint, one view)
  views     render_views forward and backward (adjoint over a batch of views)
  light     Scene.render_light_tracing
  fog       Scene.render_vpt (volumetric path tracing)
  photons   Scene.render_sppm
  rays      gy_trace_closest_device and gy_trace_any_device on a ray batch
"""
import math

import numpy as np
import torch  # before gyunity_amd: one HIP runtime for both

import gyunity_amd as g
from gyunity_amd.torch_render import render_textures, render_views

LAMBERT, CONDUCTOR, GLASS, ROUGH_GLASS = 0, 1, 2, 3
OBJECTS = {"lambert": LAMBERT, "ggx": CONDUCTOR, "glass": GLASS, "rough_glass": ROUGH_GLASS}
ROOM = 12  # triangles of the room and its light


def listed():
    return [
        # an interactive viewer's thumbnail, the smallest call: launches and host latency
        dict(name="thumbnail", kind="render", level=-1, object="lambert", width=64, height=64, spp=4, depth=5,
             form="megakernel", sampler="sobol", env=False),
        # a preview of the Cornell room at its own settings: short launches
        dict(name="cornell_preview", kind="render", level=-1, object="lambert", width=256, height=256, spp=16, depth=5,
             form="wavefront", sampler="sobol", env=False),
        # the benchmark's final frame: 1.31M triangles, 67M paths
        dict(name="final_frame", kind="render", level=8, object="ggx", width=1024, height=1024, spp=64, depth=8,
             form="wavefront", sampler="sobol", env=False),
        # a ragged frame with Halton samples and a rough dielectric, one path per thread
        dict(name="ragged_megakernel", kind="render", level=6, object="rough_glass", width=701, height=523, spp=9,
             depth=10, form="megakernel", sampler="halton", env=False),
        # a frame lit by an environment map
        dict(name="sky", kind="render", level=7, object="ggx", width=640, height=360, spp=16, depth=6,
             form="wavefront", sampler="sobol", env=True),
        # a set of scenes of uneven size rendered together
        dict(name="scene_batch", kind="batch", entries=16, res=256, spp=16, max_tri=60000),
        # one optimisation step of the textures of a room seen from one view
        dict(name="texture_step", kind="gradient", res=256, spp=64, tex=64),
        # one optimisation step over several views of the 1.31M-triangle textured object
        dict(name="views_step", kind="views", views=8, res=256, spp=16, tex=512),
        # light tracing
        dict(name="light_tracing", kind="light", level=7, object="ggx", width=512, height=512, spp=16, depth=8,
             form="wavefront", sampler="sobol"),
        # volumetric path tracing in fog, equi-angular sampling
        dict(name="fog", kind="fog", level=7, object="ggx", width=512, height=512, spp=16, depth=8, form="wavefront",
             sampler="sobol", equiangular=True),
        # progressive photon mapping at the reference's settings, a few iterations
        dict(name="photon_map", kind="photons", level=6, object="ggx", width=512, height=512, iterations=4,
             photons=300000, depth=20, sampler="halton"),
        # ray queries of a program with its own integrator: camera rays and scattered rays
        dict(name="ray_queries", kind="rays", level=5, object="ggx", rays=1 << 20),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _frame(rng, budget, depth):
    """Width, height and samples with at most `budget` path vertices."""
    w, h = _log(rng, 48, 1100), _log(rng, 48, 1100)
    spp = min(_log(rng, 1, 64), max(1, budget // (w * h * depth)))
    return w, h, spp


def draw(rng):
    kind = rng.choice(["render", "render", "render", "render", "batch", "gradient", "views", "light", "fog", "photons", "rays"])
    obj = rng.choice(list(OBJECTS))
    if kind == "render":
        env = rng.random() < 0.25
        level = rng.randint(3, 8) if env else rng.choice([-1, 3, 4, 5, 6, 7, 8])
        form = rng.choice(["megakernel", "wavefront", "wavefront"])
        depth = rng.randint(3, 12)
        w, h, spp = _frame(rng, (1 << 28) if form == "wavefront" and not env else (1 << 26), depth)
        return dict(kind=kind, level=level, object="lambert" if level < 0 else obj, width=w, height=h, spp=spp,
                    depth=depth, form=form, sampler=rng.choice(["sobol", "sobol", "halton"]), env=env)
    if kind == "batch":
        return dict(kind=kind, entries=rng.randint(3, 24), res=rng.choice([96, 128, 200, 256, 320]), spp=rng.randint(2, 24),
                    max_tri=_log(rng, 1000, 200000))
    if kind == "gradient":
        return dict(kind=kind, res=_log(rng, 64, 320), spp=_log(rng, 4, 64), tex=_log(rng, 16, 256))
    if kind == "views":
        return dict(kind=kind, views=rng.randint(2, 8), res=_log(rng, 96, 256), spp=rng.randint(4, 16), tex=rng.randint(128, 1024))
    if kind in ("light", "fog"):
        depth = rng.randint(3, 10)
        form = rng.choice(["megakernel", "wavefront", "wavefront"])
        w, h, spp = _frame(rng, 1 << 25, depth)
        case = dict(kind=kind, level=rng.randint(3, 8), object=obj, width=w, height=h, spp=spp, depth=depth, form=form,
                    sampler=rng.choice(["sobol", "sobol", "halton"]))
        if kind == "fog":
            case["equiangular"] = rng.random() < 0.6
        return case
    if kind == "photons":
        return dict(kind=kind, level=rng.randint(3, 7), object=obj, width=_log(rng, 64, 640), height=_log(rng, 64, 640),
                    iterations=rng.randint(1, 6), photons=_log(rng, 10000, 300000), depth=rng.randint(5, 20),
                    sampler=rng.choice(["sobol", "halton"]))
    return dict(kind=kind, level=rng.randint(2, 8), object=obj, rays=_log(rng, 1 << 12, 1 << 23))


# ------------------------------------------------------------------ inputs
class _State:
    """The handles of one case; freed with it."""

    def __init__(self):
        self.ctx = g.Context(0)
        self.scenes = []
        self.batch = None

    def scene(self, arrays):
        sc = g.Scene(self.ctx, arrays)
        self.scenes.append(sc)
        return sc

    def __del__(self):
        try:
            if self.batch is not None:
                self.batch.close()
            for sc in self.scenes:
                sc.close()
            self.ctx.close()
        except Exception:  # the interpreter is going down
            pass


def _camera(rng, width, height):
    """The Cornell camera, moved a little by the seed."""
    x, y, z = rng.uniform(-0.04, 0.04, 3)
    return g.camera((0.5 + x, 0.5 + y, 2.35 + z), (0.5, 0.5, 0.0), (0.0, 1.0, 0.0), 40.0, width, height)


def _room(case, seed, rng):
    """The Cornell room (level -1) or the icosphere room, lights scaled by the seed."""
    if case["level"] < 0:
        sa, _, _ = g.generate_scene(g.GY_SCENE_CORNELL, 0, 64)
    else:
        sa, _, _ = g.generate_scene(g.GY_SCENE_ICOSPHERE_GGX, seed & 0xFFFF, case["level"])
        mat = sa.mats[-1]
        mat[0] = OBJECTS[case["object"]]
        if mat[0] == LAMBERT:
            mat[2:5] = rng.uniform(0.2, 0.9, 3).astype(np.float32).view(np.uint32)
        else:
            mat[1] = 3 if mat[0] == CONDUCTOR else 1  # alpha given directly, Schlick Fresnel for the conductor
            mat[8:10] = np.full(2, rng.uniform(0.1, 0.4), np.float32).view(np.uint32)
    sa.light_le *= np.float32(rng.uniform(0.7, 1.4))
    return sa


def _sky(sa, rng, w=1024, h=512):
    """The room's floor and back wall under a seeded sky with a sun."""
    keep = np.r_[0:2, 4:6, ROOM:sa.n_tri]
    out = g.SceneArrays(sa.pos[keep], sa.nrm[keep], sa.face_n[keep], sa.mat[keep], np.full(len(keep), -1, np.int32),
                        sa.mats, np.zeros(0, np.int32), np.zeros((0, 3), np.float32),
                        uv=sa.uv[keep] if sa.uv is not None else None)
    v = (np.arange(h) + 0.5)[:, None] / h
    u = (np.arange(w) + 0.5)[None, :] / w
    at, up = rng.uniform(0.2, 0.8), rng.uniform(0.15, 0.35)
    sun = 200.0 * np.exp(-(((u - at) / 0.02) ** 2 + ((v - up) / 0.03) ** 2))
    sky = np.stack([0.3 + 0.5 * (1 - v), 0.4 + 0.4 * (1 - v), 0.7 + 0.3 * (1 - v)], -1) * np.ones((1, w, 1))
    return out, (sky + sun[..., None] * np.array([1.0, 0.9, 0.75])).astype(np.float32)


def _fog(sa, rng, lo=(0.06, 0.01, 0.06), hi=(0.94, 0.9, 0.94)):
    """The room with a material-less box of homogeneous fog in it."""
    c = np.array([[(lo, hi)[(i >> k) & 1][k] for k in range(3)] for i in range(8)], np.float32)
    quads = [((0, 1, 5, 4), (0, -1, 0)), ((2, 6, 7, 3), (0, 1, 0)), ((0, 4, 6, 2), (-1, 0, 0)),
             ((1, 3, 7, 5), (1, 0, 0)), ((0, 2, 3, 1), (0, 0, -1)), ((4, 5, 7, 6), (0, 0, 1))]
    box = np.array([[c[q[0]], c[q[i]], c[q[i + 1]]] for q, _ in quads for i in (1, 2)], np.float32).reshape(-1, 9)
    bn = np.repeat(np.array([n for _, n in quads], np.float32), 2, axis=0)
    n = box.shape[0]
    uv = sa.uv if sa.uv is not None else np.zeros((sa.n_tri, 6), np.float32)
    out = g.SceneArrays(np.concatenate([sa.pos, box]), np.concatenate([sa.nrm, np.tile(bn, (1, 3))]),
                        np.concatenate([sa.face_n, bn]), np.concatenate([sa.mat, np.zeros(n, np.uint32)]),
                        np.concatenate([sa.light, np.full(n, -1, np.int32)]), sa.mats, sa.light_tri, sa.light_le,
                        uv=np.concatenate([uv, np.zeros((n, 6), np.float32)]))
    media = np.zeros(1, g.MEDIUM_DTYPE)
    media["sigma_a"], media["sigma_s"] = rng.uniform(0.03, 0.1, 3), rng.uniform(0.5, 0.9, 3)
    media["g"] = rng.uniform(0.0, 0.5)
    tri = np.zeros(out.n_tri, g.TRI_MEDIUM_DTYPE)
    tri["inside"], tri["outside"] = -1, -1
    tri["inside"][sa.n_tri:] = 0
    tri["no_material"][sa.n_tri:] = 1
    return out, media, tri


def _params(case, spp, depth):
    return g.render_params(spp, depth, 5, g.GY_RENDER_MEGAKERNEL if case["form"] == "megakernel" else g.GY_RENDER_WAVEFRONT,
                           sampler=g.GY_SAMPLER_HALTON if case["sampler"] == "halton" else g.GY_SAMPLER_SOBOL)


def _rays(n, seed):
    """Half camera rays in scan order, half scattered rays between points of the
    room, (n, 8) float32: origin, tmin, direction, tmax."""
    gen = torch.Generator().manual_seed(seed)
    rays = torch.empty(n, 8)
    half = n // 2
    side = max(1, math.isqrt(half))
    i = torch.arange(half)
    target = torch.stack([(i % side + torch.rand(half, generator=gen)) / side,
                          ((i // side) % side + torch.rand(half, generator=gen)) / side, torch.full((half,), 0.5)], 1)
    rays[:half, :3] = torch.tensor([0.5, 0.5, 2.35])
    rays[:half, 4:7] = target - rays[:half, :3]
    a, b = torch.rand(n - half, 3, generator=gen), torch.rand(n - half, 3, generator=gen)
    rays[half:, :3] = a
    rays[half:, 4:7] = b - a
    rays[:, 4:7] /= rays[:, 4:7].norm(dim=1, keepdim=True)
    rays[:, 3] = 0.0
    rays[:, 7] = float("inf")
    return rays


def prepare(case, seed):
    st = _State()
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind in ("render", "light", "fog", "photons", "rays"):
        sa = _room(case, seed, rng)
        img = media = None
        if kind == "render" and case["env"]:
            sa, img = _sky(sa, rng)
        if kind == "fog":
            sa, media, tri = _fog(sa, rng)
        st.sc = st.scene(sa)
        if img is not None:
            st.sc.set_environment(img)
        if media is not None:
            st.sc.set_media(media, tri)
        if kind == "rays":
            st.rays = _rays(case["rays"], seed).cuda()
            st.hits = torch.empty(case["rays"], 4, device="cuda")
            st.occluded = torch.empty(case["rays"], dtype=torch.int32, device="cuda")
        else:
            st.cam = _camera(rng, case["width"], case["height"])
        if kind == "photons":
            st.params = g.sppm_params(case["iterations"], case["photons"], case["depth"], 0.01, 0.75,
                                      sampler=g.GY_SAMPLER_HALTON if case["sampler"] == "halton" else g.GY_SAMPLER_SOBOL)
        elif kind != "rays":
            st.params = _params(case, case["spp"], case["depth"])
    elif kind == "batch":
        st.batch = g.Batch(st.ctx)
        sizes = _entry_sizes(case)
        for e in range(case["entries"]):
            sa, _, prm = g.generate_scene(g.GY_SCENE_BATCH_MEMBER, (seed + 7919 * e) & 0xFFFF, max(100, case["max_tri"] >> (e % 5)))
            prm.spp, prm.mode, prm.max_depth = sizes[e][1], g.GY_RENDER_WAVEFRONT, 4 + e % 7
            st.batch.add(st.scene(sa), _camera(rng, sizes[e][0], sizes[e][0]), prm)
    elif kind == "gradient":
        sa, cam, prm = g.generate_scene(g.GY_SCENE_ADJOINT, seed & 0xFFFF, case["tex"])
        prm.spp, prm.mode = case["spp"], g.GY_RENDER_WAVEFRONT
        cam.width = cam.height = case["res"]
        st.sc, st.cam, st.params = st.scene(sa), cam, prm
        st.textures, st.target = _optimisation(sa, rng, (case["res"], case["res"], 3))
    elif kind == "views":
        sa, _, prm = g.generate_scene(g.GY_SCENE_ICOSPHERE_TEXTURED, seed & 0xFFFF, case["tex"])
        prm.spp, prm.mode = case["spp"], g.GY_RENDER_WAVEFRONT
        st.sc = st.scene(sa)
        st.batch = g.Batch(st.ctx)
        for cam in g.orbit_views(case["views"], case["res"], seed=seed):
            st.batch.add(st.sc, cam, prm)
        st.textures, st.target = _optimisation(sa, rng, (case["views"] * case["res"] ** 2 * 3,))
    else:
        raise ValueError(kind)
    st.kind, st.case = kind, case
    torch.cuda.synchronize()
    return st


def _entry_sizes(case):
    """(side, samples) of each batch entry: whole, half and quarter sides, uneven budgets."""
    return [(max(16, case["res"] >> (e % 3)), max(1, case["spp"] >> (e % 2))) for e in range(case["entries"])]


def _optimisation(sa, rng, shape):
    """Texels part of the way to the scene's own, and a target image."""
    start = sa.tex_data * np.float32(0.8) + rng.uniform(0.02, 0.15, sa.tex_data.size).astype(np.float32)
    tex = torch.from_numpy(start).cuda().requires_grad_(True)
    return tex, torch.from_numpy(rng.uniform(0.0, 0.6, shape).astype(np.float32)).cuda()


# ------------------------------------------------------------------ one pass
def run(st):
    if st.kind == "render":
        return st.sc.render(st.cam, st.params)
    if st.kind == "batch":
        st.batch.render()
        return [st.batch.film(e) for e in range(st.case["entries"])]
    if st.kind in ("gradient", "views"):
        st.textures.grad = None
        if st.kind == "gradient":
            image = render_textures(st.sc, st.cam, st.params, st.textures)
        else:
            image = render_views(st.sc, st.batch, st.textures)
        loss = ((image - st.target) ** 2).mean()
        loss.backward()
        return image.detach(), st.textures.grad
    if st.kind == "light":
        return st.sc.render_light_tracing(st.cam, st.params)
    if st.kind == "fog":
        return st.sc.render_vpt(st.cam, st.params, equiangular=st.case["equiangular"])
    if st.kind == "photons":
        return st.sc.render_sppm(st.cam, st.params)
    n, lib = st.case["rays"], g.lib()
    for call, out in ((lib.gy_trace_closest_device, st.hits), (lib.gy_trace_any_device, st.occluded)):
        if call(st.sc.h, st.rays.data_ptr(), n, out.data_ptr()) != 0:
            raise RuntimeError(lib.gy_last_error())
    return st.hits[:, 0], st.hits.view(torch.int32)[:, 1], st.hits[:, 2:], st.occluded


# ------------------------------------------------------------------ what a pass cannot do without
def _triangles(case):
    if case["kind"] in ("gradient",):
        return 20492
    if case["kind"] == "views":
        return 1310732
    return 36 if case["level"] < 0 else 20 * 4 ** case["level"] + ROOM


def _ray_flops(n_tri):
    """One ray through a binary hierarchy over n_tri triangles: two slab tests
    (24 operations each) on each of about log2(n) + 4 nodes and three triangle
    tests of 50."""
    return 48 * (math.log2(n_tri) + 4) + 150


def work(case):
    kind = case["kind"]
    if kind == "rays":
        n = _triangles(case)
        return {"bytes": n * 48 + case["rays"] * (32 + 16 + 32 + 4), "flops": 2 * case["rays"] * _ray_flops(n)}
    if kind == "batch":
        out = {"bytes": 0.0, "flops": 0.0}
        for e, (res, spp) in enumerate(_entry_sizes(case)):
            n = max(100, case["max_tri"] >> (e % 5))
            out["bytes"] += n * 176 + res * res * 16
            out["flops"] += res * res * spp * (4 + e % 7) * 0.8 * (2 * _ray_flops(n) + 1000)
        return out
    n = _triangles(case)
    scene = n * 176  # 48 bytes to intersect and 128 to shade a triangle
    if kind == "photons":
        px = case["width"] * case["height"]
        vertices = case["iterations"] * (px * 2 + case["photons"] * 5)
        return {"bytes": scene + px * 20, "flops": vertices * (_ray_flops(n) + 1000)}
    if kind == "gradient":
        paths, px, depth, passes, floats = case["res"] ** 2 * case["spp"], case["res"] ** 2, 5, 2, 16 * case["tex"] ** 2
    elif kind == "views":
        px = case["views"] * case["res"] ** 2
        paths, depth, passes, floats = px * case["spp"], 6, 2, 4 * case["tex"] ** 2
    else:
        px = case["width"] * case["height"]
        paths, depth, passes, floats = px * case["spp"], case["depth"], 1, 0
    return {"bytes": passes * (scene + px * 16 + floats * 4), "flops": passes * paths * depth * 0.8 * (2 * _ray_flops(n) + 1000)}


def tolerance(case):
    if case["kind"] == "rays":
        # the hit distance is one triangle's own; exact ties at shared edges may name either triangle
        return {"rel": 1e-5, "max": 1e-3, "differ": 1e-4}
    # Every path's arithmetic is fixed; sums over a pixel's samples, splats and
    # texel gradients (float atomics) may be taken in another order.
    return {"rel": 1e-5}


def exact(case, seed):
    """Ray queries against every triangle in 64 bits: the nearest hit's distance
    and barycentrics, and whether there is one.  Images are estimates over
    paths that branch on 32-bit comparisons and have no 64-bit value."""
    if case["kind"] != "rays":
        return None
    n_tri = _triangles(case)
    if case["rays"] * n_tri > 1 << 35:
        return None
    rng = np.random.default_rng(seed)
    pos = torch.from_numpy(_room(case, seed, rng).pos).cuda().double().reshape(-1, 3, 3)
    rays = _rays(case["rays"], seed).cuda().double()
    p0, e1, e2 = pos[:, 0], pos[:, 1] - pos[:, 0], pos[:, 2] - pos[:, 0]
    t_out = torch.zeros(case["rays"], dtype=torch.float64, device="cuda")
    b_out = torch.zeros(case["rays"], 2, dtype=torch.float64, device="cuda")
    chunk = max(1, (1 << 27) // n_tri)
    for i in range(0, case["rays"], chunk):
        o, d = rays[i:i + chunk, :3], rays[i:i + chunk, 4:7]
        # det and the barycentrics as products of per-ray and per-triangle 3-vectors
        m = torch.linalg.cross(o, d, dim=1)
        nrm = torch.linalg.cross(e1, e2, dim=1)
        det = -(d @ nrm.T)
        b1 = (m @ e2.T - d @ torch.linalg.cross(e2, p0, dim=1).T) / det
        b2 = (d @ torch.linalg.cross(e1, p0, dim=1).T - m @ e1.T) / det
        t = (o @ nrm.T - (p0 * nrm).sum(1)) / det
        ok = (b1 >= 0) & (b2 >= 0) & (b1 + b2 <= 1) & (t >= 0) & (det != 0)
        t = torch.where(ok, t, torch.inf)
        best, k = t.min(dim=1)
        hit = torch.isfinite(best)
        t_out[i:i + chunk] = torch.where(hit, best, 0.0)
        bary = torch.stack([b1.gather(1, k[:, None])[:, 0], b2.gather(1, k[:, None])[:, 0]], 1)
        b_out[i:i + chunk] = torch.where(hit[:, None], bary, 0.0)
    return t_out, None, b_out, None
