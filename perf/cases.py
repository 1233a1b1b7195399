"""What a program that uses this package has the GPU do, as cases that can be timed and
compared: ray batches against a mesh, the setup of a scene, lightmap bakes (plain, layered,
learned), per-vertex lighting, the filter chain with the writeback, and a training step of
the surrogate.

listed() names the cases, draw() gives more of the same ranges, prepare() makes what a
program holds before the call, run() is one pass through the public entry points, work() the
bytes and operations a pass cannot do without, tolerance() what another correct
implementation may differ by, exact() the same outputs in 64 bits where brute force allows.
"""
import ctypes
import math

import numpy as np
import torch

from lightsprintsdk_amd import learned as LG
from lightsprintsdk_amd import native as N
from lightsprintsdk_amd import scenes as S
from lightsprintsdk_amd.bake import BakePlan, GatherParams, GatherScene, VertexPlan, SUBTEXEL_DTYPE
from lightsprintsdk_amd.collider import RRCollider, make_rrrays


def listed():
    return [
        # a picking or visibility query of an application frame: few rays, small mesh, latency
        dict(name="hit_4k", kind="hit", frequency=12, rays=4096),
        # the collider's headline batch: 1M random rays, 100,820-triangle displaced icosphere
        dict(name="hit_1m", kind="hit", frequency=71, rays=1_000_000),
        # intersectBatch over the caller's own 128-byte RRRay records in host memory, odd count
        dict(name="rrrays_100k", kind="rrrays", frequency=47, rays=100_003),
        # loading a scene: tree build, scene upload, rasterisation of 21 lightmaps
        dict(name="setup_room", kind="setup", scene="room", objects=20, tris=50_000, size=256),
        # preview bake of a small level, as the solver adapter calls it (no graph)
        dict(name="bake_preview", kind="bake", scene="room", objects=12, tris=10_000, size=63, quality=256, env=0, graph=False),
        # the headline bake: box room of about 50k triangles, 21 lightmaps of 256x256, 1024 rays
        dict(name="bake_room", kind="bake", scene="room", objects=20, tris=50_000, size=256, quality=1024, env=0, graph=True),
        # open field: sun and four point lights, panorama sky, lightmaps of mixed odd sizes
        dict(name="bake_field", kind="bake", scene="field", objects=36, tris=150_000, size=320, quality=300, env=1, graph=False),
        # directional lightmaps and bent normals of a level (five output layers)
        dict(name="layers_room", kind="layers", scene="room", objects=9, tris=20_000, size=97, quality=128, env=0),
        # per-vertex lighting of a level, sun-and-sky gather smoothed into the vertices
        dict(name="vertex_field", kind="vertex", scene="field", objects=25, tris=60_000, size=32, quality=200, env=1),
        # the learned bake of a room the surrogate was not trained on
        dict(name="learned_room", kind="learned", objects=20, tris=50_000, size=256),
        # eight optimiser steps of the surrogate at its training batch
        dict(name="train_8k", kind="train", rows=8192, steps=8),
        # filter chain of gathered maps and the writeback into byte lightmaps, odd sizes
        dict(name="filter_maps", kind="filter", maps=5, width=1013, height=731, spread=1000, sigma=1.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["hit", "hit", "rrrays", "setup", "bake", "bake", "layers", "vertex", "learned", "train", "filter"])
    if kind in ("hit", "rrrays"):
        return dict(kind=kind, frequency=rng.randint(8, 71 if kind == "hit" else 47),
                    rays=_log(rng, 1000, 1_000_000 if kind == "hit" else 100_000))
    if kind == "train":
        return dict(kind=kind, rows=_log(rng, 300, 16384), steps=rng.randint(2, 8))
    if kind == "filter":
        return dict(kind=kind, maps=rng.randint(1, 12), width=_log(rng, 24, 900), height=_log(rng, 24, 700),
                    spread=rng.choice([0, 2, 40, 1000]), sigma=rng.choice([0.0, 0.5, 1.0, 2.0]))
    if kind == "learned":
        return dict(kind=kind, objects=rng.randint(6, 20), tris=_log(rng, 8000, 50_000), size=rng.randint(96, 256))
    scene = rng.choice(["room", "field"])
    c = dict(kind=kind, scene=scene, objects=rng.randint(3, 20), tris=_log(rng, 2000, 50_000), size=rng.randint(33, 200))
    if kind != "setup":
        c.update(quality=_log(rng, 16, 600), env=rng.choice([0, 1]))
    if kind == "bake":
        c.update(graph=rng.choice([False, True]))
    return c


# ---- inputs ---------------------------------------------------------------------------

def _scene(case, seed):
    """The case's level (its shapes and unwraps follow from the sizes) with the seed's colours,
    lights, scale and order of triangles within each object."""
    if case["scene"] == "room":
        sc = S.box_room(seed=case["objects"], n_boxes=case["objects"], target_tris=case["tris"], lightmap_size=case["size"])
    else:
        # lightmap sides between size/8 and size, about 15 m of ground per object
        sc = S.object_field(seed=case["objects"], n_objects=case["objects"], target_tris=case["tris"],
                            lightmap_range=(max(16, case["size"] // 8), case["size"]), area=15.0 * math.sqrt(case["objects"]))
    rng = np.random.default_rng(seed)
    scale = np.float32(rng.uniform(0.95, 1.05))
    sc.verts = sc.verts * scale
    order = np.arange(sc.ntri)
    for ob in sc.objects:
        own = slice(ob.tri_begin, ob.tri_begin + ob.tri_count)
        order[own] = ob.tri_begin + _shuffled_strips(rng, ob.tri_count)
        sc.albedo[own] = rng.uniform(0.2, 0.8, 3)
    for k in ("idx", "tri_uv", "side_bits", "albedo", "emittance"):
        setattr(sc, k, np.ascontiguousarray(getattr(sc, k)[order]))
    sc.emittance = sc.emittance * np.float32(rng.uniform(0.7, 1.3))
    for light in sc.lights:
        light["color"] = tuple(c * f for c, f in zip(light["color"], rng.uniform(0.7, 1.2, 3)))
        light["position"] = tuple(float(scale) * p + m for p, m in zip(light["position"], rng.uniform(-0.3, 0.3, 3)))
        d = np.asarray(light["direction"], np.float64) + rng.uniform(-0.2, 0.2, 3)
        light["direction"] = tuple(d / np.linalg.norm(d))
    return sc


def _shuffled_strips(rng, n):
    """0..n-1 in runs of 64 whose order is random: neighbours mostly stay together, as exporters leave them."""
    starts = np.arange(0, n, 64)
    rng.shuffle(starts)
    return np.concatenate([np.arange(a, min(n, a + 64)) for a in starts]) if n else np.zeros(0, np.int64)


def _sky(seed):
    """A panorama sky of 64 x 32 texels: bright towards the zenith, with a blotch of haze."""
    rng = np.random.default_rng(seed)
    v = np.linspace(-1, 1, 32)[:, None, None]
    base = np.array([0.5, 0.7, 1.0]) * (0.35 + 0.6 * np.clip(v, 0, 1))
    return (base * rng.uniform(0.8, 1.2, (32, 64, 1))).astype(np.float32)


def _params(case, scene, seed):
    return GatherParams(quality=case["quality"], ray_length_min=S.minimal_safe_distance(scene.verts), seed=seed & 0x7FFFFFFF,
                        environment_multiplier=1.0 if case["env"] else 0.0)


class _Device:
    """A torch view of a device buffer the library owns."""

    def __init__(self, ptr, shape, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=typestr, data=(int(ptr), False), version=2)


def _view(ptr, shape, typestr, owner):
    return torch.as_tensor(_Device(ptr, shape, typestr, owner), device="cuda")


class _FilterPlan:
    def __init__(self, maps):
        h = ctypes.c_void_p()
        N.check(N.lib().lsg_filter_plan_create(maps, len(maps), ctypes.byref(h)), "filter plan")
        self.handle = h

    def __del__(self):
        N.lib().lsg_filter_plan_destroy(self.handle)


def _filter_input(case, seed):
    """Gathered RGBA maps: rectangular charts with gutters over about 60% of a map, alpha =
    coverage flags / 255 (full inside, some quadrants and edges at chart borders), HDR values
    smooth within a chart with the noise of a gather."""
    g = torch.Generator().manual_seed(seed)
    w, h, n = case["width"], case["height"], case["maps"]
    out = torch.zeros(n, h, w, 4)
    for m in range(n):
        k = int(torch.randint(2, 6, (1,), generator=g))
        ys = [round(i * h / k) for i in range(k + 1)]
        xs = [round(i * w / k) for i in range(k + 1)]
        for a in range(k):
            for b in range(k):
                f = 0.02 + 0.2 * torch.rand(4, generator=g)
                y0, y1 = ys[a] + int(f[0] * (ys[a + 1] - ys[a])), ys[a + 1] - int(f[1] * (ys[a + 1] - ys[a]))
                x0, x1 = xs[b] + int(f[2] * (xs[b + 1] - xs[b])), xs[b + 1] - int(f[3] * (xs[b + 1] - xs[b]))
                if y1 <= y0 or x1 <= x0:
                    continue
                level = torch.exp(torch.randn(3, generator=g))
                rgb = level * (1 + 0.03 * torch.randn(y1 - y0, x1 - x0, 3, generator=g))
                flags = torch.full((y1 - y0, x1 - x0), 255, dtype=torch.int32)
                rim = torch.zeros(y1 - y0, x1 - x0, dtype=torch.bool)
                rim[0], rim[-1], rim[:, 0], rim[:, -1] = True, True, True, True
                flags[rim] = torch.randint(1, 256, (int(rim.sum()),), generator=g, dtype=torch.int32)
                out[m, y0:y1, x0:x1, :3] = rgb.clamp_min(0)
                out[m, y0:y1, x0:x1, 3] = flags / 255.0
    return out


def _train_input(case, seed):
    """Feature rows and targets with the scales of the gathered ones: log1p radiances, window
    means near them, positions, unit normals, albedos, spreads; corrections of a few percent."""
    g = torch.Generator().manual_seed(seed)
    n = case["rows"] * case["steps"]
    x = torch.empty(n, 32)
    base = torch.log1p(torch.exp(0.8 * torch.randn(n, 3, generator=g)))
    for k in (0, 6, 9, 12):
        x[:, k:k + 3] = base + 0.15 / (1 + k) * torch.randn(n, 3, generator=g)
    for k in (3, 15):
        x[:, k:k + 3] = torch.log1p(torch.relu(torch.randn(n, 1, generator=g)) * torch.tensor([1.0, 0.9, 0.8]))
    x[:, 18:21] = 2 * torch.rand(n, 3, generator=g) - 1
    nrm = torch.randn(n, 3, generator=g)
    x[:, 21:24] = nrm / nrm.norm(dim=1, keepdim=True)
    x[:, 24:27] = 0.2 + 0.6 * torch.rand(n, 3, generator=g)
    x[:, 27:29] = torch.log(0.01 + torch.rand(n, 2, generator=g))
    x[:, 29] = torch.rand(n, generator=g)
    x[:, 30] = torch.log1p(torch.relu(torch.randn(n, generator=g)))
    x[:, 31] = 1
    t = 0.2 * (x[:, 12:15] - x[:, 0:3]) + 0.05 * torch.sin(3 * x[:, 18:21]) + 0.03 * torch.randn(n, 3, generator=g)
    return x, t


def _mesh(case, seed):
    return S.icosphere(case["frequency"], seed=seed)


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind in ("hit", "rrrays"):
        V, I = _mesh(case, seed)
        R = S.random_rays(V, case["rays"], seed=seed + 1)
        st["col"] = RRCollider.create(V, I)
        if kind == "rrrays":
            st["rays"] = make_rrrays(R)
            return st
        st["ro"] = torch.from_numpy(np.ascontiguousarray(R[:, :4])).cuda()
        st["rd"] = torch.from_numpy(np.ascontiguousarray(R[:, 4:])).cuda()
        st["hits"] = torch.empty(case["rays"], 4, dtype=torch.int32, device="cuda")
        st["front"] = torch.empty(case["rays"], dtype=torch.uint8, device="cuda")
        return st
    if kind == "train":
        x, t = _train_input(case, seed)
        st["x"], st["t"] = x.cuda(), t.cuda()
        st["net"] = LG.Surrogate(max_batch=(case["rows"] + 15) // 16 * 16, seed=seed)
        return st
    if kind == "filter":
        st["input"] = _filter_input(case, seed).cuda()
        n, h, w = st["input"].shape[:3]
        st["rgba"] = torch.empty_like(st["input"])
        st["rgbf"] = torch.empty(n, h, w, 3, device="cuda")
        st["bytes"] = torch.empty((3 * n * h * w + 3) // 4 * 4, dtype=torch.uint8, device="cuda")
        maps = (N.Lightmap * n)(*[N.Lightmap(k * w * h, w, h, k * w * h) for k in range(n)])
        st["plan"] = _FilterPlan(maps)
        return st
    if kind == "learned":
        sc = _scene(dict(case, scene="room"), seed)
        st["ls"] = LG.LearnedScene(sc, seed=seed & 0x7FFFFFFF)
        st["net"], bound, _ = LG.load_weights()
        st["target"] = bound["target"]
        sb = st["ls"].sb
        st["out"] = dict(rgba=_view(sb.d_out.ptr, (sb.nout, 4), "<f4", sb), rgbf=_view(sb.d_rgbf.ptr, (sb.nout, 3), "<f4", sb))
        return st
    st["scene"] = sc = _scene(case, seed)
    if kind == "setup":
        return st
    st["params"] = p = _params(case, sc, seed)
    if kind == "vertex":
        ex = np.zeros((sc.ntri, 8), np.float32)
        ex[:, :3] = sc.emittance + 0.3 * sc.albedo
        gs = GatherScene(sc.verts, sc.idx, sc.normals, sc.side_bits, ex, sc.lights)
        st["vertex"] = VertexPlan(gs, sc)
    else:
        st["plan"] = plan = BakePlan(sc, p)
        gs = plan.gs
        inf = plan.info()
        st["out"] = dict(rgba=_view(inf.rgba, (inf.num_slots, 4), "<f4", plan), rgbf=_view(inf.rgbf, (inf.num_slots, 3), "<f4", plan))
    if case["env"]:
        gs.set_environment(GatherScene.ENV_PANORAMA, 64, 32, _sky(seed))
    return st


def run(st):
    case, L = st["case"], N.lib()
    kind = case["kind"]
    if kind == "hit":
        N.check(L.lsg_collider_intersect_device(st["col"]._h, st["ro"].data_ptr(), st["rd"].data_ptr(), case["rays"],
                                                st["hits"].data_ptr(), st["front"].data_ptr(), None), "hit")
        return dict(tri=st["hits"][:, 0], tuv=st["hits"][:, 1:].view(torch.float32), front=st["front"])
    if kind == "rrrays":
        r = st["rays"]
        mask = st["col"].intersect_rrrays(r)
        return dict(mask=mask, t=r["hitDistance"], tri=r["hitTriangle"], uv=r["hitPoint2d"], plane=r["hitPlane"],
                    point=r["hitPoint3d"], front=r["hitFrontSide"])
    if kind == "train":
        net, n = st["net"], case["rows"]
        for k in range(case["steps"]):
            N.check(L.lsg_mlp_train_step(net._h, st["x"].data_ptr() + 4 * 32 * n * k, st["t"].data_ptr() + 12 * n * k, n,
                                         LG.LAMBDA, 2e-3, None, None), "train_step")
        return net.get_params()
    if kind == "filter":
        st["rgba"].copy_(st["input"])           # the gather's output, which the chain works on in place
        bg = (ctypes.c_float * 4)(0.0, 0.0, 0.0, 0.0)
        fp = N.FilterParams(case["sigma"], case["spread"], bg, 0)
        N.check(L.lsg_filter_plan_run(st["plan"].handle, st["rgba"].data_ptr(), st["rgbf"].data_ptr(), ctypes.byref(fp), None), "filter")
        N.check(L.lsg_lightmap_encode(st["rgba"].data_ptr(), st["rgba"].numel() // 4, 0, 1, 0.45, 0.45, bg,
                                      st["bytes"].data_ptr(), None), "encode")
        return dict(rgba=st["rgba"], rgbf=st["rgbf"], bytes=st["bytes"][:st["rgbf"].numel()])
    if kind == "learned":
        st["ls"].learned(st["net"], target=st["target"])
        return st["out"]
    if kind == "setup":
        sc = st["scene"]
        plan = BakePlan(sc, GatherParams(ray_length_min=S.minimal_safe_distance(sc.verts)))
        inf = plan.info()
        words = SUBTEXEL_DTYPE.itemsize // 4
        subs = _view(inf.subtexels, (inf.num_subtexels, words), "<i4", plan)
        return dict(texels=_view(inf.texels, (inf.num_texels, 4), "<i4", plan), triangle=subs[:, 0],
                    uv_area=subs[:, 1:].view(torch.float32))
    if kind == "vertex":
        return st["vertex"].gather(st["params"])[0]
    plan = st["plan"]
    if kind == "layers":
        plan.run_layers()
        maps = range(len(plan.scene.objects))
        return [np.concatenate([plan.lightmap_layer(k, l).reshape(-1) for k in maps]) for l in range(5)]
    plan.run(first=True, graph=case["graph"])
    return st["out"]


# ---- what a pass cannot do without ----------------------------------------------------

def _ray_flops(ntri):
    """One ray through a tree of ntri triangles: log2(ntri) node visits, each four box tests
    of 12 operations, and two triangle tests of 30."""
    return 48.0 * math.log2(max(ntri, 2)) + 60.0


def work(case):
    kind = case["kind"]
    if kind in ("hit", "rrrays"):
        nt, n = 20 * case["frequency"] ** 2, case["rays"]
        return dict(bytes=49.0 * n + 110.0 * nt if kind == "hit" else 256.0 * n + 110.0 * nt, flops=n * _ray_flops(nt))
    if kind == "train":
        weights = 32 * 64 + 3 * 64 * 64 + 64 * 4
        rows = case["rows"] * case["steps"]
        return dict(bytes=140.0 * rows + 28.0 * weights * case["steps"], flops=6.0 * weights * rows)
    if kind == "filter":
        n = case["maps"] * case["width"] * case["height"]
        return dict(bytes=(16.0 + 16 + 12 + 3) * n, flops=60.0 * n)
    if kind == "learned":
        texels = 0.55 * (case["objects"] + 1) * case["size"] ** 2
        rays = 22.5 * texels                     # 16 + 2 of the cheap gather, a quarter of it again
        return dict(bytes=130.0 * texels + 150.0 * case["tris"], flops=rays * _ray_flops(case["tris"]) + 29000.0 * texels)
    maps = case["objects"] + (1 if case["scene"] == "room" else 0)
    # about 0.55 of a room's map is covered; a field's sides are log-uniform, mean square 0.24 of the largest
    texels = (0.55 if case["scene"] == "room" else 0.13) * maps * case["size"] ** 2
    if kind == "setup":
        return dict(bytes=150.0 * case["tris"] + (16 + 96.0) * texels, flops=400.0 * texels + 500.0 * case["tris"])
    lights = 1 if case["scene"] == "room" else 5
    if kind == "vertex":
        rays = case["tris"] * (case["quality"] + lights * (case["quality"] // 10 + 1))
        return dict(bytes=200.0 * case["tris"], flops=rays * _ray_flops(case["tris"]))
    rays = texels * (case["quality"] + lights * (case["quality"] // 10 + 1))
    rays += case["tris"] * lights * (case["quality"] // 20 + 1)
    return dict(bytes=(112.0 + 28 * (5 if kind == "layers" else 1)) * texels + 150.0 * case["tris"],
                flops=rays * _ray_flops(case["tris"]))


def tolerance(case):
    kind = case["kind"]
    if kind in ("hit", "rrrays", "setup"):
        return "exact"                           # hits and texel lists are pinned bit for bit
    if kind == "filter":
        return dict(rel=1e-6, max=1e-5, differ=0.0)
    if kind == "train":
        # rows in another order move the weights by 6e-8 (largest 4e-6); another order inside a
        # product also rounds some bf16 activations the other way
        return dict(rel=1e-4, max=1e-2)
    if kind == "learned":
        return dict(rel=2e-3, max=0.5)           # bf16 network; a texel at the bound may fall back or not
    # up to 1024 radiances summed in another order move a map by 5.4e-8 (largest 6.5e-7)
    return dict(rel=1e-6, max=1e-4)


# ---- the same outputs in 64 bits -------------------------------------------------------

def _brute_force(V, I, R, chunk=1 << 26):
    """Closest hits by testing every triangle in binary64: (triangle or -1, t, u, v, unit normal), on the GPU."""
    v = torch.from_numpy(V.astype(np.float64)).cuda()
    i = torch.from_numpy(I.astype(np.int64)).cuda()
    r = torch.from_numpy(R.astype(np.float64)).cuda()
    a = v[i[:, 0]]
    e1, e2 = v[i[:, 1]] - a, v[i[:, 2]] - a
    nrm = torch.linalg.cross(e1, e2)
    e11, e12, e22 = (e1 * e1).sum(1), (e1 * e2).sum(1), (e2 * e2).sum(1)
    inv = 1 / (e11 * e22 - e12 * e12)
    pu = (e22[:, None] * e1 - e12[:, None] * e2) * inv[:, None]      # u = pu . (p - a), v = pv . (p - a)
    pv = (e11[:, None] * e2 - e12[:, None] * e1) * inv[:, None]
    na, ua, va = (nrm * a).sum(1), (pu * a).sum(1), (pv * a).sum(1)
    out = []
    for q in torch.split(r, max(1, chunk // len(I))):
        o, tmin, d, tmax = q[:, :3], q[:, 3:4], q[:, 4:7], q[:, 7:8]
        t = (na - o @ nrm.T) / (d @ nrm.T)
        u = o @ pu.T + t * (d @ pu.T) - ua
        w = o @ pv.T + t * (d @ pv.T) - va
        ok = (u >= 0) & (w >= 0) & (u + w <= 1) & (t >= tmin) & (t <= tmax)
        t = torch.where(ok, t, math.inf)
        best, k = t.min(1)
        hit = torch.isfinite(best)
        k = torch.where(hit, k, 0)
        pick = lambda x: torch.where(hit, x.gather(1, k[:, None])[:, 0], 0.0)      # noqa: E731
        out.append((torch.where(hit, k, -1), torch.where(hit, best, 0.0), pick(u), pick(w)))
    tri, t, u, w = (torch.cat(x) for x in zip(*out))
    n = nrm / nrm.norm(dim=1, keepdim=True)
    return tri, t, u, w, torch.cat([n, -(n * a).sum(1, keepdim=True)], 1)


def _exact_filter(case, seed):
    rgba = _filter_input(case, seed).double().cuda()
    flags_of = lambda a: (a.float() * 255 + 0.5).to(torch.int64)      # noqa: E731
    F = torch.nn.functional
    alpha = rgba[..., 3]
    rgb = rgba[..., :3]
    near = [(jj, ii) for jj in (-1, 0, 1) for ii in (-1, 0, 1)]
    n, h, w = alpha.shape

    def shifted(x, jj, ii, mode="constant"):
        x = x.movedim(-1, 1)
        x = F.pad(x, (1, 1, 1, 1), mode=mode)[:, :, 1 + jj:1 + jj + h, 1 + ii:1 + ii + w]
        return x.movedim(1, -1)

    if case["sigma"] > 0:
        cf = flags_of(alpha)
        masks = []
        for jj, ii in near:
            nf = shifted(cf[..., None].double(), jj, ii)[..., 0].to(torch.int64)
            inside = shifted(torch.ones_like(alpha)[..., None], jj, ii)[..., 0] > 0
            both = lambda a, b: ((cf & a) > 0) & ((nf & b) > 0)      # noqa: E731
            ok = inside
            if ii < 0: ok = ok & both(16, 32)      # noqa: E701
            if ii > 0: ok = ok & both(32, 16)      # noqa: E701
            if jj < 0: ok = ok & both(64, 128)     # noqa: E701
            if jj > 0: ok = ok & both(128, 64)     # noqa: E701
            masks.append(ok)
        x = torch.cat([rgb, (alpha > 0).double()[..., None]], -1)
        left = np.float32(min(case["sigma"], 10.0)) ** 2
        while left > 0:
            s2 = min(left, np.float32(0.34))
            left = np.float32(left - s2)
            wt = [1.0, math.exp(-0.5 / s2), math.exp(-1 / s2)]
            y = torch.zeros_like(x)
            for (jj, ii), ok in zip(near, masks):
                y += x * wt[0] if not (ii or jj) else shifted(x, jj, ii) * (ok.double() * wt[abs(ii) + abs(jj)])[..., None]
            x = torch.where((x[..., 3] != 0)[..., None], y / y[..., 3:], x)
        rgb = torch.where((alpha > 0)[..., None], x[..., :3], rgb)
    full = torch.cat([rgb, alpha[..., None]], -1)
    total = torch.zeros_like(full)
    for jj, ii in near:
        nb = shifted(full, jj, ii)
        f = flags_of(nb[..., 3])
        q = torch.zeros_like(f, dtype=torch.bool)
        for bit, fits in ((8, ii < 1 and jj < 1), (1, ii > -1 and jj > -1), (2, ii < 1 and jj > -1), (4, ii > -1 and jj < 1)):
            if fits:
                q |= (f & bit) > 0
        wgt = 1.0 if ii and jj else 1.6
        total += torch.cat([nb[..., :3], torch.ones_like(nb[..., 3:])], -1) * (q.double() * wgt)[..., None]
    grown = torch.cat([total[..., :3] / total[..., 3:].clamp_min(1e-30), torch.full_like(total[..., 3:], 0.001)], -1)
    c = torch.where(((alpha <= 0.002) & (total[..., 3] > 0))[..., None], grown, full)
    g = torch.where((c[..., 3:] > 0), torch.cat([c[..., :3], torch.ones_like(c[..., 3:])], -1), torch.zeros_like(c))
    for _ in range(int(case["spread"])):
        d = sum(shifted(g, jj, ii, "replicate") * (1.0 if ii and jj else 1.6) for jj, ii in near if ii or jj)
        fill = (g[..., 3] == 0) & (d[..., 3] > 0)
        if not bool(fill.any()):
            break
        g = torch.where(fill[..., None], d / d[..., 3:].clamp_min(1e-30), g)
    c = torch.where(((c[..., 3] <= 0) & (g[..., 3] > 0))[..., None], torch.cat([g[..., :3], torch.full_like(g[..., 3:], 0.001)], -1), c)
    c = torch.where((c[..., 3:] > 0), c, torch.zeros_like(c))
    return dict(rgba=c, rgbf=c[..., :3].contiguous(), bytes=None)


def _exact_train(case, seed):
    x, t = (v.double() for v in _train_input(case, seed))
    shapes = LG.Surrogate.layer_shapes()
    rng = np.random.default_rng(seed)
    p = []
    for k, (i, o) in enumerate(shapes):           # the surrogate's initial weights for this seed
        w = rng.normal(size=(i, o)) * math.sqrt(2.0 / i) * (0.1 if k == 4 else 1.0)
        if k == 4:
            w[:, 4:] = 0
        p += [torch.from_numpy(w.astype(np.float32)).double(), torch.zeros(o, dtype=torch.float64)]
    p = [v.requires_grad_() for v in p]
    m, s = [torch.zeros_like(v) for v in p], [torch.zeros_like(v) for v in p]
    for k in range(case["steps"]):
        a, y = x[k * case["rows"]:(k + 1) * case["rows"]], t[k * case["rows"]:(k + 1) * case["rows"]]
        for j in range(5):
            a = a @ p[2 * j] + p[2 * j + 1]
            a = torch.relu(a) if j < 4 else a
        d = a[:, :3] - y
        e = (d * d).mean(1).sqrt().detach()
        loss = ((d * d).sum(1) + LG.LAMBDA * (a[:, 3] - e) ** 2).mean()
        for j, gr in enumerate(torch.autograd.grad(loss, p)):
            m[j] = 0.9 * m[j] + 0.1 * gr
            s[j] = 0.999 * s[j] + 0.001 * gr * gr
            with torch.no_grad():
                p[j] -= 2e-3 * (m[j] / (1 - 0.9 ** (k + 1))) / ((s[j] / (1 - 0.999 ** (k + 1))).sqrt() + 1e-8)
    return torch.cat([v.detach().reshape(-1) for v in p]).numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_train(case, seed)
    if kind == "filter":
        return _exact_filter(case, seed)
    if kind in ("hit", "rrrays") and case["rays"] * case["frequency"] ** 2 <= 1e9:
        V, I = _mesh(case, seed)
        R = S.random_rays(V, case["rays"], seed=seed + 1)
        tri, t, u, v, plane = _brute_force(V, I, R)
        if kind == "hit":
            return dict(tri=None, tuv=torch.stack([t, u, v], 1), front=None)
        r = make_rrrays(R)                       # what misses keep
        hit = (tri >= 0).cpu().numpy()
        old = lambda f, x: np.where(hit[:, None], x.cpu().numpy(), r[f].astype(np.float64).reshape(len(r), -1))      # noqa: E731
        d = torch.from_numpy(R[:, 4:7].astype(np.float64)).cuda()
        o = torch.from_numpy(R[:, :3].astype(np.float64)).cuda()
        return dict(mask=None, tri=None, front=None, t=old("hitDistance", t[:, None])[:, 0], uv=old("hitPoint2d", torch.stack([u, v], 1)),
                    plane=old("hitPlane", plane[tri.clamp_min(0)]), point=old("hitPoint3d", o + d * t[:, None]))
    # gathers and bakes: every ray of every texel against every triangle, after the texels'
    # pieces are clipped, is minutes of work; a scene's setup is tested against an oracle
    return None
