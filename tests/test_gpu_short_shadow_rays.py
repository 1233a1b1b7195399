"""Shadow rays whose whole range lies within rugDistance (the light, or the end of the scene on
the way to it, is that near, or rugDistance is larger than the scene): any blocker makes them
unreliable (gather.cpp:493-511), and a ray is not done before it has tested every triangle of its
last leaf.  Floor cells of which every other one is covered, the covers' triangles in the floor
triangles' leaves, through every gather kernel, against the CPU oracle on the same seeded rays."""
import numpy as np
import pytest

from lightsprintsdk_amd import scenes as S

pytestmark = pytest.mark.gpu

CELLS = 4
HEIGHT = 5e-4            # of the covers
# (top of the scene, rugDistance, light): covers that are the top of the scene, a directional light; a
# rugDistance larger than the scene, a point light
SCENES = {
    "near_exit": (HEIGHT, 1e-3, dict(type=1, position=(0, 0, 0), direction=(-0.1, -0.2, -1.0), color=(3.0, 2.0, 1.0))),
    "large_rug": (4.0, 50.0, dict(type=0, position=(3.5, 0.5, 3.0), direction=(0, 0, -1.0), color=(9.0, 8.0, 7.0))),
}


def _scene(what):
    top, rug, light = SCENES[what]
    light = dict(light, direction=tuple(np.float64(light["direction"]) / np.linalg.norm(light["direction"])), cast_shadows=1)
    v, i, uv, objects = [], [], [], []
    none = [0.0] * 6
    for k in range(CELLS):
        # a floor triangle and its cover share a box but for a height the Morton order does not see: they
        # follow one another in the leaf order, and share leaves of two and of four
        first = len(i)
        for corners, c_uv in (((0, 1, 2), [0, 0, 1, 0, 1, 1]), ((0, 2, 3), [0, 0, 1, 1, 0, 1])):
            for z in (0.0, HEIGHT) if k % 2 == 0 else (0.0,):
                b = len(v)
                v += [(2 * k + x, y, z) for x, y in [((0, 0), (1, 0), (1, 1), (0, 1))[c] for c in corners]]
                i.append((b, b + 1, b + 2))
                uv.append(c_uv if z == 0.0 else none)
        objects.append(S.LightmapObject(f"cell{k}", first, len(i) - first, 12, 12, (0.5, 0.5, 0.5)))
    for z, x in ((-1.0, -1.0), (top, 9.0)):          # ground below all, and the scene's top corner
        b = len(v)
        v += [(x, -1, z), (x + 1, -1, z), (x, 0, z)]
        i.append((b, b + 1, b + 2))
        uv.append(none)
    v, i = np.float32(v), np.uint32(i)
    sc = S.BakeScene(v, i, np.tile(np.float32([0, 0, 1]), (len(v), 1)), np.float32(uv), np.full(len(i), 5, np.uint8),
                     np.full((len(i), 3), 0.5, np.float32), np.zeros((len(i), 3), np.float32), objects, [light])
    return sc, rug


def _texels(sc, n, seed):
    """n texels of two small subtexels on random floor triangles."""
    from lightsprintsdk_amd import bake as B
    rng = np.random.default_rng(seed)
    tex, sub = np.zeros(n, B.TEXEL_DTYPE), np.zeros(2 * n, B.SUBTEXEL_DTYPE)
    k = np.arange(n)
    floor = np.flatnonzero((sc.verts[sc.idx][:, :, 2] == 0).all(1))
    tex["out_index"], tex["sub_begin"], tex["key"] = k, 2 * k, 500 + k
    tex["sub_count_flags"] = 2 | (255 << 16)
    sub["triangle"] = np.repeat(rng.choice(floor, n), 2)
    c = rng.uniform(0.1, 0.4, (2 * n, 1, 2)) + rng.uniform(-0.05, 0.05, (2 * n, 3, 2))
    sub["uv"] = c.reshape(2 * n, 6)
    sub["area"] = rng.uniform(0.2, 1.0, 2 * n) / 100
    return tex, sub


def _compare(got, ref, sel, what):
    """Covered cells dark, open ones lit, both as the oracle has them (float32 sums of
    up to 110 terms against binary64 ones)."""
    g, r = got[sel].astype(np.float64), ref[sel]
    np.testing.assert_array_equal(g[:, 3].astype(np.float32), r[:, 3].astype(np.float32), err_msg=what)
    err = np.abs(g[:, :3] - r[:, :3]) / np.maximum(np.abs(r[:, :3]), 1e-6)
    assert err.max() <= 1e-4, (what, err.max())
    assert (r[:, 0] == 0).any() and (r[:, 0] > 0).any(), what


# kernel: (texels, quality, light rounds)
KERNELS = {
    "wave": (400, 64, 20),
    "group16": (400, 16, 16),
    "group32": (400, 24, 30),
    "persistent": (20_000, 40, 12),
    "lanes": (16 * 64 * 16 * 256, 12, 4),
    "layers": (400, 64, 20),
    "layers16": (400, 16, 16),
}


@pytest.mark.parametrize("leaf", [2, 4])
@pytest.mark.parametrize("what", list(SCENES))
@pytest.mark.parametrize("kernel", list(KERNELS))
def test_gpu_short_shadow_rays_vs_oracle(gpu, oracle, kernel, what, leaf):
    from lightsprintsdk_amd import bake as B
    from lightsprintsdk_amd.collider import RRCollider
    n, quality, rounds = KERNELS[kernel]
    sc, rug = _scene(what)
    ex = np.zeros((sc.ntri, 8), np.float32)
    gs = B.GatherScene(sc.verts, sc.idx, sc.normals, sc.side_bits, ex, sc.lights,
                       collider=RRCollider.create(sc.verts, sc.idx, leaf_size=leaf))
    p = B.GatherParams(quality=quality, ray_length_min=1e-6, rug_distance=rug, seed=31, light_rounds=rounds)
    tex, sub = _texels(sc, n, quality + leaf)
    sel = np.unique(np.linspace(0, n - 1, 400).astype(np.int64))
    print(f"short shadow rays: {kernel}, {what}, leaf {leaf}, {n} texels", flush=True)
    if kernel.startswith("layers"):
        got = gs.gather_layers(tex, sub, p, layers=(0,))[0]
    else:
        got = gs.gather(tex, sub, p)
    ref, _ = oracle.gather(gs.oracle_arrays(ex), p.as_dict(), tex[sel].view(np.uint32).reshape(-1, 4), sub,
                           tree=gs.col.download_tree(), threads=16)
    _compare(got, ref, tex["out_index"][sel], kernel)
    gs.close()


@pytest.mark.parametrize("refill", [1, 2])
@pytest.mark.parametrize("what", list(SCENES))
def test_gpu_short_shadow_rays_plan_vs_oracle(gpu, oracle, what, refill):
    from lightsprintsdk_amd import bake as B
    sc, rug = _scene(what)
    p = B.GatherParams(quality=100, ray_length_min=1e-6, rug_distance=rug, seed=33, light_rounds=50)
    plan = B.BakePlan(sc, p)
    plan.set_tuning(lane_refill=refill)
    print(f"short shadow rays: plan, {what}, lane refill {refill}", flush=True)
    plan.run(first=False, filtering=False)
    got = plan.rgba()
    sb = B.SceneBake(sc, p)                       # the plan's texels, in its order
    ex = np.zeros((sc.ntri, 8), np.float32)
    ref, _ = oracle.gather(sb.gs.oracle_arrays(ex), p.as_dict(), sb.texels.view(np.uint32).reshape(-1, 4), sb.subs,
                           tree=sb.gs.col.download_tree(), threads=16)
    _compare(got, ref, sb.texels["out_index"], what)
    sb.gs.close()
