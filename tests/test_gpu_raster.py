"""GPU texel rasteriser (lsg_rasterize_texels: each triangle clipped against the squares of
its candidate texels, pairs sorted by texel) against the oracle's restatement of the
reference's method (oracle/lsg_oracle_raster.c: each texel square clipped by the triangle's
sides in triangle space, lightmap.cpp:147-331).  The two clip in different frames and
triangulate from different first vertices, so they are compared on what the gather and the
filters read: the set of covered texels, each texel's flags, and for every (texel, triangle)
the covered area and the polygon's corners; plus the orders (texels row-major, pieces in
triangle order) and the closed forms the oracle is pinned by."""
import ctypes

import numpy as np
import pytest

from lightsprintsdk_amd import scenes as S

pytestmark = pytest.mark.gpu


def _gpu(uv, w, h, ids=None, obj=0, base=0):
    from lightsprintsdk_amd import bake as B
    uv = np.asarray(uv, np.float32).reshape(-1, 6)
    ids = np.arange(len(uv), dtype=np.uint32) if ids is None else np.asarray(ids, np.uint32)
    return B.rasterize(uv, ids, w, h, obj, base)


def _clip64(tri, x, y):
    """triangle (3x2 texel units) intersected with the texel square [x,x+1]x[y,y+1] in
    binary64 (Sutherland-Hodgman); returns (area in texel units, corners)"""
    poly = [tuple(p) for p in tri]
    for axis, lim, sg in ((0, x, 1), (0, x + 1, -1), (1, y, 1), (1, y + 1, -1)):
        out = []
        for i in range(len(poly)):
            p, c = poly[i - 1], poly[i]
            dp, dc = sg * (p[axis] - lim), sg * (c[axis] - lim)
            if (dp >= 0) != (dc >= 0):
                t = dp / (dp - dc)
                out.append((p[0] + (c[0] - p[0]) * t, p[1] + (c[1] - p[1]) * t))
            if dc >= 0:
                out.append(c)
        poly = out
        if len(poly) < 3:
            return 0.0, []
    a = 0.0
    for i in range(1, len(poly) - 1):
        a += (poly[i][0] - poly[0][0]) * (poly[i + 1][1] - poly[0][1]) - (poly[i][1] - poly[0][1]) * (poly[i + 1][0] - poly[0][0])
    return abs(a) * 0.5, poly


def _truth(uv, w, h):
    """{(texel slot, triangle): (area in the pieces' unit, corners in texel units)} in binary64"""
    out = {}
    for t, u in enumerate(uv.astype(np.float64)):
        tri = u.reshape(3, 2) * np.array([w, h])
        e1, e2 = tri[1] - tri[0], tri[2] - tri[0]
        if e1[0] * e2[1] - e1[1] * e2[0] == 0:
            continue
        lo, hi = np.floor(tri.min(axis=0)), np.floor(tri.max(axis=0))
        for y in range(max(int(lo[1]), 0), min(int(hi[1]), h - 1) + 1):
            for x in range(max(int(lo[0]), 0), min(int(hi[0]), w - 1) + 1):
                a, poly = _clip64(tri, x, y)
                if a > 0:
                    out[(x + y * w, t)] = (0.5 * a / (w * h), poly)
    return out


def _pieces(tex, sub):
    """{(texel slot, triangle): (stored area, corner list in triangle space)}"""
    out = {}
    for t in tex:
        n = t["sub_count_flags"] & 0xFFFF
        for s in sub[t["sub_begin"]:t["sub_begin"] + n]:
            key = (int(t["out_index"]), int(s["triangle"]))
            a, pts = out.get(key, (0.0, []))
            pts = pts + [tuple(s["uv"][0:2]), tuple(s["uv"][2:4]), tuple(s["uv"][4:6])]
            out[key] = (a + float(s["area"]), pts)
    return out


def _corners(pts, uv, w, h):
    """distinct polygon corners in texel units (triangle space -> map -> texels)"""
    p = np.array(pts, np.float64)
    u0, e1, e2 = uv[0:2].astype(np.float64), (uv[2:4] - uv[0:2]).astype(np.float64), (uv[4:6] - uv[0:2]).astype(np.float64)
    m = (u0 + p[:, :1] * e1 + p[:, 1:2] * e2) * np.array([w, h])
    keep = []
    for q in m:
        if not any(np.abs(q - k).max() < 2e-3 for k in keep):
            keep.append(q)
    return np.array(keep)


def _distinct(poly):
    keep = []
    for q in np.array(poly, np.float64):
        if not any(np.abs(q - k).max() < 2e-3 for k in keep):
            keep.append(q)
    return np.array(keep)


def compare(uv, w, h, label, sliver=1e-6, flag_frac=1 / 2000):
    """GPU and oracle against the binary64 intersections, and against each other"""
    uv = np.asarray(uv, np.float32).reshape(-1, 6)
    import oracle_py as O
    gt, gs = _gpu(uv, w, h)
    ot, os_ = O.rasterize(uv, np.arange(len(uv), dtype=np.uint32), w, h)
    unit = 0.5 / (w * h)                      # a whole texel in the pieces' area unit
    # orders: texels row-major, pieces in triangle order
    for tx, sb in ((gt, gs), (ot, os_)):
        assert np.all(np.diff(tx["out_index"].astype(np.int64)) > 0), label
        for t in tx:
            n = t["sub_count_flags"] & 0xFFFF
            assert np.all(np.diff(sb["triangle"][t["sub_begin"]:t["sub_begin"] + n].astype(np.int64)) >= 0), label
    T = _truth(uv, w, h)
    G, Oo = _pieces(gt, gs), _pieces(ot, os_)
    bad = dict(gpu_area=0, gpu_corner=0, gpu_set=0, oracle_area=0, oracle_set=0)
    for key in set(T) | set(G) | set(Oo):
        at = T.get(key, (0.0, []))[0]
        # GPU: binary32 clipping of texel-local corners, about 1e-7 texel per coordinate;
        # oracle: the reference's binary32 Heron formula in triangle space
        for name, D, rel, ab in (("gpu", G, 1e-5, 2e-6), ("oracle", Oo, 2e-3, 2e-6)):
            if key not in D:
                bad[name + "_set"] += at > sliver * unit            # only slivers may be missing
                continue
            ad = D[key][0]
            if abs(ad - at) > rel * at + ab * unit and abs(ad - at) > rel * 1e-3 * unit:
                if key in T or ad > sliver * unit:
                    bad[name + "_area"] += 1
        if key in G and key in T and at > 1e-3 * unit:
            cg = _corners(G[key][1], uv[key[1]], w, h)
            ct = _distinct(T[key][1])
            same = len(cg) == len(ct) and all(np.abs(ct - q).max(axis=1).min() < 2e-3 for q in cg)
            bad["gpu_corner"] += not same
    # the texels both cover by more than a sliver carry the same flags
    flags_g = {int(t["out_index"]): int(t["sub_count_flags"]) >> 16 for t in gt}
    flags_o = {int(t["out_index"]): int(t["sub_count_flags"]) >> 16 for t in ot}
    cover = {k[0] for k, v in T.items() if v[0] > sliver * unit}
    bad_flags = sum(flags_g.get(s) != flags_o.get(s) for s in cover)
    print(f"{label}: {len(gt)} texels / {len(gs)} pieces on the GPU, {len(ot)} / {len(os_)} in the oracle, "
          f"{len(cover)} covered; mismatches {bad}, flags {bad_flags}", flush=True)
    assert all(v == 0 for v in bad.values()), (label, bad)
    assert bad_flags <= max(1, int(len(cover) * flag_frac)), label
    return gt, gs


def test_gpu_raster_full_quad_closed_form(gpu):
    """Two triangles covering the unit square of a 4x4 map: 16 texels in row-major order,
    each covered to 1/16 of the map, the triangles' pieces summing to half their map area."""
    tex, sub = _gpu([[0, 0, 1, 0, 1, 1], [0, 0, 1, 1, 0, 1]], 4, 4)
    assert len(tex) == 16 and np.all(tex["out_index"] == np.arange(16))
    for t in range(2):
        assert abs(sub["area"][sub["triangle"] == t].astype(np.float64).sum() - 0.25) < 1e-6
    cover = np.add.reduceat(sub["area"].astype(np.float64), tex["sub_begin"])
    np.testing.assert_allclose(cover, 0.5 / 16, rtol=1e-5)
    assert np.all(((tex["sub_count_flags"] >> 16) & 15) == 15)
    # only the four texels the diagonal crosses hold pieces of both triangles
    two = [len(set(sub["triangle"][b:b + (c & 0xFFFF)])) for b, c in zip(tex["sub_begin"], tex["sub_count_flags"])]
    assert sorted(two) == [1] * 12 + [2] * 4


def test_gpu_raster_outside_and_degenerate(gpu):
    tex, sub = _gpu([[2, 2, 3, 2, 2, 3], [0.1, 0.1, 0.1, 0.1, 0.1, 0.1], [0.5, 0.5, 0.5, 0.5, 0.5, 0.5]], 8, 8)
    assert len(tex) == 0 and len(sub) == 0


def test_gpu_raster_random_triangles_vs_oracle(gpu):
    rng = np.random.default_rng(7)
    for w, h, n, size in [(16, 16, 40, 0.3), (64, 48, 300, 0.08), (256, 256, 500, 0.02), (37, 91, 40, 0.5)]:
        c = rng.uniform(-0.1, 1.1, (n, 1, 2))
        uv = (c + rng.uniform(-size, size, (n, 3, 2))).reshape(n, 6)
        compare(uv, w, h, f"random {w}x{h}")


def test_gpu_raster_grid_aligned_vs_oracle(gpu):
    """Corners on texel corners and centres, edges along grid lines and diagonals.  A polygon
    corner exactly on a texel's centre line sets no quadrant bit here (its centred
    coordinate is exactly 0); the oracle, like the reference, reaches it through triangle
    space and decides by the rounding of the round trip, so a few such texels may differ."""
    rng = np.random.default_rng(8)
    w = h = 32
    q = rng.integers(0, 2 * w + 1, (300, 3, 2)) / (2.0 * w)
    compare(q.reshape(-1, 6), w, h, "grid-aligned", sliver=1e-5, flag_frac=0.01)


def test_gpu_raster_scene_objects_vs_oracle(gpu):
    sc = S.box_room(seed=3, n_boxes=6, target_tris=8000, lightmap_size=96)
    for ob in sc.objects[:3]:
        compare(sc.tri_uv[ob.tri_begin:ob.tri_begin + ob.tri_count], ob.width, ob.height, f"box room object {ob.tri_begin}")
    fs = S.object_field(seed=5, n_objects=4, target_tris=8_000, lightmap_range=(16, 128), area=20.0)
    for ob in fs.objects:
        compare(fs.tri_uv[ob.tri_begin:ob.tri_begin + ob.tri_count], ob.width, ob.height, f"object field {ob.tri_begin}")


def test_gpu_raster_deterministic_and_ids(gpu):
    sc = S.box_room(seed=4, n_boxes=4, target_tris=4000, lightmap_size=64)
    ob = sc.objects[1]
    uv = sc.tri_uv[ob.tri_begin:ob.tri_begin + ob.tri_count]
    ids = np.arange(ob.tri_begin, ob.tri_begin + ob.tri_count, dtype=np.uint32)
    a = _gpu(uv, ob.width, ob.height, ids, obj=3, base=1000)
    b = _gpu(uv, ob.width, ob.height, ids, obj=3, base=1000)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1].view(np.uint32), b[1].view(np.uint32))
    assert np.all(a[0]["out_index"] >= 1000)
    assert np.all((a[0]["key"] - np.uint32(3 * 0x9E3779B1 & 0xFFFFFFFF)) == a[0]["out_index"] - 1000)
    assert set(np.unique(a[1]["triangle"])) <= set(ids)


@pytest.mark.parametrize("groups", [1, 2])
def test_gpu_plan_rasterises_objects_together(gpu, groups):
    """A bake plan's texel and piece lists (all objects rasterised together) are the lists of
    its objects rasterised one at a time, one after another: odd map sizes, an object without
    triangles, one whose triangles cover nothing, one with a single texel.  With two maps of
    6000^2 crossed by a sliver (36M candidates each, few texels) the objects do not fit one
    group of 2^26 candidates."""
    from lightsprintsdk_amd import bake as B
    from lightsprintsdk_amd import native as N
    rng = np.random.default_rng(4)
    sizes = [(33, 17), (8, 8), (1, 1), (64, 65), (5, 3)]
    counts = [40, 0, 3, 120, 6]
    if groups == 2:
        sizes, counts = [(6000, 6000), (9, 7), (8, 8), (6000, 6000), (5, 3)], [1, 20, 0, 1, 6]
    nt = sum(counts)
    verts = rng.uniform(-1, 1, (3 * nt, 3)).astype(np.float32)
    idx = np.arange(3 * nt, dtype=np.uint32).reshape(-1, 3)
    uv = rng.uniform(0, 1, (nt, 6)).astype(np.float32)
    uv[nt - 6:] = 2.0                                     # the last object's cover nothing
    if groups == 2:
        uv[0] = (0, 0, 1, 1, 1, 0.9998)
        uv[21] = (0, 1, 1, 0, 0.9997, 0)
    ids = rng.permutation(nt).astype(np.uint32)
    gs = B.GatherScene(verts, idx, np.zeros_like(verts), np.full(nt, 3, np.uint8), np.zeros((nt, 8), np.float32), [])
    objs = (N.BakeObject * len(sizes))()
    ref_t, ref_s, keep, t, slot = [], [], [], 0, 0
    for k, ((w, h), c) in enumerate(zip(sizes, counts)):
        u, i = np.ascontiguousarray(uv[t:t + c]), np.ascontiguousarray(ids[t:t + c])
        keep += [u, i]
        objs[k] = N.BakeObject(u.ctypes.data, i.ctypes.data, c, w, h)
        tex, sub = B.rasterize(u, i, w, h, k, slot)
        tex = tex.copy()
        tex["sub_begin"] += sum(len(q) for q in ref_s)
        ref_t.append(tex)
        ref_s.append(sub)
        t += c
        slot += w * h
    zero = np.zeros((nt, 3), np.float32)
    h = ctypes.c_void_p()
    N.check(N.lib().lsg_bake_create(gs._h, objs, len(sizes), zero.ctypes.data, zero.ctypes.data, ctypes.byref(h)), "lsg_bake_create")
    try:
        inf = N.BakeInfo()
        N.check(N.lib().lsg_bake_info_get(h, ctypes.byref(inf)), "info")
        rt, rs = np.concatenate(ref_t), np.concatenate(ref_s)
        assert (inf.num_texels, inf.num_subtexels) == (len(rt), len(rs)) and len(rt)
        gt, gs_ = np.empty_like(rt), np.empty_like(rs)
        N.check(N.lib().lsg_memcpy_d2h(gt.ctypes.data, inf.texels, gt.nbytes), "d2h")
        N.check(N.lib().lsg_memcpy_d2h(gs_.ctypes.data, inf.subtexels, gs_.nbytes), "d2h")
        assert gt.tobytes() == rt.tobytes() and gs_.tobytes() == rs.tobytes()
    finally:
        N.lib().lsg_bake_destroy(h)
