"""The collider cache on the GPU (lsg_collider_create_cached / save / load): a tree loaded from
its file equals the tree that was built, node for node, with the same leaf order and the same
hits; a file of another mesh, another build setting or a damaged file is not used (the tree is
rebuilt and the file rewritten); small trees and "*" write no file."""
import os

import numpy as np
import pytest

from lightsprintsdk_amd import scenes as S

pytestmark = pytest.mark.gpu


def _files(d):
    return sorted(f for f in os.listdir(d) if f.endswith(".lsgbvh"))


def _same_tree(a, b, rays):
    ia, ib = a.info(), b.info()
    for f in ("num_triangles", "num_valid", "num_nodes", "root_ref", "depth", "leaf_size", "num_nodes4", "stack_need"):
        assert getattr(ia, f) == getattr(ib, f), f
    ta, tb = a.download_tree(), b.download_tree()
    np.testing.assert_array_equal(ta["nodes"].view(np.uint32), tb["nodes"].view(np.uint32))
    np.testing.assert_array_equal(ta["prim"], tb["prim"])
    ha, fa = a.intersect_batch(rays)
    hb, fb = b.intersect_batch(rays)
    np.testing.assert_array_equal(ha.view(np.uint8), hb.view(np.uint8))
    np.testing.assert_array_equal(fa, fb)


def test_gpu_cache_round_trip(gpu, tmp_path):
    from lightsprintsdk_amd.collider import RRCollider
    V, I = S.icosphere(S.ICOSPHERE_100K_FREQUENCY, seed=1)
    R = S.random_rays(V, 200_000, seed=5)
    loc = str(tmp_path) + "/"
    a = RRCollider.create(V, I, cacheLocation=loc)
    assert not a.from_cache and len(_files(tmp_path)) == 1
    b = RRCollider.create(V, I, cacheLocation=loc)
    assert b.from_cache
    _same_tree(a, b, R)
    print(f"build {a.info().build_ms:.1f} ms, load {b.info().build_ms:.1f} ms", flush=True)
    # explicit save / load
    path = str(tmp_path / "tree.bin")
    a.save(path)
    c = RRCollider.load(V, I, path)
    _same_tree(a, c, R)
    # LBVH-only and another leaf size are other trees: rebuilt and written again
    d = RRCollider.create(V, I, cacheLocation=loc, lbvh_only=True)
    assert not d.from_cache
    e = RRCollider.create(V, I, cacheLocation=loc, lbvh_only=True)
    assert e.from_cache
    _same_tree(d, e, R[:20_000])
    f = RRCollider.create(V, I, cacheLocation=loc, leaf_size=4)
    assert not f.from_cache
    g = RRCollider.create(V, I, cacheLocation=loc, leaf_size=4)
    assert g.from_cache and g.info().leaf_size == 4
    _same_tree(f, g, R[:20_000])
    for col in (a, b, c, d, e, f, g):
        col.close()


def test_gpu_cache_refuses_other_mesh_and_damage(gpu, tmp_path):
    from lightsprintsdk_amd import native as N
    from lightsprintsdk_amd.collider import RRCollider
    V, I = S.icosphere(20, seed=2)
    R = S.random_rays(V, 20_000, seed=6)
    loc = str(tmp_path) + "/"
    a = RRCollider.create(V, I, cacheLocation=loc)
    path = tmp_path / _files(tmp_path)[0]
    # the same triangle count with one vertex moved: another mesh, another file name
    V2 = V.copy()
    V2[7] += 0.01
    b = RRCollider.create(V2, I, cacheLocation=loc)
    assert not b.from_cache and len(_files(tmp_path)) == 2
    with pytest.raises(N.LsgError):
        RRCollider.load(V2, I, str(path))          # the first mesh's file
    # one flipped payload byte: refused, rebuilt, rewritten
    raw = bytearray(path.read_bytes())
    raw[len(raw) // 2] ^= 0x40
    path.write_bytes(bytes(raw))
    with pytest.raises(N.LsgError):
        RRCollider.load(V, I, str(path))
    c = RRCollider.create(V, I, cacheLocation=loc)
    assert not c.from_cache
    d = RRCollider.create(V, I, cacheLocation=loc)
    assert d.from_cache
    _same_tree(a, d, R)
    # a truncated file
    path.write_bytes(path.read_bytes()[:-100])
    with pytest.raises(N.LsgError):
        RRCollider.load(V, I, str(path))
    for col in (a, b, c, d):
        col.close()


def _payload_sum(p):
    """The tree files' payload checksum."""
    mask, prime = (1 << 64) - 1, 0x100000001b3
    h = [0xcbf29ce484222325, 0x84222325cbf29ce4, 0x9e3779b97f4a7c15, 0xc2b2ae3d27d4eb4f]
    n = len(p) // 32 * 32
    for k, w in enumerate(np.frombuffer(p[:n], "<u8").tolist()):
        h[k & 3] = (h[k & 3] ^ w) * prime & mask
    r = h[0] ^ (h[1] * 3 & mask) ^ (h[2] * 5 & mask) ^ (h[3] * 7 & mask)
    for b in p[n:]:
        r = (r ^ b) * prime & mask
    return (r ^ len(p)) * prime & mask


@pytest.mark.parametrize("what", ["sound", "cycle", "node_past_end", "leaf_past_end"])
def test_gpu_cache_walks_the_stored_tree(gpu, tmp_path, what):
    """A file whose checksum is right but whose 4-wide tree could lead the traversal out of
    its arrays is refused before it reaches the GPU."""
    from lightsprintsdk_amd import native as N
    from lightsprintsdk_amd.collider import RRCollider
    V, I = S.icosphere(8, seed=2)
    a = RRCollider.create(V, I)
    path = str(tmp_path / "t.lsgbvh")
    a.save(path)
    n4 = a.info().num_nodes4
    a.close()
    raw = bytearray(open(path, "rb").read())
    head = 8 + 4 + 4 + 20 + 4 + 8          # magic, version, header bytes, mesh hash, padding, then past the checksum
    head_bytes = int.from_bytes(raw[12:16], "little")
    refs = len(raw) - 128 * n4 + 96        # child refs of the 4-wide root
    assert _payload_sum(bytes(raw[head_bytes:])) == int.from_bytes(raw[head - 8:head], "little")
    bad = dict(sound=None, cycle=0, node_past_end=n4, leaf_past_end=-(1 << 31) | (len(I) << 4))[what]
    if bad is not None:
        raw[refs:refs + 4] = int(bad & 0xFFFFFFFF).to_bytes(4, "little")
    raw[head - 8:head] = _payload_sum(bytes(raw[head_bytes:])).to_bytes(8, "little")
    open(path, "wb").write(raw)
    if bad is None:
        RRCollider.load(V, I, path).close()
        return
    with pytest.raises(N.LsgError, match="4-wide tree"):
        RRCollider.load(V, I, path)


@pytest.mark.parametrize("field,value", [("stack_need", 0xFFFFFFFF), ("stack_need", 32), ("stack_need", -1),
                                         ("depth", 0xFFFFFFFF), ("depth", 64)])
def test_gpu_cache_stack_claims(gpu, tmp_path, field, value):
    """The header's depth and stack entries are outside the checksum: a file that states more than
    the traversal stack holds, however large the number, or fewer entries than its tree needs (-1:
    one less) is refused before it reaches the GPU."""
    from lightsprintsdk_amd import native as N
    from lightsprintsdk_amd.collider import RRCollider
    V, I = S.icosphere(8, seed=2)
    a = RRCollider.create(V, I)
    path = str(tmp_path / "t.lsgbvh")
    a.save(path)
    info = a.info()
    a.close()
    assert info.depth <= 31
    raw = bytearray(open(path, "rb").read())
    at = dict(depth=76, stack_need=80)[field]
    assert int.from_bytes(raw[at:at + 4], "little") == getattr(info, field)
    if value == -1:
        value = info.stack_need - 1
    raw[at:at + 4] = value.to_bytes(4, "little")
    open(path, "wb").write(raw)
    with pytest.raises(N.LsgError, match="stack"):
        RRCollider.load(V, I, path)


@pytest.mark.parametrize("lbvh_only", [False, True])
def test_gpu_cache_saves_a_loaded_tree(gpu, tmp_path, lbvh_only):
    """A loaded tree saved again is the file it came from, byte for byte, whichever tree it is."""
    from lightsprintsdk_amd.collider import RRCollider
    V, I = S.icosphere(16, seed=3)
    a = RRCollider.create(V, I, lbvh_only=lbvh_only)
    p, q = str(tmp_path / "a.lsgbvh"), str(tmp_path / "b.lsgbvh")
    a.save(p)
    b = RRCollider.load(V, I, p)
    b.save(q)
    assert open(p, "rb").read() == open(q, "rb").read()
    c = RRCollider.load(V, I, q)
    _same_tree(a, c, S.random_rays(V, 5_000, seed=8))
    for col in (a, b, c):
        col.close()


def test_gpu_cache_saves_another_collapse(gpu, tmp_path):
    """A file whose 4-wide tree is a sound one, but not the one this build collapses to (its nodes all of
    two children: the BVH2 itself), loads, and saving it states the tree that is written."""
    from lightsprintsdk_amd.collider import RRCollider
    V, I = S.icosphere(8, seed=2)
    a = RRCollider.create(V, I)
    p, q = str(tmp_path / "a.lsgbvh"), str(tmp_path / "b.lsgbvh")
    a.save(p)
    raw = bytearray(open(p, "rb").read())
    info, head_bytes = a.info(), int.from_bytes(raw[12:16], "little")
    n, at = info.num_nodes, head_bytes + 4 * info.num_valid
    nodes = np.frombuffer(bytes(raw[at:at + 64 * n]), np.float32).reshape(n, 16)
    wide = np.zeros((n, 8, 4), np.float32)
    wide[:, :6, 0], wide[:, :6, 1] = nodes[:, :6], nodes[:, 6:12]
    refs = np.full((n, 4), 0x7FFFFFFE, np.int32)
    refs[:, :2] = nodes[:, 12:14].view(np.int32)
    wide[:, 6] = refs.view(np.float32)
    payload = bytes(raw[head_bytes:at + 64 * n]) + wide.tobytes()
    raw = raw[:head_bytes] + payload
    raw[72:76] = n.to_bytes(4, "little")                       # 4-wide nodes
    raw[80:84] = info.depth.to_bytes(4, "little")              # stack entries: one a level at most
    raw[40:48] = _payload_sum(payload).to_bytes(8, "little")
    raw[120:128] = len(payload).to_bytes(8, "little")
    open(p, "wb").write(raw)
    b = RRCollider.load(V, I, p)
    assert b.info().num_nodes4 == n != info.num_nodes4
    R = S.random_rays(V, 5_000, seed=8)
    ha, hb = a.intersect_batch(R), b.intersect_batch(R)
    np.testing.assert_array_equal(ha[0].view(np.uint8), hb[0].view(np.uint8))
    b.save(q)
    c = RRCollider.load(V, I, q)
    _same_tree(a, c, R)
    for col in (a, b, c):
        col.close()


@pytest.mark.parametrize("what", ["cycle", "root_ref", "two_parents", "node_past_end", "leaf_past_end", "root", "root_leaf"])
def test_gpu_cache_checks_the_stored_bvh2(gpu, tmp_path, what):
    """Saving a loaded tree walks its BVH2 on the GPU: a file with the right checksum whose BVH2 could
    lead out of its arrays, or is no tree, is refused before it reaches the GPU."""
    from lightsprintsdk_amd import native as N
    from lightsprintsdk_amd.collider import RRCollider
    V, I = S.icosphere(8, seed=2)
    a = RRCollider.create(V, I)
    path = str(tmp_path / "t.lsgbvh")
    a.save(path)
    info = a.info()
    a.close()
    raw = bytearray(open(path, "rb").read())
    head_bytes = int.from_bytes(raw[12:16], "little")
    n, nodes = info.num_nodes, head_bytes + 4 * info.num_valid
    assert info.root_ref == 0
    ref = lambda i, k: nodes + 64 * i + 48 + 4 * k

    def inner(i):                                    # an inner child ref of node i, or None
        for k in range(2):
            c = int.from_bytes(raw[ref(i, k):ref(i, k) + 4], "little", signed=True)
            if c >= 0:
                return ref(i, k), c
    deep = next(i for i in range(n - 1, 0, -1) if inner(i))
    at, child = inner(deep)
    other = next(inner(i)[1] for i in range(n) if inner(i) and inner(i)[1] != child)
    where, bad = dict(cycle=(at, deep), root_ref=(at, 0), two_parents=(at, other), node_past_end=(at, n),
                      leaf_past_end=(at, -(1 << 31) | (len(I) << 4)), root=(84, n), root_leaf=(84, -(1 << 31)))[what]
    raw[where:where + 4] = int(bad & 0xFFFFFFFF).to_bytes(4, "little")
    raw[40:48] = _payload_sum(bytes(raw[head_bytes:])).to_bytes(8, "little")
    open(path, "wb").write(raw)
    with pytest.raises(N.LsgError, match="2-wide tree"):
        RRCollider.load(V, I, path)


def test_gpu_cache_small_trees_and_star(gpu, tmp_path):
    from lightsprintsdk_amd.collider import RRCollider
    v = np.float32([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]])
    i = np.uint32([[0, 1, 2], [0, 2, 3]])
    a = RRCollider.create(v, i, cacheLocation=str(tmp_path) + "/")
    assert not _files(tmp_path)                    # under 1024 bytes: not written
    V, I = S.icosphere(20, seed=2)
    b = RRCollider.create(V, I, cacheLocation="*")
    assert not b.from_cache and not _files(tmp_path)
    a.close()
    b.close()


def test_gpu_cache_large_mesh_load_time(gpu, tmp_path):
    """The 10M-triangle city: the cached tree skips the GPU build (LBVH, SAH rebuild, collapse)."""
    import time
    from lightsprintsdk_amd.collider import RRCollider
    sc = S.city_terrain(seed=5, sun_direction=S.sun_sweep(0, 60))
    loc = str(tmp_path) + "/"
    t0 = time.perf_counter()
    a = RRCollider.create(sc.verts, sc.idx, cacheLocation=loc)
    t1 = time.perf_counter()
    b = RRCollider.create(sc.verts, sc.idx, cacheLocation=loc)
    t2 = time.perf_counter()
    assert not a.from_cache and b.from_cache
    size = os.path.getsize(tmp_path / _files(tmp_path)[0])
    print(f"city {sc.ntri} triangles: build + write {t1 - t0:.2f} s (tree {a.info().build_ms:.0f} ms), "
          f"load {t2 - t1:.2f} s (tree {b.info().build_ms:.0f} ms), file {size / 1e6:.0f} MB", flush=True)
    R = S.random_rays(sc.verts, 100_000, seed=7)
    _same_tree(a, b, R)
    a.close()
    b.close()
