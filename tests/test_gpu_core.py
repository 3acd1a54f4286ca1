"""GPU parity of the LBVH build, traversal and luminance histogram against the
CPU oracle, called through the C ABI (librtgl1_amd.so).

Integer and index outputs (Morton codes, sort order, topology, node child
references, primitive ids, histogram bins) must be bit-exact; FP32 outputs of
the same IEEE operation sequence (boxes, hit t/u/v, average luminance) must be
equal as floats.
"""
import ctypes as C

import numpy as np
import pytest

from raytracedgl1_amd import ffi, scenes
from raytracedgl1_amd.ffi import (HIT_DTYPE, RAY_DTYPE, RG_EXT_MISS, RG_EXT_TRACE_ANY_HIT, RG_EXT_TRACE_COLLECT_STATS,
                                  RG_EXT_TRACE_CULL_FRONT_FACE, Bvh, DeviceArray)

pytestmark = pytest.mark.gpu


def _random_tris(n, seed, spread=10.0, size=1.0):
    r = np.random.default_rng(seed)
    c = r.uniform(-spread, spread, (n, 1, 3))
    return (c + r.uniform(-size, size, (n, 3, 3))).reshape(n, 9).astype(np.float32)


def _gpu_bvh(tris, leaf=3):
    d = DeviceArray.from_numpy(tris)
    b = Bvh()
    b.build(d, len(tris), leaf)
    return b, d


def _assert_same_bvh(g, o):
    assert g["n"] == o["n"]
    assert np.array_equal(g["codes"], o["codes"])
    assert np.array_equal(g["scene_min"], o["scene_min"])
    assert np.array_equal(g["scene_max"], o["scene_max"])
    assert np.array_equal(g["sorted_idx"], o["sorted_idx"])
    assert np.array_equal(g["children"], o["children"])
    assert np.array_equal(g["bounds"], o["bounds"])  # float equality (+0 == -0)
    assert g["node_count"] == o["node_count"]
    for f in ("lo_x", "hi_x", "lo_y", "hi_y", "lo_z", "hi_z"):
        assert np.array_equal(g["nodes"][f], o["nodes"][f]), f
    assert np.array_equal(g["nodes"]["child"], o["nodes"]["child"])


@pytest.mark.parametrize("n,leaf", [(1, 3), (2, 1), (3, 3), (7, 1), (64, 3), (1000, 4), (4097, 2), (70000, 3)])
def test_lbvh_bit_exact_random(gpu, oracle, n, leaf):
    print(f"lbvh random n={n} leaf={leaf}", flush=True)
    tris = _random_tris(n, seed=n)
    b, _ = _gpu_bvh(tris, leaf)
    _assert_same_bvh(b.download(), oracle.bvh(tris, leaf).download())


def test_lbvh_bit_exact_duplicates(gpu, oracle):
    base = _random_tris(1, seed=5)
    tris = np.repeat(base, 5000, axis=0)
    tris[:, 0] += np.linspace(-1e-3, 1e-3, 5000, dtype=np.float32)
    b, _ = _gpu_bvh(tris, 3)
    _assert_same_bvh(b.download(), oracle.bvh(tris, 3).download())


@pytest.mark.parametrize("kind", ["even", "nested"])
@pytest.mark.parametrize("n", [255, 257, 1024, 2049, 32768, 32769, 50001])
def test_lbvh_bit_exact_at_run_and_tile_edges(gpu, oracle, n, kind):
    """Sizes about the hierarchy's runs (256 and 1024 triangles), the sort's
    tiles (2048) and the change between the runs (32768); "nested" halves the
    distances again and again towards one place with thousands of equal
    triangles, which makes the longest root paths across runs."""
    tris = _random_tris(n, seed=n)
    if kind == "nested":
        r = np.random.default_rng(n)
        k = np.minimum(r.integers(0, 40, n), 22)  # 45% of them at the last distance
        tris = np.broadcast_to(np.float32([0, 0, 0, 1e-3, 0, 0, 0, 1e-3, 0]), (n, 9)) + np.repeat(np.float32(2.0) ** -k[:, None], 9, 1)
        tris = np.ascontiguousarray(tris, np.float32)
    for leaf in (1, 3):
        b, _ = _gpu_bvh(tris, leaf)
        _assert_same_bvh(b.download(), oracle.bvh(tris, leaf).download())


def test_lbvh_bit_exact_terrain_boxes(gpu, oracle):
    s = scenes.terrain_boxes_scene()
    b, _ = _gpu_bvh(s.tris, 3)
    _assert_same_bvh(b.download(), oracle.bvh(s.tris, 3).download())


def test_lbvh_bit_exact_terrain_spheres_1m(gpu, oracle):
    print("lbvh terrain-spheres 1M tris", flush=True)
    s = scenes.terrain_spheres_scene()
    b, _ = _gpu_bvh(s.tris, 3)
    _assert_same_bvh(b.download(), oracle.bvh(s.tris, 3).download())


def test_lbvh_rebuild_is_deterministic_and_order_invariant(gpu):
    # Tests/RtglTest.cpp:510-511 shuffles primitives because upload order must
    # not change the image: the set of leaf triangles and the tree shape are
    # the same after a permutation that keeps ids stable by construction.
    s = scenes.terrain_boxes_scene()
    b, d = _gpu_bvh(s.tris, 3)
    first = b.download()
    b.build(d, s.n, 3)
    again = b.download()
    _assert_same_bvh(first, again)


def _trace_gpu(b, rays, flags):
    dr = DeviceArray.from_numpy(rays)
    dh = DeviceArray(len(rays), HIT_DTYPE)
    b.trace(dr, len(rays), dh, flags)
    out = dh.download()
    assert b.trace_errors() == 0, "traversal reported a dropped stack entry or a step-limit stop"
    return out


def _assert_same_hits(g, o, any_hit=False):
    assert np.array_equal(g["prim"] == RG_EXT_MISS, o["prim"] == RG_EXT_MISS)
    if any_hit:
        return
    assert np.array_equal(g["prim"], o["prim"])
    for f in ("t", "u", "v"):
        assert np.array_equal(g[f], o[f]), f


@pytest.mark.parametrize("flags", [0, RG_EXT_TRACE_CULL_FRONT_FACE, RG_EXT_TRACE_ANY_HIT])
def test_trace_bit_exact_terrain_boxes_primary(gpu, oracle, flags):
    print(f"trace terrain-boxes flags={flags}", flush=True)
    s = scenes.terrain_boxes_scene()
    rays = scenes.primary_rays(scenes.terrain_boxes_camera(), 640, 360)
    b, _ = _gpu_bvh(s.tris, 3)
    _assert_same_hits(_trace_gpu(b, rays, flags), oracle.bvh(s.tris, 3).trace(rays, flags),
                      any_hit=bool(flags & RG_EXT_TRACE_ANY_HIT))


@pytest.mark.parametrize("flags", [0, RG_EXT_TRACE_ANY_HIT])
def test_trace_visit_counts_match_oracle(gpu, oracle, flags):
    # Node visits and triangle tests are the traversal's algorithmic work
    # (they price its memory traffic); the GPU must visit exactly what the
    # oracle's traversal of the same tree visits, for primary and random rays.
    print(f"trace stats flags={flags}", flush=True)
    s = scenes.terrain_boxes_scene()
    r = np.random.default_rng(5)
    rnd = np.zeros(20000, RAY_DTYPE)
    rnd["origin"] = r.uniform(-30, 30, (20000, 3)) + np.array([0, 4, 0])
    d = r.normal(size=(20000, 3))
    rnd["direction"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rnd["tmax"] = 1000.0
    rays = np.concatenate([scenes.primary_rays(scenes.terrain_boxes_camera(), 640, 360), rnd])
    b, _ = _gpu_bvh(s.tris, 3)
    g = _trace_gpu(b, rays, flags | RG_EXT_TRACE_COLLECT_STATS)
    nodes, tris = b.trace_stats()
    o, onodes, otris = oracle.bvh(s.tris, 3).trace(rays, flags, stats=True)
    _assert_same_hits(g, o, any_hit=bool(flags & RG_EXT_TRACE_ANY_HIT))
    assert (nodes, tris) == (onodes, otris)
    assert nodes >= len(rays)
    # without the flag the counters are not touched
    _trace_gpu(b, rays[:100], flags)
    assert b.trace_stats() == (nodes, tris)


def test_trace_matches_bruteforce_fp64(gpu, oracle):
    s = scenes.terrain_boxes_scene()
    rays = scenes.primary_rays(scenes.terrain_boxes_camera(), 640, 360)[::29]
    b, _ = _gpu_bvh(s.tris, 3)
    g = _trace_gpu(b, rays, 0)
    t, u, v, p = oracle.bruteforce(s.tris, rays, 0)
    miss = p == RG_EXT_MISS
    assert np.array_equal(g["prim"] == RG_EXT_MISS, miss)
    h = ~miss
    assert (np.abs(g["t"][h] - t[h]) / t[h]).max() < 1e-5
    diff = h & (g["prim"] != p)
    assert np.all(np.abs(g["t"][diff] - t[diff]) <= 1e-6 * t[diff] + 1e-7)


def test_trace_random_rays_and_empty(gpu, oracle):
    s = scenes.terrain_boxes_scene()
    r = np.random.default_rng(3)
    rays = np.zeros(50000, RAY_DTYPE)
    rays["origin"] = r.uniform(-40, 40, (50000, 3))
    d = r.normal(size=(50000, 3))
    rays["direction"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays["tmin"] = r.uniform(0, 1, 50000)
    rays["tmax"] = r.uniform(1, 100, 50000)
    b, _ = _gpu_bvh(s.tris, 3)
    _assert_same_hits(_trace_gpu(b, rays, 0), oracle.bvh(s.tris, 3).trace(rays, 0))
    # zero rays is a no-op
    dh = DeviceArray(1, HIT_DTYPE)
    dr = DeviceArray(1, RAY_DTYPE)
    b.trace(dr, 0, dh, 0)


def test_trace_terrain_spheres_1080p(gpu, oracle):
    print("trace terrain-spheres 1080p", flush=True)
    s = scenes.terrain_spheres_scene()
    rays = scenes.primary_rays(scenes.orbit_camera(0), 1920, 1080)
    b, _ = _gpu_bvh(s.tris, 3)
    g = _trace_gpu(b, rays, 0)
    ob = oracle.bvh(s.tris, 3)
    sub = np.arange(0, len(rays), 7)
    _assert_same_hits(g[sub], ob.trace(rays[sub], 0))
    # size-independent property over the full image: hit points lie on the hit triangle
    h = g["prim"] != RG_EXT_MISS
    assert h.mean() > 0.5
    tri = s.tris.reshape(-1, 3, 3)[g["prim"][h]].astype(np.float64)
    u, v = g["u"][h, None].astype(np.float64), g["v"][h, None].astype(np.float64)
    pb = (1 - u - v) * tri[:, 0] + u * tri[:, 1] + v * tri[:, 2]
    pr = rays["origin"][h] + rays["direction"][h] * g["t"][h, None]
    assert np.abs(pb - pr).max() < 1e-2


def _edge_scene(kind, r):
    """Triangles at the limits of the traversal nodes' grids, and their spread."""
    if kind.startswith("n"):  # leaves per node, and nodes of one child
        return _random_tris(int(kind[1:]), seed=int(kind[1:])), 10.0
    t = _random_tris(3000, seed=7)
    if kind == "flat":  # no extent on one axis
        t[:, 1::3] = 2.5
    elif kind == "thin":  # extents of 1e-30 and 0 beside 10
        t[:, 1::3] = np.where(r.random((3000, 3)) < 0.5, 0.0, 1e-30)
    elif kind == "far":  # 20,000 units out: a grid step is a few units in the last place
        t += np.float32(20000.0)
    elif kind == "huge":
        t *= np.float32(1e10)
    elif kind == "broken":  # triangles that nothing hits, in every part of the tree
        bad = r.random(3000) < 0.03
        t[bad, 4] = np.where(r.random(bad.sum()) < 0.5, np.inf, np.nan)
        t[::701] = np.nan
    return t, 10.0


@pytest.mark.parametrize("kind", ["n1", "n2", "n7", "n8", "n9", "n15", "n57", "n500", "flat", "thin", "far", "huge", "broken"])
def test_traversal_nodes_at_their_limits(gpu, kind):
    """Hits through the traversal's grid nodes against the walk of the
    published FP32 nodes: the same, or a hit that the FP32 boxes' rounding
    hid, nearer by rounding (1e-5 t bounds the triangle test's error) or as
    near with a lower id.  At most 1e-4 of the rays differ, but where all
    triangles lie in one plane and overlap: there every ray meets several
    within rounding of each other, and a ray in that plane meets them edge
    on, where the triangle test is all rounding and no bound on t holds."""
    print(f"traversal nodes {kind}", flush=True)
    r = np.random.default_rng(11)
    tris, spread = _edge_scene(kind, r)
    finite = tris[np.isfinite(tris).all(1)].reshape(-1, 3, 3)
    n = 60000
    rays = np.zeros(n, RAY_DTYPE)
    target = finite[r.integers(0, len(finite), n)].mean(1).astype(np.float64)
    scale = max(1.0, np.abs(finite).max() if kind == "huge" else spread)
    origin = target + r.normal(size=(n, 3)) * scale
    if kind in ("flat", "thin"):
        origin[: n // 4, 1] = finite[0, 0, 1]  # in the plane of the triangles
    d = target - origin + r.normal(size=(n, 3)) * scale * 0.02
    d[: n // 8, r.integers(0, 3)] = 0.0  # parallel to a slab
    d[n // 8: n // 6, :2] = 0.0
    rays["origin"] = origin
    rays["direction"] = d / np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-30)
    rays["tmin"] = np.where(r.random(n) < 0.5, 0.0, 0.1 * scale)
    rays["tmax"] = np.where(r.random(n) < 0.2, np.inf, 100.0 * scale)
    b, _ = _gpu_bvh(tris, 1)
    g = _trace_gpu(b, rays, 0)
    v = _trace_gpu(b, rays, RG_EXT_TRACE_COLLECT_STATS)
    assert (v["prim"] != RG_EXT_MISS).mean() > 0.02
    diff = (g["prim"] != v["prim"]) | (g["t"] != v["t"]) | (g["u"] != v["u"]) | (g["v"] != v["v"])
    assert kind in ("flat", "thin") or diff.mean() <= 1e-4, diff.sum()
    near = diff & ((np.arange(n) >= n // 4) if kind in ("flat", "thin") else True)
    assert (v["t"][near] - g["t"][near] <= 1e-5 * g["t"][near]).all()
    assert ((g["t"] < v["t"]) | ((g["t"] == v["t"]) & (g["prim"] < v["prim"])))[diff].all()
    occ = _trace_gpu(b, rays, RG_EXT_TRACE_ANY_HIT)["prim"] != RG_EXT_MISS
    assert np.array_equal(occ, g["prim"] != RG_EXT_MISS)


def _nested_clusters():
    """20 clusters of 64 triangles at halving distances from the origin, each
    triangle as large as its cluster: boxes within boxes, and from the origin
    outwards every cluster lies behind the ones nested in it."""
    r = np.random.default_rng(3)
    out = []
    for k in range(20):
        v = r.uniform(-1, 1, (64, 3, 3))
        out.append((r.uniform(0.55, 0.95, (64, 1, 3)) + 0.4 * (v - v.mean(1, keepdims=True))) * 2.0 ** -k)
    return np.concatenate(out).reshape(-1, 9).astype(np.float32)


def _deepest_group_stack(b, tris, origin, direction):
    """The traversal restated for one ray over the same keys (the scene is a
    cube): the binary tree collapsed by area, subtrees of up to 8 triangles
    last, and the most groups that wait on its stack."""
    ch, bd, I = b["children"], b["bounds"], b["n"] - 1
    size = np.ones(2 * I + 1, int)
    order = [0]
    for x in order:
        order += [int(c) for c in ch[x] if c < I]
    for x in reversed(order):
        size[x] = size[ch[x]].sum()
    d = bd[:, 3:] - bd[:, :3]
    area = d[:, 0] * d[:, 1] + d[:, 1] * d[:, 2] + d[:, 2] * d[:, 0]

    def children(x):
        kids = [int(c) for c in ch[x]]
        while True:
            opens = [i for i, c in enumerate(kids) if c < I and size[c] > 8 and len(kids) < 8] or \
                    [i for i, c in enumerate(kids) if c < I and size[c] - 1 <= 8 - len(kids)]
            if not opens:
                return kids
            i = max(opens, key=lambda i: area[kids[i]])
            kids[i:i + 1] = [int(c) for c in ch[kids[i]]]

    best, stack, group, deepest = np.inf, [], [0], 0
    while group or stack:
        if not group:
            group = stack.pop()
        hit = []
        for c in children(group.pop(0)):
            t = (bd[c].reshape(2, 3) - origin) / direction
            near, far = max(t.min(0).max(), 0.0), min(t.max(0).min(), best)
            if near <= far and c < I:
                hit.append((near, c))
            elif near <= far:
                p = tris[b["sorted_idx"][c - I]].reshape(3, 3).astype(np.float64)
                m = np.stack([p[1] - p[0], p[2] - p[0], -direction], 1)
                u, v, t = np.linalg.solve(m, origin - p[0])
                best = t if u >= 0 and v >= 0 and u + v <= 1 and 0 <= t < best else best
        if hit:
            if group:
                stack.append(group)
                deepest = max(deepest, len(stack))
            group = [c for _, c in sorted(hit)]
    return deepest


def test_traversal_stack_beyond_lds(gpu, oracle):
    """Rays that leave more groups waiting than the stack has in LDS (8, 12 or
    16 of them by the tuning, 12 of 32 in the variant without allocations):
    the rest goes through global memory.  Against the oracle's walk, whose
    stack has no end (these rays need up to 140 entries of one child each)."""
    tris = _nested_clusters()
    r = np.random.default_rng(1)
    n = 40000
    rays = np.zeros(n, RAY_DTYPE)
    rays["origin"] = 1e-7
    d = r.uniform(0.6, 1.4, (n, 3))
    rays["direction"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays["tmax"] = 100.0
    o = oracle.bvh(tris, 1)
    ob = o.download()
    deep = [_deepest_group_stack(ob, tris, np.full(3, 1e-7), rays["direction"][k].astype(np.float64)) for k in range(20)]
    print(f"groups on the stack: {min(deep)} to {max(deep)}", flush=True)
    assert 17 <= max(deep) <= 32
    b, _ = _gpu_bvh(tris, 1)
    v = o.trace(rays, 0)
    assert (v["prim"] != RG_EXT_MISS).mean() > 0.5
    dr, dh = DeviceArray.from_numpy(rays), DeviceArray(n, HIT_DTYPE)
    for _ in range(6):
        _assert_same_hits(_trace_gpu(b, rays, 0), v)
        _assert_same_hits(_trace_gpu(b, rays, RG_EXT_TRACE_ANY_HIT), v, any_hit=True)
        for flags in (0, RG_EXT_TRACE_ANY_HIT):
            ffi.call("rgExtTraceRaysNoAlloc", b.h, dr.ptr, n, dh.ptr, flags, None)
            _assert_same_hits(dh.download(), v, any_hit=bool(flags))
            assert b.trace_errors() == 0
        print(f"  next: {b.autotune(dr, n, dh).stackLdsEntries} words in LDS", flush=True)


@pytest.mark.parametrize("kind", ["n9", "n57", "n500", "flat", "thin", "far", "huge", "broken"])
def test_traversal_nodes_against_a_loop_over_all_triangles(gpu, oracle, kind):
    """The same scenes against the FP64 loop, with rays at the middle of a
    triangle from outside the plane of flat scenes: a ray that hits a triangle
    there hits it or a nearer one."""
    print(f"loop over all triangles {kind}", flush=True)
    r = np.random.default_rng(29)
    tris, spread = _edge_scene(kind, r)
    n = 5000
    good = np.flatnonzero(np.isfinite(tris).all(1))
    scale = max(1.0, np.abs(tris[good]).max() if kind == "huge" else spread)
    t = tris[good[r.integers(0, len(good), n)]].reshape(n, 3, 3).astype(np.float64)
    target = (t * r.dirichlet([8, 8, 8], n)[..., None]).sum(1)
    nrm = np.cross(t[:, 1] - t[:, 0], t[:, 2] - t[:, 0])
    nrm /= np.maximum(np.linalg.norm(nrm, axis=1, keepdims=True), 1e-300)
    d = nrm * r.choice([-1.0, 1.0], (n, 1)) + r.normal(size=(n, 3)) * 0.3
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    rays = np.zeros(n, RAY_DTYPE)
    rays["origin"] = target - d * (r.uniform(0.5, 3.0, (n, 1)) * scale)
    rays["direction"] = d
    rays["tmax"] = 100.0 * scale
    tb, _, _, p = oracle.bruteforce(tris[good], rays)
    hit = p != RG_EXT_MISS
    p = np.where(hit, good[np.where(hit, p, 0)], RG_EXT_MISS)
    assert hit.mean() > 0.9
    v = tris[np.where(hit, p, good[0])].reshape(n, 3, 3).astype(np.float64)
    nrm = np.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0])
    cos = np.abs((nrm * d).sum(1)) / np.maximum(np.linalg.norm(nrm, axis=1), 1e-300)
    b, _ = _gpu_bvh(tris, 1)
    g = _trace_gpu(b, rays, 0)
    same = g["prim"] == p
    # One flat plane of overlapping triangles: any of those within rounding may
    # be the nearest.  Else a ray meets another triangle only at an edge.
    if kind not in ("flat", "thin"):
        assert (g["prim"] == p).mean() >= 0.999
    assert np.array_equal(g["prim"] != RG_EXT_MISS, hit)
    # A ray is placed on the triangle within a few roundings of its distance or
    # of the triangle's size, and the depth there by weights off by as much over the
    # triangle's height: across the plane 8 roundings times the aspect, along the
    # ray over the cosine.
    edge = np.linalg.norm(v - np.roll(v, 1, 1), axis=2).max(1)
    aspect = edge ** 2 / np.maximum(np.linalg.norm(np.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]), axis=1), 1e-300)
    err = (np.abs(g["t"] - tb) * cos / (np.maximum(np.abs(tb), edge) * aspect))[hit]
    print(f"  error at most {err.max() * 2.0 ** 24:.1f} roundings", flush=True)
    assert err.max() <= 8 * 2.0 ** -24


def _grid_wall():
    """3200 triangles side by side in the plane x = 0."""
    y, z = np.meshgrid(np.arange(40.0) - 20.0, np.arange(40.0) - 20.0, indexing="ij")
    p = [np.stack([np.zeros(1600), y.ravel() + a, z.ravel() + b], 1) for a, b in ((0, 0), (1, 0), (0, 1), (1, 1))]
    return np.concatenate([np.concatenate([p[0], p[1], p[2]], 1), np.concatenate([p[3], p[2], p[1]], 1)]).astype(np.float32)


@pytest.mark.parametrize("kind", ["wall", "soup", "axis"])
def test_boxes_behind_the_origin_and_beyond_the_range(gpu, oracle, kind):
    """Hits of both walks against an FP64 loop over all triangles: at negative
    distances (tmin < 0), where a slack on the far planes must not move them
    nearer, down to boxes without thickness; and along rays parallel to an axis
    on which the boxes reach out to 1e19, where distances overflow."""
    print(f"boxes {kind}", flush=True)
    r = np.random.default_rng(23)
    n = 20000
    rays = np.zeros(n, RAY_DTYPE)
    if kind == "axis":
        far = np.zeros((8, 3, 3))
        far[np.arange(8), :, np.arange(8) % 2] = np.repeat([1e19, -1e19], 4)[:, None]
        far += r.uniform(-1e13, 1e13, far.shape)
        tris = np.concatenate([_random_tris(300, 4, spread=4.0), far.reshape(8, 9).astype(np.float32)])
        rays["origin"] = r.uniform(-5, 5, (n, 3))
        rays["origin"][:50, 0] = 1e25  # outside, and nowhere
        rays["origin"][50:100, 1] = -np.inf
        rays["direction"] = r.choice([0.0, -0.0, 1e-30, -1e-30], (n, 3))
        rays["direction"][:, 2] = r.choice([-1.0, 1.0], n)
        rays["tmax"] = 1000.0
    else:
        tris = _grid_wall() if kind == "wall" else _random_tris(3000, 5, size=0.2)
        t = tris[r.integers(0, len(tris), n)].reshape(n, 3, 3).astype(np.float64)
        d = r.normal(size=(n, 3)) + np.array([4.0, 0.0, 0.0])
        d /= np.linalg.norm(d, axis=1, keepdims=True)
        dist = -(10.0 ** r.uniform(0, 5 if kind == "wall" else 3, n))
        rays["origin"] = (t * r.dirichlet([4, 4, 4], n)[..., None]).sum(1) - d * dist[:, None]
        rays["direction"] = d
        rays["tmin"] = dist * 1.5
        rays["tmax"] = np.where(r.random(n) < 0.5, 0.0, 100.0)
    b, _ = _gpu_bvh(tris, 1)
    tb, _, _, p = oracle.bruteforce(tris, rays)
    hit = p != RG_EXT_MISS
    v = tris[np.where(hit, p, 0)].reshape(n, 3, 3).astype(np.float64)
    nrm = np.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0])
    cos = np.abs((nrm * rays["direction"]).sum(1)) / np.linalg.norm(nrm, axis=1)
    assert hit.mean() > 0.3
    for flags in (0, RG_EXT_TRACE_COLLECT_STATS):
        g = _trace_gpu(b, rays, flags)
        same = g["prim"] == p
        # the FP32 triangle test and the FP64 one part at edges and ties only:
        # a ray is placed within some 1e-7 of its distance, of triangles of 1 (wall) and 0.2
        assert same.mean() >= 0.98, (flags, same.mean())
        assert (hit & (g["prim"] == RG_EXT_MISS)).mean() <= 5e-3, flags
        # that error (16 roundings of the distance bound it) across the plane,
        # along the ray: over the cosine of incidence
        assert (np.abs(g["t"] - tb) * cos <= 16 * 2.0 ** -24 * np.abs(tb) + 1e-6)[same & hit].all(), flags
    occ = _trace_gpu(b, rays, RG_EXT_TRACE_ANY_HIT)["prim"] != RG_EXT_MISS
    assert np.array_equal(occ, _trace_gpu(b, rays, 0)["prim"] != RG_EXT_MISS)


@pytest.mark.parametrize("n", [1, 5, 4097, 16383, 16385, 65537, 131073, 262145, 300001])
def test_launch_widths(gpu, n):
    """Ray counts about the change between the lanes per wave that take rays
    (powers of two times the resident waves): every ray has its hit, those of
    the walk over the published nodes."""
    print(f"launch width {n}", flush=True)
    s = scenes.terrain_boxes_scene()
    r = np.random.default_rng(n)
    rays = np.zeros(n, RAY_DTYPE)
    rays["origin"] = r.uniform(-30, 30, (n, 3)) + np.array([0, 8, 0])
    d = r.normal(size=(n, 3)) - np.array([0, 0.5, 0])
    rays["direction"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays["tmax"] = 1000.0
    b, _ = _gpu_bvh(s.tris, 1)
    v = _trace_gpu(b, rays, RG_EXT_TRACE_COLLECT_STATS)
    for _ in range(2):  # the second launch finds the counters of the first
        _assert_same_hits(_trace_gpu(b, rays, 0), v)
        _assert_same_hits(_trace_gpu(b, rays, RG_EXT_TRACE_ANY_HIT), v, any_hit=True)


def _free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert C.CDLL("libamdhip64.so.7").hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_published_bvh_memory(gpu):
    """What a published BVH keeps, per triangle: its own arrays, the
    traversal's tree (48 and some 25 bytes) and both builds' scratch, that of
    the traversal's tree mostly inside the arrays that are written last."""
    n = 1_000_000
    d = DeviceArray.from_numpy(_random_tris(n, 3, spread=300.0, size=0.5))
    _gpu_bvh(_random_tris(4, 1))
    b = Bvh()
    before = _free_bytes()
    for _ in range(2):  # a second build takes nothing more
        b.build(d, n, 3)
        per = (before - _free_bytes()) / n
        print(f"published BVH: {per:.0f} bytes a triangle", flush=True)
        assert 200 < per <= 410


def test_histogram_bit_exact(gpu, oracle):
    r = np.random.default_rng(11)
    w, h = 1920, 1080
    lum = np.exp(r.uniform(-12, 12, w * h)).astype(np.float32)
    lum[::97] = 0.0
    lum[::101] = np.nan
    lum[::103] = np.inf
    lum[1::89] = 0.001
    min_log, max_log = np.log2(np.exp2(-4.0) * 12.5 / 100), np.log2(np.exp2(12.0) * 12.5 / 100)
    d = DeviceArray.from_numpy(lum)
    dh = DeviceArray(256, np.uint32, zero=True)
    ffi.call("rgExtLuminanceHistogram", d.ptr, w, h, float(min_log), float(max_log), dh.ptr, None)
    g = dh.download()
    o = oracle.lum_histogram(lum, float(np.float32(min_log)), float(np.float32(max_log)))
    assert np.array_equal(g, o)
    assert g.sum() == w * h
    # average: equal to the oracle's FP32 evaluation, and the histogram is cleared
    davg = DeviceArray.from_numpy(np.array([0.5], np.float32))
    ffi.call("rgExtLuminanceAverage", dh.ptr, w * h, float(min_log), float(max_log), 0.016, 0, davg.ptr, None)
    ga = davg.download()[0]
    oa = oracle.lum_average(o, w * h, float(np.float32(min_log)), float(np.float32(max_log)), 0.016, False, 0.5)
    assert ga == np.float32(oa)
    assert np.all(dh.download() == 0)


def test_device_copy_kernel(gpu):
    a = np.random.default_rng(2).integers(0, 2**32, 4096 * 4 + 8, dtype=np.uint32)
    src = DeviceArray.from_numpy(a)
    dst = DeviceArray(a.shape, a.dtype, zero=True)
    ffi.call("rgExtCopyDeviceToDevice", dst.ptr, src.ptr, a.nbytes, None)
    assert np.array_equal(dst.download(), a)
    ffi.call("rgExtCopyDeviceToDevice", dst.ptr, src.ptr, 0, None)
    with pytest.raises(ffi.RgError):
        ffi.call("rgExtCopyDeviceToDevice", dst.ptr, src.ptr, 20, None)



def _decode_half_nodes(nodes):
    """Child boxes of FP16 nodes as the traversal decodes them: origin +
    float(offset), rounded to FP32."""
    o = nodes["origin"].astype(np.float32)
    out = {}
    for f, axis in (("lo_x", 0), ("hi_x", 0), ("lo_y", 1), ("hi_y", 1), ("lo_z", 2), ("hi_z", 2)):
        out[f] = o[:, axis:axis + 1] + nodes[f].view(np.float16).astype(np.float32)
    return out


@pytest.mark.parametrize("case", ["terrain_boxes", "far_soup"])
def test_fp16_nodes_contain_fp32_boxes_and_hit_the_same(gpu, case):
    """FP16 nodes (FP32 origin + half offsets rounded outward) have the FP32
    build's topology and boxes that contain its boxes, so closest-hit traversal
    finds the same hits bit for bit (the hit rule is order-independent)."""
    print(f"fp16 nodes {case}", flush=True)
    if case == "terrain_boxes":
        tris = scenes.terrain_boxes_scene().tris
        rays = np.concatenate([scenes.primary_rays(scenes.terrain_boxes_camera(), 640, 360)])
    else:
        # 200k small triangles 20,000 units from the origin: absolute FP16
        # coordinates there are 16 units apart
        tris = _random_tris(200_000, 9, spread=500.0, size=0.3) + np.float32(20000.0)
        r = np.random.default_rng(4)
        rays = np.zeros(100_000, RAY_DTYPE)
        rays["origin"] = r.uniform(-600, 600, (100_000, 3)) + 20000.0
        d = r.normal(size=(100_000, 3))
        rays["direction"] = d / np.linalg.norm(d, axis=1, keepdims=True)
        rays["tmax"] = 2000.0
    d = DeviceArray.from_numpy(tris)
    b32, b16 = Bvh(), Bvh()
    b32.build(d, len(tris), 1, ffi.RG_EXT_BVH_NODE_FP32)
    b16.build(d, len(tris), 1, ffi.RG_EXT_BVH_NODE_FP16)
    g32, g16 = b32.download(), b16.download()
    assert b16.view().nodeStrideBytes == 144
    assert g16["node_count"] == g32["node_count"]
    assert np.array_equal(g16["nodes"]["child"], g32["nodes"]["child"])
    assert np.array_equal(g16["sorted_tris"], g32["sorted_tris"])
    dec = _decode_half_nodes(g16["nodes"])
    full = g32["nodes"]["child"] != 0xFFFFFFFF
    for f in ("lo_x", "lo_y", "lo_z"):
        assert (dec[f][full] <= g32["nodes"][f][full]).all(), f
    for f in ("hi_x", "hi_y", "hi_z"):
        assert (dec[f][full] >= g32["nodes"][f][full]).all(), f
    # outward rounding costs ~2^-11 of the node's extent, not of the coordinates
    ext32 = g32["nodes"]["hi_x"][full].astype(np.float64) - g32["nodes"]["lo_x"][full]
    ext16 = dec["hi_x"][full].astype(np.float64) - dec["lo_x"][full]
    grow = (ext16 - ext32) / np.maximum(ext32, 1e-6)
    print(f"fp16 box growth (x): median {np.median(grow):.2e}, p99 {np.quantile(grow, 0.99):.2e}", flush=True)
    assert np.median(grow) < 2e-2
    for flags in (0, RG_EXT_TRACE_ANY_HIT):
        h32 = _trace_gpu(b32, rays, flags | RG_EXT_TRACE_COLLECT_STATS)
        n32 = b32.trace_stats()
        h16 = _trace_gpu(b16, rays, flags | RG_EXT_TRACE_COLLECT_STATS)
        n16 = b16.trace_stats()
        print(f"flags {flags}: node visits fp32 {n32[0]} fp16 {n16[0]}, triangle tests {n32[1]} {n16[1]}", flush=True)
        assert b16.trace_errors() == 0
        _assert_same_hits(h16, h32, any_hit=bool(flags & RG_EXT_TRACE_ANY_HIT))
