"""GPU parity of the HIP hot path against the FP32 oracle (marked gpu).

* BVH invariants of the GPU LBVH: every triangle in exactly one leaf, every
  internal node reached once, each parent box contains its children.
* Closest / any hit on fixed ray batches: instance and primitive ids, t,
  barycentrics and facing bit-exact against the oracle (which is itself
  pinned to brute force).
* Per-sample radiance of whole frames against the FP32 oracle, same seeds:
  required within 1e-4 relative for >= 99.9 % of samples (bit equality is
  expected); rgba running mean, albedo and normal targets likewise.
"""
import ctypes as C
import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import oracle
from kuafu_amd import abi, api, scenes
from kuafu_amd.api import GpuScene, Renderer, push_constants

pytestmark = pytest.mark.gpu


def node_boxes(n):
    L = np.array([[n[0], n[2], n[8]], [n[1], n[3], n[9]]])
    R = np.array([[n[4], n[6], n[10]], [n[5], n[7], n[11]]])
    return L, R


def check_blas(gs, g):
    verts, tris, _, _ = gs.data.geoms[g]
    nodes, root, order = gs.read_blas(g)
    nt = len(tris)
    assert sorted(order.tolist()) == list(range(nt))
    if nt == 1:
        assert root == ~0
        return 0
    assert len(nodes) == nt - 1 and root == 0
    refs = nodes[:, 12:14].copy().view(np.int32)
    seen_nodes = np.zeros(nt - 1, int)
    seen_leaves = np.zeros(nt, int)
    pos = verts["pos"].astype(np.float64)
    depth = 0
    stack = [(0, None, 1)]
    while stack:
        r, parent_box, d = stack.pop()
        depth = max(depth, d)
        seen_nodes[r] += 1
        L, R = node_boxes(nodes[r])
        for ref, box in ((refs[r, 0], L), (refs[r, 1], R)):
            if parent_box is not None:
                assert (box[0] >= parent_box[0]).all() and (box[1] <= parent_box[1]).all()
            if ref >= 0:
                stack.append((ref, box, d + 1))
            else:
                slot = ~ref
                seen_leaves[slot] += 1
                p = pos[tris[order[slot]]]
                assert (p.min(0) >= box[0] - 1e-7).all() and (p.max(0) <= box[1] + 1e-7).all()
    assert (seen_nodes == 1).all() and (seen_leaves == 1).all()
    return depth


# Batches around a chunk, a wave, one query per lane of the resident grid
# (4 waves per SIMD on 256 CUs, 5 for shadow rays) and several refills of it:
# a ray's hit does not depend on the batch it is traced in.
@pytest.mark.parametrize("n", [1, 7, 8, 9, 63, 64, 65, 513, 262143, 262145, 327680, 700001])
def test_batch_sizes_give_the_same_hits(gpu, n):
    gs = GpuScene(scenes.config1().data)
    rng = np.random.default_rng(5)
    base = np.zeros(1009, abi.RAY_DTYPE)
    base["org"] = rng.uniform(-3, 3, (1009, 3)) + (0.0, 3.0, 0.0)
    d = rng.normal(size=(1009, 3))
    base["dir"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    base["tmin"], base["tmax"] = 0.001, 1e4
    base["tmax"][::97] = -1.0  # nothing to trace: a miss
    hits = np.concatenate([gs.trace_closest(base[i:i + 64]) for i in range(0, 1009, 64)])
    occ = np.concatenate([gs.trace_any(base[i:i + 64]) for i in range(0, 1009, 64)])
    idx = np.arange(n) % 1009
    got = gs.trace_closest(base[idx])
    assert got.tobytes() == hits[idx].tobytes()
    assert np.array_equal(gs.trace_any(base[idx]), occ[idx])
    if n == 65:
        ref = oracle.Scene(scenes.config1().data).trace_closest(base)
        assert np.array_equal(hits["inst"], ref["inst"]) and np.array_equal(hits["prim"], ref["prim"])


# Batches around the size up to which rays and hits stay in pinned memory, and
# beyond what a scene keeps on the device, in an order that grows, shrinks and
# skips its workspace; from several threads at once the same hits.
@pytest.mark.parametrize("sizes", [(131072, 131073, 100, 131072), (1250000, 200000, 5), (3, 131073, 4096, 1)])
def test_trace_workspace(gpu, sizes):
    gs = GpuScene(scenes.config1().data)
    rng = np.random.default_rng(len(sizes))
    base = np.zeros(997, abi.RAY_DTYPE)
    base["org"] = rng.uniform(-3, 3, (997, 3)) + (0.0, 3.0, 0.0)
    d = rng.normal(size=(997, 3))
    base["dir"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    base["tmin"], base["tmax"] = 0.001, 1e4
    hits, occ = gs.trace_closest(base), gs.trace_any(base)
    for n in sizes:
        idx = np.arange(n) % 997
        assert gs.trace_closest(base[idx]).tobytes() == hits[idx].tobytes()
        assert np.array_equal(gs.trace_any(base[idx]), occ[idx])

    def some(k):
        idx = (np.arange(min(sizes[k % len(sizes)], 20000)) + 31 * k) % 997
        return gs.trace_closest(base[idx]).tobytes() == hits[idx].tobytes() and np.array_equal(gs.trace_any(base[idx]), occ[idx])

    with ThreadPoolExecutor(4) as pool:
        assert all(pool.map(some, range(24)))


# Triangles one behind the other whose boxes every ray meets: three children
# stay on the stack per BVH4 level (log4 n levels), below, at and beyond what
# the LDS ring holds.  Half the rays pass all triangles but the last one.
@pytest.mark.parametrize("n", [4, 64, 300, 1024, 4096, 40000])
def test_stack_depths(gpu, n):
    v = np.zeros(3 * n, abi.VERTEX_DTYPE)
    z = np.repeat(np.arange(n) / n, 3)
    v["pos"] = np.stack([np.tile([0.0, 1.0, 0.0], n), np.tile([0.0, 0.0, 1.0], n), z], 1)
    v["pos"][-3:, :2] = [[-4.0, -4.0], [8.0, -4.0], [-4.0, 8.0]]
    v["normal"] = (0.0, 0.0, 1.0)
    s = scenes.SceneData()
    s.add_geometry(v, np.arange(3 * n, dtype=np.uint32).reshape(-1, 3), scenes.material())
    s.add_instance(0, scenes.mat_from_rows(np.eye(3), (0.0, 0.0, 0.0)))
    rng = np.random.default_rng(n)
    rays = np.zeros(500, abi.RAY_DTYPE)
    xy = rng.uniform(0.05, 0.95, (500, 2))
    up = rng.random(500) < 0.5
    rays["org"] = np.concatenate([xy, np.where(up, -1.0, 2.0)[:, None]], 1)
    d = np.concatenate([rng.uniform(-1e-3, 1e-3, (500, 2)), np.where(up, 1.0, -1.0)[:, None]], 1)
    rays["dir"] = d
    rays["tmin"], rays["tmax"] = 0.001, 1e4
    ref = oracle.Scene(s).trace_closest(rays)
    gs = GpuScene(s)
    hits = gs.trace_closest(rays)
    for f in ("inst", "prim", "t", "b1", "b2"):
        assert hits[f].tobytes() == ref[f].tobytes(), f
    assert (hits["prim"] == n - 1).any() and (n < 64 or (hits["prim"] != n - 1).any())
    assert gs.trace_any(rays).all()
    rays["tmax"] = 2.0 - 1.5 / n  # upwards: past all but the last triangle
    far = up & (ref["prim"] == n - 1)
    assert not gs.trace_any(rays)[far].any()


# Instances per TLAS around the block sizes of the one-launch build (64, 256,
# 1024) and beyond it, created directly and by an update from another count.
@pytest.mark.parametrize("n", [1, 2, 3, 63, 64, 65, 256, 257, 1024, 1025, 3000])
def test_tlas_sizes(gpu, n):
    rng = np.random.default_rng(n)
    s = scenes.SceneData()
    sv, si = scenes.uv_sphere(6, 4, 0.5)
    one_v, one_t = scenes.quad(1.0)
    s.add_geometry(sv, si, scenes.material())
    s.add_geometry(one_v, one_t[:1], scenes.material())  # its BLAS root is a triangle
    s.add_geometry(sv, si, scenes.material(), hidden=True)
    for k in range(n):
        pos = rng.uniform(-8, 8, 3) if k % 5 else (1.0, 2.0, 3.0)  # equal Morton codes too
        s.add_instance(int(rng.choice(3, p=[0.8, 0.15, 0.05])),
                       scenes.mat_from_rows(scenes.random_rotation(rng) * rng.uniform(0.3, 1.2), pos))
    rays = np.zeros(600, abi.RAY_DTYPE)
    rays["org"] = rng.uniform(-12, 12, (600, 3))
    d = rng.uniform(-6, 6, (600, 3)) - rays["org"]
    rays["dir"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays["tmin"], rays["tmax"] = 0.001, 1e4
    ref = oracle.Scene(s).trace_closest(rays)
    gs = GpuScene(s)
    few = scenes.SceneData()
    few.__dict__.update(s.__dict__)
    few.instances = s.instances[:max(1, n // 2)]
    updated = GpuScene(few)
    updated.update_instances(s.arrays()["inst"])
    for g in (gs, updated):
        hits = g.trace_closest(rays)
        for f in ("inst", "prim", "t", "b1", "b2"):
            hit = ref["inst"] != 0xFFFFFFFF if f in ("t", "b1", "b2") else slice(None)
            assert np.array_equal(hits[f][hit], ref[f][hit]), f
        nodes, roots = g.read_bvh4(1)
        leaves, todo = [], [int(roots[0])] if n > 1 else []
        while todo:
            for c in nodes[todo.pop(), 24:28].copy().view(np.uint32):
                if c == 0xFFFFFFFF:
                    continue
                if c >> 30 == 0:
                    todo.append(int(c))
                else:
                    assert c >> 30 == 2
                    leaves.append(int(c & 0x3FFFFFFF))
        assert sorted(leaves) == (list(range(n)) if n > 1 else [])


def test_blas_invariants(gpu):
    w = scenes.config1()
    gs = GpuScene(w.data)
    for g in range(len(w.data.geoms)):
        check_blas(gs, g)
    s = scenes.SceneData()
    v, t = scenes.icosphere(4)
    s.add_geometry(v, t, scenes.material())
    s.add_geometry(*scenes.quad(1.0), scenes.material())
    one_v, one_t = scenes.quad(1.0)
    s.add_geometry(one_v, one_t[:1], scenes.material())
    s.add_instance(0)
    gs2 = GpuScene(s)
    d = check_blas(gs2, 0)
    assert d < 48
    check_blas(gs2, 1)
    check_blas(gs2, 2)
    info = gs2.bvh_info()
    assert info.triangles == 5120 + 2 + 1 and info.max_blas_depth == d


# Triangles per geometry: around the runs of 512 leaves that one pyramid block
# reduces, around sort tiles (2048 keys), many segments per wave (geometries of
# one to three triangles) and a geometry after them.
@pytest.mark.parametrize("counts", [(2,), (3,), (511,), (512,), (513,), (1025,), (2049, 1, 2, 3), (1,) * 100 + (2, 70, 3) * 30,
                                    (5000, 262145)])
def test_blas_boxes_are_the_unions_of_their_triangles(gpu, counts):
    rng = np.random.default_rng(len(counts) + counts[0])
    s = scenes.SceneData()
    m = s.add_material(scenes.material())
    for n in counts:
        pos = (rng.uniform(-5, 5, (n, 1, 3)) + rng.normal(0, 0.1, (n, 3, 3))).reshape(-1, 3).astype(np.float32)
        s.add_geometry(api.vertices(pos), np.arange(3 * n, dtype=np.uint32).reshape(n, 3), m)
    for g in range(len(counts)):
        s.add_instance(g)
    gs = GpuScene(s)
    moved = s.geoms[-1][0].copy()
    moved["pos"] = moved["pos"][:, [1, 2, 0]] * np.float32(1.5)
    for step in range(2):
        for g in ([0, len(counts) // 2, len(counts) - 1] if step == 0 else [len(counts) - 1]):
            pos = (moved if step else s.geoms[g][0])["pos"].reshape(-1, 3, 3)
            nodes, root, order = gs.read_blas(g)
            n = counts[g]
            assert sorted(order.tolist()) == list(range(n))
            lo, hi = pos.min(1)[order], pos.max(1)[order]
            refs = nodes[:, 12:14].copy().view(np.int32)
            # ranges of leaves, children before parents
            todo, seen = [root] if n > 1 else [], []
            while todo:
                r = todo.pop()
                seen.append(r)
                todo += [int(c) for c in refs[r] if c >= 0]
            assert len(seen) == n - 1 == len(set(seen))
            box = {}
            for r in reversed(seen):
                L, R = node_boxes(nodes[r])
                for ref, b in ((int(refs[r, 0]), L), (int(refs[r, 1]), R)):
                    want = np.stack([lo[~ref], hi[~ref]]) if ref < 0 else box[ref]
                    assert np.array_equal(b, want)
                box[r] = np.stack([np.minimum(L[0], R[0]), np.maximum(L[1], R[1])])
        if step == 0:
            gs.update_geometry(len(counts) - 1, moved)


def contact_rays(data, n, seed):
    """Rays from within 5 mm of the lines where the bodies of a scene stand on
    its ground (instance 0), half of them from the ground itself."""
    rng = np.random.default_rng(seed)
    inst = data.arrays()["inst"]
    ends = []
    for i in range(1, len(inst)):
        m = inst[i]["transform"].reshape(4, 4)
        p = data.geoms[int(inst[i]["geometry_index"])][0]["pos"] @ m[:3, :3] + m[3, :3]
        foot = p[p[:, 2] < p[:, 2].min() + 1e-4]
        ends += [foot[rng.integers(len(foot), size=2)] for _ in range(8)]
    a, b = np.array(ends)[rng.integers(len(ends), size=n)].transpose(1, 0, 2)
    org = a + rng.uniform(size=(n, 1)) * (b - a) + rng.uniform(-0.005, 0.005, (n, 3))
    org[:, 2] = np.where(np.arange(n) % 2 == 0, 0.0, np.abs(org[:, 2]))
    d = rng.uniform(-1, 1, (n, 3))
    rays = np.zeros(n, abi.RAY_DTYPE)
    rays["org"], rays["dir"] = org, d / np.linalg.norm(d, axis=1, keepdims=True)
    rays["tmin"], rays["tmax"] = 0.001, 1e4
    return rays


@pytest.mark.parametrize("seed", [0, 1, 2, 3])
def test_hits_do_not_follow_the_numbering_of_instances(gpu, seed):
    """Children entered at the same distance are visited in the order of their
    places in the node, so the same instances in another order give the same
    hits, also where two surfaces are hit within a rounding of each other."""
    w = scenes.config3(seed=seed)
    inst = w.data.arrays()["inst"].copy()
    rays = contact_rays(w.data, 1 << 18, seed)
    gs = GpuScene(w.data)
    hits = gs.trace_closest(rays)
    for order in (np.arange(len(inst))[::-1], np.random.default_rng(seed).permutation(len(inst))):
        gs.update_instances(np.ascontiguousarray(inst[order]))
        assert gs.trace_closest(rays)["t"].tobytes() == hits["t"].tobytes()


# (seed, ray of contact_rays, instance, primitive, distance): hits that turn on
# the order of children entered at the same distance.  closest: whether that
# order finds the closest one; the other hits lie within 5e-7 m of it, a few
# roundings of a distance over the 4 m ground.
@pytest.mark.parametrize("seed,ray,inst,prim,t,closest", [
    (0, 5399, 0, 0, "0x1.1648460000000p-10", True), (2, 27307, 58, 57, "0x1.f301880000000p-10", True),
    (3, 9363, 19, 11, "0x1.c2e5e60000000p-10", False), (0, 959, 23, 49, "0x1.99dd400000000p-6", False),
    (1, 151, 54, 43, "0x1.0cabb40000000p-7", False), (3, 10955, 34, 10, "0x1.28a4e60000000p-5", False)])
def test_hits_at_contact_lines(gpu, seed, ray, inst, prim, t, closest):
    w = scenes.config3(seed=seed)
    rays = contact_rays(w.data, 1 << 18, seed)[ray:ray + 1]
    (hit,) = GpuScene(w.data).trace_closest(rays)
    assert (hit["inst"], hit["prim"], float(hit["t"])) == (inst, prim, float.fromhex(t))
    (ref,) = oracle.Scene(w.data).trace_closest(rays, brute=True)
    if closest:
        assert (ref["inst"], ref["prim"], ref["t"]) == (hit["inst"], hit["prim"], hit["t"])
    else:
        assert 0.0 < hit["t"] - ref["t"] < 5e-7


EMPTY_ITEM = 0xFFFFFFFF


def walk_bvh4(nodes, root, leaf_box_check, inner_kind):
    """Visit a BVH4 from root: every node once, returns the leaf indices seen.
    Children are items kind << 30 | index (inner_kind for inner nodes,
    inner_kind + 2 for leaves).  leaf_box_check(leaf, lo, hi) asserts the
    leaf lies in its child box."""
    items = nodes[:, 24:28].copy().view(np.uint32)
    seen = np.zeros(len(nodes), int)
    leaves = []
    stack = [root]
    while stack:
        r = stack.pop()
        seen[r] += 1
        n = nodes[r]
        lo = np.stack([n[0:4], n[8:12], n[16:20]], 1).astype(np.float64)
        hi = np.stack([n[4:8], n[12:16], n[20:24]], 1).astype(np.float64)
        used = items[r] != EMPTY_ITEM
        assert used.sum() >= 2
        assert used[:used.sum()].all(), "unused child slots come last"
        for c in range(4):
            if not used[c]:
                continue
            kind, idx = int(items[r, c]) >> 30, int(items[r, c]) & 0x3FFFFFFF
            assert kind in (inner_kind, inner_kind + 2)
            assert (lo[c] <= hi[c]).all()
            if kind == inner_kind:
                child = nodes[idx]
                clo = np.stack([child[0:4], child[8:12], child[16:20]], 1)
                chi = np.stack([child[4:8], child[12:16], child[20:24]], 1)
                cu = items[idx] != EMPTY_ITEM
                assert (clo[cu] >= lo[c]).all() and (chi[cu] <= hi[c]).all()
                stack.append(idx)
            else:
                leaves.append(idx)
                leaf_box_check(idx, lo[c], hi[c])
    return seen, leaves


@pytest.mark.parametrize("shift", [1, 2, 3])
def test_bvh4_into_a_buffer_aligned_for_floats(gpu, shift):
    """The nodes arrive whole in a buffer that starts 4, 8 or 12 bytes off a
    16-byte line."""
    gs = GpuScene(scenes.config1().data)
    for which in (0, 1):
        want, _ = gs.read_bvh4(which)
        raw = np.zeros(want.size + 8, np.float32)
        at = (-raw.ctypes.data // 4) % 4 + shift
        n = C.c_uint32()
        abi.check(abi.lib().kf_scene_read_bvh4(gs.h, which, raw.ctypes.data + 4 * at, len(want), C.byref(n), None, 0))
        assert (raw.ctypes.data + 4 * at) % 16 == 4 * shift and n.value == len(want)
        assert raw[at:at + want.size].tobytes() == want.tobytes()


def check_blas4(gs, s):
    """Every triangle slot of a geometry in exactly one BVH4 leaf whose box
    holds the triangle (at its current vertex positions), every node
    reached once, geometry g's nodes packed at the start of its range
    [node_off[g], node_off[g] + n_g - 1), fewer nodes than the BVH2."""
    nodes4, roots4 = gs.read_bvh4(0)
    info = gs.bvh_info()
    assert len(nodes4) == info.blas_nodes and info.blas4_nodes < info.blas_nodes
    toff = np.cumsum([0] + [len(g[1]) for g in s.geoms])
    node_off = np.cumsum([0] + [max(len(g[1]) - 1, 0) for g in s.geoms])
    all_seen = np.zeros(len(nodes4), int)
    for g, (verts, tris, _, _) in enumerate(s.geoms):
        nt = len(tris)
        _, _, order = gs.read_blas(g)
        pos = verts["pos"].astype(np.float64)
        if nt == 1:
            assert roots4[g] == ~int(toff[g])
            continue

        def tri_in_box(slot, lo, hi):
            local = slot - toff[g]
            assert 0 <= local < nt
            p = pos[tris[order[local]]]
            assert (p.min(0) >= lo).all() and (p.max(0) <= hi).all()

        assert roots4[g] == node_off[g]
        seen, leaves = walk_bvh4(nodes4, int(roots4[g]), tri_in_box, 1)
        used = np.nonzero(seen)[0]
        assert used.min() >= node_off[g] and used.max() < node_off[g + 1]
        assert used.max() - used.min() + 1 == len(used)  # packed from the start of the range
        all_seen += seen
        assert sorted(leaves) == list(range(toff[g], toff[g] + nt))
    assert all_seen.max() == 1 and all_seen.sum() == info.blas4_nodes
    return info


def test_bvh4_invariants(gpu):
    """The BVH4 the traversal reads (check_blas4); the TLAS BVH4 holds every
    instance once."""
    s = scenes.SceneData()
    v, t = scenes.icosphere(4)
    s.add_geometry(v, t, scenes.material())
    s.add_geometry(*scenes.quad(1.0), scenes.material())
    one_v, one_t = scenes.quad(1.0)
    s.add_geometry(one_v, one_t[:1], scenes.material())
    cube_v, cube_t = scenes.box((0.5, 0.5, 0.5))
    s.add_geometry(cube_v, cube_t, scenes.material())
    rng = np.random.default_rng(3)
    for i in range(37):
        m = np.eye(4, dtype=np.float32)
        m[:3, 3] = rng.uniform(-5, 5, 3)
        s.add_instance(i % 4, m)
    gs = GpuScene(s)
    info = check_blas4(gs, s)
    # TLAS
    tl, troot = gs.read_bvh4(1)
    assert info.tlas4_nodes == len(tl) and len(tl) < 36
    seen, leaves = walk_bvh4(tl, int(troot[0]), lambda i, lo, hi: None, 0)
    assert (seen == 1).all() and sorted(leaves) == list(range(37))


def rays_toward(rng, n, center, spread, origin_box):
    r = np.zeros(n, abi.RAY_DTYPE)
    r["org"] = rng.uniform(-origin_box, origin_box, (n, 3))
    tgt = np.asarray(center) + rng.uniform(-spread, spread, (n, 3))
    d = tgt - r["org"]
    r["dir"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    r["tmin"] = 0.001
    r["tmax"] = 1e4
    return r


def assert_hits_equal(g, o):
    assert (g["inst"] == o["inst"]).all(), np.nonzero(g["inst"] != o["inst"])[0][:10]
    m = o["inst"] != 0xFFFFFFFF
    assert m.sum() > 0
    for k in ("prim", "back", "t", "b1", "b2"):
        assert (g[k][m] == o[k][m]).all(), k


@pytest.mark.parametrize("which", ["config1", "tiny", "icospheres"])
def test_traversal_parity(gpu, which):
    rng = np.random.default_rng(7)
    if which == "config1":
        data = scenes.config1().data
        rays = rays_toward(rng, 200000, (0, 0.5, 0), 3.0, 6.0)
    elif which == "tiny":
        data = scenes.tiny_scene(3, n_spheres=6)
        rays = rays_toward(rng, 100000, (0, 0.5, 0), 2.5, 5.0)
    else:
        data = scenes.config2(width=64, height=36, n_inst=48, subdiv=3).data
        rays = rays_toward(rng, 200000, (0, 0, 0), 10.0, 14.0)
    gs = GpuScene(data)
    o = oracle.Scene(data)
    assert_hits_equal(gs.trace_closest(rays), o.trace_closest(rays, threads=8))
    rays["tmax"] = rng.uniform(0.1, 12.0, len(rays)).astype(np.float32)
    assert (gs.trace_any(rays) == o.trace_any(rays, threads=8)).all()


def test_traversal_shared_edges(gpu):
    # rays aimed exactly at vertices and edge midpoints of a tessellated sphere
    s = scenes.SceneData()
    v, t = scenes.icosphere(2)
    s.add_geometry(v, t, scenes.material())
    s.add_instance(0)
    p = v["pos"].astype(np.float64)
    targets = np.concatenate([p, 0.5 * (p[t[:, 0]] + p[t[:, 1]]), 0.5 * (p[t[:, 1]] + p[t[:, 2]])])
    rng = np.random.default_rng(3)
    org = targets * 3.0 + rng.normal(0, 0.2, targets.shape)
    r = np.zeros(len(targets), abi.RAY_DTYPE)
    r["org"] = org
    r["dir"] = targets - org
    r["tmin"] = 0.0
    r["tmax"] = 1e4
    g = GpuScene(s).trace_closest(r)
    assert (g["inst"] == 0).all()  # watertight: nothing falls through
    assert_hits_equal(g, oracle.Scene(s).trace_closest(r))


def render_both(w, spp_batch=0, seed=0, frames=1, rgba0=None):
    gs = GpuScene(w.data)
    rd = Renderer(w.width, w.height)
    o = oracle.Scene(w.data)
    out = []
    rg = rgba0
    ro = rgba0
    for f in range(frames):
        pc = w.pc
        pc.frame_count = f
        st = rd.render(gs, w.cam, pc, seed=seed, samples_per_batch=spp_batch, keep_samples=True)
        ref = o.render(w.cam, pc, w.width, w.height, seed=seed, threads=8, keep_samples=True,
                       rgba=None if ro is None else ro.copy())
        ro = ref["rgba"]
        out.append((st, rd.read_samples(pc.spp), rd.read(0), rd.read(1), rd.read(2), ref))
    return out


def assert_frame_parity(st, smp, rgba, alb, nrm, ref):
    rs = ref["samples"]
    close = (np.abs(smp - rs) <= 1e-4 * np.maximum(1.0, np.abs(rs))) | (np.isnan(smp) & np.isnan(rs))
    frac = close.all(-1).mean()
    exact = ((smp == rs) | (np.isnan(smp) & np.isnan(rs))).all(-1).mean()
    print("per-sample within 1e-4: %.6f, bit-exact: %.6f" % (frac, exact))
    assert frac >= 0.999
    assert (alb == ref["albedo"]).mean() > 0.999 and (nrm == ref["normal"]).mean() > 0.999
    ok = np.abs(rgba - ref["rgba"]) <= 1e-4 * np.maximum(1.0, np.abs(ref["rgba"]))
    assert ok.mean() > 0.999
    c = ref["counts"]
    assert st.primary_rays == c[0]
    # ray counts follow the paths; allow the few diverged samples
    assert abs(int(st.extension_rays) - int(c[1])) <= 0.001 * c[1] + 2
    assert abs(int(st.shadow_rays) - int(c[2])) <= 0.001 * c[2] + 2


def test_render_parity_config1_small(gpu):
    w = scenes.config1(64, 64, spp=4)
    (res,) = render_both(w)
    assert_frame_parity(*res)


def test_render_parity_config1_full(gpu):
    w = scenes.config1()   # 256x256, 4 spp, depth 4
    (res,) = render_both(w, spp_batch=1)
    assert_frame_parity(*res)


@pytest.mark.parametrize("soft", [False, True])
def test_render_parity_tiny_lights(gpu, soft):
    # soft lights exercise the inline shadow-ray path (perturbation draws)
    data = scenes.tiny_scene(5, n_spheres=5, soft=soft)
    from kuafu_amd.api import camera_ubo
    cam = camera_ubo((0.0, 2.5, 5.0), (0, -0.4, -1.0), (0, 1, 0), 48, 40, fx=50.0, fy=50.0)
    pc = push_constants(spp=3, path_depth=6, clear_color=(0.8, 0.9, 1.0, 0.5))
    w = scenes.Workload("tiny", data, cam, pc, 48, 40)
    (res,) = render_both(w)
    assert_frame_parity(*res)


def test_render_parity_alpha_tested_geometry(gpu):
    # non-opaque spheres with alpha 0.5 and 0.2 run the any-hit alpha test
    # on path rays; the coin is seeded by (sample stream, bounce) and so is
    # the same whatever order the traversal meets the triangles in
    data = scenes.tiny_scene(2, n_spheres=2)
    sv, si = scenes.uv_sphere(12, 8, 0.6)
    for a, pos in ((0.5, (-0.6, 0.7, 0.8)), (0.2, (0.7, 0.6, 1.2))):
        g = data.add_geometry(sv, si, scenes.material(diffuse=(0.3, 0.8, 0.4), alpha=a), opaque=False)
        data.add_instance(g, scenes.mat_from_rows(np.eye(3), pos))
    from kuafu_amd.api import camera_ubo
    cam = camera_ubo((0.0, 2.0, 5.0), (0, -0.3, -1.0), (0, 1, 0), 48, 40, fx=50.0, fy=50.0)
    pc = push_constants(spp=4, path_depth=5, clear_color=(0.8, 0.9, 1.0, 0.5))
    w = scenes.Workload("alpha", data, cam, pc, 48, 40)
    (res,) = render_both(w)
    assert_frame_parity(*res)


def test_instance_update_matches_fresh_scene(gpu):
    """kf_scene_update_instances (asynchronous TLAS rebuild) with every
    instance moved and one re-pointed to another geometry: the frame equals, bit for bit, the frame of
    a scene created with the new instances, and matches the oracle."""
    import copy
    w = scenes.config2(width=48, height=27, spp=2, path_depth=4, n_inst=40, subdiv=2)
    gs = GpuScene(w.data)
    rd = Renderer(w.width, w.height)
    pc = w.pc
    pc.frame_count = 0
    rd.render(gs, w.cam, pc, seed=3)
    moved = copy.deepcopy(w.data)
    rng = np.random.default_rng(5)
    moved.instances = [(np.asarray(t, np.float32).copy(), g) for t, g in moved.instances]
    for t, g in moved.instances:
        t[3, :3] += rng.uniform(-1.0, 1.0, 3).astype(np.float32)  # column-major: column 3 is the translation
    moved.instances[7] = (moved.instances[7][0], len(moved.geoms) - 1)  # another geometry
    inst = moved.arrays()["inst"]
    for _ in range(3):  # back-to-back updates reuse the pinned staging buffer
        gs.update_instances(inst)
    rd.render(gs, w.cam, pc, seed=11)
    a = rd.read(0).copy()
    gs2 = GpuScene(moved)
    rd2 = Renderer(w.width, w.height)
    rd2.render(gs2, w.cam, pc, seed=11)
    assert (a == rd2.read(0)).all()
    o = oracle.Scene(moved)
    ref = o.render(w.cam, pc, w.width, w.height, seed=11, threads=8)
    close = np.abs(a - ref["rgba"]) <= 1e-4 * np.maximum(1.0, np.abs(ref["rgba"]))
    assert close.mean() > 0.999


def test_geometry_refit_matches_fresh_scene(gpu):
    """kf_scene_update_geometry (refit of one geometry's BLAS on the GPU,
    then the TLAS) after two geometries were deformed: BVH2 and BVH4
    invariants hold at the new positions, closest hits equal the oracle's,
    and the frame equals, bit for bit, the frame of a scene created with the
    deformed vertices (whose BVHs are built from scratch)."""
    import copy
    w = scenes.config2(width=48, height=27, spp=2, path_depth=4, n_inst=12, subdiv=3)
    gs = GpuScene(w.data)
    rd = Renderer(w.width, w.height)
    pc = w.pc
    pc.frame_count = 0
    rd.render(gs, w.cam, pc, seed=3)
    moved = copy.deepcopy(w.data)
    rng = np.random.default_rng(17)
    for g in (3, 7):
        v, t, mi, fl = moved.geoms[g]
        v = v.copy()
        p = v["pos"].astype(np.float64)
        # anisotropic stretch and a twist about z: boxes change everywhere
        p *= rng.uniform(0.6, 1.8, 3)
        a = 0.8 * p[:, 2]
        p[:, 0], p[:, 1] = p[:, 0] * np.cos(a) - p[:, 1] * np.sin(a), p[:, 0] * np.sin(a) + p[:, 1] * np.cos(a)
        v["pos"] = p.astype(np.float32)
        moved.geoms[g] = (v, t, mi, fl)
        gs.update_geometry(g, v)
    check_blas4(gs, moved)
    view = type("View", (), {})()  # the refit BVH2 against the moved vertices
    view.data, view.read_blas = moved, gs.read_blas
    for g in (3, 7):
        check_blas(view, g)
    rng2 = np.random.default_rng(5)
    rays = rays_toward(rng2, 4000, np.zeros(3), 10.0, 25.0)
    assert_hits_equal(gs.trace_closest(rays), oracle.Scene(moved).trace_closest(rays))
    rd.render(gs, w.cam, pc, seed=11)
    a = rd.read(0).copy()
    rd2 = Renderer(w.width, w.height)
    rd2.render(GpuScene(moved), w.cam, pc, seed=11)
    assert (a == rd2.read(0)).all()
    with pytest.raises(RuntimeError, match="vertex count"):
        gs.update_geometry(3, moved.geoms[3][0][:-1])


@pytest.mark.parametrize("camera", ["left", "right"])
def test_render_parity_projector_pattern(gpu, camera):
    # active-light sensing scene: 64 boxes / cylinders, IR projector whose
    # Bernoulli dot pattern is a texture sampled through the projector's
    # frustum (rchit:262-316), stereo IR cameras 55 mm apart
    w = scenes.config3(width=96, height=54, spp=2, path_depth=4, camera=camera)
    (res,) = render_both(w)
    assert_frame_parity(*res)
    # the pattern reaches the image: some pixels are lit by the projector only
    assert res[2][..., 0].max() > 0.0


def test_render_accumulation_frames(gpu):
    w = scenes.config1(32, 32, spp=2)
    for res in render_both(w, frames=3):
        assert_frame_parity(*res)


def test_render_parity_icospheres_gradient_env(gpu):
    w = scenes.config2(width=160, height=90, spp=2, n_inst=32, subdiv=3)
    (res,) = render_both(w)
    assert_frame_parity(*res)


def test_bgra8_download_matches_oracle_encoding(gpu):
    w = scenes.config1(40, 24, spp=2)
    gs = GpuScene(w.data)
    rd = Renderer(w.width, w.height)
    rd.render(gs, w.cam, w.pc)
    rgba = rd.read(0)
    rgba[0, :8, 0] = [np.nan, -1.0, 0.0, 0.0031308, 0.5, 1.0, 2.0, 0.04]
    rd.write(0, rgba)
    assert (rd.download_bgra8() == oracle.to_bgra8(rgba)).all()


def test_empty_instance_list_renders_background(gpu):
    s = scenes.SceneData()
    v, t = scenes.quad(1.0)
    s.add_geometry(v, t, scenes.material())
    from kuafu_amd.api import camera_ubo
    cam = camera_ubo((0, 0, 3.0), (0, 0, -1.0), (0, 1, 0), 16, 16)
    pc = push_constants(spp=2, path_depth=2, clear_color=(0.2, 0.4, 0.6, 0.5))
    rd = Renderer(16, 16)
    rd.render(GpuScene(s), cam, pc)
    img = rd.read(0)
    assert np.allclose(img[..., :3], [0.1, 0.2, 0.3]) and (img[..., 3] == 1).all()
