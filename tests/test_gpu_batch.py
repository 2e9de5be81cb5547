"""Batches of scenes (rtbvh_gpu_create_batch / rtbvh_gpu_intersect_batch).

No reference counterpart: the reference builds and traces one scene per
call.  The bar is that a batch is exactly the per-scene work done together:
  * every scene's subtree of the batch forest equals, node for node (bounds
    bit for bit, same child order, same leaf primitives), the PLOC tree of
    that scene built alone (which is itself bit-identical to the oracle's
    LOCB);
  * the batched launch returns, bit for bit, the hits and occlusion flags of
    tracing each scene alone, and those equal the oracle's brute force.
"""
import numpy as np
import pytest

from oracle import refcpu as ref
from rtbvh_amd import scenes
from tests.helpers import as_rays, flat, hits_equal, prep, ray_set, teapot

torch = pytest.importorskip("torch")
import rtbvh_amd as rt  # noqa: E402
from rtbvh_amd import _lib as L  # noqa: E402

pytestmark = pytest.mark.gpu


def _dev(a, dtype=torch.float32):
    return torch.from_numpy(np.ascontiguousarray(a)).view(dtype).cuda()


def _scene_list():
    return [
        scenes.random_soup(3, 0.2, seed=1),
        teapot(),
        scenes.random_soup(100, 0.1, seed=4),
        scenes.noisy_sphere(60, 40, seed=5),
        np.repeat(scenes.random_soup(400, 0.05, seed=6), 3, axis=0),
        scenes.torus(120, 60),
        scenes.random_soup(7, 0.3, seed=8),
    ]


def _subtree_equal(na, ia, ra, off_a, nb, ib, rb):
    """Node-for-node equality of the subtree of (na, ia) at ra, whose leaves
    hold batch-wide ids offset by off_a, and the tree (nb, ib) at rb."""
    ua = flat(na).view(np.uint32).reshape(-1, 8)
    ub = flat(nb).view(np.uint32).reshape(-1, 8)
    stack = [(ra, rb)]
    count = 0
    while stack:
        a, b = stack.pop()
        count += 1
        if not np.array_equal(ua[a][[0, 1, 2, 4, 5, 6]], ub[b][[0, 1, 2, 4, 5, 6]]):
            return False, f"bounds differ at {a}/{b}"
        ca, cb = int(na[a]["count"]), int(nb[b]["count"])
        if ca != cb:
            return False, f"count differs at {a}/{b}"
        la, lb = int(na[a]["left_first"]), int(nb[b]["left_first"])
        if ca >= 0:
            pa = ia[la:la + ca].astype(np.int64) - off_a
            pb = ib[lb:lb + cb].astype(np.int64)
            if not np.array_equal(pa, pb):
                return False, f"leaf prims differ at {a}/{b}"
        else:
            stack.append((la + 1, lb + 1))
            stack.append((la, lb))
    return True, count


def _build_batch(verts_list):
    counts = [len(v) for v in verts_list]
    offs = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    verts = np.concatenate(verts_list)
    aabbs, centers = prep(verts)
    batch = rt.SceneBatch(_dev(centers), offs.tolist(), aabbs=_dev(flat(aabbs)))
    return batch, verts, offs


def test_batch_trees_equal_single_scene_builds():
    print("[batch_trees]", flush=True)
    vl = _scene_list()
    batch, verts, offs = _build_batch(vl)
    assert batch.scene_count == len(vl)
    assert batch.bvh_node_count == 2 * len(verts) - len(vl)
    nodes = batch.bvh_nodes().cpu().numpy().view(ref.AABB).reshape(-1)
    idx = batch.indices().cpu().numpy().view(np.uint32)
    assert sorted(idx.tolist()) == list(range(len(verts)))
    for s, v in enumerate(vl):
        aabbs, centers = prep(v)
        want_n, want_i = ref.build_locb(aabbs, centers)
        ok, info = _subtree_equal(nodes, idx, s, int(offs[s]), want_n, want_i, 0)
        assert ok, f"scene {s}: {info}"
        assert info == 2 * len(v) - 1


def test_batch_trace_equals_per_scene_trace():
    print("[batch_trace]", flush=True)
    vl = _scene_list()
    batch, verts, offs = _build_batch(vl)
    batch.attach_triangles(_dev(verts))
    rays_l = [ray_set(v, 3000 + 500 * s, seed=20 + s, kind="box") for s, v in enumerate(vl)]
    rays_l[2] = rays_l[2][:0]  # a scene without rays
    for r in rays_l[::2]:
        if len(r):
            r[::4, 7] = np.float32(0.5)
    counts = [len(r) for r in rays_l]
    rays = np.concatenate(rays_l)
    roff = rt.SceneBatch.ray_offsets(counts, "cuda")
    got = batch.intersect(_dev(rays), roff).cpu().numpy()
    got_occ = batch.occluded(_dev(rays), roff).cpu().numpy()
    torch.cuda.synchronize()
    start = 0
    for s, v in enumerate(vl):
        r = rays_l[s]
        g = got[start:start + len(r)]
        go = got_occ[start:start + len(r)]
        start += len(r)
        if not len(r):
            continue
        aabbs, centers = prep(v)
        bvh = rt.Builder(_dev(centers), aabbs=_dev(flat(aabbs))).construct_locally_ordered_clustered()
        m = rt.Mbvh.from_bvh(bvh)
        m.attach_triangles(_dev(v))
        want = m.intersect_prepared(_dev(r)).cpu().numpy()
        want_occ = m.occluded_prepared(_dev(r)).cpu().numpy()
        assert np.array_equal(g.view(np.uint32), want.view(np.uint32)), f"scene {s}"
        assert np.array_equal(go, want_occ), f"scene {s} occluded"
        brute = ref.trace_brute(v, as_rays(r), threads=8)
        assert hits_equal(g.view(ref.HIT).reshape(-1), brute).all(), f"scene {s} vs brute force"
    m.status()


@pytest.mark.parametrize("n_scenes", [2500, 4096])
def test_batch_many_small_scenes(n_scenes):
    """More scenes than the clustering's usual tail threshold (2048), up to
    RTBVH_MAX_BATCH_SCENES: the tail then starts at one cluster per scene
    and holds up to 4096 clusters.  Sampled scenes' subtrees equal the
    oracle's LOCB and their batched hits equal brute force."""
    print(f"[batch_many] scenes={n_scenes}", flush=True)
    rng = np.random.default_rng(n_scenes)
    sizes = rng.integers(3, 13, n_scenes)
    vl = [scenes.random_soup(int(c), 0.2, seed=1000 + i) for i, c in enumerate(sizes)]
    batch, verts, offs = _build_batch(vl)
    assert batch.scene_count == n_scenes
    nodes = batch.bvh_nodes().cpu().numpy().view(ref.AABB).reshape(-1)
    idx = batch.indices().cpu().numpy().view(np.uint32)
    assert sorted(idx.tolist()) == list(range(len(verts)))
    sample = list(range(0, n_scenes, 97)) + [n_scenes - 1]
    for s in sample:
        aabbs, centers = prep(vl[s])
        want_n, want_i = ref.build_locb(aabbs, centers)
        ok, info = _subtree_equal(nodes, idx, s, int(offs[s]), want_n, want_i, 0)
        assert ok, f"scene {s}: {info}"
    batch.attach_triangles(_dev(verts))
    rays_l = [ray_set(v, 40, seed=s, kind="box") for s, v in enumerate(vl)]
    roff = rt.SceneBatch.ray_offsets([len(r) for r in rays_l], "cuda")
    got = batch.intersect(_dev(np.concatenate(rays_l)), roff).cpu().numpy()
    starts = np.concatenate([[0], np.cumsum([len(r) for r in rays_l])])
    for s in sample:
        g = got[starts[s]:starts[s + 1]].view(ref.HIT).reshape(-1)
        brute = ref.trace_brute(vl[s], as_rays(rays_l[s]), threads=1)
        assert hits_equal(g, brute).all(), f"scene {s}"


def test_batch_autotune_keeps_results():
    """rtbvh_gpu_autotune_batch times the launch shapes on the batch's own
    rays; the shape it keeps returns the same hits as the default shape."""
    print("[batch_autotune]", flush=True)
    vl = _scene_list()
    batch, verts, offs = _build_batch(vl)
    batch.attach_triangles(_dev(verts))
    rays_l = [ray_set(v, 2000, seed=40 + s, kind="box") for s, v in enumerate(vl)]
    rays = _dev(np.concatenate(rays_l))
    roff = rt.SceneBatch.ray_offsets([len(r) for r in rays_l], "cuda")
    rt.set_trace_config()
    try:
        want = batch.intersect(rays, roff).cpu().numpy()
        best = rt.autotune(batch, rays, roff)
        assert best == rt.get_trace_config()
        assert best["block"] in (64, 128) and best["kernel"] == 0
        got = batch.intersect(rays, roff).cpu().numpy()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        with pytest.raises(ValueError):
            rt.autotune(batch, rays)
    finally:
        rt.set_trace_config()


@pytest.mark.parametrize("per_scene", [600, 20_000])
def test_autotune_of_few_rays_keeps_the_shape(per_scene):
    """A compressed tree traces up to 98,304 rays in a shape of their own: the
    autotuner has nothing to time there and leaves the device's shape as it
    is (postpone is 0 in every shape it tries), while it still writes the hits.
    Above that it times the shapes, and every shape returns the same hits."""
    vl = _scene_list()
    batch, verts, offs = _build_batch(vl)
    batch.attach_triangles(_dev(verts))
    rays = _dev(np.concatenate([ray_set(v, per_scene, seed=60 + s, kind="box")
                                for s, v in enumerate(vl)]))
    roff = rt.SceneBatch.ray_offsets([per_scene] * len(vl), "cuda")
    aabbs, centers = prep(vl[3])
    dv = _dev(vl[3])
    tree = rt.Builder(_dev(centers), aabbs=_dev(flat(aabbs))) \
        .construct_locally_ordered_clustered().trace_tree(dv)
    few = len(rays) <= 98_304
    try:
        for shape in ((128, 4, 400, 0, 8, 1, 16), (64, 10, 1600, 0, 32, 1, 3)):
            rt.set_trace_config(*shape)
            before = rt.get_trace_config()
            want = batch.intersect(rays, roff)
            for target, args in ((batch, (rays, roff)), (tree, (rays,))):
                best = rt.autotune(target, *args)
                assert best == rt.get_trace_config()
                assert (best == before) == few, (shape, best)
                assert torch.equal(batch.intersect(rays, roff).view(torch.int32),
                                   want.view(torch.int32))
                rt.set_trace_config(*shape)
        hits = torch.zeros_like(want)
        c = L.RTTraceConfig()
        L.check(L.lib().rtbvh_gpu_autotune_batch(
            batch._h, rays.data_ptr(), roff.data_ptr(), len(rays), hits.data_ptr(),
            torch.cuda.current_stream().cuda_stream, c), "rtbvh_gpu_autotune_batch")
        assert torch.equal(hits.view(torch.int32), want.view(torch.int32))
    finally:
        rt.set_trace_config()


def test_batch_errors():
    print("[batch_errors]", flush=True)
    v = scenes.random_soup(50, 0.1, seed=3)
    aabbs, centers = prep(v)
    with pytest.raises(rt.RTBvhError, match="InvalidArgument"):
        rt.SceneBatch(_dev(centers), [0, 2, 50], aabbs=_dev(flat(aabbs)))  # scene of 2
    batch = rt.SceneBatch(_dev(centers), [0, 20, 50], aabbs=_dev(flat(aabbs)))
    rays = _dev(ray_set(v, 64, seed=1))
    roff = rt.SceneBatch.ray_offsets([32, 32], "cuda")
    with pytest.raises(rt.RTBvhError):
        batch.intersect(rays, roff)  # no triangles attached
    batch.attach_triangles(_dev(v))
    out = batch.intersect(rays, roff)
    torch.cuda.synchronize()
    assert out.shape == (64, 4)
    with pytest.raises(rt.RTBvhError, match="InvalidArgument"):
        rt._lib.check(rt._lib.lib().rtbvh_gpu_intersect_batch(
            batch._h, rays.data_ptr(), roff.data_ptr(), 64, out.data_ptr(), 1, None), "flags")


@pytest.mark.parametrize("scene_count", [2, 127, 128, 129, 300])
def test_batch_of_tiny_scenes_around_a_block_of_nodes(scene_count):
    """The compressed tree's first level holds one node per scene and is built
    128 nodes to a block, eight lanes to a node: scenes of 3 to 12 triangles
    give nodes of 3 to 8 slots, with and without children."""
    vl = [scenes.random_soup(3 + s % 10, 0.3, seed=500 + s) for s in range(scene_count)]
    batch, verts, offs = _build_batch(vl)
    batch.attach_triangles(_dev(verts))
    rays_l = [ray_set(v, 24, seed=900 + s, kind="box") for s, v in enumerate(vl)]
    roff = rt.SceneBatch.ray_offsets([len(r) for r in rays_l], "cuda")
    got = batch.intersect(_dev(np.concatenate(rays_l)), roff).cpu().numpy()
    got = got.view(ref.HIT).reshape(-1)
    for s, v in enumerate(vl):
        want = ref.trace_brute(v, as_rays(rays_l[s]))
        assert hits_equal(got[24 * s:24 * s + 24], want).all(), s
