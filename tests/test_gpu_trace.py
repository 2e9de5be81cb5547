"""GPU traversal parity: the HIP kernels against the CPU oracle, through the
C ABI (rtbvh_gpu_intersect*, rtbvh_gpu_occluded*).

Trees are built by the oracle and uploaded, so these tests isolate the
traversal + Moller-Trumbore kernels.  The bar is bit-exact hit records
(t, u, v, prim) in both tie modes, and exact occlusion flags.
"""
import numpy as np
import pytest

from oracle import refcpu as ref
from rtbvh_amd import scenes
from tests.helpers import as_rays, flat, hits_equal, prep, ray_set, teapot

torch = pytest.importorskip("torch")
import rtbvh_amd as rt  # noqa: E402

pytestmark = pytest.mark.gpu

SCENES = {
    "teapot": lambda: teapot(),
    "torus": lambda: scenes.torus(80, 40),
    "soup": lambda: scenes.random_soup(3000, 0.05, seed=3),
    "sphere": lambda: scenes.noisy_sphere(60, 40, seed=5),
}


def _dev(a, dtype=torch.float32):
    return torch.from_numpy(np.ascontiguousarray(a)).view(dtype).cuda()


def _trees(verts, builder):
    aabbs, centers = prep(verts)
    if builder == "locb":
        nodes, idx = ref.build_locb(aabbs, centers)
    else:
        nodes, idx = ref.build_binned_sah(aabbs, centers)
    m = ref.build_mbvh(nodes)
    return nodes, idx, m


def _gpu_hits(tree, verts, rays, reference_order):
    out = tree.intersect(_dev(verts.reshape(-1, 9)), _dev(rays), reference_order=reference_order)
    torch.cuda.synchronize()
    tree.status()
    return out.cpu().numpy().view(ref.HIT).reshape(-1)


@pytest.mark.parametrize("scene", list(SCENES))
@pytest.mark.parametrize("builder", ["locb", "binned"])
@pytest.mark.parametrize("kind", ["sphere", "box"])
def test_trace_parity(scene, builder, kind):
    print(f"[trace_parity] scene={scene} builder={builder} rays={kind}", flush=True)
    verts = SCENES[scene]()
    nodes, idx, m = _trees(verts, builder)
    rays8 = ray_set(verts, 20000, seed=11, kind=kind)
    rays = as_rays(rays8)
    bvh = rt.Bvh.from_arrays(_dev(flat(nodes)), _dev(idx, torch.int32))
    mbvh = rt.Mbvh.from_arrays(_dev(flat(m)), _dev(idx, torch.int32))
    for mode, ref_order in ((ref.MODE_LOWEST_ID, False), (ref.MODE_VISIT_ORDER, True)):
        want_m = ref.trace_mbvh(m, idx, verts, rays, mode=mode, threads=8)
        got_m = _gpu_hits(mbvh, verts, rays8, ref_order)
        bad = ~hits_equal(got_m, want_m)
        assert not bad.any(), f"MBVH mode={mode}: {bad.sum()} rays differ, first {np.nonzero(bad)[0][:5]}"
        want_b = ref.trace_bvh(nodes, idx, verts, rays, mode=mode, threads=8)
        got_b = _gpu_hits(bvh, verts, rays8, ref_order)
        bad = ~hits_equal(got_b, want_b)
        assert not bad.any(), f"BVH mode={mode}: {bad.sum()} rays differ"


@pytest.mark.parametrize("builder", ["locb", "binned"])
def test_occluded_parity(builder):
    print(f"[occluded_parity] builder={builder}", flush=True)
    verts = teapot()
    nodes, idx, m = _trees(verts, builder)
    rays8 = ray_set(verts, 20000, seed=12, kind="box")
    rays8[:, 7] = np.random.default_rng(0).uniform(0.0, 3.0, len(rays8)).astype(np.float32)
    rays = as_rays(rays8)
    want_m = ref.occluded_mbvh(m, idx, verts, rays, threads=8)
    want_b = ref.occluded_bvh(nodes, idx, verts, rays, threads=8)
    brute = ref.occluded_brute(verts, rays, threads=8)
    mbvh = rt.Mbvh.from_arrays(_dev(flat(m)), _dev(idx, torch.int32))
    bvh = rt.Bvh.from_arrays(_dev(flat(nodes)), _dev(idx, torch.int32))
    dv = _dev(verts.reshape(-1, 9))
    # the reference order is bit-exact with the oracle's traversal of the
    # same tree; on trees whose boxes contain their primitives (LOCB) every
    # mode equals brute force.  Binned-SAH trees built with the reference's
    # stale left-box count (binned_sah.rs:188-235) can lose hits, so only the reference-order result is pinned.
    assert np.array_equal(mbvh.occluded(dv, _dev(rays8), reference_order=True).cpu().numpy(),
                          want_m)
    assert np.array_equal(bvh.occluded(dv, _dev(rays8), reference_order=True).cpu().numpy(),
                          want_b)
    if builder == "locb":
        assert np.array_equal(want_m, brute) and np.array_equal(want_b, brute)
        for tree in (mbvh, bvh):
            got = tree.occluded(dv, _dev(rays8), reference_order=False).cpu().numpy()
            assert np.array_equal(got, brute)


def test_ffi_intersect_kat_gpu():
    """rtbvh_ffi/src/lib.rs:945-1019: quad at z = 1, ray from the origin
    along +z hits at t == 1 for the BVH and the MBVH (the hit point lies on
    the shared diagonal, so both triangles tie)."""
    print("[ffi_kat_gpu]", flush=True)
    v = np.array([[-1, -1, 1, 1, -1, 1, 1, 1, 1], [-1, -1, 1, 1, 1, 1, -1, 1, 1]], np.float32)
    aabbs, _ = prep(v)
    aabbs["min"] -= np.float32(1e-4)  # aabb! macro pads by 1e-4 (src/aabb.rs:470-482)
    aabbs["max"] += np.float32(1e-4)
    centers = ((aabbs["min"] + aabbs["max"]) * np.float32(0.5)).astype(np.float32)
    nodes, idx = ref.build_binned_sah(aabbs, centers)
    m = ref.build_mbvh(nodes)
    rays8 = np.array([[0, 0, 0, 1e-4, 0, 0, 1, 1e26]], np.float32)
    bvh = rt.Bvh.from_arrays(_dev(flat(nodes)), _dev(idx, torch.int32))
    mbvh = rt.Mbvh.from_arrays(_dev(flat(m)), _dev(idx, torch.int32))
    for tree in (bvh, mbvh):
        for ro in (False, True):
            h = _gpu_hits(tree, v, rays8, ro)
            assert h["t"][0] == np.float32(1.0)
    # lowest-id tie rule picks triangle 0; the reference order picks whichever
    # it visits first, as the oracle does
    assert _gpu_hits(mbvh, v, rays8, False)["prim"][0] == 0
    want = ref.trace_mbvh(m, idx, v, as_rays(rays8), mode=ref.MODE_VISIT_ORDER)
    assert hits_equal(_gpu_hits(mbvh, v, rays8, True), want).all()


def test_trace_edge_cases():
    """NaN rays, axis-parallel rays (inf inverse), zero-length t range, empty
    ray set, empty tree."""
    print("[trace_edge_cases]", flush=True)
    verts = scenes.torus(20, 10)
    nodes, idx, m = _trees(verts, "locb")
    rays8 = ray_set(verts, 4000, seed=3, kind="box")
    rays8[0, 0] = np.nan
    rays8[1, 4:7] = (0.0, 0.0, 1.0)
    rays8[2, 4:7] = (1.0, 0.0, 0.0)
    rays8[3, 4:7] = (0.0, -1.0, 0.0)
    rays8[4, 7] = rays8[4, 3]
    rays8[5, 0:3] = (0.0, 0.0, 0.0)
    rays8[5, 4:7] = (0.0, 0.0, 1.0)
    rays8[6, 4:7] = (-0.0, 0.0, 1.0)
    rays = as_rays(rays8)
    mbvh = rt.Mbvh.from_arrays(_dev(flat(m)), _dev(idx, torch.int32))
    bvh = rt.Bvh.from_arrays(_dev(flat(nodes)), _dev(idx, torch.int32))
    for mode, ro in ((0, False), (1, True)):
        assert hits_equal(_gpu_hits(mbvh, verts, rays8, ro),
                          ref.trace_mbvh(m, idx, verts, rays, mode=mode)).all()
        assert hits_equal(_gpu_hits(bvh, verts, rays8, ro),
                          ref.trace_bvh(nodes, idx, verts, rays, mode=mode)).all()
    got = _gpu_hits(mbvh, verts, rays8, False)
    assert got["prim"][0] == 0xFFFFFFFF
    # empty ray set
    empty = mbvh.intersect(_dev(verts.reshape(-1, 9)), torch.empty((0, 8), device="cuda"))
    assert empty.shape == (0, 4)
    # empty tree: every ray misses with t = t_max
    e = rt.Mbvh.from_arrays(torch.empty((0, 32), device="cuda"),
                            torch.empty((0,), dtype=torch.int32, device="cuda"))
    h = _gpu_hits(e, verts, rays8, False)
    assert (h["prim"] == 0xFFFFFFFF).all()


def test_trace_brute_force_large():
    """200k rays on a 120k-triangle scene: GPU lowest-id hits equal brute
    force exactly."""
    print("[trace_brute_force_large]", flush=True)
    verts = np.concatenate([scenes.noisy_sphere(250, 200, seed=9),
                            scenes.random_soup(20000, 0.01, seed=10)])
    aabbs, centers = prep(verts)
    nodes, idx = ref.build_locb(aabbs, centers)
    m = ref.build_mbvh(nodes)
    rays8 = ray_set(verts, 2000, seed=13, kind="box")
    want = ref.trace_brute(verts, as_rays(rays8), threads=8)
    mbvh = rt.Mbvh.from_arrays(_dev(flat(m)), _dev(idx, torch.int32))
    got = _gpu_hits(mbvh, verts, rays8, False)
    assert hits_equal(got, want).all()
    big = ray_set(verts, 200000, seed=14, kind="box")
    got = _gpu_hits(mbvh, verts, big, False)
    want = ref.trace_mbvh(m, idx, verts, as_rays(big), threads=8)
    assert hits_equal(got, want).all()


def test_launch_shapes_and_autotune_keep_results():
    """The traversal's launch shape (block size, LDS stack depth, persistent
    grid size, one-item or per-node-leaves kernel) changes speed only: every
    shape gives the same hit records, the autotuner's pick included, with deep
    stacks spilling from LDS to private memory at depth 0."""
    print("[launch_shapes]", flush=True)
    verts = scenes.noisy_sphere(100, 80, seed=11)
    aabbs, centers = prep(verts)
    bvh = rt.Builder(_dev(centers), aabbs=_dev(flat(aabbs))).construct_locally_ordered_clustered()
    m = rt.Mbvh.from_bvh(bvh)
    dv = _dev(verts)
    m.attach_triangles(dv)
    rays = _dev(ray_set(verts, 50000, seed=21, kind="box"))
    default = rt.get_trace_config()
    want = m.intersect_prepared(rays).cpu().numpy()
    try:
        shapes = ((64, 0, 100, 0, 1, 0), (128, 4, 50, 0, 8, 0), (256, 24, 200, 0, 64, 0),
                  (64, 32, 400, 0, 16, 0), (64, 8, 200, 0, 32, 1), (64, 8, 800, 0, 1, 1),
                  (256, 4, 3200, 0, 4, 1), (64, 0, 100, 1, 1, 0), (256, 12, 100, 1, 1, 0),
                  (128, 32, 200, 1, 1, 0))
        for block, depth, occ, kernel, refill, sched in shapes:
            rt.set_trace_config(block, depth, occ, kernel, refill, sched)
            got = m.intersect_prepared(rays).cpu().numpy()
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (block, depth, occ,
                                                                              kernel, refill,
                                                                              sched)
            occ_got = m.occluded_prepared(rays).cpu().numpy()
            assert np.array_equal(occ_got, (want[:, 3].view(np.uint32) != 0xFFFFFFFF).astype(np.uint8))
        with pytest.raises(rt.RTBvhError, match="InvalidArgument"):
            rt.set_trace_config(96, 4, 100)
        best = rt.autotune(m, rays)
        assert rt.get_trace_config() == best
        got = m.intersect_prepared(rays).cpu().numpy()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        m.status()
    finally:
        rt.set_trace_config(None)
    assert rt.get_trace_config() == default


def test_compressed_tree_launch_shapes_and_autotune():
    """The same for the compressed 8-wide tree's kernel: every launch shape
    (LDS stack depth 0 puts the whole group stack in private memory; both
    ray schedules -- 1.2M rays, so that wave ranges engage with refill 1;
    triangle postponing) and the autotuner's pick give the 4-wide tree's hit records
    and occlusion flags."""
    print("[launch_shapes_cw8]", flush=True)
    verts = np.concatenate([scenes.noisy_sphere(100, 80, seed=12),
                            scenes.random_soup(5000, 0.02, seed=13)])
    aabbs, centers = prep(verts)
    bvh = rt.Builder(_dev(centers), aabbs=_dev(flat(aabbs))).construct_locally_ordered_clustered()
    dv = _dev(verts)
    # 1.2M rays: about 2 per resident lane, so the wave-range schedule engages
    rays = _dev(ray_set(verts, 1_200_000, seed=22, kind="box"))
    rt.set_trace_config(64, 8, 100, 0, 1, 0)
    want = bvh.trace_tree(dv, width=4).intersect(rays).cpu().numpy()
    rt.set_trace_config(None)
    want_occ = (want[:, 3].view(np.uint32) != 0xFFFFFFFF).astype(np.uint8)
    tt = bvh.trace_tree(dv)
    assert tt.width == 8
    default = rt.get_trace_config()
    try:
        for block, depth, occ, refill, sched, post in (
                (64, 0, 100, 1, 0, 0), (128, 4, 50, 8, 0, 16), (256, 24, 200, 64, 0, 0),
                (64, 32, 1600, 16, 0, 64), (64, 12, 3200, 1, 0, 0), (64, 8, 400, 1, 1, 0),
                (128, 0, 100, 2, 1, 32), (256, 8, 3200, 1, 1, 0), (64, 8, 800, 64, 1, 0)):
            rt.set_trace_config(block, depth, occ, 0, refill, sched, post)
            got = tt.intersect(rays).cpu().numpy()
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (block, depth, occ)
            assert np.array_equal(tt.occluded(rays).cpu().numpy(), want_occ), (block, depth, occ)
        best = rt.autotune(tt, rays)
        assert rt.get_trace_config() == best
        got = tt.intersect(rays).cpu().numpy()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        tt.status()
    finally:
        rt.set_trace_config(None)
    assert rt.get_trace_config() == default


def test_ray_packets_unpack_and_trace():
    """RayPacket4 records (src/ray.rs:44-59) unpack to the rays
    RayPacket4::ray gives (src/ray.rs:118-146: t_min 1e-4, t_max = t[i]), and
    tracing them gives lane-for-lane the hits of those single rays."""
    print("[packets]", flush=True)
    verts = teapot()
    rays8 = ray_set(verts, 4000, seed=31, kind="box")
    rays8[:, 3] = np.float32(1e-4)
    rays8[::5, 7] = np.float32(0.75)
    p = len(rays8) // 4
    r = rays8[: 4 * p].reshape(p, 4, 8)
    packets = np.empty((p, 40), np.float32)
    for k, col in enumerate((0, 1, 2, 4, 5, 6)):
        packets[:, 4 * k: 4 * k + 4] = r[:, :, col]
    with np.errstate(divide="ignore"):
        for k, col in enumerate((4, 5, 6)):
            packets[:, 24 + 4 * k: 28 + 4 * k] = np.float32(1.0) / r[:, :, col]
    packets[:, 36:40] = r[:, :, 7]
    got = rt.rays_from_packets(_dev(packets))
    assert np.array_equal(got.cpu().numpy().view(np.uint32),
                          rays8[: 4 * p].view(np.uint32))
    nodes, idx, m = _trees(verts, "locb")
    mbvh = rt.Mbvh.from_arrays(_dev(flat(m)), _dev(idx, torch.int32))
    hp = mbvh.intersect(_dev(verts.reshape(-1, 9)), got).cpu().numpy()
    want = ref.trace_mbvh(m, idx, verts, as_rays(rays8[: 4 * p]), mode=ref.MODE_LOWEST_ID,
                          threads=8)
    assert hits_equal(hp.view(ref.HIT).reshape(-1), want).all()


@pytest.mark.parametrize("rays_n", [1, 65, 5000, 1_300_000])
@pytest.mark.parametrize("per_leaf", [1, 24])
def test_vertex_traversals_over_ray_counts_and_leaf_sizes(rays_n, per_leaf):
    """The traversals over the caller's vertex array hand out rays one per
    lane up to two per resident lane (about a million), in ranges per wave
    beyond, and test a leaf's triangles one per iteration: every count of
    rays, leaves of 1 to 24 triangles, both tie rules and any hit."""
    verts = scenes.random_soup(700, 0.2, seed=17)
    aabbs, centers = prep(verts)
    bvh = rt.Builder(_dev(centers), aabbs=_dev(flat(aabbs)),
                     primitives_per_leaf=per_leaf).construct_binned_sah()
    mbvh = rt.Mbvh.from_bvh(bvh)
    nodes = bvh.nodes().cpu().numpy().view(ref.AABB).reshape(-1)
    quads = mbvh.quad_nodes().cpu().numpy().view(ref.MBVH).reshape(-1)
    idx = bvh.indices().cpu().numpy().view(np.uint32)
    rays8 = ray_set(verts, rays_n, seed=18 + rays_n, kind="box")
    rays8[::3, 7] = np.float32(0.4)
    rays = as_rays(rays8)
    for mode, ref_order in ((ref.MODE_LOWEST_ID, False), (ref.MODE_VISIT_ORDER, True)):
        want_b = ref.trace_bvh(nodes, idx, verts, rays, mode=mode, threads=8)
        want_m = ref.trace_mbvh(quads, idx, verts, rays, mode=mode, threads=8)
        for tree, want in ((bvh, want_b), (mbvh, want_m)):
            assert hits_equal(_gpu_hits(tree, verts, rays8, ref_order), want).all(), mode
            occ = tree.occluded(_dev(verts), _dev(rays8), reference_order=ref_order).cpu().numpy()
            assert np.array_equal(occ, (want["prim"] != 0xFFFFFFFF).astype(np.uint8)), mode


@pytest.mark.parametrize("any_hit", [False, True])
def test_large_launches_equal_their_parts(any_hit):
    """Rays are handed out by the size of the launch: a vertex traversal above
    1,572,864 rays keeps one lane a ray to the end, the binary one deals runs
    in up to 8 times the resident blocks (2^25 rays and more), and compressed
    and 4-wide trees give each wave one range where the grid is 4 times the
    resident one (from 2^24 rays, refilled by 8), without a tail of groups for
    ordered rays there and for closest hits at 8 times (2^25 rays).  Every ray's result is that
    of a launch of fewer rays."""
    g = torch.Generator("cuda").manual_seed(5)
    verts = _dev(np.concatenate([scenes.noisy_sphere(40, 30, seed=51),
                                 scenes.random_soup(800, 0.1, seed=52)]))
    aabbs, centers = prep(verts.cpu().numpy())
    bvh = rt.Builder(_dev(centers), aabbs=_dev(flat(aabbs))).construct_locally_ordered_clustered()
    mbvh = rt.Mbvh.from_bvh(bvh)
    tree8, tree4 = bvh.trace_tree(verts), bvh.trace_tree(verts, width=4)
    n = (1 << 25) + 321
    rays = torch.rand((n, 8), device="cuda", generator=g)
    rays[:, 3] = 1e-4
    rays[:, 4:7] -= 0.5
    rays[:, 7] = 1e30
    rays[::3, 7] = 0.3

    def check(name, fn, count, part):
        whole = fn(rays[:count])
        for b in range(0, count, part):
            want = fn(rays[b:min(count, b + part)])
            assert torch.equal(whole[b:b + part].view(torch.int32) if not any_hit
                               else whole[b:b + part],
                               want.view(torch.int32) if not any_hit else want), (name, b)
        return whole

    kind = "occluded" if any_hit else "intersect"
    for ref_order in (False, True):
        check("bvh", lambda r: getattr(bvh, kind)(verts, r, reference_order=ref_order), n, 5 << 20)
    check("mbvh", lambda r: getattr(mbvh, kind)(verts, r), 1_600_003, 400_001)
    check("mbvh", lambda r: getattr(mbvh, kind)(verts, r), 3 << 20, 3 << 19)
    try:
        rt.set_trace_config(64, 8, 3200, 0, 8, 1)
        for tree in (tree8, tree4):
            got = check(str(tree.width), getattr(tree, kind), n, 1 << 20)
            if tree is tree8:
                ordered = getattr(tree, kind)(rays, order_rays=True)
                assert torch.equal(ordered if any_hit else ordered.view(torch.int32),
                                   got if any_hit else got.view(torch.int32))
            if any_hit:
                assert torch.equal(got, bvh.occluded(verts, rays))
            else:
                assert torch.equal(got.view(torch.int32), bvh.intersect(verts, rays)
                                   .view(torch.int32))
    finally:
        rt.set_trace_config(None)


@pytest.mark.parametrize("rays_n", [5, 5_000, 300_001])
@pytest.mark.parametrize("per_leaf", [1, 24])
def test_vertex_traversal_with_any_stack_in_lds(rays_n, per_leaf):
    """The last sixteen rays of a wave go to groups of four lanes, whose stack
    starts in the LDS of the ray's lane and goes on in private memory: with 0
    to 32 entries in LDS the results are the oracle's."""
    verts = np.concatenate([scenes.noisy_sphere(40, 30, seed=55),
                            scenes.random_soup(900, 0.15, seed=56)])
    aabbs, centers = prep(verts)
    bvh = rt.Builder(_dev(centers), aabbs=_dev(flat(aabbs)),
                     primitives_per_leaf=per_leaf).construct_binned_sah()
    mbvh = rt.Mbvh.from_bvh(bvh)
    quads = mbvh.quad_nodes().cpu().numpy().view(ref.MBVH).reshape(-1)
    idx = bvh.indices().cpu().numpy().view(np.uint32)
    rays8 = ray_set(verts, rays_n, seed=57, kind="box")
    rays8[::3, 7] = np.float32(0.4)
    rays8[::7, 4] = 0.0
    want = ref.trace_mbvh(quads, idx, verts, as_rays(rays8), mode=ref.MODE_LOWEST_ID, threads=8)
    flags = (want["prim"] != 0xFFFFFFFF).astype(np.uint8)
    try:
        for block, depth in ((64, 0), (128, 1), (256, 2), (64, 4), (64, 32)):
            rt.set_trace_config(block, depth, 100)
            assert hits_equal(_gpu_hits(mbvh, verts, rays8, False), want).all(), depth
            assert np.array_equal(mbvh.occluded(_dev(verts), _dev(rays8)).cpu().numpy(), flags)
    finally:
        rt.set_trace_config(None)


def _chains(depth):
    """(binary nodes, 4-wide nodes) of a chain of `depth` interior nodes that
    one ray along +z walks to the end, with one entry left on the stack by
    every level: the sibling, an interior node without children, lies behind."""
    box = np.zeros(2 * depth + 1, ref.AABB)
    box["min"], box["max"] = -2.0, 10.0
    box["count"], box["left_first"] = -1, -1
    box["left_first"][0] = 1
    box["left_first"][1:-2:2] = np.arange(3, 2 * depth, 2)
    box["max"][2::2] = 9.0
    box["min"][2::2] = -1.0
    box["count"][-2], box["left_first"][-2] = 1, 0
    quad = np.zeros(depth + 1, ref.MBVH)
    for ax in "xyz":
        quad[f"min_{ax}"], quad[f"max_{ax}"] = 3.0e38, 3.0e38
        quad[f"min_{ax}"][:-1, 0:2], quad[f"max_{ax}"][:-1, 0:2] = -2.0, 10.0
    quad["min_z"][:-1, 1] = 0.5  # the sibling is entered later
    quad["children"], quad["counts"] = -1, -1
    quad["children"][:-1, 0] = np.arange(1, depth + 1)
    quad["children"][:-1, 1] = depth
    quad["children"][-2, 0], quad["counts"][-2, 0] = 0, 1
    return box, quad


@pytest.mark.parametrize("rays_n", [3, 64, 1000])
@pytest.mark.parametrize("depth", [2, 100, 255, 256, 257, 258, 300])
def test_stack_limit(depth, rays_n):
    """RTBVH_MAX_STACK (256) entries: the binary traversal holds the child in
    hand beside the siblings of 254 levels, the 4-wide one 256 siblings; a ray
    that needs more ends with t = NaN, no hit, and a sticky StackOverflow."""
    verts = np.array([[-1, -1, 1, 1, -1, 1, 0, 1, 1]], np.float32)
    idx = _dev(np.zeros(1, np.int32), torch.int32)
    rays = _dev(np.repeat(np.array([[0, 0, 0, 1e-4, 0, 0, 1, 1e26]], np.float32), rays_n, axis=0))
    box, quad = _chains(depth)
    bvh = rt.Bvh.from_arrays(_dev(flat(box)), idx)
    mbvh = rt.Mbvh.from_arrays(_dev(flat(quad)), idx)
    try:
        for tree, orders, most in ((bvh, (False, True), 255), (mbvh, (False,), 257)):
            for lds in (8, 0, 32):
                rt.set_trace_config(64, lds, 100)
                for ref_order in orders:
                    hits = tree.intersect(_dev(verts), rays, reference_order=ref_order)
                    prim = hits.view(torch.int32)[:, 3]
                    if depth <= most:
                        tree.status()
                        assert bool((prim == 0).all()) and bool((hits[:, 0] == 1.0).all())
                    else:
                        with pytest.raises(rt.RTBvhError, match="StackOverflow"):
                            tree.status()
                        assert bool((prim == -1).all()) and bool(hits[:, 0].isnan().all())
                    occ = tree.occluded(_dev(verts), rays, reference_order=ref_order)
                    assert bool((occ == (1 if depth <= most else 0)).all())
                    if depth > most:
                        with pytest.raises(rt.RTBvhError, match="StackOverflow"):
                            tree.status()
    finally:
        rt.set_trace_config(None)


@pytest.mark.parametrize("first, count, tested", [(-1, 3, 0), (-2, 4, 0), (1, 2, 2), (1, 7, 2),
                                                  (3, 1, 0), (2, 1, 1)])
def test_leaf_outside_the_index_array(first, count, tested):
    """A leaf's triangles end with the index array, and a leaf that starts
    outside it has none (src/iter.rs:337 skips missing primitives): at the
    root and below it, in both tie rules and any hit."""
    quad = np.array([[-1, -1, 1, 1, -1, 1, 0, 1, 1]], np.float32)
    verts = np.repeat(quad, 3, axis=0)
    idx = np.array([2, 1, 0], np.int32)
    rays8 = np.array([[0, 0, 0, 1e-4, 0, 0, 1, 1e26]], np.float32)
    box = np.zeros(3, ref.AABB)
    box["min"], box["max"] = -2.0, 2.0
    box["count"], box["left_first"] = [-1, 0, count], [1, 0, first]
    leaf = box[2:].copy()
    ids = idx[first:first + tested] if tested else []
    for nodes in (leaf, box):
        bvh = rt.Bvh.from_arrays(_dev(flat(nodes)), _dev(idx, torch.int32))
        for ref_order in (False, True):
            hit = _gpu_hits(bvh, verts, rays8, ref_order)["prim"][0]
            if len(ids):
                assert hit == (ids[0] if ref_order else min(ids))
            else:
                assert hit == 0xFFFFFFFF
            occ = bvh.occluded(_dev(verts), _dev(rays8), reference_order=ref_order)
            assert int(occ[0]) == (1 if len(ids) else 0)


@pytest.mark.parametrize("rays_n", [1, 7, 9, 31, 33, 4097, 98_304, 98_305, 300_001])
def test_compressed_tree_over_ray_counts(rays_n):
    """Up to 98,304 rays eight lanes hold a ray and test a node's triangles
    at once, above a lane holds one: both equal brute force, for one tree, a
    batch and in any launch shape, with zero direction components, short t_max
    and duplicated triangles (the lowest id of equal t)."""
    verts = np.concatenate([scenes.random_soup(300, 0.25, seed=31)] * 2)
    aabbs, centers = prep(verts)
    dv, dc, da = _dev(verts), _dev(centers), _dev(flat(aabbs))
    tree = rt.Builder(dc, aabbs=da).construct_locally_ordered_clustered().trace_tree(dv)
    rays8 = ray_set(verts, rays_n, seed=rays_n, kind="box")
    rays8[::5, 4] = 0.0
    rays8[::11, 5] = 0.0
    rays8[::3, 7] = np.float32(0.3)
    want = ref.trace_brute(verts, as_rays(rays8), threads=8)
    flags = (want["prim"] != 0xFFFFFFFF).astype(np.uint8)
    dr = _dev(rays8)
    batch = rt.SceneBatch(dc, [0, len(verts)], aabbs=da)
    batch.attach_triangles(dv)
    off = rt.SceneBatch.ray_offsets([rays_n], "cuda")
    try:
        for shape in (None, (64, 0, 100, 0, 1, 0), (128, 8, 1600, 0, 16, 1)):
            rt.set_trace_config(None) if shape is None else rt.set_trace_config(*shape)
            for got in (tree.intersect(dr), batch.intersect(dr, off),
                        tree.intersect(dr, order_rays=True)):
                assert hits_equal(got.cpu().numpy().view(ref.HIT).reshape(-1), want).all(), shape
            for got in (tree.occluded(dr), batch.occluded(dr, off)):
                assert np.array_equal(got.cpu().numpy(), flags), shape
    finally:
        rt.set_trace_config(None)
    tree.status()


@pytest.mark.parametrize("rays_n", [98_305, 600_000, 1_200_000])
def test_compressed_tree_long_rays_end_in_groups(rays_n):
    """A wave's last eight rays are taken over by groups of eight lanes: rays
    along a fan of slivers visit hundreds of nodes while the others miss, in
    the one-ray-per-lane schedule and in runs, with stacks in LDS and (depth
    0) in private memory."""
    fan = scenes.noisy_sphere(400, 60, seed=41)  # slivers around both poles
    verts = np.concatenate([fan, scenes.random_soup(200, 0.1, seed=42)]) * np.float32(8.0)
    aabbs, centers = prep(verts)
    dv = _dev(verts)
    tree = rt.Builder(_dev(centers), aabbs=_dev(flat(aabbs))) \
        .construct_locally_ordered_clustered().trace_tree(dv)
    rays8 = ray_set(verts, rays_n, seed=43, kind="box")
    rays8[:, 4:7] = (0.0, 0.0, 1.0)  # parallel to the axis through the poles
    rays8[::997, 0:2] = np.float32(4.0)  # and some through them
    check = np.unique(np.concatenate([np.arange(0, rays_n, 997), np.arange(0, rays_n, 61)]))
    want = ref.trace_brute(verts, as_rays(rays8[check]), threads=8)
    dr = _dev(rays8)
    try:
        for shape in (None, (64, 0, 800, 0, 16, 1), (128, 8, 1600, 0, 16, 0)):
            rt.set_trace_config(None) if shape is None else rt.set_trace_config(*shape)
            got = tree.intersect(dr).cpu().numpy().view(ref.HIT).reshape(-1)
            assert hits_equal(got[check], want).all(), shape
            occ = tree.occluded(dr).cpu().numpy()
            assert np.array_equal(occ, (got["prim"] != 0xFFFFFFFF).astype(np.uint8)), shape
    finally:
        rt.set_trace_config(None)
    tree.status()
