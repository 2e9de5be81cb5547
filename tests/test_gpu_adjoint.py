"""Adjoint of the closest hit (rtbvh_gpu_adjoint, rtbvh_amd.diff.trace_tuv).

No reference counterpart (the reference's triangle test is forward only), so
the gradient is pinned by mathematics, not by reference outputs:
  * an FP64 CPU gradient computed a different way (numpy linear solves of
    M x = s and M^T lambda = g, M = [-d | e1 | e2]) against the kernel's
    closed form in FP32: relative error (norm of the difference over the norm
    of the FP64 gradient) <= 1e-4 for vertex, origin and direction
    gradients;
  * central finite differences of the FP64 forward with the hit triangles
    fixed, against the FP64 gradient: relative error <= 2e-2 at h = 1e-3
    (the truncation error is ~(h / edge)^2 with edges ~0.03) and <= 1e-5 at
    h = 1e-5;
  * central finite differences, h = 1e-3, of the GPU forward itself (full
    re-trace, shared vertex positions moved together so the mesh stays
    watertight), against the GPU gradient of L = sum of w_t t: relative
    error <= 5e-2 (FP32 forward, and rays near an edge may change triangle;
    t is continuous there, u and v are not, so they are left out).
Loss otherwise: L = sum over hit rays of w_t t + w_u u + w_v v, w ~ N(0, 1).
"""
import threading

import numpy as np
import pytest

from rtbvh_amd import scenes

torch = pytest.importorskip("torch")
import rtbvh_amd as rt  # noqa: E402
from rtbvh_amd import _lib as L  # noqa: E402
from rtbvh_amd import diff  # noqa: E402
from rtbvh_amd.diff import trace_tuv  # noqa: E402

pytestmark = pytest.mark.gpu


def _tree(verts, dev):
    aabbs, centers = scenes.triangle_aabbs_centers(verts)
    bvh = rt.Builder(torch.from_numpy(centers).to(dev),
                     aabbs=torch.from_numpy(aabbs).to(dev)).construct_locally_ordered_clustered()
    return rt.Mbvh.from_bvh(bvh)


def _setup(seed=3, n_rays=20000):
    # rays from a sphere of radius 3 aimed at the middle of the displaced
    # sphere (radius 0.35 +- 0.1): no grazing hits, no silhouette crossings
    verts = scenes.noisy_sphere(60, 40, seed=5).astype(np.float32)
    rays = scenes.rays_sphere_to_box(n_rays, (0.42, 0.42, 0.42), (0.58, 0.58, 0.58), seed=seed)
    dev = torch.device("cuda:0")
    tree = _tree(verts, dev)
    rng = np.random.default_rng(seed)
    w = rng.normal(size=(n_rays, 3))
    return verts, rays, tree, w, dev


def _solve_f64(verts64, o, d, prim):
    """(t, u, v) and M for the given triangles, by a float64 linear solve."""
    tri = verts64[prim].reshape(-1, 3, 3)
    v0, v1, v2 = tri[:, 0], tri[:, 1], tri[:, 2]
    m = np.stack([-d, v1 - v0, v2 - v0], axis=-1)
    x = np.linalg.solve(m, (o - v0)[..., None])[..., 0]
    return x, m


def _grad_f64(verts64, o, d, prim, g):
    x, m = _solve_f64(verts64, o, d, prim)
    lam = np.linalg.solve(np.transpose(m, (0, 2, 1)), g[..., None])[..., 0]
    t, u, v = x[:, 0], x[:, 1], x[:, 2]
    gv = np.zeros((len(verts64), 9))
    np.add.at(gv[:, 0:3], prim, -(1.0 - u - v)[:, None] * lam)
    np.add.at(gv[:, 3:6], prim, -u[:, None] * lam)
    np.add.at(gv[:, 6:9], prim, -v[:, None] * lam)
    return gv, lam, t[:, None] * lam, x


def _loss_f64(verts64, o, d, prim, w):
    x, _ = _solve_f64(verts64, o, d, prim)
    return float(np.sum(w * x))


def _rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def _forward_backward(verts, rays, tree, w, dev):
    vt = torch.from_numpy(verts).to(dev).requires_grad_(True)
    o = torch.from_numpy(np.ascontiguousarray(rays[:, 0:3])).to(dev).requires_grad_(True)
    d = torch.from_numpy(np.ascontiguousarray(rays[:, 4:7])).to(dev).requires_grad_(True)
    t, u, v, prim = trace_tuv(tree, vt, o, d)
    hit = prim >= 0
    wt = torch.from_numpy(w).to(dev, torch.float32)
    loss = (wt[:, 0] * torch.where(hit, t, 0) + wt[:, 1] * u + wt[:, 2] * v)[hit].sum()
    loss.backward()
    torch.cuda.synchronize()
    return (t.detach().cpu().numpy(), u.detach().cpu().numpy(), v.detach().cpu().numpy(),
            prim.cpu().numpy(), vt.grad.cpu().numpy(), o.grad.cpu().numpy(), d.grad.cpu().numpy())


def test_calls_beside_a_capture_of_another_thread():
    """A call of 2^19 rays or more takes a workspace: while another thread
    records a graph (torch's default mode, in which an allocation anywhere
    invalidates the recording) its first calls, which allocate and grow the
    workspace, and later ones leave the recording alone.  The first test of
    the file, so that nothing is allocated yet."""
    print("[adjoint_beside_capture]", flush=True)
    verts = torch.rand((100, 9), device="cuda") * 4.0
    source = torch.rand(1000, device="cuda")
    for rays_n in (1 << 19, 1 << 20, 1 << 20, 1 << 22):
        rays, hits, grad = _random_hits(verts, rays_n, rays_n)
        got, want = (torch.zeros((100, 9), device="cuda") for _ in range(2))
        out = torch.zeros(1000, device="cuda")
        torch.cuda.synchronize()
        started, go, errors = threading.Event(), threading.Event(), []

        def record():
            try:
                graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
                with torch.cuda.stream(stream):
                    graph.capture_begin()
                    try:
                        torch.mul(source, 2.0, out=out)
                        started.set()
                        go.wait(60)
                    finally:
                        graph.capture_end()
                for _ in range(3):
                    out.zero_()
                    torch.cuda.synchronize()
                    graph.replay()
                    torch.cuda.synchronize()
                    assert torch.equal(out, source * 2.0)
            except Exception as e:
                errors.append(e)
            finally:
                started.set()

        thread = threading.Thread(target=record)
        thread.start()
        started.wait(60)
        try:
            _add_adjoint(verts, rays, hits, grad, got, torch.cuda.current_stream())
        finally:
            go.set()
            thread.join()
        assert not errors, (rays_n, errors)
        _add_adjoint(verts, rays, hits, grad, want, torch.cuda.current_stream())
        assert torch.allclose(got, want, rtol=1e-4, atol=1e-4 * float(want.abs().max()))


def test_adjoint_matches_fp64_gradient():
    print("[adjoint_fp64]", flush=True)
    verts, rays, tree, w, dev = _setup()
    t, u, v, prim, g_v, g_o, g_d = _forward_backward(verts, rays, tree, w, dev)
    hit = prim >= 0
    assert hit.mean() > 0.5
    verts64 = verts.astype(np.float64)
    o64 = rays[hit, 0:3].astype(np.float64)
    d64 = rays[hit, 4:7].astype(np.float64)
    gv, go, gd, x = _grad_f64(verts64, o64, d64, prim[hit], w[hit])
    # forward agrees with the float64 solve
    assert _rel(np.stack([t[hit], u[hit], v[hit]], 1), x) < 1e-5
    errs = (_rel(g_v, gv), _rel(g_o[hit], go), _rel(g_d[hit], gd))
    print(f"[adjoint_fp64] relative error vertices {errs[0]:.2e} origin {errs[1]:.2e} "
          f"direction {errs[2]:.2e}", flush=True)
    assert max(errs) <= 1e-4, errs
    assert not g_o[~hit].any() and not g_d[~hit].any()


def test_fp64_gradient_matches_central_differences():
    print("[adjoint_fd64]", flush=True)
    verts, rays, tree, w, dev = _setup(seed=4, n_rays=5000)
    _, _, _, prim, _, _, _ = _forward_backward(verts, rays, tree, w, dev)
    hit = prim >= 0
    verts64 = verts.astype(np.float64)
    o64 = rays[hit, 0:3].astype(np.float64)
    d64 = rays[hit, 4:7].astype(np.float64)
    p, wh = prim[hit], w[hit]
    gv, go, gd, _ = _grad_f64(verts64, o64, d64, p, wh)
    # h = 1e-3: truncation error ~ (h / edge)^2 with edges ~0.03, so ~1e-2;
    # h = 1e-5 shrinks it to ~1e-7 and pins the formula tightly
    for h, tol in ((1e-3, 2e-2), (1e-5, 1e-5)):
        rng = np.random.default_rng(0)
        fd, an = [], []
        for tri in rng.choice(np.unique(p), 12, replace=False):
            for c in rng.choice(9, 3, replace=False):
                vp, vm = verts64.copy(), verts64.copy()
                vp[tri, c] += h
                vm[tri, c] -= h
                fd.append((_loss_f64(vp, o64, d64, p, wh) - _loss_f64(vm, o64, d64, p, wh))
                          / (2 * h))
                an.append(gv[tri, c])
        for r in rng.choice(len(p), 12, replace=False):
            for arr, g in ((o64, go), (d64, gd)):
                c = int(rng.integers(3))
                ap, am = arr.copy(), arr.copy()
                ap[r, c] += h
                am[r, c] -= h
                if arr is o64:
                    lp, lm = _loss_f64(verts64, ap, d64, p, wh), _loss_f64(verts64, am, d64, p, wh)
                else:
                    lp, lm = _loss_f64(verts64, o64, ap, p, wh), _loss_f64(verts64, o64, am, p, wh)
                fd.append((lp - lm) / (2 * h))
                an.append(g[r, c])
        err = _rel(np.asarray(an), np.asarray(fd))
        print(f"[adjoint_fd64] h={h:g}: relative error {err:.2e} over {len(fd)} coordinates",
              flush=True)
        assert err <= tol, (h, err)


def test_gpu_gradient_matches_gpu_central_differences():
    print("[adjoint_fd_gpu]", flush=True)
    verts, rays, tree, w, dev = _setup(seed=5, n_rays=20000)
    # t alone: with shared positions moved together t stays continuous, while
    # u and v jump where a ray changes triangle
    w[:, 1:] = 0.0
    _, _, _, prim, g_v, _, _ = _forward_backward(verts, rays, tree, w, dev)
    corners = verts.reshape(-1, 3)
    keys, inverse = np.unique(corners, axis=0, return_inverse=True)
    inverse = inverse.reshape(-1)
    rays_d = torch.from_numpy(rays).to(dev)
    hit0 = prim >= 0

    def loss(vs):
        # the closest hit under the lowest-(t, id) rule does not depend on the
        # tree, so each perturbed mesh gets a tree of its own
        vs = np.ascontiguousarray(vs)
        vd = torch.from_numpy(vs).to(dev)
        hits = _tree(vs, dev).intersect(vd, rays_d).cpu().numpy()
        t, u, v = (hits[:, k].astype(np.float64) for k in range(3))
        hit = hits[:, 3].view(np.uint32) != 0xFFFFFFFF
        return w[:, 0] * t + w[:, 1] * u + w[:, 2] * v, hit

    rng = np.random.default_rng(1)
    used = np.unique(prim[hit0])
    h = 1e-3
    fd, an = [], []
    for tri in rng.choice(used, 10, replace=False):
        corner = int(tri) * 3 + int(rng.integers(3))
        group = np.nonzero(inverse == inverse[corner])[0]  # every copy of this position
        c = int(rng.integers(3))
        vp, vm = corners.copy(), corners.copy()
        vp[group, c] += np.float32(h)
        vm[group, c] -= np.float32(h)
        step = float(vp[group[0], c]) - float(vm[group[0], c])  # 2h after fp32 rounding
        lp, hp = loss(vp.reshape(-1, 9))
        lm, hm = loss(vm.reshape(-1, 9))
        assert np.array_equal(hp, hit0) and np.array_equal(hm, hit0)
        fd.append((lp[hit0].sum() - lm[hit0].sum()) / step)
        an.append(float(sum(g_v.reshape(-1, 3)[k, c] for k in group)))
    err = _rel(np.asarray(an), np.asarray(fd))
    print(f"[adjoint_fd_gpu] relative error {err:.2e} over {len(fd)} shared vertices", flush=True)
    assert err <= 5e-2


def test_trace_tree_snapshot_guard():
    """A TraceTree traces the snapshot of the vertices it was built from;
    trace_tuv refuses vertices that are another tensor or were modified in
    place since, because its gradients would belong to other geometry."""
    print("[adjoint_snapshot_guard]", flush=True)
    verts_np = scenes.noisy_sphere(60, 40, seed=5).astype(np.float32)
    rays = scenes.rays_sphere_to_box(2000, (0.42, 0.42, 0.42), (0.58, 0.58, 0.58), seed=6)
    dev = torch.device("cuda:0")
    aabbs, centers = scenes.triangle_aabbs_centers(verts_np)
    verts = torch.from_numpy(verts_np).to(dev)
    bvh = rt.Builder(torch.from_numpy(centers).to(dev),
                     aabbs=torch.from_numpy(aabbs).to(dev)).construct_locally_ordered_clustered()
    tree = bvh.trace_tree(verts)
    o = torch.from_numpy(np.ascontiguousarray(rays[:, 0:3])).to(dev)
    d = torch.from_numpy(np.ascontiguousarray(rays[:, 4:7])).to(dev)
    t, _, _, prim = trace_tuv(tree, verts.detach().requires_grad_(True), o, d)
    assert (prim >= 0).float().mean().item() > 0.5
    with pytest.raises(ValueError):
        trace_tuv(tree, verts.clone(), o, d)  # equal values, another tensor
    verts[:, 1] += 0.01                       # moved in place after the build
    with pytest.raises(ValueError):
        trace_tuv(tree, verts, o, d)
    # a tree rebuilt over the moved vertices is accepted
    a2, c2 = scenes.triangle_aabbs_centers(verts.cpu().numpy())
    bvh2 = rt.Builder(torch.from_numpy(c2).to(dev),
                      aabbs=torch.from_numpy(a2).to(dev)).construct_locally_ordered_clustered()
    tree2 = bvh2.trace_tree(verts)
    t2, _, _, _ = trace_tuv(tree2, verts, o, d)
    assert not torch.equal(t, t2)


@pytest.mark.parametrize("rays_n, prims", [((1 << 19) - 1, 65), (1 << 19, 64), (1 << 19, 65),
                                           ((1 << 19) + 4097, 3), ((1 << 19) + 4097, 1000),
                                           ((1 << 22) + 5, 70_001), (1 << 20, 1_048_576),
                                           (1 << 20, 1_048_577)])
def test_vertex_gradients_of_many_rays(rays_n, prims):
    """From 2^19 rays on the vertex terms go through buckets of triangles (64
    to a bucket up to 65,536 triangles, then 128 and more; above 1,048,576 they
    go by atomics), tiles of 4096 rays and passes of 2^22.  lambda is dL/d(origin), so the sums have an exact
    reference: the same float32 terms added in float64.  A float32 sum of k
    terms is within (k + 2) 2^-24 of it, relative to the sum of magnitudes."""
    g = torch.Generator("cuda").manual_seed(rays_n + prims)
    verts = torch.rand((prims, 9), device="cuda", generator=g) * 4.0
    rays = torch.rand((rays_n, 8), device="cuda", generator=g) + 0.1
    hits = torch.rand((rays_n, 4), device="cuda", generator=g) * 0.5
    prim = torch.randint(0, prims, (rays_n,), device="cuda", generator=g, dtype=torch.int32)
    prim[::7] = -1  # misses
    hits[:, 3] = prim.view(torch.float32)
    grad = torch.randn((rays_n, 3), device="cuda", generator=g)
    d_v, d_o, d_d = diff.adjoint(verts, rays, hits, grad)
    hit = prim >= 0
    u, v = hits[hit, 1], hits[hit, 2]
    lam = d_o[hit]
    assert not d_o[~hit].any() and not d_d[~hit].any()
    assert torch.equal(d_d[hit], hits[hit, 0:1] * lam)
    w = torch.stack([-((1.0 - u) - v), -u, -v], dim=1)
    terms = (w[:, :, None] * lam[:, None, :]).reshape(-1, 9)
    idx = prim[hit].long()
    want = torch.zeros((prims, 9), dtype=torch.float64, device="cuda")
    size = torch.zeros_like(want)
    want.index_add_(0, idx, terms.double())
    size.index_add_(0, idx, terms.double().abs())
    k = torch.zeros(prims, dtype=torch.float64, device="cuda")
    k.index_add_(0, idx, torch.ones(len(idx), dtype=torch.float64, device="cuda"))
    bound = (k[:, None] + 2.0) * 2.0 ** -24 * size
    assert bool(((d_v.double() - want).abs() <= bound).all())


def _random_hits(verts, rays_n, seed):
    """(rays, hits, gradients of t, u, v) of rays_n rays on random triangles
    of verts.  A ray within 1e-5 of parallel to its triangle (the determinant
    whose inverse scales lambda) is a miss, as the triangle test decides: one
    of 786,432 rays on 40 triangles has 1.0e-7, which rounds to zero in 32
    bits, so that no sum over it is finite."""
    prims = verts.shape[0]
    g = torch.Generator("cuda").manual_seed(seed)
    rays = torch.rand((rays_n, 8), device="cuda", generator=g) + 0.1
    hits = torch.rand((rays_n, 4), device="cuda", generator=g) * 0.5
    prim = torch.randint(0, prims, (rays_n,), device="cuda", generator=g, dtype=torch.int32)
    tri = verts.double().view(-1, 3, 3)[prim.long()]
    normal = torch.linalg.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0])
    prim[(normal * rays[:, 4:7].double()).sum(1).abs() < 1e-5] = -1
    hits[:, 3] = prim.view(torch.float32)
    return rays, hits, torch.randn((rays_n, 3), device="cuda", generator=g)


def _add_adjoint(verts, rays, hits, grad, grad_verts, stream, origin=None):
    """rtbvh_gpu_adjoint adding to grad_verts on `stream`."""
    L.check(L.lib().rtbvh_gpu_adjoint(
        verts.data_ptr(), verts.shape[0], rays.data_ptr(), hits.data_ptr(), rays.shape[0],
        grad.data_ptr(), grad_verts.data_ptr(), origin.data_ptr() if origin is not None else None,
        None, stream.cuda_stream), "rtbvh_gpu_adjoint")


@pytest.mark.parametrize("prims", [40, 3000, 70_001])
@pytest.mark.parametrize("counts", [(1 << 20,), (1 << 20, 1 << 18), (1 << 19, 3 << 18)])
def test_calls_on_several_streams_add_to_one_gradient(counts, prims):
    """The vertex gradients are added to what the buffer holds, also while
    calls on other streams add to it: by buckets (2^19 rays or more) and by
    single atomics at once.  The float32 sum of an initial value and k terms in
    any order is within (k + 2) 2^-24 of the float64 sum, relative to the sum
    of magnitudes."""
    g = torch.Generator("cuda").manual_seed(prims)
    verts = torch.rand((prims, 9), device="cuda", generator=g) * 4.0
    start = torch.randn((prims, 9), device="cuda", generator=g)
    got, want, size = start.clone(), start.double(), start.double().abs()
    k = torch.zeros(prims, dtype=torch.float64, device="cuda")
    calls = []
    for c, rays_n in enumerate(counts):
        rays, hits, grad = _random_hits(verts, rays_n, 100 * prims + c)
        lam = torch.empty((rays_n, 3), device="cuda")
        calls.append((rays, hits, grad, lam, torch.cuda.Stream()))
    torch.cuda.synchronize()
    for rays, hits, grad, lam, stream in calls:
        _add_adjoint(verts, rays, hits, grad, got, stream, lam)
    torch.cuda.synchronize()
    for rays, hits, grad, lam, stream in calls:
        prim = hits[:, 3].contiguous().view(torch.int32)
        hit = prim >= 0
        u, v, idx = hits[hit, 1], hits[hit, 2], prim[hit].long()
        w = torch.stack([-((1.0 - u) - v), -u, -v], dim=1)
        terms = (w[:, :, None] * lam[hit][:, None, :]).reshape(-1, 9).double()
        want.index_add_(0, idx, terms)
        size.index_add_(0, idx, terms.abs())
        k.index_add_(0, idx, torch.ones(len(idx), dtype=torch.float64, device="cuda"))
    bound = (k[:, None] + 2.0) * 2.0 ** -24 * size
    assert bool(((got.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("n", [0, 1, 255, 257])
def test_packed_rays_and_split_hits_equal_the_field_copies(n):
    """One-pass packing and splitting against the per-field forms, with
    arguments that take the general form (other types, strides, tensors for
    t_min) beside them."""
    g = torch.Generator("cuda").manual_seed(n)
    o = torch.rand((n, 3), device="cuda", generator=g)
    d = torch.rand((n, 3), device="cuda", generator=g)
    want = rt.rays_tensor(o, d, 0.25, 7.5)
    assert torch.equal(diff._pack_rays(o, d, 0.25, 7.5), want)
    assert torch.equal(diff._pack_rays(o.double(), d, 0.25, 7.5), want)
    wide = torch.empty((n, 6), device="cuda")
    wide[:, ::2] = o
    assert torch.equal(diff._pack_rays(wide[:, ::2], d, 0.25, 7.5), want)
    t0 = torch.full((n,), 0.25, device="cuda")
    assert torch.equal(diff._pack_rays(o, d, t0, 7.5), want)
    hits = torch.rand((n, 4), device="cuda", generator=g)
    ids = torch.randint(-1, 5, (n,), device="cuda", generator=g, dtype=torch.int32)
    hits[:, 3] = ids.view(torch.float32)
    if n > 4:  # an id beyond 2^31
        hits.view(torch.int32)[3, 3] = -5
    t, u, v, prim = diff._split_hits(hits)
    for got, column in ((t, 0), (u, 1), (v, 2)):
        assert torch.equal(got, hits[:, column])
    assert prim.dtype == torch.int64 and torch.equal(prim, rt.hits_prim(hits))


@pytest.mark.parametrize("x", [1e39, -3.5e38, 1 << 70, 3.4028235e38, 3.4028234663852886e38,
                               float("inf"), float("nan"), 1e-50, True, 7, (1 << 60) + (1 << 36) + 1,
                               np.float64(0.1), np.float32(0.1)])
def test_ray_ends_are_taken_or_refused_as_by_rays_tensor(x):
    """t_min and t_max beyond the 32-bit range are refused, everything else is
    rounded once, whichever form packs the rays."""
    o, d = torch.rand((3, 3), device="cuda"), torch.rand((3, 3), device="cuda")

    def packed(pack, *ends):
        try:
            return pack(o, d, *ends).view(torch.int32)
        except Exception as e:
            return type(e)

    for ends in ((x, 7.5), (0.25, x)):
        want, got = packed(rt.rays_tensor, *ends), packed(diff._pack_rays, *ends)
        assert torch.equal(got, want) if isinstance(want, torch.Tensor) else got is want, ends


@pytest.mark.parametrize("cut", ["vertices", "rays", "hits"])
def test_saved_tensors_of_another_shape_are_refused(cut):
    """Saved-tensor hooks may hand back other tensors than were saved: shapes
    that disagree are an error before anything is launched."""
    verts = torch.rand((5, 9), device="cuda") * 4.0
    aabbs, centers = scenes.triangle_aabbs_centers(verts.cpu().numpy())
    bvh = rt.Builder(torch.from_numpy(centers).cuda(),
                     aabbs=torch.from_numpy(aabbs).cuda()).construct_locally_ordered_clustered()
    columns = {"vertices": 9, "rays": 8, "hits": 4}[cut]

    def unpack(x):
        if x.shape[-1] != columns:
            return x
        return x.reshape(-1)[:-1] if cut == "vertices" else x[:-1].contiguous()

    verts.requires_grad_()
    with torch.autograd.graph.saved_tensors_hooks(lambda x: x, unpack):
        t, u, v, _ = trace_tuv(bvh, verts, torch.rand((7, 3), device="cuda"),
                               torch.rand((7, 3), device="cuda"))
    with pytest.raises((ValueError, RuntimeError)):
        (t + u + v).sum().backward()


@pytest.mark.parametrize("n", [1, 2, 700])
def test_lazily_negated_inputs_and_gradients(n):
    """A complex loss gives a gradient that is a lazily negated view (for one
    ray a contiguous one), and rays may be such views: values count, not what
    the memory holds."""
    verts = torch.tensor([[-4.0, -4.0, 0.0, 4.0, -4.0, 0.5, 0.0, 5.0, 1.0]], device="cuda")
    aabbs, centers = scenes.triangle_aabbs_centers(verts.cpu().numpy())
    bvh = rt.Builder(torch.from_numpy(centers).cuda(),
                     aabbs=torch.from_numpy(aabbs).cuda()).construct_locally_ordered_clustered()
    g = torch.Generator("cuda").manual_seed(n)
    o = torch.rand((n, 3), device="cuda", generator=g) - torch.tensor([0.5, 0.5, 4.0]).cuda()
    d = torch.rand((n, 3), device="cuda", generator=g) * 0.1 + torch.tensor([0, 0, 1.0]).cuda()
    assert torch.equal(diff._pack_rays(torch._neg_view(o), torch._neg_view(d), 0.25, 7.5),
                       rt.rays_tensor(-o, -d, 0.25, 7.5))
    verts.requires_grad_(), o.requires_grad_(), d.requires_grad_()
    t, u, v, prim = trace_tuv(bvh, verts, o, d)
    assert bool((prim == 0).all())
    weight = torch.complex(torch.rand(n, device="cuda", generator=g), torch.ones(n, device="cuda"))

    def loss(a, b):
        return (torch.complex(a, b).conj() * weight).abs().sum()

    seen = []
    u.register_hook(lambda x: seen.append(x.is_neg()))
    got = torch.autograd.grad(loss(t, u), [verts, o, d])
    assert seen == [True]
    leaves = [x.detach().clone().requires_grad_() for x in (t, u)]
    gt, gu = (x.resolve_neg() for x in torch.autograd.grad(loss(*leaves), leaves))
    grad = torch.stack([gt, gu, torch.zeros_like(gt)], dim=1)
    hits = torch.stack([t, u, v, prim.to(torch.int32).view(torch.float32)], 1).detach()
    want = diff.adjoint(verts.detach(), rt.rays_tensor(o.detach(), d.detach()),
                        hits.contiguous(), grad.contiguous())
    assert torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])
    # the float atomics' order differs from run to run: (n + 2) 2^-24 of each
    # magnitude, of which every term here is at most |dL/do|
    size = want[1].abs().sum(0).repeat(3)
    assert bool(((got[0] - want[0]).abs() <= 2 * (n + 2) * 2.0 ** -24 * size).all())


def test_backward_of_one_output_and_of_expanded_gradients():
    """Gradients that autograd leaves out are zeros, and a sum's gradient is
    one number expanded over the rays (stride 0)."""
    verts = torch.from_numpy(scenes.noisy_sphere(40, 30, seed=3)).cuda().requires_grad_()
    aabbs, centers = scenes.triangle_aabbs_centers(verts.detach().cpu().numpy())
    bvh = rt.Builder(torch.from_numpy(centers).cuda(),
                     aabbs=torch.from_numpy(aabbs).cuda()).construct_locally_ordered_clustered()
    rays = torch.from_numpy(scenes.rays_sphere_to_box(3000, [0.2] * 3, [0.8] * 3, seed=4)).cuda()
    o = rays[:, 0:3].contiguous().requires_grad_()
    d = rays[:, 4:7].contiguous().requires_grad_()
    t, u, v, prim = trace_tuv(bvh, verts, o, d)
    assert int((prim >= 0).sum()) > 1000
    got = torch.autograd.grad(u.sum(), [verts, o, d])
    hits = torch.stack([t.detach(), u.detach(), v.detach(),
                        prim.to(torch.int32).view(torch.float32)], dim=1).contiguous()
    grad = torch.zeros((len(rays), 3), device="cuda")
    grad[:, 1] = 1.0
    want = diff.adjoint(verts.detach(), rays, hits, grad)
    assert torch.allclose(got[0], want[0], rtol=1e-5, atol=1e-5 * float(want[0].abs().max()))
    assert torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])
