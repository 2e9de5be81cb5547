"""Differentiable closest hit: a torch.autograd.Function over the C ABI.

Forward: rtbvh_gpu_intersect / rtbvh_gpu_intersect_mbvh (lowest-(t, id)
rule).  Backward: rtbvh_gpu_adjoint_parts, the analytic adjoint of
o + t d = (1-u-v) v0 + u v1 + v v2 with the hit triangle fixed by the
forward pass (no counterpart in the reference, whose triangle test,
src/builders/spatial_sah.rs:132-163, is forward only).
"""
from __future__ import annotations

import ctypes
import math

import torch

from . import _lib as L
from .api import RAY_FLOATS, TraceTree, _ptr, _require_device, _stream, rays_tensor


def adjoint(vertices: torch.Tensor, rays: torch.Tensor, hits: torch.Tensor,
            grad_tuv: torch.Tensor, grad_vertices: bool = True, grad_rays: bool = True):
    """dL/d(vertices) (N, 9), dL/d(origin) (R, 3), dL/d(direction) (R, 3) from
    dL/d(t, u, v) (R, 3) of the hits (R, 4) of `rays` (R, 8)."""
    _require_device(vertices, "vertices")
    _require_device(rays, "rays")
    _require_device(hits, "hits")
    _require_device(grad_tuv, "grad_tuv")
    verts = vertices.reshape(-1)
    n = verts.numel() // 9
    r = rays.shape[0]
    if rays.shape[1] != RAY_FLOATS or hits.shape != (r, 4) or grad_tuv.shape != (r, 3):
        raise ValueError("rays (R, 8), hits (R, 4) and grad_tuv (R, 3) must agree")
    gv = torch.zeros((n, 9), dtype=torch.float32, device=vertices.device) if grad_vertices else None
    go = torch.empty((r, 3), dtype=torch.float32, device=rays.device) if grad_rays else None
    gd = torch.empty((r, 3), dtype=torch.float32, device=rays.device) if grad_rays else None
    L.check(L.lib().rtbvh_gpu_adjoint(_ptr(verts), n, _ptr(rays), _ptr(hits), r, _ptr(grad_tuv),
                                      _ptr(gv), _ptr(go), _ptr(gd), _stream(rays)),
            "rtbvh_gpu_adjoint")
    return gv, go, gd


_FLOAT32_MAX = torch.finfo(torch.float32).max


def _float32_number(x):
    """A number that a 32-bit float takes as the general form stores it: not
    beyond its range (refused there), nor an integer that is rounded twice."""
    if isinstance(x, int):
        return abs(x) <= 1 << 53
    return isinstance(x, float) and (not math.isfinite(x)
                                     or abs(x) <= _FLOAT32_MAX)


def _pack_rays(origins, directions, t_min, t_max):
    """rays_tensor in one pass where the library's kernel applies: contiguous
    (R, 3) float32 arrays on one device and plain numbers for t_min, t_max."""
    same = (origins.dim() == 2 and origins.shape == directions.shape and origins.shape[1] == 3
            and origins.dtype == directions.dtype == torch.float32
            and origins.device.type == "cuda" and origins.device == directions.device
            and origins.is_contiguous() and directions.is_contiguous())
    if not same or not all(_float32_number(x) for x in (t_min, t_max)):
        return rays_tensor(origins, directions, t_min, t_max)
    # the kernel reads memory: a lazily negated view is not what it holds
    origins, directions = origins.resolve_neg(), directions.resolve_neg()
    r = torch.empty((origins.shape[0], RAY_FLOATS), dtype=torch.float32, device=origins.device)
    L.check(L.lib().rtbvh_gpu_pack_rays(_ptr(origins), _ptr(directions), r.shape[0], float(t_min),
                                        float(t_max), _ptr(r), _stream(r)), "rtbvh_gpu_pack_rays")
    return r


def _split_hits(hits):
    """(t, u, v, prim id as int64, -1 on a miss) of (R, 4) hit records."""
    r = hits.shape[0]
    t, u, v = (torch.empty(r, dtype=torch.float32, device=hits.device) for _ in range(3))
    prim = torch.empty(r, dtype=torch.int64, device=hits.device)
    L.check(L.lib().rtbvh_gpu_split_hits(_ptr(hits), r, _ptr(t), _ptr(u), _ptr(v), _ptr(prim),
                                         _stream(hits)), "rtbvh_gpu_split_hits")
    return t, u, v, prim


class TraceTUV(torch.autograd.Function):
    """(vertices, origins, directions) -> (t, u, v, prim) of the closest hit."""

    @staticmethod
    def forward(ctx, vertices, origins, directions, tree, t_min, t_max):
        verts = vertices.detach().contiguous()
        rays = _pack_rays(origins.detach().contiguous(), directions.detach().contiguous(),
                          t_min, t_max)
        if isinstance(tree, TraceTree):
            # a traversal tree traces its own snapshot of the triangles: the
            # gradients are only those of `vertices` if the snapshot is theirs
            if not tree.built_from(vertices):
                raise ValueError("the TraceTree was built from other vertices, or these were "
                                 "modified since: rebuild it (Bvh.trace_tree) from the vertices "
                                 "passed here")
            hits = tree.intersect(rays)
        else:
            hits = tree.intersect(verts.reshape(-1, 9), rays)
        t, u, v, prim = _split_hits(hits)
        ctx.save_for_backward(verts, rays, hits)
        ctx.mark_non_differentiable(prim)
        return t, u, v, prim

    @staticmethod
    def backward(ctx, gt, gu, gv, _gprim):
        verts, rays, hits = ctx.saved_tensors
        # resolve_neg: complex losses hand back lazily negated views, whose
        # memory holds the opposite sign
        parts = [None if g is None else g.resolve_neg().contiguous() for g in (gt, gu, gv)]
        for name, x in (("vertices", verts), ("rays", rays), ("hits", hits),
                        *((f"grad_{k}", g) for k, g in zip("tuv", parts) if g is not None)):
            _require_device(x, name)
        (n, rest), r = divmod(verts.numel(), 9), rays.shape[0]
        # saved-tensor hooks may have handed back anything
        if rest or rays.shape != (r, RAY_FLOATS) or hits.shape != (r, 4) \
                or any(g is not None and g.shape != (r,) for g in parts):
            raise ValueError("the saved rays (R, 8) and hits (R, 4) and the gradients (R,) "
                             "must agree")
        need_v = ctx.needs_input_grad[0]
        need_r = ctx.needs_input_grad[1] or ctx.needs_input_grad[2]
        d_v = (torch.zeros((n, 9), dtype=torch.float32, device=verts.device) if need_v else None)
        d_o, d_d = ((torch.empty((r, 3), dtype=torch.float32, device=rays.device)
                     for _ in range(2)) if need_r else (None, None))
        L.check(L.lib().rtbvh_gpu_adjoint_parts(_ptr(verts), n, _ptr(rays), _ptr(hits), r,
                                                *(_ptr(g) for g in parts), _ptr(d_v), _ptr(d_o),
                                                _ptr(d_d), _stream(rays)),
                "rtbvh_gpu_adjoint_parts")
        d_v = d_v.view(verts.shape) if d_v is not None else None
        return (d_v, d_o if ctx.needs_input_grad[1] else None,
                d_d if ctx.needs_input_grad[2] else None, None, None, None)


def trace_tuv(tree, vertices: torch.Tensor, origins: torch.Tensor, directions: torch.Tensor,
              t_min: float = 1e-4, t_max: float = 1e34):
    """Closest hit (t, u, v, prim id) of rays against `tree` (a Bvh, Mbvh or
    TraceTree over `vertices`), differentiable in vertices, origins and
    directions.
    Misses return t = t_max, u = v = 0, prim = -1 and zero gradients."""
    return TraceTUV.apply(vertices, origins, directions, tree, t_min, t_max)


__all__ = ["adjoint", "trace_tuv", "TraceTUV", "ctypes"]
