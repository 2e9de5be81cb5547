"""The compressed tree's edge cases on the kernel that gives a ray one lane.

Up to 98,304 rays a compressed tree is traced with eight lanes a ray, so the
scenes that pin its box tests (zero direction components, face planes, t_min
and t_max at a hit, far-off and huge scenes, duplicated and degenerate
triangles, deep chains, spatial splits) reach the kernel of larger launches
only when their rays are repeated past that count.
"""
import pytest

from tests import test_gpu_build, test_gpu_spatial

torch = pytest.importorskip("torch")
import rtbvh_amd as rt  # noqa: E402

pytestmark = pytest.mark.gpu

FEW = 98_304


@pytest.fixture(autouse=True)
def rays_repeated(monkeypatch):
    """TraceTree traversals of few rays trace them in turn until there are more
    than 98,304, and return the first of the equal results."""
    used = []

    def many(method):
        def call(self, rays, out=None, order_rays=False):
            n = rays.shape[0]
            if n == 0 or n > FEW or self.width != 8 or order_rays or out is not None:
                return method(self, rays, out, order_rays)
            reps = FEW // n + 1
            got = method(self, rays.repeat(reps, 1))
            bits = got.view(torch.int32) if got.dtype == torch.float32 else got
            assert bool((bits.view(reps, n, -1) == bits[:n].view(1, n, -1)).all())
            used.append(n)
            return got[:n].contiguous()
        return call

    monkeypatch.setattr(rt.TraceTree, "intersect", many(rt.TraceTree.intersect))
    monkeypatch.setattr(rt.TraceTree, "occluded", many(rt.TraceTree.occluded))
    yield
    assert used


@pytest.mark.parametrize("kind,ppl", [("ploc", None), ("binned", 4)])
def test_structure_and_hits(kind, ppl):
    test_gpu_build.test_trace_tree8_structure_and_hits(kind, ppl)


@pytest.mark.parametrize("n", [1, 2, 9, 100])
def test_small(n):
    test_gpu_build.test_trace_tree8_small(n)


@pytest.mark.parametrize("offset", [0.0, 3.0e4])
def test_flat_scene_axis_rays(offset):
    test_gpu_build.test_trace_tree8_flat_scene_axis_rays(offset)


@pytest.mark.parametrize("scale,offset", [(0.1, 0.0), (1.0, 1.0e6), (1.0e12, 0.0),
                                          (1.0, -3.0e4)])
def test_scales_and_offsets(scale, offset):
    test_gpu_build.test_trace_tree8_scales_and_offsets(scale, offset)


def test_duplicates_and_degenerates():
    test_gpu_build.test_trace_tree8_duplicates_and_degenerates()


def test_spatial_duplicates_degenerates_and_flat():
    test_gpu_spatial.test_spatial_duplicates_degenerates_and_flat()


def test_spatial_deep_chain():
    test_gpu_spatial.test_spatial_deep_chain(None)
