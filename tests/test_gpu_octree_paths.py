"""Octree extraction's kernels (lhmc_kernels.hip) where their new paths can go
wrong, against the oracle byte for byte.

Nodes are evaluated over the operations that can change a value among a
wavefront's 64 (runs longer than 64 operations, operands below on the value
stack, nested translations, programs whose bounds are not sound), depths of
fewer nodes than a wavefront and of many workgroups, primal vertices on a bit
lattice or sorted, and every buffer starts too small in a fresh context, or
larger than needed after a larger call."""
import ctypes as C

import numpy as np
import pytest

from isosurface_amd import Context, LinearHashedMarchingCubes, _abi as A
from isosurface_amd import workloads as W
from isosurface_amd.sources import (DemoSource, Difference, RectangularPrism, SmoothUnion, Sphere,
                                    Torus, Translate, Union, smooth_union_all, union_all)
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def spheres(n, k):
    r = W.SplitMix64(21)
    parts = [Translate(tuple(r.uniform(-0.4, 0.4) for _ in range(3)), Sphere(r.uniform(0.02, 0.1)))
             for _ in range(n)]
    return DemoSource(smooth_union_all(parts, k) if k else union_all(parts))


def tree():
    left = Union(Sphere(0.12), Translate((0.1, 0.1, 0.1), RectangularPrism((0.05, 0.3, 0.05))))
    right = Difference(Torus(0.25, 0.05), Translate((0.0, 0.1, 0.0), RectangularPrism((0.3, 0.1, 0.2))))
    return DemoSource(SmoothUnion(Translate((0.02, -0.03, 0.01), left), right, 0.05))


SOURCES = {
    "spheres70": lambda: spheres(70, 0.0),
    "smooth130": lambda: spheres(130, 0.03),
    "tree": tree,
    "unbounded": lambda: DemoSource(Union(Sphere(0.3), Translate((1e30, 0.0, 0.0), Sphere(0.1)))),
    "empty": lambda: DemoSource(Translate((5.0, 0.0, 0.0), Sphere(0.1))),
    "full": lambda: DemoSource(Sphere(5.0)),
}


def same(ctx, src, depth):
    gpu = LinearHashedMarchingCubes(depth, ctx).extract_mesh(src)
    ref = O.extract_lhmc(src.program(), depth, 0)
    assert np.array_equal(gpu.indices, ref.indices)
    assert gpu.vertices.tobytes() == ref.vertices.tobytes()
    return ref


@pytest.mark.parametrize("name", sorted(SOURCES))
def test_programs_match_the_oracle(ctx, name):
    for depth in (2, 3, 4, 6):
        same(ctx, SOURCES[name](), depth)


@pytest.mark.parametrize("depth", [8, 9])  # the deepest bit lattice, the first sorted list
def test_both_sides_of_the_bit_lattice(ctx, depth):
    same(ctx, DemoSource(Sphere(0.2)), depth)


def test_buffers_grow_and_are_reused(ctx):
    fresh = Context(0)
    try:
        for depth in (8, 3, 7, 9, 2):
            same(fresh, DemoSource(Sphere(0.3)), depth)
    finally:
        fresh.close()


def test_device_buffers_too_small(ctx):
    import torch
    src = DemoSource(Sphere(0.3))
    ref = O.extract_lhmc(src.program(), 6, 0)
    ctx.upload_program(src.program())
    nv, ni = len(ref.vertices), len(ref.indices)
    for short_v, short_i in ((0, 0), (1, 0), (0, 1)):
        v = torch.zeros((nv + 8, 3), device="cuda")
        i = torch.zeros(ni + 8, dtype=torch.int32, device="cuda")
        out = A.IsoMeshOut(v.data_ptr(), i.data_ptr(), nv - short_v, ni - short_i, 0, 0,
                           A.ISO_MEMORY_DEVICE, 0)
        st = ctx.lib.iso_extract_lhmc(ctx.handle, 6, C.byref(out))
        assert st == (A.ISO_ERR_CAPACITY if short_v or short_i else 0)
        assert (out.vertex_count, out.index_count) == (nv, ni)
        ctx.synchronize()
        # nothing past the capacities, everything below them
        assert np.array_equal(v[:nv - short_v].cpu().numpy(), ref.vertices[:nv - short_v])
        assert np.array_equal(i[:ni - short_i].cpu().numpy().view(np.uint32), ref.indices[:ni - short_i])
        assert not v[nv - short_v:].any() and not i[ni - short_i:].any()
