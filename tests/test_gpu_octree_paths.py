"""Octree extraction's kernels (lhmc_kernels.hip) where their new paths can go
wrong, against the oracle byte for byte.

Nodes are evaluated over the operations that can change a value among a
wavefront's 64 (runs longer than 64 operations, operands below on the value
stack, nested translations, programs whose bounds are not sound), depths of
fewer nodes than a wavefront and of many workgroups, primal vertices on a bit
lattice or sorted, and buffers that are too small in a fresh context, each in
its turn, or larger than needed after a larger call."""
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


# From depth 6 on a fresh context has room for 131072 nodes and primal vertices,
# 32768 cubes and vertices, 131072 indices and a table for 43690 triangles.
# (radius, depth): nodes, primal vertices, mesh vertices (two less than cubes),
# indices.
OUTGROWN = {
    "nothing": (0.2, 6),
    "table_and_indices": (0.3, 7),     # 84113, 101269, 27768, 166596
    "cubes_and_vertices": (0.33, 7),   # 104465, 124903, 33552, 201300
    "primal_vertices": (0.35, 7),      # 116561, 139567, 37920, 227508
    "nodes_of_last_depth": (0.3, 8),   # 339153 (84113 without it)
    "nodes_before_it": (0.45, 8),      # 772689 (193169 without it)
}


@pytest.mark.parametrize("device", [False, True])
@pytest.mark.parametrize("what", sorted(OUTGROWN))
def test_each_buffer_outgrown_on_the_bit_lattice(what, device):
    import torch
    radius, depth = OUTGROWN[what]
    src = DemoSource(Sphere(radius))
    fresh = Context(0)
    try:
        if not device:
            ref = same(fresh, src, depth)
        else:
            ref = O.extract_lhmc(src.program(), depth, 0)
            nv, ni = len(ref.vertices), len(ref.indices)
            v = torch.zeros((nv, 3), device="cuda")
            i = torch.zeros(ni, dtype=torch.int32, device="cuda")
            torch.cuda.synchronize()
            fresh.upload_program(src.program())
            out = A.IsoMeshOut(v.data_ptr(), i.data_ptr(), nv, ni, 0, 0, A.ISO_MEMORY_DEVICE, 0)
            assert fresh.lib.iso_extract_lhmc(fresh.handle, depth, C.byref(out)) == 0
            assert (out.vertex_count, out.index_count) == (nv, ni)
            assert v.cpu().numpy().tobytes() == ref.vertices.tobytes()
            assert np.array_equal(i.cpu().numpy().view(np.uint32), ref.indices)
    finally:
        fresh.close()
    nodes = len(O.lhmc_octree(src.program(), depth)[0])
    assert (nodes > 131072) == what.startswith("nodes")
    assert (len(ref.vertices) > 32768) == (what not in ("nothing", "table_and_indices"))
    assert (len(ref.indices) > 131072) == (what != "nothing")


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
