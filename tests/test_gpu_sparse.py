"""Sparse program classification (sparse_kernels.hip) against the oracle.

Bounds prove the sign of whole 4^3 bricks and only the others are evaluated,
over the operations that matter in their 16^3 tile.  The cases sit where that
can go wrong: lattice sides around the brick and tile edges (all of at least
92^3 samples, where the sparse pass takes over), every primitive and operator
(runs longer than 64 operands, tiles whose list does not fit, nested
translations, operands below on the value stack), surfaces that pass exactly
through lattice points, negative spacings, and programs or lattices whose bounds
are not sound.  The mesh must equal the oracle's byte for byte.  (The splits of a
tile among wavefronts: test_gpu_wavefronts.py.)"""
import numpy as np
import pytest

from isosurface_amd import _abi as A
from isosurface_amd import workloads as W
from isosurface_amd.sources import (Cylinder, DemoSource, Difference, Intersection,
                                    RectangularPrism, SmoothUnion, Sphere, Torus, Translate, Union,
                                    smooth_union_all, union_all)
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def desc(nx, ny, nz, origin=(0.0, 0.0, 0.0), spacing=None):
    d = A.IsoGridDesc()
    d.nx, d.ny, d.nz = nx, ny, nz
    s = spacing or (1.0 / (nx - 1), 1.0 / (ny - 1), 1.0 / (nz - 1))
    for i in range(3):
        d.origin[i], d.spacing[i] = origin[i], float(np.float32(s[i]))
    d.source = A.ISO_SOURCE_PROGRAM
    return d


def check(ctx, src, d, want_mesh=True):
    assert d.nx * d.ny * d.nz >= 786432 and d.nx >= 16
    prog = src.program()
    grid = O.sample_lattice_threads(prog, O.as_desc(d), threads=8)
    ref = O.extract_mc(grid=grid, desc=O.as_desc(d))
    ctx.upload_program(prog)
    gpu = ctx.extract_mc(d)
    assert np.array_equal(gpu.indices, ref.indices)
    assert gpu.vertices.tobytes() == ref.vertices.tobytes()
    if want_mesh:
        assert len(ref.indices) > 0
    cloud = ctx.extract_point_cloud(d)
    assert cloud.tobytes() == O.extract_point_cloud(grid=grid, desc=O.as_desc(d)).tobytes()


def shapes(seed, n):
    r = W.SplitMix64(seed)
    out = []
    for i in range(n):
        c = tuple(r.uniform(-0.4, 0.4) for _ in range(3))
        p = [Sphere(r.uniform(0.03, 0.2)), Torus(r.uniform(0.08, 0.2), r.uniform(0.02, 0.05)),
             RectangularPrism(tuple(r.uniform(0.03, 0.15) for _ in range(3))),
             Cylinder(r.uniform(0.03, 0.15), r.uniform(0.05, 0.2))][i % 4]
        out.append(Translate(c, p))
    return out


def tree(seed, n):
    """Every operator over every primitive, operands below the top included."""
    s = shapes(seed, n)
    left, right = union_all(s[: n // 2]), s[n // 2]
    for i, p in enumerate(s[n // 2 + 1:]):
        right = [Union, Intersection, Difference][i % 3](p, right) if i % 3 != 1 else \
            Union(right, Intersection(p, Translate((0.05, 0.0, -0.03), Sphere(0.3))))
    both = SmoothUnion(Translate((0.02, -0.03, 0.01), left), right, 0.05)
    cut = Union(Sphere(0.06), Translate((0.1, 0.1, 0.1), RectangularPrism((0.05, 0.3, 0.05))))
    return DemoSource(Difference(cut, both))


# sides of 16 q + 0 to 5: the last brick and tile hold one sample, or are full
@pytest.mark.parametrize("n", [(96, 96, 96), (97, 100, 101), (18, 213, 210), (64, 2, 6200),
                               (16, 1000, 50), (1003, 34, 24), (113, 65, 112)])
@pytest.mark.parametrize("seed", [1, 2])
def test_trees_on_ragged_lattices(ctx, n, seed):
    check(ctx, tree(seed, 12), desc(*n), want_mesh=min(n) > 2)


def test_one_wavefront_per_tile(ctx):
    # 27 * 26 * 27 tiles: above the line where one wavefront takes a tile
    check(ctx, tree(3, 8), desc(417, 403, 418))


@pytest.mark.parametrize("n_ops,k", [(70, 0.0), (70, 0.02), (700, 0.0), (600, 0.3)])
def test_long_runs(ctx, n_ops, k):
    r = W.SplitMix64(9)
    parts = [Translate(tuple(r.uniform(-0.45, 0.45) for _ in range(3)),
                       Sphere(r.uniform(0.01, 0.08))) for _ in range(n_ops)]
    # with k = 0.3 almost every operand matters everywhere: the list does not fit
    check(ctx, DemoSource(smooth_union_all(parts, k) if k else union_all(parts)), desc(93, 93, 92))


def cluster(n, far=0):
    """n spheres whose values differ by less than the blend's width everywhere, and
    some that matter nowhere near them."""
    r = W.SplitMix64(9)
    return smooth_union_all([Translate(tuple(r.uniform(-0.02, 0.02) for _ in range(3)),
                                       Sphere(r.uniform(0.2, 0.25))) for _ in range(n)] +
                            [Translate((5.0 + i, 0.0, 0.0), Sphere(0.1)) for i in range(far)], 0.15)


@pytest.mark.parametrize("n,name", [
    ((93, 93, 92), "run"), ((93, 93, 92), "stack"), ((93, 93, 92), "pruned_run"),
    ((93, 93, 92), "pruned_stack"), ((33000, 5, 5), "run"), ((33000, 5, 5), "stack"),
    ((262129, 2, 2), "run"), ((262129, 2, 2), "stack")])  # 8, 4, 1 wavefronts
def test_lists_that_do_not_fit(ctx, n, name):
    long = cluster(550, 100 if "pruned" in name else 0)
    src = DemoSource(long) if name.endswith("run") else DemoSource(
        Union(Difference(Sphere(0.2), long), Difference(Sphere(0.1), Torus(0.3, 0.05))))
    check(ctx, src, desc(*n) if n[1] > 5 else
          desc(*n, origin=(0.0, 0.44, 0.46), spacing=(1.0 / (n[0] - 1), 0.03, 0.03)))


def test_batch_lists_that_do_not_fit(ctx):
    from isosurface_amd import BatchedMarchingCubes, chunk_desc
    for src in (DemoSource(cluster(550)), DemoSource(cluster(550, 100)),
                DemoSource(Union(Difference(Sphere(0.2), cluster(520, 100)),
                                 Difference(Sphere(0.1), Torus(0.3, 0.05))))):
        chunks = [(src, chunk_desc(s)) for s in (16, 33, 48)]
        for (_, d), m in zip(chunks, BatchedMarchingCubes(ctx).extract_meshes(chunks)):
            ref = O.extract_mc(src.program(), desc=O.as_desc(d))
            assert len(ref.indices) > 0 and np.array_equal(m.indices, ref.indices)
            assert m.vertices.tobytes() == ref.vertices.tobytes()


def test_surface_through_lattice_points(ctx):
    # faces on lattice planes: the samples there are exactly 0
    check(ctx, Translate((48.0, 48.0, 48.0), RectangularPrism((20.0, 20.0, 15.0))),
          desc(96, 96, 96, spacing=(1.0, 1.0, 1.0)))
    check(ctx, Translate((48.0, 48.0, 48.0), Sphere(25.0)),
          desc(97, 97, 97, spacing=(1.0, 1.0, 1.0)))


def test_descending_lattice(ctx):
    check(ctx, tree(4, 12), desc(97, 96, 98, origin=(1.0, 0.0, 1.0),
                                 spacing=(-1.0 / 96, 1.0 / 95, -1.0 / 97)))


@pytest.mark.parametrize("radius", [float("inf"), 3.0e38, 1.0e30])
def test_programs_without_sound_bounds(ctx, radius):
    src = DemoSource(Intersection(Sphere(radius), union_all(shapes(5, 6))))
    check(ctx, src, desc(93, 93, 93))


def test_lattice_without_sound_bounds(ctx):
    check(ctx, Sphere(1.0e16), desc(93, 93, 93, origin=(-2.0e16,) * 3, spacing=(4.4e14,) * 3))


def test_empty_and_full(ctx):
    check(ctx, Sphere(0.5), desc(93, 93, 93, origin=(3.0, 3.0, 3.0)), want_mesh=False)
    check(ctx, Sphere(50.0), desc(93, 93, 93), want_mesh=False)


def test_graph_replay_follows_the_program(ctx):
    """A captured extraction replays with the kernel its program needs: another
    program of the same length, with a value stack or without sound bounds,
    captures anew."""
    d = desc(93, 93, 93)
    a = DemoSource(Union(Sphere(0.3), Translate((0.2, 0.1, 0.0), Sphere(0.2))))
    b = DemoSource(Union(Sphere(0.25), Translate((0.1, 0.1, 0.0), Sphere(float("inf")))))
    for src in (a, a, b, a):
        check(ctx, src, d, want_mesh=src is a)
        ref = O.extract_mc(src.program(), desc=O.as_desc(d))
        got = device_mesh(ctx, d, A.ISO_MESH_GRAPH, len(ref.vertices) + 8, len(ref.indices) + 8)
        assert np.array_equal(got[1], ref.indices)
        assert got[0].tobytes() == ref.vertices.tobytes()


def device_mesh(ctx, d, flags, nv, ni):
    import ctypes as C
    v, i = C.c_void_p(), C.c_void_p()
    ctx.check(ctx.lib.iso_device_alloc(ctx.handle, 12 * nv, C.byref(v)), "alloc")
    ctx.check(ctx.lib.iso_device_alloc(ctx.handle, 4 * ni, C.byref(i)), "alloc")
    out = A.IsoMeshOut(v, i, nv, ni, 0, 0, A.ISO_MEMORY_DEVICE, flags)
    try:
        ctx.check(ctx.lib.iso_extract_mc(ctx.handle, C.byref(d), C.byref(out)), "extract")
        hv = np.empty((int(out.vertex_count), 3), np.float32)
        hi = np.empty(int(out.index_count), np.uint32)
        ctx.lib.iso_memcpy_to_host(ctx.handle, hv.ctypes.data, v, hv.nbytes)
        ctx.lib.iso_memcpy_to_host(ctx.handle, hi.ctypes.data, i, hi.nbytes)
    finally:
        ctx.lib.iso_device_free(ctx.handle, v)
        ctx.lib.iso_device_free(ctx.handle, i)
    return hv, hi


@pytest.mark.parametrize("unbounded", [False, True])
def test_batches(ctx, unbounded):
    """Chunks of every size class over trees with a value stack; one program
    without sound bounds takes the whole batch to the dense pass."""
    from isosurface_amd import BatchedMarchingCubes, chunk_desc
    sizes = [15, 16, 2, 17, 31, 32, 3, 33, 48, 63, 64, 65, 1]
    chunks = [(tree(20 + i, 5 + i % 4), chunk_desc(s)) for i, s in enumerate(sizes)]
    if unbounded:
        chunks[4] = (DemoSource(Intersection(Sphere(float("inf")), Sphere(0.4))), chunks[4][1])
    meshes = BatchedMarchingCubes(ctx).extract_meshes(chunks)
    for (src, d), m in zip(chunks, meshes):
        ref = O.extract_mc(src.program(), desc=O.as_desc(d))
        assert np.array_equal(m.indices, ref.indices)
        assert m.vertices.tobytes() == ref.vertices.tobytes()
