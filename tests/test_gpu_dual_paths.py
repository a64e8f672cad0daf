"""Dual contouring's sparse samples and brick normals (sparse_kernels.hip,
dc_kernels.hip) against the oracle byte for byte.

Lattices of at least 92^3 samples take the sparse samples: sides around the
4^3 bricks and 16^3 tiles, one wavefront a tile (the other splits:
test_gpu_wavefronts.py), surfaces through lattice points and dual points,
descending lattices.  Normals of every kind of program: long runs, operands below
on the value stack, nested translations, programs whose bounds are not sound; by
central differences of small and large steps, and the program's own."""
import numpy as np
import pytest

from isosurface_amd import _abi as A
from isosurface_amd import workloads as W
from isosurface_amd.sources import (DemoSource, Difference, RectangularPrism, SmoothUnion, Sphere,
                                    Torus, Translate, Union, smooth_union_all, union_all)
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def desc(n, origin=(0.0, 0.0, 0.0), spacing=None):
    d = A.IsoGridDesc()
    d.nx, d.ny, d.nz = n
    s = spacing or tuple(1.0 / (k - 1) for k in n)
    for i in range(3):
        d.origin[i], d.spacing[i] = origin[i], float(np.float32(s[i]))
    d.source = A.ISO_SOURCE_PROGRAM
    return d


def check(ctx, src, d, eps=1e-6, want_mesh=True):
    ctx.upload_program(src.program())
    gpu = ctx.extract_dc(d, eps)
    ref = O.extract_dc(src.program(), O.as_desc(d), eps)
    assert np.array_equal(gpu.indices, ref.indices)
    assert gpu.vertices.tobytes() == ref.vertices.tobytes()
    assert not want_mesh or len(ref.indices) > 0


def spheres(n, k, more=()):
    r = W.SplitMix64(31)
    parts = [Translate(tuple(r.uniform(-0.4, 0.4) for _ in range(3)), Sphere(r.uniform(0.02, 0.1)))
             for _ in range(n)] + list(more)
    return DemoSource(smooth_union_all(parts, k) if k else union_all(parts))


def tree():
    left = Union(Sphere(0.12), Translate((0.1, 0.1, 0.1), RectangularPrism((0.05, 0.3, 0.05))))
    right = Difference(Torus(0.25, 0.05),
                       Translate((0.0, 0.1, 0.0), RectangularPrism((0.3, 0.1, 0.2))))
    return DemoSource(SmoothUnion(Translate((0.02, -0.03, 0.01), left), right, 0.05))


SOURCES = {
    "boxes": lambda: W.boxes_union(32, seed=4),
    "spheres70": lambda: spheres(70, 0.0),
    "smooth130": lambda: spheres(130, 0.03),
    "tree": tree,
    "unbounded": lambda: DemoSource(Union(Sphere(0.3), Translate((1e30, 0.0, 0.0), Sphere(0.1)))),
    "unbounded100": lambda: spheres(100, 0.03, [Translate((1e30, 0.0, 0.0), Sphere(0.1))]),
}


@pytest.mark.parametrize("name", sorted(SOURCES))
@pytest.mark.parametrize("n", [(96, 97, 98), (99, 100, 81), (17, 19, 2600)])
def test_programs_on_ragged_lattices(ctx, name, n):
    check(ctx, SOURCES[name](), desc(n), want_mesh=min(n) > 20)


@pytest.mark.parametrize("n", [(5, 4, 6), (33, 34, 35)])  # dense samples, brick normals
@pytest.mark.parametrize("eps", [1e-3, 0.25])
def test_small_lattices(ctx, n, eps):
    check(ctx, tree(), desc(n), eps, want_mesh=min(n) > 20)


@pytest.mark.parametrize("eps", [1e11, 1e16])  # beyond what bounds of the points allow, too
def test_lattice_without_sound_bounds(ctx, eps):
    src = Union(Sphere(1.0e16), Translate((0.0, 0.0, 1.0e16), Sphere(5.0e15)))
    check(ctx, src, desc((41, 42, 43), origin=(-2.0e16,) * 3, spacing=(1.0e15,) * 3), eps)


def test_steps_without_sound_bounds(ctx):
    check(ctx, tree(), desc((33, 34, 35)), 1e16)


def test_lists_that_do_not_fit(ctx):
    # spheres whose values differ by less than the blend's width everywhere, and
    # some that matter nowhere near them
    r = W.SplitMix64(9)
    long = smooth_union_all([Translate(tuple(r.uniform(-0.02, 0.02) for _ in range(3)),
                                       Sphere(r.uniform(0.2, 0.25))) for _ in range(550)] +
                            [Translate((5.0 + i, 0.0, 0.0), Sphere(0.1)) for i in range(100)], 0.15)
    d = desc((16384, 7, 7), origin=(0.0, 0.47, 0.47), spacing=(1.0 / 16383, 0.01, 0.01))
    check(ctx, DemoSource(long), d)
    check(ctx, DemoSource(Union(Difference(Sphere(0.2), long),
                                Difference(Sphere(0.1), Torus(0.3, 0.05)))), d)


def test_analytic_normals(ctx):
    check(ctx, W.boxes_union(32, seed=4), desc((96, 97, 98)), 0.0)


def test_one_wavefront_per_tile(ctx):
    # 16384 tiles of at most 16 x 3 x 3 samples
    src = Union(Sphere(0.3), Translate((100.0, 0.1, 0.0), RectangularPrism((40.0, 0.2, 0.4))))
    check(ctx, src, desc((262144, 3, 3), origin=(-0.5, -0.3, -0.35), spacing=(0.001, 0.3, 0.31)))


@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_surfaces_on_lattice_and_dual_points(ctx, sign):
    # faces at samples (a multiple of 1/64) and between them (dual values of 0)
    src = Union(RectangularPrism((0.25, 0.125, 0.3125)),
                Translate((0.0078125, 0.0078125, 0.0078125), RectangularPrism((0.125, 0.25, 0.0625))))
    s = sign / 64.0
    check(ctx, src, desc((96, 96, 96), origin=(-48 * s, -48 * s, -48 * s), spacing=(s, s, s)))
