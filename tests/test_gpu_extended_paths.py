"""Extended marching cubes' sparse directed values and listed crossings
(sparse_kernels.hip, emc_kernels.hip) against the oracle byte for byte.

Lattices of at least 92^3 samples take the sparse values: every primitive and
operator (lines that miss, tori, which no bound proves, operands below on the
value stack, nested translations, runs of more than 64), sides around bricks
and tiles, surfaces on lattice points, one wavefront a tile (the other splits:
test_gpu_wavefronts.py), crossings off their edges, unbounded programs; analytic
normals and central differences of small and large steps."""
import numpy as np
import pytest

from isosurface_amd import _abi as A
from isosurface_amd import workloads as W
from isosurface_amd.sources import (Cylinder, DemoSource, Difference, Intersection,
                                    RectangularPrism, Sphere, Torus, Translate, Union, union_all)
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


def check(ctx, src, d, eps, want_mesh=True):
    ctx.upload_program(src.program())
    gpu = ctx.extract_emc(d, eps)
    ref = O.extract_emc(src.program(), O.as_desc(d), epsilon=eps)
    assert np.array_equal(gpu.indices, ref.indices)
    assert gpu.vertices.tobytes() == ref.vertices.tobytes()
    assert not want_mesh or len(ref.indices) > 0


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
    s = shapes(seed, n)
    left, right = union_all(s[: n // 2]), s[n // 2]
    for i, p in enumerate(s[n // 2 + 1:]):
        right = [Union, Intersection, Difference][i % 3](p, right) if i % 3 != 1 else \
            Union(right, Intersection(p, Translate((0.05, 0.0, -0.03), Sphere(0.3))))
    return DemoSource(Difference(Translate((0.1, 0.1, 0.1), RectangularPrism((0.05, 0.3, 0.05))),
                                 Union(Translate((0.02, -0.03, 0.01), left), right)))


@pytest.mark.parametrize("n", [(96, 97, 98), (99, 100, 81), (17, 19, 2600)])
@pytest.mark.parametrize("eps", [1e-6, 0.125])
def test_trees_on_ragged_lattices(ctx, n, eps):
    check(ctx, tree(2, 12), desc(n), eps, want_mesh=min(n) > 20)


@pytest.mark.parametrize("eps", [0.0, 1e-4])
@pytest.mark.parametrize("name", ["boxes", "shapes80", "unbounded"])
def test_unions(ctx, name, eps):
    src = {"boxes": lambda: W.boxes_union(32, seed=4),
           "shapes80": lambda: DemoSource(union_all(shapes(5, 80))),
           "unbounded": lambda: DemoSource(Union(RectangularPrism((0.2, 0.3, 0.1)),
                                                 Translate((1e30, 0.0, 0.0), Sphere(0.1))))}[name]()
    check(ctx, src, desc((96, 97, 98)), eps)


# With the coordinates of the last scale times 2^25, bounds of the crossings' box
# are not sound any more.
@pytest.mark.parametrize("scale", [1.0, 2.0**20, 2.0**40])
def test_crossings_off_their_edges(ctx, scale):
    """Inside a spindle torus a corner can be positive in one component only, and
    the crossing of an edge along another lies far outside the edge."""
    src = Union(Torus(0.05 * scale, 0.3 * scale),
                union_all(Translate(tuple(scale * c for c in (0.1 * i - 0.4, 0.05 * i, -0.3)),
                                    Sphere(0.1 * scale)) for i in range(8)))
    d = desc((40, 41, 42), tuple(scale * c for c in (-0.437, -0.463, -0.4)),
             tuple(0.9 * scale / k for k in (39, 40, 41)))
    x, y = (float(np.float32(d.origin[a]) + np.float32(i) * np.float32(d.spacing[a]))
            for a, i in ((0, 12), (1, 20)))
    column = [O.sample_vector(src.program(), x, y,
                              float(np.float32(d.origin[2]) + np.float32(i) * np.float32(d.spacing[2])))
              for i in range(d.nz)]
    ends = [(a[2], b[2]) for a, b in zip(column, column[1:]) if (a > 0).any() != (b > 0).any()]
    assert any(a * b > 0 for a, b in ends)  # a crossing that no interpolation gives
    check(ctx, src, d, 1e-4 * scale)


def test_small_lattices(ctx):
    for n in ((2, 3, 2), (9, 8, 7), (33, 34, 35)):
        check(ctx, tree(3, 8), desc(n), 1e-5, want_mesh=min(n) > 20)


def test_one_wavefront_per_tile(ctx):
    # 16384 tiles of at most 16 x 3 x 3 samples
    src = Union(Sphere(0.3), Translate((100.0, 0.1, 0.0), RectangularPrism((40.0, 0.2, 0.4))))
    check(ctx, src, desc((262144, 3, 3), origin=(-0.5, -0.3, -0.35), spacing=(0.001, 0.3, 0.31)),
          0.0)


@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_surfaces_on_lattice_points(ctx, sign):
    src = Union(Difference(Cylinder(0.125, 0.5), RectangularPrism((0.25, 0.125, 0.3125))),
                Union(Sphere(0.1875), Translate((0.0078125, 0.0, 0.0),
                                                RectangularPrism((0.125, 0.25, 0.0625)))))
    s = sign / 64.0
    check(ctx, src, desc((96, 96, 96), origin=(-48 * s, -48 * s, -48 * s), spacing=(s, s, s)), 1e-3)
