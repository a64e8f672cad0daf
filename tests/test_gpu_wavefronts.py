"""The sparse kernels' splits of a tile among wavefronts (sparse_kernels.hip)
against the oracle byte for byte: eight for up to 2048 tiles, four for fewer
than 16384, one from there on, each side of both lines; signs, dual contouring's
samples and directed values of a lattice, and a batch's signs (four or one, or
the flat pass where many tiles are nearly empty); programs without a value stack
and with one.  The lattices are long rows of
tiles, most of them a few samples thick."""
import numpy as np
import pytest

from isosurface_amd import BatchedMarchingCubes, _abi as A, chunk_desc
from isosurface_amd.sources import Difference, RectangularPrism, Sphere, Torus, Translate, Union, union_all
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def desc(n, width):
    d = A.IsoGridDesc()
    d.nx, d.ny, d.nz = n
    extent = (width, 0.6, 0.62)
    for i, o in enumerate((-0.5, -0.3, -0.35)):
        d.origin[i], d.spacing[i] = o, float(np.float32(extent[i] / (n[i] - 1)))
    d.source = A.ISO_SOURCE_PROGRAM
    return d


def row(n, first, step):
    return union_all(Translate((first + step * i, 0.1, 0.05 * (i % 3)),
                               RectangularPrism((0.3 + 0.02 * i, 0.25, 0.4)) if i % 2 else Sphere(0.45))
                     for i in range(n))


def plain():
    return row(16, 3.0, 16.0)


def stacked():
    return Union(Difference(Sphere(0.3), row(9, 3.0, 27.0)),
                 Difference(row(5, 3.2, 60.0), Translate((20.0, 0.0, 0.0), Torus(9.0, 0.2))))


# 2048 and 2049 tiles, 16383 and 16384
ROWS = [(32768, 5, 5), (32769, 5, 5), (262128, 3, 3), (262129, 3, 3)]
SOURCES = {"plain": plain, "stacked": stacked}


def same(mesh, ref):
    assert len(ref.indices) > 0
    assert np.array_equal(mesh.indices, ref.indices)
    assert mesh.vertices.tobytes() == ref.vertices.tobytes()


@pytest.mark.parametrize("name", sorted(SOURCES))
@pytest.mark.parametrize("n", ROWS)
def test_signs(ctx, n, name):
    src, d = SOURCES[name](), desc(n, 236.0)
    ctx.upload_program(src.program())
    same(ctx.extract_mc(d), O.extract_mc(src.program(), desc=O.as_desc(d)))


@pytest.mark.parametrize("name", sorted(SOURCES))
@pytest.mark.parametrize("n", ROWS)
def test_dual_samples(ctx, n, name):
    src, d = SOURCES[name](), desc(n, 236.0)
    ctx.upload_program(src.program())
    same(ctx.extract_dc(d, 1e-6), O.extract_dc(src.program(), O.as_desc(d), 1e-6))


@pytest.mark.parametrize("name", sorted(SOURCES))
@pytest.mark.parametrize("n", ROWS)
def test_directed_values(ctx, n, name):
    src, d = SOURCES[name](), desc(n, 236.0)
    ctx.upload_program(src.program())
    same(ctx.extract_emc(d, 1e-4), O.extract_emc(src.program(), O.as_desc(d), epsilon=1e-4))


def same_batch(ctx, parts):
    meshes = BatchedMarchingCubes(ctx).extract_meshes(parts)
    found = 0
    for (src, d), m in zip(parts, meshes):
        grid = O.sample_lattice_threads(src.program(), O.as_desc(d), threads=8)
        ref = O.extract_mc(grid=grid, desc=O.as_desc(d))
        assert np.array_equal(m.indices, ref.indices)
        assert m.vertices.tobytes() == ref.vertices.tobytes()
        found += len(ref.indices) > 0
    assert found > len(parts) // 10


@pytest.mark.parametrize("name", sorted(SOURCES))
@pytest.mark.parametrize("chunks", [64, 512])  # of 32 tiles of 1280 samples
def test_batch_signs(ctx, chunks, name):
    same_batch(ctx, [(Translate((-0.25 * i, 0.0, 0.0), SOURCES[name]()), desc((512, 16, 5), 4.0))
                     for i in range(chunks)])


@pytest.mark.parametrize("chunks", [4096, 4097])  # of one tile of 125: the flat pass for more
def test_batches_of_nearly_empty_tiles(ctx, chunks):
    ball = Union(Difference(Sphere(0.25), Sphere(0.3)), Difference(Torus(0.2, 0.1), Sphere(0.2)))
    same_batch(ctx, [(Translate((0.5 + 0.0001 * i, 0.5, 0.5), ball), chunk_desc(4))
                     for i in range(chunks)])
