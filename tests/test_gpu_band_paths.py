"""The band's tiles and listed certificates (band_kernels.hip) and the fused
training step (mlp_kernels.hip) where they can go wrong.

The certified band's mesh must be the oracle's byte for byte: sides around the
4^3 blocks, the 16^3 tiles and both brick sizes, runs longer than a list,
operands below on the value stack, nested translations, descending lattices,
programs whose bounds are not sound.  Gradients at batches around a
workgroup's 64 samples and above one workgroup per compute unit, against the
float64 restatement; training twice gives the same bits."""
import numpy as np
import pytest

from isosurface_amd import _abi as A
from isosurface_amd import workloads as W
from isosurface_amd.band import NarrowBand
from isosurface_amd.sources import (Cylinder, DemoSource, Difference, RectangularPrism, SmoothUnion,
                                    Sphere, Torus, Translate, Union, smooth_union_all)
from oracle import mlp as M
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


def cluster(far):
    """Spheres whose values differ by less than the blend's width everywhere, and
    some that matter nowhere near them."""
    r = W.SplitMix64(9)
    return smooth_union_all([Translate(tuple(r.uniform(-0.02, 0.02) for _ in range(3)),
                                       Sphere(r.uniform(0.2, 0.25))) for _ in range(550)] +
                            [Translate((5.0 + i, 0.0, 0.0), Sphere(0.1)) for i in range(far)], 0.15)


def smooth(n, more=()):
    r = W.SplitMix64(41)
    return DemoSource(smooth_union_all(
        [Translate(tuple(r.uniform(-0.4, 0.4) for _ in range(3)), Sphere(r.uniform(0.02, 0.06)))
         for _ in range(n)] + list(more), 0.02))


def tree():
    left = Union(Sphere(0.12), Translate((0.1, 0.1, 0.1), RectangularPrism((0.05, 0.3, 0.05))))
    right = Difference(Torus(0.25, 0.05), Translate((0.0, 0.1, 0.0), Cylinder(0.2, 0.3)))
    return DemoSource(SmoothUnion(Translate((0.02, -0.03, 0.01), left), right, 0.05))


SOURCES = {
    "smooth40": lambda: smooth(40),
    "smooth700": lambda: smooth(700),
    "tree": tree,
    "unbounded": lambda: DemoSource(Union(Sphere(0.3), Translate((1e30, 0.0, 0.0), Sphere(0.1)))),
    "unbounded100": lambda: smooth(100, [Translate((1e30, 0.0, 0.0), Sphere(0.1))]),
    "cluster550": lambda: DemoSource(cluster(0)),
    "cluster650": lambda: DemoSource(cluster(100)),
    "cluster650_stack": lambda: DemoSource(Union(Difference(Sphere(0.2), cluster(100)),
                                                 Difference(Sphere(0.1), Torus(0.3, 0.05)))),
}


@pytest.mark.parametrize("name", sorted(SOURCES))
@pytest.mark.parametrize("brick", [0, A.ISO_BAND_BRICK8])
@pytest.mark.parametrize("n", [(17, 33, 18), (33, 32, 31), (67, 50, 40), (9, 8, 130), (83, 81, 70)])
def test_certified_band_is_the_oracles_mesh(ctx, name, brick, n):
    # (the last has more than 128 tiles: lists however long the program, and
    # programs without sound bounds by four wavefronts)
    src = SOURCES[name]()
    band = NarrowBand(ctx)
    ctx.upload_program(src.program())
    for d in (desc(n), desc(n, (1.0, 1.0, 1.0), tuple(-1.0 / (k - 1) for k in n))):
        mesh, stats = band.extract_mesh(d, 0.0, A.ISO_BAND_NO_NETWORK | brick)
        ref = O.extract_mc(src.program(), desc=O.as_desc(d))
        assert np.array_equal(mesh.indices, ref.indices)
        assert mesh.vertices.tobytes() == ref.vertices.tobytes()
        assert stats.exact_samples <= n[0] * n[1] * n[2]
        assert band.missed_cells(d) == 0


@pytest.mark.parametrize("n", [16, 48, 64, 80, 128, 16384, 16400, 16448, 40000])
def test_gradient_at_batch_sizes(ctx, n):
    band = NarrowBand(ctx)
    theta = M.init(3)
    band.set_params(theta)
    rng = np.random.default_rng(n)
    p = rng.random((n, 3)).astype(np.float32)
    t = rng.normal(0, 0.05, n).astype(np.float32)
    w = (rng.random(n) + 0.5).astype(np.float32)
    loss, g = band.gradient(p, t, w, clamp=0.05)
    ref_loss, ref = M.loss_and_grad(theta, p, np.clip(t, -0.05, 0.05), w, 1.0)
    assert abs(loss - ref_loss) <= 1e-3 * ref_loss
    # bf16 weights and activations: 2^-8 an operand, a few layers deep
    assert np.linalg.norm(g - ref) <= 2e-2 * np.linalg.norm(ref)


def test_training_is_reproducible(ctx):
    rng = np.random.default_rng(0)
    p = rng.random((4096, 3)).astype(np.float32)
    t = (np.linalg.norm(p - 0.5, axis=1) - 0.3).astype(np.float32)
    out = []
    for _ in range(2):
        band = NarrowBand(ctx)
        band.init(7)
        band.train(p, t, steps=25, batch=1040, lr=3e-3, clamp=0.05, seed=2)
        out.append(band.get_params().tobytes())
    assert out[0] == out[1]
