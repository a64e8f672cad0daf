"""The sparse evaluators' square root (f_sqrt, sdf_eval.h) is correctly rounded:
every mesh that must equal the dense evaluation's bit for bit rests on it.
Every nonnegative float is compared on the GPU with the compiler's root, and
that, with f_sqrt where a wavefront holds values of both its branches, with
numpy's IEEE root."""
import ctypes as C

import numpy as np
import pytest

from isosurface_amd.build import SQRT_CHECK

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    assert SQRT_CHECK.exists(), "build the library first (python -m isosurface_amd.build)"
    return C.CDLL(str(SQRT_CHECK))


@pytest.mark.parametrize("points", [1, 4])
def test_every_nonnegative_float(lib, points):
    differing = C.c_uint64(1)
    st = lib.sqrt_differing(C.c_uint32(0), C.c_uint64(0x7F800001), points,  # up to infinity
                            C.byref(differing))
    assert st == 0
    assert differing.value == 0


def test_roots_beside_others_of_their_wavefront(lib):
    rng = np.random.default_rng(5)
    x = rng.integers(0, 0x7F800001, 1 << 20, dtype=np.uint32).view(np.float32)
    ends = np.float32([0.0, 2.0**-96, 2.0**120, np.inf, 1e-45, 2.0**-126])
    edge = np.concatenate([ends.view(np.uint32) + np.uint32(k) for k in range(3)] +
                          [ends[1:3].view(np.uint32) - np.uint32(k) for k in (1, 2)])
    edge = edge[edge <= 0x7F800000].view(np.float32)
    x[rng.integers(0, len(x), 1 << 12)] = rng.choice(edge, 1 << 12)
    # long stretches within the fast branch, with single values outside it
    x[1 << 18:1 << 19] = np.float32(rng.random(1 << 18) * 4)
    x[(1 << 18) + 640 * np.arange(16)] = edge[:16]
    out = np.zeros_like(x)
    assert lib.sqrt_roots(x.ctypes.data_as(C.c_void_p), out.ctypes.data_as(C.c_void_p), len(x)) == 0
    assert out.tobytes() == np.sqrt(x).tobytes()
