"""Window tiles (plane tiles of a convolution, a stage of channels held for
all taps) on the GPU against float64, with each tile forced and by size:
images smaller than a tile and not dividing it, channel counts that are no
multiple of a stage, columns at the edges of blocks, and operands, of either
side, that do not split into bf16 planes.

Bound: as of the plane tiles, K * 2^-24 of the sum of the products'
magnitudes, and 2^-24 of it for the products left out."""
import numpy as np
import pytest

from tests import contractions as ct
from tests.test_gpu_planes import F32, _check, _fini, _init
from tinyhvm_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=["WINDOW0", "WINDOW1", "WINDOW2", "WINDOW3"], ids=["128x128", "128x64", "64x64", "256x64"])
def hip(request):
    L, saved = _init("1", "0", str(FIRST + int(request.param[-1])))
    yield L
    _fini(L, saved)


FIRST = 18    # the first window tile's number

SHAPES = [(3, 8, 20, 7, 9, 3), (40, 17, 33, 5, 7, 3), (2, 33, 65, 11, 13, 5), (5, 16, 24, 10, 10, 2), (1, 40, 16, 40, 41, 3),
          (70, 64, 64, 9, 8, 3)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_convolution_edges(hip, shape):
    prog, sa, sb = ct.conv("cf", *shape)
    assert "vpos_" in _lib.dense_source(prog)
    rng = np.random.default_rng(sum(shape))
    _check(hip, "cf", prog, rng.standard_normal(sa).astype(np.float32), rng.standard_normal(sb).astype(np.float32),
           shape[1] * shape[5] ** 2, F32)


@pytest.mark.parametrize("side", ["input", "weights"])
@pytest.mark.parametrize("what", ["inf", "nan", "huge", "tiny"])
@pytest.mark.parametrize("shape", [(6, 24, 40, 13, 11, 3), (70, 64, 64, 9, 8, 3)], ids=["in-kernel", "marked"])
def test_operands_that_do_not_split(hip, shape, what, side):
    """The second shape has a shaped f32 kernel, which computes the marked tiles."""
    prog, sa, sb = ct.conv("cf", *shape)
    rng = np.random.default_rng(5)
    x, w = rng.standard_normal(sa).astype(np.float32), rng.standard_normal(sb).astype(np.float32)
    bad, other = (x, w) if side == "input" else (w, x)
    v = bad.reshape(-1)
    at = v.size // 3
    if what == "inf":
        v[at] = np.inf
    elif what == "nan":
        v[at] = np.nan
    elif what == "huge":
        v[at] = np.float32(3.4028235e38)
        other *= np.float32(2.0 ** -10)
    else:
        v[at:at + v.size // 4] *= np.float32(2.0 ** -119)
        other *= np.float32(2.0 ** 100)
    _check(hip, "cf", prog, x, w, shape[1] * shape[5] ** 2, F32)


def test_by_size():
    """The 64-channel convolution keeps its f32 kernel behind the window tile."""
    L, saved = _init("0", "0", "0")
    try:
        shape = (40, 64, 64, 56, 56, 3)
        prog, sa, sb = ct.conv("cf", *shape)
        src = _lib.dense_source(prog)
        assert "vpos_" in src and "redo_(fl_, m0, n0)" in src
        rng = np.random.default_rng(3)
        x, w = rng.standard_normal(sa).astype(np.float32), rng.standard_normal(sb).astype(np.float32)
        _check(L, "cf", prog, x, w, 576, F32)
        x.reshape(-1)[77777] = np.inf
        _check(L, "cf", prog, x, w, 576, F32)
    finally:
        _fini(L, saved)
