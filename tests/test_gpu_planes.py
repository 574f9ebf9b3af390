"""Plane tiles on the GPU: every committed trace with each tile forced, under
the kernel-boundary parity of tests/test_gpu_parity.py; contractions at the
edges of tiles, groups and K splits against float64; operands that do not
split into bf16 planes (infinities, NaN, the largest and the smallest
values); and the routes by size.

Bounds: a sum of K products in any order of f32 additions is within
K * 2^-24 of the sum of the products' magnitudes; the products left out of
the split add at most 2^-24 of it. f16 results are rounded once more
(2^-11, and half the smallest f16 step)."""
import ctypes as C
import os

import numpy as np
import pytest

from tests import contractions as ct
from tests import tracetools as tt
from tests.test_gpu_dense import dense_tolerance
from tests.test_gpu_parity import _oracle, kernel_parity
from tinyhvm_amd import _lib, abi

pytestmark = pytest.mark.gpu
F32, F16 = abi.DTYPE_F32, abi.DTYPE_F16
KNOBS = ("THVM_HIP_DENSE_FORCE", "THVM_HIP_DENSE_SPLITS", "THVM_HIP_DENSE_TILE")


def _init(force, splits, tile):
    saved = {k: os.environ.get(k) for k in KNOBS}
    os.environ.update(zip(KNOBS, (force, splits, tile)))
    L = _lib.lib()
    L.thvm_hip_shutdown()
    assert L.thvm_hip_init() == 0
    return L, saved


def _fini(L, saved):
    L.thvm_hip_shutdown()
    for k, v in saved.items():
        if v is None:
            os.environ.pop(k, None)
        else:
            os.environ[k] = v


# (split-K, tile): 12 and 13 128x128 (two LDS stages, one), 14 and 15 128x64, 16 and 17 64x64; 0 by size
@pytest.fixture(scope="module", params=[("1", "12"), ("3", "13"), ("2", "14"), ("1", "15"), ("3", "16"), ("1", "17"), ("0", "0")],
                ids=["128x128d", "128x128-split3", "128x64d-split2", "128x64", "64x64d-split3", "64x64", "by-size"])
def hip(request):
    L, saved = _init("1" if request.param[1] != "0" else "0", *request.param)
    yield L
    _fini(L, saved)


@pytest.mark.parametrize("path", tt.fixtures(), ids=lambda p: p.split("/")[-1])
def test_trace_parity(hip, path):
    kr, e2e = kernel_parity(hip.thvm_hip_backend(), hip.thvm_hip_buf_read, hip.thvm_hip_synchronize, _oracle(), path,
                            tol_fn=dense_tolerance)
    assert not [r for r in kr if not r[1]], kr
    assert not [r for r in e2e if not r[1]], e2e


def _dispatch(L, k, a, b, n_out, out_dt):
    ids = []
    try:
        for x in (a, b):
            i = L.thvm_hip_buf_alloc(x.nbytes)
            L.thvm_hip_buf_write(i, x.ctypes.data_as(C.c_void_p), x.nbytes)
            ids.append(i)
        out = np.full(n_out, np.nan, np.float16 if out_dt == F16 else np.float32)
        o = L.thvm_hip_buf_alloc(out.nbytes)
        L.thvm_hip_buf_write(o, out.ctypes.data_as(C.c_void_p), out.nbytes)
        ids.append(o)
        L.thvm_hip_dispatch_uop_kernel(o, (C.c_uint32 * 2)(*ids[:2]), 2, C.byref(k), 0)
        L.thvm_hip_buf_read(o, out.ctypes.data_as(C.c_void_p), out.nbytes)
        assert L.thvm_hip_synchronize() == 0
        return out
    finally:
        for i in ids:
            L.thvm_hip_buf_free(i)


def _check(L, kind, k, a, b, kk, dt):
    with np.errstate(all="ignore"):
        want, mag = ct.reference(kind, a, b)
    got = _dispatch(L, k, a, b, want.size, dt).astype(np.float64).reshape(want.shape)
    with np.errstate(all="ignore"):
        ref = want.astype(np.float16 if dt == F16 else np.float32).astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    assert np.array_equal(got[inf], ref[inf])
    ok = np.isfinite(ref)
    bound = (kk + 2) * 2.0 ** -24 * mag[ok] + 2.0 ** -149
    if dt == F16:
        bound = bound + np.abs(want[ok]) * 2.0 ** -11 + 2.0 ** -25
    worst = np.max(np.abs(got[ok] - want[ok]) / bound) if ok.any() else 0.0
    assert worst <= 1.0, worst


# edges of tiles (64, 128), of groups (4, 8), of stages (32, 64), and of pairs of rows
SIZES = [(64, 64, 64), (128, 96, 128), (65, 33, 63), (129, 771, 130), (63, 4, 17), (16, 257, 16), (200, 130, 72), (17, 8, 300)]


@pytest.mark.parametrize("dt", [F32, F16], ids=["f32", "f16"])
@pytest.mark.parametrize("m,k,n", SIZES, ids=lambda v: str(v))
@pytest.mark.parametrize("kind", ["nn", "nt", "tn"])
def test_matmul_edges(hip, kind, m, k, n, dt):
    prog, sa, sb = ct.matmul(kind, m, k, n, dt)
    rng = np.random.default_rng(m * 7 + k * 3 + n)
    f = np.float16 if dt == F16 else np.float32
    _check(hip, kind, prog, rng.uniform(-1, 1, sa).astype(f), rng.uniform(-1, 1, sb).astype(f), k, dt)


@pytest.mark.parametrize("shape", [(3, 8, 20, 7, 9, 3), (2, 33, 17, 11, 13, 5), (5, 16, 24, 10, 10, 1), (1, 4, 70, 12, 16, 3)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("kind", ["cf", "dw"])
def test_convolution_edges(hip, kind, shape):
    prog, sa, sb = ct.conv(kind, *shape)
    rng = np.random.default_rng(sum(shape))
    b, ci, _co, h, w, ks = shape
    kk = ci * ks * ks if kind == "cf" else b * h * w
    _check(hip, kind, prog, rng.standard_normal(sa).astype(np.float32), rng.standard_normal(sb).astype(np.float32), kk, F32)


@pytest.mark.parametrize("what", ["inf", "nan", "huge", "tiny", "subnormal"])
def test_operands_that_do_not_split(hip, what):
    """One row, or one element, that has no exact bf16 planes; the tile it is
    in keeps the f32 instruction's result, and its neighbours theirs."""
    m, k, n = 200, 260, 150
    prog, sa, sb = ct.matmul("nn", m, k, n)
    rng = np.random.default_rng(5)
    a, b = rng.uniform(-1, 1, sa).astype(np.float32), rng.uniform(-1, 1, sb).astype(np.float32)
    if what == "inf":
        a[3, 7], b[200, 100] = np.inf, -np.inf
        a[150, 200] = 0.0                    # 0 * -inf is NaN
    elif what == "nan":
        a[70, 1] = np.nan
    elif what == "huge":
        a[5, 5] = a[5, 9] = np.float32(3.4028235e38)     # rounds past the bf16 range
        b[5, :], b[9, :] = 0.5, 0.25
    elif what == "tiny":
        a[:64] *= np.float32(2.0 ** -119)
        b *= np.float32(2.0 ** 100)
    else:
        a[10] = rng.integers(1, 1000, k).astype(np.float32) * np.float32(1e-45)
        b *= np.float32(2.0 ** 110)
    _check(hip, "nn", prog, a, b, k, F32)


def test_f16_subnormals_and_infinities(hip):
    prog, sa, sb = ct.matmul("nt", 70, 130, 66, F16)
    rng = np.random.default_rng(6)
    a, b = rng.uniform(-1, 1, sa).astype(np.float16), rng.uniform(-1, 1, sb).astype(np.float16)
    a[3] = (rng.integers(1, 1000, 130) * 2.0 ** -24).astype(np.float16)
    b[5] *= np.float16(512)
    a[40, 7], b[9, 20] = np.inf, np.nan
    _check(hip, "nt", prog, a, b, 130, F16)


@pytest.mark.parametrize("what", ["plain", "inf", "tiny"])
@pytest.mark.parametrize("case", [("nn", 2048, 1024, 2048), ("dw", 16, 128, 64, 56, 56, 3)], ids=["matmul", "weight-gradient"])
def test_marked_tiles_take_the_f32_kernel(case, what):
    """Contractions with a shaped f32 kernel run as a plane tile whose tiles
    that did not split exactly that kernel computes, split over K or not."""
    kind = case[0]
    prog, sa, sb = ct.matmul(*case) if kind == "nn" else ct.conv(*case)
    assert "redo_(" in _lib.dense_source(prog) and "bf_" in _lib.dense_source(prog)
    rng = np.random.default_rng(11)
    a, b = rng.uniform(-1, 1, sa).astype(np.float32), rng.uniform(-1, 1, sb).astype(np.float32)
    if what == "inf":
        a.reshape(-1)[12345] = np.inf
    elif what == "tiny":
        a.reshape(-1)[: a.size // 20] *= np.float32(2.0 ** -118)
        b *= np.float32(2.0 ** 90)
    L, saved = _init("0", "0", "0")
    try:
        _check(L, kind, prog, a, b, case[2] if kind == "nn" else case[1] * case[4] * case[5], F32)
    finally:
        _fini(L, saved)


@pytest.mark.parametrize("kind,m,k,n", [("nn", 1031, 771, 600), ("nt", 1031, 771, 501)])
def test_buffers_shorter_than_the_plan_was_made_for(kind, m, k, n):
    """A program that ran as a plane tile, dispatched with a left operand that
    ends early (what lies past the end reads as 0): the f32 kernel that the
    plane tile takes the place of runs it, and full buffers take the tile again."""
    prog, sa, sb = ct.matmul(kind, m, k, n)
    assert "split2" in _lib.dense_source(prog) and "redo_(" not in _lib.dense_source(prog)
    rng = np.random.default_rng(k)
    a, b = rng.uniform(-1, 1, sa).astype(np.float32), rng.uniform(-1, 1, sb).astype(np.float32)
    short = a.reshape(-1)[: a.size - 3 * k - 5].copy()
    padded = np.concatenate([short, np.zeros(a.size - short.size, np.float32)]).reshape(sa)
    L, saved = _init("0", "0", "0")
    try:
        cnt = (C.c_uint64 * 2)()
        for x, full in ((a, a), (short, padded), (a, a)):
            L.thvm_hip_counters(cnt, 2)
            n0 = cnt[1]
            want, mag = ct.reference(kind, full, b)
            got = _dispatch(L, prog, x, b, want.size, F32).reshape(want.shape)
            L.thvm_hip_counters(cnt, 2)
            assert cnt[1] == n0 + 1                     # on the matrix cores
            assert np.all(np.abs(got - want) <= (k + 2) * 2.0 ** -24 * mag + 2.0 ** -149)
    finally:
        _fini(L, saved)


# (program, forced tile): a plane tile, and a window tile
SMALL = [("nn", (200, 260, 150), "17"), ("cf", (9, 24, 40, 29, 37, 5), "20")]


@pytest.mark.parametrize("e", [-50, -60, -64, -68], ids=lambda e: "2^%d" % e)
@pytest.mark.parametrize("kind,shape,tile", SMALL, ids=["plane", "window"])
def test_small_products(kind, shape, tile, e):
    """Operands that split exactly, but whose planes' products are subnormal:
    a step of the K / 16 * 6 in the sum may lose half of 2^-149 besides."""
    prog, sa, sb = ct.matmul(kind, *shape) if kind == "nn" else ct.conv(kind, *shape)
    kk = shape[1] if kind == "nn" else shape[1] * shape[5] ** 2
    rng = np.random.default_rng(8)
    a, b = (rng.uniform(1, 2, s) * rng.choice([-1, 1], s) for s in (sa, sb))
    a, b = ((v * 2.0 ** e).astype(np.float32) for v in (a, b))
    L, saved = _init("1", "0", tile)
    try:
        assert "split2" in _lib.dense_source(prog)
        want, mag = ct.reference(kind, a, b)
        got = _dispatch(L, prog, a, b, want.size, F32).reshape(want.shape)
        assert np.all(np.abs(got - want) <= (kk + 2) * 2.0 ** -24 * mag + (kk * 6 / 16 + 8) * 2.0 ** -150)
    finally:
        _fini(L, saved)


@pytest.mark.parametrize("factor", ["power-of-two", "any"])
@pytest.mark.parametrize("kind,shape,tile", [("nn", (192, 192, 150), "17"), ("cf", (5, 32, 32, 13, 11, 3), "20")], ids=["plane", "window"])
def test_sums_of_one_product(kind, shape, tile, factor):
    """A diagonal operand: the product itself, exactly where the factor is a
    power of two; else the products left out (2^-24 of it), the rounding of
    the small ones' sum (2^-31) and that of the result (2^-24)."""
    prog, sa, sb = ct.matmul(kind, *shape) if kind == "nn" else ct.conv(kind, *shape)
    rng = np.random.default_rng(9)
    n = sa[1]
    d = 2.0 ** rng.integers(-3, 4, n) if factor == "power-of-two" else rng.uniform(1, 2, n)
    worst = np.array([0x3F807FC0], np.uint32).view(np.float32)[0]     # its square loses nearly 2^-24
    x = rng.uniform(1, 2, sb if kind == "nn" else sa)
    x.reshape(-1)[::7] = worst
    x = x.astype(np.float32)
    if factor == "any":
        d[::5] = worst
    d = d.astype(np.float32)
    if kind == "nn":
        a, b = np.diag(d), x
    else:
        a, b = x, np.zeros(sb, np.float32)
        b[np.arange(n), np.arange(n), 1, 1] = d
    L, saved = _init("1", "0", tile)
    try:
        assert "split2" in _lib.dense_source(prog)
        want, _ = ct.reference(kind, a, b)
        got = _dispatch(L, prog, a, b, want.size, F32).reshape(want.shape)
        if factor == "any":
            assert np.all(np.abs(got - want) <= (2 + 2.0 ** -7) * 2.0 ** -24 * np.abs(want))
        else:
            assert np.array_equal(got, want)
    finally:
        _fini(L, saved)


def test_timing_covers_the_kernel_behind_the_plane_tile():
    """The events of thvm_hip_time_contraction hold the f32 kernel that
    computes the marked tiles: with every tile marked the pair measures more
    than the plane tile's time and most of the f32 kernel's."""
    hip = C.CDLL("libamdhip64.so")
    hip.hipEventCreate.argtypes = [C.POINTER(C.c_void_p)]
    hip.hipEventSynchronize.argtypes = [C.c_void_p]
    hip.hipEventElapsedTime.argtypes = [C.POINTER(C.c_float), C.c_void_p, C.c_void_p]
    m, k, n = 2048, 2048, 2048
    prog, sa, sb = ct.matmul("nn", m, k, n)
    rng = np.random.default_rng(2)
    a, b = rng.uniform(-1, 1, sa).astype(np.float32), rng.uniform(-1, 1, sb).astype(np.float32)
    bad = a.copy()
    bad[::16, 0] = np.inf                     # a row of every tile
    leaves = lambda ids: (C.c_uint32 * 2)(*ids)  # noqa: E731

    def best(x, planes):
        os.environ.pop("THVM_HIP_DENSE_NOPLANES", None)
        if not planes:
            os.environ["THVM_HIP_DENSE_NOPLANES"] = "1"
        L, saved = _init("0", "0", "0")
        ids = []
        for v in (x, b):
            ids.append(L.thvm_hip_buf_alloc(v.nbytes))
            L.thvm_hip_buf_write(ids[-1], v.ctypes.data_as(C.c_void_p), v.nbytes)
        out = L.thvm_hip_buf_alloc(4 * m * n)
        e = [C.c_void_p(), C.c_void_p()]
        for v in e:
            assert hip.hipEventCreate(C.byref(v)) == 0
        times = []
        for _ in range(8):
            L.thvm_hip_time_contraction(*e)
            L.thvm_hip_dispatch_uop_kernel(out, leaves(ids), 2, C.byref(prog), 0)
            assert L.thvm_hip_time_contraction(None, None) == 1
            t = C.c_float()
            assert hip.hipEventSynchronize(e[1]) == 0 and hip.hipEventElapsedTime(C.byref(t), *e) == 0
            times.append(t.value)
        _fini(L, saved)
        os.environ.pop("THVM_HIP_DENSE_NOPLANES", None)
        return min(times)

    plain, f32, both = best(a, True), best(a, False), best(bad, True)
    assert both > plain + 0.6 * f32, (plain, f32, both)
