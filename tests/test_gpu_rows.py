"""Row sequences on the GPU: every buffer as the same programs leave it when
each is a launch of its own, bit for bit, and the softmax against float64.
Shapes at the edges: the fewest rows, rows that are no multiple of a
workgroup's elements, rows that threads of four straddle (not taken), long
rows. Programs that must not be taken by row follow ones that are: a shifted
row, a column vector of a row vector's buffer, an update in place."""
import ctypes as C

import numpy as np
import pytest

from tests import rowprograms as rp
from tests.rowprograms import COL, MAT, VEC
from tinyhvm_amd import _lib, abi

pytestmark = pytest.mark.gpu
SUM, RMAX, ADD, MUL, SUB, DIV, EXP = (abi.UOP_SUM, abi.UOP_RMAX, abi.UOP_ADD, abi.UOP_MUL, abi.UOP_SUB, abi.UOP_DIV, abi.UOP_EXP)


def two(u):
    return lambda o, a, b: o(u, a, b)


def one(o, v):
    return v


def exp_diff(o, a, b):
    return o(EXP, o(SUB, a, b))


def steps(m, n):
    """(output, leaves, program): buffers by name."""
    p = lambda *a, **kw: rp.program(m, n, *a, **kw)  # noqa: E731
    softmax = [("mx", ["x"], p([MAT], one, reduce=RMAX)),
               ("pick", ["h", "x"], p([MAT, MAT], two(MUL), reduce=SUM, dtypes=[rp.F16, rp.F32])),
               ("se", ["x", "mx"], p([MAT, VEC], exp_diff, reduce=SUM)),
               ("e", ["x", "mx"], p([MAT, VEC], exp_diff)),
               ("s", ["e"], p([MAT], one, reduce=SUM)),
               ("p", ["e", "s"], p([MAT, VEC], two(DIV))),
               ("q", ["p", "c"], p([MAT, COL], two(MUL)))]
    shifted = [("t", ["q"], p([MAT], one, reduce=SUM)),
               ("r", ["q", "t"], p([MAT, (1, 0, 1)], two(ADD))),        # the next row's sum
               ("u", ["q", "t"], p([(n, 1, n), VEC], two(ADD))),        # the next row
               ("v", ["r"], p([MAT], one, reduce=RMAX)),
               ("w", ["r", "v"], p([MAT, (0, 1, 0)], two(ADD)))]        # rows' maxima along a row
    in_place = [("a", ["y"], p([MAT], one, reduce=SUM)),
                ("y", ["y", "a"], p([MAT, VEC], two(ADD))),
                ("b", ["y"], p([MAT], one, reduce=RMAX)),
                ("x", ["y", "b"], p([MAT, VEC], two(SUB))),
                ("a", ["x", "a"], p([MAT, VEC], two(MUL), reduce=SUM))]
    return softmax + shifted + in_place


def run(m, n, data):
    L = _lib.lib()
    L.thvm_hip_shutdown()
    assert L.thvm_hip_init() == 0
    ids = {}
    for k, v in data.items():
        ids[k] = L.thvm_hip_buf_alloc(v.nbytes)
        L.thvm_hip_buf_write(ids[k], v.ctypes.data_as(C.c_void_p), v.nbytes)
    st = steps(m, n)
    for out, leaves, k in st:
        L.thvm_hip_dispatch_uop_kernel(ids[out], (C.c_uint32 * len(leaves))(*[ids[q] for q in leaves]), len(leaves), C.byref(k), 0)
    outs = {}
    for k, v in data.items():
        outs[k] = np.empty_like(v)
        L.thvm_hip_buf_read(ids[k], outs[k].ctypes.data_as(C.c_void_p), v.nbytes)
    assert L.thvm_hip_synchronize() == 0
    L.thvm_hip_shutdown()
    return outs


@pytest.mark.parametrize("m,n", [(2, 256), (65, 260), (64, 1000), (33, 1001), (700, 1024), (4096, 1000), (2100, 5000), (300, 8192), (40, 8196)])
def test_rows_as_separate_launches(m, n, monkeypatch):
    rng = np.random.default_rng(m * 7 + n)
    f = lambda *s: rng.standard_normal(s).astype(np.float32)  # noqa: E731
    data = {"x": 3 * f(m, n), "h": f(m, n).astype(np.float16), "y": f(m, n), "c": f(n)}
    data["x"][0, 5] = np.inf if m == 65 else data["x"][0, 5]
    for k in "epqruw":
        data[k] = np.full((m, n), -7, np.float32)
    for k in ("mx", "pick", "se", "s", "t", "v", "a", "b"):
        data[k] = np.full(m, -7, np.float32)
    monkeypatch.setenv("THVM_HIP_NO_SEQ", "1")
    want = run(m, n, data)
    monkeypatch.delenv("THVM_HIP_NO_SEQ")
    got = run(m, n, data)
    for k in data:
        assert got[k].tobytes() == want[k].tobytes(), k
    if m != 65:
        x = data["x"].astype(np.float64)
        e = np.exp(x - x.max(1, keepdims=True))
        # exp's own error, the difference's and n additions', each within 2^-24 of a term
        err = np.abs(got["p"] - e / e.sum(1, keepdims=True)) / (e / e.sum(1, keepdims=True))
        assert err.max() <= (n + 64) * 2.0 ** -24


def test_passes_are_the_same_kernels_however_many_run_on(monkeypatch):
    """A pass over one matrix, dispatched 1 to 9 times before its launches go
    out: the kernels of the first passes serve all of them."""
    m, n = 300, 512
    st = [("e", ["x", "c"], rp.program(m, n, [MAT, COL], two(MUL))), ("s", ["e"], rp.program(m, n, [MAT], one, reduce=SUM)),
          ("p", ["e", "s"], rp.program(m, n, [MAT, VEC], two(SUB)))]
    L = _lib.lib()
    L.thvm_hip_shutdown()
    assert L.thvm_hip_init() == 0
    rng = np.random.default_rng(3)
    data = {k: rng.standard_normal(s).astype(np.float32) for k, s in (("x", (m, n)), ("c", n), ("e", (m, n)), ("s", m), ("p", (m, n)))}
    ids = {}
    for k, v in data.items():
        ids[k] = L.thvm_hip_buf_alloc(v.nbytes)
        L.thvm_hip_buf_write(ids[k], v.ctypes.data_as(C.c_void_p), v.nbytes)

    def passes(count):
        for _ in range(count):
            for out, leaves, k in st:
                L.thvm_hip_dispatch_uop_kernel(ids[out], (C.c_uint32 * len(leaves))(*[ids[q] for q in leaves]), len(leaves), C.byref(k), 0)
        assert L.thvm_hip_synchronize() == 0
        c, p = (C.c_uint64 * 16)(), np.empty_like(data["p"])
        L.thvm_hip_counters(c, 16)
        L.thvm_hip_buf_read(ids["p"], p.ctypes.data_as(C.c_void_p), p.nbytes)
        return c[2], c[11], p

    compiled, batched, want = passes(2)
    for count in (1, 3, 4, 6, 9):
        c, b, p = passes(count)
        assert c == compiled and b - batched == 3 * count, count    # the three launches of a pass in one
        assert p.tobytes() == want.tobytes()
        batched = b
    L.thvm_hip_shutdown()


@pytest.mark.parametrize("m,n,rows", [(2, 4092, True), (64, 4096, False), (64, 8192, False), (256, 4096, True), (300, 8192, True), (300, 8196, False)],
                         ids=str)
def test_which_rows_are_a_sequence(m, n, rows):
    st = [("e", ["x", "c"], rp.program(m, n, [MAT, COL], two(MUL))), ("s", ["e"], rp.program(m, n, [MAT], one, reduce=RMAX)),
          ("p", ["e", "s"], rp.program(m, n, [MAT, VEC], two(SUB)))]
    L = _lib.lib()
    L.thvm_hip_shutdown()
    assert L.thvm_hip_init() == 0
    x = np.random.default_rng(m + n).standard_normal((m, n)).astype(np.float32)
    c = np.linspace(0.5, 2, n, dtype=np.float32)
    ids = {k: L.thvm_hip_buf_alloc(4 * m * n) for k in "xep"}
    ids.update(c=L.thvm_hip_buf_alloc(4 * n), s=L.thvm_hip_buf_alloc(4 * m))
    for k, v in (("x", x), ("c", c)):
        L.thvm_hip_buf_write(ids[k], v.ctypes.data_as(C.c_void_p), v.nbytes)
    batched = []
    for _ in range(2):
        for out, leaves, k in st:
            L.thvm_hip_dispatch_uop_kernel(ids[out], (C.c_uint32 * len(leaves))(*[ids[q] for q in leaves]), len(leaves), C.byref(k), 0)
        assert L.thvm_hip_synchronize() == 0
        cnt = (C.c_uint64 * 16)()
        L.thvm_hip_counters(cnt, 16)
        batched.append(cnt[11])
    assert batched[1] - batched[0] == (3 if rows else 0)
    p = np.empty_like(x)
    L.thvm_hip_buf_read(ids["p"], p.ctypes.data_as(C.c_void_p), p.nbytes)
    e = x * c
    assert np.array_equal(p, e - e.max(1, keepdims=True))
    L.thvm_hip_shutdown()


def test_passes_in_a_graph():
    """Two passes captured into a graph and launched several times, other
    inputs and eager passes in between: every buffer as the eager passes leave it."""
    m, n = 300, 512
    st = [("e", ["x", "c"], rp.program(m, n, [MAT, COL], two(MUL))), ("s", ["e"], rp.program(m, n, [MAT], one, reduce=SUM)),
          ("p", ["e", "s"], rp.program(m, n, [MAT, VEC], two(SUB))), ("x", ["p"], rp.program(m, n, [MAT], one))]
    L = _lib.lib()
    L.thvm_hip_shutdown()
    assert L.thvm_hip_init() == 0
    rng = np.random.default_rng(4)
    shapes = {"x": (m, n), "c": (n,), "e": (m, n), "s": (m,), "p": (m, n)}
    ids = {k: L.thvm_hip_buf_alloc(4 * int(np.prod(s))) for k, s in shapes.items()}

    def put(k, v):
        L.thvm_hip_buf_write(ids[k], v.ctypes.data_as(C.c_void_p), v.nbytes)

    def get():
        out = {}
        for k, s in shapes.items():
            out[k] = np.empty(s, np.float32)
            L.thvm_hip_buf_read(ids[k], out[k].ctypes.data_as(C.c_void_p), out[k].nbytes)
        return out

    def passes(count):
        for _ in range(count):
            for out, leaves, k in st:
                L.thvm_hip_dispatch_uop_kernel(ids[out], (C.c_uint32 * len(leaves))(*[ids[q] for q in leaves]), len(leaves), C.byref(k), 0)

    c = (1 + rng.random(n)).astype(np.float32) / 2
    put("c", c)
    put("x", rng.standard_normal((m, n)).astype(np.float32))
    passes(2)
    assert L.thvm_hip_synchronize() == 0
    assert L.thvm_hip_graph_begin() == 0
    passes(2)
    g = L.thvm_hip_graph_end()
    assert g
    for _ in range(4):
        x = rng.standard_normal((m, n)).astype(np.float32)
        put("x", x)
        passes(2)
        want = get()
        for k in ("e", "s", "p"):
            put(k, np.full(shapes[k], -7, np.float32))
        put("x", x)
        assert L.thvm_hip_graph_launch(g) == 0
        got = get()
        for k in shapes:
            assert got[k].tobytes() == want[k].tobytes(), k
        passes(1)
        assert L.thvm_hip_synchronize() == 0
    L.thvm_hip_graph_destroy(g)
    L.thvm_hip_shutdown()
