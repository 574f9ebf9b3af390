"""Column sums (a workgroup per 4 to 16 columns, or 2 to 8 of 16 bits) on the GPU,
against float64: rows and columns at the edges of slices, steps and column
blocks, f32 and f16, a product of two tensors, and a factor per column; and
which programs take them.

Bound: the result of n f32 additions in any order is within n * 2^-24 of the
sum of the magnitudes; here an output goes through at most rows / 64 + 32
(the tests' shapes: 16 to 512 slices), and an f16 result is
rounded once more."""
import ctypes as C

import numpy as np
import pytest

from tinyhvm_amd import _lib, abi

F32, F16 = abi.DTYPE_F32, abi.DTYPE_F16


def column_sum(m, n, dt=F32, kind="plain"):
    """out[g] = sum over r of x[r, g] (plain), x[r, g] * y[r, g] (product) or x[r, g] * w[g] (factor)."""
    k = abi.UOpKernel()
    c = [0]

    def op(t, a=0, b=0, imm=0):
        o = k.ops[c[0]]
        o.type, o.arg[0], o.arg[1], o.imm.u = t, a, b, imm
        c[0] += 1
        return c[0] - 1

    gid, acc, loop = op(abi.KOP_GID), op(abi.KOP_ACC_INIT), op(abi.KOP_RANGE, imm=m)
    row = op(abi.KOP_IDX, op(abi.KOP_MOD, loop, imm=m), op(abi.KOP_CONST_U), n)
    col = op(abi.KOP_MOD, op(abi.KOP_GID), imm=n)
    v = op(abi.KOP_LOAD, op(abi.KOP_IDX, row, col, 1), imm=1)
    if kind != "plain":
        u = op(abi.KOP_LOAD, op(abi.KOP_IDX, row, col, 1) if kind == "product" else col, imm=2)
        v = op(abi.KOP_ALU, v, u, abi.UOP_MUL)
    op(abi.KOP_ACC, acc, v, abi.UOP_SUM)
    op(abi.KOP_ENDRANGE, loop)
    op(abi.KOP_STORE, gid, acc)
    leaves = 1 if kind == "plain" else 2
    k.n_ops, k.n_leaves, k.n_bufs = c[0], leaves, 1 + leaves
    k.rank = k.full_shape.rank = 2
    k.full_shape.dims[0], k.full_shape.dims[1] = m, n
    k.grid[0], k.grid[1], k.grid[2] = n, 1, 1
    k.local_size, k.reduce_numel, k.out_dtype = 256, m, dt
    for i in range(leaves):
        k.leaf_dtypes[i] = dt
    return k


def _main(k):
    return _lib.kernel_source(k)[0].split('extern "C" __global__')[1]


def test_routes():
    for m, n in [(4096, 4096), (1031, 1501), (100000, 33)]:
        k = column_sum(m, n)
        if not _lib.window_analyze(k):
            assert "csum_<" in _main(k) or n < 32 or m >= 8192 and n <= 256, (m, n)
            assert _lib.compile_check(k) > 0
    assert "csum_<16u, 64u>" in _main(column_sum(4096, 4096)) and "csum_<8u, 128u>" in _main(column_sum(4096, 4096, F16))
    assert "csum_<" not in _main(column_sum(256, 120))        # small: a workgroup per output
    # row sums keep their workgroup per output
    k = column_sum(2048, 2048)
    for i in range(k.n_ops):                                   # swap the strides of r and g
        o = k.ops[i]
        if o.type == abi.KOP_IDX and o.imm.u == 2048:
            o.imm.u = 1
        elif o.type == abi.KOP_IDX and o.imm.u == 1:
            o.type, o.arg[0], o.arg[1], o.imm.u = abi.KOP_IDX, o.arg[1], o.arg[0], 2048
    assert "csum_<" not in _main(k)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [F32, F16], ids=["f32", "f16"])
@pytest.mark.parametrize("kind", ["plain", "product", "factor"])
@pytest.mark.parametrize("m,n", [(1031, 1501), (4096, 512), (257, 4099), (260, 4112), (4096, 333), (64, 16400), (513, 2049)])
def test_column_sums(m, n, kind, dt):
    k = column_sum(m, n, dt, kind)
    assert "csum_<" in _main(k)
    f = np.float16 if dt == F16 else np.float32
    rng = np.random.default_rng(m + n)
    xs = [rng.uniform(-1, 1, (m, n)).astype(f)]
    if kind != "plain":
        xs.append(rng.uniform(-1, 1, (m, n) if kind == "product" else n).astype(f))
    L = _lib.lib()
    L.thvm_hip_shutdown()
    assert L.thvm_hip_init() == 0
    ids = []
    for x in xs + [np.full(n, np.nan, f)]:
        i = L.thvm_hip_buf_alloc(x.nbytes)
        L.thvm_hip_buf_write(i, x.ctypes.data_as(C.c_void_p), x.nbytes)
        ids.append(i)
    L.thvm_hip_dispatch_uop_kernel(ids[-1], (C.c_uint32 * (len(ids) - 1))(*ids[:-1]), len(ids) - 1, C.byref(k), 0)
    out = np.empty(n, f)
    L.thvm_hip_buf_read(ids[-1], out.ctypes.data_as(C.c_void_p), out.nbytes)
    assert L.thvm_hip_synchronize() == 0
    L.thvm_hip_shutdown()
    v = xs[0].astype(np.float64)
    if kind != "plain":      # the product is rounded to f32 before it is added
        v = v * xs[1].astype(np.float64)
    want, mag = v.sum(0), np.abs(v).sum(0)
    bound = (m / 64 + 32 + 1) * 2.0 ** -24 * mag + (np.abs(want) * 2.0 ** -11 + 2.0 ** -25 if dt == F16 else 0)
    worst = np.max(np.abs(out.astype(np.float64) - want) / bound)
    assert worst <= 1.0, worst


# fewer columns a workgroup where the grid is small, and grids that are no multiple of the XCDs
NARROW = [(65536, 257, F32, 4), (8200, 300, F32, 4), (8188, 132, F32, 4), (4096, 1000, F32, 4), (4096, 1030, F32, 8), (2048, 2049, F32, 16),
          (20000, 320, F16, 4), (8188, 132, F16, 2), (8191, 131, F16, 2), (1200, 1030, F16, 8)]


@pytest.mark.parametrize("m,n,dt,cols", NARROW, ids=str)
def test_narrow_grids(m, n, dt, cols):
    src = _main(column_sum(m, n, dt))
    assert "csum_<%du" % cols in src
    assert (n + cols - 1) // cols >= min(n // 4, 128)      # a workgroup for half of the compute units, or per four columns


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,dt,cols", NARROW, ids=str)
def test_narrow_column_sums(m, n, dt, cols):
    test_column_sums(m, n, "plain", dt)
