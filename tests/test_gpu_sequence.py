"""A held launch whose output an earlier-dispatched step of the same held
sequence already reads stays where it is: a consumer that could fuse after
it becomes a later step of its own. The second layer of a small perceptron
with two classes, its row maxima and the exponentials of the differences.

Bound: the contraction rounds k products and k additions, the bias adds one,
each within 2^-24 of the magnitudes' sum; a difference of logits doubles
that, and exp turns it into a relative error (2^-21 is left for exp's own)."""
import ctypes as C

import numpy as np
import pytest

from tinyhvm_amd import _lib, abi
from tests.contractions import matmul


def program(n_out, leaves, body, loop=0):
    """One load per (row stride, column stride) of `leaves`, combined by
    `body`; over (n_out, loop) if loop, else elementwise over rows of 2."""
    k = abi.UOpKernel()
    c = [0]

    def op(t, a=0, b=0, imm=0, f=None):
        o = k.ops[c[0]]
        o.type, o.arg[0], o.arg[1] = t, a, b
        if f is None:
            o.imm.u = imm
        else:
            o.imm.f = f
        c[0] += 1
        return c[0] - 1

    gid = op(abi.KOP_GID)
    if loop:
        acc, rng = op(abi.KOP_ACC_INIT, f=-1e30), op(abi.KOP_RANGE, imm=loop)
        row, col = op(abi.KOP_GID), op(abi.KOP_MOD, rng, imm=loop)
        row = op(abi.KOP_MOD, row, imm=n_out)
    else:
        cur = op(abi.KOP_GID)
        col = op(abi.KOP_MOD, cur, imm=2)
        row = op(abi.KOP_MOD, op(abi.KOP_DIV, cur, imm=2), imm=n_out // 2)
    vals = []
    for i, (rs, cs) in enumerate(leaves):
        at = op(abi.KOP_CONST_U)
        if rs:
            at = op(abi.KOP_IDX, at, op(abi.KOP_IDX, row, op(abi.KOP_CONST_U), rs), 1)
        if cs:
            at = op(abi.KOP_IDX, at, op(abi.KOP_IDX, col, op(abi.KOP_CONST_U), cs), 1)
        vals.append(op(abi.KOP_LOAD, at, imm=i + 1))
    v = body(op, *vals)
    if loop:
        op(abi.KOP_ACC, acc, v, abi.UOP_RMAX)
        op(abi.KOP_ENDRANGE, rng)
        v = acc
    op(abi.KOP_STORE, gid, v)
    k.n_ops, k.n_leaves, k.n_bufs = c[0], len(leaves), 1 + len(leaves)
    k.rank = k.full_shape.rank = 2
    k.full_shape.dims[0], k.full_shape.dims[1] = (n_out, loop) if loop else (n_out // 2, 2)
    k.grid[0], k.grid[1], k.grid[2] = n_out, 1, 1
    return k


@pytest.mark.gpu
@pytest.mark.parametrize("m,k", [(56, 29), (8, 33), (64, 30)])
def test_consumer_after_a_step_that_reads_the_same_output(m, k, monkeypatch):
    monkeypatch.delenv("THVM_HIP_DENSE_FORCE", raising=False)    # below the matrix tiles' least work: a generated loop

    def alu(u):
        return lambda op, a, b: op(abi.KOP_ALU, a, b, u)

    def exp_diff(op, v, x):
        return op(abi.KOP_ALU, op(abi.KOP_ALU, v, x, abi.UOP_SUB), 0, abi.UOP_EXP)

    rng = np.random.default_rng(m)
    x, w, b = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((m, k), (k, 2), (2,)))
    L = _lib.lib()
    L.thvm_hip_shutdown()
    assert L.thvm_hip_init() == 0

    def buf(v):
        i = L.thvm_hip_buf_alloc(v.nbytes)
        L.thvm_hip_buf_write(i, v.ctypes.data_as(C.c_void_p), v.nbytes)
        return i

    ix, iw, ib = buf(x), buf(w), buf(b)
    iz, iy, ie = (buf(np.full((m, 2), -7, np.float32)) for _ in range(3))
    im = buf(np.full(m, -7, np.float32))
    assert L.thvm_hip_synchronize() == 0
    for out, leaves, p in [(iz, (ix, iw), matmul("nn", m, k, 2)[0]),
                           (iy, (iz, ib), program(2 * m, [(2, 1), (0, 1)], alu(abi.UOP_ADD))),
                           (im, (iy,), program(m, [(2, 1)], lambda op, v: v, loop=2)),
                           (ie, (iy, im), program(2 * m, [(2, 1), (1, 0)], exp_diff))]:
        L.thvm_hip_dispatch_uop_kernel(out, (C.c_uint32 * len(leaves))(*leaves), len(leaves), C.byref(p), 0)
    mx, e = np.empty(m, np.float32), np.empty((m, 2), np.float32)
    for i, v in ((im, mx), (ie, e)):
        L.thvm_hip_buf_read(i, v.ctypes.data_as(C.c_void_p), v.nbytes)
    assert L.thvm_hip_synchronize() == 0
    L.thvm_hip_shutdown()
    y = x.astype(np.float64) @ w + b
    bound = (2 * k + 1) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w) + np.abs(b))
    worst = np.max(np.abs(mx - y.max(1)) / bound.max(1))
    assert worst <= 1.0, worst
    want = np.exp(y - y.max(1, keepdims=True))
    worst = np.max(np.abs(e - want) / (want * (2.2 * bound.max(1, keepdims=True) + 2.0 ** -21)))
    assert worst <= 1.0, worst
