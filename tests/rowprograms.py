"""Programs over a matrix [rows, cols] as the lowering writes them, their
leaves given by strides: reductions of each row, and elementwise ones."""
from tinyhvm_amd import abi

F32, F16 = abi.DTYPE_F32, abi.DTYPE_F16
MAT, VEC, COL = "matrix", "vector", "column"


def strides(kind, cols):
    """(row stride, column stride, offset) of a leaf."""
    return {MAT: (cols, 1, 0), VEC: (1, 0, 0), COL: (0, 1, 0)}.get(kind, kind)


def program(rows, cols, leaves, body, reduce=None, dtypes=None, split=1):
    """body over a load per leaf (a kind or its strides); reduce: SUM or RMAX
    over the columns. split: the columns as two axes, the inner of this size."""
    k = abi.UOpKernel()
    n = [0]

    def op(t, a=0, b=0, imm=0, f=None):
        o = k.ops[n[0]]
        o.type, o.arg[0], o.arg[1] = t, a, b
        if f is None:
            o.imm.u = imm
        else:
            o.imm.f = f
        n[0] += 1
        return n[0] - 1

    gid = op(abi.KOP_GID)
    if reduce:
        acc = op(abi.KOP_ACC_INIT, f=0.0 if reduce == abi.UOP_SUM else -1e30)
        col = rng = op(abi.KOP_RANGE, imm=cols)
        row = op(abi.KOP_MOD, op(abi.KOP_GID), imm=rows)
    else:
        col = op(abi.KOP_GID)
        row = op(abi.KOP_MOD, op(abi.KOP_DIV, col, imm=cols), imm=rows)
    zero = op(abi.KOP_CONST_U)
    inner = op(abi.KOP_MOD, col, imm=split if split > 1 else cols)
    outer = op(abi.KOP_MOD, op(abi.KOP_DIV, col, imm=split), imm=cols // split) if split > 1 else None
    vals = []
    for i, kind in enumerate(leaves):
        rs, cs, off = strides(kind, cols)
        at = op(abi.KOP_CONST_U, imm=off)
        if rs:
            at = op(abi.KOP_IDX, at, op(abi.KOP_IDX, row, zero, rs), 1)
        if cs:
            if outer is not None:
                at = op(abi.KOP_IDX, at, op(abi.KOP_IDX, outer, zero, cs * split), 1)
            at = op(abi.KOP_IDX, at, op(abi.KOP_IDX, inner, zero, cs), 1)
        k.leaf_dtypes[i] = dtypes[i] if dtypes else F32
        vals.append(op(abi.KOP_LOAD, at, imm=i + 1))
    v = body(lambda u, a, b=0: op(abi.KOP_ALU, a, b, u), *vals)
    if reduce:
        op(abi.KOP_ACC, acc, v, reduce)
        op(abi.KOP_ENDRANGE, rng)
        v = acc
    op(abi.KOP_STORE, gid, v)
    k.n_ops, k.n_leaves, k.n_bufs = n[0], len(leaves), 1 + len(leaves)
    k.rank = k.full_shape.rank = 2
    k.full_shape.dims[0], k.full_shape.dims[1] = rows, cols
    k.grid[0], k.grid[1], k.grid[2] = rows if reduce else rows * cols, 1, 1
    k.out_dtype = F32
    k.tg[0] = k.tg[1] = k.tg[2] = 1
    if reduce and cols >= 256:
        k.local_size = k.tg[0] = 256
        k.reduce_numel = cols
    return k
