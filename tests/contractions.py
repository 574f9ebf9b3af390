"""Lowered contraction programs of any size, for tests: matmuls with either
operand held transposed and stride-1 convolutions (forward and weight
gradient), with the index forms the engine lowers them to, and the same sums
in numpy float64 with the sum of the products' magnitudes."""
import numpy as np

from tinyhvm_amd import abi


def program(full, reduce, views, dtypes, out_dtype=abi.DTYPE_F32):
    """out[...] = sum over `reduce` of the product of two loads, each read at
    sum(coordinate * stride) over the axes of `full`."""
    k = abi.UOpKernel()
    n = [0]

    def op(t, a=0, b=0, imm=0):
        o = k.ops[n[0]]
        o.type, o.arg[0], o.arg[1], o.imm.u = t, a, b, imm
        n[0] += 1
        return n[0] - 1

    total = rn = 1
    for a, e in enumerate(full):
        if a in reduce:
            rn *= e
        else:
            total *= e
    gid = op(abi.KOP_GID)
    acc = op(abi.KOP_ACC_INIT)
    loop = op(abi.KOP_RANGE, imm=rn)
    coord = {}
    for inside in (False, True):
        cur = loop if inside else op(abi.KOP_GID)
        axes = [a for a in range(len(full)) if (a in reduce) == inside and full[a] > 1]
        for i, a in enumerate(reversed(axes)):
            coord[a] = op(abi.KOP_MOD, cur, imm=full[a])
            if i + 1 < len(axes):
                cur = op(abi.KOP_DIV, cur, imm=full[a])
    vals = []
    for i, strides in enumerate(views):
        at = op(abi.KOP_CONST_U)
        for a, s in enumerate(strides):
            if s and a in coord:
                at = op(abi.KOP_IDX, at, op(abi.KOP_IDX, coord[a], op(abi.KOP_CONST_U), s), 1)
        vals.append(op(abi.KOP_LOAD, at, imm=i + 1))
        k.leaf_dtypes[i] = dtypes[i]
    op(abi.KOP_ACC, acc, op(abi.KOP_ALU, vals[0], vals[1], abi.UOP_MUL), abi.UOP_SUM)
    op(abi.KOP_ENDRANGE, loop)
    op(abi.KOP_STORE, gid, acc)
    k.n_ops, k.n_leaves, k.n_bufs = n[0], 2, 3
    k.rank = k.full_shape.rank = len(full)
    for a, e in enumerate(full):
        k.full_shape.dims[a] = e
    k.grid[0], k.grid[1], k.grid[2] = total, 1, 1
    k.out_dtype = out_dtype
    if rn >= 256:
        k.local_size, k.reduce_numel = 256, rn
    return k


def matmul(kind, m, k, n, dt=abi.DTYPE_F32):
    """kind: nn, nt (the right operand held [n, k]) or tn (the left one held
    [k, m]). Returns the program and both operands' shapes."""
    va = (1, m, 0) if kind == "tn" else (k, 1, 0)
    vb = (0, 1, k) if kind == "nt" else (0, n, 1)
    return (program((m, k, n), {1}, [va, vb], [dt, dt], dt), (k, m) if kind == "tn" else (m, k),
            (n, k) if kind == "nt" else (k, n))


def conv(kind, b, ci, co, h, w, ks):
    """A stride-1 convolution over an input held padded: cf (forward, the
    second operand the weights) or dw (the weights' gradient, the second
    operand the output's)."""
    hp, wp = h + ks - 1, w + ks - 1
    xs = (b, ci, hp, wp)
    if kind == "cf":
        full, red = (b, 1, co, h, w, ci, ks, ks), {5, 6, 7}
        va = (ci * hp * wp, 0, 0, wp, 1, hp * wp, wp, 1)
        vb = (0, 0, ci * ks * ks, 0, 0, ks * ks, ks, 1)
        return program(full, red, [va, vb], [0, 0]), xs, (co, ci, ks, ks)
    full, red = (co, ci, ks, ks, b, h, w), {4, 5, 6}
    va = (0, hp * wp, wp, 1, ci * hp * wp, wp, 1)
    vb = (h * w, 0, 0, 0, co * h * w, w, 1)
    return program(full, red, [va, vb], [0, 0]), xs, (b, co, h, w)


def reference(kind, a, b):
    """The result in float64 and the sum of the magnitudes of its products."""
    a, b = a.astype(np.float64), b.astype(np.float64)
    out = []
    for x, y in ((a, b), (np.abs(a), np.abs(b))):
        if kind in ("nn", "nt", "tn"):
            out.append((x.T if kind == "tn" else x) @ (y.T if kind == "nt" else y))
            continue
        ks = (x.shape[2] - y.shape[2] + 1) if kind == "dw" else y.shape[2]
        h, w = x.shape[2] - ks + 1, x.shape[3] - ks + 1
        win = np.lib.stride_tricks.sliding_window_view(x, (h, w), axis=(2, 3))    # [b, ci, ky, kx, h, w]
        if kind == "cf":
            out.append(np.einsum("bikjhw,oikj->bohw", win, y, optimize=True))
        else:
            out.append(np.einsum("bikjhw,bohw->oikj", win, y, optimize=True))
    return out
