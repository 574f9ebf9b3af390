"""The work that programs have this backend do, as measurable cases.

A program hands the backend lowered kernel programs (`UOpKernel`) over buffers
it holds, through the flat C entry points (`tinyhvm_amd._lib`). The builders
below lower the layers, losses and training steps of the engine's workloads to
the same programs the engine records for them (index digits of the output
position and the reduce counter, strided views, pad masks), at any size.

Families and what each stands for in use:

  mlp      a whole training step of a small two-layer network, dispatched
           kernel by kernel: the smallest calls, where launches count.
  lenet    a whole LeNet-5 training step (forward, backward, SGD through
           ASSIGN), captured once as a HIP graph and launched per step, or
           dispatched kernel by kernel.
  linear   a linear layer: y = relu(x W + b) and the gradients of x, W and b,
           in 32-bit or 16-bit storage.
  conv     a convolution layer: padded forward, weight gradient, and input
           gradient through the flipped weights.
  bnpool   batch normalisation (train mode), relu and max-pool, forward and
           backward, with the running statistics updated in place.
  fused    an elementwise chain with a row reduction, and its gradient.
  ce       the softmax cross-entropy head on logits: loss and gradient.

Inputs are made on the GPU from the seed; `exact` computes the same in 64-bit
torch.
"""
import ctypes as C
import math

import torch

from tinyhvm_amd import _lib, abi

SUM, RMAX = abi.UOP_SUM, abi.UOP_RMAX
ADD, SUB, MUL, DIV, CMP = abi.UOP_ADD, abi.UOP_SUB, abi.UOP_MUL, abi.UOP_DIV, abi.UOP_CMP
RELU, EXP, LOG, SQRT = abi.UOP_RELU, abi.UOP_EXP, abi.UOP_LOG, abi.UOP_SQRT
F32, F16 = abi.DTYPE_F32, abi.DTYPE_F16
DEV = "cuda:0"
EPS, MOMENTUM, LR = 1e-5, 0.1, 0.01


# ---- the cases ---------------------------------------------------------

def listed():
    return [
        # a small classifier's training step, each kernel dispatched on its own
        {"name": "mlp_b64", "family": "mlp", "batch": 64, "inp": 784, "hidden": 128, "classes": 10},
        # LeNet-5 at the benchmark's batch, launched as a graph per step
        {"name": "lenet_b256_graph", "family": "lenet", "batch": 256, "graph": True},
        # LeNet-5's first fully connected layer at batch 256
        {"name": "linear_256x400x120", "family": "linear", "m": 256, "k": 400, "n": 120, "dtype": "f32"},
        # a layer whose sizes fit no tile: odd rows, columns and depth
        {"name": "linear_1031x771x1501", "family": "linear", "m": 1031, "k": 771, "n": 1501, "dtype": "f32"},
        # the benchmark's largest layer
        {"name": "linear_4096", "family": "linear", "m": 4096, "k": 4096, "n": 4096, "dtype": "f32"},
        # a layer held in 16-bit storage
        {"name": "linear_2048_f16", "family": "linear", "m": 2048, "k": 2048, "n": 2048, "dtype": "f16"},
        # the benchmark's convolution
        {"name": "conv_b64_64to64_56", "family": "conv", "batch": 64, "cin": 64, "cout": 64, "h": 56, "w": 56, "ksize": 3},
        # a deeper layer of a convolutional network: more channels, a smaller image
        {"name": "conv_b32_128to128_28", "family": "conv", "batch": 32, "cin": 128, "cout": 128, "h": 28, "w": 28, "ksize": 3},
        # an odd batch, image and channel count, with a wider kernel
        {"name": "conv_b9_24to40_29x37", "family": "conv", "batch": 9, "cin": 24, "cout": 40, "h": 29, "w": 37, "ksize": 5},
        # what stands between two convolutions of the benchmark's block
        {"name": "bnpool_b64_64x56", "family": "bnpool", "batch": 64, "ch": 64, "h": 56, "w": 56},
        # the benchmark's fused chain: bound by memory
        {"name": "fused_8192", "family": "fused", "rows": 8192, "cols": 8192},
        # a classifier head over many classes
        {"name": "ce_4096x1000", "family": "ce", "rows": 4096, "cols": 1000},
    ]


def _log(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi]: odd ones as likely as their neighbours."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    f = rng.choice(["mlp", "lenet", "linear", "linear", "linear", "conv", "conv", "conv", "bnpool", "fused", "ce"])
    if f == "mlp":
        return {"family": f, "batch": _log(rng, 8, 512), "inp": _log(rng, 16, 2048), "hidden": _log(rng, 16, 1024),
                "classes": _log(rng, 2, 100)}
    if f == "lenet":
        return {"family": f, "batch": _log(rng, 8, 512), "graph": rng.random() < 0.5}
    if f == "linear":
        d = "f16" if rng.random() < 0.25 else "f32"
        m, k, n = _log(rng, 8, 4096), _log(rng, 16, 4096), _log(rng, 10, 4096)
        if rng.random() < 0.5:   # widths are often round, batches less so
            k, n = max(16, k // 16 * 16), max(16, n // 16 * 16)
        return {"family": f, "m": m, "k": k, "n": n, "dtype": d}
    if f == "conv":
        c = {"family": f, "batch": _log(rng, 1, 128), "cin": _log(rng, 1, 256), "cout": _log(rng, 6, 256),
             "h": _log(rng, 7, 112), "w": 0, "ksize": rng.choice([1, 3, 3, 3, 5])}
        c["w"] = c["h"] if rng.random() < 0.6 else _log(rng, 7, 112)
        if rng.random() < 0.5:
            c["cin"], c["cout"] = max(8, c["cin"] // 8 * 8), max(8, c["cout"] // 8 * 8)
        # no larger than the largest listed convolution
        while _conv_flops(c) > 4.5e10 or c["batch"] * max(c["cin"], c["cout"]) * c["h"] * c["w"] > 13e6:
            if c["batch"] > 1:
                c["batch"] = max(1, c["batch"] // 2)
            else:
                c["cin"], c["cout"] = max(1, c["cin"] // 2), max(6, c["cout"] // 2)
        return c
    if f == "bnpool":
        c = {"family": f, "batch": _log(rng, 2, 128), "ch": _log(rng, 6, 256), "h": 2 * _log(rng, 5, 56), "w": 0}
        c["w"] = c["h"] if rng.random() < 0.6 else 2 * _log(rng, 5, 56)
        while c["batch"] * c["ch"] * c["h"] * c["w"] > 13e6:
            c["batch"] = max(2, c["batch"] // 2)
            c["ch"] = max(6, c["ch"] * 3 // 4)
        return c
    if f == "fused":
        return {"family": f, "rows": _log(rng, 64, 8192), "cols": _log(rng, 256, 8192)}
    return {"family": "ce", "rows": _log(rng, 32, 8192), "cols": _log(rng, 10, 4096)}


def _conv_flops(c):
    return 6.0 * c["batch"] * c["h"] * c["w"] * c["cin"] * c["cout"] * c["ksize"] ** 2


# ---- buffers -----------------------------------------------------------

_live = 0


class Buffers:
    """The backend buffers (and the graph) of one state; given back when the
    last user of them (the state, or a tensor over one of them) is gone."""

    def __init__(self):
        global _live
        self.L, self.ids, self.graph = _lib.lib(), [], None
        _live += 1
        if _live == 1:
            if self.L.thvm_hip_stream() is None:
                if self.L.thvm_hip_init() != 0:
                    raise RuntimeError("the HIP backend does not initialise on this device")
            else:
                self.L.thvm_hip_pool_reset(0)   # no buffer is in use: numbering starts again
        self.L.thvm_hip_synchronize()           # torch fills buffers that earlier work may have used

    def alloc(self, nbytes):
        i = self.L.thvm_hip_buf_alloc(max(4, nbytes))
        if not i:
            raise RuntimeError("out of memory: no backend buffer of %d bytes" % nbytes)
        self.ids.append(i)
        return i

    def __del__(self):
        global _live
        if self.graph:
            self.L.thvm_hip_graph_destroy(self.graph)
        for i in self.ids:
            self.L.thvm_hip_buf_free(i)
        _live -= 1


class _Memory:
    """A buffer's device memory as torch sees it."""

    def __init__(self, bufs, i, shape, dtype):
        self.bufs = bufs
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f2" if dtype == F16 else "<f4", "version": 3,
                                         "strides": None, "data": (bufs.L.thvm_hip_buf_device_ptr(i), False)}


class T:
    """A row-major tensor in a backend buffer."""

    def __init__(self, net, shape, dtype=F32):
        self.net, self.shape, self.dtype = net, tuple(shape), dtype
        n = 1
        for d in self.shape:
            n *= d
        self.numel, self.nbytes = n, n * abi.DTYPE_SIZE[dtype]
        self.id = net.bufs.alloc(self.nbytes)

    def torch(self):
        return torch.as_tensor(_Memory(self.net.bufs, self.id, self.shape, self.dtype), device=DEV)

    def fill(self, values):
        self.torch().copy_(values.reshape(self.shape))
        return self

    def strides(self):
        s, out = 1, []
        for d in reversed(self.shape):
            out.append(s)
            s *= d
        return out[::-1]

    def view(self, *strides, offset=0, mask=()):
        """Read at sum(coordinate * stride) + offset; 0 outside mask = [(axis, begin, end), ...]."""
        return (self, strides, offset, mask)


# ---- programs ----------------------------------------------------------

class Prog:
    """One lowered kernel over the iteration space `full`: outputs are its
    axes outside `reduce` in order, the loop counts through those inside."""

    def __init__(self, full, reduce=(), kind=SUM, out_dtype=F32):
        self.k = abi.UOpKernel()
        self.n = 0
        self.slots = []
        self.reduce = bool(reduce)
        k = self.k
        total = rn = 1
        for a, e in enumerate(full):
            if a in reduce:
                rn *= e
            else:
                total *= e
        self.gid = self.op(abi.KOP_GID)
        if self.reduce:
            self.acc = self.op(abi.KOP_ACC_INIT, imm=0.0 if kind == SUM else -1e30, f=True)
            self.loop = self.op(abi.KOP_RANGE, imm=rn)
            self.kind = kind
        self.full, self.red = full, set(reduce)
        self.cur = {False: (self.op(abi.KOP_GID), len(full)), True: (self.loop if self.reduce else 0, len(full))}
        self.coords = {}
        k.rank = k.full_shape.rank = len(full)
        for a, e in enumerate(full):
            k.full_shape.dims[a] = e
        k.grid[0], k.grid[1], k.grid[2] = total, 1, 1
        k.out_dtype = out_dtype
        if self.reduce and rn >= 256:    # the lowering's rule: a workgroup of 256 lanes per output
            k.local_size = 256
            k.tg[0], k.tg[1], k.tg[2] = 256, 1, 1
            k.reduce_numel = rn
        else:
            k.tg[0] = k.tg[1] = k.tg[2] = 1

    def op(self, t, a=0, b=0, imm=0, f=False):
        o = self.k.ops[self.n]
        o.type, o.arg[0], o.arg[1] = t, a, b
        if f:
            o.imm.f = imm
        else:
            o.imm.u = imm & 0xFFFFFFFF
        self.n += 1
        return self.n - 1

    def coord(self, axis):
        """The op of an axis's coordinate, by dividing down from the innermost axis of its kind."""
        if axis not in self.coords:
            r = axis in self.red
            cur, at = self.cur[r]
            for a in range(at - 1, axis - 1, -1):
                if (a in self.red) != r or self.full[a] == 1:
                    continue
                self.coords[a] = self.op(abi.KOP_MOD, cur, imm=self.full[a])
                if any((b in self.red) == r and self.full[b] > 1 for b in range(a)):
                    cur = self.op(abi.KOP_DIV, cur, imm=self.full[a])
                self.cur[r] = (cur, a)
        return self.coords[axis]

    def load(self, leaf):
        """Leaf: a T (read along all axes, its strides set by its shape), or T.view(...)."""
        if isinstance(leaf, T):
            assert len(leaf.shape) == len(self.full)
            leaf = leaf.view(*[s if d > 1 else 0 for s, d in zip(leaf.strides(), leaf.shape)])
        t, strides, offset, mask = leaf
        cond = None
        for a, lo, hi in mask:
            c = self.coord(a)
            for x, y in ((c, self.op(abi.KOP_CONST_U, imm=lo - 1) if lo else None), (self.op(abi.KOP_CONST_U, imm=hi), c)):
                if y is None:
                    continue
                one = self.alu(CMP, x, y)
                cond = one if cond is None else self.alu(MUL, cond, one)
        acc = self.op(abi.KOP_CONST_U, imm=offset) if offset else None
        for a, s in enumerate(strides):
            if s == 0 or self.full[a] == 1:
                continue
            c = self.coord(a)
            term = c if s == 1 else self.op(abi.KOP_IDX, c, self.op(abi.KOP_CONST_U, imm=0), s)
            acc = term if acc is None else self.op(abi.KOP_IDX, acc, term, 1)
        if acc is None:
            acc = self.op(abi.KOP_CONST_U, imm=0)
        self.slots.append(t)
        self.k.leaf_dtypes[len(self.slots) - 1] = t.dtype
        v = self.op(abi.KOP_LOAD, acc, imm=len(self.slots))
        return v if cond is None else self.op(abi.KOP_MASK, cond, v)

    def alu(self, uop, a, b=0):
        return self.op(abi.KOP_ALU, a, b, uop)

    def done(self, val):
        if self.reduce:
            self.op(abi.KOP_ACC, self.acc, val, self.kind)
            self.op(abi.KOP_ENDRANGE, self.loop)
            val = self.acc
        self.op(abi.KOP_STORE, self.gid, val)
        self.k.n_ops = self.n
        self.k.n_leaves = len(self.slots)
        self.k.n_bufs = 1 + len(self.slots)
        return self


class Net:
    """A state: tensors, and the backend calls of one pass in order."""

    def __init__(self):
        self.bufs = Buffers()
        self.L = self.bufs.L
        self.calls = []
        self.scalars = []
        self.outs = {}

    def t(self, shape, dtype=F32):
        return T(self, shape, dtype)

    def scalar(self, v):
        s = self.t((1,))
        self.scalars.append((s.id, C.c_float(v)))
        self.L.thvm_hip_buf_write(s.id, C.byref(self.scalars[-1][1]), 4)
        return s

    def kernel(self, out, full, leaves, body, reduce=(), kind=SUM):
        """out[...] = body(loads of leaves...) over `full`, reduced over the axes `reduce`."""
        p = Prog(full, reduce, kind, out.dtype)
        leaves = [v.view(*([0] * len(full))) if isinstance(v, T) and v.shape == (1,) and full != (1,) else v for v in leaves]
        vals = [p.load(v) for v in leaves]
        p.done(body(p.alu, *vals))
        ids = (C.c_uint32 * max(1, len(p.slots)))(*[s.id for s in p.slots])
        self.calls.append((self.L.thvm_hip_dispatch_uop_kernel, (out.id, ids, len(p.slots), C.byref(p.k), 0)))
        return out

    def copy(self, dst, src):
        self.calls.append((self.L.thvm_hip_buf_copy, (dst.id, src.id, dst.nbytes)))

    # -- layers, as the engine lowers them --

    def matmul(self, a, b, m, k, n, ta=False, tb=False, dtype=F32):
        """[m, n] = a b over [m, k, n]; ta: a is held [k, m], tb: b is held [n, k]."""
        va = a.view(1, m, 0) if ta else a.view(k, 1, 0)
        vb = b.view(0, 1, k) if tb else b.view(0, n, 1)
        return self.kernel(self.t((m, n), dtype), (m, k, n), [va, vb], lambda o, x, y: o(MUL, x, y), reduce=(1,))

    def bias(self, x, b, relu):
        m, n = x.shape

        def f(o, v, w):
            s = o(ADD, v, w)
            return o(RELU, s) if relu else s
        return self.kernel(self.t((m, n), x.dtype), (m, n), [x, b.view(0, 1)], f)

    def relu_mask(self, d, y):
        zero = self.scalar(0.0)
        return self.kernel(self.t(d.shape), d.shape, [d, y, zero], lambda o, g, v, z: o(MUL, g, o(CMP, v, z)))

    def colsum(self, x):
        m, n = x.shape
        return self.kernel(self.t((n,), x.dtype), (m, n), [x], lambda o, v: v, reduce=(0,))

    def conv(self, x, w, b, ci, co, h, ww, ks):
        """x held [b, ci, h+ks-1, ww+ks-1] (padded already), w [co, ci, ks, ks]."""
        hp, wp = h + ks - 1, ww + ks - 1
        full = (b, 1, co, h, ww, ci, ks, ks)
        vx = x.view(ci * hp * wp, 0, 0, wp, 1, hp * wp, wp, 1)
        vw = w.view(0, 0, ci * ks * ks, 0, 0, ks * ks, ks, 1)
        return self.kernel(self.t((b, co, h, ww)), full, [vx, vw], lambda o, p, q: o(MUL, p, q), reduce=(5, 6, 7))

    def conv_dw(self, x, dy, b, ci, co, h, ww, ks):
        hp, wp = h + ks - 1, ww + ks - 1
        full = (co, ci, ks, ks, b, h, ww)
        vx = x.view(0, hp * wp, wp, 1, ci * hp * wp, wp, 1)
        vy = dy.view(h * ww, 0, 0, 0, co * h * ww, ww, 1)
        return self.kernel(self.t((co, ci, ks, ks)), full, [vx, vy], lambda o, p, q: o(MUL, p, q), reduce=(4, 5, 6))

    def conv_dx(self, dy, w, b, ci, co, h, ww, ks, pad):
        """The gradient of the unpadded input [b, ci, h, ww]: dy padded, convolved with the flipped weights."""
        oh, ow = h + 2 * pad - ks + 1, ww + 2 * pad - ks + 1
        flip = self.t((ks * ks, ks * ks)).fill(torch.eye(ks * ks, device=DEV).flip(1))
        wf = self.matmul(w, flip, co * ci, ks * ks, ks * ks)
        one = self.scalar(1.0)
        wt = self.kernel(self.t((ci, co, ks, ks)), (ci, co, ks, ks), [wf.view(ks * ks, ci * ks * ks, ks, 1), one],
                         lambda o, v, s: o(MUL, v, s))
        dyp = self.pad(dy, b, co, oh, ow, ks - 1 - pad)
        return self.conv(dyp, wt, b, co, ci, h, ww, ks)

    def pad(self, x, b, c, h, w, p):
        if p == 0:
            return x
        full = (b, c, h + 2 * p, w + 2 * p)
        zero = self.scalar(0.0)
        v = x.view(c * h * w, h * w, w, 1, offset=-(p * w + p), mask=((2, p, p + h), (3, p, p + w)))
        return self.kernel(self.t(full), full, [v, zero], lambda o, q, z: o(ADD, q, z))

    def per_channel(self, x, b):
        """x + b per channel, relu."""
        return self.kernel(self.t(x.shape), x.shape, [x, b.view(0, 1, 0, 0)], lambda o, v, w: o(RELU, o(ADD, v, w)))

    def channel_sum(self, x, *more, body=lambda o, v: v):
        _n, c, _h, _w = x.shape
        return self.kernel(self.t((c,)), x.shape, [x, *more], body, reduce=(0, 2, 3))

    def maxpool(self, x):
        b, c, h, w = x.shape
        full = (b, c, h // 2, w // 2, 2, 2)
        v = x.view(c * h * w, h * w, 2 * w, 2, w, 1)
        return self.kernel(self.t(full[:4]), full, [v], lambda o, q: q, reduce=(4, 5), kind=RMAX)

    def maxpool_relu_back(self, dp, pooled, y):
        """dy = dp * (1 - (pooled > y)) * (y > 0): the gradient goes to every maximum of a window."""
        b, c, h, w = y.shape
        ph, pw = h // 2, w // 2
        full = (b, c, ph, 2, pw, 2)
        vp = (c * ph * pw, ph * pw, pw, 0, 1, 0)
        vy = (c * h * w, h * w, 2 * w, w, 2, 1)
        one, zero = self.scalar(1.0), self.scalar(0.0)
        return self.kernel(self.t(y.shape), full, [dp.view(*vp), one, pooled.view(*vp), y.view(*vy), y.view(*vy), zero],
                           lambda o, g, s, q, v, u, z: o(MUL, o(MUL, g, o(SUB, s, o(CMP, q, v))), o(CMP, u, z)))

    def cross_entropy(self, logits, onehot):
        """Mean cross-entropy and its gradient, as the engine composes them."""
        m, n = logits.shape
        row = lambda t: t.view(1, 0)  # noqa: E731

        def rowmax():
            return self.kernel(self.t((m,)), (m, n), [logits], lambda o, v: v, reduce=(1,), kind=RMAX)
        mx = rowmax()
        picked = self.kernel(self.t((m,)), (m, n), [onehot, logits], lambda o, p, v: o(MUL, p, v), reduce=(1,))
        se = self.kernel(self.t((m,)), (m, n), [logits, row(mx)], lambda o, v, x: o(EXP, o(SUB, v, x)), reduce=(1,))
        total = self.kernel(self.t((1,)), (m, 1), [row(mx), row(se), row(picked)],
                            lambda o, x, s, p: o(SUB, o(ADD, x, o(LOG, s)), p), reduce=(0,))
        loss = self.kernel(self.t((1,)), (1,), [total, self.scalar(1.0 / m)], lambda o, t, s: o(MUL, t, s))
        mx2 = rowmax()
        e = self.kernel(self.t((m, n)), (m, n), [logits, row(mx2)], lambda o, v, x: o(EXP, o(SUB, v, x)))
        s = self.kernel(self.t((m,)), (m, n), [e], lambda o, v: v, reduce=(1,))
        p = self.kernel(self.t((m, n)), (m, n), [e, row(s)], lambda o, v, z: o(DIV, v, z))
        d = self.kernel(self.t((m, n)), (m, n), [p, onehot, self.scalar(1.0 / m)],
                        lambda o, v, t, z: o(MUL, o(SUB, v, t), z))
        return loss, d

    def sgd(self, param, grad):
        """param <- param - lr * grad, assigned in place."""
        lr = self.scalar(LR)
        new = self.kernel(self.t(param.shape), param.shape, [param, grad, lr], lambda o, p, g, r: o(SUB, p, o(MUL, g, r)))
        self.copy(param, new)

    # -- a pass --

    def dispatch(self):
        for fn, args in self.calls:
            fn(*args)

    def capture(self):
        """The pass as a HIP graph (a step dispatched once before, so that its kernels are built)."""
        self.L.thvm_hip_synchronize()
        if self.L.thvm_hip_graph_begin() != 0:
            raise RuntimeError("no graph capture")
        for i, v in self.scalars:     # a captured step writes its scalars, as the engine's steps do
            self.L.thvm_hip_buf_write(i, C.byref(v), 4)
        self.dispatch()
        self.bufs.graph = self.L.thvm_hip_graph_end()
        if not self.bufs.graph:
            raise RuntimeError("the step was not captured")

    def give(self, **tensors):
        self.outs = {name: t.torch() for name, t in tensors.items()}
        return self


# ---- inputs ------------------------------------------------------------

class Inputs:
    """Tensors drawn one after the other from a seed, the same for prepare and exact."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.g, device=DEV)

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.g, device=DEV) * (hi - lo) + lo

    def kaiming(self, fan_in, *shape):
        a = math.sqrt(6.0 / fan_in)
        return self.uniform(-a, a, *shape)

    def onehot(self, m, n):
        c = torch.randint(0, n, (m,), generator=self.g, device=DEV)
        return torch.nn.functional.one_hot(c, n).float()


def _inputs(case, seed):
    r, f = Inputs(seed), case["family"]
    if f == "mlp":
        b, i, h, c = case["batch"], case["inp"], case["hidden"], case["classes"]
        return {"x": r.normal(b, i), "w1": r.kaiming(i, i, h), "b1": r.uniform(-0.1, 0.1, h), "w2": r.kaiming(h, h, c),
                "b2": r.uniform(-0.1, 0.1, c), "onehot": r.onehot(b, c)}
    if f == "lenet":
        b, out = case["batch"], {}
        out["x"], out["onehot"] = r.uniform(0, 1, b, 1, 28, 28), r.onehot(b, 10)
        for name, shape, fan in _LENET:
            out[name] = r.kaiming(fan, *shape) if len(shape) > 1 else r.uniform(-0.05, 0.05, *shape)
        return out
    if f == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        out = {"x": r.uniform(-1, 1, m, k), "w": r.kaiming(k, k, n), "b": r.uniform(-1, 1, n), "g": r.normal(m, n)}
        return {q: v.half() if case["dtype"] == "f16" else v for q, v in out.items()}
    if f == "conv":
        b, ci, co, h, w, ks = (case[q] for q in ("batch", "cin", "cout", "h", "w", "ksize"))
        return {"x": r.normal(b, ci, h, w), "w": r.kaiming(ci * ks * ks, co, ci, ks, ks), "g": r.normal(b, co, h, w)}
    if f == "bnpool":
        b, c, h, w = (case[q] for q in ("batch", "ch", "h", "w"))
        return {"y": r.normal(b, c, h, w), "gamma": r.uniform(0.5, 1.5, c), "beta": r.uniform(-0.5, 0.5, c),
                "mean": r.uniform(-0.5, 0.5, c), "var": r.uniform(0.5, 1.5, c), "g": r.normal(b, c, h // 2, w // 2)}
    if f == "fused":
        s = (case["rows"], case["cols"])
        return {"a": r.normal(*s), "b": r.normal(*s), "c": r.normal(*s)}
    s = (case["rows"], case["cols"])
    return {"logits": r.normal(*s) * 3, "onehot": r.onehot(*s)}


_LENET = [("w1", (6, 1, 5, 5), 25), ("b1", (6,), 0), ("w2", (16, 6, 5, 5), 150), ("b2", (16,), 0),
          ("f1", (400, 120), 400), ("c1", (120,), 0), ("f2", (120, 84), 120), ("c2", (84,), 0),
          ("f3", (84, 10), 84), ("c3", (10,), 0)]


# ---- states and passes ---------------------------------------------------

def prepare(case, seed):
    net = Net()
    vals = _inputs(case, seed)
    t = {k: net.t(v.shape, F16 if v.dtype == torch.float16 else F32).fill(v) for k, v in vals.items()}
    _BUILD[case["family"]](net, case, t)
    torch.cuda.synchronize()     # the inputs are in place before the backend's stream reads them
    if case.get("graph"):
        net.dispatch()           # builds the kernels
        net.L.thvm_hip_synchronize()
        for k, v in vals.items():
            t[k].fill(v)
        torch.cuda.synchronize()
        net.capture()
    return net


def run(net):
    if net.bufs.graph:
        net.L.thvm_hip_graph_launch(net.bufs.graph)
    else:
        net.dispatch()
        net.L.thvm_hip_flush()
    return net.outs


def _mlp(net, case, t):
    b, i, h, c = case["batch"], case["inp"], case["hidden"], case["classes"]
    hid = net.bias(net.matmul(t["x"], t["w1"], b, i, h), t["b1"], True)
    logits = net.bias(net.matmul(hid, t["w2"], b, h, c), t["b2"], False)
    loss, d2 = net.cross_entropy(logits, t["onehot"])
    dw2 = net.matmul(hid, d2, h, b, c, ta=True)
    db2 = net.colsum(d2)
    d1 = net.relu_mask(net.matmul(d2, t["w2"], b, c, h, tb=True), hid)
    dw1 = net.matmul(t["x"], d1, i, b, h, ta=True)
    db1 = net.colsum(d1)
    net.give(loss=loss, logits=logits, dw1=dw1, db1=db1, dw2=dw2, db2=db2)


def _lenet(net, case, t):
    b = case["batch"]
    xp = net.pad(t["x"], b, 1, 28, 28, 2)
    a1 = net.per_channel(net.conv(xp, t["w1"], b, 1, 6, 28, 28, 5), t["b1"])
    p1 = net.maxpool(a1)
    a2 = net.per_channel(net.conv(p1, t["w2"], b, 6, 16, 10, 10, 5), t["b2"])
    p2 = net.maxpool(a2)
    h1 = net.bias(net.matmul(p2, t["f1"], b, 400, 120), t["c1"], True)
    h2 = net.bias(net.matmul(h1, t["f2"], b, 120, 84), t["c2"], True)
    logits = net.bias(net.matmul(h2, t["f3"], b, 84, 10), t["c3"], False)
    loss, d3 = net.cross_entropy(logits, t["onehot"])
    grads = {"f3": net.matmul(h2, d3, 84, b, 10, ta=True), "c3": net.colsum(d3)}
    d2 = net.relu_mask(net.matmul(d3, t["f3"], b, 10, 84, tb=True), h2)
    grads["f2"], grads["c2"] = net.matmul(h1, d2, 120, b, 84, ta=True), net.colsum(d2)
    d1 = net.relu_mask(net.matmul(d2, t["f2"], b, 84, 120, tb=True), h1)
    grads["f1"], grads["c1"] = net.matmul(p2, d1, 400, b, 120, ta=True), net.colsum(d1)
    dp2 = net.matmul(d1, t["f1"], b, 120, 400, tb=True)
    da2 = net.maxpool_relu_back(dp2, p2, a2)
    grads["w2"], grads["b2"] = net.conv_dw(p1, da2, b, 6, 16, 10, 10, 5), net.channel_sum(da2)
    da1 = net.maxpool_relu_back(net.conv_dx(da2, t["w2"], b, 6, 16, 14, 14, 5, 0), p1, a1)
    grads["w1"], grads["b1"] = net.conv_dw(xp, da1, b, 1, 6, 28, 28, 5), net.channel_sum(da1)
    for name, _shape, _fan in _LENET:
        net.sgd(t[name], grads[name])
    net.give(loss=loss, logits=logits, **{name: t[name] for name, _s, _f in _LENET})


def _linear(net, case, t):
    m, k, n = case["m"], case["k"], case["n"]
    dt = F16 if case["dtype"] == "f16" else F32
    y = net.bias(net.matmul(t["x"], t["w"], m, k, n, dtype=dt), t["b"], True)
    dx = net.matmul(t["g"], t["w"], m, n, k, tb=True, dtype=dt)
    dw = net.matmul(t["x"], t["g"], k, m, n, ta=True, dtype=dt)
    db = net.colsum(t["g"])
    net.give(y=y, dx=dx, dw=dw, db=db)


def _conv(net, case, t):
    b, ci, co, h, w, ks = (case[q] for q in ("batch", "cin", "cout", "h", "w", "ksize"))
    p = ks // 2
    xp = net.pad(t["x"], b, ci, h, w, p)
    y = net.conv(xp, t["w"], b, ci, co, h, w, ks)
    dw = net.conv_dw(xp, t["g"], b, ci, co, h, w, ks)
    dx = net.conv_dx(t["g"], t["w"], b, ci, co, h, w, ks, p)
    net.give(y=y, dw=dw, dx=dx)


def _bnpool(net, case, t):
    b, c, h, w = (case[q] for q in ("batch", "ch", "h", "w"))
    y, n = t["y"], b * h * w
    ch = lambda v: v.view(0, 1, 0, 0)  # noqa: E731
    vec = lambda leaves, body: net.kernel(net.t((c,)), (1, c, 1, 1), [ch(v) if v.shape == (c,) else v for v in leaves], body)  # noqa: E731
    mean = vec([net.channel_sum(y), net.scalar(1.0 / n)], lambda o, s, r: o(MUL, s, r))
    cen = net.kernel(net.t(y.shape), y.shape, [y, ch(mean)], lambda o, v, m: o(SUB, v, m))
    var = vec([net.channel_sum(cen, body=lambda o, v: o(MUL, v, v)), net.scalar(1.0 / n)], lambda o, s, r: o(MUL, s, r))
    inv = vec([net.scalar(1.0), var, net.scalar(EPS)], lambda o, one, v, e: o(DIV, one, o(SQRT, o(ADD, v, e))))
    xhat = net.kernel(net.t(y.shape), y.shape, [cen, ch(inv)], lambda o, v, s: o(MUL, v, s))
    z = net.kernel(net.t(y.shape), y.shape, [xhat, ch(t["gamma"]), ch(t["beta"])], lambda o, v, g, s: o(ADD, o(MUL, v, g), s))
    for stat, new, f in ((t["mean"], mean, 1.0), (t["var"], var, n / (n - 1.0))):
        upd = net.kernel(net.t((c,)), (c,), [stat, net.scalar(1.0 - MOMENTUM), new, net.scalar(MOMENTUM * f)],
                         lambda o, s, p, v, q: o(ADD, o(MUL, s, p), o(MUL, v, q)))
        net.copy(stat, upd)
    a = net.kernel(net.t(y.shape), y.shape, [z], lambda o, v: o(RELU, v))
    pooled = net.maxpool(a)
    dz = net.maxpool_relu_back(t["g"], pooled, a)
    dbeta = net.channel_sum(dz)
    dgamma = net.channel_sum(dz, xhat, body=lambda o, v, u: o(MUL, v, u))
    dxh = net.kernel(net.t(y.shape), y.shape, [dz, ch(t["gamma"])], lambda o, v, g: o(MUL, v, g))
    s1 = net.channel_sum(dxh)
    s2 = net.channel_sum(dxh, xhat, body=lambda o, v, u: o(MUL, v, u))
    scale = vec([inv, net.scalar(1.0 / n)], lambda o, s, r: o(MUL, s, r))
    dy = net.kernel(net.t(y.shape), y.shape, [dxh, net.scalar(float(n)), ch(s1), xhat, ch(s2), ch(scale)],
                    lambda o, v, k, p, u, q, s: o(MUL, o(SUB, o(SUB, o(MUL, v, k), p), o(MUL, u, q)), s))
    net.give(pooled=pooled, mean=t["mean"], var=t["var"], dgamma=dgamma, dbeta=dbeta, dy=dy)


def _fused(net, case, t):
    s = (case["rows"], case["cols"])
    chain = lambda o, a, b, c: o(ADD, o(MUL, a, b), c)  # noqa: E731
    y = net.kernel(net.t((s[0],)), s, [t["a"], t["b"], t["c"]], lambda o, a, b, c: o(RELU, chain(o, a, b, c)), reduce=(1,))
    da = net.kernel(net.t(s), s, [t["a"], t["b"], t["c"], net.scalar(0.0)],
                    lambda o, a, b, c, z: o(MUL, o(CMP, chain(o, a, b, c), z), b))
    net.give(y=y, da=da)


def _ce(net, case, t):
    loss, d = net.cross_entropy(t["logits"], t["onehot"])
    net.give(loss=loss, dlogits=d)


_BUILD = {"mlp": _mlp, "lenet": _lenet, "linear": _linear, "conv": _conv, "bnpool": _bnpool, "fused": _fused, "ce": _ce}


# ---- what a pass cannot do without ----------------------------------------

def work(case):
    f = case["family"]
    if f == "mlp":
        b, i, h, c = case["batch"], case["inp"], case["hidden"], case["classes"]
        return {"bytes": 4.0 * (b * i + 2 * (i * h + h * c + h + c) + 2 * b * c + 1), "flops": 2.0 * b * (2 * i * h + 3 * h * c)}
    if f == "lenet":
        b, params = case["batch"], 61706
        conv = 784 * 6 * 25 * 2 + 100 * 16 * 150 * 3
        fc = 3 * (400 * 120 + 120 * 84 + 84 * 10)
        return {"bytes": 4.0 * (b * 784 + 2 * params + 2 * b * 10 + 1), "flops": 2.0 * b * (conv + fc)}
    if f == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        e = 2.0 if case["dtype"] == "f16" else 4.0
        return {"bytes": e * (2 * m * k + 2 * k * n + 2 * n + 2 * m * n), "flops": 6.0 * m * k * n}
    if f == "conv":
        b, ci, co, h, w, ks = (case[q] for q in ("batch", "cin", "cout", "h", "w", "ksize"))
        return {"bytes": 4.0 * (2 * b * ci * h * w + 2 * ci * co * ks * ks + 2 * b * co * h * w), "flops": _conv_flops(case)}
    if f == "bnpool":
        b, c, h, w = (case[q] for q in ("batch", "ch", "h", "w"))
        n = b * c * h * w
        return {"bytes": 4.0 * (2.5 * n + 8 * c), "flops": 26.0 * n}
    n = case["rows"] * case["cols"]
    if f == "fused":
        return {"bytes": 4.0 * (4 * n + case["rows"]), "flops": 8.0 * n}
    return {"bytes": 4.0 * (3 * n + 1), "flops": 10.0 * n}


def tolerance(case):
    f = case["family"]
    if f == "linear" and case["dtype"] == "f16":
        # results rounded to 11 bits: a sum in another order moves some by a unit in the last place
        return {"rel": 1e-3, "max": 2e-2}
    if f == "bnpool":
        # a rounding apart, a few of the millions of relu signs and window maxima fall the other way
        return {"rel": 4e-3, "max": 0.9}
    # 32-bit sums in another order
    return {"rel": 1e-5}


# ---- the same in 64 bits ----------------------------------------------------

def _conv64(x, w, p):
    """2-d convolution by taps: one matrix product per tap."""
    co, ci, ks, _ = w.shape
    b, _c, h, ww = x.shape
    x = torch.nn.functional.pad(x, (p, p, p, p))
    oh, ow = h + 2 * p - ks + 1, ww + 2 * p - ks + 1
    xt = x.permute(1, 0, 2, 3)
    y = 0
    for i in range(ks):
        for j in range(ks):
            y = y + w[:, :, i, j] @ xt[:, :, i:i + oh, j:j + ow].reshape(ci, -1)
    return y.reshape(co, b, oh, ow).permute(1, 0, 2, 3)


def exact(case, seed):
    f = case["family"]
    v = {k: t.double() for k, t in _inputs(case, seed).items()}
    nn = torch.nn.functional
    if f == "linear":
        return {"y": (v["x"] @ v["w"] + v["b"]).relu(), "dx": v["g"] @ v["w"].t(), "dw": v["x"].t() @ v["g"], "db": v["g"].sum(0)}
    if f == "conv":
        x, w = v["x"].requires_grad_(), v["w"].requires_grad_()
        y = _conv64(x, w, case["ksize"] // 2)
        dx, dw = torch.autograd.grad(y, (x, w), v["g"])
        return {"y": y.detach().contiguous(), "dw": dw.contiguous(), "dx": dx.contiguous()}
    if f == "fused":
        s = v["a"] * v["b"] + v["c"]
        return {"y": s.relu().sum(1), "da": (s > 0) * v["b"]}
    if f == "ce":
        x = v["logits"].requires_grad_()
        loss = -(v["onehot"] * nn.log_softmax(x, 1)).sum() / case["rows"]
        return {"loss": loss.detach().reshape(1), "dlogits": torch.autograd.grad(loss, x)[0]}
    if f == "mlp":
        ps = [v[q].requires_grad_() for q in ("w1", "b1", "w2", "b2")]
        logits = (v["x"] @ ps[0] + ps[1]).relu() @ ps[2] + ps[3]
        loss = -(v["onehot"] * nn.log_softmax(logits, 1)).sum() / case["batch"]
        g = torch.autograd.grad(loss, ps)
        return {"loss": loss.detach().reshape(1), "logits": logits.detach(), "dw1": g[0], "db1": g[1], "dw2": g[2], "db2": g[3]}
    if f == "lenet":
        ps = {name: v[name].requires_grad_() for name, _s, _f in _LENET}
        a = nn.max_pool2d((_conv64(v["x"], ps["w1"], 2) + ps["b1"].view(1, -1, 1, 1)).relu(), 2)
        a = nn.max_pool2d((_conv64(a, ps["w2"], 0) + ps["b2"].view(1, -1, 1, 1)).relu(), 2)
        h = (a.reshape(case["batch"], 400) @ ps["f1"] + ps["c1"]).relu()
        h = (h @ ps["f2"] + ps["c2"]).relu()
        logits = h @ ps["f3"] + ps["c3"]
        loss = -(v["onehot"] * nn.log_softmax(logits, 1)).sum() / case["batch"]
        g = torch.autograd.grad(loss, list(ps.values()))
        out = {name: (p - LR * d).detach() for (name, p), d in zip(ps.items(), g)}
        return {"loss": loss.detach().reshape(1), "logits": logits.detach(), **out}
    # bnpool: what follows the relu's signs and the windows' maxima backwards
    # has no 64-bit value to hold a 32-bit pass to
    n = case["batch"] * case["h"] * case["w"]
    mean = v["y"].mean((0, 2, 3))
    var = (v["y"] - mean.view(1, -1, 1, 1)).square().mean((0, 2, 3))
    z = (v["y"] - mean.view(1, -1, 1, 1)) / (var + EPS).sqrt().view(1, -1, 1, 1)
    z = z * v["gamma"].view(1, -1, 1, 1) + v["beta"].view(1, -1, 1, 1)
    return {"pooled": nn.max_pool2d(z.relu(), 2), "mean": v["mean"] * (1 - MOMENTUM) + mean * MOMENTUM,
            "var": v["var"] * (1 - MOMENTUM) + var * (MOMENTUM * n / (n - 1.0)), "dgamma": None, "dbeta": None, "dy": None}
