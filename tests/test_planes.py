"""Plane tiles (the matrix-core kernels that stage operands as 16-bit
planes), without a device: the index functions of the generated source,
compiled for the host, against the contraction's own offsets.

- The groups of the reduce index visit every (left, right) pair of k offsets
  exactly once (elements a group shares with the one before it count as 0).
- No load of a group leaves its buffer, also of elements that count as 0.
- Every such kernel compiles for gfx950.
- A contraction the direct kernel is as fast for keeps it, and one whose
  operands differ in type, or have no run of a group's length along k, takes
  no plane tile."""
import ctypes as C
import re
import subprocess
from collections import Counter

import pytest

from tests import contractions as ct
from tinyhvm_amd import _lib, abi

F32, F16 = abi.DTYPE_F32, abi.DTYPE_F16
FN = re.compile(r"^__device__ __forceinline__ u32 (gid_[mn]|row[b]?_[pq]|koff_[pq]|kg_[pq]o?|kz|vpos_|tapq_)\(u32 \w\) \{.*?^\}|"
                r"^__device__ __forceinline__ u32 (?:row_[pq]|kg_q)\(u32 \w\) \{.*?\}$", re.M | re.S)
CST = re.compile(r"constexpr u32 KG = (\d+)u, NGRP = (\d+)u, ICP = (\d+)u, ICQ = (\d+)u;")

CASES = [ct.matmul(*a) for a in [
    ("nn", 300, 771, 500), ("nt", 600, 1501, 260), ("tn", 601, 1030, 517), ("nn", 64, 4099, 64), ("nt", 640, 512, 640),
    ("nn", 512, 512, 512, F16), ("nt", 300, 1502, 262, F16), ("nt", 300, 1501, 262, F16), ("tn", 302, 1030, 258, F16),
    ("tn", 301, 1030, 259, F16)]] + [ct.conv(*a) for a in [
        ("cf", 32, 32, 128, 28, 28, 7), ("cf", 9, 24, 40, 29, 37, 7), ("dw", 9, 24, 40, 29, 37, 5),
        ("dw", 16, 64, 80, 14, 14, 3), ("cf", 7, 33, 70, 39, 43, 6), ("dw", 7, 33, 70, 39, 43, 3), ("cf", 16, 64, 96, 28, 28, 1), ("cf", 4, 6, 130, 60, 61, 5)]]


def _host(src, tmp_path):
    """The source's index functions as a host library."""
    text = "typedef unsigned u32;\n#define constexpr const\n" + "\n".join(
        m.group(0).replace("__device__ __forceinline__", "") for m in FN.finditer(src))
    c, so = tmp_path / "f.c", tmp_path / "f.so"
    c.write_text(text)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", str(c), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))

    def f(name):
        fn = getattr(lib, name)
        fn.restype, fn.argtypes = C.c_uint32, [C.c_uint32]
        return fn
    return f


@pytest.mark.parametrize("case", CASES, ids=lambda c: "%s-%s" % ("x".join(map(str, c[1])), "x".join(map(str, c[2]))))
def test_groups_cover_the_reduce_index_once(case, tmp_path):
    k, sa, sb = case
    m, n, kk, _splits = _lib.dense_analyze(k)
    src = _lib.dense_source(k)
    cst = CST.search(src)
    assert cst, "no plane tile"
    g, ng, icp, icq = map(int, cst.groups())
    f = _host(src, tmp_path)
    packed = "kg_qo(" in src
    kg_q, icq_own = f("kg_qo" if packed else "kg_q"), icq
    if packed:
        icq_own = int(re.search(r"kg_qo\(g\) \+ j \* (\d+)u", src).group(1))
    koff_p, koff_q, kg_p, kz = f("koff_p"), f("koff_q"), f("kg_p"), f("kz")
    want = Counter((koff_p(r), koff_q(r)) for r in range(kk))
    got, all_p, all_q = Counter(), 0, 0
    for grp in range(ng):
        p, q, z = kg_p(grp), kg_q(grp), kz(grp)
        assert 0 <= z < g
        for j in range(g):
            all_p, all_q = max(all_p, p + j * icp), max(all_q, q + j * icq_own)
            if j >= z:
                got[(p + j * icp, q + j * icq_own)] += 1
    assert got == want
    na = nb = 1
    for d in sa:
        na *= d
    for d in sb:
        nb *= d
    rowb_p, rowb_q, gid_m, gid_n = f("rowb_p"), f("rowb_q"), f("gid_m"), f("gid_n")
    assert max(rowb_p(gid_m(x)) for x in range(m)) + all_p < na
    assert max(rowb_q(gid_n(x)) for x in range(n)) + all_q < nb
    if packed:
        # the packed side: rows of NGRP groups one after the other
        row_q, kq = f("row_q"), f("kg_q")
        assert icq == 1 and row_q(1) == ng * g and [kq(i) for i in (0, 1, ng - 1)] == [0, g, (ng - 1) * g]
    # a stage past the last group counts as 0 as a whole
    if ng % 8:
        assert kz(ng) == g
    assert _lib.dense_compile_check(k) > 0


WINDOWS = [("cf", 64, 64, 64, 56, 56, 3), ("cf", 32, 128, 128, 28, 28, 3), ("cf", 9, 24, 40, 29, 37, 3), ("cf", 300, 40, 48, 9, 7, 3),
           ("cf", 16, 64, 128, 39, 43, 5), ("cf", 4, 96, 128, 130, 131, 2)]


@pytest.mark.parametrize("case", WINDOWS, ids=lambda c: "x".join(map(str, c[1:])))
def test_window_positions_are_the_contractions_offsets(case, tmp_path):
    """A row's position plus a tap's offset, and a channel's stride, give the
    element the contraction reads there; the positions of a tile stay inside
    its LDS run, and every load inside the buffer."""
    k, sx, _sw = ct.conv(*case)
    m, n, kk, _splits = _lib.dense_analyze(k)
    src = _lib.dense_source(k)
    f = _host(src, tmp_path)
    koff_p, koff_q, rowb_p, gid_m, vpos, tapq = (f(x) for x in ("koff_p", "koff_q", "rowb_p", "gid_m", "vpos_", "tapq_"))
    bm = int(re.findall(r"constexpr u32 BM = (\d+)u, BN = \d+u, M", src)[-1])
    sp, nt = map(int, re.search(r"NT = (\d+)u, SP = (\d+)u", src).groups()[::-1])
    off = [int(x) for x in re.findall(r"\(rp\[i\] \+ (\d+)u\)", src)]
    cp = int(re.search(r"\(int\)\(c \* (\d+)u\)", src).group(1)) // 4
    vt = int(re.search(r"v = v < (\d+)u \? v : ", src).group(1))
    u, sb, cst = map(int, re.search(r"oA\[e\] = \(v / (\d+)u \* (\d+)u \+ v % \d+u \+ (\d+)u\) \* 4u", src).groups())
    cq = int(re.search(r"tapq_\(tap\) \+ c0 \* (\d+)u", src).group(1))
    e = kk // nt
    assert len(off) == nt and e * nt == kk
    taps = Counter((off[t] + c * cp, tapq(t) + c * cq) for t in range(nt) for c in range(e))
    assert taps == Counter((koff_p(r), koff_q(r)) for r in range(kk))
    v = [vpos(i) for i in range(m)]
    for i in range(m):
        a = (v[i] // u) * sb + v[i] % u + cst
        assert a == rowb_p(gid_m(i)) and v[i] % u + max(off) < u, i
    assert v[-1] + max(off) < vt
    for i in range(0, m, bm):
        t = v[i:i + bm]
        assert min(t) == t[0] and max(t) - t[0] + max(off) < sp
    size = 1
    for d in sx:
        size *= d
    assert (vt - 1) // u * sb + u - 1 + cst + (e - 1) * cp < size
    assert _lib.dense_compile_check(k) > 0


def test_small_and_mixed_contractions_take_no_plane_tile():
    for kind, m, k, n in [("tn", 400, 256, 120), ("nn", 92, 48, 64), ("nn", 38, 288, 16)]:
        assert "NGRP" not in _lib.dense_source(ct.matmul(kind, m, k, n)[0])
    va, vb = (771, 1, 0), (0, 500, 1)
    mixed = ct.program((300, 771, 500), {1}, [va, vb], [F32, F16])
    assert "NGRP" not in _lib.dense_source(mixed)
    # a 3x3 convolution of one channel: K = (1, 3, 3) has no run of four
    assert "NGRP" not in _lib.dense_source(ct.conv("cf", 16, 1, 64, 24, 24, 3)[0])


def test_a_packed_operand_counts_as_a_launch():
    """The weights of a convolution of few channels would be packed first: it
    keeps the direct kernel, where a larger one takes the packed plane tile."""
    assert "NGRP" not in _lib.dense_source(ct.conv("cf", 2, 5, 224, 91, 12, 3)[0])
    assert "kg_qo(" in _lib.dense_source(ct.conv("cf", 6, 120, 232, 103, 10, 3)[0])
