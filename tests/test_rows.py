"""Which programs are steps of a row sequence, without a GPU: how each buffer
is taken is compared with the elements its strides reach."""
import pytest

from tests import rowprograms as rp
from tests.rowprograms import COL, MAT, VEC
from tinyhvm_amd import _lib, abi

SUM, RMAX = abi.UOP_SUM, abi.UOP_RMAX
MATRIX, VECTOR, OTHER = 1, 2, 3
ROWS, COLS = 12, 512
KINDS = [MAT, VEC, COL, (1, ROWS, 0), (COLS, 1, 1), (1, 0, 1), (COLS, 2, 0), (2 * COLS, 1, 0), (2, 0, 0), (0, 0, 0), (COLS, 1, COLS),
         (COLS, 0, 0), (ROWS, 1, 0)]


@pytest.mark.parametrize("split", [1, 32])
@pytest.mark.parametrize("reduce", [None, SUM, RMAX])
@pytest.mark.parametrize("kind", KINDS, ids=str)
def test_classes_are_the_elements_reached(kind, reduce, split):
    k = rp.program(ROWS, COLS, [kind], lambda o, v: v, reduce=reduce, split=split)
    got = _lib.row_classes(k)
    assert got[0] == ((VECTOR, 0) if reduce else (MATRIX, 0))
    rs, cs, off = rp.strides(kind, COLS)
    at = {(i, j): i * rs + j * cs + off for i in range(ROWS) for j in range(COLS)}
    matrix = all(v == i * COLS + j for (i, j), v in at.items())
    vector = all(v == i for (i, j), v in at.items())
    cls, div = got[1]
    assert (cls == MATRIX) == matrix
    if vector:
        assert cls == VECTOR and (reduce or div == COLS)
    elif not matrix:   # a vector of other rows: its div is not a row
        assert cls == OTHER or (not reduce and cls == VECTOR and div != COLS)


def test_two_ways_to_take_a_buffer_are_neither():
    k = rp.program(ROWS, COLS, [MAT, VEC], lambda o, a, b: o(abi.UOP_ADD, a, b))
    for i in range(k.n_ops):
        if k.ops[i].type == abi.KOP_LOAD:
            k.ops[i].imm.u = 1
    assert _lib.row_classes(k)[1][0] == OTHER


def test_softmax_compiles_as_one_kernel():
    sub = lambda o, a, b: o(abi.UOP_SUB, a, b)  # noqa: E731
    ks = [rp.program(64, 1000, [MAT], lambda o, v: v, reduce=RMAX),
          rp.program(64, 1000, [MAT, VEC], lambda o, a, b: o(abi.UOP_EXP, sub(o, a, b))),
          rp.program(64, 1000, [MAT], lambda o, v: v, reduce=SUM),
          rp.program(64, 1000, [MAT, VEC], lambda o, a, b: o(abi.UOP_DIV, a, b))]
    assert _lib.row_compile_check(ks) > 0
    with pytest.raises(ValueError):   # rows of another length
        _lib.row_compile_check(ks[:1] + [rp.program(64, 996, [MAT], lambda o, v: v)])
    with pytest.raises(ValueError):   # a thread's four elements cross the row's end
        _lib.row_compile_check([rp.program(64, 1001, [MAT], lambda o, v: v, reduce=RMAX),
                                rp.program(64, 1001, [MAT], lambda o, v: o(abi.UOP_EXP, v))])


def test_a_thread_of_pieces_of_two_rows_is_no_step(monkeypatch):
    """With several vectors a thread, a thread's elements lie far apart: a
    workgroup's threads would reach rows that other workgroups still reduce."""
    ks = [rp.program(4096, 1000, [MAT], lambda o, v: v, reduce=RMAX),
          rp.program(4096, 1000, [MAT, VEC], lambda o, a, b: o(abi.UOP_EXP, o(abi.UOP_SUB, a, b)))]
    assert _lib.row_compile_check(ks) > 0
    for per in "28":
        monkeypatch.setenv("THVM_HIP_EW_PER_THREAD", per)
        assert "w_ < %su" % per in _lib.kernel_source(ks[1])[0]
        with pytest.raises(ValueError):
            _lib.row_compile_check(ks)
