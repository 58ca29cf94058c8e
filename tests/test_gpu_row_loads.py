"""Row kernels written by hand whose loads are not all along the row: a value per row loaded in the row loop beside rows that registers hold."""
import ctypes as C

import numpy as np
import pytest

import ug_amd
from ug_amd import SsaKernel
from ug_amd.api import A, Instr

ADD, MUL = 0, 2
F32, I32 = int(ug_amd.F32), int(ug_amd.I32)


class Text:
    """Instructions one behind the other; every method gives the line of what it appends."""

    def __init__(self):
        self.ins = []

    def put(self, op, dtype=0, sub=0, v=0, n=0, a=None, b=None):
        self.ins.append(Instr(op, dtype, sub, v, n, self.operand(a), self.operand(b)))
        return len(self.ins) - 1

    @staticmethod
    def operand(x):
        if x is None:
            return A()
        if isinstance(x, tuple):  # a constant
            return A(1, I32, 0, 0, x[0], 0.0, 0) if isinstance(x[0], int) else A(1, F32, 0, 0, 0, x[0], 0)
        return A(0, I32, 0, x, 0, 0.0, 0)

    def arg(self, i):
        return self.put(1, F32, n=i)

    def binary(self, op, a, b, dtype=F32):
        return self.put(6, dtype, sub=op, a=a, b=b)

    def load(self, src, at):
        return self.put(8, F32, v=src, a=at)

    def store(self, dst, at, value):
        self.put(13, F32, v=dst, a=at, b=value)

    def loop(self, n):
        return self.put(7, a=(0,), b=(n,), n=1)

    def end(self, begin):
        self.ins[begin].v = self.put(10, v=begin)

    def kernel(self):
        return SsaKernel.from_instrs(self.ins)


def scaled(rows, width, of_row=lambda t, row, width: row):
    """dst[row, :] = a[row, :] * b[of_row] * sum(a[row, :]), arguments a, b, dst."""
    t = Text()
    a, b, dst = t.arg(0), t.arg(1), t.arg(2)
    row = t.loop(rows)
    s = t.load(b, of_row(t, row, width))
    acc = t.put(0, a=(0.0,))
    first = t.binary(MUL, row, (width,), I32)
    j = t.loop(width)
    t.put(9, v=acc, a=t.binary(ADD, acc, t.load(a, t.binary(ADD, first, j, I32))))
    t.end(j)
    c = t.loop(width)
    at = t.binary(ADD, first, c, I32)
    t.store(dst, at, t.binary(MUL, t.binary(MUL, t.load(a, at), s), acc))
    t.end(c)
    t.end(row)
    return t.kernel()


def first_of_row(t, row, width):
    return t.binary(MUL, row, (width,), I32)


def builds(source):
    lib = ug_amd.ughip_lib()
    assert lib.ughip_rtc_check(source.encode(), b"gfx950", None) == 0, lib.ughip_last_error().decode()


def joined(first, second, shared, keep):
    """The source of two kernels as one launch, '' where they stay two: what lies between is the last argument of `first`."""
    a, b, lib, n = first.wire(), second.wire(), ug_amd.ughip_lib(), C.c_size_t()
    args = (C.byref(a), C.byref(b), (C.c_char_p * 2)(b"first", b"second"), (C.c_int * len(shared))(*shared), C.c_size_t(len(shared)), C.c_int(a.n_args - 1), C.c_int(keep))
    assert lib.ughip_codegen_rows_pair(*args, None, C.c_size_t(0), C.byref(n)) == 0, lib.ughip_last_error()
    buf = C.create_string_buffer(n.value + 1)
    assert lib.ughip_codegen_rows_pair(*args, buf, C.c_size_t(n.value + 1), C.byref(n)) == 0
    return buf.value.decode()


SHAPES = [(8, 300), (3, 64), (9, 1024), (2, 8193)]


@pytest.mark.parametrize("rows, width", SHAPES)
@pytest.mark.parametrize("of_row, asked", [(lambda t, row, width: row, lambda r, w: r), (first_of_row, lambda r, w: (r - 1) * w + 1), (lambda t, row, width: (0,), lambda r, w: 1)],
                         ids=["per row", "row start", "one for all"])
def test_a_value_per_row_is_loaded_once_and_where_it_is(rows, width, of_row, asked):
    k = scaled(rows, width, of_row)
    assert k.min_lens() == [rows * width, asked(rows, width), rows * width]
    source, info = k.hip_code("scaled")
    assert info["strategy"] == "row_block"
    builds(source)
    assert source[source.index("__global__"):].count("v1[") == 1


@pytest.mark.parametrize("rows, width", SHAPES)
@pytest.mark.parametrize("keep", [0, 1])
def test_a_value_per_row_in_either_half_of_a_pair(rows, width, keep):
    k = scaled(rows, width)
    src = joined(k, k, [2, -1, -1], keep)   # the second's rows are the first's result, its values per row a buffer of their own
    assert "ug_link" in src
    builds(src)
    assert joined(k, k, [2, 1, -1], keep)   # and the same values per row
    # values per row read from the first's result are other rows' elements or one that another thread holds
    assert joined(k, k, [-1, 2, -1], keep) == "" and joined(k, scaled(rows, width, first_of_row), [-1, 2, -1], keep) == ""


@pytest.mark.gpu
@pytest.mark.parametrize("rows, width", SHAPES)
def test_values_per_row(hip, rows, width):
    rng = np.random.default_rng(7)
    a, b = rng.standard_normal((rows, width)).astype(np.float32), rng.standard_normal(rows).astype(np.float32)
    dst = hip.slice_from(np.zeros(rows * width, np.float32))
    hip.run(hip.compile(scaled(rows, width), "scaled"), [hip.slice_from(a), hip.slice_from(b), dst])
    x = a.astype(np.float64)
    want = x * b[:, None] * x.sum(1, keepdims=True)
    # a sum of `width` terms of size 1 in a tree, two products: against the terms' own size, not the sum's
    np.testing.assert_allclose(dst.to_vec().reshape(a.shape), want, rtol=4 * 2.0 ** -24, atol=(2 + np.log2(width)) * 2.0 ** -24 * np.abs(x).sum(1).max() * np.abs(x * b[:, None]).max())
