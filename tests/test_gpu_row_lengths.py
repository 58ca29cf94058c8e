"""Row kernels of lazy graphs on rows that are no multiple of four elements: the last group of four overlaps the one before it."""
import numpy as np
import pytest

import ug_amd
from ug_amd import LazyBuffer as LB, Schedule, rng

pytestmark = pytest.mark.gpu


# one element more and less than whole groups, waves and workgroups (64, 128, 1024 threads of four); rows in one pass and in several
@pytest.mark.parametrize("cols", [257, 258, 259, 509, 513, 1023, 1025, 4093, 4095, 4097, 4099, 9001])
@pytest.mark.parametrize("rows", [1, 7])
def test_rows_of_any_length(hip, rows, cols):
    x, alpha = rng.normal(cols, rows * cols, 3.0).reshape(rows, cols), rng.normal(cols + 1, cols, 1.0)
    x[0, cols // 2] = -np.inf        # no weight in the softmax, the smallest of its row
    x[-1, -1] = 50.0                 # the last element, folded once only: it is nearly all of its row's sum
    x64, finite = x.astype(np.float64), np.where(np.isfinite(x), x, 0).astype(np.float32)
    lx, lf = LB.copy(x, (rows, cols), hip), LB.copy(finite, (rows, cols), hip)
    whole = LB.copy(finite.astype(np.int32), (rows, cols), hip)
    sm, rn = ug_amd.llama.softmax(lx), ug_amd.llama.rms_norm(lf, LB.copy(alpha, (cols,), hip), 1e-5)
    red = {op: lf.reduce(op, 1) for op in ("sum", "max", "min")}
    ints = whole.reduce("sum", 1)
    sched = Schedule.create([sm, rn, ints, *red.values()])
    sched.compile().run()
    e = np.exp(x64 - x64.max(1, keepdims=True))
    np.testing.assert_allclose(sm.data_vec().reshape(rows, cols), e / e.sum(1, keepdims=True), rtol=1e-5, atol=1e-30)
    f64 = finite.astype(np.float64)
    np.testing.assert_allclose(rn.data_vec().reshape(rows, cols), f64 / np.sqrt((f64 ** 2).mean(1, keepdims=True) + 1e-5) * alpha, rtol=1e-5, atol=1e-30)
    got = {op: lb.data_vec().reshape(rows, -1)[:, 0] for op, lb in red.items()}
    np.testing.assert_array_equal(got["max"], finite.max(1))
    np.testing.assert_array_equal(got["min"], finite.min(1))
    assert np.all(np.abs(got["sum"] - f64.sum(1)) <= cols * np.finfo(np.float32).eps * np.abs(f64).sum(1))
    np.testing.assert_array_equal(ints.data_vec().reshape(rows, -1)[:, 0], finite.astype(np.int32).sum(1))


def test_a_row_with_not_a_number(hip):
    x = np.ones((2, 1531), np.float32)
    x[1, 1529] = np.nan
    lx = LB.copy(x, (2, 1531), hip)
    s = lx.reduce("sum", 1)
    Schedule.create_one(s).compile().run()
    got = s.data_vec().reshape(2, -1)[:, 0]
    assert got[0] == 1531 and np.isnan(got[1])
