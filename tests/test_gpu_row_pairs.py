"""Row kernels that hold their rows in registers, and two of them as one launch: widths around the groups of four, the waves and the rows per
workgroup, what somebody else can see of the buffer between the two, and neighbours that must stay two launches."""
import ctypes as C

import numpy as np
import pytest

import test_gpu_parity as parity
import ug_amd
from ug_amd import LazyBuffer as LB
from ug_amd import Schedule

EPS32 = 2.0 ** -24


def _x(seed, *shape):
    return np.random.default_rng(seed).standard_normal(shape).astype(np.float32)


def _softmax(x):
    e = np.exp(x.astype(np.float64) - x.max(-1, keepdims=True))
    return e / e.sum(-1, keepdims=True)


def _parts(x, weight=None, dev=None):
    """The softmax in steps, so that the buffer between its kernels has a name here: (exponentials, result)."""
    wide = lambda r: r.broadcast(x.shape)  # noqa: E731
    lx = LB.copy(x, x.shape, dev)
    e = lx.binary("sub", wide(lx.reduce("max", len(x.shape) - 1))).unary("exp")
    out = e.binary("div", wide(e.reduce("sum", len(x.shape) - 1)))
    return e, out if weight is None else out.binary("mul", wide(LB.copy(weight, (1,) * (len(x.shape) - 1) + weight.shape, dev)))


def _bare(*buffers):
    """The same buffers without the operands that their Python objects hold: only the graph does then."""
    for b in buffers:
        b._keep = [k for k in b._keep if not isinstance(k, LB)]
    return buffers


def _whole_numbers(x, dev):
    """(x - max) times the sum of that, row by row."""
    wide = lambda r: r.broadcast(x.shape)  # noqa: E731
    lx = LB.copy(x, x.shape, dev)
    e = lx.binary("sub", wide(lx.reduce("max", 1)))
    return _bare(e.binary("mul", wide(e.reduce("sum", 1))))[0]


def _joined(lb, keep=0):
    """The source of the first two items of a graph as one launch, '' where they stay two; needs no device."""
    s = Schedule.create_one(lb)
    ka, kb = s.item_ssa(0), s.item_ssa(1)
    a, b, lib = ka.wire(), kb.wire(), ug_amd.ughip_lib()
    names, n = (C.c_char_p * 2)(b"first", b"second"), C.c_size_t()
    shared = (C.c_int * b.n_args)(*([a.n_args - 1] + [-1] * (b.n_args - 1)))
    args = (C.byref(a), C.byref(b), names, shared, C.c_size_t(b.n_args), C.c_int(a.n_args - 1), C.c_int(keep))
    assert lib.ughip_codegen_rows_pair(*args, None, C.c_size_t(0), C.byref(n)) == 0, lib.ughip_last_error()
    buf = C.create_string_buffer(n.value + 1)
    assert lib.ughip_codegen_rows_pair(*args, buf, C.c_size_t(n.value + 1), C.byref(n)) == 0
    return buf.value.decode()


def test_which_neighbours_are_joined(cpu):
    kernel = lambda src: src[src.index("__global__"):]  # noqa: E731
    for shape in [(1, 4), (7, 333), (5, 256), (3, 8192), (2, 3, 49152)]:
        src = kernel(_joined(_parts(_x(1, *shape), dev=cpu)[1]))
        assert "ug_link" in src and src.count("__restrict__") == 2, shape  # what lies between is no argument
        assert kernel(_joined(_parts(_x(1, *shape), dev=cpu)[1], keep=1)).count("__restrict__") == 3
    assert _joined(_parts(_x(1, 2, 3), dev=cpu)[1]) == ""  # rows shorter than a group
    assert _joined(_parts(_x(1, 2, 49153), dev=cpu)[1]) == ""  # more than a thread holds
    e, _ = _parts(_x(1, 64, 64), dev=cpu)
    t = e.transpose(0, 1)
    assert _joined(t.binary("div", t.reduce("sum", 1).broadcast((64, 64)))) == ""  # another row's elements


@pytest.mark.parametrize("each, joins", [(8, True), (30, True), (31, False), (40, False)])
def test_a_pair_has_no_more_arguments_than_a_launch_takes(cpu, each, joins):
    """Two kernels of 64 buffers at most each run; as one they would have up to twice that, which a launch refuses."""
    x = _x(1, 3, 8)
    more = lambda b: [b := b.binary("mul", LB.copy(x, x.shape, cpu)) for _ in range(each)][-1]  # noqa: E731
    lx = LB.copy(x, x.shape, cpu)
    e = more(lx.binary("sub", lx.reduce("max", 1).broadcast(x.shape)))
    [out] = _bare(more(e.binary("div", e.reduce("sum", 1).broadcast(x.shape))))
    args = [Schedule.create_one(out).item_ssa(i).wire().n_args for i in range(2)]
    assert args == [each + 2, each + 2] and (_joined(out, keep=1) != "") == joins


WIDTHS = [4, 5, 7, 63, 64, 65, 128, 255, 256, 257, 259, 260, 767, 768, 769, 1020, 1023, 1531, 4095, 4096, 4097, 8191, 8193, 16380, 49151, 49152, 49153]


@pytest.mark.gpu
@pytest.mark.parametrize("width", WIDTHS)
@pytest.mark.parametrize("rows", [1, 3, 9])
def test_softmax_and_norm_of_any_width(hip, width, rows):
    x, w = 3 * _x(width, rows, width), 1 + 0.1 * _x(5, width)
    got = ug_amd.llama.softmax(LB.copy(x, x.shape, hip)).data_vec().reshape(x.shape)
    # an exponential is 2 ulp of its argument's rounding off (|x - max| up to some 30), a sum of n terms in a tree at most log2(n) roundings
    np.testing.assert_allclose(got, _softmax(x), rtol=(40 + np.log2(width)) * 2 * EPS32, atol=1e-30)
    got = ug_amd.llama.rms_norm(LB.copy(x, x.shape, hip), LB.copy(w, w.shape, hip), 1e-5).data_vec().reshape(x.shape)
    want = x / np.sqrt((x.astype(np.float64) ** 2).mean(-1, keepdims=True) + 1e-5) * w
    np.testing.assert_allclose(got, want, rtol=(10 + width / 1024 + np.log2(width)) * EPS32, atol=1e-30)


@pytest.mark.gpu
@pytest.mark.parametrize("width", [4, 5, 255, 256, 257, 4099, 24577, 49152, 49153])
@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_rows_of_whole_numbers(hip, width, dtype):
    x = np.random.default_rng(width).integers(-90, 90, (5, width)).astype(dtype)
    out = _whole_numbers(x, hip)
    cs = Schedule.create_one(out).compile()
    assert ("ug_link" in cs.funcs()[0]["source"]) == (width <= 49152)
    cs.run()
    e = x - x.max(1, keepdims=True)
    assert np.array_equal(out.data_vec().reshape(x.shape), e * e.sum(1, keepdims=True, dtype=dtype))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(3, 5), (9, 130), (4, 3, 257), (33, 2052)])
def test_what_others_see_of_the_buffer_between(hip, shape):
    """Held by a handle it is written, and the same as ever; held by nobody it is never realised; both give the result's same bits."""
    x, w = _x(2, *shape), _x(3, shape[-1])
    e, out = _parts(x, w, dev=hip)
    Schedule.create_one(out).compile().run()
    assert e.realized()
    np.testing.assert_allclose(e.data_vec().reshape(shape), np.exp(x.astype(np.float64) - x.max(-1, keepdims=True)), rtol=40 * EPS32)
    kept = out.data_vec()
    e, out = _bare(*_parts(x, w, dev=hip))
    del e
    Schedule.create_one(out).compile().run()
    assert np.array_equal(kept, out.data_vec())
    np.testing.assert_allclose(kept.reshape(shape), _softmax(x) * w, rtol=60 * EPS32, atol=1e-30)
    # both at once: the buffer is an output itself
    e, out = _parts(x, w, dev=hip)
    Schedule.create([e, out]).compile().run()
    assert np.array_equal(kept, out.data_vec()) and e.realized()


@pytest.mark.gpu
def test_everything_is_compiled_when_compile_returns(hip):
    """One of a pair's kernels by itself, on the cache that the pair was compiled with: its code is made by compile, not by run."""
    objects, cache, x = lambda: parity.n_code_objects(hip), ug_amd.CompilationCache(), _x(8, 37, 1234)  # noqa: E731  (a shape of its own: nothing of it is compiled yet)
    e, out = _bare(*_parts(x, dev=hip))
    del e
    before = objects()
    pair = Schedule.create_one(out).compile(cache)
    assert objects() == before + 1 and len(cache) == 1
    info = pair.funcs()
    assert len(info) == 2 and all("ug_link" in f["source"] and f["info"]["strategy"] == "row_block" for f in info)
    for alone in (lambda: _parts(x, dev=hip)[0], lambda: _quotient(hip, x)):
        lb = alone()
        cs = Schedule.create_one(lb).compile(cache)
        compiled = objects()
        cs.run()
        assert objects() == compiled > before + 1
    pair.run()
    assert objects() == compiled
    np.testing.assert_allclose(out.data_vec().reshape(x.shape), _softmax(x), rtol=60 * EPS32, atol=1e-30)


def _quotient(dev, x):
    e = LB.copy(np.exp(x), x.shape, dev)
    return e.binary("div", e.reduce("sum", 1).broadcast(x.shape))


def _reads(dev):
    """Who may come to see the buffer between a softmax's kernels: name -> (what to schedule from (e, out), what holds it beside that, what it should
    read of the exponentials)."""
    shape, w = (5, 6), _x(9, 6, 3)
    ones = LB.copy(np.ones(shape, np.float32), shape, dev)
    return {
        "a handle": (lambda e, out: [out], lambda e: e, lambda e: e),
        "a sibling": (lambda e, out: [out], lambda e: e.binary("add", ones), lambda e: e + 1),
        "a sibling's sibling": (lambda e, out: [out], lambda e: e.binary("mul", ones).unary("neg").reduce("sum", 1), lambda e: np.broadcast_to(-e.sum(1, keepdims=True), shape)),
        "a reshape": (lambda e, out: [out], lambda e: e.reshape((30,)), lambda e: e.reshape(30)),
        "a view": (lambda e, out: [out], lambda e: e.narrow(1, 2, 3), lambda e: e[:, 2:5]),
        "an output": (lambda e, out: [e, out], None, None),
        "a later kernel": (lambda e, out: [out, e.reduce("sum", 0)], None, None),
        "a product": (lambda e, out: [out, e.matmul(LB.copy(w, w.shape, dev))], None, None),
        "a product held elsewhere": (lambda e, out: [out], lambda e: e.matmul(LB.copy(w, w.shape, dev)), lambda e: e @ w),
        "a custom op": (lambda e, out: [out, LB.custom(lambda s: s[1].copy_host_to_device(s[0].to_vec()), [e], shape, ug_amd.F32, dev)], None, None),
        "another schedule": (lambda e, out: [out], lambda e: Schedule.create_one(e.binary("add", ones)), None),
    }


READS = ["a handle", "a sibling", "a sibling's sibling", "a reshape", "a view", "an output", "a later kernel", "a product", "a product held elsewhere", "a custom op", "another schedule"]


def _read(dev, name):
    make, hold, _ = _reads(dev)[name]
    e, out = _parts(_x(6, 5, 6), dev=dev)
    roots = make(e, out)
    held = hold(e) if hold else None
    _bare(*[b for b in [e, out, held, *roots] if isinstance(b, LB)])
    if isinstance(held, Schedule):
        _bare(*held._keep)
        held._keep = []
    del e
    s = Schedule.create(roots)
    return s, roots, held


@pytest.mark.parametrize("name", READS)
def test_a_buffer_that_somebody_can_reach_is_written(cpu, name):
    s, roots, held = _read(cpu, name)
    assert s.pair(0) is True


def test_a_buffer_that_nobody_can_reach_is_not_written(cpu):
    for weight in (None, _x(1, 6)):
        e, out = _bare(*_parts(_x(6, 5, 6), weight, cpu))
        del e
        s = Schedule.create_one(out)
        assert s.pair(0) is False and s.pair(1) is None
        compiled = s.compile()
        assert s.pair(0) is True    # (this device's two launches hold it)
        del compiled
        assert s.pair(0) is False
    # one behind the other
    [out] = _bare(ug_amd.llama.softmax(ug_amd.llama.softmax(LB.copy(_x(6, 5, 6), (5, 6), cpu))))
    s = Schedule.create_one(out)
    assert [s.pair(i) for i in range(len(s.items()))] == [False, False, False, None]
    # kernels without a reduction are not row kernels
    e = LB.copy(_x(1, 4, 8), (4, 8), cpu).unary("exp")
    out = e.binary("mul", e)
    s = Schedule.create_one(out)
    assert [s.pair(i) for i in range(len(s.items()))] == [None] * len(s.items())


@pytest.mark.gpu
@pytest.mark.parametrize("name", READS)
def test_everybody_sees_what_is_between(hip, name):
    s, roots, held = _read(hip, name)
    cs = s.compile()
    assert "ug_link" in cs.funcs()[0]["source"]
    cs.run()
    x = _x(6, 5, 6).astype(np.float64)
    e = np.exp(x - x.max(-1, keepdims=True))
    want = {"an output": [e, _softmax(x)], "a later kernel": [_softmax(x), np.broadcast_to(e.sum(0), x.shape)], "a product": [_softmax(x), e @ _x(9, 6, 3)], "a custom op": [_softmax(x), e]}.get(name, [_softmax(x)])
    for got, v in zip(roots, want):
        np.testing.assert_allclose(got.data_vec().reshape(v.shape), v, rtol=1e-5, atol=1e-6)
    if _reads(hip)[name][2]:
        v = _reads(hip)[name][2](e)
        np.testing.assert_allclose(held.data_vec().reshape(v.shape), v, rtol=1e-5, atol=1e-6)


@pytest.mark.gpu
def test_neighbours_that_stay_two_launches(hip):
    x = _x(4, 64, 64)
    e, _ = _parts(x, dev=hip)
    t = e.transpose(0, 1)
    out = t.binary("div", t.reduce("sum", 1).broadcast((64, 64)))
    del e, t
    want = np.exp(x.astype(np.float64) - x.max(-1, keepdims=True)).T
    np.testing.assert_allclose(out.data_vec().reshape(64, 64), want / want.sum(-1, keepdims=True), rtol=60 * EPS32)


@pytest.mark.gpu
@pytest.mark.parametrize("row", [[np.inf, 1, 2, 3, 4], [-np.inf, 1, 2, 3, 4], [np.nan, 1, 2, 3, 4], [-3.4028235e38] * 5, [3.4028235e38, 1, 2, 3, -3.4028235e38]])
def test_extreme_rows(hip, cpu, row):
    """Infinities, NaN and the lowest value give what the oracle's two kernels give."""
    x = np.array([row * 70, [0.5] * (5 * 70)], np.float32)
    got, want = (ug_amd.llama.softmax(LB.copy(x, x.shape, d)).data_vec().reshape(x.shape) for d in (hip, cpu))
    np.testing.assert_allclose(got, want, rtol=1e-5, atol=1e-30)
