"""Products of one row where the workgroup's shape changes: columns per workgroup and their remainders, row lengths around whole waves and the
longest row held in registers, parts of lanes, of waves and of neither, experts' rows side by side."""
import ctypes as C

import numpy as np
import pytest

import plain_hybrid as ph
from gpu_calls import GLU, SWIGLU, Gpu, RowStep, close, get, rand

pytestmark = pytest.mark.gpu
EPS = 1e-3


@pytest.fixture(scope="module")
def gpu(hip):
    return Gpu(hip)


def bound(k):
    """Sums of k products in f32, in any order: their roundings add up like the root of k; the norms' and gates' own are a few ulp."""
    return 2.0 ** -24 * (16 + 4 * k ** 0.5)


@pytest.mark.parametrize("k, n", [(8, 1), (8, 1399), (8, 2801), (8, 5603), (8, 11205), (8, 22401), (504, 9), (512, 257), (520, 3), (1024, 2801), (8184, 5), (8192, 1025), (8200, 5)])
@pytest.mark.parametrize("bf16", [False, True])
def test_columns_and_row_lengths(gpu, k, n, bf16):
    x, y, yn, norm, extra, bias = rand(1, k), rand(2, k), rand(3, k) + 1, rand(4, k) + 1, rand(5, k), rand(6, n)
    w = rand(7, n, k, std=k ** -0.5)
    dw, dyn, dn, db = gpu.up(w, bf16=bf16), gpu.up(yn), gpu.up(norm), gpu.up(bias)
    buf, ex, dst, out = gpu.up(np.concatenate([x, y])), gpu.up(extra), gpu.out(n + k), gpu.out(n)
    gpu.call("ughip_product_row", C.byref(RowStep(x=buf.raw(), w=dw.raw(), n=n, k=k, bias=db.raw(), dst=out.raw())))
    close(get(out, n), w @ x + bias, bound(k))
    gpu.call("ughip_product_row", C.byref(RowStep(x=buf.raw(), y=buf.raw(), y_offset=k, y_norm=dyn.raw(), norm=dn.raw(), extra=ex.raw(), eps=EPS, keep_x=1, x_out=n, w=dw.raw(), n=n, k=k,
                                                  dst=dst.raw())))
    joined = x + ph.rms(y, EPS) * yn + extra
    close(get(dst, n + k)[n:], joined, 3e-6)
    close(get(dst, n + k)[:n], w @ (ph.rms(joined, EPS) * norm), bound(k))


@pytest.mark.parametrize("k, n", [(8, 700), (8, 1399), (8, 2803), (8, 5603), (8, 11205), (1032, 1401), (8192, 9)])
def test_gated_columns(gpu, k, n):
    x, w, bias = rand(1, k), rand(2, 2 * n, k, std=k ** -0.5), rand(3, 2 * n)
    sx, dw, db, out = gpu.up(x), gpu.up(w, bf16=True), gpu.up(bias), gpu.out(n)
    gpu.call("ughip_product_row", C.byref(RowStep(x=sx.raw(), w=dw.raw(), bias=db.raw(), n=n, k=k, act=GLU, act_alpha=1.5, act_shift=1.0, act_limit=2.0, dst=out.raw())))
    v = w @ x + bias
    g, u = np.minimum(v[:n], 2.0), np.clip(v[n:], -2.0, 2.0)
    close(get(out, n), g / (1 + np.exp(-1.5 * g)) * (u + 1), 2 * bound(k))


@pytest.mark.parametrize("k, parts", [(1024, 256), (1024, 128), (1024, 64), (1024, 4), (1024, 2), (2048, 2), (3072, 2), (1536, 2), (1536, 3), (8192, 8), (520, 1), (520, 65), (2560, 2), (3840, 3), (8192, 32), (768, 3), (8, 2), (520, 130), (8192, 2048)])
@pytest.mark.parametrize("after", [False, True])
def test_parts_of_the_row(gpu, k, parts, after):
    n = 33
    x, gate, norm, w = rand(1, k), rand(2, k), rand(3, k) + 1, rand(4, n, k, std=k ** -0.5)
    sx, sg, dn, dw, out = gpu.up(x), gpu.up(gate), gpu.up(norm), gpu.up(w, bf16=True), gpu.out(n)
    gpu.call("ughip_product_row", C.byref(RowStep(x=sx.raw(), gate=sg.raw(), gate_after=int(after), norm=dn.raw(), norm_groups=parts, eps=EPS, w=dw.raw(), n=n, k=k, dst=out.raw())))
    v = ph.rms((x if after else x * ph.silu(gate)).reshape(parts, -1), EPS).reshape(-1) * norm
    close(get(out, n), w @ (v / (1 + np.exp(-gate)) if after else v), bound(k))


@pytest.mark.parametrize("k, n, top", [(8, 1, 1), (16, 1401, 4), (1024, 257, 3), (1408, 96, 5), (1368, 40, 6), (2048, 300, 4), (2056, 20, 4), (8, 5, 32)])
def test_chosen_experts(gpu, k, n, top):
    """Both routed forms against the same choice; with 32 of them on rows of 8 a wave holds all experts' rows."""
    experts = max(top, 7)
    x, w1, w2, logits = rand(1, k), rand(2, experts, 2 * n, k, std=k ** -0.5), rand(3, experts, n, k, std=k ** -0.5), rand(4, experts)
    sx, d1, d2, sl, ids, wts, out = gpu.up(x), gpu.up(w1, bf16=True), gpu.up(w2, bf16=True), gpu.up(logits), gpu.ints(top), gpu.out(top), gpu.out(top * n)
    route = dict(experts=experts, groups=1, keep=1, top=top, route_ids=ids.raw(), route_weights=wts.raw())
    gpu.call("ughip_product_row", C.byref(RowStep(x=sx.raw(), w=d1.raw(), n=n, k=k, act=SWIGLU, route=1, logits=sl.raw(), dst=out.raw(), **route)))
    best = np.argsort(-logits, kind="stable")[:top]
    assert ids.to_vec().tolist() == best.tolist()
    v = np.stack([w1[e] @ x for e in best])
    close(get(out, (top, n)), ph.silu(v[:, :n]) * v[:, n:], 2 * bound(k))
    a = rand(5, top, k)
    sa, o2 = gpu.up(a), gpu.out(n)
    gpu.call("ughip_product_row", C.byref(RowStep(x=sa.raw(), w=d2.raw(), n=n, k=k, route=2, dst=o2.raw(), **route)))
    close(get(o2, n), sum(get(wts, top)[j] * (w2[e] @ a[j]) for j, e in enumerate(best)), bound(top * k))
