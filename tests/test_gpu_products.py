"""Product kernels at the sizes where they can go wrong -- tile edges, remainders, the shortest loops -- against float64."""
import ctypes as C

import numpy as np
import pytest

import ug_amd
from gpu_calls import BF16, F32, GELU_MUL, GLU, NONE, SWIGLU, Gpu, Product, close, get, p, rand, view
from test_gpu_parity import _raw_matmul
from ug_amd import rng

pytestmark = pytest.mark.gpu

RING = {"10": "256x128", "12": "128x128", "13": "64x128", "9": "64x64"}  # GEMM_SHAPE -> tile


def rounded(dtype, v):
    return rng.bf16_round(v) if dtype == "bf16" else v.astype(np.float16).astype(np.float32)


# 4 .. 9 K tiles: the ring's first and last rounds alone, then odd and even counts of steady ones
@pytest.mark.parametrize("bmnk", [(1, 300, 264, 256), (2, 257, 136, 320), (3, 9, 8, 384), (1, 63, 392, 448), (1, 128, 128, 512), (1, 65, 1000, 576)])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("rhs_nk", [True, False], ids=["NT", "NN"])
def test_ring_tiles(hip, tune, bmnk, dtype, rhs_nk):
    """Every tile of the ring on rows and columns that hang over it: the bound of an f32 sum rounded once, and small integers exactly."""
    b, m, n, k = bmnk
    dt = ug_amd.BF16 if dtype == "bf16" else ug_amd.F16
    a, w = rounded(dtype, rng.uniform_pm1(1, b * m * k)).reshape(b, m, k), rounded(dtype, rng.uniform_pm1(2, b * k * n)).reshape(b, k, n)
    exact = np.matmul(a.astype(np.float64), w.astype(np.float64))
    bound = (2.0 ** -8 if dtype == "bf16" else 2.0 ** -11) * np.abs(exact) + k * np.finfo(np.float32).eps * np.matmul(np.abs(a).astype(np.float64), np.abs(w).astype(np.float64))
    ai, wi = np.floor(a * 4), np.floor(w * 4)
    whole = rounded(dtype, np.matmul(ai, wi).ravel()).reshape(exact.shape)  # (sums below 2^24)
    for shape, tile in RING.items():
        if shape == "9" and not rhs_nk:
            continue  # the transposing reads want 128 columns
        tune.setenv("UGHIP_GEMM_SHAPE", shape)
        print("ring", dtype, bmnk, "NT" if rhs_nk else "NN", tile, flush=True)
        got = _raw_matmul(hip, dt, a, w, rhs_nk)
        assert ug_amd.last_kernel() == f"gemm_dma4<{dtype},{'NT' if rhs_nk else 'NN'},{tile},512t,ring>"
        assert np.all(np.abs(got - exact) <= bound * 1.001 + 1e-7)
        np.testing.assert_array_equal(_raw_matmul(hip, dt, ai, wi, rhs_nk), whole)


@pytest.mark.parametrize("m, n, k, groups", [(1, 8, 64, 0), (17, 72, 128, 0), (193, 392, 192, 0), (70, 136, 320, 0), (300, 264, 384, 0), (301, 40, 448, 5), (40, 136, 576, 3)])
@pytest.mark.parametrize("act", [NONE, SWIGLU, GLU])
def test_ring_rows(hip, tune, m, n, k, groups, act):
    """Products of rows on every tile of the ring: bias, gated units, rows gathered and sorted by matrix (one matrix without any)."""
    gpu, rows, mats = Gpu(hip), n if act == NONE else 2 * n, max(1, groups)
    x, w, bias = rand(1, m, k), rand(2, mats, rows, k, std=k ** -0.5), rand(3, rows, std=0.5)
    if groups:
        gen = np.random.default_rng(4)
        end = np.sort(gen.integers(0, m + 1, groups)).astype(np.int32)
        end[0], end[-1] = 0, m
        src, bias = gen.integers(0, m, m).astype(np.int32), 0 * bias
        of = np.searchsorted(end, np.arange(m), side="right")
        y = np.stack([w[of[i]] @ x[src[i]] for i in range(m)])
    else:
        y = x @ w[0].T + bias
    if act != NONE:
        limit, alpha, shift = (1.5, 1.702, 1.0) if act == GLU else (1e9, 1.0, 0.0)
        g, u = np.minimum(y[:, :n], limit), np.clip(y[:, n:], -limit, limit)
        y = g / (1 + np.exp(-alpha * g)) * (u + shift)
    dx, dw, db = gpu.up(x, bf16=True), gpu.up(w, bf16=True), gpu.up(bias)
    idx = (gpu.up(src), gpu.up(end)) if groups else (None, None)
    for shape, tile in {**RING, "11": "192x192"}.items():
        tune.setenv("UGHIP_GEMM_SHAPE", shape)
        dst = gpu.out(m * n + 8)
        q = Product(x=view(dx, 0, k), dst=view(dst, 0, n), w=dw.raw(), bias=None if groups else db.raw(), m=m, n=n, k=k, product=BF16, act=act, row_index=idx[0].raw() if groups else None,
                    group_end=idx[1].raw() if groups else None, groups=groups, x_rows=m if groups else 0, act_alpha=1.702 if act == GLU else 0, act_shift=1.0 if act == GLU else 0,
                    act_limit=1.5 if act == GLU else 0)
        print("ring rows", m, n, k, groups, act, tile, flush=True)
        gpu.call("ughip_product_rows", C.byref(q))
        assert f"{tile},512t,ring,rows" in ug_amd.last_kernel()
        out = get(dst, m * n + 8)
        assert np.all(np.isnan(out[m * n :])), "wrote past the end"
        close(out[: m * n].reshape(m, n), y, 2e-5)


# columns of a last tile that hang over it (192; 96 gated), one row to three tiles of them; four K tiles, the fewest, and odd and even counts
@pytest.mark.parametrize("m, n, k, groups", [(1, 8, 256, 0), (257, 192, 320, 0), (300, 200, 384, 0), (520, 392, 256, 0), (301, 104, 448, 4)])
@pytest.mark.parametrize("act", [NONE, SWIGLU, GLU])
@pytest.mark.parametrize("bf16_out", [False, True], ids=["f32", "bf16"])
def test_rows_on_256x192_tiles(hip, tune, m, n, k, groups, act, bf16_out):
    """Rows on 256 x 192 tiles with one wave per SIMD: the bits of the ring's 256 x 128 tiles, nothing behind the result."""
    gpu, rows, mats = Gpu(hip), n if act == NONE else 2 * n, max(1, groups)
    dx, dw, db = gpu.up(rand(1, m, k), bf16=True), gpu.up(rand(2, mats, rows, k, std=k ** -0.5), bf16=True), gpu.up(rand(3, rows, std=0.5))
    idx = (gpu.up(np.random.default_rng(4).integers(0, m, m).astype(np.int32)), gpu.up(np.array([0, m // 3, m // 3, m], np.int32))) if groups else (None, None)
    got = {}
    for shape, name in (("14", "256x192,256t,rows"), ("10", "256x128,512t,ring,rows")):
        tune.setenv("UGHIP_GEMM_SHAPE", shape)
        dst = gpu.out(m * n + 8, bf16=bf16_out)
        q = Product(x=view(dx, 0, k), dst=view(dst, 0, n), w=dw.raw(), bias=None if groups else db.raw(), m=m, n=n, k=k, product=BF16, act=act, row_index=idx[0].raw() if groups else None,
                    group_end=idx[1].raw() if groups else None, groups=groups, x_rows=m if groups else 0, act_alpha=1.702 if act == GLU else 0, act_shift=1.0 if act == GLU else 0,
                    act_limit=1.5 if act == GLU else 0)
        print("256x192 rows", m, n, k, groups, act, shape, flush=True)
        gpu.call("ughip_product_rows", C.byref(q))
        assert name in ug_amd.last_kernel(), ug_amd.last_kernel()
        got[shape] = get(dst, m * n + 8)
        assert np.all(np.isnan(got[shape][m * n :])) and not np.any(np.isnan(got[shape][: m * n]))
    np.testing.assert_array_equal(got["14"][: m * n], got["10"][: m * n])


@pytest.mark.parametrize("m, n, k", [(385, 264, 256), (400, 136, 448)])
def test_ring_planes(hip, tune, m, n, k):
    """Three bf16 terms on the ring's tiles, with a K split where it divides: the bound of an f32 sum."""
    gpu, Z = Gpu(hip), C.c_size_t
    x, w, r = rng.normal(1, m * k).reshape(m, k), rand(2, n, k, std=k ** -0.5), rng.normal(3, m * n).reshape(m, n)
    want = x.astype(np.float64) @ w.T + r
    bound = k * np.finfo(np.float32).eps * (np.abs(x).astype(np.float64) @ np.abs(w).T) + 4 * np.finfo(np.float32).eps * np.abs(want) + 1e-7
    dx, dw, dr = gpu.up(x), gpu.up(w, bf16=True), gpu.up(r)
    for shape, tile in RING.items():
        if shape == "10":
            continue  # not a tile of this product
        for split in ("1", "2"):
            if split == "2" and (k // 64) % 2:
                continue
            tune.setenv("UGHIP_X3_DMA", shape)
            tune.setenv("UGHIP_X3_SPLIT", split)
            dst = gpu.out(m * n)
            print("ring planes", m, n, k, tile, split, flush=True)
            gpu.call("ughip_linear_add_rows", p(dx), p(dw), p(dr), p(dst), Z(m), Z(n), Z(k), 1)
            assert f"{tile},512t,ring,3 planes" in ug_amd.last_kernel()
            assert np.all(np.abs(get(dst, (m, n)) - want) <= bound)


# tile edges (64; 128 where that many tiles fill the chip), K steps of 64 / 32 elements: none whole, one, one and a remainder, several; single rows
# and columns, and fewer than eight of them (another kernel's)
@pytest.mark.parametrize("bmnk", [(1, 1, 1, 1), (2, 8, 9, 7), (1, 63, 65, 33), (3, 65, 64, 31), (1, 129, 8, 64), (2, 9, 77, 65), (1, 64, 7, 129), (1, 7, 200, 128), (1, 130, 66, 200), (1, 2049, 2001, 70)])
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("rhs_nk", [True, False], ids=["NT", "NN"])
@pytest.mark.parametrize("lhs_mk", [True, False], ids=["rows", "transposed"])
def test_products_of_any_size(hip, bmnk, dtype, rhs_nk, lhs_mk):
    """Any size, operands that start at any element and lie either way: the bound of an f32 sum (rounded once for 16 bits), nothing written past the
    result, nothing read from behind the operands (not-a-number there)."""
    b, m, n, k = bmnk
    dt, enc = {"f32": (ug_amd.F32, lambda v: v), "f16": (ug_amd.F16, lambda v: v.astype(np.float16)), "bf16": (ug_amd.BF16, rng.to_bf16_bits)}[dtype]
    a, w = rng.uniform_pm1(1, b * m * k), rng.uniform_pm1(2, b * k * n)
    if dtype != "f32":
        a, w = rounded(dtype, a), rounded(dtype, w)
    a, w = a.reshape(b, m, k), w.reshape(b, k, n)
    nan = np.full(3, np.nan, np.float32)
    sa = hip.slice_from(enc(np.concatenate([nan, (a if lhs_mk else np.swapaxes(a, 1, 2)).ravel(), nan]).astype(np.float32)))
    sw = hip.slice_from(enc(np.concatenate([nan, (np.swapaxes(w, 1, 2) if rhs_nk else w).ravel(), nan]).astype(np.float32)))
    dst = hip.slice_from(enc(np.full(b * m * n + 9, 7.0, np.float32)))
    print("any size", dtype, bmnk, rhs_nk, lhs_mk, flush=True)
    hip.matmul(dst, sa, sw, (b, m, n, k), ((b, m, k), (m * k, k, 1) if lhs_mk else (m * k, 1, m), 3), ((b, k, n), (k * n, 1, k) if rhs_nk else (k * n, n, 1), 3))
    got = dst.to_vec()
    got = (rng.from_bf16_bits(got) if dtype == "bf16" else got).astype(np.float64)
    assert np.all(got[b * m * n :] == 7.0), "wrote past the end"
    exact = np.matmul(a.astype(np.float64), w.astype(np.float64))
    bound = {"f32": 0, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype] * np.abs(exact) + (k + 1) * np.finfo(np.float32).eps * np.matmul(np.abs(a).astype(np.float64), np.abs(w).astype(np.float64))
    assert np.all(np.abs(got[: b * m * n].reshape(exact.shape) - exact) <= bound * 1.001 + 1e-7)


# products of one tile, of several, of tiles of both sizes, in batches; f32 on both sides of one step by element
@pytest.mark.parametrize("b, m, n, k, dtype, kernel", [(300, 33, 17, 40, "f32", "gemm_any<f32>"), (17, 9, 70, 65, "f16", "gemm_any<f16>"), (9, 65, 129, 130, "bf16", "gemm_any<bf16,words>"),
                                                       (3, 1155, 1155, 130, "bf16", "gemm_any<bf16,128x128,words>"), (5, 70, 130, 16, "f32", "gemm_any<f32,by element>"),
                                                       (5, 70, 131, 17, "f32", "gemm_any<f32>"), (2, 20, 7, 100, "f16", "gemm_any<f16,by element>")])
@pytest.mark.parametrize("shared", [False, True], ids=["batched", "one lhs"])
def test_batches_of_products_of_any_size(hip, b, m, n, k, dtype, kernel, shared):
    """Batches, a left operand with padded rows that is each product's own or all products' (batch stride 0), and the kernel by its name."""
    gap = 3
    a, w = rng.uniform_pm1(1, b * m * k), rng.uniform_pm1(2, b * k * n)
    dt, enc = {"f32": (ug_amd.F32, lambda v: v), "f16": (ug_amd.F16, lambda v: v.astype(np.float16)), "bf16": (ug_amd.BF16, rng.to_bf16_bits)}[dtype]
    if dtype != "f32":
        a, w = rounded(dtype, a), rounded(dtype, w)
    a, w = a.reshape(b, m, k)[: 1 if shared else b], w.reshape(b, k, n)
    padded = np.full((a.shape[0], m, k + gap), np.nan, np.float32)
    padded[:, :, :k] = a
    sa, sw, dst = hip.slice_from(enc(padded.ravel())), hip.slice_from(enc(w.ravel())), hip.slice_from(enc(np.full(b * m * n + 9, 7.0, np.float32)))
    print("batches", dtype, b, m, n, k, shared, flush=True)
    hip.matmul(dst, sa, sw, (b, m, n, k), ((b, m, k), (0 if shared else m * (k + gap), k + gap, 1), 0), ((b, k, n), (k * n, n, 1), 0))
    assert ug_amd.last_kernel() == kernel
    got = dst.to_vec()
    got = (rng.from_bf16_bits(got) if dtype == "bf16" else got).astype(np.float64)
    assert np.all(got[b * m * n :] == 7.0), "wrote past the end"
    exact = np.matmul(a.astype(np.float64), w.astype(np.float64))
    bound = {"f32": 0, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype] * np.abs(exact) + (k + 1) * np.finfo(np.float32).eps * np.matmul(np.abs(a).astype(np.float64), np.abs(w).astype(np.float64))
    assert np.all(np.abs(got[: b * m * n].reshape(exact.shape) - exact) <= bound * 1.001 + 1e-7)


# tiles of 32, 64 and 128, whole and with K shared; K of one step and one element, of whole steps behind a remainder of 1, 63 and 64; slabs that begin behind K's first step
@pytest.mark.parametrize("b, m, n, k", [(1, 40, 33, 65), (3, 31, 70, 129), (1, 65, 67, 191), (1, 1000, 777, 320), (2, 900, 130, 447), (1, 2001, 2050, 193), (1, 39, 801, 2113), (1, 392, 113, 3457)])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("rhs_nk", [True, False], ids=["NT", "NN"])
def test_rows_that_start_inside_a_word(hip, b, m, n, k, dtype, rhs_nk):
    """16-bit rows at odd elements, all of them or every second one, have the bits of the same rows at whole words; behind and between them is not-a-number."""
    dt, enc = (ug_amd.F16, lambda v: v.astype(np.float16)) if dtype == "f16" else (ug_amd.BF16, rng.to_bf16_bits)
    a, w = rounded(dtype, rng.uniform_pm1(1, b * m * k)).reshape(b, m, k), rounded(dtype, rng.uniform_pm1(2, b * k * n)).reshape(b, k, n)
    lines = np.swapaxes(w, 1, 2) if rhs_nk else w

    def placed(x, pitch, offset):
        full = np.full(offset + x.shape[0] * x.shape[1] * pitch + 1, np.nan, np.float32)
        full[offset:-1].reshape(x.shape[0], x.shape[1], pitch)[:, :, : x.shape[2]] = x
        return hip.slice_from(enc(full)), pitch

    def product(odd_a, odd_w, offset):
        sa, pa = placed(a, k + 2 + (k + odd_a) % 2, offset)
        sw, pw = placed(lines, lines.shape[2] + 2 + (lines.shape[2] + odd_w) % 2, offset)
        dst = hip.allocate_uninit(dt, b * m * n)
        hip.matmul(dst, sa, sw, (b, m, n, k), ((b, m, k), (m * pa, pa, 1), offset), ((b, k, n), (lines.shape[1] * pw, 1, pw) if rhs_nk else (k * pw, pw, 1), offset))
        name = ug_amd.last_kernel()
        assert name.startswith("gemm_any<") and name.endswith(",words>") == bool(odd_a and odd_w or offset), name
        return dst.to_vec().view(np.uint16)

    print("inside a word", dtype, b, m, n, k, rhs_nk, flush=True)
    want = product(0, 0, 0)
    exact = np.matmul(a.astype(np.float64), w.astype(np.float64))
    got = rng.from_bf16_bits(want) if dtype == "bf16" else want.view(np.float16)
    bound = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype] * np.abs(exact) + (k + 1) * np.finfo(np.float32).eps * np.matmul(np.abs(a).astype(np.float64), np.abs(w).astype(np.float64))
    assert np.all(np.abs(got.astype(np.float64).reshape(exact.shape) - exact) <= bound * 1.001 + 1e-7)
    for odd_a, odd_w, offset in ((1, 1, 0), (1, 1, 1), (0, 0, 1), (1, 0, 1)):
        assert np.array_equal(product(odd_a, odd_w, offset), want), (odd_a, odd_w, offset)


# one group, a wave's 64 and one more, several rounds of them; groups without rows, ends in front of their predecessors' and behind the rows
@pytest.mark.parametrize("groups", [1, 2, 63, 64, 65, 128, 300])
@pytest.mark.parametrize("rows", [0, 3, 700])
def test_rows_by_group(hip, tune, groups, rows):
    """Which matrix a row meets, on every tile of rows: against the same product with each row's matrix looked up."""
    gpu, n, k, m = Gpu(hip), 24, 256, max(1, rows)
    gen = np.random.default_rng(groups + rows)
    x, w = rand(1, m, k), rand(2, groups, n, k, std=k ** -0.5)
    end = np.sort(gen.integers(0, rows + 1, groups)).astype(np.int32)
    end[-1] = rows
    said = end.copy()
    if groups > 2:
        said[1:-1:7] = -5              # an empty group, whatever is behind it
        end = np.maximum.accumulate(np.maximum(said, 0)).astype(np.int32)
    if rows == 700:
        said[-1] = rows + 1000
    src, of = gen.integers(0, m, m).astype(np.int32), np.searchsorted(end, np.arange(rows), side="right")
    y = np.stack([w[of[i]] @ x[src[i]] for i in range(rows)]) if rows else np.zeros((0, n))
    dx, dw, di, de = gpu.up(x, bf16=True), gpu.up(w, bf16=True), gpu.up(src), gpu.up(said)
    for shape in (None, "0", "3", *RING, "11"):
        if shape is not None:
            tune.setenv("UGHIP_GEMM_SHAPE", shape)
        dst = gpu.out(m * n + 8)
        print("rows by group", groups, rows, shape, flush=True)
        gpu.call("ughip_product_rows", C.byref(Product(x=view(dx, 0, k), dst=view(dst, 0, n), w=dw.raw(), m=m, n=n, k=k, product=BF16, act=NONE, row_index=di.raw(), group_end=de.raw(),
                                                       groups=groups, x_rows=m)))
        out = get(dst, m * n + 8)
        assert np.all(np.isnan(out[rows * n :])), "wrote what belongs to no group"
        if rows:
            close(out[: rows * n].reshape(rows, n), y, 2e-5)


# groups of every height's first and last size, of none, one and two tiles and more; the shortest K loops and an odd one; columns that hang over the tile
@pytest.mark.parametrize("n, k", [(96, 64), (200, 128), (264, 192), (136, 448)])
@pytest.mark.parametrize("act", [NONE, SWIGLU])
def test_tiles_as_high_as_their_groups(hip, tune, n, k, act):
    """Every k order is the other tiles': the same bits, gathered rows and bf16 results too."""
    sizes = [0, 1, 16, 17, 63, 64, 65, 0, 127, 128, 129, 191, 192, 193, 255, 256, 257, 300, 511, 512, 513, 770]
    gpu, m, rows = Gpu(hip), sum(sizes), n if act == NONE else 2 * n
    x, w = rand(1, m, k), rand(2, len(sizes), rows, k, std=k ** -0.5)
    dx, dw = gpu.up(x, bf16=True), gpu.up(w, bf16=True)
    src, end = gpu.up(np.random.default_rng(3).integers(0, m, m).astype(np.int32)), gpu.up(np.cumsum(sizes).astype(np.int32))
    got = {}
    for shape, tile in (("9", "64x64"), ("15", "256x192"), ("16", "256x128")):
        tune.setenv("UGHIP_GEMM_SHAPE", shape)
        dst = gpu.out(m * n + 8)
        print("as high as their groups", n, k, act, tile, flush=True)
        gpu.call("ughip_product_rows", C.byref(Product(x=view(dx, 0, k), dst=view(dst, 0, n), w=dw.raw(), m=m, n=n, k=k, product=BF16, act=act, row_index=src.raw(), group_end=end.raw(),
                                                       groups=len(sizes), x_rows=m)))
        assert f"{tile},512t,ring,rows" in ug_amd.last_kernel()
        got[tile] = get(dst, m * n + 8)
        assert np.all(np.isnan(got[tile][m * n :])) and np.all(np.isfinite(got[tile][: m * n]))
    np.testing.assert_array_equal(got["256x192"], got["64x64"])
    np.testing.assert_array_equal(got["256x128"], got["64x64"])


# (groups, rows of one in the mean, n, k, act): us on the tile named and on the one that prices fitted to 16 groups of two matrices took, or that took them before
@pytest.mark.parametrize("groups, per, n, k, act, tile", [(8, 1900, 8192, 4096, NONE, "256x256"),  # 820 .. 1016 / 1228 on 256 x 192
                                                          (4, 1000, 1408, 2048, SWIGLU, "256x256"),  # 53 / 78 on 256 x 192
                                                          (16, 260, 1408, 2048, SWIGLU, "192x192"),  # 72 / 57 .. 107 on 256 x 256, one round or two
                                                          (16, 127, 1408, 2048, SWIGLU, "256x192")])  # 59 / 84 on 192 x 192
def test_groups_take_the_tile_priced_lowest(hip, groups, per, n, k, act, tile):
    gpu, m, rows = Gpu(hip), groups * per, n if act == NONE else 2 * n
    dx, dw, dst = hip.allocate_uninit(ug_amd.BF16, m * k), hip.allocate_uninit(ug_amd.BF16, groups * rows * k), hip.allocate_uninit(ug_amd.BF16, m * n)
    src, end = gpu.up(np.arange(m, dtype=np.int32)), gpu.up(np.arange(1, groups + 1, dtype=np.int32) * per)
    gpu.call("ughip_product_rows", C.byref(Product(x=view(dx, 0, k), dst=view(dst, 0, n), w=dw.raw(), m=m, n=n, k=k, product=BF16, act=act, row_index=src.raw(), group_end=end.raw(), groups=groups, x_rows=m)))
    assert f"NT,{tile}," in ug_amd.last_kernel(), ug_amd.last_kernel()


@pytest.mark.parametrize("shape, kernel", [("3", "gemm_dma4<bf16,NT,256x256,256t,rows>"), ("4", "gemm_dma4<bf16,NT,256x128,512t,ring,rows>"), ("5", "gemm_dma4<bf16,NT,128x128,512t,ring,rows>"),
                                           ("0", "rows_product<bf16,none>"), ("6", "rows_product<bf16,none>"), ("7", "rows_product<bf16,none>")])
def test_forced_tiles_of_rows(hip, tune, shape, kernel):
    gpu, m, n, k = Gpu(hip), 70, 136, 320
    x, w = rand(1, m, k), rand(2, n, k, std=k ** -0.5)
    dx, dw, dst = gpu.up(x, bf16=True), gpu.up(w, bf16=True), gpu.out(m * n)
    tune.setenv("UGHIP_GEMM_SHAPE", shape)
    gpu.call("ughip_product_rows", C.byref(Product(x=view(dx, 0, k), dst=view(dst, 0, n), w=dw.raw(), m=m, n=n, k=k, product=BF16, act=NONE)))
    assert ug_amd.last_kernel() == kernel
    close(get(dst, (m, n)), x @ w.T, 2e-5)


def _random_products():
    gen = np.random.default_rng(17)
    out = [(1, 130, 136, 64, "bf16", True), (2, 65, 264, 128, "f16", False), (1, 300, 72, 192, "bf16", False), (1, 257, 392, 64, "f16", False), (3, 9, 8, 128, "bf16", False), (1, 64, 64, 192, "f16", True)]
    for _ in range(18):
        b, m, n, kt = int(gen.integers(1, 4)), int(gen.integers(9, 600)), 8 * int(gen.integers(1, 60)), int(gen.integers(1, 12))
        out.append((b, m, n, 64 * kt, ("bf16", "f16")[int(gen.integers(2))], bool(gen.integers(2))))
    return out


# one to three K tiles, where only the tail of the loop runs, in both layouts and types, and sizes as they come
@pytest.mark.parametrize("b, m, n, k, dtype, rhs_nk", _random_products())
def test_ring_tiles_give_the_other_kernels_bits(hip, tune, b, m, n, k, dtype, rhs_nk):
    """Every tile of the ring sums in the order of the register-staged kernel (without a K split): the same bits, on values that any other order would
    round otherwise."""
    dt = ug_amd.BF16 if dtype == "bf16" else ug_amd.F16
    a, w = rounded(dtype, rng.normal(1, b * m * k)).reshape(b, m, k), rounded(dtype, rng.normal(2, b * k * n)).reshape(b, k, n)
    tune.setenv("UGHIP_GEMM_SPLIT", "1")
    ref = None
    if rhs_nk or n % 128 == 0:  # (whole column tiles for a [k, n]-major rhs)
        tune.setenv("UGHIP_GEMM_SHAPE", "1")
        ref = _raw_matmul(hip, dt, a, w, rhs_nk)
        assert ug_amd.last_kernel().startswith("gemm_tiled<")
    elif k >= 256:
        tune.setenv("UGHIP_GEMM_SHAPE", "5")
        ref = _raw_matmul(hip, dt, a, w, rhs_nk)
        assert ug_amd.last_kernel().startswith("gemm_dma4<") and "ring" not in ug_amd.last_kernel()
    exact = np.matmul(a.astype(np.float64), w.astype(np.float64))
    bound = (2.0 ** -8 if dtype == "bf16" else 2.0 ** -11) * np.abs(exact) + k * np.finfo(np.float32).eps * np.matmul(np.abs(a).astype(np.float64), np.abs(w).astype(np.float64))
    for shape, tile in RING.items():
        if shape == "9" and not rhs_nk:
            continue
        tune.setenv("UGHIP_GEMM_SHAPE", shape)
        print("ring bits", dtype, b, m, n, k, "NT" if rhs_nk else "NN", tile, flush=True)
        got = _raw_matmul(hip, dt, a, w, rhs_nk)
        assert ug_amd.last_kernel() == f"gemm_dma4<{dtype},{'NT' if rhs_nk else 'NN'},{tile},512t,ring>"
        assert np.all(np.abs(got - exact) <= bound * 1.001 + 1e-7)
        if ref is None:
            ref = got  # (neither of the others takes it: the tiles among themselves)
        np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("m, n, k", [(1, 8, 64), (70, 136, 320), (193, 72, 192), (300, 264, 128)])
@pytest.mark.parametrize("table_bf16", [True, False])
@pytest.mark.parametrize("out_bf16", [True, False])
def test_ring_rows_times_a_lookup(hip, tune, m, n, k, table_bf16, out_bf16):
    """gelu(y) times an element of a table row, on every tile that has the form: tables and results of either type, ids outside the table."""
    gpu, rows, col = Gpu(hip), 13, 4
    x, w, bias, table = rand(1, m, k), rand(2, n, k, std=k ** -0.5), rand(3, n, std=0.5), rand(4, rows, n + 6)
    ids = (np.arange(m) * 5 % rows).astype(np.int32)
    ids[m // 2], ids[m - 1] = (-1, rows) if m > 1 else (rows, rows)
    y = x @ w.T + bias
    inside = (ids >= 0) & (ids < rows)
    want = 0.5 * y * (1 + np.tanh(np.sqrt(2 / np.pi) * (y + 0.044715 * y ** 3))) * table[np.where(inside, ids, 0)][:, col : col + n]
    dx, dw, db, dt, di = gpu.up(x, bf16=True), gpu.up(w, bf16=True), gpu.up(bias), gpu.up(table, bf16=table_bf16), gpu.up(ids)
    for shape in (None, "10", "12", "13", "9"):
        if shape:
            tune.setenv("UGHIP_GEMM_SHAPE", shape)
        dst = gpu.out(m * n + 8, bf16=out_bf16)
        print("lookup rows", m, n, k, table_bf16, out_bf16, shape, flush=True)
        gpu.call("ughip_product_rows", C.byref(Product(x=view(dx, 0, k), dst=view(dst, 0, n), w=dw.raw(), bias=db.raw(), m=m, n=n, k=k, product=BF16, act=GELU_MUL, table=dt.raw(), ids=di.raw(),
                                                       table_rows=rows, table_stride=n + 6, table_col=col)))
        assert ",512t,ring,rows,lookup>" in ug_amd.last_kernel() and (shape is None or RING[shape] in ug_amd.last_kernel())
        out = get(dst, m * n + 8)
        assert np.all(np.isnan(out[m * n :])), "wrote past the end"
        out = out[: m * n].reshape(m, n)
        assert np.all(np.isnan(out[~inside]))
        if inside.any():
            close(out[inside], want[inside], 2e-5, rel=2.0 ** -8 if out_bf16 else 0.0)


@pytest.mark.parametrize("k", [512, 516, 2048, 9000])
@pytest.mark.parametrize("n", [1, 77, 2000])
@pytest.mark.parametrize("w_bf16, mode", [(True, BF16), (False, BF16), (False, F32)])
def test_one_row_keeps_its_f32_values(hip, n, k, w_bf16, mode):
    """One dense f32 row goes to the decode kernels: neither it nor an F32 matrix is rounded to bf16, whatever the product is called."""
    gpu, eps = Gpu(hip), np.finfo(np.float32).eps
    x, w = rng.normal(1, k).astype(np.float64), (rand(2, n, k, std=k ** -0.5) if w_bf16 else rng.normal(2, n * k, k ** -0.5).reshape(n, k).astype(np.float64))
    dx, dw, dst = gpu.up(np.concatenate([x, np.full(8, np.nan)])), gpu.up(w, bf16=w_bf16), gpu.out(n + 8)
    gpu.call("ughip_product_rows", C.byref(Product(x=view(dx, 0, k + 8), dst=view(dst, 0, n), w=dw.raw(), m=1, n=n, k=k, product=mode, act=NONE)))
    assert ug_amd.last_kernel() == f"rows_product<{'f32' if mode == F32 else 'bf16'},one row>"
    out = get(dst, n + 8)
    assert np.all(np.isnan(out[n:])), "wrote past the end"
    assert np.all(np.abs(out[:n] - w @ x) <= k * eps * (np.abs(w) @ np.abs(x)))


@pytest.mark.parametrize("k, bias, offset", [(256, False, 0), (511, False, 0), (512, True, 0), (512, False, 4)])
def test_one_row_elsewhere_is_rounded(hip, k, bias, offset):
    """A row with a bias, at an offset, or short: rounded to bf16 in front of the product, as several rows are."""
    gpu, n = Gpu(hip), 40
    x, w, b = rng.normal(1, k), rand(2, n, k, std=k ** -0.5), rand(3, n)
    want = w @ rng.bf16_round(x).astype(np.float64) + (b if bias else 0)
    dx, dw, db, dst = gpu.up(np.concatenate([np.zeros(offset), x])), gpu.up(w, bf16=True), gpu.up(b), gpu.out(n)
    gpu.call("ughip_product_rows", C.byref(Product(x=view(dx, offset, k), dst=view(dst, 0, n), w=dw.raw(), bias=db.raw() if bias else None, m=1, n=n, k=k, product=BF16, act=NONE)))
    assert "one row" not in ug_amd.last_kernel()
    close(get(dst, n), want, 2e-5)


# 32 x 32 tiles: one to nine K tiles (the ring has eight stages) and more, rows and columns that hang over, rows by group, a lookup behind, bf16 results
@pytest.mark.parametrize("m, n, k", [(1, 8, 64), (33, 40, 128), (31, 72, 192), (65, 136, 448), (40, 24, 512), (32, 32, 576), (70, 264, 640), (100, 96, 1088)])
@pytest.mark.parametrize("form", ["plain", "groups", "lookup", "bf16"])
def test_smallest_ring_tile_gives_the_next_ones_bits(hip, tune, m, n, k, form):
    gpu, gen = Gpu(hip), np.random.default_rng(7)
    mats = 3 if form == "groups" else 1
    dx, dw = gpu.up(rand(1, m, k), bf16=True), gpu.up(rand(2, mats, n, k, std=k ** -0.5), bf16=True)
    keep, kw = [dx, dw, gpu.up(rand(3, n))], {}
    if form == "plain":
        kw = dict(bias=keep[2].raw())
    if form == "groups":
        keep += [gpu.up(gen.integers(0, m, m).astype(np.int32)), gpu.up(np.array([m // 3, m // 3, m], np.int32))]
        kw = dict(row_index=keep[3].raw(), group_end=keep[4].raw(), groups=3, x_rows=m)
    if form == "lookup":
        keep += [gpu.up(rand(4, 50, n + 3)), gpu.up(gen.integers(0, 50, m).astype(np.int32))]
        kw = dict(table=keep[3].raw(), ids=keep[4].raw(), table_rows=50, table_stride=n + 3, table_col=2)
    got = {}
    for shape, tile in (("9", "64x64,512t"), ("17", "32x32,256t")):
        tune.setenv("UGHIP_GEMM_SHAPE", shape)
        dst = gpu.out(m * n + 8, bf16=form == "bf16")
        print("smallest ring tile", m, n, k, form, tile, flush=True)
        gpu.call("ughip_product_rows", C.byref(Product(x=view(dx, 0, k), dst=view(dst, 0, n), w=dw.raw(), m=m, n=n, k=k, product=BF16, act=GELU_MUL if form == "lookup" else NONE, **kw)))
        assert f"{tile},ring,rows" in ug_amd.last_kernel()
        got[tile] = get(dst, m * n + 8)
        assert np.all(np.isnan(got[tile][m * n :])) and np.all(np.isfinite(got[tile][: m * n]))
    np.testing.assert_array_equal(got["64x64,512t"], got["32x32,256t"])


@pytest.mark.parametrize("m, n, k", [(300, 264, 128), (257, 128, 64), (17, 392, 192)])
@pytest.mark.parametrize("half", [False, True])
def test_lookups_on_every_tile_of_the_ring(hip, tune, m, n, k, half):
    """gelu(y) times the token's row of an f32 or a bf16 table, ids outside of it among them: the same bits on every tile, values against 64 bits."""
    gpu, gen = Gpu(hip), np.random.default_rng(9)
    x, w, bias, table, ids = rand(1, m, k), rand(2, n, k, std=k ** -0.5), rand(3, n), rand(4, 50, n + 3), gen.integers(0, 50, m)
    ids[::7] = 50
    ids[3::11] = -1
    keep = [gpu.up(x, bf16=True), gpu.up(w, bf16=True), gpu.up(bias), gpu.up(table, bf16=half), gpu.up(ids.astype(np.int32))]
    got = {}
    for shape, tile in (("10", "256x128"), ("12", "128x128"), ("13", "64x128"), ("9", "64x64"), ("17", "32x32")):
        tune.setenv("UGHIP_GEMM_SHAPE", shape)
        dst = gpu.out(m * n + 8)
        print("lookup", m, n, k, half, tile, flush=True)
        gpu.call("ughip_product_rows", C.byref(Product(x=view(keep[0], 0, k), dst=view(dst, 0, n), w=keep[1].raw(), bias=keep[2].raw(), m=m, n=n, k=k, product=BF16, act=GELU_MUL, table=keep[3].raw(),
                                                       ids=keep[4].raw(), table_rows=50, table_stride=n + 3, table_col=2)))
        assert f"NT,{tile}," in ug_amd.last_kernel() and "ring,rows" in ug_amd.last_kernel()
        out = get(dst, m * n + 8)
        assert np.all(np.isnan(out[m * n :]))
        got[tile] = out[: m * n].reshape(m, n)
    known = (ids >= 0) & (ids < 50)
    y = x @ w.T + bias
    want = 0.5 * y * (1 + np.tanh(np.sqrt(2 / np.pi) * (y + 0.044715 * y ** 3))) * table[np.where(known, ids, 0), 2 : 2 + n]
    for out in got.values():
        np.testing.assert_array_equal(out, got["64x64"])
    assert np.all(np.isnan(got["64x64"][~known]))
    close(got["64x64"][known], want[known], 2e-5)


# f32 rows on 128 x 128, 64 x 128 and 64 x 64 tiles as the rounds of 256 have it, a few tiles and one past a round too; K of a step less and a step more, gated and plain, even and uneven groups
@pytest.mark.parametrize("m, n, k, groups, act, tile", [
    (70, 2050, 33, 0, SWIGLU, "64x128"), (129, 1040, 64, 0, SWIGLU, "64x128"), (300, 5632, 40, 0, SWIGLU, "64x128"), (513, 6592, 36, 0, NONE, "64x128"), (700, 6592, 31, 0, NONE, "64x64"),
    (1531, 2048, 24, 0, NONE, "128x128"), (150, 300, 20, 0, NONE, "64x64"), (1200, 1408, 28, 16, SWIGLU, "64x128"), (1200, 2048, 28, 16, NONE, "64x128"), (2036, 264, 20, 5, SWIGLU, "64x128"),
    (128, 256, 72, 0, NONE, "64x64"), (256, 16, 65, 0, NONE, "64x64"), (100, 128, 40, 0, SWIGLU, "64x128"), (5504, 768, 20, 0, NONE, "64x128"), (2048, 2048, 20, 0, NONE, "128x128")])
def test_f32_rows_of_every_tile(hip, m, n, k, groups, act, tile):
    gpu, rows, mats = Gpu(hip), n if act == NONE else 2 * n, max(1, groups)
    gen = np.random.default_rng(6)
    x, w = gen.standard_normal((m, k)).astype(np.float32), (gen.standard_normal((mats, rows, k)) / np.sqrt(k)).astype(np.float32)
    kw, of = {}, np.zeros(m, int)
    if groups:
        end = np.sort(gen.integers(0, m + 1, groups)).astype(np.int32)
        end[-1] = m
        of = np.searchsorted(end, np.arange(m), side="right")
        keep = gpu.up(np.arange(m, dtype=np.int32)), gpu.up(end)
        kw = dict(row_index=keep[0].raw(), group_end=keep[1].raw(), groups=groups, x_rows=m)
    y = np.concatenate([x[of == g].astype(np.float64) @ w[g].T.astype(np.float64) for g in range(mats)])
    if act == SWIGLU:
        y = y[:, :n] / (1 + np.exp(-y[:, :n])) * y[:, n:]
    dx, dw, dst = gpu.up(x), gpu.up(w), gpu.out(m * n + 8)
    print("f32 rows", m, n, k, groups, act, flush=True)
    gpu.call("ughip_product_rows", C.byref(Product(x=view(dx, 0, k), dst=view(dst, 0, n), w=dw.raw(), m=m, n=n, k=k, product=F32, act=act, **kw)))
    assert ug_amd.last_kernel() == f"rows_product<f32,{'swiglu' if act == SWIGLU else 'none'}{',grouped' if groups else ''},{tile}>"
    out = get(dst, m * n + 8)
    assert np.all(np.isnan(out[m * n :])), "wrote past the end"
    close(out[: m * n].reshape(m, n), y, 1e-5)  # k eps and the gate's few units, against sums of some standard deviations


# rows a little further apart than they are long, behind others; gathered and by group (with rows that nobody asks for)
@pytest.mark.parametrize("m, n, k, groups, act", [(*size, 0, act) for size in [(1, 8, 640), (16, 264, 512), (33, 136, 384), (70, 520, 320)] for act in (SWIGLU, GLU, GELU_MUL)] +
                         [(40, 136, 576, 3, act) for act in (SWIGLU, GLU)] + [(40, 136, 832, 3, NONE), (40, 136, 64, 70, NONE), (140, 136, 1024, 0, NONE), (33, 8, 768, 0, NONE)])
def test_f32_rows_of_a_bf16_product_have_the_bits_of_rounded_ones(hip, m, n, k, groups, act):
    gpu, rows, mats, rx = Gpu(hip), 2 * n if act in (SWIGLU, GLU) else n, max(1, groups), m + 3
    gen = np.random.default_rng(8)
    x = gen.standard_normal((rx, k + 8)).astype(np.float32)
    dx, db = gpu.up(np.concatenate([np.full(4, np.nan, np.float32), x.ravel()])), gpu.up(np.concatenate([np.full(8, np.nan, np.float32), x.ravel()]), bf16=True)
    dw, dt, di = gpu.up(rand(2, mats, rows, k, std=k ** -0.5), bf16=True), gpu.up(rand(3, 50, n)), gpu.up(gen.integers(-1, 51, m).astype(np.int32))
    kw = {}
    if groups:
        idx, end = gpu.up(gen.integers(0, rx, m).astype(np.int32)), gpu.up(np.array([0, m // 3] + [m] * (groups - 2), np.int32))
        kw = dict(row_index=idx.raw(), group_end=end.raw(), groups=groups, x_rows=rx)
    if act == GELU_MUL:
        kw = dict(table=dt.raw(), ids=di.raw(), table_rows=50, table_stride=n)
    got = []
    for rows_of, offset in ((dx, 4), (db, 8)):
        dst = gpu.out(m * n + 8)
        print("rounded rows", m, n, k, groups, act, flush=True)
        gpu.call("ughip_product_rows", C.byref(Product(x=view(rows_of, offset, k + 8), dst=view(dst, 0, n), w=dw.raw(), m=m, n=n, k=k, product=BF16, act=act, act_alpha=1.702 if act == GLU else 0,
                                                       act_shift=1.0 if act == GLU else 0, act_limit=1.5 if act == GLU else 0, **kw)))
        assert ug_amd.last_kernel().startswith("gemm_dma4<bf16,NT,"), ug_amd.last_kernel()
        got.append(get(dst, m * n + 8))
    np.testing.assert_array_equal(got[0], got[1])
    assert np.all(np.isnan(got[0][m * n :])) and np.any(np.isfinite(got[0][: m * n]))


# tiles of bf16 rows and, K no multiple of 64, the kernel of any size; many more rows than are asked for, of which one that nobody asks for is not-a-number
@pytest.mark.parametrize("k", [1024, 2048, 1020])
@pytest.mark.parametrize("act", [NONE, SWIGLU])
@pytest.mark.parametrize("bf16_rows", [False, True], ids=["f32", "bf16"])
def test_rows_by_group_that_name_no_row(hip, k, act, bf16_rows):
    """F32 rows: zeros.  BF16 rows: the others are what they are, and so is what lies behind them."""
    gpu, m, n, rx, groups = Gpu(hip), 70, 136, 5000, 3
    rows = 2 * n if act else n
    gen = np.random.default_rng(5)
    idx = gen.integers(0, rx - 1, m).astype(np.int32)
    idx[[0, 7, 30, 69]] = -1, rx, 0x7fffffff, -0x80000000
    x = gen.standard_normal((rx, k)).astype(np.float32)
    x[rx - 1] = np.nan
    x[0] = np.nan  # (what an index below would be taken for)
    idx[idx == 0] = 1
    w = rand(2, groups, rows, k, std=k ** -0.5)
    dx, dw, di, de, dst = gpu.up(x, bf16=bf16_rows), gpu.up(w, bf16=True), gpu.up(idx), gpu.up(np.array([20, 21, m], np.int32)), gpu.out(m * n + 8)
    print("rows that are none", k, act, bf16_rows, flush=True)
    gpu.call("ughip_product_rows", C.byref(Product(x=view(dx, 0, k), dst=view(dst, 0, n), w=dw.raw(), m=m, n=n, k=k, product=BF16, act=act, row_index=di.raw(), group_end=de.raw(), groups=groups,
                                                   x_rows=rx)))
    assert ug_amd.last_kernel().startswith("rows_product<" if k % 64 else "gemm_dma4<bf16,NT,"), ug_amd.last_kernel()
    got, there = get(dst, m * n + 8), (idx >= 0) & (idx < rx)
    assert np.all(np.isnan(got[m * n :]))
    got = got[: m * n].reshape(m, n)
    assert bf16_rows or np.all(got[~there] == 0)
    y = np.stack([rng.bf16_round(x[idx[r] if there[r] else 1]).astype(np.float64) @ w[0 if r < 20 else 1 if r < 21 else 2].T for r in range(m)])
    if act:
        y = y[:, :n] / (1 + np.exp(-y[:, :n])) * y[:, n:]
    close(got[there], y[there], 2e-5)


# K shared and whole, 32-, 64- and 128-row tiles and rows and columns that hang over them; bias, gates and lookups in the fold, results between other rows' elements
@pytest.mark.parametrize("m, n, k", [(2, 8, 512), (17, 1032, 2048), (33, 136, 1056), (70, 520, 1024), (130, 264, 2048), (200, 1032, 2048)])
@pytest.mark.parametrize("act, bias, gap", [(NONE, False, 0), (NONE, True, 0), (NONE, False, 3), (SWIGLU, True, 0), (GLU, False, 5), (GELU_MUL, False, 0), (GELU_MUL, True, 1)])
def test_f32_rows_that_share_their_k(hip, m, n, k, act, bias, gap):
    gpu, rows = Gpu(hip), 2 * n if act in (SWIGLU, GLU) else n
    gen = np.random.default_rng(8)
    x, w, b = gen.standard_normal((m, k), np.float32), (gen.standard_normal((rows, k)) / np.sqrt(k)).astype(np.float32), gen.standard_normal(rows).astype(np.float32)
    table, ids = gen.standard_normal((50, n + 6)).astype(np.float32), gen.integers(-1, 51, m).astype(np.int32)
    y = x.astype(np.float64) @ w.T.astype(np.float64) + (b if bias else 0)
    if act in (SWIGLU, GLU):
        limit, alpha, shift = (1.5, 1.702, 1.0) if act == GLU else (1e9, 1.0, 0.0)
        g, u = np.minimum(y[:, :n], limit), np.clip(y[:, n:], -limit, limit)
        y = g / (1 + np.exp(-alpha * g)) * (u + shift)
    known = (ids >= 0) & (ids < 50)
    if act == GELU_MUL:
        y = 0.5 * y * (1 + np.tanh(np.sqrt(2 / np.pi) * (y + 0.044715 * y ** 3))) * table[np.where(known, ids, 0), 2 : 2 + n]
    else:
        known |= True
    dx, dw, db, dt, di, dst = gpu.up(x), gpu.up(w), gpu.up(b), gpu.up(table), gpu.up(ids), gpu.out(m * (n + gap) + 8)
    print("f32 rows, K shared", m, n, k, act, bias, gap, flush=True)
    kw = dict(table=dt.raw(), ids=di.raw(), table_rows=50, table_stride=n + 6, table_col=2) if act == GELU_MUL else {}
    gpu.call("ughip_product_rows", C.byref(Product(x=view(dx, 0, k), dst=view(dst, 0, n + gap), w=dw.raw(), bias=db.raw() if bias else None, m=m, n=n, k=k, product=F32, act=act,
                                                   act_alpha=1.702 if act == GLU else 0, act_shift=1.0 if act == GLU else 0, act_limit=1.5 if act == GLU else 0, **kw)))
    assert ug_amd.last_kernel().startswith("gemm_tiled<f32,NT,"), ug_amd.last_kernel()
    out = get(dst, m * (n + gap) + 8)
    assert np.all(np.isnan(out[m * (n + gap) :]))
    out = out[: m * (n + gap)].reshape(m, n + gap)
    assert np.all(np.isnan(out[:, n:])) and np.all(np.isnan(out[~known, :n]))
    # sums of 2048 are off by 8e-7 of their spread in the mean square, five times that at most here; in a gated unit times the other factor, of up to 4.5
    close(out[known, :n], y[known], 5 * 8e-7 * 4.5 if act != NONE else 1e-5)


# sums of 131 MB and of 137; rows rounded to 128 MiB and to a row more
@pytest.mark.parametrize("m, n, k, kind, kernel", [(5000, 6592, 1024, F32, "gemm_tiled<f32,NT,"), (5200, 6592, 1024, F32, "rows_product<f32,"), (16384, 1024, 4096, BF16, "gemm_dma4<bf16,NT,"),
                                                   (16385, 1024, 4096, BF16, "rows_product<bf16,")])
def test_rows_take_a_share_of_the_devices_block_at_most(hip, m, n, k, kind, kernel):
    gpu = Gpu(hip)
    x, w, b = rng.normal(1, m * k, 1.0).reshape(m, k), rand(2, n, k, std=k ** -0.5), rand(3, n)
    dx, dw, db, dst = gpu.up(x), gpu.up(w, bf16=kind == BF16), gpu.up(b), gpu.out(m * n)
    print("the block's share", m, n, k, flush=True)
    gpu.call("ughip_product_rows", C.byref(Product(x=view(dx, 0, k), dst=view(dst, 0, n), w=dw.raw(), bias=db.raw(), m=m, n=n, k=k, product=kind, act=NONE)))
    assert ug_amd.last_kernel().startswith(kernel), ug_amd.last_kernel()
    some = [0, 1, 255, m // 2, m - 130, m - 1]
    rows = rng.bf16_round(x[some]) if kind == BF16 else x[some]
    close(get(dst, (m, n))[some], rows.astype(np.float64) @ w.T + b, 1e-5)


def test_f32_rows_of_more_tile_rows_than_a_grid_has(hip):
    """64-row tiles would be more than the 65535 that a grid's second dimension takes."""
    gpu, m, n, k = Gpu(hip), 65535 * 64 + 1, 8, 8
    gen = np.random.default_rng(3)
    x, w = gen.standard_normal((m, k), np.float32), gen.standard_normal((n, k), np.float32)
    dx, dw, dst = gpu.up(x), gpu.up(w), hip.allocate_uninit(ug_amd.F32, m * n)
    gpu.call("ughip_product_rows", C.byref(Product(x=view(dx, 0, k), dst=view(dst, 0, n), w=dw.raw(), m=m, n=n, k=k, product=F32, act=NONE)))
    np.testing.assert_allclose(dst.to_vec().reshape(m, n), x @ w.T, rtol=0, atol=2e-5)  # 8 products of normal deviates in f32 on either side


# Rows leave in 16-byte pieces through LDS where a bf16 row starts on one, else fragment by fragment: the same bits either way, edges of tiles and of pieces, nothing behind a row touched.
# (17, 32 x 32 tiles: plain rows alone)
@pytest.mark.parametrize("shape, m, n, act", [(shape, *size) for size in [(300, 200, NONE), (257, 392, NONE), (16, 520, NONE), (271, 136, SWIGLU), (97, 200, SWIGLU)]
                                              for shape in ["3", "10", "11", "12", "13", "9"] + ["17"] * (size[2] == NONE)])
def test_rows_leave_in_pieces_with_the_same_bits(hip, tune, shape, m, n, act):
    gpu, k, rows = Gpu(hip), 512, 2 * n if act == SWIGLU else n
    dx, dw, bias = gpu.up(rand(1, m, k), bf16=True), gpu.up(rand(2, rows, k, std=k ** -0.5), bf16=True), gpu.up(rand(3, rows))
    tune.setenv("UGHIP_GEMM_SHAPE", shape)
    got = {}
    for bf16, gap in ((True, 8), (True, 4), (False, 8)):
        print("rows out", shape, m, n, act, bf16, gap, flush=True)
        dst = gpu.out(m * (n + gap), bf16=bf16)
        gpu.call("ughip_product_rows", C.byref(Product(x=view(dx, 0, k), dst=view(dst, 0, n + gap), w=dw.raw(), bias=bias.raw(), m=m, n=n, k=k, product=BF16, act=act)))
        assert "rows" in ug_amd.last_kernel() and "gemm_dma4" in ug_amd.last_kernel()
        out = get(dst, m * (n + gap)).reshape(m, n + gap)
        assert np.all(np.isnan(out[:, n:])) and np.all(np.isfinite(out[:, :n]))
        got[bf16, gap] = out[:, :n]
    np.testing.assert_array_equal(got[True, 8], got[True, 4])
    np.testing.assert_array_equal(got[True, 8], rng.bf16_round(got[False, 8].ravel()).reshape(m, n))
