"""Three bf16 terms on the 256 x 192 tile of the one-wave-per-SIMD kernel, at the edges of the tile and over splits of K."""
import ctypes as C

import numpy as np
import pytest

import test_gpu_parity as parity
import ug_amd

pytestmark = pytest.mark.gpu


# rows and columns one tile and a bit, one short, exactly; the shortest K the tile takes, odd numbers of K tiles, a few columns (the bounds are the oracle test's: k eps against float64)
@pytest.mark.parametrize("t,k,n,split", [(513, 128, 200, None), (511, 192, 184, None), (512, 128, 192, None), (512, 256, 96, "2"), (400, 512, 392, "4"), (390, 448, 8, None)])
def test_wide_tile(hip, tune, t, k, n, split):
    parity.test_three_bf16_terms_on_the_one_wave_per_simd_kernel(hip, tune, t, k, n, "14", split)
    assert "256x192" in ug_amd.last_kernel()


# gate and up columns of a tile gated in registers: 96 columns one short, exact and a bit; as planes, bit for bit what the f32 rows give
@pytest.mark.parametrize("t,k,inter,n", [(513, 128, 192, 64), (511, 192, 64, 72), (512, 128, 128, 64), (400, 256, 1088, 136), (385, 128, 320, 64), (449, 448, 448, 64)])
def test_wide_tile_gated(hip, tune, monkeypatch, t, k, inter, n):
    names, last = [], ug_amd.last_kernel
    monkeypatch.setattr(ug_amd, "last_kernel", lambda: names.append(last()) or names[-1])
    tune.setenv("UGHIP_X3_DMA", "14")
    tune.setenv("UGHIP_X3_SPLIT", "1")
    parity.test_norm_and_mlp_folded_into_the_products_of_rows(hip, t, k, inter, n, 1, True)
    tile = "gemm_dma4<bf16,NT,256x192,256t,3 planes,f32 out,in-register swiglu fold"
    assert tile + ">" in names and any(tile + " onto planes> -> " in name for name in names), names


@pytest.mark.parametrize("inter", [96, 200])
def test_gates_of_every_size(hip, tune, inter):
    """Gates of one row each, up values of one: what leaves is silu alone.  No further from 64 bits than the fold of slabs has it (expf and a division) on another tile; gates that overflow the
    sums, and none, among the others."""
    gen = np.random.default_rng(4)
    g = np.concatenate([gen.standard_normal(2000), gen.uniform(-88.7, 88.7, 2000), gen.uniform(-88.72, -87.2, 300), [0.0, -0.0, 20, -20, -87, -88.5, 100, -100, -104, 1e-30, -1e-30, 1e30, -1e30]]).astype(np.float32)
    many, k = len(g), 128
    x = np.zeros((many + 3, k), np.float32)
    x[:many, 0], x[:, 1] = g, 1
    x[many, 2], x[many + 1, 2], x[many + 2, 0] = 2.0 ** 127, -(2.0 ** 127), np.nan  # times 2^20: infinities
    w = np.zeros((2 * inter, k), np.float32)
    w[:inter, 0], w[:inter, 2], w[inter:, 1] = 1, 2.0 ** 20, 1
    dx, dw = hip.slice_from(x.ravel()), hip.slice_from(ug_amd.rng.to_bf16_bits(w.ravel()))
    lib, raw, z = ug_amd.ughip_lib(), lambda s: C.c_void_p(s.raw()), C.c_size_t
    got = {}
    for shape, name in (("14", "256x192,256t,3 planes,f32 out,in-register swiglu"), ("3", "256x256,256t,3 planes,f32 out,swiglu fold")):
        tune.setenv("UGHIP_X3_DMA", shape)
        tune.setenv("UGHIP_X3_SPLIT", "1")
        dst = hip.slice_from(np.full((many + 3) * inter, 7, np.float32))
        assert lib.ughip_linear_swiglu_rows(C.c_void_p(hip.raw_hip()), raw(dx), raw(dw), raw(dst), z(many + 3), z(inter), z(k), C.c_int(1)) == 0, lib.ughip_last_error()
        assert name in ug_amd.last_kernel(), ug_amd.last_kernel()
        y = dst.to_vec().reshape(many + 3, inter)
        assert np.all((y == y[:, :1]) | np.isnan(y) & np.isnan(y[:, :1]))
        got[shape] = y[:, 0]
        assert y[many, 0] == np.inf and np.isnan(y[many + 1, 0]) and np.isnan(y[many + 2, 0])  # -inf / (1 + inf) is none in f32 either
    g64 = g.astype(np.float64)
    with np.errstate(over="ignore"):
        want = g64 / (1 + np.exp(-g64))
    whole = g > -88.72  # 1 + exp(-z) is finite in f32
    assert np.all(np.abs(got["14"][:many][~whole]) <= 2.7e-37)
    unit = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(want[whole]), 2.0 ** -126))) - 23)
    units = {s: np.abs(v[:many].astype(np.float64) - want)[whole] / unit for s, v in got.items()}
    print("units of the last place, in registers / fold: most %.2f / %.2f, rms %.3f / %.3f" % tuple(f(units[s]) for f in (np.max, lambda u: np.sqrt(np.mean(u * u))) for s in ("14", "3")), flush=True)
    # exp2, its product's rounding, the sum's, the quotient's: one unit and three halves, each up to twice that where the next binade begins
    assert np.max(units["14"]) <= 5
    assert np.sqrt(np.mean(units["14"] ** 2)) <= 1.02 * np.sqrt(np.mean(units["3"] ** 2))


# up to 64 rows the split inside the product has tiles of 64: rows one tile, one short and the fewest, columns that hang over, fewer units than the ring has stages, as many and more, runs that begin
# and end anywhere in a column tile and a last one that hangs over behind a whole one
@pytest.mark.parametrize("t,k,n,units", [(64, 64, 8, None), (63, 320, 392, "7"), (64, 384, 136, "6"), (33, 448, 264, "5"), (64, 1024, 640, "16"), (50, 2048, 11264, None), (64, 5632, 1000, None), (40, 640, 2056, "11")])
def test_split_inside_the_product_on_64_rows(hip, tune, t, k, n, units):
    parity.test_three_bf16_terms_split_inside_the_product(hip, tune, t, k, n, units)
