"""Three bf16 terms on the 256 x 192 tile of the one-wave-per-SIMD kernel, at the edges of the tile and over splits of K."""
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
