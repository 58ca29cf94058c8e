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
