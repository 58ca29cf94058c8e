"""Products of any size whose K several workgroups share, and the rules for the larger tile: what each plan leaves, against the bound of an f32 sum."""
import numpy as np
import pytest

import test_gpu_products as products
import test_zz_no_alloc as no_alloc
import ug_amd

pytestmark = pytest.mark.gpu


# sums that are split in 32 bits, the shorter ones on 32 x 32 tiles without a split in 16: a whole last step and one element of one, uneven slabs, a tile over the edge, slabs of 1, 2 and 3 elements behind the last four,
# as many slabs as there may be, tiles times slabs on either side of a round of the chip; a product in a batch
@pytest.mark.parametrize("bmnk", [(1, 9, 9, 1600), (1, 9, 9, 1601), (1, 65, 67, 1407), (1, 21, 11, 4096), (1, 63, 65, 3000), (3, 70, 9, 2050), (1, 150, 500, 4001), (1, 500, 1001, 2001)])
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("rhs_nk", [True, False], ids=["NT", "NN"])
@pytest.mark.parametrize("lhs_mk", [True, False], ids=["rows", "transposed"])
def test_split_sums(hip, bmnk, dtype, rhs_nk, lhs_mk):
    products.test_products_of_any_size(hip, bmnk, dtype, rhs_nk, lhs_mk)
    if dtype == "f32" and bmnk[1] < 100 and bmnk[3] % 64:
        assert ",splitK=" in ug_amd.last_kernel(), ug_amd.last_kernel()


# 16 bits, fewer than 256 large tiles: four small ones and three to a CU, on both sides of the sums that pay for the large one
@pytest.mark.parametrize("bmnk, large", [((1, 1729, 1729, 257), True), ((1, 1729, 1729, 255), False), ((1, 1601, 1601, 1537), True), ((1, 1601, 1601, 1535), False)])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_three_and_four_tiles_to_a_cu(hip, bmnk, large, dtype):
    products.test_products_of_any_size(hip, bmnk, dtype, True, True)
    assert ug_amd.last_kernel() == f"gemm_any<{dtype}{',128x128' if large else ''},words>"


@pytest.mark.parametrize("dtype", [ug_amd.F32, ug_amd.BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("bmnk", [(1, 70, 65, 6001), (2, 33, 9, 5999)])
def test_the_call_that_may_not_allocate(hip, dtype, bmnk):
    ref, got, kernel = no_alloc._both(hip, dtype, bmnk, True, 91)
    assert ",splitK=" in kernel
    np.testing.assert_array_equal(got, ref)


# K of a step less one, a step, one and a bit, two less one: the step in front of K's end overlaps the one before by nothing to all but one; columns and rows that end
# inside a piece of 16 bytes, at its first element and at its last
@pytest.mark.parametrize("bmnk", [(1, 9, 9, 31), (1, 66, 71, 32), (2, 67, 65, 33), (1, 71, 66, 63), (1, 12, 79, 64), (2, 77, 12, 65), (1, 73, 9, 95), (3, 9, 10, 127), (1, 68, 95, 128)])
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("rhs_nk", [True, False], ids=["NT", "NN"])
@pytest.mark.parametrize("lhs_mk", [True, False], ids=["rows", "transposed"])
def test_last_step(hip, bmnk, dtype, rhs_nk, lhs_mk):
    products.test_products_of_any_size(hip, bmnk, dtype, rhs_nk, lhs_mk)


# one step of K or less on the large tile, whose form has no loop: a few elements, an odd number, a whole step
@pytest.mark.parametrize("bmnk", [(16, 130, 1023, 9), (16, 130, 1023, 51), (16, 130, 1023, 64)])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("rhs_nk", [True, False], ids=["NT", "NN"])
@pytest.mark.parametrize("lhs_mk", [True, False], ids=["rows", "transposed"])
def test_one_step_on_the_large_tile(hip, bmnk, dtype, rhs_nk, lhs_mk):
    products.test_products_of_any_size(hip, bmnk, dtype, rhs_nk, lhs_mk)
    assert ug_amd.last_kernel() == f"gemm_any<{dtype},128x128>"


# 32 x 32 tiles, a few and several to a CU: fewer steps of K than waves, as many, one more, uneven parts and a last wave without one; tiles over both edges; batches
@pytest.mark.parametrize("bmnk", [(1, 100, 100, 65), (1, 33, 65, 120), (1, 300, 300, 300), (2, 31, 97, 257), (1, 330, 9, 350), (1, 625, 319, 353), (15, 19, 18, 640), (1, 23, 148, 1355), (8, 200, 200, 200)])
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("rhs_nk", [True, False], ids=["NT", "NN"])
@pytest.mark.parametrize("lhs_mk", [True, False], ids=["rows", "transposed"])
def test_small_tiles(hip, bmnk, dtype, rhs_nk, lhs_mk):
    products.test_products_of_any_size(hip, bmnk, dtype, rhs_nk, lhs_mk)


# aligned products of few tiles: on either side of where the kernel with larger tiles takes over (steps of K in all tiles; 32 tiles and K; 255 tiles and 256), small integers exactly
@pytest.mark.parametrize("bmnk, small", [((1, 64, 64, 4096), True), ((1, 64, 64, 4128), False), ((1, 64, 2048, 2048), True), ((1, 64, 2112, 2048), False), ((8, 192, 64, 320), True),
                                         ((1, 512, 512, 512), True), ((1, 576, 1600, 1024), True), ((1, 576, 1600, 1056), False), ((255, 64, 64, 64), True), ((256, 64, 64, 64), False), ((1, 64, 384, 64), True), ((1, 64, 384, 32), False)])
@pytest.mark.parametrize("rhs_nk", [True, False], ids=["NT", "NN"])
def test_aligned_products_of_few_tiles(hip, bmnk, small, rhs_nk):
    b, m, n, k = bmnk
    a, w = np.floor(products.rng.uniform_pm1(1, b * m * k) * 4).reshape(b, m, k), np.floor(products.rng.uniform_pm1(2, b * k * n) * 4).reshape(b, k, n)
    got = products._raw_matmul(hip, ug_amd.F32, a, w, rhs_nk)
    assert ug_amd.last_kernel().startswith("gemm_any<") == (small and not rhs_nk), ug_amd.last_kernel()
    np.testing.assert_array_equal(got, np.matmul(a.astype(np.float32), w.astype(np.float32)))  # sums below 2^24: exact in any order
