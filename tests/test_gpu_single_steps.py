"""One position of the delta rule and of grouped attention at the sizes where their kernels' forms begin and end."""
import pytest

import test_gpu_tugelorn as tugelorn
from gpu_calls import Gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu(hip):
    return Gpu(hip)


# heads of 128 elements and values in whole runs of 32 are held in registers whole: both sides of that, and of pieces of eight in the matrices' rows
@pytest.mark.parametrize("sizes", [(2, 2, 128, 128, 4, 128, 128), (4, 2, 128, 96, 4, 16, 8), (2, 1, 128, 32, 4, 136, 264), (1, 1, 128, 100, 4, 24, 16), (2, 2, 128, 64, 4, 12, 16), (2, 2, 120, 64, 4, 16, 16)])
@pytest.mark.parametrize("cuts", [(1, 1, 1, 1, 1, 1, 1), (66, 1, 1, 1, 1)])
@pytest.mark.parametrize("decay", ["mild", "strong", "none"])
def test_delta_steps(gpu, sizes, cuts, decay):
    tugelorn.test_delta_rule_rows_and_steps(gpu, sizes, cuts, decay)


# few key heads: a workgroup per 32 value elements, the last ones with some left, one, or none; many: the whole head to a workgroup
@pytest.mark.parametrize("sizes", [(4, 2, 64, 33, 32), (2, 2, 128, 32, 128), (8, 1, 128, 97, 64), (34, 1, 64, 64, 64), (2, 1, 192, 128, 64), (128, 128, 16, 40, 8), (129, 129, 64, 40, 32), (130, 65, 128, 72, 24)])
@pytest.mark.parametrize("cuts, window", [((1, 1, 1), 0), ((70, 1, 1), 0), ((95, 1, 1, 1), 33)])
@pytest.mark.parametrize("bf16", [False, True])
def test_attention_of_one_position(gpu, sizes, cuts, window, bf16):
    tugelorn.test_grouped_attention(gpu, sizes, cuts, window, bf16)


def test_attention_of_one_position_over_many_splits(gpu):
    tugelorn.test_grouped_attention_over_many_splits(gpu)
