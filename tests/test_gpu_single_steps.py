"""One position of the delta rule at the sizes where its kernel's forms begin and end."""
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
