"""Weight gradients on either side of the line between one wave and four an adapter (wgrad_split): against the oracle bit
for bit on exactly representable inputs, and several projections against calls of one, whose line must be the same."""
import pytest

from test_gpu_backward_multi import test_multi_dyadic_bit_exact as dyadic_exact
from test_gpu_backward_multi import test_multi_equals_single_calls_and_oracle as multi_equals_single
from test_gpu_parity import K  # noqa: F401

pytestmark = pytest.mark.gpu

# adapters, rank, rows an adapter from which four waves share them
LINES = [(1, 16, 128), (4, 8, 192), (12, 16, 512), (1, 24, 128), (3, 32, 288), (6, 32, 512), (2, 64, 256), (1, 72, 256),
         (8, 32, 512), (8, 64, 512), (3, 136, 512)]   # (the line's end)


def case(NA, r, from_, below, unequal=False):
    rows = NA * from_ - (1 if below else 0)
    tp = [0] + [rows * i // NA for i in range(1, NA)] + [rows]
    if unequal:   # the first adapter has all rows but 1, 2, 3, ... of the others
        tp = [0] + [rows - sum(range(i, NA)) for i in range(1, NA + 1)]
    return ("line", tp, list(range(NA)), NA, [(128, 192), (192, 64)], r)


@pytest.mark.parametrize("below", [True, False], ids=["one-wave", "four-waves"])
@pytest.mark.parametrize("NA,r,from_", LINES)
def test_either_side_of_the_line(K, oracle, gpu_device, NA, r, from_, below):  # noqa: F811
    dyadic_exact(K, oracle, gpu_device, case(NA, r, from_, below), "bf16")
    multi_equals_single(K, oracle, gpu_device, case(NA, r, from_, below), "bf16", True)


@pytest.mark.parametrize("below", [True, False], ids=["one-wave", "four-waves"])
@pytest.mark.parametrize("NA,r,from_", [(4, 16, 192), (3, 32, 288), (4, 64, 512)])
def test_one_long_adapter_among_short_ones(K, oracle, gpu_device, NA, r, from_, below):  # noqa: F811
    dyadic_exact(K, oracle, gpu_device, case(NA, r, from_, below, unequal=True), "bf16")
