"""bf16 3x3 convolution with more than 64 reduction channels at widths that are no multiple of eight: the passes over a
copy of the input with wider rows (rows shorter than a granule, one column off one, last strips of one column)."""
import pytest

from test_gpu_conv_bf16 import test_bf16_conv_small_vs_oracle as check_passes_vs_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,N,Cin,Cout,H,W", [(1, 1, 65, 66, 1, 1), (2, 2, 72, 130, 3, 7), (1, 2, 130, 72, 5, 33), (3, 1, 192, 65, 4, 65),
                                              (1, 3, 128, 128, 6, 23), (1, 1, 80, 16, 9, 97), (2, 1, 16, 80, 2, 12)])
def test_odd_widths_vs_oracle(oracle, K, N, Cin, Cout, H, W):
    check_passes_vs_oracle(oracle, K, N, Cin, Cout, H, W)
