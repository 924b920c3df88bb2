"""The native argument conversion refuses what a launch could not take before it reaches the library."""
import pytest
import torch

from arraydiff_cuda_amd import capi


@pytest.mark.parametrize("call,error", [
    (lambda: capi.relu_fwd(torch.zeros(4), torch.zeros(4)), ValueError),  # not on the GPU
    (lambda: capi._n().adh_relu_fwd(0, 4, [], None), TypeError),  # a sequence where one tensor belongs
    (lambda: capi._n().adh_relu_fwd(0, 4, None), TypeError),  # an argument too few
    (lambda: capi.flat_store([torch.zeros(2)], torch.zeros(2)), ValueError)])
def test_refused_arguments(call, error):
    with pytest.raises(error):
        call()
