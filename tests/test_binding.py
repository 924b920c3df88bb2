"""The native argument conversion refuses what a launch could not take before it reaches the library."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from arraydiff_cuda_amd import capi


@pytest.mark.parametrize("call,error", [
    (lambda: capi.relu_fwd(torch.zeros(4), torch.zeros(4)), ValueError),  # not on the GPU
    (lambda: capi._n().adh_relu_fwd(0, 4, [], None), TypeError),  # a sequence where one tensor belongs
    (lambda: capi._n().adh_relu_fwd(0, 4, None), TypeError),  # an argument too few
    (lambda: capi.flat_store([torch.zeros(2)], torch.zeros(2)), ValueError),
    # integers are no addresses, alone or in a table (of no element: nothing is launched where they are taken for some)
    (lambda: capi._n().adh_relu_fwd(0, 0, None, 4096), TypeError),
    (lambda: capi._n().adh_relu_fwd(0, 0, True, None), TypeError),
    (lambda: capi._n().adh_sum_fwd(0, 2, 0, [4096, 4096], None), TypeError),
    (lambda: capi._n().adh_sum_fwd(0, 2, 0, [None, None], None), TypeError)])  # nor does a table have gaps
def test_refused_arguments(call, error):
    with pytest.raises(error):
        call()


@pytest.mark.parametrize("call", [lambda t: capi.relu_fwd(t, t), lambda t: capi.sum_fwd([t], t)])
def test_a_tensor_without_an_address_raises(call):
    """Under vmap a tensor has no storage: torch's C++ exception arrives as a Python one."""
    with FakeTensorMode(), pytest.raises(RuntimeError, match="storage"):
        torch.vmap(lambda t: (call(t), t)[1])(torch.empty(3, 4, device="cuda"))
