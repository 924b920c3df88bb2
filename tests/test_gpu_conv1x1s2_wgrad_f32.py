"""Filter gradients of the 1x1 window at stride 2 in fp32 over tiles without halo: three bf16 parts on the matrix cores, at the sizes where
steps, octets and groups of channels end, with values that are not finite, and in small workspaces; rows of fewer than four outputs
go past them."""
import pytest
import torch

from arraydiff_cuda_amd import capi
from test_gpu_conv_s2_wgrad import _reference, _run

pytestmark = pytest.mark.gpu


def _check(K, N, Ci, Co, Ht, W, beta=0.0):
    g = torch.Generator().manual_seed(Ci + 31 * Co + W)
    x = torch.rand((N, Ci, Ht * K, W), generator=g) * 2 - 1
    dy = torch.randn((N, Co, Ht * K // 2, W // 2), generator=g)
    got, want = _run(x, dy, 1, K, beta), _reference(x, dy, 1)
    # every rounding is one of a partial sum, which is no more than the terms' magnitudes; a few of them add up (and of the old value)
    assert bool(((got - want).abs() <= 2.0 ** -22 * _reference(x.abs(), dy.abs(), 1) + (1e-6 if beta else 0.0)).all())


@pytest.mark.parametrize("Ci,Co", [(1, 1), (16, 16), (31, 33), (33, 32), (64, 40), (65, 129), (128, 7)])
@pytest.mark.parametrize("W", [2, 6, 8, 14, 18, 34, 66, 130])
def test_channels_and_widths(Ci, Co, W):
    _check(2, 2, Ci, Co, 6, W)


@pytest.mark.parametrize("K,N,Ht,W", [(1, 1, 2, 8), (8, 2, 2, 16), (1, 5, 4, 32), (2, 3, 14, 70), (5, 9, 6, 20), (4, 8, 16, 64)])
def test_images_and_tiles(K, N, Ht, W):
    _check(K, N, 40, 80, Ht, W)
    _check(K, N, 24, 48, Ht, W, beta=1.0)


@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_values_that_are_not_finite(value):
    g = torch.Generator().manual_seed(3)
    x = torch.rand((2, 20, 12, 22), generator=g) * 2 - 1
    dy = torch.randn((2, 36, 6, 11), generator=g)
    x[1, 3, 10, 4] = value  # read
    x[0, 7, 11, 21] = value  # an odd row and column: read by no output
    dy[1, 9, 5, 10] = value
    got, want = _run(x, dy, 1, 2), _reference(x, dy, 1)
    assert torch.equal(got.isnan(), want.isnan()) and not want[0, 7].isnan().any()
    fine = want.isfinite()
    assert torch.equal(got[~fine & ~want.isnan()], want[~fine & ~want.isnan()])
    assert (got - want)[fine].norm() <= 1e-6 * want[fine].norm()


def test_small_workspaces():
    """Fewer parts, down to what is refused."""
    g = torch.Generator().manual_seed(5)
    x = torch.rand((4, 70, 16, 40), generator=g) * 2 - 1
    dy = torch.randn((4, 90, 8, 20), generator=g)
    want = _reference(x, dy, 1)
    query = capi.conv2d_unpadded_workspace_bytes(capi.ADH_CONV_BWD_FILTER, capi.ADH_F32, 2, 4, 70, 90, 8, 40, 1, 1, 2, 2, 1, 1, 0, 0)
    served = 0
    for part in (1, 2, 3, 5, 9, 20):
        try:
            got = _run(x, dy, 1, 2, workspace=query // part // 256 * 256)
        except capi.AdhError as e:
            assert "workspace" in str(e)
            continue
        served += 1
        assert (got - want).norm() <= 1e-6 * want.norm()
    assert served
