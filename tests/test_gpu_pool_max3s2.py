"""Backward of 3x3 max pooling at stride 2 over tiles without halo, rows of whole groups of four: the kernel that keeps its
windows in registers, at the sizes where it can go wrong (one group of columns, tiles of two rows, an odd number of window rows
per tile, bands of every length), against the oracle's pooling of the unsplit padded tensor; ties, infinities and NaN with
tiles off their alignment (test_gpu_pool_max3s2_widths.py: against the banded kernel)."""
import pytest
import torch

from arraydiff_cuda_amd import capi
from test_gpu_pool_unpadded import test_pool_unpadded_f32_vs_unsplit_oracle as check_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,N,C,Ht,W", [(1, 1, 1, 2, 4), (3, 1, 2, 2, 8), (2, 3, 5, 6, 12), (4, 2, 3, 14, 56), (1, 2, 65, 64, 20), (8, 2, 64, 128, 260),
                                        (2, 1, 3, 22, 516)])
def test_vs_unsplit_oracle(oracle, K, N, C, Ht, W):
    check_f32(oracle, capi.ADH_POOL_MAX, K, N, C, Ht, W, 3, 3, 2, 2, 1, 1)


def _backward(xs, dys, shape, offset=0):
    """offset: elements by which the gradient tiles are off their alignment."""
    N, C, Ht, W = shape
    gs = [torch.empty(N * C * Ht * W + offset, device="cuda", dtype=xs[0].dtype)[offset:].view(shape) for _ in xs]
    capi.check(capi.pool_unpadded_bwd_tiles(capi.ADH_POOL_MAX, xs, None, dys, gs, *shape, 3, 3, 2, 2, 1, 1), "bwd")
    return torch.cat(gs, 2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("K,Ht,W", [(1, 6, 8), (3, 10, 28)])
def test_same_as_the_banded_kernel(dtype, K, Ht, W):
    """Ties in every window (values of few levels) and special values: the same places, the same order of additions."""
    g = torch.Generator().manual_seed(4)
    shape = (2, 3, Ht, W)
    x = torch.randint(-2, 3, (K,) + shape, generator=g).float()
    special = torch.tensor([float("inf"), -float("inf"), float("nan"), torch.finfo(dtype).min])
    where = torch.rand(x.shape, generator=g) < 0.2
    x[where] = special[torch.randint(0, 4, (int(where.sum()),), generator=g)]
    x[:, 0, 0] = -float("inf")  # a plane of nothing but the lowest value, and one of nothing but NaN
    x[:, 1, 2] = float("nan")
    xs = [t.to(dtype).cuda() for t in x]
    dys = [torch.randn((2, 3, Ht // 2, W // 2), generator=g).to(dtype).cuda() for _ in range(K)]
    assert torch.equal(_backward(xs, dys, shape), _backward(xs, dys, shape, offset=1))
