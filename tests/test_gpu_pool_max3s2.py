"""Backward of 3x3 max pooling at stride 2 over tiles without halo, rows of whole groups of four: the kernel that keeps its
windows in registers, at the sizes where it can go wrong (one group of columns, tiles of two rows, an odd number of window rows
per tile, bands of every length), against the oracle's pooling of the unsplit padded tensor, below and above the size from which
forward is that kernel's too; ties, infinities and NaN against the banded kernel."""
import pytest
import torch

from arraydiff_cuda_amd import capi
from test_gpu_pool_unpadded import test_pool_unpadded_f32_vs_unsplit_oracle as check_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,N,C,Ht,W", [(1, 1, 1, 2, 4), (3, 1, 2, 2, 8), (2, 3, 5, 6, 12), (4, 2, 3, 14, 56), (1, 2, 65, 64, 20), (8, 2, 64, 128, 260),
                                        (2, 1, 3, 22, 516), (1, 40, 128, 2, 4), (3, 20, 70, 2, 8), (2, 9, 31, 6, 12), (4, 4, 10, 14, 56)])
def test_vs_unsplit_oracle(oracle, K, N, C, Ht, W):
    check_f32(oracle, capi.ADH_POOL_MAX, K, N, C, Ht, W, 3, 3, 2, 2, 1, 1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("K,Ht,W", [(1, 2, 4), (3, 2, 8), (1, 6, 8), (2, 14, 12), (3, 10, 28)])
def test_same_as_the_banded_kernel(dtype, K, Ht, W):
    """Ties in every window (values of few levels), special values, and whole planes of -inf and of NaN: the same places as the
    bands, which serve the same pooling over one halo-padded tile (whole gradients: their sums are exact in any order)."""
    N = 2
    C = (1 << 15) // (N * K * Ht * W) + 3  # (forward, smaller tensors are the bands')
    g = torch.Generator().manual_seed(4)
    x = torch.randint(-2, 3, (N, C, K * Ht, W), generator=g).float()
    special = torch.tensor([float("inf"), -float("inf"), float("nan"), torch.finfo(dtype).min])
    where = torch.rand(x.shape, generator=g) < 0.2
    x[where] = special[torch.randint(0, 4, (int(where.sum()),), generator=g)]
    x[0, 0] = -float("inf")  # a plane of nothing but the lowest value, and one of nothing but NaN
    x[1, 2] = float("nan")
    x = x.to(dtype).cuda()
    dy = torch.randint(-9, 10, (N, C, K * Ht // 2, W // 2), generator=g).to(dtype).cuda()
    xs, dys = ([t.contiguous() for t in v.chunk(K, 2)] for v in (x, dy))
    ys, dxs = [torch.full_like(t, 7.0) for t in dys], [torch.full_like(t, 7.0) for t in xs]
    capi.check(capi.pool_unpadded_fwd_tiles(capi.ADH_POOL_MAX, xs, ys, N, C, Ht, W, 3, 3, 2, 2, 1, 1), "fwd")
    capi.check(capi.pool_unpadded_bwd_tiles(capi.ADH_POOL_MAX, xs, None, dys, dxs, N, C, Ht, W, 3, 3, 2, 2, 1, 1), "bwd")
    padded = torch.nn.functional.pad(x, (1, 1, 1, 1))
    y, dx = torch.empty_like(dy), torch.zeros_like(padded)
    capi.check(capi.pool_fwd_tiles(capi.ADH_POOL_MAX, [padded], [y], N, C, K * Ht + 2, W + 2, 3, 3, 2, 2), "padded fwd")
    capi.check(capi.pool_bwd_tiles(capi.ADH_POOL_MAX, [padded], [y], [dy], [dx], N, C, K * Ht + 2, W + 2, 3, 3, 2, 2), "padded bwd")
    assert torch.equal(torch.cat(ys, 2).nan_to_num(nan=123.0), y.nan_to_num(nan=123.0))
    assert torch.equal(torch.cat(dxs, 2), dx[:, :, 1:-1, 1:-1])
