"""Rows whose length is no multiple of a vector: the last vector of a row ends with the row (pack, unpack and the tiles' zeroed
borders), rows shorter than a vector go element by element.  Copies: exact."""
import pytest
import torch

from arraydiff_cuda_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("W", [1, 3, 4, 5, 7, 8, 9, 15, 17, 255])
@pytest.mark.parametrize("p", [1, 2])
def test_pack_and_unpack(dtype, W, p):
    K, N, C, Ht = 2, 2, 3, 4
    g = torch.Generator().manual_seed(W)
    x = torch.randn((N, C, K * Ht, W), generator=g).to(dtype).cuda()
    tiles = [torch.full((N, C, Ht + 2 * p, W + 2 * p), float("nan"), device="cuda", dtype=dtype) for _ in range(K)]
    capi.check(capi.tiles_pack(K, p, W, K * Ht, C, N, x, tiles), "pack")
    wide = torch.nn.functional.pad(x, (p, p, p, p))
    for r in range(K):
        assert torch.equal(tiles[r], wide[:, :, r * Ht:r * Ht + Ht + 2 * p])
    guard = torch.full((N * C * K * Ht * W + 16,), 7.0, device="cuda", dtype=dtype)
    y = guard[8:-8].view(x.shape)
    capi.check(capi.tiles_unpack(K, p, W, K * Ht, C, N, tiles, y), "unpack")
    assert torch.equal(y, x) and (guard[:8] == 7).all() and (guard[-8:] == 7).all()
