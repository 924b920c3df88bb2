"""Filter gradients at stride 2 over tiles without halo, 3x3 (fp32, bf16) and 1x1 (bf16), at the sizes where steps, octets of pixels
and groups of channels end, in small workspaces, and with values that are not finite beside the last row, against float64."""
import pytest
import torch
import torch.nn.functional as F

from arraydiff_cuda_amd import capi

pytestmark = pytest.mark.gpu
CODES = {torch.float32: capi.ADH_F32, torch.bfloat16: capi.ADH_BF16}


def _reference(x, dy, k):
    """In double, as sums over what exists: a tap's padding contributes nothing."""
    N, Ci, H, W = x.shape
    Co, OH, OW = dy.shape[1:]
    xp = F.pad(x.double(), (k // 2,) * 4)
    out = torch.zeros((Co, Ci, k, k), dtype=torch.float64)
    d = dy.double().permute(1, 0, 2, 3).reshape(Co, -1)
    for a in range(k):
        for b in range(k):
            p = xp[:, :, a:a + 2 * OH - 1:2, b:b + 2 * OW - 1:2].permute(1, 0, 2, 3).reshape(Ci, -1)
            out[:, :, a, b] = d @ p.T
    return out


def _run(x, dy, k, K, beta=0.0, workspace=None):
    N, Ci, H, W = x.shape
    Co = dy.shape[1]
    size = (N, Ci, Co, H // K, W, k, k, 2, 2, 1, 1, k // 2, k // 2)
    query = capi.conv2d_unpadded_workspace_bytes(capi.ADH_CONV_BWD_FILTER, CODES[x.dtype], K, *size)
    ws = torch.full(((query if workspace is None else workspace) // 4 + 64,), float("nan"), device="cuda")
    old = torch.randn((Co, Ci, k, k), generator=torch.Generator().manual_seed(1))
    dw = old.cuda()
    xs, dys = ([t.contiguous().cuda() for t in v.chunk(K, 2)] for v in (x, dy))
    ws = ws[:(query if workspace is None else workspace) // 4]
    capi.check(capi.conv2d_unpadded_bwd_filter_tiles(xs, dys, dw, *size, beta=beta, ws=ws), "filter gradient")
    return dw.cpu().double() - (old.double() if beta else 0.0)


def _check(dtype, k, K, N, Ci, Co, Ht, W, beta=0.0):
    g = torch.Generator().manual_seed(Ci + 31 * Co + W)
    x = (torch.rand((N, Ci, Ht * K, W), generator=g) * 2 - 1).to(dtype)
    dy = torch.randn((N, Co, Ht * K // 2, W // 2), generator=g).to(dtype)
    got, want = _run(x, dy, k, K, beta), _reference(x, dy, k)
    # fp32 sums of products of 8 (exact) or 24 bits: 2^-24 a term, random in sign
    assert (got - want).norm() <= 1e-6 * want.norm() + (2e-7 * want.numel() ** 0.5 if beta else 0.0)


BOTH = [(torch.float32, 3), (torch.bfloat16, 3), (torch.bfloat16, 1)]


@pytest.mark.parametrize("dtype,k", BOTH)
@pytest.mark.parametrize("Ci,Co", [(1, 1), (16, 16), (31, 33), (32, 32), (33, 32), (64, 40), (65, 129), (20, 100), (128, 7)])
def test_channels(dtype, k, Ci, Co):
    _check(dtype, k, 2, 2, Ci, Co, 6, 20)


@pytest.mark.parametrize("dtype,k", BOTH)
@pytest.mark.parametrize("W", [2, 4, 6, 8, 10, 12, 14, 16, 18, 30, 32, 34, 46, 62, 64, 66, 126, 128, 130, 256, 258])
@pytest.mark.parametrize("Ci", [20, 40])
def test_widths(dtype, k, W, Ci):
    _check(dtype, k, 2, 3, Ci, 36, 4, W)


@pytest.mark.parametrize("dtype,k", BOTH)
@pytest.mark.parametrize("K,N,Ht", [(1, 1, 2), (3, 1, 2), (8, 2, 2), (1, 5, 4), (2, 3, 14), (1, 2, 66), (5, 9, 6)])
@pytest.mark.parametrize("W", [8, 16, 32, 70])
def test_images_and_tiles(dtype, k, K, N, Ht, W):
    _check(dtype, k, K, N, 24, 48, Ht, W)


@pytest.mark.parametrize("dtype,k", BOTH)
def test_accumulates(dtype, k):
    _check(dtype, k, 2, 3, 40, 70, 8, 22, beta=1.0)


@pytest.mark.parametrize("dtype,k", BOTH)
def test_many_steps(dtype, k):
    _check(dtype, k, 4, 8, 128, 96, 16, 64)


@pytest.mark.parametrize("dtype,k", [(torch.float32, 3), (torch.bfloat16, 3)])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
def test_not_finite_values_stay_in_their_taps(dtype, k, value):
    """The last row and column of x reach the taps of existing outputs only, dy's zeros beyond multiply nothing that counts."""
    g = torch.Generator().manual_seed(3)
    K, N, Ci, Co, H, W = 2, 2, 20, 36, 12, 22
    x = (torch.rand((N, Ci, H, W), generator=g) * 2 - 1).to(dtype)
    dy = torch.randn((N, Co, H // 2, W // 2), generator=g).to(dtype)
    x[1, 3, H - 1, 5] = value
    x[0, 7, 4, W - 1] = value
    x[0, 11, 0, 0] = value
    dy[1, 9, H // 2 - 1, 2] = value
    got, want = _run(x, dy, k, K), _reference(x, dy, k)
    # (the reference's padding is zeros, which times what is not finite is NaN, as here: both have to agree)
    assert torch.equal(got.isnan(), want.isnan())
    fine = want.isfinite()
    assert torch.equal(got[~fine & ~want.isnan()], want[~fine & ~want.isnan()])
    assert (got - want)[fine].norm() <= 1e-6 * want[fine].norm()


@pytest.mark.parametrize("dtype,k", BOTH)
def test_small_workspaces(dtype, k):
    """The least that the entry point took before it had this kernel: the same sums in fewer parts."""
    g = torch.Generator().manual_seed(5)
    x = (torch.rand((4, 70, 16, 40), generator=g) * 2 - 1).to(dtype)
    dy = torch.randn((4, 90, 8, 20), generator=g).to(dtype)
    want = _reference(x, dy, k)
    query = capi.conv2d_unpadded_workspace_bytes(capi.ADH_CONV_BWD_FILTER, CODES[dtype], 2, 4, 70, 90, 8, 40, k, k, 2, 2, 1, 1, k // 2, k // 2)
    served = 0
    for part in (1, 2, 3, 5, 9, 20):
        try:
            got = _run(x, dy, k, 2, workspace=query // part // 256 * 256)
        except capi.AdhError as e:
            assert "workspace" in str(e)
            continue
        served += 1
        assert (got - want).norm() <= 1e-6 * want.norm()
    assert served


@pytest.mark.parametrize("K,N,Ci,Co,H,W,former", [(8, 3, 12, 80, 88, 196, 3.41e-7), (8, 13, 17, 17, 86, 122, 4.68e-7), (3, 3, 28, 398, 38, 324, 3.62e-7)])
def test_fp32_sums_over_many_pixels(K, N, Ci, Co, H, W, former):
    """Against double precision on the GPU, where a workgroup adds thousands of pixels.  former: the error of the general kernel's fp32 sums
    (measured; 6.57e-7, 7.34e-7 and 4.89e-7 with six roundings a step)."""
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand((N, Ci, K * H, W), device="cuda", generator=g) * 2 - 1
    dy = torch.randn((N, Co, K * H // 2, W // 2), device="cuda", generator=g)
    xp, d = F.pad(x, (1,) * 4), dy.double().transpose(0, 1).reshape(Co, -1)
    want = torch.stack([torch.stack([d @ xp[:, :, a:a + K * H - 1:2, b:b + W - 1:2].double().permute(0, 2, 3, 1).reshape(-1, Ci) for b in range(3)], -1)
                        for a in range(3)], -2)
    dw, size = torch.empty((Co, Ci, 3, 3), device="cuda"), (N, Ci, Co, H, W, 3, 3, 2, 2, 1, 1, 1, 1)
    ws = torch.empty(capi.conv2d_unpadded_workspace_bytes(capi.ADH_CONV_BWD_FILTER, capi.ADH_F32, K, *size) // 4, device="cuda")
    xs, dys = ([t.contiguous() for t in v.chunk(K, 2)] for v in (x, dy))
    capi.check(capi.conv2d_unpadded_bwd_filter_tiles(xs, dys, dw, *size, ws=ws), "filter gradient")
    assert ((dw.double() - want).norm() / want.norm()).item() <= former
