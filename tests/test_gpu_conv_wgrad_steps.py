"""bf16 filter gradients of the 3x3 stride-1 window over padded tiles and over tiles without halo, at the sizes where steps, octets of
pixels and groups of channels end, in small workspaces, and with values that are not finite beside the last row, against float64."""
import pytest
import torch
import torch.nn.functional as F

from arraydiff_cuda_amd import capi

pytestmark = pytest.mark.gpu


def _reference(x, dy, K, stacked):
    """In double.  x, dy: the whole tensor (stacked) or the tiles one after the other."""
    xp = F.pad(x.double(), (1,) * 4) if stacked else x.double()
    OH, OW = dy.shape[2:]
    d = dy.double().permute(1, 0, 2, 3).reshape(dy.shape[1], -1)
    taps = [[d @ xp[:, :, a:a + OH, b:b + OW].permute(1, 0, 2, 3).reshape(x.shape[1], -1).T for b in range(3)] for a in range(3)]
    return torch.stack([torch.stack(row, -1) for row in taps], -2)


def _tensors(K, N, Ci, Co, H, W, stacked, seed=0):
    g = torch.Generator().manual_seed(seed + Ci + 31 * Co + W)
    xs, ds = ((N, Ci, H * K, W), (N, Co, H * K, W)) if stacked else ((K * N, Ci, H + 2, W + 2), (K * N, Co, H, W))
    return (torch.rand(xs, generator=g) * 2 - 1).bfloat16(), torch.randn(ds, generator=g).bfloat16()


def _run(x, dy, K, stacked, beta=0.0, part=1):
    N, Ci, Co = x.shape[0] // (1 if stacked else K), x.shape[1], dy.shape[1]
    size = (N, Ci, Co, dy.shape[2] // (K if stacked else 1), dy.shape[3])
    query = capi.conv_workspace_bytes(capi.ADH_CONV_BWD_FILTER, capi.ADH_BF16, K, *size)
    ws = torch.full((query // 4 // part,), float("nan"), device="cuda")
    old = torch.randn((Co, Ci, 3, 3), generator=torch.Generator().manual_seed(1))
    dw = old.cuda()
    xs, dys = ([t.contiguous().cuda() for t in v.chunk(K, 2 if stacked else 0)] for v in (x, dy))
    f = capi.conv_unpadded_bwd_filter_tiles if stacked else capi.conv_bwd_filter_tiles
    capi.check(f(xs, dys, dw, *size, beta=beta, ws=ws), "filter gradient")
    return dw.cpu().double() - (old.double() if beta else 0.0)


def _check(K, N, Ci, Co, H, W, stacked, beta=0.0):
    x, dy = _tensors(K, N, Ci, Co, H, W, stacked)
    got, want = _run(x, dy, K, stacked, beta), _reference(x, dy, K, stacked)
    # fp32 sums of exact products: 2^-24 a term, random in sign
    assert (got - want).norm() <= 1e-6 * want.norm() + (2e-7 * want.numel() ** 0.5 if beta else 0.0)


@pytest.mark.parametrize("stacked", [False, True])
@pytest.mark.parametrize("Ci,Co", [(1, 1), (16, 16), (31, 33), (32, 32), (33, 32), (64, 40), (65, 129), (20, 100), (128, 7)])
def test_channels(Ci, Co, stacked):
    _check(2, 2, Ci, Co, 5, 24, stacked)


@pytest.mark.parametrize("Ci", [20, 40])
@pytest.mark.parametrize("W", [7, 8, 9, 10, 11, 13, 15, 16, 17, 23, 31, 32, 33, 47, 57, 63, 64, 65, 71, 72, 127, 129, 200])
def test_widths_with_halo(W, Ci):
    _check(2, 3, Ci, 36, 4, W, False)


@pytest.mark.parametrize("Ci,Co", [(20, 36), (40, 36), (40, 20), (20, 20)])
@pytest.mark.parametrize("W", [8, 16, 24, 32, 40, 56, 64, 72, 120, 128, 136])
def test_widths_without_halo(W, Ci, Co):
    _check(2, 3, Ci, Co, 4, W, True)


@pytest.mark.parametrize("stacked", [False, True])
@pytest.mark.parametrize("K,N,H", [(1, 1, 1), (3, 1, 1), (16, 2, 2), (1, 5, 3), (2, 3, 13), (1, 2, 67), (5, 9, 6)])
@pytest.mark.parametrize("W", [8, 16, 32, 72])
def test_images_and_tiles(K, N, H, W, stacked):
    _check(K, N, 24, 48, H, W, stacked)


@pytest.mark.parametrize("stacked", [False, True])
def test_accumulates(stacked):
    _check(2, 3, 40, 70, 7, 24, stacked, beta=1.0)


@pytest.mark.parametrize("stacked", [False, True])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
def test_not_finite_values_stay_in_their_taps(value, stacked):
    """The last row and column of x reach the taps of existing outputs only, dy's zeros beyond multiply nothing that counts."""
    K = 2 if stacked else 1
    x, dy = _tensors(K, 2, 20, 36, 5, 24, stacked, 3)
    x[1, 3, -1, 5] = value
    x[0, 7, 4, -1] = value
    x[0, 11, 0, 0] = value
    dy[1, 9, -1, 2] = value
    got, want = _run(x, dy, K, stacked), _reference(x, dy, K, stacked)
    # (the reference's padding is zeros, which times what is not finite is NaN, as here: both have to agree)
    assert torch.equal(got.isnan(), want.isnan())
    fine = want.isfinite()
    assert torch.equal(got[~fine & ~want.isnan()], want[~fine & ~want.isnan()])
    assert (got - want)[fine].norm() <= 1e-6 * want[fine].norm()


@pytest.mark.parametrize("stacked,W", [(False, 40), (True, 40), (False, 41)])
def test_small_workspaces(stacked, W):
    """What the entry points took before they had this kernel: the same sums in fewer parts."""
    x, dy = _tensors(2, 4, 70, 90, 8, W, stacked, 5)
    want, served = _reference(x, dy, 2, stacked), 0
    for part in (1, 2, 3, 5, 9, 20):
        try:
            got = _run(x, dy, 2, stacked, part=part)
        except capi.AdhError as e:
            assert "workspace" in str(e)
            continue
        served += 1
        assert (got - want).norm() <= 1e-6 * want.norm()
    assert served


def _error(K, N, Ci, Co, H, W):
    """Relative error against double precision, computed on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(1)
    xs = [(torch.rand((N, Ci, H + 2, W + 2), device="cuda", generator=g) * 2 - 1).bfloat16() for _ in range(K)]
    dys = [torch.randn((N, Co, H, W), device="cuda", generator=g).bfloat16() for _ in range(K)]
    want = torch.zeros((Co, Ci, 3, 3), device="cuda", dtype=torch.float64)
    for x, dy in zip(xs, dys):
        d = dy.double().transpose(0, 1).reshape(Co, -1)
        for a in range(3):
            for b in range(3):
                want[:, :, a, b] += d @ x[:, :, a:a + H, b:b + W].double().permute(0, 2, 3, 1).reshape(-1, Ci)
    dw = torch.empty((Co, Ci, 3, 3), device="cuda")
    ws = torch.empty(capi.conv_workspace_bytes(capi.ADH_CONV_BWD_FILTER, capi.ADH_BF16, K, N, Ci, Co, H, W) // 4, device="cuda")
    capi.check(capi.conv_bwd_filter_tiles(xs, dys, dw, N, Ci, Co, H, W, ws=ws), "filter gradient")
    return ((dw.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("shape,walks", [((3, 7, 263, 135, 11, 272), 1.58e-7), ((7, 31, 103, 287, 13, 50), 1.64e-7), ((8, 24, 48, 256, 10, 170), 2.27e-7),
                                         ((6, 3, 339, 228, 5, 342), 1.18e-7), ((5, 25, 38, 377, 3, 295), 1.46e-7)])
def test_chains_of_no_more_pixels_than_walks_down_64_columns(shape, walks):
    """Layers of several channel groups, of which few splits run at once.  walks: the error of conv3x3_bf16_wgrad.hip's sums (measured; 2.48e-7,
    3.16e-7, 2.39e-7, 2.19e-7 and 2.09e-7 with chains as long as such splits)."""
    assert _error(*shape) <= 1.02 * walks


# (few rows and many channels: chains of 1, 2, 3, 4 and 5 steps, one group of 32 channels on either side, groups and splits that are not full)
LINKED = [(8, 6, 206, 148, 3, 29), (6, 23, 54, 226, 3, 79), (3, 21, 128, 32, 2, 507), (4, 17, 16, 256, 2, 92), (6, 2, 85, 203, 4, 551), (8, 11, 29, 212, 5, 145),
          (7, 22, 375, 95, 4, 12)]


@pytest.mark.parametrize("shape", LINKED)
def test_linked_chains(shape):
    # the rounding of a split's sum and of the result (2^-24 each), and of chains of at most 1024 pixels, 32 of an addition
    assert _error(*shape) <= 2.0 ** -24 * (2 + 32 / 3) ** 0.5


@pytest.mark.parametrize("shape", [LINKED[1], LINKED[2], LINKED[3]])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf"), 3e38])
def test_not_finite_values_in_linked_chains(shape, value):
    """What is not finite, or becomes so in a chain, is summed again in plain fp32."""
    K, N, Ci, Co, H, W = shape
    x, dy = _tensors(K, N, Ci, Co, H, W, False, 3)
    x[1, 3, 2, 5] = value
    x[-1, 7, 1, 40] = value
    got, want = _run(x, dy, K, False, beta=1.0), _reference(x, dy, K, False)
    if value == 3e38:
        want = torch.where(want.abs() > 3.4e38, want.sign() * float("inf"), want)
    assert torch.equal(got.isnan(), want.isnan())
    sure = want.isinf() if value != 3e38 else want.abs() > 1e39
    assert torch.equal(got[sure], want[sure])
    fine = want.abs() < 1e30
    assert fine.any() and not fine.all()
    assert (got - want)[fine].norm() <= 1e-6 * want[fine].norm()
