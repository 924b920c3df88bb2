"""3x3 and 1x1 convolutions of bf16 tensors from patches in LDS, through the general entry points: strides 1 and 2, forward and
backward-data, at the sizes where tiles, pairs of pixels and chunks of channels end, against float64 on the CPU."""
import pytest
import torch
import torch.nn.functional as F

from arraydiff_cuda_amd import capi

pytestmark = pytest.mark.gpu


def _check(K, N, Ci, Co, Ht, W, k, s, d=1, beta=0.0, padded=False):
    """Row tiles of one tensor without halo, or (padded) independent tiles that hold theirs."""
    g = torch.Generator().manual_seed(Ci * 131 + Co * 17 + W)
    p = d * (k // 2)
    bf = lambda t: t.to(torch.bfloat16)
    x = bf(torch.rand((N, Ci, Ht * K, W), generator=g) * 2 - 1)
    w = bf(torch.randn((Co, Ci, k, k), generator=g) * (2.0 / (Ci * k * k)) ** 0.5)
    OHt, OW = Ht // s, (W + 2 * p - d * (k - 1) - 1) // s + 1
    dy = bf(torch.randn((N, Co, OHt * K, OW), generator=g))
    x64 = x.double().requires_grad_()
    if padded:
        tiles = [F.pad(t, (p, p, p, p)).contiguous() for t in x.chunk(K, 2)]
        ins = [t.double().requires_grad_() for t in tiles]
        outs = [F.conv2d(t, w.double(), stride=s, dilation=d) for t in ins]
        ys64 = outs
        OHt, OW = outs[0].shape[2:]
        dys = [bf(torch.randn(o.shape, generator=g)) for o in outs]
        torch.autograd.backward(outs, [t.double() for t in dys])
        dx64 = [t.grad for t in ins]
    else:
        tiles = [t.contiguous() for t in x.chunk(K, 2)]
        y = F.conv2d(x64, w.double(), stride=s, padding=p, dilation=d)
        y.backward(dy.double())
        ys64, dx64, dys = y.detach().chunk(K, 2), x64.grad.chunk(K, 2), [t.contiguous() for t in dy.chunk(K, 2)]
    H, WI = tiles[0].shape[2:]
    cu = lambda ts: [t.cuda() for t in ts]
    tiles, dys, wd = cu(tiles), cu(dys), w.cuda()
    old_y = [bf(torch.randn(t.shape, generator=g)) for t in ys64]
    old_x = [bf(torch.randn(t.shape, generator=g)) for t in dx64]
    ys, dxs = cu(old_y) if beta else [torch.full(t.shape, float("nan"), device="cuda", dtype=torch.bfloat16) for t in old_y], None
    dxs = cu(old_x) if beta else [torch.full(t.shape, float("nan"), device="cuda", dtype=torch.bfloat16) for t in old_x]
    geometry = (k, k, s, s, d, d) + (() if padded else (p, p))
    query = capi.conv2d_workspace_bytes if padded else capi.conv2d_unpadded_workspace_bytes
    fwd = capi.conv2d_fwd_tiles if padded else capi.conv2d_unpadded_fwd_tiles
    bwd = capi.conv2d_bwd_data_tiles if padded else capi.conv2d_unpadded_bwd_data_tiles
    size = (N, Ci, Co, H, WI) + geometry
    ws = [torch.empty(query(q, capi.ADH_BF16, K, *size) // 4 + 64, device="cuda") for q in (capi.ADH_CONV_FWD, capi.ADH_CONV_BWD_DATA)]
    capi.check(fwd(tiles, wd, ys, *size, beta=beta, ws=ws[0]), "forward")
    capi.check(bwd(wd, dys, dxs, *size, beta=beta, ws=ws[1]), "backward-data")
    for got, want, old in list(zip(ys, ys64, old_y)) + list(zip(dxs, dx64, old_x)):
        want = want.detach() + (old.double() if beta else 0.0)
        err = (got.cpu().double() - want).abs()
        # one rounding to the 8 significant bits of bf16 (at most 2^-8 of the value) of a sum whose own error is 2^-20 of its terms' size
        assert bool((err <= 2.0 ** -8 * 1.001 * want.abs() + 2e-5 * (1 + want.abs().max())).all()), err.max()


CHANNELS = [(1, 1), (3, 16), (8, 17), (16, 33), (31, 64), (32, 65), (33, 7), (64, 48), (72, 130), (130, 20)]


@pytest.mark.parametrize("Ci,Co", CHANNELS)
@pytest.mark.parametrize("s", [1, 2])
def test_3x3_channels(Ci, Co, s):
    _check(2, 2, Ci, Co, 6, 14, 3, s)


@pytest.mark.parametrize("W", [2, 4, 6, 8, 10, 16, 30, 34, 62, 66, 128, 130, 258, 514])
@pytest.mark.parametrize("s,k", [(2, 3), (2, 1), (1, 1), (1, 3)])
def test_widths(W, s, k):
    _check(3, 1, 20, 24, 4, W, k, s)


@pytest.mark.parametrize("W", [3, 5, 7, 9, 15, 17, 31, 33, 63, 65, 127, 129, 255, 257])
def test_odd_widths(W):
    _check(2, 1, 20, 24, 5, W, 3, 1)
    _check(2, 1, 20, 24, 5, W, 1, 1)


@pytest.mark.parametrize("N,K,Ht,W", [(1, 1, 2, 2), (5, 1, 2, 2), (7, 3, 2, 4), (33, 1, 4, 4), (4, 8, 2, 16), (2, 2, 30, 18), (1, 5, 64, 12), (70, 2, 6, 6)])
@pytest.mark.parametrize("s,k", [(2, 3), (2, 1), (1, 3)])
def test_images_and_tiles(N, K, Ht, W, s, k):
    _check(K, N, 18, 20, Ht, W, k, s)


@pytest.mark.parametrize("s,k", [(2, 3), (2, 1), (1, 1), (1, 3)])
def test_accumulates(s, k):
    _check(2, 3, 40, 24, 8, 22, k, s, beta=1.0)


@pytest.mark.parametrize("d", [1, 2, 3, 8])
def test_dilated_and_padded_tiles(d):
    _check(2, 2, 20, 36, 18, 21, 3, 1, d, padded=True)
    _check(2, 2, 20, 36, 18, 21, 3, 1, d)


@pytest.mark.parametrize("Ci,Co", CHANNELS)
def test_1x1_channels(Ci, Co):
    _check(2, 2, Ci, Co, 6, 14, 1, 1)
    _check(2, 2, Ci, Co, 6, 14, 1, 2)


@pytest.mark.parametrize("H,W", [(5, 7), (6, 9), (9, 4)])
def test_1x1_stride_2_over_odd_tiles(H, W):
    _check(2, 2, 24, 40, H, W, 1, 2, padded=True)


def test_many_blocks():
    _check(2, 8, 96, 160, 32, 64, 3, 2)
    _check(2, 8, 96, 160, 16, 60, 3, 1)


def _check_3x3(K, N, Ci, Co, H, W, halo, beta=0.0, skew=0, spoil=None):
    """The entry points of the 3x3 window, over padded tiles (backward-data: the whole padded slab) or tiles without halo."""
    g = torch.Generator().manual_seed(Ci * 7 + Co + W)
    bf = lambda t: t.to(torch.bfloat16)
    w = bf(torch.randn((Co, Ci, 3, 3), generator=g) * (2.0 / (Ci * 9)) ** 0.5)
    if spoil:
        spoil(w)
    if halo:
        xs = [bf(torch.rand((N, Ci, H + 2, W + 2), generator=g) * 2 - 1) for _ in range(K)]
        dys = [bf(torch.randn((N, Co, H, W), generator=g)) for _ in range(K)]
        ins = [x.double().requires_grad_() for x in xs]
        ys64 = [F.conv2d(x, w.double()) for x in ins]
        torch.autograd.backward(ys64, [d.double() for d in dys])
        dx64 = [x.grad for x in ins]
    else:
        x, dy = bf(torch.rand((N, Ci, H * K, W), generator=g) * 2 - 1), bf(torch.randn((N, Co, H * K, W), generator=g))
        x64 = x.double().requires_grad_()
        y = F.conv2d(x64, w.double(), padding=1)
        y.backward(dy.double())
        xs, dys, ys64, dx64 = x.chunk(K, 2), dy.chunk(K, 2), y.detach().chunk(K, 2), x64.grad.chunk(K, 2)

    def put(t):  # `skew` elements off alignment
        d = torch.empty(t.numel() + skew, device="cuda", dtype=torch.bfloat16)[skew:].view(t.shape)
        return d.copy_(t)
    old_y, old_x = [bf(torch.randn(t.shape, generator=g)) for t in ys64], [bf(torch.randn(t.shape, generator=g)) for t in dx64]
    wd, xd, dyd, ys, dxs = put(w), [put(t) for t in xs], [put(t) for t in dys], [put(t) for t in old_y], [put(t) for t in old_x]
    size = (N, Ci, Co, H, W)
    ws = [torch.empty(capi.conv_workspace_bytes(q, capi.ADH_BF16, K, *size) // 4 + 64, device="cuda") for q in (capi.ADH_CONV_FWD, capi.ADH_CONV_BWD_DATA)]
    fwd, bwd = (capi.conv_fwd_tiles, capi.conv_bwd_data_tiles) if halo else (capi.conv_unpadded_fwd_tiles, capi.conv_unpadded_bwd_data_tiles)
    capi.check(fwd(xd, wd, ys, *size, beta=beta, ws=ws[0]), "forward")
    capi.check(bwd(wd, dyd, dxs, *size, beta=beta, ws=ws[1]), "backward-data")
    for got, want, old in list(zip(ys, ys64, old_y)) + list(zip(dxs, dx64, old_x)):
        want, got = want.detach() + (old.double() if beta else 0.0), got.cpu().double()
        # (of a spoiled channel the kernels also multiply the padding's zeros; the others have to be as ever)
        fine = want.isfinite().all(3, keepdim=True).all(2, keepdim=True).all(0, keepdim=True).expand_as(want)
        scale = want[fine].abs()
        err = (got - want)[fine].abs()
        assert bool((err <= 2.0 ** -8 * 1.001 * scale + 2e-5 * (1 + scale.max())).all()), err.max()


def _patches(which, K, N, Ci, Co, H, W):
    return "patch_kernel" in capi.conv_kernel_name(which, capi.ADH_BF16, K, N, Ci, Co, H, W)


@pytest.mark.parametrize("Ci,Co", CHANNELS + [(224, 16), (16, 224), (97, 300)])
@pytest.mark.parametrize("halo", [True, False])
def test_small_3x3_channels(Ci, Co, halo):
    assert _patches(capi.ADH_CONV_FWD, 2, 3, Ci, Co, 5, 16) and _patches(capi.ADH_CONV_BWD_DATA, 2, 3, Ci, Co, 5, 16)
    _check_3x3(2, 3, Ci, Co, 5, 16, halo)


@pytest.mark.parametrize("W", [1, 2, 3, 7, 8, 9, 31, 64, 65, 250, 515])
def test_small_3x3_widths(W):
    _check_3x3(2, 2, 24, 40, 6, W, True, beta=1.0)


@pytest.mark.parametrize("halo", [True, False])
def test_the_filter_in_order_first(halo):
    """Large enough a launch to put the filter in order, with partial groups of 64 channels on both sides."""
    for which in (capi.ADH_CONV_FWD, capi.ADH_CONV_BWD_DATA):
        assert capi.conv_kernel_name(which, capi.ADH_BF16, 4, 8, 76, 140, 32, 40).endswith("9, true>")
    _check_3x3(4, 8, 76, 140, 32, 40, halo)


@pytest.mark.parametrize("skew", [1, 3])
def test_tiles_off_alignment(skew):
    _check_3x3(2, 3, 20, 24, 5, 17, True, skew=skew)


def test_an_infinite_filter_element_stays_in_its_channel():
    def spoil(w):
        w[3, 17, 1, 1] = float("inf")  # channels of a partial chunk
        w[5, 19, 0, 2] = float("nan")
    for halo in (True, False):
        _check_3x3(2, 2, 20, 24, 6, 16, halo, spoil=spoil)
        _check_3x3(2, 2, 33, 24, 6, 16, halo, spoil=spoil)  # (a chunk of one channel)
