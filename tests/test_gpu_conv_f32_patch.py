"""fp32 windows of 3x3 and 1x1 on small tensors from patches in LDS, forward and backward-data, at stride 1 and 2, over padded tiles and
tiles without halo, at the sizes where blocks, octets and chunks of channels end, and with values that are not finite, against float64."""
import pytest
import torch
import torch.nn.functional as F

from arraydiff_cuda_amd import capi

pytestmark = pytest.mark.gpu
FWD, BWD = capi.ADH_CONV_FWD, capi.ADH_CONV_BWD_DATA


def _uniform(g, *shape):
    return torch.rand(shape, generator=g) * 2 - 1


def _split(t, K):
    return [a.contiguous().cuda() for a in t.chunk(K, 2)]


def _unpadded(which, k, s, K, N, Ci, Co, H, W, beta=0.0, spoil=None):
    """H x W: a tile of the activation.  Result and reference."""
    g = torch.Generator().manual_seed(Ci + 31 * Co + W)
    w = _uniform(g, Co, Ci, k, k)
    x, y = _uniform(g, N, Ci, H * K, W), _uniform(g, N, Co, H * K // s, W // s)
    if spoil:
        spoil(w, y if which == BWD else x)
    size = (N, Ci, Co, H, W, k, k, s, s, 1, 1, k // 2, k // 2)
    ws = torch.empty(capi.conv2d_unpadded_workspace_bytes(which, capi.ADH_F32, K, *size) // 4 + 64, device="cuda")
    if which == FWD:
        want, old, out = F.conv2d(x.double(), w.double(), padding=k // 2, stride=s), y, _split(y, K)
        capi.check(capi.conv2d_unpadded_fwd_tiles(_split(x, K), w.cuda(), out, *size, beta=beta, ws=ws))
    else:
        want, old, out = F.conv_transpose2d(y.double(), w.double(), padding=k // 2, stride=s, output_padding=s - 1), x, _split(x, K)
        capi.check(capi.conv2d_unpadded_bwd_data_tiles(w.cuda(), _split(y, K), out, *size, beta=beta, ws=ws))
    return torch.cat([o.cpu() for o in out], 2).double() - (old.double() if beta else 0.0), want


def _close(got, want, beta=0.0):
    # 24 bits of every factor and fp32 sums: 2^-24 a term, random in sign; rounding what is accumulated
    assert (got - want).norm() <= 3e-7 * want.norm() + (1e-7 * want.numel() ** 0.5 if beta else 0.0)


FORMS = [(which, k, s) for which in (FWD, BWD) for k, s in ((3, 1), (3, 2), (1, 1), (1, 2))]


@pytest.mark.parametrize("which,k,s", FORMS)
@pytest.mark.parametrize("Ci,Co", [(1, 1), (16, 16), (7, 33), (31, 17), (32, 64), (33, 32), (64, 65), (100, 20), (130, 48)])
def test_channels(which, k, s, Ci, Co):
    _close(*_unpadded(which, k, s, 2, 2, Ci, Co, 6, 22))


@pytest.mark.parametrize("which,k,s", FORMS)
@pytest.mark.parametrize("W", [4, 6, 8, 10, 14, 16, 18, 30, 32, 34, 62, 64, 66, 126, 130, 258])
def test_widths(which, k, s, W):
    _close(*_unpadded(which, k, s, 2, 3, 20, 36, 4, W))


@pytest.mark.parametrize("which,k,s", FORMS)
@pytest.mark.parametrize("K,N,H", [(1, 1, 2), (3, 1, 2), (8, 2, 2), (1, 5, 4), (2, 3, 14), (1, 2, 66), (5, 9, 6)])
def test_images_and_tiles(which, k, s, K, N, H):
    _close(*_unpadded(which, k, s, K, N, 24, 40, H, 12))


# What the larger tiles serve (two tiles of H x W): 16 MT channels by 64 NT pixels, MT and NT of 1 and 2 as the plan takes them there
LARGER_TILES = [(FWD, 3, 1, 2, 20, 24, 30, 130), (FWD, 3, 1, 4, 33, 31, 14, 130), (BWD, 3, 1, 2, 24, 20, 30, 130), (BWD, 3, 1, 4, 31, 33, 14, 130),
                (FWD, 3, 2, 4, 16, 24, 30, 130), (FWD, 3, 2, 8, 33, 17, 14, 130), (FWD, 1, 1, 4, 16, 16, 30, 130), (FWD, 1, 1, 2, 16, 24, 30, 130),
                (FWD, 1, 1, 8, 70, 17, 14, 130), (FWD, 1, 2, 16, 16, 16, 30, 130), (FWD, 1, 2, 16, 16, 24, 14, 130), (FWD, 1, 2, 16, 20, 33, 30, 88),
                (BWD, 1, 1, 4, 16, 16, 30, 130), (BWD, 1, 1, 4, 24, 16, 14, 130), (BWD, 1, 1, 8, 24, 70, 14, 130), (BWD, 1, 2, 16, 16, 16, 30, 130),
                (BWD, 1, 2, 16, 24, 16, 14, 130), (BWD, 1, 2, 16, 33, 20, 30, 88)]


@pytest.mark.parametrize("which,k,s,N,Ci,Co,H,W", LARGER_TILES)
@pytest.mark.parametrize("beta", [0.0, 1.0])
def test_larger_tiles(which, k, s, N, Ci, Co, H, W, beta):
    if k == 3 and s == 1:  # (which the name is of)
        assert "conv_f32_patch_kernel<2, 2, 0, 9>" in capi.conv_kernel_name(which, capi.ADH_F32, 2, N, Ci, Co, H, W)
    _close(*_unpadded(which, k, s, 2, N, Ci, Co, H, W, beta=beta), beta=beta)


@pytest.mark.parametrize("which,k,s", FORMS)
def test_accumulates(which, k, s):
    _close(*_unpadded(which, k, s, 2, 3, 40, 24, 8, 22, beta=1.0), beta=1.0)


@pytest.mark.parametrize("which", [FWD, BWD])
@pytest.mark.parametrize("W", [1, 2, 3, 5, 7, 13, 17, 31, 33, 63, 65])
@pytest.mark.parametrize("K,N,H", [(1, 2, 5), (3, 2, 3)])
def test_padded_tiles(which, W, K, N, H):
    g = torch.Generator().manual_seed(W)
    Ci, Co = 33, 20
    w, x, y = _uniform(g, Co, Ci, 3, 3), _uniform(g, K * N, Ci, H + 2, W + 2), _uniform(g, K * N, Co, H, W)
    tiles = lambda t: [a.contiguous().cuda() for a in t.chunk(K, 0)]
    if which == FWD:
        out, want = tiles(y), F.conv2d(x.double(), w.double())
        capi.check(capi.conv_fwd_tiles(tiles(x), w.cuda(), out, N, Ci, Co, H, W))
    else:
        out, want = tiles(x), F.conv_transpose2d(y.double(), w.double())
        capi.check(capi.conv_bwd_data_tiles(w.cuda(), tiles(y), out, N, Ci, Co, H, W))
    _close(torch.cat([o.cpu() for o in out]).double(), want)


def test_residual():
    g = torch.Generator().manual_seed(4)
    K, N, Ci, Co, H, W = 2, 3, 40, 50, 5, 19
    w, x, r = _uniform(g, Co, Ci, 3, 3), _uniform(g, N, Ci, H * K, W), _uniform(g, N, Co, H * K, W)
    out = [torch.full((N, Co, H, W), float("nan"), device="cuda") for _ in range(K)]
    capi.check(capi.conv_unpadded_fwd_residual_tiles(_split(x, K), w.cuda(), _split(r, K), out, N, Ci, Co, H, W))
    _close(torch.cat([o.cpu() for o in out], 2).double(), F.conv2d(x.double(), w.double(), padding=1) + r.double(), 1.0)


@pytest.mark.parametrize("which,k,s", FORMS)
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf"), 3.4e38])
def test_not_finite_values_stay_in_their_windows(which, k, s, value):
    def spoil(w, t):
        t[0, 3, 1, 2] = value
        t[1, 5, -1, -1] = value
        t[1, 7, 0, 0] = value
        w[w != 0] = w[w != 0].sign() * w[w != 0].abs().clamp(min=0.1)  # (3.4e38 times less is no sum of fp32 here)

    got, want = _unpadded(which, k, s, 2, 2, 20, 36, 6, 22, spoil=spoil)
    want = want.float().double()  # beyond fp32: infinite
    touched = ~want.isfinite() | (want.abs() > 1e30)
    if value != value or abs(value) == float("inf"):
        assert torch.equal(got.isnan(), want.isnan())
        assert torch.equal(got[touched & ~want.isnan()], want[touched & ~want.isnan()])
    else:
        near = touched & (want.abs() < 3.3e38)
        assert ((got - want)[near].abs() <= 1e-6 * want[near].abs()).all()
    fine = ~touched
    assert (got - want)[fine].norm() <= 3e-7 * want[fine].norm()


@pytest.mark.parametrize("which,k,s,N,Ci,Co,H,W", LARGER_TILES[1::3])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_not_finite_values_in_larger_tiles(which, k, s, N, Ci, Co, H, W, value):
    def spoil(w, t):
        t[0, 3, 1, 2] = value
        t[1, 5, -1, -1] = value
        t[-1, 7, 0, 64 // s] = value  # (a pixel that every form reads)

    got, want = _unpadded(which, k, s, 2, N, Ci, Co, H, W, spoil=spoil)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    fine = want.isfinite()
    assert fine.any() and not fine.all()
    assert (got - want)[fine].norm() <= 3e-7 * want[fine].norm()


@pytest.mark.parametrize("which,s", [(FWD, 1), (FWD, 2), (BWD, 1)])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_the_padding_is_data_to_the_filter(which, s, value):
    """An infinite element of it times a zero beside the tensor is NaN, as in sums over a padded tensor."""
    def spoil(w, t):
        w[5, 7, 1, 2] = value

    got, _ = _unpadded(which, 3, s, 2, 2, 20, 36, 6, 22, spoil=spoil)
    g = torch.Generator().manual_seed(20 + 31 * 36 + 22)
    w = _uniform(g, 36, 20, 3, 3)
    x, y = _uniform(g, 2, 20, 12, 22), _uniform(g, 2, 36, 12 // s, 22 // s)
    spoil(w, None)
    t, f = (x, w) if which == FWD else (y, w.transpose(0, 1).flip(2, 3))
    want = F.conv2d(F.pad(t, (1,) * 4).double(), f.double(), stride=s)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
