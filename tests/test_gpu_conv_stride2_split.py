"""The fp32 3x3 convolution at stride 2 over tiles without halo on the bf16 matrix cores, forward and backward-data, at the
sizes where its tiling can go wrong (one pixel, blocks of many images, rows that are no multiple of four quads, channels around
the chunks of 32 and the groups of 16 and 64, several tiles in one block, widths of many blocks), against double precision, at
the accuracy of fp32 sums, and with values whose bf16 parts are not finite."""
import pytest
import torch

from arraydiff_cuda_amd import capi

pytestmark = pytest.mark.gpu

GEO = (3, 3, 2, 2, 1, 1, 1, 1)


def _tiles(a, K):
    return [t.contiguous().cuda() for t in torch.chunk(a, K, dim=2)]


def _rel(got, want):
    return ((got.cpu().double() - want).abs().max() / want.abs().max()).item()


def _inputs(N, Cin, Cout, H, W, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.rand((N, Cin, H, W), generator=g) * 2 - 1, torch.randn((Cout, Cin, 3, 3), generator=g) * (2.0 / (Cin * 9)) ** 0.5,
            torch.randn((N, Cout, H // 2, W // 2), generator=g))


def _passes(x, w, dy, K, beta=0.0, workspace=True):
    N, Cin, H, W = x.shape
    size = (N, Cin, w.shape[0], H // K, W) + GEO
    xs, dys = _tiles(x, K), _tiles(dy, K)
    ys, gs = [torch.ones_like(t) for t in dys], [torch.ones_like(t) for t in xs]
    ws = [torch.empty(capi.conv2d_unpadded_workspace_bytes(q, capi.ADH_F32, K, *size) // 4 + 64, device="cuda")
          for q in (capi.ADH_CONV_FWD, capi.ADH_CONV_BWD_DATA)]
    capi.check(capi.conv2d_unpadded_fwd_tiles(xs, w.cuda(), ys, *size, beta=beta, ws=ws[0]), "fwd")
    capi.check(capi.conv2d_unpadded_bwd_data_tiles(w.cuda(), dys, gs, *size, beta=beta, ws=ws[1]), "bwd-data")
    return torch.cat(ys, 2), torch.cat(gs, 2)


def _want(x, w, dy):
    y = torch.nn.functional.conv2d(x.double(), w.double(), stride=2, padding=1)
    return y, torch.nn.functional.conv_transpose2d(dy.double(), w.double(), stride=2, padding=1, output_padding=1)


@pytest.mark.parametrize("K,N,Cin,Cout,Ht,W", [
    (1, 1, 1, 1, 2, 2), (2, 3, 31, 17, 2, 10), (1, 2, 5, 70, 18, 6), (3, 1, 33, 16, 4, 626), (4, 9, 32, 65, 4, 16), (4, 5, 64, 64, 2, 8),
    (1, 2, 65, 33, 34, 34), (2, 1, 96, 130, 16, 64), (5, 2, 16, 48, 6, 24), (2, 7, 48, 16, 14, 14), (3, 3, 512, 256, 2, 8),
    # 2.1 M results and more, which conv_f32_patch.hip takes no part of: forward, backward-data
    (2, 9, 33, 70, 58, 116), (1, 9, 4, 140, 64, 122), (2, 9, 70, 33, 58, 116), (1, 9, 140, 17, 64, 122)])
def test_passes_vs_double_precision(K, N, Cin, Cout, Ht, W):
    x, w, dy = _inputs(N, Cin, Cout, K * Ht, W, 60 + Cin + W)
    y, g = _want(x, w, dy)
    for beta in (0.0, 1.0):
        got_y, got_g = _passes(x, w, dy, K, beta)
        assert _rel(got_y, y + beta) <= 1e-5
        assert _rel(got_g, g + beta) <= 1e-5


def test_sums_are_as_close_to_double_precision_as_fp32_ones():
    x, w, dy = _inputs(2, 256, 256, 32, 32, 9)
    plain_y = torch.nn.functional.conv2d(x, w, stride=2, padding=1)
    plain_g = torch.nn.functional.conv_transpose2d(dy, w, stride=2, padding=1, output_padding=1)
    for got, want, plain in zip(_passes(x, w, dy, 2), _want(x, w, dy), (plain_y, plain_g)):
        err = ((got.cpu().double() - want).norm() / want.norm()).item()
        ref = ((plain.double() - want).norm() / want.norm()).item()
        assert err <= max(2 * ref, 1.5e-6), (err, ref)  # 2304 terms: fp32 sums in order are 1e-6 off


@pytest.mark.parametrize("N,C,H,W", [(1, 40, 10, 20), (16, 44, 100, 128)])  # the second beyond what conv_f32_patch.hip takes
@pytest.mark.parametrize("bad", [float("inf"), -float("inf"), 3.4e38, float("nan")])
def test_values_without_finite_bf16_parts(bad, N, C, H, W):
    """What an infinity or a number that rounds to an infinite bf16 touches is what plain sums over the zero-padded tensor give."""
    x, w, dy = _inputs(N, C, C, H, W, 3)
    x, w, dy = (x.abs() + 0.5).cuda(), (w.abs() + 0.01).cuda(), (dy.abs() + 0.5).cuda()
    for where in ("data", "filter"):
        xb, wb, db = x.clone(), w.clone(), dy.clone()
        if where == "data":
            xb[0, 3, 4, 10] = db[0, 3, 2, 7] = bad
        else:
            wb[5, 7, 1, 2] = bad
        y, g = torch.zeros((N, C, H // 2, W // 2), device="cuda"), torch.zeros((N, C, H + 2, W + 2), device="cuda")
        xp, dp = torch.nn.functional.pad(xb, (1, 1, 1, 1)), torch.nn.functional.pad(db, (0, 1, 0, 1))
        for a in range(3):
            for b in range(3):
                y += (xp[:, None, :, a:a + H:2, b:b + W:2] * wb[None, :, :, a, b, None, None]).sum(2)
                # gradient row 2i + a - 1 from gradient row i: quads past the last one read the zero padding, as data
                g[:, :, a:a + H + 1:2, b:b + W + 1:2] += (dp[:, :, None] * wb[None, :, :, a, b, None, None]).sum(1)[..., :(H + 3 - a) // 2, :(W + 3 - b) // 2]
        for got, want in zip(_passes(xb, wb, db, 1), (y, g[:, :, 1:-1, 1:-1])):
            assert torch.equal(torch.isnan(got), torch.isnan(want))
            assert torch.equal(torch.isinf(got), torch.isinf(want))
            fine = torch.isfinite(want)
            assert ((got[fine].double() - want[fine].double()).abs() <= 2e-6 * want[fine].double().abs()).all()
            assert fine.any()


@pytest.mark.parametrize("Cin,Cout", [(8, 320), (12, 384), (512, 128), (5, 576)])
def test_forward_on_either_side_of_the_line_between_the_kernels(Cin, Cout):
    """24 images of 16 x 16 results are 48 blocks per 64 channels: 240 and 96 (one round), 288 and 432 (two, of which 224 and 80 idle)."""
    g = torch.Generator().manual_seed(14)
    x, w = torch.rand((24, Cin, 32, 32), generator=g) * 2 - 1, torch.randn((Cout, Cin, 3, 3), generator=g) * (2.0 / (9 * Cin)) ** 0.5
    want = torch.nn.functional.conv2d(x.double(), w.double(), stride=2, padding=1)
    geo = (3, 3, 2, 2, 1, 1, 1, 1)
    for beta in (0.0, 1.0):
        y = torch.ones((24, Cout, 16, 16), device="cuda")
        ws = torch.empty(capi.conv2d_unpadded_workspace_bytes(capi.ADH_CONV_FWD, capi.ADH_F32, 1, 24, Cin, Cout, 32, 32, *geo) // 4, device="cuda")
        capi.check(capi.conv2d_unpadded_fwd_tiles([x.cuda()], w.cuda(), [y], 24, Cin, Cout, 32, 32, *geo, beta=beta, ws=ws), "fwd")
        assert ((y.cpu().double() - want - beta).abs().max() / want.abs().max()).item() <= 1e-5
