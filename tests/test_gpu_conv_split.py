"""The fp32 3x3 convolution and its filter gradient on the bf16 matrix cores at the sizes where their tiling can go wrong
(rows shorter than a load and column tiles of every width, blocks of one row and of many images, channels around the chunks of 32 and the groups of 16 and 64, rows that are no multiple of four, several
row tiles in one block) against the CPU oracle, at the accuracy of fp32 arithmetic against double precision, and with
values whose bf16 parts are not finite."""
import numpy as np
import pytest
import torch

from arraydiff_cuda_amd import capi
from gpu_util import dev, host, rel_err

pytestmark = pytest.mark.gpu


def _tiles(a, K):
    return [t.contiguous() for t in torch.chunk(a, K, dim=2)]


@pytest.mark.parametrize("K,N,Cin,Cout,Ht,W", [
    (1, 1, 1, 1, 1, 1), (2, 3, 31, 17, 1, 5), (1, 2, 5, 70, 9, 3), (2, 2, 40, 20, 7, 2), (1, 1, 64, 64, 5, 41), (2, 1, 33, 33, 8, 48), (3, 1, 33, 16, 2, 640), (4, 9, 32, 65, 4, 16), (4, 5, 64, 64, 2, 8), (1, 2, 65, 33, 17, 33),
    (2, 1, 96, 130, 16, 32), (5, 2, 8, 48, 3, 12)])
def test_unpadded_passes_vs_oracle(oracle, K, N, Cin, Cout, Ht, W):
    rng = np.random.default_rng(810 + Cin + W)
    H = K * Ht
    x = rng.uniform(-1, 1, size=(N, Cin, H, W)).astype(np.float32)
    w = (rng.standard_normal((Cout, Cin, 3, 3)) * np.sqrt(2.0 / (Cin * 9))).astype(np.float32)
    dy = rng.standard_normal((N, Cout, H, W)).astype(np.float32)
    xp = np.zeros((N, Cin, H + 2, W + 2), np.float32)
    xp[:, :, 1:-1, 1:-1] = x
    y_want, g_want = np.empty((N, Cout, H, W), np.float32), np.empty((N, Cin, H + 2, W + 2), np.float32)
    oracle.conv_slab_fwd(xp, w, y_want)
    oracle.conv_slab_bwd_data(w, dy, g_want)
    dw_want = np.zeros((Cout, Cin, 3, 3), np.float32)
    oracle.conv_slab_bwd_filter(xp, dy, dw_want)
    g_want = g_want[:, :, 1:-1, 1:-1]
    xs, dys = _tiles(dev(x), K), _tiles(dev(dy), K)
    for beta in (0.0, 1.0):
        ys, gs = [torch.ones_like(t) for t in dys], [torch.ones_like(t) for t in xs]
        capi.check(capi.conv_unpadded_fwd_tiles(xs, dev(w), ys, N, Cin, Cout, Ht, W, beta=beta), "fwd")
        capi.check(capi.conv_unpadded_bwd_data_tiles(dev(w), dys, gs, N, Cin, Cout, Ht, W, beta=beta), "bwd-data")
        assert rel_err(host(torch.cat(ys, 2)), y_want + beta) <= 1e-5
        assert rel_err(host(torch.cat(gs, 2)), g_want + beta) <= 1e-5
        dw = torch.ones((Cout, Cin, 3, 3), device="cuda")
        ws = torch.empty(capi.conv_workspace_bytes(capi.ADH_CONV_BWD_FILTER, capi.ADH_F32, K, N, Cin, Cout, Ht, W) // 4, device="cuda")
        capi.check(capi.conv_unpadded_bwd_filter_tiles(xs, dys, dw, N, Cin, Cout, Ht, W, beta=beta, ws=ws), "bwd-filter")
        assert rel_err(host(dw), dw_want + beta) <= 1e-5


def test_sums_are_as_close_to_double_precision_as_fp32_ones():
    g = torch.Generator().manual_seed(5)
    N, C, H, W = 2, 256, 16, 32
    x = torch.rand((N, C, H, W), generator=g) * 2 - 1
    w = torch.randn((C, C, 3, 3), generator=g) * (2.0 / (C * 9)) ** 0.5
    want = torch.nn.functional.conv2d(x.double(), w.double(), padding=1)
    y = torch.empty((N, C, H, W), device="cuda")
    capi.check(capi.conv_unpadded_fwd_tiles([x.cuda()], w.cuda(), [y], N, C, C, H, W), "fwd")
    err = ((y.cpu().double() - want).norm() / want.norm()).item()
    plain = ((torch.nn.functional.conv2d(x, w, padding=1).double() - want).norm() / want.norm()).item()
    assert err <= max(2 * plain, 1.5e-6), (err, plain)  # 2304 terms: fp32 sums in order are 1e-6 off


def test_many_chunks_dealt_to_several_workgroups():
    """512 channels over 2 x 8 tiles through the entry points with a workspace: sums of channel chunks added by a second kernel."""
    K, N, C, Ht, W = 4, 3, 512, 2, 8
    geo = (3, 3, 1, 1, 1, 1, 1, 1)
    g = torch.Generator().manual_seed(6)
    x = torch.rand((N, C, K * Ht, W), generator=g) * 2 - 1
    w = torch.randn((C, C, 3, 3), generator=g) * (2.0 / (C * 9)) ** 0.5
    want = torch.nn.functional.conv2d(x.double(), w.double(), padding=1)
    nbytes = capi.conv2d_unpadded_workspace_bytes(capi.ADH_CONV_FWD, capi.ADH_F32, K, N, C, C, Ht, W, *geo)
    for beta in (0.0, 1.0):
        ys = [torch.ones((N, C, Ht, W), device="cuda") for _ in range(K)]
        capi.check(capi.conv2d_unpadded_fwd_tiles(_tiles(x.cuda(), K), w.cuda(), ys, N, C, C, Ht, W, *geo, beta=beta,
                                                  ws=torch.empty(nbytes // 4 + 64, device="cuda")), "fwd")
        assert rel_err(torch.cat(ys, 2).cpu().numpy(), want.numpy() + beta) <= 1e-5


@pytest.mark.parametrize("bad", [float("inf"), -float("inf"), 3.4e38, float("nan")])
def test_values_without_finite_bf16_parts(bad):
    """An infinity (or a number that rounds to an infinite bf16) in the input or the filter gives what fp32 sums give: the
    outputs it touches, and only those, are infinite, huge or NaN."""
    N, C, H, W = 1, 40, 9, 21
    g = torch.Generator().manual_seed(7)
    x, w = torch.rand((N, C, H, W), generator=g) + 0.5, torch.rand((C, C, 3, 3), generator=g) * 0.1 + 0.01
    for where in ("input", "filter"):
        xb, wb = x.clone(), w.clone()
        if where == "input":
            xb[0, 3, 4, 10] = bad
        else:
            wb[5, 7, 1, 2] = bad
        y = torch.empty((N, C, H, W), device="cuda")
        capi.check(capi.conv_unpadded_fwd_tiles([xb.cuda()], wb.cuda(), [y], N, C, C, H, W), "fwd")
        # taps in order, the zero padding as data (zero times an infinity is NaN)
        xp = torch.nn.functional.pad(xb, (1, 1, 1, 1))
        want = torch.zeros((N, C, H, W))
        for a in range(3):
            for b in range(3):
                want = want + (xp[:, None, :, a:a + H, b:b + W] * wb[None, :, :, a, b, None, None]).sum(2)
        got = y.cpu()
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        assert torch.equal(torch.isinf(got), torch.isinf(want))
        fine = torch.isfinite(want)
        assert ((got[fine].double() - want[fine].double()).abs() <= 2e-6 * want[fine].double().abs()).all()
        assert fine.any() and not torch.equal(want, torch.nn.functional.conv2d(x, w, padding=1))


# Layers just beyond what conv_f32_patch.hip takes: chunks of channels and groups of 16, 32 and 64 that are not full, rows of any width,
# every number of channels on which the order of additions hangs
BEYOND = [(2, 3, 33, 70, 30, 187), (3, 2, 40, 90, 41, 96), (1, 4, 4, 96, 61, 90), (2, 9, 17, 16, 80, 92), (2, 9, 16, 33, 80, 91), (4, 9, 64, 130, 14, 33), (2, 4, 100, 72, 30, 124)]


def _slab(which, K, N, Cin, Cout, H, W, beta=0.0, spoil=None):
    """A pass over padded tiles by the persistent workgroups, and its sums in double precision, both with the padding as data."""
    assert "conv3x3_split_kernel" in capi.conv_kernel_name(which, capi.ADH_F32, K, N, Cin, Cout, H, W)
    g = torch.Generator(device="cuda").manual_seed(Cin + W)
    fwd = which == capi.ADH_CONV_FWD
    w = torch.randn((Cout, Cin, 3, 3), device="cuda", generator=g) * (2.0 / (Cin * 9)) ** 0.5
    t = torch.rand((K * N, Cin if fwd else Cout, H + 2 if fwd else H, W + 2 if fwd else W), device="cuda", generator=g) * 2 - 1
    if spoil:
        spoil(w, t)
    M, OH, OW = (Cout, H, W) if fwd else (Cin, H + 2, W + 2)
    tp = t.double() if fwd else torch.nn.functional.pad(t, (2,) * 4).double()
    wd = (w if fwd else w.transpose(0, 1).flip(2, 3)).double()
    want = torch.zeros((M, K * N * OH * OW), device="cuda", dtype=torch.float64)
    for a in range(3):
        for b in range(3):
            want += wd[:, :, a, b].contiguous() @ tp[:, :, a:a + OH, b:b + OW].transpose(0, 1).reshape(t.shape[1], -1)
    want = want.reshape(M, K * N, OH, OW).transpose(0, 1)
    outs = [torch.full((N, M, OH, OW), 2.0, device="cuda") for _ in range(K)]
    tiles = [v.contiguous() for v in t.chunk(K, 0)]
    if fwd:
        capi.check(capi.conv_fwd_tiles(tiles, w, outs, N, Cin, Cout, H, W, beta=beta), "fwd")
    else:
        capi.check(capi.conv_bwd_data_tiles(w, tiles, outs, N, Cin, Cout, H, W, beta=beta), "bwd-data")
    return torch.cat(outs).double() - (2.0 if beta else 0.0), want


@pytest.mark.parametrize("which", [capi.ADH_CONV_FWD, capi.ADH_CONV_BWD_DATA])
@pytest.mark.parametrize("beta", [0.0, 1.0])
@pytest.mark.parametrize("shape", BEYOND)
def test_persistent_workgroups_vs_double(which, beta, shape):
    if which == capi.ADH_CONV_BWD_DATA:
        K, N, Cin, Cout, H, W = shape
        shape = (K, N, Cout, Cin, H, W)  # (as many results)
    got, want = _slab(which, *shape, beta=beta)
    # 24 bits of every factor and fp32 sums: 2^-24 a term, random in sign; the old output's rounding
    assert (got - want).norm() <= 3e-7 * want.norm() + (2e-7 * want.numel() ** 0.5 if beta else 0.0)


@pytest.mark.parametrize("which", [capi.ADH_CONV_FWD, capi.ADH_CONV_BWD_DATA])
@pytest.mark.parametrize("bad", [float("inf"), -float("inf"), 3.4e38, float("nan")])
@pytest.mark.parametrize("where", ["input", "filter"])
def test_persistent_workgroups_of_values_without_finite_bf16_parts(which, bad, where):
    def spoil(w, t):
        w.copy_(w.sign() * w.abs().clamp(min=0.01))
        if where == "input":
            t[0, 3, 4, 10] = t[-1, 5, -1, -1] = bad
        else:
            w[5, 7, 1, 2] = bad

    got, want = _slab(which, 2, 3, 70, 70, 30, 187, spoil=spoil)
    want32 = want.float().double()  # beyond fp32: infinite
    assert torch.equal(got.isnan(), want32.isnan())
    far = want32.isinf() | (want.abs() > 3.3e38)  # (which side of the largest number a sum near it falls on is its rounding's)
    assert torch.equal(got[want32.isinf() & (bad != 3.4e38)], want32[want32.isinf() & (bad != 3.4e38)])
    large = (want.abs() > 1e30) & ~far
    assert ((got - want)[large].abs() <= 2e-6 * want[large].abs()).all()
    fine = want.abs() <= 1e30
    assert fine.any() and (~fine).any()
    # 630 terms of 24 bits in one chain of 27 sums, each rounded (2^-24, random in sign) at the size it has by then
    assert (got - want)[fine].norm() <= 2.0 ** -24 * 27 ** 0.5 * 2 * want[fine].norm()


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_filter_gradient_of_values_without_finite_bf16_parts(bad):
    N, Cin, Cout, H, W = 1, 20, 40, 6, 21
    g = torch.Generator().manual_seed(8)
    x, dy = torch.rand((N, Cin, H, W), generator=g) + 0.5, torch.rand((N, Cout, H, W), generator=g) + 0.5
    ws = torch.empty(capi.conv_workspace_bytes(capi.ADH_CONV_BWD_FILTER, capi.ADH_F32, 1, N, Cin, Cout, H, W) // 4, device="cuda")
    for where in ("input", "gradient"):
        xb, db = x.clone(), dy.clone()
        (xb[0, 3, 2] if where == "input" else db[0, 30, 4])[10] = bad
        dw = torch.empty((Cout, Cin, 3, 3), device="cuda")
        capi.check(capi.conv_unpadded_bwd_filter_tiles([xb.cuda()], [db.cuda()], dw, N, Cin, Cout, H, W, ws=ws), "bwd-filter")
        xp = torch.nn.functional.pad(xb, (1, 1, 1, 1))
        want = torch.stack([torch.stack([(db[:, :, None] * xp[:, None, :, a:a + H, b:b + W]).sum((0, 3, 4)) for b in range(3)], -1)
                            for a in range(3)], -2)
        got = dw.cpu()
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        assert torch.equal(torch.isinf(got), torch.isinf(want))
        fine = torch.isfinite(want)
        assert ((got[fine].double() - want[fine].double()).abs() <= 2e-6 * want[fine].double().abs()).all()
        assert fine.any() and not fine.all()


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("halo", [False, True])
@pytest.mark.parametrize("K,H,W", [(1, 6, 56), (1, 7, 21), (3, 5, 32), (1, 9, 8), (2, 1, 13)])
def test_filter_gradient_of_a_bad_value_at_the_border(K, H, W, halo, bad):
    """A step of the kernel multiplies pixels past the last column and row of dy, which are zero, with what x has beside them: a
    NaN there belongs to the taps that reach it from a pixel that exists, and to no other."""
    N, Cin, Cout = 2, 20, 40
    g = torch.Generator().manual_seed(9)
    p = 1 if halo else 0
    x, dy = torch.rand((K, N, Cin, H + 2 * p, W + 2 * p), generator=g) + 0.5, torch.rand((K, N, Cout, H, W), generator=g) + 0.5
    ws = torch.empty(capi.conv_workspace_bytes(capi.ADH_CONV_BWD_FILTER, capi.ADH_F32, K, N, Cin, Cout, H, W) // 4, device="cuda")
    fn = capi.conv_bwd_filter_tiles if halo else capi.conv_unpadded_bwd_filter_tiles
    for row, col in ((0, -1), (-1, 0), (-1, -1), (H // 2, W // 2), (0, 0), (0, -2), (-2, 0)):
        if not (-x.shape[3] <= row and -x.shape[4] <= col):
            continue
        xb = x.clone()
        xb[K - 1, 1, 3, row, col] = bad
        dw = torch.empty((Cout, Cin, 3, 3), device="cuda")
        capi.check(fn(list(xb.cuda()), list(dy.cuda()), dw, N, Cin, Cout, H, W, ws=ws), "bwd-filter")
        if halo:
            xp, d, h = xb.transpose(0, 1).reshape(N, K, Cin, H + 2, W + 2), dy.transpose(0, 1), H
        else:  # the row tiles of one tensor
            h = K * H
            xp = torch.nn.functional.pad(torch.cat(list(xb), 2), (1, 1, 1, 1))[:, None]
            d = torch.cat(list(dy), 2)[:, None]
        want = torch.stack([torch.stack([(d.double()[:, :, :, None] * xp.double()[:, :, None, :, a:a + h, b:b + W]).sum((0, 1, 4, 5))
                                         for b in range(3)], -1) for a in range(3)], -2)
        got = dw.cpu()
        assert torch.equal(torch.isnan(got), torch.isnan(want)), (row, col)
        assert torch.equal(torch.isinf(got), torch.isinf(want)), (row, col)
        fine = torch.isfinite(want)
        # positive sums of K N H W terms, each addition rounded once
        assert ((got[fine].double() - want[fine]).abs() <= (K * N * H * W + 4) * 2.0 ** -24 * want[fine]).all() and fine.any()


@pytest.mark.parametrize("K,N,Cin,Cout,H,W", [(5, 4, 128, 64, 7, 7), (1, 1, 65, 65, 3, 5), (2, 3, 20, 100, 9, 33), (1, 2, 40, 30, 4, 4), (1, 1, 3, 5, 2, 2)])
def test_filter_gradient_in_a_small_workspace(K, N, Cin, Cout, H, W):
    """A workspace below the query's answer: fewer workgroups share the pixels, then the channel groups run in turn."""
    g = torch.Generator().manual_seed(10)
    x, dy = torch.rand((N, Cin, K * H, W), generator=g) * 2 - 1, torch.randn((N, Cout, K * H, W), generator=g)
    want = torch.nn.grad.conv2d_weight(x.double(), (Cout, Cin, 3, 3), dy.double(), padding=1).numpy()
    xs, dys = _tiles(x.cuda(), K), _tiles(dy.cuda(), K)
    unit = 4 * 9 * 1024 * (2 if Cin > 32 else 1) * (2 if Cout > 32 else 1)  # a workgroup's sums
    groups = -(-Cin // 64) * -(-Cout // 64)
    full = capi.conv_workspace_bytes(capi.ADH_CONV_BWD_FILTER, capi.ADH_F32, K, N, Cin, Cout, H, W)
    for nbytes in {unit, groups * unit - 4, groups * unit, 2 * groups * unit + 4, full // 2, full}:
        if not unit <= nbytes <= full:
            continue
        ws = torch.full((nbytes // 4 + 64,), 7.0, device="cuda")
        dw = torch.ones((Cout, Cin, 3, 3), device="cuda")
        capi.check(capi.conv_unpadded_bwd_filter_tiles(xs, dys, dw, N, Cin, Cout, H, W, beta=1.0, ws=ws[:nbytes // 4]), "bwd-filter")
        assert rel_err(host(dw), want + 1.0) <= 1e-5, nbytes
        assert (ws[nbytes // 4:] == 7.0).all()
    dw = torch.ones((Cout, Cin, 3, 3), device="cuda")
    small = torch.empty(unit // 4 - 1, device="cuda")
    assert capi.conv_unpadded_bwd_filter_tiles(xs, dys, dw, N, Cin, Cout, H, W, ws=small) == capi.ADH_EWORKSPACE
