"""Sums of fp32 products on the bf16 matrix cores are as close to double precision as fp32 sums taken term by term, in every pass:
few channels and many, chunks that are full and such that are not, signed and rectified inputs.  And what is left of values
near the smallest ones."""
import pytest
import torch

from arraydiff_cuda_amd import capi

pytestmark = pytest.mark.gpu


def _data(N, Cin, Cout, H, W, k, s, pad, kind):
    g = torch.Generator().manual_seed(12)
    x = torch.rand((N, Cin, H, W), generator=g) * 2 - 1 if kind == "uniform" else torch.relu(torch.randn((N, Cin, H, W), generator=g))
    w = torch.randn((Cout, Cin, k, k), generator=g) * (2.0 / (Cin * k * k)) ** 0.5
    dy = torch.randn((N, Cout, (H + 2 * pad - k) // s + 1, (W + 2 * pad - k) // s + 1), generator=g)
    return x.cuda(), w.cuda(), dy.cuda()


def _sums(x, w, dy, s, pad, dtype):
    """y, dx and dw, one term after another, each addition rounded to `dtype` (the products are exact in double precision)."""
    N, Cin, H, W = x.shape
    Cout, k, (OH, OW) = w.shape[0], w.shape[2], dy.shape[2:]
    cols = torch.nn.functional.unfold(torch.nn.functional.pad(x, (pad,) * 4).double(), k, stride=s)  # [N][Cin k k][pixel]
    wd, dd = w.double().reshape(Cout, -1), dy.double().reshape(N, Cout, -1)
    y = torch.zeros((N, Cout, OH * OW), dtype=dtype, device="cuda")
    for t in range(cols.shape[1]):
        y = (y.double() + wd[None, :, t, None] * cols[:, None, t]).to(dtype)
    dw = torch.zeros((Cout, Cin * k * k), dtype=dtype, device="cuda")
    for n in range(N):
        for p in range(OH * OW):
            dw = (dw.double() + dd[n, :, None, p] * cols[n, None, :, p]).to(dtype)
    dx = torch.zeros((N, Cin, H + 2 * pad, W + 2 * pad), dtype=dtype, device="cuda")
    for co in range(Cout):
        for a in range(k):
            for b in range(k):
                at = dx[:, :, a:a + (OH - 1) * s + 1:s, b:b + (OW - 1) * s + 1:s]
                at.copy_((at.double() + w.double()[None, co, :, a, b, None, None] * dy.double()[:, co, None]).to(dtype))
    return y.reshape(dy.shape), dx[:, :, pad:pad + H, pad:pad + W], dw.reshape(w.shape)


def _passes(x, w, dy, k, s, pad):
    N, Cin, H, W = x.shape
    Cout = w.shape[0]
    geo = (k, k, s, s, 1, 1) + ((pad, pad) if pad else ())
    ws = lambda which: torch.empty((capi.conv2d_unpadded_workspace_bytes if pad else capi.conv2d_workspace_bytes)(
        which, capi.ADH_F32, 1, N, Cin, Cout, H, W, *geo) // 4 + 64, device="cuda")
    y, dx, dw = torch.empty_like(dy), torch.empty_like(x), torch.empty_like(w)
    fwd, bwd, wgrad = ((capi.conv2d_unpadded_fwd_tiles, capi.conv2d_unpadded_bwd_data_tiles, capi.conv2d_unpadded_bwd_filter_tiles) if pad
                       else (capi.conv2d_fwd_tiles, capi.conv2d_bwd_data_tiles, capi.conv2d_bwd_filter_tiles))
    capi.check(fwd([x], w, [y], N, Cin, Cout, H, W, *geo, ws=ws(capi.ADH_CONV_FWD)), "fwd")
    capi.check(bwd(w, [dy], [dx], N, Cin, Cout, H, W, *geo, ws=ws(capi.ADH_CONV_BWD_DATA)), "bwd-data")
    capi.check(wgrad([x], [dy], dw, N, Cin, Cout, H, W, *geo, ws=ws(capi.ADH_CONV_BWD_FILTER)), "bwd-filter")
    return y, dx, dw


@pytest.mark.parametrize("kind", ["uniform", "rectified"])
@pytest.mark.parametrize("Cin,Cout,k,s,pad", [(1, 64, 3, 1, 1), (3, 40, 3, 1, 1), (5, 33, 3, 1, 1), (16, 16, 3, 1, 1), (40, 20, 3, 1, 1), (64, 64, 3, 1, 1),
                                              (2, 3, 3, 2, 1), (16, 48, 3, 2, 1), (64, 16, 3, 2, 1), (3, 64, 7, 1, 0), (3, 48, 7, 2, 0), (1, 16, 3, 1, 0),
                                              (20, 48, 1, 1, 0), (70, 33, 1, 2, 0)])
def test_sums_are_as_close_to_double_precision_as_fp32_ones(Cin, Cout, k, s, pad, kind):
    x, w, dy = _data(2, Cin, Cout, 16, 24, k, s, pad, kind)
    want, plain, got = _sums(x, w, dy, s, pad, torch.float64), _sums(x, w, dy, s, pad, torch.float32), _passes(x, w, dy, k, s, pad)
    err = lambda a, b: ((a.double() - b).norm() / b.norm()).item()
    for name, v, p, t in zip(("fwd", "bwd-data", "bwd-filter"), got, plain, want):
        if name == "bwd-data" and k > 3:
            continue  # on the fp32 matrix cores
        assert err(v, t) <= err(p, t), (name, err(v, t), err(p, t))


@pytest.mark.parametrize("kind", ["uniform", "rectified"])
@pytest.mark.parametrize("Cin,Cout", [(3, 64), (33, 40), (40, 33), (64, 64), (100, 64)])
def test_persistent_workgroups_sums(Cin, Cout, kind):
    """Layers beyond what conv_f32_patch.hip takes (2.1 M results), forward and backward-data."""
    H = W = 96
    N = 2100000 // (min(Cin, Cout) * H * W) + 1
    x, w, dy = _data(N, Cin, Cout, H, W, 3, 1, 1, kind)
    geo = (3, 3, 1, 1, 1, 1, 1, 1)
    for name, which, t, out, M in (("fwd", capi.ADH_CONV_FWD, x, dy, Cout), ("bwd-data", capi.ADH_CONV_BWD_DATA, dy, x, Cin)):
        assert "conv3x3_split_kernel" in capi.conv_kernel_name(which, capi.ADH_F32, 1, N, Cin, Cout, H, W)
        f = (w if which == capi.ADH_CONV_FWD else w.transpose(0, 1).flip(2, 3)).reshape(M, -1).double()
        sums = {}
        for dtype in (torch.float64, torch.float32):
            at = sums[dtype] = torch.zeros((N, M, H * W), dtype=dtype, device="cuda")
            tp = torch.nn.functional.pad(t, (1,) * 4).double()
            for c in range(t.shape[1]):
                for a in range(9):
                    col = tp[:, c, a // 3:a // 3 + H, a % 3:a % 3 + W].reshape(N, 1, -1)
                    at.copy_((at.double() + f[None, :, c * 9 + a, None] * col).to(dtype))
        got = torch.empty((N, M, H, W), device="cuda")
        ws = torch.empty(capi.conv2d_unpadded_workspace_bytes(which, capi.ADH_F32, 1, N, Cin, Cout, H, W, *geo) // 4 + 64, device="cuda")
        if which == capi.ADH_CONV_FWD:
            capi.check(capi.conv2d_unpadded_fwd_tiles([x], w, [got], N, Cin, Cout, H, W, *geo, ws=ws), name)
        else:
            capi.check(capi.conv2d_unpadded_bwd_data_tiles(w, [dy], [got], N, Cin, Cout, H, W, *geo, ws=ws), name)
        err = lambda v: ((v.double().reshape(N, M, -1) - sums[torch.float64]).norm() / sums[torch.float64].norm()).item()
        assert err(got) <= err(sums[torch.float32]), (name, err(got), err(sums[torch.float32]))


@pytest.mark.parametrize("Cin,Cout,k,s,pad", [(5, 33, 3, 1, 1), (64, 64, 3, 1, 1), (16, 48, 3, 2, 1), (3, 48, 7, 2, 0), (20, 48, 1, 1, 0), (70, 33, 1, 2, 0)])
@pytest.mark.parametrize("scale", [2.0 ** -109, 2.0 ** -118])
def test_values_near_the_smallest(Cin, Cout, k, s, pad, scale):
    """Three bf16 parts hold a value down to 2^-134: an input of 2^-110 and more whole, a smaller one to that much."""
    x, w, dy = _data(2, Cin, Cout, 16, 24, k, s, pad, "uniform")
    x = torch.where(x.abs() < 0.5, x + torch.sign(x) * 0.5, x)  # from half the scale on
    dy = torch.where(dy.abs() < 0.5, dy + torch.sign(dy) * 0.5, dy)
    for side in ("input", "gradient"):
        xs, ds = (x * scale, dy) if side == "input" else (x, dy * scale)
        want, size = _sums(xs, w, ds, s, pad, torch.float64), _sums(xs.abs(), w.abs(), ds.abs(), s, pad, torch.float64)
        one = torch.ones_like
        lost = 2.0 ** -134 if scale < 2.0 ** -109 else 0.0
        got = _passes(xs, w, ds, k, s, pad)
        for i, name in enumerate(("fwd", "bwd-data", "bwd-filter")):
            if (side, name) in (("input", "bwd-data"), ("gradient", "fwd")):
                continue
            terms = (Cin * k * k, Cout * k * k, dy.numel() // Cout)[i]
            # a value's lost part times the other operand's sizes, and fp32 sums' roundings
            other = (_sums(one(xs), w.abs(), one(ds), s, pad, torch.float64)[i] if i < 2 else
                     _sums(one(xs), one(w), ds.abs(), s, pad, torch.float64)[2] if side == "input" else
                     _sums(xs.abs(), one(w), one(ds), s, pad, torch.float64)[2])
            bound = lost * other + terms * 2.0 ** -24 * size[i]
            assert ((got[i].double() - want[i]).abs() <= bound).all(), (side, name)
