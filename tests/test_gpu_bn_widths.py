"""Batch norm at the row and plane lengths where the vectorised passes can go wrong: planes that are no whole number of
16-byte groups, padded gradients with odd rows, gradients written over their input, channels of many splits, and tensors
larger than the on-package cache (non-temporal accesses), against float64."""
import pytest
import torch

from arraydiff_cuda_amd import capi

pytestmark = pytest.mark.gpu
EPS = 1e-5


def _reference(x, dy, scale, shift):
    x, dy = x.double(), dy.double()
    mean = x.mean((0, 2, 3), keepdim=True)
    xhat = (x - mean) / torch.sqrt(x.var((0, 2, 3), unbiased=False, keepdim=True) + EPS)
    y = xhat * scale.double().view(1, -1, 1, 1) + shift.double().view(1, -1, 1, 1)
    d = torch.where(y > 0, dy, torch.zeros_like(dy))
    m = d.mean((0, 2, 3), keepdim=True)
    k = (d * xhat).mean((0, 2, 3), keepdim=True)
    dx = (d - m - xhat * k) * scale.double().view(1, -1, 1, 1) / torch.sqrt(x.var((0, 2, 3), unbiased=False, keepdim=True) + EPS)
    return y, dx, (d * xhat).sum((0, 2, 3)), d.sum((0, 2, 3))


def _close(got, want, rel):
    assert (got.double() - want).norm() <= rel * want.norm() + 1e-30


def _run(dtype, K, N, C, H, W, p=0, beta=0.0, over_dy=False):
    g = torch.Generator(device="cuda").manual_seed(H * W + C)
    xs = [(torch.randn((N, C, H, W), device="cuda", generator=g) + torch.randn((1, C, 1, 1), device="cuda", generator=g)).to(dtype) for _ in range(K)]
    dys = [torch.randn((N, C, H, W), device="cuda", generator=g).to(dtype) for _ in range(K)]
    scales = [torch.rand((C,), device="cuda", generator=g) + 0.5 for _ in range(K)]
    shifts = [torch.randn((C,), device="cuda", generator=g) * 0.1 for _ in range(K)]
    # within rounding of zero the rectifier may fall either way (1e-5: some 100 roundings of values of order 1): no gradient there
    for x, d, a, b in zip(xs, dys, scales, shifts):
        d[_reference(x, d, a, b)[0].abs() <= 1e-5] = 0
    # (dy beyond the interior must not be read into the sums)
    padded = [torch.full((N, C, H + 2 * p, W + 2 * p), float("nan"), device="cuda", dtype=dtype) for _ in range(K)]
    for t, d in zip(padded, dys):
        t[:, :, p:p + H, p:p + W] = d
    vec = lambda: [torch.empty((C,), device="cuda") for _ in range(K)]
    means, invs, dscales, dshifts = vec(), vec(), vec(), vec()
    ys = [torch.full((N, C, H, W), 9.0, device="cuda", dtype=dtype) for _ in range(K)]
    olds = [torch.randn((N, C, H, W), device="cuda", generator=g).to(dtype) for _ in range(K)]
    dxs = padded if over_dy else [o.clone() for o in olds]
    ws = torch.empty(capi.batchnorm_workspace_bytes(K, N, C) // 4 + 64, device="cuda")
    capi.check(capi.batchnorm_fwd_tiles(xs, scales, shifts, ys, N, C, H, W, relu=1, run_means=vec(), run_vars=vec(), save_means=means,
                                        save_invstds=invs, ws=ws), "forward")
    capi.check(capi.batchnorm_bwd_tiles(xs, padded, scales, shifts, means, invs, dxs, dscales, dshifts, N, C, H, W, relu=1, dy_halo=p,
                                        beta_data=beta, ws=ws), "backward")
    # one rounding of a result to bf16; fp32: sums over the channel in another order
    rel = 4e-3 if dtype is torch.bfloat16 else 2e-6
    for k in range(K):
        y, dx, dscale, dshift = _reference(xs[k], dys[k], scales[k], shifts[k])
        _close(ys[k], y.clamp(min=0), rel)
        _close(dxs[k], dx + (olds[k].double() if beta else 0.0), rel)
        _close(dscales[k], dscale, 2e-5)
        _close(dshifts[k], dshift, 2e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,W", [(1, 7), (1, 9), (2, 11), (3, 21), (5, 13), (1, 65), (2, 33), (4, 129), (3, 257), (9, 455), (64, 67)])
@pytest.mark.parametrize("p", [0, 1, 3])
@pytest.mark.parametrize("beta", [0.0, 1.0])
def test_lengths(dtype, H, W, p, beta):
    _run(dtype, 2, 3, 5, H, W, p, beta)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,W", [(1, 9), (5, 13), (4, 129), (64, 67)])
def test_gradient_over_its_input(dtype, H, W):
    _run(dtype, 2, 3, 5, H, W, over_dy=True)


def _many(H, W, dtype):
    """Channels of 2 tiles of 16 images that are more than a workgroup per compute unit by 16-byte groups (as the apply pass deals them)."""
    groups = -(-H * W // (4 if dtype is torch.float32 else 8))
    threads = 256 if groups > 128 else max(16, 1 << (groups - 1).bit_length())
    return 256 * 4 * (256 // threads) // 32 + 3


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,W", [(5, 13), (1, 65), (2, 33), (4, 129), (64, 67), (3, 257)])
@pytest.mark.parametrize("p,beta", [(0, 0.0), (0, 1.0), (1, 1.0)])
def test_lengths_by_groups(dtype, H, W, p, beta):
    _run(dtype, 2, 16, _many(H, W, dtype), H, W, p, beta)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,W", [(5, 13), (4, 129), (64, 67)])
def test_gradient_over_its_input_by_groups(dtype, H, W):
    _run(dtype, 2, 16, _many(H, W, dtype), H, W, over_dy=True)


@pytest.mark.parametrize("K,N,C", [(1, 37, 1), (1, 70, 3), (2, 9, 130)])
def test_splits(K, N, C):
    _run(torch.float32, K, N, C, 6, 11)


@pytest.mark.parametrize("dtype,W", [(torch.float32, 1100), (torch.float32, 1099), (torch.bfloat16, 2200), (torch.bfloat16, 2199)])
def test_larger_than_the_cache(dtype, W):
    _run(dtype, 2, 2, 33, 512, W)


def test_more_planes_than_workgroups_of_a_launch():
    """2^24 planes of more than 1024 groups (16 tiles that share their memory): a workgroup per plane would be 2^32 threads."""
    K, N, C, H, W = capi.ADH_MAX_TILES, 1024, 1024, 94, 11
    g = torch.Generator(device="cuda").manual_seed(2)
    x = torch.randn((N, C, H, W), device="cuda", generator=g, dtype=torch.bfloat16)
    dy = torch.randn((N, C, H + 2, W + 2), device="cuda", generator=g, dtype=torch.bfloat16)
    dx = torch.full((N, C, H, W), 7.0, device="cuda", dtype=torch.bfloat16)
    scale, mean, invstd = torch.rand(C, device="cuda", generator=g) + 0.5, torch.randn(C, device="cuda", generator=g) * 0.1, torch.rand(C, device="cuda", generator=g) + 0.5
    dscale, dshift = torch.empty(C, device="cuda"), torch.empty(C, device="cuda")
    ws = torch.empty(capi.batchnorm_workspace_bytes(K, N, C) // 4, device="cuda")
    capi.check(capi.batchnorm_bwd_tiles([x] * K, [dy] * K, [scale] * K, [scale] * K, [mean] * K, [invstd] * K, [dx] * K, [dscale] * K, [dshift] * K, N, C, H, W,
                                        dy_halo=1, ws=ws))
    for c in (0, 1, 700, C - 1):
        xc, d = x[:, c].double() - mean[c].double(), dy[:, c, 1:-1, 1:-1].double()
        i, m = invstd[c].double(), N * H * W
        want = scale[c].double() * i * (d - d.sum() / m - xc * i * (d * xc * i).sum() / m)
        # rounded to bf16, and sums of a million fp32 terms behind the small corrections
        assert ((dx[:, c].double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all()
