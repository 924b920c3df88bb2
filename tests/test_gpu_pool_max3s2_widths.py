"""3x3 max pooling at stride 2 over tiles without halo at any row length, forward and backward, by the kernels that keep
their windows in registers: every remainder of a group of columns (4 fp32, 8 bf16), rows of one group, bit for bit against the
banded kernels, which serve the same pooling over one halo-padded tile."""
import pytest
import torch
import torch.nn.functional as F

from arraydiff_cuda_amd import capi

pytestmark = pytest.mark.gpu

WINDOW = (3, 3, 2, 2)


def _inputs(dtype, K, N, C, Ht, W, seed):
    """Values of few levels, so that most windows have ties, and some special ones."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randint(-2, 3, (N, C, Ht * K, W), generator=g).float()
    special = torch.tensor([float("inf"), -float("inf"), float("nan"), torch.finfo(dtype).min, -0.0])
    where = torch.rand(x.shape, generator=g) < 0.2
    x[where] = special[torch.randint(0, 5, (int(where.sum()),), generator=g)]
    dy = torch.randn((N, C, Ht * K // 2, (W - 1) // 2 + 1), generator=g)
    return x.to(dtype).cuda(), dy.to(dtype).cuda()


def _same(a, b):
    return torch.equal(a.nan_to_num(nan=123.0), b.nan_to_num(nan=123.0)) and torch.equal(torch.signbit(a), torch.signbit(b))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("W", [4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17, 31, 255, 350, 515])
@pytest.mark.parametrize("K,Ht", [(1, 6), (3, 8)])
@pytest.mark.parametrize("beta", [0.0, 1.0])
def test_same_as_the_banded_kernels(dtype, W, K, Ht, beta):
    N, C, H, OW = 2, 700 if W < 32 else 40, Ht * K, (W - 1) // 2 + 1  # (below 2^15 pixels the bands serve both)
    x, dy = _inputs(dtype, K, N, C, Ht, W, W)
    xs = [t.contiguous() for t in x.chunk(K, 2)]
    dys = [t.contiguous() for t in dy.chunk(K, 2)]
    ys = [torch.full_like(t, 7.0) for t in dys]
    old = torch.randint(-4, 5, x.shape, generator=torch.Generator().manual_seed(9)).to(dtype).cuda()
    dxs = [t.clone().contiguous() for t in old.chunk(K, 2)]
    capi.check(capi.pool_unpadded_fwd_tiles(capi.ADH_POOL_MAX, xs, ys, N, C, Ht, W, *WINDOW, 1, 1), "forward")
    capi.check(capi.pool_unpadded_bwd_tiles(capi.ADH_POOL_MAX, xs, None, dys, dxs, N, C, Ht, W, *WINDOW, 1, 1, beta=beta), "backward")
    padded = F.pad(x, (1, 1, 1, 1))
    want_y, want_dx = torch.empty((N, C, H // 2, OW), device="cuda", dtype=dtype), F.pad(old, (1, 1, 1, 1))
    capi.check(capi.pool_fwd_tiles(capi.ADH_POOL_MAX, [padded], [want_y], N, C, H + 2, W + 2, *WINDOW), "padded forward")
    capi.check(capi.pool_bwd_tiles(capi.ADH_POOL_MAX, [padded], [want_y], [dy], [want_dx], N, C, H + 2, W + 2, *WINDOW, beta=beta), "padded backward")
    assert _same(torch.cat(ys, 2), want_y)
    assert _same(torch.cat(dxs, 2), want_dx[:, :, 1:-1, 1:-1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_larger_than_the_cache(dtype):
    """Where the accesses are non-temporal."""
    N, C, Ht, W, K = 2, 33, 512 if dtype is torch.float32 else 1024, 1100, 2
    x, dy = _inputs(dtype, K, N, C, Ht, W, 3)
    assert x.numel() * x.element_size() > 256 << 20
    xs = [t.contiguous() for t in x.chunk(K, 2)]
    dys = [t.contiguous() for t in dy.chunk(K, 2)]
    ys, dxs = [torch.empty_like(t) for t in dys], [torch.empty_like(t) for t in xs]
    capi.check(capi.pool_unpadded_fwd_tiles(capi.ADH_POOL_MAX, xs, ys, N, C, Ht, W, *WINDOW, 1, 1), "forward")
    capi.check(capi.pool_unpadded_bwd_tiles(capi.ADH_POOL_MAX, xs, None, dys, dxs, N, C, Ht, W, *WINDOW, 1, 1), "backward")
    for n in range(N):  # one image is small enough for the cache
        small, sdy = [t[n:n + 1].contiguous() for t in xs], [t[n:n + 1].contiguous() for t in dys]
        y1, d1 = [torch.empty_like(t) for t in sdy], [torch.empty_like(t) for t in small]
        capi.check(capi.pool_unpadded_fwd_tiles(capi.ADH_POOL_MAX, small, y1, 1, C, Ht, W, *WINDOW, 1, 1), "forward")
        capi.check(capi.pool_unpadded_bwd_tiles(capi.ADH_POOL_MAX, small, None, sdy, d1, 1, C, Ht, W, *WINDOW, 1, 1), "backward")
        for t in range(K):
            assert _same(ys[t][n:n + 1], y1[t]) and _same(dxs[t][n:n + 1], d1[t])


@pytest.mark.parametrize("W", [8, 9, 11, 13, 15, 16, 17, 22, 255, 520])
def test_eight_columns_a_thread(W):
    """bf16 tensors of 24 MB and more: the same bits as image by image, by fours."""
    N, K, Ht = 3, 2, 10
    C = (26 << 20) // (2 * N * K * Ht * W) + 1
    g = torch.Generator(device="cuda").manual_seed(W)
    x = torch.randint(-2, 3, (N, C, K * Ht, W), device="cuda", generator=g).bfloat16()
    special = torch.tensor([float("inf"), -float("inf"), float("nan"), torch.finfo(torch.bfloat16).min, -0.0], device="cuda").bfloat16()
    x = torch.where(torch.rand(x.shape, device="cuda", generator=g) < 0.2, special[torch.randint(0, 5, x.shape, device="cuda", generator=g)], x)
    dy = torch.randn((N, C, K * Ht // 2, (W - 1) // 2 + 1), device="cuda", generator=g).bfloat16()

    def run(x, dy, old):
        xs, dys, dxs = ([t.clone(memory_format=torch.contiguous_format) for t in v.chunk(K, 2)] for v in (x, dy, old))
        ys = [torch.full_like(t, 7.0) for t in dys]
        capi.check(capi.pool_unpadded_fwd_tiles(capi.ADH_POOL_MAX, xs, ys, x.shape[0], C, Ht, W, *WINDOW, 1, 1), "forward")
        capi.check(capi.pool_unpadded_bwd_tiles(capi.ADH_POOL_MAX, xs, None, dys, dxs, x.shape[0], C, Ht, W, *WINDOW, 1, 1, beta=1.0), "backward")
        return torch.cat(ys, 2), torch.cat(dxs, 2)

    old = torch.randint(-4, 5, x.shape, device="cuda", generator=g).bfloat16()
    y, dx = run(x, dy, old)
    for n in range(N):
        y1, dx1 = run(x[n:n + 1], dy[n:n + 1], old[n:n + 1])
        assert _same(y[n:n + 1], y1) and _same(dx[n:n + 1], dx1)


@pytest.mark.parametrize("W", [256, 260])
@pytest.mark.parametrize("offset", [0, 1])
def test_larger_than_the_cache_at_any_alignment(W, offset):
    """Forward, fp32, rows of whole lines and of whole 16-byte groups: off 16 bytes the same bits as image by image, and no more
    than 1.7 times as long (1.1 and 1.2 without LDS; the bands, which would stage element by element, 2.1 times)."""
    N, C, Ht, K = 18, 64, 64, 4

    def off(t, by):
        flat = torch.empty(t.numel() + 4, device="cuda")[by:by + t.numel()].view(t.shape)
        return flat.copy_(t)

    def run(xs, ys):
        capi.check(capi.pool_unpadded_fwd_tiles(capi.ADH_POOL_MAX, xs, ys, xs[0].shape[0], C, Ht, W, *WINDOW, 1, 1), "forward")

    def fastest(xs, ys):
        run(xs, ys)
        events = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(10)]
        for a, b in events:
            a.record()
            run(xs, ys)
            b.record()
        torch.cuda.synchronize()
        return min(a.elapsed_time(b) for a, b in events)

    x, _ = _inputs(torch.float32, K, N, C, Ht, W, 5)
    assert x.numel() * 4 > 256 << 20
    aligned = [t.contiguous() for t in x.chunk(K, 2)]
    xs = [off(t, offset) for t in aligned]
    ys = [off(torch.full((N, C, Ht // 2, W // 2), 7.0, device="cuda"), offset) for _ in xs]
    run(xs, ys)
    for n in range(0, N, 5):
        small = [t[n:n + 1].contiguous() for t in aligned]
        y1 = [torch.empty_like(y[n:n + 1]).contiguous() for y in ys]
        run(small, y1)
        assert all(_same(ys[t][n:n + 1], y1[t]) for t in range(K))
    if offset:
        assert fastest(xs, ys) < 1.7 * fastest(aligned, [torch.empty_like(y).contiguous() for y in ys])
