"""bf16 3x3 strips over rows that start on any element: odd widths forward, widths that are no whole granules backward-data, where
the staged rows begin one element off and granules hold the ends of neighbouring rows, against float64."""
import pytest
import torch

from arraydiff_cuda_amd import capi

pytestmark = pytest.mark.gpu

# (strips: the smallest tiles that patches don't take; one and several launches, channels off 64 and 128, heights off four rows)
FWD = [(4, 4, 64, 64, 34, 255), (4, 8, 61, 64, 34, 127), (2, 3, 1, 144, 64, 255), (8, 2, 128, 128, 34, 127), (8, 2, 128, 128, 64, 65),
       (8, 8, 128, 256, 16, 33), (4, 1, 66, 320, 34, 255), (8, 4, 96, 96, 34, 127), (4, 1, 128, 128, 64, 257)]
BWD = [(4, 6, 64, 64, 16, 255), (4, 12, 61, 64, 16, 127), (8, 12, 64, 64, 16, 132), (4, 8, 48, 48, 64, 130), (8, 3, 128, 128, 16, 127),
       (4, 6, 128, 128, 34, 65), (4, 6, 128, 128, 34, 70), (4, 8, 192, 128, 34, 33), (4, 4, 130, 128, 16, 132), (2, 3, 320, 66, 16, 255),
       (8, 1, 384, 256, 16, 255), (8, 3, 384, 256, 16, 132), (4, 6, 128, 128, 33, 132)]


def _correlate(x, w):
    """Valid correlation of (N, Ci, H, W) with (Co, Ci, 3, 3) in float64."""
    H, W = x.shape[2] - 2, x.shape[3] - 2
    y = 0
    for i in range(3):
        for j in range(3):
            y = y + torch.matmul(w[:, :, i, j].contiguous(), x[:, :, i:i + H, j:j + W].reshape(x.shape[0], x.shape[1], H * W))
    return y.reshape(x.shape[0], w.shape[0], H, W)


@pytest.mark.parametrize("beta", [0.0, 1.0])
@pytest.mark.parametrize("which,K,N,Cin,Cout,H,W", [("fwd",) + s for s in FWD] + [("bwd",) + s for s in BWD])
def test_vs_float64(which, K, N, Cin, Cout, H, W, beta):
    fwd = which == "fwd"
    code = capi.ADH_CONV_FWD if fwd else capi.ADH_CONV_BWD_DATA
    name = capi.conv_kernel_name(code, capi.ADH_BF16, K, N, Cin, Cout, H, W, beta)
    assert "w8" in name or "k128" in name, name
    g = torch.Generator(device="cuda").manual_seed(W * 31 + Cin)
    bf = lambda shape: torch.randn(shape, generator=g, device="cuda").to(torch.bfloat16)
    w = (bf((Cout, Cin, 3, 3)).float() * (2.0 / (9 * (Cin if fwd else Cout))) ** 0.5).to(torch.bfloat16)
    ins = [bf((N, Cin, H + 2, W + 2) if fwd else (N, Cout, H, W)) for _ in range(K)]
    olds = [bf((N, Cout, H, W) if fwd else (N, Cin, H + 2, W + 2)) for _ in range(K)]
    # infinite at one end of some rows: only the outputs that reach it may see it
    ins[0][:, :, 5, 0] = float("inf")
    ins[-1][:, :, 8, -1] = float("inf")
    outs = [t.clone() if beta else torch.full_like(t, float("nan")) for t in olds]
    ws = torch.empty(capi.conv_workspace_bytes(code, capi.ADH_BF16, K, N, Cin, Cout, H, W) // 4 + 64, device="cuda")
    if fwd:
        capi.check(capi.conv_fwd_tiles(ins, w, outs, N, Cin, Cout, H, W, beta=beta, ws=ws), name)
    else:
        capi.check(capi.conv_bwd_data_tiles(w, ins, outs, N, Cin, Cout, H, W, beta=beta, ws=ws), name)
    filt = w.double() if fwd else w.double().flip(2, 3).transpose(0, 1)
    for k in range(K):
        src = ins[k].double()
        if not fwd:
            src = torch.nn.functional.pad(src, (2, 2, 2, 2))
        want = _correlate(src, filt) + (olds[k].double() if beta else 0.0)
        far = torch.isfinite(want)
        got = outs[k].double()
        assert far.float().mean() > 0.8 and bool(torch.isfinite(got[far]).all())
        err, ref = (got - want)[far].abs(), want[far].abs()
        # one rounding to bf16 (at most 2^-8 of the value) of fp32 sums of at most 2304 terms, added to an old value of bf16
        assert bool((err <= 2.0 ** -8 * 1.001 * ref + 2e-5 * (1 + ref.max())).all()), err.max()


@pytest.mark.parametrize("which,C,W,at", [("fwd", 128, 255, 1), ("bwd", 128, 255, 1), ("bwd", 128, 130, 1), ("fwd", 128, 255, 2),
                                          ("fwd", 320, 129, 2), ("fwd", 192, 129, 2), ("fwd", 64, 129, 2)])
def test_tiles_off_16_bytes(which, C, W, at):
    """Tiles `at` elements off 16 bytes: over copies, or (forward, on 4 bytes, no room for copies) strips over rows as they lie."""
    K, N, H = 2, 3, 34
    fwd = which == "fwd"
    g = torch.Generator(device="cuda").manual_seed(2)
    bf = lambda shape: torch.randn(shape, generator=g, device="cuda").to(torch.bfloat16)
    w = bf((C, C, 3, 3))
    ins = [bf((N, C, H + 2, W + 2) if fwd else (N, C, H, W)) for _ in range(K)]
    code = capi.ADH_CONV_FWD if fwd else capi.ADH_CONV_BWD_DATA
    full = capi.conv_workspace_bytes(code, capi.ADH_BF16, K, N, C, C, H, W)
    groups = (C + 63) // 64
    small = groups * groups * 9 * 2 * 64 * 32 * 2 + (K * ((4 * N * C * H * W + 255) // 256 * 256) if groups > 1 else 0)

    def off(t):
        u = torch.empty(t.numel() + at, device="cuda", dtype=t.dtype)[at:].view(t.shape)
        return u.copy_(t)
    got = []
    for tiles, nbytes in ((ins, full), ([off(t) for t in ins], small if at == 2 else full)):
        outs = [torch.empty((N, C, H, W) if fwd else (N, C, H + 2, W + 2), device="cuda", dtype=torch.bfloat16) for _ in range(K)]
        ws = torch.empty(nbytes // 4, device="cuda")
        if fwd:
            capi.check(capi.conv_fwd_tiles(tiles, w, outs, N, C, C, H, W, ws=ws), "fwd")
        else:
            capi.check(capi.conv_bwd_data_tiles(w, tiles, outs, N, C, C, H, W, ws=ws), "bwd-data")
        got.append(torch.cat(outs).float())
    # both round one fp32 sum of the same products to bf16
    assert (got[0] - got[1]).abs().max().item() <= 2 ** -7 * got[1].abs().max().item()
