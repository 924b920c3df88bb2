"""bf16 3x3 convolution with more than 64 reduction channels at widths that are no multiple of eight: the passes over a
copy of the input with wider rows (rows shorter than a granule, one column off one, last strips of one column)."""
import numpy as np
import pytest
import torch

from arraydiff_cuda_amd import capi

from test_gpu_conv_bf16 import test_bf16_conv_small_vs_oracle as check_passes_vs_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,N,Cin,Cout,H,W", [(1, 1, 65, 66, 1, 1), (2, 2, 72, 130, 3, 7), (1, 2, 130, 72, 5, 33), (3, 1, 192, 65, 4, 65),
                                              (1, 3, 128, 128, 6, 23), (1, 1, 80, 16, 9, 97), (2, 1, 16, 80, 2, 12)])
def test_odd_widths_vs_oracle(oracle, K, N, Cin, Cout, H, W):
    check_passes_vs_oracle(oracle, K, N, Cin, Cout, H, W)


@pytest.mark.parametrize("which,K,N,Cin,Cout,H,W", [("fwd", 2, 2, 320, 72, 3, 7), ("bwd", 1, 3, 66, 260, 5, 9)])
def test_a_workspace_without_room_for_the_copy(oracle, which, K, N, Cin, Cout, H, W):
    """The reordered filter and the fp32 sums alone: the kernels that run without the copy give the same result."""
    rng = np.random.default_rng(3)
    bf = lambda shape: torch.from_numpy(rng.standard_normal(shape).astype(np.float32)).to(torch.bfloat16).cuda()
    w, fwd = bf((Cout, Cin, 3, 3)), which == "fwd"
    ins = [bf((N, Cin, H + 2, W + 2) if fwd else (N, Cout, H, W)) for _ in range(K)]
    cred, cout = (Cin, Cout) if fwd else (Cout, Cin)
    shape = (N, cout, H, W) if fwd else (N, cout, H + 2, W + 2)
    small = (cout + 63) // 64 * ((cred + 63) // 64) * 9 * 2 * 64 * 32 * 2 + K * ((4 * int(np.prod(shape)) + 255) // 256 * 256)
    full = capi.conv_workspace_bytes(capi.ADH_CONV_FWD if fwd else capi.ADH_CONV_BWD_DATA, capi.ADH_BF16, K, N, Cin, Cout, H, W)
    assert full > small
    got = []
    for nbytes in (small, full):
        outs = [torch.empty(shape, device="cuda", dtype=torch.bfloat16) for _ in range(K)]
        ws = torch.empty(nbytes // 4, device="cuda")
        if fwd:
            capi.check(capi.conv_fwd_tiles(ins, w, outs, N, Cin, Cout, H, W, ws=ws), "fwd")
        else:
            capi.check(capi.conv_bwd_data_tiles(w, ins, outs, N, Cin, Cout, H, W, ws=ws), "bwd-data")
        got.append(torch.cat(outs).float())
    # both round one fp32 sum of the same products to bf16
    assert (got[0] - got[1]).abs().max().item() <= 2 ** -7 * got[1].abs().max().item()


@pytest.mark.parametrize("which,K,N,Cin,Cout,H,W", [("fwd", 2, 9, 320, 66, 64, 255), ("bwd", 2, 5, 66, 320, 64, 255),  # images in turn
                                                    ("fwd", 3, 2, 320, 65, 64, 501),  # two tiles, then one
                                                    ("bwd", 2, 1, 1, 144, 120, 2043)])  # a tile at a time, each larger than the least room
def test_copies_in_turn(which, K, N, Cin, Cout, H, W):
    """A workspace with room for some of the copies: every image's bits are those of a call for it alone, and nothing is written
    past the workspace."""
    fwd = which == "fwd"
    g = torch.Generator(device="cuda").manual_seed(4)
    bf = lambda shape: torch.randn(shape, generator=g, device="cuda").to(torch.bfloat16)
    w = bf((Cout, Cin, 3, 3))
    ins = [bf((N, Cin, H + 2, W + 2) if fwd else (N, Cout, H, W)) for _ in range(K)]
    olds = [bf((N, Cout, H, W) if fwd else (N, Cin, H + 2, W + 2)) for _ in range(K)]
    code = capi.ADH_CONV_FWD if fwd else capi.ADH_CONV_BWD_DATA
    query = lambda k, n: capi.conv_workspace_bytes(code, capi.ADH_BF16, k, n, Cin, Cout, H, W)

    def run(ins, outs, n, nbytes):
        ws = torch.full((nbytes // 4 + 64,), 7.0, device="cuda")
        if fwd:
            capi.check(capi.conv_fwd_tiles(ins, w, outs, n, Cin, Cout, H, W, beta=1.0, ws=ws[:nbytes // 4]), "fwd")
        else:
            capi.check(capi.conv_bwd_data_tiles(w, ins, outs, n, Cin, Cout, H, W, beta=1.0, ws=ws[:nbytes // 4]), "bwd-data")
        assert (ws[nbytes // 4:] == 7.0).all()

    cred, cout, oh, ow = (Cin, Cout, H, W) if fwd else (Cout, Cin, H + 2, W + 2)
    filt = ((cout + 63) // 64) * ((cred + 63) // 64) * 9 * 2 * 64 * 32 * 2
    sums = K * ((N * cout * oh * ow * 4 + 255) // 256 * 256)
    least = filt + max(sums, 64 << 20, query(1, 1) - filt)
    got, all_at_once = [t.clone() for t in olds], [t.clone() for t in olds]
    run(ins, all_at_once, N, query(K, N))
    run(ins, got, N, least)
    for k in range(K):
        assert torch.equal(got[k], all_at_once[k])
        for n in range(N):
            alone = olds[k][n:n + 1].clone()
            run([ins[k][n:n + 1].clone()], [alone], 1, query(1, 1))
            assert torch.equal(got[k][n:n + 1], alone), (k, n)
