"""Convolution of at most three input channels on the bf16 matrix cores at the sizes where its tiling can go wrong (windows of every
width, column stride 1 and 2, output channels around the groups of 16 and 64, rows around 16 and 32 columns, tiles of few
rows, many tiles per workgroup) against the CPU oracle, and with values whose bf16 parts are not finite."""
import numpy as np
import pytest
import torch

from arraydiff_cuda_amd import capi
from gpu_util import dev, host, rel_err

pytestmark = pytest.mark.gpu


def _ws(which, K, N, Cin, Cout, HP, WP, geo):
    return torch.empty(capi.conv2d_workspace_bytes(which, capi.ADH_F32, K, N, Cin, Cout, HP, WP, *geo) // 4 + 64, device="cuda")


@pytest.mark.parametrize("K,N,Cin,Cout,OH,OW,kh,kw,sh,sw", [
    (1, 1, 1, 1, 1, 1, 1, 1, 1, 1), (2, 1, 3, 64, 9, 33, 7, 7, 1, 1), (1, 2, 3, 65, 17, 31, 7, 7, 2, 2), (2, 2, 3, 17, 5, 16, 3, 3, 1, 1),
    (1, 2, 1, 16, 33, 15, 5, 5, 1, 1), (3, 1, 2, 33, 4, 48, 5, 5, 2, 2), (1, 3, 3, 32, 3, 70, 3, 3, 2, 2), (2, 1, 1, 48, 6, 17, 7, 7, 2, 2),
    (1, 1, 3, 20, 8, 40, 8, 8, 1, 1), (1, 1, 2, 24, 7, 19, 2, 6, 3, 2), (1, 1, 3, 8, 6, 9, 4, 9, 1, 1), (8, 40, 1, 8, 8, 32, 3, 3, 1, 1)])
def test_passes_vs_oracle(oracle, K, N, Cin, Cout, OH, OW, kh, kw, sh, sw):
    rng = np.random.default_rng(77 + OW)
    HP, WP, geo = (OH - 1) * sh + kh, (OW - 1) * sw + kw, (kh, kw, sh, sw, 1, 1)
    xs = [rng.uniform(-1, 1, size=(N, Cin, HP, WP)).astype(np.float32) for _ in range(K)]
    w = (rng.standard_normal((Cout, Cin, kh, kw)) * np.sqrt(2.0 / (Cin * kh * kw))).astype(np.float32)
    bias = rng.standard_normal(Cout).astype(np.float32)
    dys = [rng.standard_normal((N, Cout, OH, OW)).astype(np.float32) for _ in range(K)]
    for beta in (0.0, 1.0):
        ys = [torch.ones((N, Cout, OH, OW), device="cuda") for _ in range(K)]
        capi.check(capi.conv2d_fwd_bias_tiles([dev(x) for x in xs], dev(w), [dev(bias)] * K, ys, N, Cin, Cout, HP, WP, *geo, beta=beta,
                                              ws=_ws(capi.ADH_CONV_FWD, K, N, Cin, Cout, HP, WP, geo)), "fwd")
        for x, y in zip(xs, ys):
            want = np.empty((N, Cout, OH, OW), np.float32)
            oracle.conv2d_slab_fwd(x, w, sh, sw, 1, 1, want)
            assert rel_err(host(y), want + bias[None, :, None, None] + beta) <= 1e-5
        dw = torch.ones((Cout, Cin, kh, kw), device="cuda")
        capi.check(capi.conv2d_bwd_filter_tiles([dev(x) for x in xs], [dev(d) for d in dys], dw, N, Cin, Cout, HP, WP, *geo, beta=beta,
                                                ws=_ws(capi.ADH_CONV_BWD_FILTER, K, N, Cin, Cout, HP, WP, geo)), "bwd-filter")
        dw_want = np.full((Cout, Cin, kh, kw), beta, np.float32)
        for x, d in zip(xs, dys):
            oracle.conv2d_slab_bwd_filter(x, d, sh, sw, 1, 1, dw_want, beta=1.0)
        assert rel_err(host(dw), dw_want) <= 1e-5


@pytest.mark.parametrize("bad", [float("inf"), 3.4e38, float("nan")])
@pytest.mark.parametrize("s", [1, 2])
def test_values_without_finite_bf16_parts(bad, s):
    """What they touch, and only that, is infinite, huge or NaN."""
    N, Cin, Cout, OH, OW, k = 1, 3, 40, 20, 45, 7
    HP, WP, geo = (OH - 1) * s + k, (OW - 1) * s + k, (k, k, s, s, 1, 1)
    g = torch.Generator().manual_seed(9)
    x, w = torch.rand((N, Cin, HP, WP), generator=g) + 0.5, torch.rand((Cout, Cin, k, k), generator=g) * 0.1 + 0.01
    dy = torch.rand((N, Cout, OH, OW), generator=g) + 0.5

    def same(got, want):
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
        fine = torch.isfinite(want)
        assert ((got[fine].double() - want[fine].double()).abs() <= 1e-5 * want[fine].double().abs()).all() and fine.any()

    def taps(a):
        return [a[:, :, i:i + (OH - 1) * s + 1:s, j:j + (OW - 1) * s + 1:s] for i in range(k) for j in range(k)]

    for where in ("input", "filter", "gradient"):
        xb, wb, db = x.clone(), w.clone(), dy.clone()
        if where == "input":
            xb[0, 1, 9, 11] = bad
        elif where == "filter":
            wb[5, 2, 1, 2] = bad
        else:
            db[0, 30, 4, 10] = bad
        y = torch.empty((N, Cout, OH, OW), device="cuda")
        capi.check(capi.conv2d_fwd_tiles([xb.cuda()], wb.cuda(), [y], N, Cin, Cout, HP, WP, *geo,
                                         ws=_ws(capi.ADH_CONV_FWD, 1, N, Cin, Cout, HP, WP, geo)), "fwd")
        want = torch.zeros((N, Cout, OH, OW))
        for t, xt in enumerate(taps(xb)):
            for c in range(Cin):
                want = want + xt[:, c, None] * wb.reshape(Cout, Cin, k * k)[None, :, c, t, None, None]
        same(y.cpu(), want)
        dw = torch.empty((Cout, Cin, k, k), device="cuda")
        capi.check(capi.conv2d_bwd_filter_tiles([xb.cuda()], [db.cuda()], dw, N, Cin, Cout, HP, WP, *geo,
                                                ws=_ws(capi.ADH_CONV_BWD_FILTER, 1, N, Cin, Cout, HP, WP, geo)), "bwd-filter")
        same(dw.cpu(), torch.stack([(db[:, :, None] * xt[:, None]).sum((0, 3, 4)) for xt in taps(xb)], -1).reshape(Cout, Cin, k, k))


@pytest.mark.parametrize("K,N,Cin,Cout,OH,OW,k,s,nbytes", [(4, 3, 3, 64, 9, 18, 7, 1, 1474560), (4, 4, 3, 64, 12, 1, 7, 2, 655360),
                                                           (3, 4, 3, 64, 16, 4, 3, 2, 196608), (1, 3, 3, 64, 1, 6, 3, 2, 16384)])
def test_filter_gradient_in_a_small_workspace(K, N, Cin, Cout, OH, OW, k, s, nbytes):
    """A workspace below the query's answer but enough for the general kernel: fewer workgroups share the pixels."""
    HP, WP, geo = (OH - 1) * s + k, (OW - 1) * s + k, (k, k, s, s, 1, 1)
    g = torch.Generator().manual_seed(11)
    xs = [torch.rand((N, Cin, HP, WP), generator=g) * 2 - 1 for _ in range(K)]
    dys = [torch.randn((N, Cout, OH, OW), generator=g) for _ in range(K)]
    want = torch.nn.grad.conv2d_weight(torch.cat(xs).double(), (Cout, Cin, k, k), torch.cat(dys).double(), stride=s).numpy()
    assert nbytes < capi.conv2d_workspace_bytes(capi.ADH_CONV_BWD_FILTER, capi.ADH_F32, K, N, Cin, Cout, HP, WP, *geo)
    ws = torch.full((nbytes // 4 + 64,), 7.0, device="cuda")
    dw = torch.ones((Cout, Cin, k, k), device="cuda")
    capi.check(capi.conv2d_bwd_filter_tiles([x.cuda() for x in xs], [d.cuda() for d in dys], dw, N, Cin, Cout, HP, WP, *geo, beta=1.0,
                                            ws=ws[:nbytes // 4]), "bwd-filter")
    assert (ws[nbytes // 4:] == 7.0).all()
    assert rel_err(host(dw), want + 1.0) <= 1e-5
