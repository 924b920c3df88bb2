"""The optimizer's step over vectors beyond the on-package cache, whose accesses go past the caches: the bits of the same step in pieces."""
import pytest
import torch

from arraydiff_cuda_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ranks,n", [(1, 13500003), (2, 11500002), (3, 9700001), (4, 8500000), (8, 6000003)])
@pytest.mark.parametrize("lagged,summed", [(True, False), (False, True)])
def test_bits_of_the_step_in_pieces(ranks, n, lagged, summed):
    g = torch.Generator(device="cuda").manual_seed(ranks)
    new = lambda: torch.randn((n,), device="cuda", generator=g)
    grads, param, momentum = [new() for _ in range(ranks)], new(), new()
    out = []
    for pieces in (1, 4):
        p, m = param.clone(), momentum.clone()
        lag, total = torch.zeros_like(p) if lagged else None, torch.zeros_like(p) if summed else None
        step = (n // pieces + 3) // 4 * 4
        for a in range(0, n, step):
            cut = lambda t: None if t is None else t[a:a + step]
            capi.check(capi.sgd_step([cut(t) for t in grads], cut(p), cut(m), lagged_param=cut(lag), sum_grad=cut(total), l2_reg=1e-4,
                                     momentum=0.9, step_size=1e-2, next_step_size=2e-2, nesterov=True), "step")
        out.append([t for t in (p, m, lag, total) if t is not None])
    assert (ranks + 4 + lagged) * n * 4 > 256 << 20 >= (ranks + 4 + lagged) * step * 4
    assert all(torch.equal(a, b) for a, b in zip(*out))
