"""Flat copies at the edges of their split: a launch's 64 arrays, a workgroup's 2048 floats, arrays of no elements and off
16-byte alignment, an offset into the flat vector, and the size from which the loads are non-temporal."""
import pytest
import torch

from arraydiff_cuda_amd import capi

pytestmark = pytest.mark.gpu


def _check(lens, skew=0, offset=0):
    g = torch.Generator(device="cuda").manual_seed(len(lens))
    arrays = [torch.randn(n + skew, device="cuda", generator=g)[skew:] for n in lens]
    flat = torch.full((offset + sum(lens) + 5,), 3.0, device="cuda")
    capi.check(capi.flat_store(arrays, flat, offset), "store")
    want = torch.cat([torch.full((offset,), 3.0, device="cuda")] + arrays + [torch.full((5,), 3.0, device="cuda")])
    assert torch.equal(flat, want)
    back = [torch.full((n + skew + 3,), 4.0, device="cuda") for n in lens]
    capi.check(capi.flat_load([b[skew:skew + n] for b, n in zip(back, lens)], flat, offset), "load")
    for b, a, n in zip(back, arrays, lens):
        assert torch.equal(b[skew:skew + n], a) and bool((b[:skew] == 4).all()) and bool((b[skew + n:] == 4).all())


@pytest.mark.parametrize("count", [1, 63, 64, 65, 128, 129, 200])
@pytest.mark.parametrize("skew,offset", [(0, 0), (1, 3)])
def test_counts(count, skew, offset):
    _check([(37 * i) % 301 + 1 for i in range(count)], skew, offset)


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 1024, 1025, 2044, 2047, 2048, 2049, 4095, 4096, 6145, 100003])
@pytest.mark.parametrize("skew", [0, 1, 2, 3])
def test_lengths(n, skew):
    _check([n, 7, n + 1], skew, 1)


def test_arrays_of_no_elements():
    _check([0, 5, 0, 0, 2049] + [0] * 70 + [3, 0])


@pytest.mark.parametrize("total", [(8 << 20) - 1, 8 << 20, (8 << 20) + 4097])
def test_non_temporal(total):
    _check([1000001, 13, total - 1000014])
