"""The C-ABI library loads and exports every symbol include/adh_capi.h declares; argument
validation that returns before any device work is exercised without a GPU."""
import ctypes
import os
import re
import time

import pytest
import torch

from arraydiff_cuda_amd import capi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    hdr = open(os.path.join(ROOT, "include", "adh_capi.h")).read()
    hdr = re.sub(r"/\*.*?\*/", "", hdr, flags=re.S)
    return sorted(set(re.findall(r"\b(adh_[a-z0-9_]+)\s*\(", hdr)))


def test_every_declared_symbol_is_exported_and_bound():
    names = declared_symbols()
    assert len(names) >= 28
    lib = ctypes.CDLL(capi.LIB_PATH)
    for n in names:
        assert hasattr(lib, n), "libadh.so does not export %s" % n
    assert set(names) == set(capi.SIGNATURES), "capi.SIGNATURES out of sync with the header"
    assert capi.lib().adh_version() == 1
    assert b"NULL" in capi.lib().adh_error_string(capi.ADH_ENULL)


def test_argument_errors_need_no_gpu():
    l = capi.lib()
    bogus = ctypes.c_void_p(0x1000)
    tb, keep = capi.ptr_table([0x1000, None])
    assert l.adh_halo_exchange_nchw(0, 1, 2, 1, 4, 4, 1, 1, tb, None) == capi.ADH_ENULL
    tb4, keep4 = capi.ptr_table([0x1000] * 4)
    assert l.adh_halo_exchange_nchw(0, 2, 2, 1, 4, 4, 1, 1, tb4, None) == capi.ADH_EUNIMPL
    assert l.adh_halo_exchange_nchw(7, 1, 2, 1, 4, 4, 1, 1, tb4, None) == capi.ADH_EINVAL          # dtype
    assert l.adh_halo_reduce_nchw(0, 1, 4, 3, 4, 4, 1, 1, tb4, None) == capi.ADH_EINVAL            # H < 2p
    assert l.adh_halo_exchange_nchw(0, 1, 1, 1, 4, 4, 1, 1, tb4, None) == capi.ADH_OK              # 1x1 no-op
    odd, keepo = capi.ptr_table([0x1001, 0x1000])
    assert l.adh_halo_exchange_nchw(0, 1, 2, 1, 4, 4, 1, 1, odd, None) == capi.ADH_EALIGN
    assert l.adh_tiles_pack_nchw(0, 3, 1, 4, 8, 1, 1, bogus, tb4, None) == capi.ADH_EINVAL          # H % K
    assert l.adh_tiles_pack_nchw(0, 17, 1, 4, 34, 1, 1, bogus, tb4, None) == capi.ADH_EINVAL        # > 16 tiles
    assert l.adh_slice_copy_nchw(0, 5, 1, 1, 1, bogus, 4, 4, 1, 0, 0, 0, bogus, 8, 8, 1, 0, 0, 0, None) == capi.ADH_EINVAL
    assert l.adh_conv3x3_slab_fwd(0, 1, 4, 4, 3, 3, bogus, bogus, bogus, 0.5, None, 0, None) == capi.ADH_EINVAL  # beta
    assert l.adh_conv3x3_slab_fwd(1, 1, 4, 4, 3, 3, bogus, bogus, bogus, 0.0, None, 0, None) == capi.ADH_ENULL  # bf16 needs a workspace
    assert l.adh_conv3x3_workspace_bytes(capi.ADH_CONV_FWD, 1, 1, 1, 4, 4, 3, 3) > 0
    assert l.adh_conv3x3_slab_fwd(0, 1, 4, 4, 3, 3, None, bogus, bogus, 0.0, None, 0, None) == capi.ADH_ENULL
    assert l.adh_conv3x3_slab_bwd_filter(0, 1, 4, 4, 3, 3, bogus, bogus, bogus, 0.0, bogus, 16, None) == capi.ADH_EWORKSPACE
    assert l.adh_conv3x3_workspace_bytes(capi.ADH_CONV_BWD_FILTER, 0, 4, 32, 64, 64, 14, 56) > 0
    assert l.adh_conv3x3_workspace_bytes(capi.ADH_CONV_FWD, 0, 4, 32, 64, 64, 14, 56) == 0
    assert l.adh_softmax_fwd(10, 2, None, bogus, None) == capi.ADH_ENULL
    assert l.adh_fill_f32(0, 1.0, None, None) == capi.ADH_OK                                       # empty
    assert l.adh_softmax_fwd(0, 0, None, None, None) == capi.ADH_OK
    # the shape query of the pooling over tiles without halo launches nothing
    q = l.adh_pool2d_unpadded_supported
    assert q(0, capi.ADH_POOL_MAX, 4, 32, 64, 64, 256, 3, 3, 2, 2, 1, 1) == capi.ADH_OK        # the stem's pooling
    assert q(0, capi.ADH_POOL_MAX, 4, 32, 64, 64, 8192, 3, 3, 2, 2, 1, 1) == capi.ADH_EUNIMPL  # rows too wide for a band in LDS
    assert q(0, capi.ADH_POOL_MAX, 4, 32, 64, 63, 256, 3, 3, 2, 2, 1, 1) == capi.ADH_EINVAL    # the row split does not stitch
    assert l.adh_conv_bwd_bias_workspace_bytes(4, 32, 64) > 0


def test_bf16_conv_workspace_holds_the_sums_of_every_route_that_needs_them():
    """More than 64 reduction channels at a width the eight-wave kernels do not take run one launch per 64 channels
    with fp32 sums between them: the workspace query has to count those sums whatever one launch of 128 channels
    would have needed at a friendlier width (host logic only, no GPU)."""
    l = capi.lib()
    group = 9 * 2 * 64 * 32 * 2  # bytes of the reordered filter per (64 outputs, 64 reduction channels)

    def need(which, K, N, Cin, Cout, H, W):
        cred, cout = (Cin, Cout) if which == capi.ADH_CONV_FWD else (Cout, Cin)
        oh, ow = (H, W) if which == capi.ADH_CONV_FWD else (H + 2, W + 2)
        filt = ((cout + 63) // 64) * ((cred + 63) // 64) * group
        part = K * ((N * cout * oh * ow * 4 + 255) // 256 * 256)
        return filt, part

    for (K, N, Cin, Cout, H, W) in [(2, 1, 128, 128, 9, 7), (1, 2, 100, 70, 5, 13), (3, 1, 65, 65, 3, 1), (1, 1, 128, 96, 4, 27)]:
        for which in (capi.ADH_CONV_FWD, capi.ADH_CONV_BWD_DATA):
            filt, part = need(which, K, N, Cin, Cout, H, W)
            got = l.adh_conv3x3_workspace_bytes(which, capi.ADH_BF16, K, N, Cin, Cout, H, W)
            assert got >= filt + part, (which, K, N, Cin, Cout, H, W, got, filt, part)
    # one launch of 128 channels (even width forward, a multiple of 8 backward): the filter alone
    for which in (capi.ADH_CONV_FWD, capi.ADH_CONV_BWD_DATA):
        filt, part = need(which, 2, 1, 128, 128, 9, 72)
        assert l.adh_conv3x3_workspace_bytes(which, capi.ADH_BF16, 2, 1, 128, 128, 9, 72) == filt


def test_bf16_conv_workspace_does_not_hold_every_copy_of_an_odd_width():
    """The copies of the input with wider rows, and their sums, are made some images at a time: 512 MiB of them, or one image."""
    l = capi.lib()
    for (K, N, Cin, Cout, H, W) in [(6, 128, 1, 512, 64, 33), (8, 64, 128, 128, 64, 255), (2, 3, 512, 1, 128, 501), (2, 40, 512, 512, 128, 501)]:
        for which in (capi.ADH_CONV_FWD, capi.ADH_CONV_BWD_DATA):
            cred, cout = (Cin, Cout) if which == capi.ADH_CONV_FWD else (Cout, Cin)
            oh, ow = (H, W) if which == capi.ADH_CONV_FWD else (H + 2, W + 2)
            filt = ((cout + 63) // 64) * ((cred + 63) // 64) * 9 * 2 * 64 * 32 * 2
            sums = (N * cout * oh * ow * 4 + 255) // 256 * 256
            image = cred * (H + 2) * ((W + 2 + 7) // 8 * 8) * 2 + cout * oh * ow * 4 + 512
            got = l.adh_conv3x3_workspace_bytes(which, capi.ADH_BF16, K, N, Cin, Cout, H, W)
            assert got <= filt + max(K * sums, 512 << 20, image), (which, K, N, Cin, Cout, H, W, got)


@pytest.mark.skipif(torch.cuda.is_available(), reason="the call would be launched, on addresses that are none")
def test_bf16_filter_gradient_takes_copies_beyond_32_bit_counts():
    """2^31 granules and more of an odd width's copy (tiles above 34 GB) are no error of the arguments: without a GPU it is the
    launch that fails."""
    l = capi.lib()
    K, N, Cin, Cout, H, W = 1, 1 << 14, 512, 8, 1022, 13  # 2^33 rows of three granules
    xs, keep = capi.ptr_table([0x10000])
    nbytes = l.adh_conv3x3_workspace_bytes(capi.ADH_CONV_BWD_FILTER, capi.ADH_BF16, K, N, Cin, Cout, H, W)
    assert nbytes > 1 << 34
    rc = l.adh_conv3x3_slab_bwd_filter_tiles(capi.ADH_BF16, K, N, Cin, Cout, H, W, xs, xs, 0x10000, 0.0, 0x10000, nbytes, None)
    assert rc > 0


def test_the_choice_of_a_tile_is_made_in_microseconds():
    """Every fp32 3x3 call chooses its tile anew: the search has to cost little beside a launch (it took 10 us and more for wide
    rows while every tile was priced).  The best of many repetitions, with room for a slow host."""
    l = capi.lib()
    name = ctypes.create_string_buffer(256)
    kernels = {(4, 32, 64, 64, 32, 128): b"<4, 4, true, 0, 4>", (4, 32, 512, 512, 4, 16): b"<4, 2, true, 0, 4>", (8, 2, 64, 64, 128, 2048): b"<4, 4, true, 0, 4>",
               (7, 3, 272, 40, 61, 1013): b"<4, 4, false, 0, 4>", (4, 32, 64, 64, 14, 56): b"<4, 4, true, 0, 4>"}
    for (K, N, Cin, Cout, H, W), kernel in kernels.items():
        args = [capi.ADH_CONV_FWD, capi.ADH_F32, K, N, Cin, Cout, H, W, 0.0, name, 256]
        best = 1e9
        for _ in range(50):
            t = time.perf_counter()
            for _ in range(20):
                assert l.adh_conv3x3_kernel_name(*args) == capi.ADH_OK
            best = min(best, (time.perf_counter() - t) / 20)
        assert name.value == b"conv3x3_split_kernel" + kernel
        assert best < 6e-6, (K, N, Cin, Cout, H, W, best)


def test_small_layers_are_planned_once():
    """The choice between patches and persistent workgroups or strips costs a small layer less than one plan of the latter takes (it
    took two to seven times as much while both sides were planned, the patches twice)."""
    l = capi.lib()
    name = ctypes.create_string_buffer(256)

    def cost(dtype, K, N, Cin, Cout, H, W):
        best = 1e9
        for _ in range(50):
            t = time.perf_counter()
            for _ in range(20):
                assert l.adh_conv3x3_kernel_name(capi.ADH_CONV_FWD, dtype, K, N, Cin, Cout, H, W, 0.0, name, 256) == capi.ADH_OK
            best = min(best, (time.perf_counter() - t) / 20)
        return best

    plan = cost(capi.ADH_F32, 4, 32, 64, 64, 14, 56)
    assert b"split" in name.value and plan < 20e-6
    for dtype in (capi.ADH_F32, capi.ADH_BF16):
        for shape in ((2, 1, 16, 16, 4, 2000), (2, 3, 20, 36, 9, 130), (4, 1, 32, 64, 14, 56)):
            us = cost(dtype, *shape)
            assert b"patch" in name.value
            assert us < plan + 0.4e-6, (dtype, shape, us, plan)


@pytest.mark.parametrize("shape,strips_us,patches_us", [((6, 10, 64, 64, 80, 324), 143, 247), ((5, 29, 64, 32, 34, 566), 181, 278), ((8, 7, 64, 32, 34, 660), 88, 116),
                                                        ((6, 6, 64, 128, 12, 153), 26, 35), ((2, 16, 128, 128, 4, 930), 43, 62)])
def test_bf16_layers_that_strips_take_faster(shape, strips_us, patches_us):
    """Forward of layers that went to patches: even widths priced with copies that are not made, rounds that are begun as parts of one."""
    name = ctypes.create_string_buffer(256)
    assert capi.lib().adh_conv3x3_kernel_name(capi.ADH_CONV_FWD, capi.ADH_BF16, *shape, 0.0, name, 256) == capi.ADH_OK
    assert b"patch" not in name.value


@pytest.mark.parametrize("shape,persistent_us,patches_us", [((8, 2, 512, 256, 36, 6), 124, 153), ((2, 2, 512, 512, 44, 11), 125, 154), ((3, 10, 512, 128, 24, 10), 124, 152)])
def test_fp32_layers_that_persistent_workgroups_take_faster(shape, persistent_us, patches_us):
    name = ctypes.create_string_buffer(256)
    assert capi.lib().adh_conv3x3_kernel_name(capi.ADH_CONV_FWD, capi.ADH_F32, *shape, 0.0, name, 256) == capi.ADH_OK
    assert b"split" in name.value
