"""Python binding of ``libadh.so``: ctypes for every symbol (``lib()``), and functions on torch tensors whose arguments a native
module converts (``csrc/binding.cc``).  There is no fallback: if the library is missing, or a
call is made without a GPU, an exception is raised."""
import ctypes
import os
import subprocess

_HERE = os.path.dirname(os.path.abspath(__file__))
# ADH_LIB names another build of the library (A/B measurements); the default is the one beside this file
LIB_PATH = os.environ.get("ADH_LIB") or os.path.join(_HERE, "libadh.so")
CSRC = os.path.join(_HERE, "csrc")

ADH_F32 = 0
ADH_BF16 = 1
ADH_OK, ADH_EINVAL, ADH_EUNIMPL, ADH_ENULL, ADH_EALIGN, ADH_EWORKSPACE = 0, -1, -2, -3, -4, -5
ADH_CONV_FWD, ADH_CONV_BWD_DATA, ADH_CONV_BWD_FILTER = 0, 1, 2
ADH_POOL_AVG, ADH_POOL_MAX = 0, 1
ADH_MAX_TILES = 16

u32, u64, i32, f32, vp, sz = (ctypes.c_uint32, ctypes.c_uint64, ctypes.c_int, ctypes.c_float,
                              ctypes.c_void_p, ctypes.c_size_t)
vpp = ctypes.POINTER(ctypes.c_void_p)

# name -> (restype, argtypes); every symbol include/adh_capi.h declares
SIGNATURES = {
    "adh_version": (i32, []),
    "adh_error_string": (ctypes.c_char_p, [i32]),
    "adh_fill_f32": (i32, [u64, f32, vp, vp]),
    "adh_add_f32": (i32, [u64, vp, vp, vp]),
    "adh_halo_exchange_nchw": (i32, [i32, u32, u32, u32, u32, u32, u32, u32, vpp, vp]),
    "adh_halo_reduce_nchw": (i32, [i32, u32, u32, u32, u32, u32, u32, u32, vpp, vp]),
    "adh_halo_exchange_nchw_rank": (i32, [i32, u32, u32, u32, u32, u32, u32, u32, u32, vpp, vp]),
    "adh_halo_reduce_nchw_rank": (i32, [i32, u32, u32, u32, u32, u32, u32, u32, u32, vpp, vp]),
    "adh_halo_pad_nchw": (i32, [i32, u32, u32, u32, u32, u32, vp, vp, vp]),
    "adh_halo_pad_add_nchw": (i32, [i32, u32, u32, u32, u32, u32, vp, vp, vp]),
    "adh_halo_unpad_nchw": (i32, [i32, u32, u32, u32, u32, u32, vp, vp, vp]),
    "adh_halo_unpad_add_nchw": (i32, [i32, u32, u32, u32, u32, u32, vp, vp, vp]),
    "adh_halo_repad_nchw": (i32, [i32, u32, u32, u32, u32, u32, u32, vp, vp, vp]),
    "adh_slice_copy_nchw": (i32, [i32, u32, u32, u32, u32, vp, u32, u32, u32, u32, u32, u32,
                                  vp, u32, u32, u32, u32, u32, u32, vp]),
    "adh_slice_add_nchw": (i32, [i32, u32, u32, u32, u32, vp, u32, u32, u32, u32, u32, u32,
                                 vp, u32, u32, u32, u32, u32, u32, vp]),
    "adh_tiles_pack_nchw": (i32, [i32, u32, u32, u32, u32, u32, u32, vp, vpp, vp]),
    "adh_tiles_unpack_nchw": (i32, [i32, u32, u32, u32, u32, u32, u32, vpp, vp, vp]),
    "adh_conv3x3_workspace_bytes": (sz, [i32, i32, u32, u32, u32, u32, u32, u32]),
    "adh_conv3x3_kernel_name": (i32, [i32, i32, u32, u32, u32, u32, u32, u32, f32, ctypes.c_char_p, sz]),
    "adh_conv3x3_slab_fwd": (i32, [i32, u32, u32, u32, u32, u32, vp, vp, vp, f32, vp, sz, vp]),
    "adh_conv3x3_slab_fwd_tiles": (i32, [i32, u32, u32, u32, u32, u32, u32, vpp, vp, vpp, f32, vp, sz, vp]),
    "adh_conv3x3_slab_fwd_tiles_unexchanged": (i32, [i32, u32, u32, u32, u32, u32, u32, vpp, vp, vpp, f32, vp, sz, vp]),
    "adh_conv3x3_slab_bwd_data_tiles_reduced": (i32, [i32, u32, u32, u32, u32, u32, u32, vp, vpp, vpp, f32, vp, sz, vp]),
    "adh_conv3x3_unpadded_fwd_tiles": (i32, [i32, u32, u32, u32, u32, u32, u32, vpp, vp, vpp, f32, vp, sz, vp]),
    "adh_conv3x3_unpadded_fwd_residual_tiles": (i32, [i32, u32, u32, u32, u32, u32, u32, vpp, vp, vpp, vpp, vp]),
    "adh_conv3x3_unpadded_bwd_data_tiles": (i32, [i32, u32, u32, u32, u32, u32, u32, vp, vpp, vpp, f32, vp, sz, vp]),
    "adh_conv3x3_unpadded_bwd_filter_tiles": (i32, [i32, u32, u32, u32, u32, u32, u32, vpp, vpp, vp, f32, vp, sz, vp]),
    "adh_conv3x3_slab_fwd_tiles_static": (i32, [i32, u32, u32, u32, u32, u32, u32, vpp, vp, vpp, f32, vp]),
    "adh_conv3x3_slab_bwd_data": (i32, [i32, u32, u32, u32, u32, u32, vp, vp, vp, f32, vp, sz, vp]),
    "adh_conv3x3_slab_bwd_data_tiles": (i32, [i32, u32, u32, u32, u32, u32, u32, vp, vpp, vpp, f32, vp, sz, vp]),
    "adh_conv3x3_slab_bwd_filter": (i32, [i32, u32, u32, u32, u32, u32, vp, vp, vp, f32, vp, sz, vp]),
    "adh_conv3x3_slab_bwd_filter_tiles": (i32, [i32, u32, u32, u32, u32, u32, u32, vpp, vpp, vp, f32, vp, sz, vp]),
    "adh_conv3x3_slab_bwd_filter_tiles_unexchanged": (i32, [i32, u32, u32, u32, u32, u32, u32, vpp, vpp, vp, f32, vp, sz,
                                                            vp]),
    "adh_conv_bias_add_tiles": (i32, [i32, u32, u32, u32, u32, u32, vpp, vpp, vp]),
    "adh_conv_bwd_bias_workspace_bytes": (sz, [u32, u32, u32]),
    "adh_conv_bwd_bias_tiles": (i32, [i32, u32, u32, u32, u32, u32, vpp, vp, f32, vp, sz, vp]),
    "adh_conv2d_workspace_bytes": (sz, [i32, i32] + [u32] * 12),
    "adh_conv2d_slab_fwd_tiles": (i32, [i32] + [u32] * 12 + [vpp, vp, vpp, f32, vp, sz, vp]),
    "adh_conv2d_slab_fwd_bias_tiles": (i32, [i32] + [u32] * 12 + [vpp, vp, vpp, vpp, f32, vp, sz, vp]),
    "adh_conv2d_slab_bwd_data_tiles": (i32, [i32] + [u32] * 12 + [vp, vpp, vpp, f32, vp, sz, vp]),
    "adh_conv2d_slab_bwd_filter_tiles": (i32, [i32] + [u32] * 12 + [vpp, vpp, vp, f32, vp, sz, vp]),
    "adh_conv2d_unpadded_workspace_bytes": (sz, [i32, i32] + [u32] * 14),
    "adh_conv2d_unpadded_fwd_tiles": (i32, [i32] + [u32] * 14 + [vpp, vp, vpp, f32, vp, sz, vp]),
    "adh_conv2d_unpadded_bwd_data_tiles": (i32, [i32] + [u32] * 14 + [vp, vpp, vpp, f32, vp, sz, vp]),
    "adh_conv2d_unpadded_bwd_filter_tiles": (i32, [i32] + [u32] * 14 + [vpp, vpp, vp, f32, vp, sz, vp]),
    "adh_batchnorm2d_workspace_bytes": (sz, [u32, u32, u32]),
    "adh_batchnorm2d_fwd_tiles": (i32, [i32, i32, u32, u32, u32, u32, u32, f32, i32, u32, vpp, vpp, vpp, vpp, vpp, vpp, vpp,
                                        vpp, vpp, vpp, vp, sz, vp]),
    "adh_batchnorm2d_bwd_tiles": (i32, [i32, u32, u32, u32, u32, u32, i32, u32, vpp, vpp, vpp, vpp, vpp, vpp, vpp, vpp, vpp,
                                        f32, f32, vp, sz, vp]),
    "adh_relu_fwd": (i32, [i32, ctypes.c_uint64, vp, vp, vp]),
    "adh_relu_bwd": (i32, [i32, ctypes.c_uint64, vp, vp, vp, f32, vp]),
    "adh_sum_fwd": (i32, [i32, u32, ctypes.c_uint64, vpp, vp, vp]),
    "adh_pool2d_slab_fwd_tiles": (i32, [i32, i32, u32, u32, u32, u32, u32, u32, u32, u32, u32, vpp, vpp, vp]),
    "adh_pool2d_slab_fwd": (i32, [i32, i32, u32, u32, u32, u32, u32, u32, u32, u32, vp, vp, vp]),
    "adh_pool2d_slab_bwd_tiles": (i32, [i32, i32, u32, u32, u32, u32, u32, u32, u32, u32, u32, vpp, vpp, vpp, vpp, f32, vp]),
    "adh_pool2d_slab_bwd": (i32, [i32, i32, u32, u32, u32, u32, u32, u32, u32, u32, vp, vp, vp, vp, f32, vp]),
    "adh_pool2d_unpadded_supported": (i32, [i32, i32] + [u32] * 11),
    "adh_pool2d_unpadded_fwd_tiles": (i32, [i32, i32] + [u32] * 11 + [vpp, vpp, vp]),
    "adh_pool2d_unpadded_bwd_tiles": (i32, [i32, i32] + [u32] * 11 + [vpp, vpp, vpp, vpp, f32, vp]),
    "adh_softmax_fwd": (i32, [u32, u32, vp, vp, vp]),
    "adh_softmax_nll_loss_fwd": (i32, [u32, u32, vp, vp, vp, vp]),
    "adh_softmax_nll_loss_bwd": (i32, [u32, u32, vp, vp, vp, vp, vp]),
    "adh_softmax_xent_fwd": (i32, [u32, u32, vp, vp, vp, vp, vp]),
    "adh_softmax_nll_loss_bwd_scaled": (i32, [u32, u32, vp, vp, vp, f32, f32, vp, vp]),
    "adh_softmax_xent_fwd_bwd": (i32, [u32, u32, vp, vp, vp, f32, vp, vp, f32, vp, vp]),
    "adh_scale_add_f32": (i32, [u64, f32, vp, f32, vp, vp]),
    "adh_add_online_f32": (i32, [u64, f32, vp, vp, vp]),
    "adh_stat_step_f32": (i32, [u64, f32, vp, vp, vp, vp]),
    "adh_flat_store_f32": (i32, [u32, vpp, ctypes.POINTER(u64), u64, vp, vp]),
    "adh_flat_load_f32": (i32, [u32, vpp, ctypes.POINTER(u64), u64, vp, vp]),
    "adh_sgd_step_f32": (i32, [u64, u32, vpp, f32, f32, f32, f32, i32, vp, vp, vp, vp, vp]),
}


def build(force=True):
    """Compile libadh.so for gfx950 with hipcc (cross-compiles without a GPU)."""
    args = ["make", "-s", "-C", CSRC, "-j8"]
    if force:
        args.append("-B")
    subprocess.check_call(args)
    return LIB_PATH


class AdhError(RuntimeError):
    def __init__(self, code, what):
        self.code = code
        super().__init__("%s failed: %d (%s)" % (what, code, lib().adh_error_string(code).decode()))


_lib = None


def lib():
    """The loaded library.  Raises if it has not been built: there is no CPU fallback."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError("libadh.so is not built (%s); run __graft_entry__.build() or "
                               "`make -C arraydiff_cuda_amd/csrc`" % LIB_PATH)
        l = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(l, name)  # AttributeError if a declared symbol is not exported
            fn.restype = res
            fn.argtypes = args
        _lib = l
    return _lib


def check(code, what="adh call"):
    if code != 0:
        raise AdhError(code, what)
    return code


def ptr_table(ptrs):
    """Host array of device pointers from ints / None."""
    arr = (ctypes.c_void_p * len(ptrs))(*[p if p else None for p in ptrs])
    return ctypes.cast(arr, vpp), arr


# ---------------------------------------------------------------------------
# torch-tensor convenience wrappers (tests / bench).  Tensors must live on the GPU.
# ---------------------------------------------------------------------------
_native = None  # the module that converts the arguments and calls


def _load_native():
    global _native
    import torch
    from . import _binding
    if not os.path.exists(LIB_PATH):
        lib()  # raises, with what to do
    _binding.load(LIB_PATH, torch._C._cuda_getDevice, torch._C._cuda_getCurrentRawStream)
    _CODES.update({torch.float32: ADH_F32, torch.bfloat16: ADH_BF16})
    _native = _binding
    return _native


_CODES = {}  # ADH_F32 / ADH_BF16 by torch dtype


def _n():
    return _native or _load_native()


def _dt(t):
    if _native is None:
        _load_native()
    code = _CODES.get(t.dtype)
    if code is None:
        raise TypeError("dtype %s not supported" % t.dtype)
    return code


def _ws(ws):
    if ws is None:
        return None, 0
    return ws, ws.numel() * ws.element_size()


def fill_f32(x, v):
    return _n().adh_fill_f32(x.numel(), v, x)


def add_f32(x, y):
    return _n().adh_add_f32(x.numel(), x, y)


def halo_exchange(tiles, grid_w, grid_h, p, W, H, C, N, rank=None):
    if rank is None:
        return _n().adh_halo_exchange_nchw(_dt(tiles[0]), grid_w, grid_h, p, W, H, C, N, tiles)
    return _n().adh_halo_exchange_nchw_rank(_dt(tiles[0]), grid_w, grid_h, rank, p, W, H, C, N, tiles)


def halo_reduce(tiles, grid_w, grid_h, p, W, H, C, N, rank=None):
    if rank is None:
        return _n().adh_halo_reduce_nchw(_dt(tiles[0]), grid_w, grid_h, p, W, H, C, N, tiles)
    return _n().adh_halo_reduce_nchw_rank(_dt(tiles[0]), grid_w, grid_h, rank, p, W, H, C, N, tiles)


def _padlike(name, p, W, H, C, N, a, b):
    return getattr(_n(), name)(_dt(a), p, W, H, C, N, a, b)


def halo_pad(p, W, H, C, N, x, y):
    return _padlike("adh_halo_pad_nchw", p, W, H, C, N, x, y)


def halo_pad_add(p, W, H, C, N, x, y):
    return _padlike("adh_halo_pad_add_nchw", p, W, H, C, N, x, y)


def halo_unpad(p, W, H, C, N, x, y):
    return _padlike("adh_halo_unpad_nchw", p, W, H, C, N, x, y)


def halo_unpad_add(p, W, H, C, N, x, y):
    return _padlike("adh_halo_unpad_add_nchw", p, W, H, C, N, x, y)


def halo_repad(ps, pd, W, H, C, N, x, y):
    return _n().adh_halo_repad_nchw(_dt(x), ps, pd, W, H, C, N, x, y)


def slice_nchw(add, count, N, src, src_dims, src_off, dst, dst_dims, dst_off):
    fn = _n().adh_slice_add_nchw if add else _n().adh_slice_copy_nchw
    return fn(_dt(src), count[0], count[1], count[2], N, src, src_dims[0], src_dims[1], src_dims[2],
              src_off[0], src_off[1], src_off[2], dst, dst_dims[0], dst_dims[1], dst_dims[2],
              dst_off[0], dst_off[1], dst_off[2])


def tiles_pack(K, p, W, H, C, N, x, tiles):
    return _n().adh_tiles_pack_nchw(_dt(x), K, p, W, H, C, N, x, tiles)


def tiles_unpack(K, p, W, H, C, N, tiles, y):
    return _n().adh_tiles_unpack_nchw(_dt(y), K, p, W, H, C, N, tiles, y)


def conv_workspace_bytes(which, dtype, K, N, Cin, Cout, H, W):
    return lib().adh_conv3x3_workspace_bytes(which, dtype, K, N, Cin, Cout, H, W)


def conv_fwd_tiles(xs, w, ys, N, Cin, Cout, H, W, beta=0.0, ws=None, unexchanged=False):
    """unexchanged: xs are the row tiles of one activation in rank order whose inner halo rows have not been
    exchanged; the result equals halo_exchange followed by the ordinary forward."""
    fn = _n().adh_conv3x3_slab_fwd_tiles_unexchanged if unexchanged else _n().adh_conv3x3_slab_fwd_tiles
    return fn(_dt(xs[0]), len(xs), N, Cin, Cout, H, W, xs, w, ys, beta, *_ws(ws))


def conv_bwd_data_tiles(w, dys, dxs, N, Cin, Cout, H, W, beta=0.0, ws=None, reduced=False):
    """reduced: dys are the row tiles of one gradient in rank order; the interior of every dx tile comes out as
    after backward-data followed by halo_reduce."""
    fn = _n().adh_conv3x3_slab_bwd_data_tiles_reduced if reduced else _n().adh_conv3x3_slab_bwd_data_tiles
    return fn(_dt(dys[0]), len(dys), N, Cin, Cout, H, W, w, dys, dxs, beta, *_ws(ws))


def conv_unpadded_fwd_tiles(xs, w, ys, N, Cin, Cout, H, W, beta=0.0, ws=None):
    """xs, ys: the row tiles (H x W, no halo) of one tensor in rank order."""
    return _n().adh_conv3x3_unpadded_fwd_tiles(_dt(xs[0]), len(xs), N, Cin, Cout, H, W, xs, w, ys, beta, *_ws(ws))


def conv_unpadded_fwd_residual_tiles(xs, w, res, ys, N, Cin, Cout, H, W):
    """ys[t] = conv(xs, w)[t] + res[t] over tiles without halo (fp32)."""
    return _n().adh_conv3x3_unpadded_fwd_residual_tiles(_dt(xs[0]), len(xs), N, Cin, Cout, H, W, xs, w, res, ys)


def conv_unpadded_bwd_data_tiles(w, dys, dxs, N, Cin, Cout, H, W, beta=0.0, ws=None):
    return _n().adh_conv3x3_unpadded_bwd_data_tiles(_dt(dys[0]), len(dys), N, Cin, Cout, H, W, w, dys, dxs, beta,
                                                    *_ws(ws))


def conv_unpadded_bwd_filter_tiles(xs, dys, dw, N, Cin, Cout, H, W, beta=0.0, ws=None):
    return _n().adh_conv3x3_unpadded_bwd_filter_tiles(_dt(xs[0]), len(xs), N, Cin, Cout, H, W, xs, dys, dw, beta,
                                                      *_ws(ws))


def conv_bias_add_tiles(biases, ys, N, C, H, W):
    """ys[t][n,c,h,w] += biases[t][c]; biases are fp32 vectors of C (entries may repeat)."""
    return _n().adh_conv_bias_add_tiles(_dt(ys[0]), len(ys), N, C, H, W, biases, ys)


def conv_bwd_bias_workspace_bytes(K, N, C):
    return lib().adh_conv_bwd_bias_workspace_bytes(K, N, C)


def conv_bwd_bias_tiles(dys, db, N, C, H, W, beta=0.0, ws=None):
    """db[c] = beta*db[c] + sum over tiles, n, h, w of dys[t][n,c,h,w]."""
    return _n().adh_conv_bwd_bias_tiles(_dt(dys[0]), len(dys), N, C, H, W, dys, db, beta, *_ws(ws))


def conv2d_workspace_bytes(which, dtype, K, N, Cin, Cout, HP, WP, kh, kw, sh, sw, dh, dw):
    return lib().adh_conv2d_workspace_bytes(which, dtype, K, N, Cin, Cout, HP, WP, kh, kw, sh, sw, dh, dw)


def conv2d_fwd_tiles(xs, w, ys, N, Cin, Cout, HP, WP, kh, kw, sh, sw, dh, dw, beta=0.0, ws=None):
    return _n().adh_conv2d_slab_fwd_tiles(_dt(xs[0]), len(xs), N, Cin, Cout, HP, WP, kh, kw, sh, sw, dh, dw, xs, w, ys,
                                          beta, *_ws(ws))


def conv2d_fwd_bias_tiles(xs, w, biases, ys, N, Cin, Cout, HP, WP, kh, kw, sh, sw, dh, dw, beta=0.0, ws=None):
    """conv2d_fwd_tiles followed by ys[t] += biases[t] per channel, in the convolution's stores where its kernel can."""
    return _n().adh_conv2d_slab_fwd_bias_tiles(_dt(xs[0]), len(xs), N, Cin, Cout, HP, WP, kh, kw, sh, sw, dh, dw, xs, w,
                                               biases, ys, beta, *_ws(ws))


def conv2d_bwd_data_tiles(w, dys, dxs, N, Cin, Cout, HP, WP, kh, kw, sh, sw, dh, dw, beta=0.0, ws=None):
    return _n().adh_conv2d_slab_bwd_data_tiles(_dt(dys[0]), len(dys), N, Cin, Cout, HP, WP, kh, kw, sh, sw, dh, dw, w,
                                               dys, dxs, beta, *_ws(ws))


def conv2d_bwd_filter_tiles(xs, dys, dw, N, Cin, Cout, HP, WP, kh, kw, sh, sw, dh, dw_, beta=0.0, ws=None):
    return _n().adh_conv2d_slab_bwd_filter_tiles(_dt(xs[0]), len(xs), N, Cin, Cout, HP, WP, kh, kw, sh, sw, dh, dw_, xs,
                                                 dys, dw, beta, *_ws(ws))


def conv2d_unpadded_workspace_bytes(which, dtype, K, N, Cin, Cout, H, W, kh, kw, sh, sw, dh, dw, pad_h, pad_w):
    return lib().adh_conv2d_unpadded_workspace_bytes(which, dtype, K, N, Cin, Cout, H, W, kh, kw, sh, sw, dh, dw, pad_h, pad_w)


def conv2d_unpadded_fwd_tiles(xs, w, ys, N, Cin, Cout, H, W, kh, kw, sh, sw, dh, dw, pad_h, pad_w, beta=0.0, ws=None):
    """Row tiles without halo, any window / stride / dilation: rows outside a tile come from its neighbours."""
    return _n().adh_conv2d_unpadded_fwd_tiles(_dt(xs[0]), len(xs), N, Cin, Cout, H, W, kh, kw, sh, sw, dh, dw, pad_h,
                                              pad_w, xs, w, ys, beta, *_ws(ws))


def conv2d_unpadded_bwd_data_tiles(w, dys, dxs, N, Cin, Cout, H, W, kh, kw, sh, sw, dh, dw, pad_h, pad_w, beta=0.0, ws=None):
    return _n().adh_conv2d_unpadded_bwd_data_tiles(_dt(dys[0]), len(dys), N, Cin, Cout, H, W, kh, kw, sh, sw, dh, dw,
                                                   pad_h, pad_w, w, dys, dxs, beta, *_ws(ws))


def conv2d_unpadded_bwd_filter_tiles(xs, dys, dw, N, Cin, Cout, H, W, kh, kw, sh, sw, dh, dw_, pad_h, pad_w, beta=0.0, ws=None):
    return _n().adh_conv2d_unpadded_bwd_filter_tiles(_dt(xs[0]), len(xs), N, Cin, Cout, H, W, kh, kw, sh, sw, dh, dw_,
                                                     pad_h, pad_w, xs, dys, dw, beta, *_ws(ws))


def batchnorm_workspace_bytes(K, N, C):
    return lib().adh_batchnorm2d_workspace_bytes(K, N, C)


def batchnorm_fwd_tiles(xs, scales, shifts, ys, N, C, H, W, eps=1e-5, relu=0, out_halo=0, training=True, fixed_means=None,
                        fixed_vars=None, run_means=None, run_vars=None, save_means=None, save_invstds=None, ws=None):
    return _n().adh_batchnorm2d_fwd_tiles(_dt(xs[0]), 1 if training else 0, len(xs), N, C, H, W, eps, relu, out_halo,
                                          xs, scales, shifts, fixed_means, fixed_vars, ys, run_means, run_vars,
                                          save_means, save_invstds, *_ws(ws))


def batchnorm_bwd_tiles(xs, dys, scales, shifts, save_means, save_invstds, dxs, dscales, dshifts, N, C, H, W, relu=0,
                        dy_halo=0, beta_data=0.0, beta_param=0.0, ws=None):
    return _n().adh_batchnorm2d_bwd_tiles(_dt(xs[0]), len(xs), N, C, H, W, relu, dy_halo, xs, dys, scales, shifts,
                                          save_means, save_invstds, dxs, dscales, dshifts, beta_data, beta_param,
                                          *_ws(ws))


def relu_fwd(x, y):
    return _n().adh_relu_fwd(_dt(x), x.numel(), x, y)


def relu_bwd(y, dy, dx, beta=0.0):
    return _n().adh_relu_bwd(_dt(y), y.numel(), y, dy, dx, beta)


def sum_fwd(xs, y):
    return _n().adh_sum_fwd(_dt(y), len(xs), y.numel(), xs, y)


def scale_add(alpha, x, beta, y):
    """y = alpha*x + beta*y over flat fp32 tensors."""
    return _n().adh_scale_add_f32(y.numel(), alpha, x, beta, y)


def add_online(alpha, x, y):
    """y = y + alpha*(x - y)."""
    return _n().adh_add_online_f32(y.numel(), alpha, x, y)


def stat_step(rate, avg_stat, running_stat, stat):
    return _n().adh_stat_step_f32(stat.numel(), rate, avg_stat, running_stat, stat)


def flat_store(arrays, flat, offset=0):
    """Copy the arrays, in order, into consecutive ranges of `flat` starting at element `offset`."""
    return _n().adh_flat_store_f32(len(arrays), arrays, arrays, offset, flat)


def flat_load(arrays, flat, offset=0):
    """The inverse of flat_store: consecutive ranges of `flat` into the arrays."""
    return _n().adh_flat_load_f32(len(arrays), arrays, arrays, offset, flat)


def sgd_step(grads, param, momentum_grad, lagged_param=None, sum_grad=None, l2_reg=0.0, momentum=0.0, step_size=0.0,
             next_step_size=0.0, nesterov=False):
    """One fused optimizer update over flat fp32 vectors; grads is the list of per-rank gradient vectors."""
    return _n().adh_sgd_step_f32(param.numel(), len(grads), grads, l2_reg, momentum, step_size, next_step_size,
                                 int(bool(nesterov)), param, momentum_grad, lagged_param, sum_grad)


def pool_fwd_tiles(mode, xs, ys, N, C, HP, WP, wh, ww, sh, sw):
    return _n().adh_pool2d_slab_fwd_tiles(_dt(xs[0]), mode, len(xs), N, C, HP, WP, wh, ww, sh, sw, xs, ys)


def pool_bwd_tiles(mode, xs, ys, dys, dxs, N, C, HP, WP, wh, ww, sh, sw, beta=0.0):
    return _n().adh_pool2d_slab_bwd_tiles(_dt(dys[0]), mode, len(dys), N, C, HP, WP, wh, ww, sh, sw, xs, ys, dys, dxs,
                                          beta)


def pool_unpadded_fwd_tiles(mode, xs, ys, N, C, H, W, wh, ww, sh, sw, pad_h, pad_w):
    """Pooling over row tiles without halo: rows outside a tile come from its neighbours, zeros outside the tensor."""
    return _n().adh_pool2d_unpadded_fwd_tiles(_dt(xs[0]), mode, len(xs), N, C, H, W, wh, ww, sh, sw, pad_h, pad_w, xs,
                                              ys)


def pool_unpadded_bwd_tiles(mode, xs, ys, dys, dxs, N, C, H, W, wh, ww, sh, sw, pad_h, pad_w, beta=0.0):
    return _n().adh_pool2d_unpadded_bwd_tiles(_dt(dys[0]), mode, len(dys), N, C, H, W, wh, ww, sh, sw, pad_h, pad_w, xs,
                                              ys, dys, dxs, beta)


def conv_bwd_filter_tiles(xs, dys, dw, N, Cin, Cout, H, W, beta=0.0, ws=None, unexchanged=False):
    fn = (_n().adh_conv3x3_slab_bwd_filter_tiles_unexchanged if unexchanged
          else _n().adh_conv3x3_slab_bwd_filter_tiles)
    return fn(_dt(xs[0]), len(xs), N, Cin, Cout, H, W, xs, dys, dw, beta, *_ws(ws))


def softmax_fwd(x, y):
    N, C = x.shape
    return _n().adh_softmax_fwd(C, N, x, y)


def softmax_xent_fwd(x, label, y, loss):
    N, C = x.shape
    return _n().adh_softmax_xent_fwd(C, N, x, label, y, loss)


def softmax_nll_loss_fwd(y, label, loss):
    N, C = y.shape
    return _n().adh_softmax_nll_loss_fwd(C, N, y, label, loss)


def softmax_nll_loss_bwd(y, label, dloss, dx):
    N, C = y.shape
    return _n().adh_softmax_nll_loss_bwd(C, N, y, label, dloss, dx)


def softmax_nll_loss_bwd_scaled(y, label, dloss, dloss_all, beta, dx):
    """dx = beta*dx + dl*(y - onehot); dloss None: every example's dl is dloss_all."""
    N, C = y.shape
    return _n().adh_softmax_nll_loss_bwd_scaled(C, N, y, label, dloss, dloss_all, beta, dx)


def softmax_xent_fwd_bwd(x, label, dloss, dloss_all, y, loss, beta, dx):
    N, C = x.shape
    return _n().adh_softmax_xent_fwd_bwd(C, N, x, label, dloss, dloss_all, y, loss, beta, dx)


def conv_kernel_name(which, dtype, K, N, Cin, Cout, H, W, beta=0.0):
    """Name of the kernel instance a 3x3 forward / backward-data call of this shape runs."""
    buf = ctypes.create_string_buffer(256)
    check(lib().adh_conv3x3_kernel_name(which, dtype, K, N, Cin, Cout, H, W, beta, buf, 256), "kernel name")
    return buf.value.decode()
