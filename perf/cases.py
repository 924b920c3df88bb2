"""What a user of this library has it do, as timed cases through the public entry points of arraydiff_cuda_amd.capi.

A case is one piece of a spatially-parallel net (an activation split into K row tiles) and one pass through it:

  halo    exchange of an activation's halos and reduction of a gradient's: what surrounds every halo-padded op
  pack    an unsplit tensor into halo-padded row tiles and the tiles' interiors back
  loss    softmax cross-entropy forward and backward, and a channel slice
  slab    a 3x3 convolution layer over halo-padded tiles, forward and backward, from the unsplit tensor to its gradient
  block   a 3x3 stride-1 convolution layer over tiles without halo, forward (with the residual sum or not) and backward
  proj    the entry of a projection block: 3x3 and 1x1 convolution at one stride over tiles without halo, forward and backward
  stem    the first convolution of a net (at most three input channels, with a bias) over halo-padded tiles, forward, filter
          gradient and bias gradient (a net wants no gradient of its image)
  shell   what stands between the convolutions: batch norm with rectifier and 3x3 / 2 max pooling, forward and backward
  update  the optimizer's step: every rank's gradients into flat vectors, the Nesterov update, the parameters back

Ht x W is one tile's interior; N images, C channels, K tiles, p the halo's width."""
import math

import torch

from arraydiff_cuda_amd import capi

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
CODES = {"f32": capi.ADH_F32, "bf16": capi.ADH_BF16}
PASSES = (capi.ADH_CONV_FWD, capi.ADH_CONV_BWD_DATA, capi.ADH_CONV_BWD_FILTER)


def listed():
    return [
        # the smallest calls: halo strips of 0.5 MB between four tiles of a 56 x 56 activation
        {"name": "halo f32 64ch 4x14x56", "kind": "halo", "dtype": "f32", "N": 32, "C": 64, "Ht": 14, "W": 56, "K": 4, "p": 1,
         "columns": False},
        # the same activation scattered and gathered
        {"name": "pack f32 64ch 4x14x56", "kind": "pack", "dtype": "f32", "N": 32, "C": 64, "Ht": 14, "W": 56, "K": 4, "p": 1},
        # the classifier's loss and a channel slice
        {"name": "loss 256x1000", "kind": "loss", "N": 256, "classes": 1000, "images": 32, "C": 64, "H": 56, "W": 56, "from": 16,
         "count": 32},
        # the padded-tile convolution layer of configs[1] and [2]
        {"name": "slab f32 64ch 4x14x56", "kind": "slab", "dtype": "f32", "N": 32, "Cin": 64, "Cout": 64, "Ht": 14, "W": 56, "K": 4},
        # the high-resolution bf16 layer of configs[4]: the largest case
        {"name": "slab bf16 64ch 8x128x2048", "kind": "slab", "dtype": "bf16", "N": 2, "Cin": 64, "Cout": 64, "Ht": 128, "W": 2048,
         "K": 8},
        # a bf16 layer at an odd width
        {"name": "slab bf16 128ch 4x64x255", "kind": "slab", "dtype": "bf16", "N": 8, "Cin": 128, "Cout": 128, "Ht": 64, "W": 255,
         "K": 4},
        # the first and the last but one stage of the trained ResNet-18 variant (256 x 256 images, batch 32)
        {"name": "block f32 64ch 4x32x128", "kind": "block", "dtype": "f32", "N": 32, "Cin": 64, "Cout": 64, "Ht": 32, "W": 128,
         "K": 4, "residual": True, "window": False},
        {"name": "block f32 512ch 4x4x16", "kind": "block", "dtype": "f32", "N": 32, "Cin": 512, "Cout": 512, "Ht": 4, "W": 16,
         "K": 4, "residual": False, "window": True},
        # its second projection block
        {"name": "proj f32 128ch 4x16x64", "kind": "proj", "dtype": "f32", "N": 32, "Cin": 128, "Cout": 256, "Ht": 16, "W": 64,
         "K": 4, "s": 2},
        # its stem
        {"name": "stem f32 7x7 4x64x256", "kind": "stem", "N": 32, "Cin": 3, "Cout": 64, "OH": 64, "OW": 256, "K": 4, "k": 7, "s": 1},
        # what follows the stem
        {"name": "shell f32 64ch 4x64x256", "kind": "shell", "dtype": "f32", "N": 32, "C": 64, "Ht": 64, "W": 256, "K": 4},
        # its optimizer step
        {"name": "update 11.7M x4", "kind": "update", "total": 11689512, "arrays": 56, "ranks": 4, "nesterov": True},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _channels(rng, lo, hi):
    """Mostly the multiples of 16 that nets have, any number otherwise."""
    c = _log(rng, lo, hi)
    return max(lo, c // 16 * 16) if rng.random() < 0.7 else c


def _draw(rng):
    kind = rng.choice(("halo", "pack", "loss", "slab", "slab", "block", "block", "proj", "stem", "shell", "update"))
    dtype = rng.choice(("f32", "bf16"))
    if kind == "halo":
        p = rng.choice((1, 1, 2, 3))
        return {"kind": kind, "dtype": dtype, "N": _log(rng, 1, 32), "C": _log(rng, 3, 256), "Ht": _log(rng, 2 * p, 128),
                "W": _log(rng, 7, 512), "K": rng.randint(2, 8), "p": p, "columns": rng.random() < 0.25}
    if kind == "pack":
        p = rng.choice((1, 1, 2, 3))
        return {"kind": kind, "dtype": dtype, "N": _log(rng, 1, 32), "C": _log(rng, 3, 256), "Ht": _log(rng, p, 128),
                "W": _log(rng, 7, 2048), "K": rng.randint(1, 8), "p": p}
    if kind == "loss":
        C = _log(rng, 4, 256)
        a = rng.randrange(C)
        return {"kind": kind, "N": _log(rng, 8, 4096), "classes": _log(rng, 10, 4000), "images": _log(rng, 1, 32), "C": C,
                "H": _log(rng, 7, 112), "W": _log(rng, 7, 112), "from": a, "count": rng.randint(1, C - a)}
    if kind == "slab":
        return {"kind": kind, "dtype": dtype, "N": _log(rng, 1, 32), "Cin": _channels(rng, 16, 512), "Cout": _channels(rng, 16, 512),
                "Ht": _log(rng, 4, 128), "W": _log(rng, 7, 2048), "K": rng.randint(1, 8)}
    if kind == "block":
        W = _log(rng, 7, 512)
        return {"kind": kind, "dtype": dtype, "N": _log(rng, 1, 32), "Cin": _channels(rng, 16, 512), "Cout": _channels(rng, 16, 512),
                "Ht": _log(rng, 4, 64), "W": W if dtype == "f32" else max(8, W // 8 * 8), "K": rng.randint(1, 8),
                "residual": dtype == "f32" and rng.random() < 0.5, "window": False}
    if kind == "proj":
        Cin = _channels(rng, 16, 256)
        return {"kind": kind, "dtype": dtype, "N": _log(rng, 1, 32), "Cin": Cin, "Cout": rng.choice((Cin, 2 * Cin)),
                "Ht": 2 * _log(rng, 2, 32), "W": 2 * _log(rng, 4, 128), "K": rng.randint(1, 8), "s": 2}
    if kind == "stem":
        s = rng.choice((1, 2))
        return {"kind": kind, "N": _log(rng, 1, 32), "Cin": rng.choice((1, 3, 3)), "Cout": rng.choice((16, 32, 48, 64, 64, 96)),
                "OH": _log(rng, 7, 64), "OW": _log(rng, 14, 256), "K": rng.randint(1, 8), "k": rng.choice((3, 5, 7, 7)), "s": s}
    if kind == "shell":
        return {"kind": kind, "dtype": dtype, "N": _log(rng, 1, 32), "C": _channels(rng, 16, 512), "Ht": 2 * _log(rng, 1, 64),
                "W": _log(rng, 7, 512), "K": rng.randint(1, 8)}
    return {"kind": kind, "total": _log(rng, 200000, 30000000), "arrays": rng.randint(8, 60), "ranks": rng.randint(1, 8),
            "nesterov": rng.random() < 0.7}


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        # the rates that a layer of its kind reaches at the least favourable shapes keep the pass under the largest listed one's
        slow = case.get("dtype") == "bf16" and case["kind"] == "slab" and case["W"] % 8 != 0
        most = {"slab": 6e10 if slow else 2e11 if case.get("dtype") == "bf16" else 6e10, "block": 2e11 if case.get("dtype") == "bf16" else 6e10,
                "proj": 2e10, "stem": 7e10}.get(case["kind"], 1e12)
        if w["bytes"] <= 1e9 and w["flops"] <= most and _tile_bytes(case) <= 1e9:
            return case


def _tile_bytes(case):
    """Bytes of a halo case's tiles, of which only the strips are touched."""
    if case["kind"] != "halo":
        return 0
    return 4 * case["N"] * case["C"] * case["K"] * (case["Ht"] + 2 * case["p"]) * (case["W"] + 2 * case["p"])


def _stem_tile(c):
    return (c["OH"] - 1) * c["s"] + c["k"], (c["OW"] - 1) * c["s"] + c["k"]


def _pool_out(c):
    return c["Ht"] // 2, (c["W"] - 1) // 2 + 1


def _lengths(c):
    """Array lengths of a net's parameters: sizes over eight octaves, in turn, that sum to the total."""
    shares = [2.0 ** -(i % 8) for i in range(c["arrays"])]
    lens = [max(16, int(c["total"] * s / sum(shares))) for s in shares]
    lens[0] += c["total"] - sum(lens)
    return lens


class _Maker:
    """Tensors of one seed on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def uniform(self, shape, dtype="f32"):
        return (torch.rand(shape, device="cuda", generator=self.g) * 2 - 1).to(DTYPES[dtype])

    def normal(self, shape, dtype="f32", std=1.0):
        return (torch.randn(shape, device="cuda", generator=self.g) * std).to(DTYPES[dtype])

    def filter(self, co, ci, kh, kw, dtype="f32"):
        return self.normal((co, ci, kh, kw), dtype, math.sqrt(2.0 / (ci * kh * kw)))

    @staticmethod
    def empty(shape, dtype="f32"):
        return torch.empty(shape, device="cuda", dtype=DTYPES[dtype])


def _workspace(nbytes):
    return torch.empty(max(nbytes, 256) // 4 + 64, device="cuda")


def prepare(case, seed):
    m, c, kind = _Maker(seed), dict(case), case["kind"]
    s = {"case": c}
    dt = c.get("dtype", "f32")
    code = CODES[dt]
    if kind == "halo":
        wide = (c["N"], c["C"], c["Ht"] + 2 * c["p"], c["W"] + 2 * c["p"])
        s["acts"] = [m.uniform(wide, dt) for _ in range(c["K"])]
        # gradients of magnitudes at which repeated reductions stay finite
        s["grads"] = [m.normal(wide, dt, 1e-2) for _ in range(c["K"])]
    elif kind == "pack":
        N, C, H, W, p, K = c["N"], c["C"], c["Ht"] * c["K"], c["W"], c["p"], c["K"]
        s["x"] = m.uniform((N, C, H, W), dt)
        s["tiles"] = [m.empty((N, C, c["Ht"] + 2 * p, W + 2 * p), dt) for _ in range(K)]
        s["dtiles"] = [m.normal((N, C, c["Ht"] + 2 * p, W + 2 * p), dt) for _ in range(K)]
        s["y"] = m.empty((N, C, H, W), dt)
    elif kind == "loss":
        s["logits"] = m.normal((c["N"], c["classes"]), std=2.0)
        s["labels"] = torch.randint(0, c["classes"], (c["N"],), device="cuda", dtype=torch.int32, generator=m.g)
        s["y"], s["loss"], s["dx"] = torch.empty_like(s["logits"]), m.empty((c["N"],)), torch.empty_like(s["logits"])
        s["act"] = m.uniform((c["images"], c["C"], c["H"], c["W"]))
        s["part"] = m.empty((c["images"], c["count"], c["H"], c["W"]))
    elif kind == "slab":
        N, Ci, Co, Ht, W, K = c["N"], c["Cin"], c["Cout"], c["Ht"], c["W"], c["K"]
        s["x"] = m.uniform((N, Ci, Ht * K, W), dt)
        s["w"] = m.filter(Co, Ci, 3, 3, dt)
        s["dys"] = [m.normal((N, Co, Ht, W), dt) for _ in range(K)]
        s["tiles"] = [m.empty((N, Ci, Ht + 2, W + 2), dt) for _ in range(K)]
        s["dtiles"] = [m.empty((N, Ci, Ht + 2, W + 2), dt) for _ in range(K)]
        s["ys"] = [m.empty((N, Co, Ht, W), dt) for _ in range(K)]
        s["dx"], s["dw"] = torch.empty_like(s["x"]), m.empty((Co, Ci, 3, 3))
        s["ws"] = [_workspace(capi.conv_workspace_bytes(q, code, K, N, Ci, Co, Ht, W)) for q in PASSES]
    elif kind == "block":
        N, Ci, Co, Ht, W, K = c["N"], c["Cin"], c["Cout"], c["Ht"], c["W"], c["K"]
        s["xs"] = [m.uniform((N, Ci, Ht, W), dt) for _ in range(K)]
        s["w"] = m.filter(Co, Ci, 3, 3, dt)
        s["dys"] = [m.normal((N, Co, Ht, W), dt) for _ in range(K)]
        s["res"] = [m.uniform((N, Co, Ht, W), dt) for _ in range(K)] if c["residual"] else None
        s["ys"] = [m.empty((N, Co, Ht, W), dt) for _ in range(K)]
        s["dxs"], s["dw"] = [torch.empty_like(x) for x in s["xs"]], m.empty((Co, Ci, 3, 3))
        s["geometry"] = (3, 3, 1, 1, 1, 1, 1, 1)
        if c["window"]:
            s["ws"] = [_workspace(capi.conv2d_unpadded_workspace_bytes(q, code, K, N, Ci, Co, Ht, W, *s["geometry"])) for q in PASSES]
        else:
            s["ws"] = [_workspace(capi.conv_workspace_bytes(q, code, K, N, Ci, Co, Ht, W)) for q in PASSES]
    elif kind == "proj":
        N, Ci, Co, Ht, W, K, st = c["N"], c["Cin"], c["Cout"], c["Ht"], c["W"], c["K"], c["s"]
        s["xs"] = [m.uniform((N, Ci, Ht, W), dt) for _ in range(K)]
        s["legs"] = []
        for k in (3, 1):  # the 3x3 and the projection itself
            geometry = (k, k, st, st, 1, 1, k // 2, k // 2)
            out = (N, Co, Ht // st, (W + 2 * (k // 2) - k) // st + 1)
            s["legs"].append({
                "geometry": geometry, "w": m.filter(Co, Ci, k, k, dt), "dys": [m.normal(out, dt) for _ in range(K)],
                "ys": [m.empty(out, dt) for _ in range(K)], "dxs": [torch.empty_like(x) for x in s["xs"]],
                "dw": m.empty((Co, Ci, k, k)),
                "ws": [_workspace(capi.conv2d_unpadded_workspace_bytes(q, code, K, N, Ci, Co, Ht, W, *geometry)) for q in PASSES]})
    elif kind == "stem":
        N, Ci, Co, K = c["N"], c["Cin"], c["Cout"], c["K"]
        HP, WP = _stem_tile(c)
        s["geometry"] = (c["k"], c["k"], c["s"], c["s"], 1, 1)
        s["xs"] = [m.uniform((N, Ci, HP, WP)) for _ in range(K)]
        s["w"], s["bias"] = m.filter(Co, Ci, c["k"], c["k"]), m.normal((Co,), std=0.1)
        s["dys"] = [m.normal((N, Co, c["OH"], c["OW"])) for _ in range(K)]
        s["ys"] = [m.empty((N, Co, c["OH"], c["OW"])) for _ in range(K)]
        s["dw"], s["db"] = m.empty((Co, Ci, c["k"], c["k"])), m.empty((Co,))
        s["ws"] = [_workspace(capi.conv2d_workspace_bytes(q, code, K, N, Ci, Co, HP, WP, *s["geometry"])) for q in PASSES]
        s["wsb"] = _workspace(capi.conv_bwd_bias_workspace_bytes(K, N, Co))
    elif kind == "shell":
        N, C, Ht, W, K = c["N"], c["C"], c["Ht"], c["W"], c["K"]
        full, pooled = (N, C, Ht, W), (N, C) + _pool_out(c)
        # a convolution's outputs: channels about means of their own
        s["xs"] = [(torch.randn(full, device="cuda", generator=m.g) + m.normal((1, C, 1, 1))).to(DTYPES[dt]) for _ in range(K)]
        s["dps"] = [m.normal(pooled, dt) for _ in range(K)]
        s["scales"], s["shifts"] = ([m.normal((C,), std=0.1) + v for _ in range(K)] for v in (1.0, 0.0))
        for name, shape in (("acts", full), ("dacts", full), ("dxs", full), ("pools", pooled)):
            s[name] = [m.empty(shape, dt) for _ in range(K)]
        for name in ("rmeans", "rvars", "means", "invstds", "dscales", "dshifts"):
            s[name] = [m.empty((C,)) for _ in range(K)]
        s["ws"] = _workspace(capi.batchnorm_workspace_bytes(K, N, C))
    elif kind == "update":
        lens = _lengths(c)
        s["params"] = [m.normal((n,), std=0.05) for n in lens]
        s["grads"] = [[m.normal((n,), std=1e-3) for n in lens] for _ in range(c["ranks"])]
        s["flat"] = [m.empty((c["total"],)) for _ in range(c["ranks"])]
        s["param"] = torch.cat(s["params"])
        s["momentum"], s["lagged"] = m.normal((c["total"],), std=1e-3), m.empty((c["total"],))
    else:
        raise ValueError(kind)
    return s


def _run_halo(s, c):
    grid = (c["K"], 1) if c["columns"] else (1, c["K"])
    size = (c["p"], c["W"], c["Ht"], c["C"], c["N"])
    capi.check(capi.halo_exchange(s["acts"], *grid, *size), "exchange")
    capi.check(capi.halo_reduce(s["grads"], *grid, *size), "reduce")
    return s["acts"], s["grads"]


def _run_pack(s, c):
    size = (c["K"], c["p"], c["W"], c["Ht"] * c["K"], c["C"], c["N"])
    capi.check(capi.tiles_pack(*size, s["x"], s["tiles"]), "pack")
    capi.check(capi.tiles_unpack(*size, s["dtiles"], s["y"]), "unpack")
    return s["tiles"], s["y"]


def _run_loss(s, c):
    capi.check(capi.softmax_xent_fwd(s["logits"], s["labels"], s["y"], s["loss"]), "softmax")
    capi.check(capi.softmax_nll_loss_bwd_scaled(s["y"], s["labels"], None, 1.0 / c["N"], 0.0, s["dx"]), "loss backward")
    capi.check(capi.slice_nchw(False, (c["W"], c["H"], c["count"]), c["images"], s["act"], (c["W"], c["H"], c["C"]), (0, 0, c["from"]),
                               s["part"], (c["W"], c["H"], c["count"]), (0, 0, 0)), "slice")
    return s["y"], s["loss"], s["dx"], s["part"]


def _run_slab(s, c):
    K, N, H = c["K"], c["N"], c["Ht"] * c["K"]
    size = (N, c["Cin"], c["Cout"], c["Ht"], c["W"])
    capi.check(capi.tiles_pack(K, 1, c["W"], H, c["Cin"], N, s["x"], s["tiles"]), "pack")
    capi.check(capi.conv_fwd_tiles(s["tiles"], s["w"], s["ys"], *size, ws=s["ws"][0]), "forward")
    capi.check(capi.conv_bwd_filter_tiles(s["tiles"], s["dys"], s["dw"], *size, ws=s["ws"][2]), "filter gradient")
    capi.check(capi.conv_bwd_data_tiles(s["w"], s["dys"], s["dtiles"], *size, ws=s["ws"][1], reduced=True), "input gradient")
    capi.check(capi.tiles_unpack(K, 1, c["W"], H, c["Cin"], N, s["dtiles"], s["dx"]), "unpack")
    return s["ys"], s["dw"], s["dx"]


def _run_block(s, c):
    size = (c["N"], c["Cin"], c["Cout"], c["Ht"], c["W"])
    if c["window"]:
        size += s["geometry"]
        capi.check(capi.conv2d_unpadded_fwd_tiles(s["xs"], s["w"], s["ys"], *size, ws=s["ws"][0]), "forward")
        capi.check(capi.conv2d_unpadded_bwd_filter_tiles(s["xs"], s["dys"], s["dw"], *size, ws=s["ws"][2]), "filter gradient")
        capi.check(capi.conv2d_unpadded_bwd_data_tiles(s["w"], s["dys"], s["dxs"], *size, ws=s["ws"][1]), "input gradient")
        return s["ys"], s["dw"], s["dxs"]
    if c["residual"]:
        capi.check(capi.conv_unpadded_fwd_residual_tiles(s["xs"], s["w"], s["res"], s["ys"], *size), "forward")
    else:
        capi.check(capi.conv_unpadded_fwd_tiles(s["xs"], s["w"], s["ys"], *size, ws=s["ws"][0]), "forward")
    capi.check(capi.conv_unpadded_bwd_filter_tiles(s["xs"], s["dys"], s["dw"], *size, ws=s["ws"][2]), "filter gradient")
    capi.check(capi.conv_unpadded_bwd_data_tiles(s["w"], s["dys"], s["dxs"], *size, ws=s["ws"][1]), "input gradient")
    return s["ys"], s["dw"], s["dxs"]


def _run_proj(s, c):
    out = []
    for leg in s["legs"]:
        size = (c["N"], c["Cin"], c["Cout"], c["Ht"], c["W"]) + leg["geometry"]
        capi.check(capi.conv2d_unpadded_fwd_tiles(s["xs"], leg["w"], leg["ys"], *size, ws=leg["ws"][0]), "forward")
        out.append(leg["ys"])
    for leg in s["legs"]:
        size = (c["N"], c["Cin"], c["Cout"], c["Ht"], c["W"]) + leg["geometry"]
        capi.check(capi.conv2d_unpadded_bwd_filter_tiles(s["xs"], leg["dys"], leg["dw"], *size, ws=leg["ws"][2]), "filter gradient")
        # the second leg's input gradient is added to the first one's
        first = s["legs"][0]["dxs"]
        capi.check(capi.conv2d_unpadded_bwd_data_tiles(leg["w"], leg["dys"], first, *size, beta=0.0 if leg is s["legs"][0] else 1.0,
                                                       ws=leg["ws"][1]), "input gradient")
        out.append(leg["dw"])
    return out, s["legs"][0]["dxs"]


def _run_stem(s, c):
    HP, WP = _stem_tile(c)
    size = (c["N"], c["Cin"], c["Cout"], HP, WP) + s["geometry"]
    capi.check(capi.conv2d_fwd_bias_tiles(s["xs"], s["w"], [s["bias"]] * c["K"], s["ys"], *size, ws=s["ws"][0]), "forward")
    capi.check(capi.conv_bwd_bias_tiles(s["dys"], s["db"], c["N"], c["Cout"], c["OH"], c["OW"], ws=s["wsb"]), "bias gradient")
    capi.check(capi.conv2d_bwd_filter_tiles(s["xs"], s["dys"], s["dw"], *size, ws=s["ws"][2]), "filter gradient")
    return s["ys"], s["dw"], s["db"]


def _run_shell(s, c):
    size = (c["N"], c["C"], c["Ht"], c["W"])
    window = (3, 3, 2, 2, 1, 1)
    capi.check(capi.batchnorm_fwd_tiles(s["xs"], s["scales"], s["shifts"], s["acts"], *size, relu=1, run_means=s["rmeans"],
                                        run_vars=s["rvars"], save_means=s["means"], save_invstds=s["invstds"], ws=s["ws"]), "batch norm")
    capi.check(capi.pool_unpadded_fwd_tiles(capi.ADH_POOL_MAX, s["acts"], s["pools"], *size, *window), "pooling")
    capi.check(capi.pool_unpadded_bwd_tiles(capi.ADH_POOL_MAX, s["acts"], s["pools"], s["dps"], s["dacts"], *size, *window), "pooling gradient")
    capi.check(capi.batchnorm_bwd_tiles(s["xs"], s["dacts"], s["scales"], s["shifts"], s["means"], s["invstds"], s["dxs"], s["dscales"],
                                        s["dshifts"], *size, relu=1, ws=s["ws"]), "batch norm gradient")
    return s["acts"], s["pools"], s["dacts"], s["dxs"], s["dscales"], s["dshifts"], s["rmeans"], s["rvars"]


def _run_update(s, c):
    for grads, flat in zip(s["grads"], s["flat"]):
        capi.check(capi.flat_store(grads, flat), "store")
    capi.check(capi.sgd_step(s["flat"], s["param"], s["momentum"], lagged_param=s["lagged"], l2_reg=1e-4, momentum=0.9, step_size=1e-3,
                             next_step_size=1e-3, nesterov=c["nesterov"]), "update")
    capi.check(capi.flat_load(s["params"], s["param"]), "load")
    return s["param"], s["momentum"], s["lagged"], s["params"]


_RUN = {"halo": _run_halo, "pack": _run_pack, "loss": _run_loss, "slab": _run_slab, "block": _run_block, "proj": _run_proj,
        "stem": _run_stem, "shell": _run_shell, "update": _run_update}


def run(state):
    return _RUN[state["case"]["kind"]](state, state["case"])


def work(case):
    """Every input read once and every output written once; a multiplication and its addition are two operations."""
    c, kind = case, case["kind"]
    e = 2 if c.get("dtype") == "bf16" else 4
    if kind == "halo":
        strip = c["p"] * c["N"] * c["C"] * (c["Ht"] if c["columns"] else c["W"]) * e
        moves = 2 * (c["K"] - 1)
        return {"bytes": moves * strip * 5, "flops": moves * strip / e}  # exchange: read, write; reduce: two reads, one write
    if kind == "pack":
        H, Hp = c["Ht"] * c["K"], (c["Ht"] + 2 * c["p"]) * c["K"]
        return {"bytes": c["N"] * c["C"] * e * (3 * H * c["W"] + Hp * (c["W"] + 2 * c["p"])), "flops": 0}
    if kind == "loss":
        rows = c["N"] * c["classes"]
        return {"bytes": 4 * (3 * rows + 2 * c["N"]) + 8 * c["images"] * c["count"] * c["H"] * c["W"], "flops": 8 * rows}
    if kind in ("slab", "block"):
        pixels = c["N"] * c["K"] * c["Ht"] * c["W"]
        y = pixels * c["Cout"]
        filt = c["Cin"] * c["Cout"] * 9
        return {"bytes": e * (2 * pixels * c["Cin"] + (3 if c.get("residual") else 2) * y + filt) + 4 * filt,
                "flops": 3 * 2 * 9 * pixels * c["Cin"] * c["Cout"]}
    if kind == "proj":
        pixels = c["N"] * c["K"] * c["Ht"] * c["W"]
        y = pixels // (c["s"] * c["s"]) * c["Cout"]
        filt = c["Cin"] * c["Cout"] * 10
        return {"bytes": e * (2 * pixels * c["Cin"] + 4 * y + filt) + 4 * filt, "flops": 3 * 2 * 10 * c["Cin"] * y}
    if kind == "stem":
        HP, WP = _stem_tile(c)
        y = c["N"] * c["K"] * c["Cout"] * c["OH"] * c["OW"]
        filt = c["Cin"] * c["Cout"] * c["k"] * c["k"]
        return {"bytes": 4 * (c["N"] * c["K"] * c["Cin"] * HP * WP + 2 * y + 2 * filt), "flops": 2 * 2 * y * c["Cin"] * c["k"] * c["k"] + 2 * y}
    if kind == "shell":
        OH, OW = _pool_out(c)
        full, pooled = c["N"] * c["C"] * c["K"] * c["Ht"] * c["W"], c["N"] * c["C"] * c["K"] * OH * OW
        return {"bytes": e * (4 * full + 2 * pooled), "flops": 20 * full}
    n, r = c["total"], c["ranks"]
    return {"bytes": 4 * n * (2 * r + 6), "flops": n * (r + 6)}


def tolerance(case):
    if case["kind"] in ("halo", "pack"):
        return "exact"  # copies, and sums of two terms
    if case.get("dtype") == "bf16":
        return {"rel": 1e-2, "max": 5e-2}  # one rounding of a result to bf16
    return {"rel": 1e-5}  # sums of 32-bit products in another order
