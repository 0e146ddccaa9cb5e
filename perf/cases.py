"""The work that a user of this engine has it do, as cases that can be timed
and compared: ggml_mul_mat and ggml_flash_attn_ext with each weight type and
precision, LayerNorm, image preprocessing, the FPN neck, the tracker's memory
attention and whole image encodes, through the C ABI's Python binding.

Sizes are the engine's own: SAM 3's ViT at 1008 px (72 × 72 tokens, width
1024, 16 heads, MLP 4736, windows of 24 × 24 tokens), SAM 2.1's Hiera
encoders, a memory bank of up to 7 frames of 64 × 64 tokens, camera frames.
Weights are random (N(0, 0.02)), quantized as the model files hold them.
"""
import math
import os
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sam3.cpp_amd"))
import s3e  # noqa: E402

DEV = "cuda"
TYPES = {"q4_0": s3e.TYPE_Q4_0, "q4_1": s3e.TYPE_Q4_1, "q8_0": s3e.TYPE_Q8_0, "f16": s3e.TYPE_F16,
         "f32": s3e.TYPE_F32}
BYTES_PER_WEIGHT = {"q4_0": 18 / 32, "q4_1": 20 / 32, "q8_0": 34 / 32, "f16": 2.0, "f32": 4.0}

# (N, K) of the linears in use: the ViT's qkv, proj, fc1 and fc2; Hiera-B+'s
# and Hiera-T's; the memory attention's
LINEARS = [(3072, 1024), (1024, 1024), (4736, 1024), (1024, 4736), (672, 224), (896, 3584), (1152, 384), (384, 1536),
           (768, 256), (256, 64), (2048, 256), (256, 2048)]


def listed():
    return [
        # a few decoder tokens through one projection: launches and latency
        {"name": "linear_tokens_q4_0", "kind": "linear", "type": "q4_0", "M": 7, "N": 1024, "K": 1024, "bias": True},
        # the ViT's fc1 over all tokens of a 1008 px image, the largest of its linears
        {"name": "linear_fc1_q4_0", "kind": "linear", "type": "q4_0", "M": 5184, "N": 4736, "K": 1024, "bias": True},
        # fc2 over part of an image's tokens: a ragged row count, a long K
        {"name": "linear_fc2_q8_0", "kind": "linear", "type": "q8_0", "M": 1601, "N": 1024, "K": 4736, "bias": True},
        # the qkv projection of an F16 file
        {"name": "linear_qkv_f16", "kind": "linear", "type": "f16", "M": 5184, "N": 3072, "K": 1024, "bias": True},
        # windowed ViT attention from f32 tensors at f32 precision (quantized files), V a strided view
        {"name": "attn_window_f32", "kind": "attn", "prec": "f32", "D": 64, "B": 9, "nh": 16, "Nq": 576, "Nkv": 576,
         "layout": "vit"},
        # global ViT attention on F16 tensors
        {"name": "attn_global_f16", "kind": "attn", "prec": "f16", "D": 64, "B": 1, "nh": 16, "Nq": 5184, "Nkv": 5184,
         "layout": "heads"},
        # LayerNorm over an image's tokens
        {"name": "layer_norm", "kind": "layer_norm", "rows": 5184, "n": 1024},
        # a full-HD camera frame to the SAM 3 encoder's input
        {"name": "preprocess_1080p", "kind": "preprocess", "w": 1920, "h": 1080, "size": 1008, "norm": 0},
        # the four FPN levels of a quantized SAM 3 file (F32 convolutions)
        {"name": "neck_q4_0", "kind": "neck", "type": "q4_0", "img": 1008},
        # the tracker's memory attention with a full bank: 7 frames and 16 object pointers
        {"name": "mem_attn_q8_0", "kind": "mem_attn", "type": "q8_0", "side": 64, "frames": 7, "ptr": 64},
        # a frame through SAM 2.1 Hiera-Tiny, F16 weights
        {"name": "hiera_t_f16", "kind": "hiera", "variant": "hiera_t", "type": "f16", "img": 1024},
        # a frame through the SAM 3 ViT and tracker neck, Q4_0 weights
        {"name": "sam3_frame_q4_0", "kind": "sam3", "type": "q4_0", "neck": 1},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges."""
    kind = rng.choice(["linear"] * 4 + ["attn"] * 3 + ["layer_norm", "preprocess", "neck", "mem_attn", "hiera", "sam3"])
    if kind == "linear":
        if rng.random() < 0.7:
            N, K = rng.choice(LINEARS)
        else:
            N, K = _log_int(rng, 33, 4736), 32 * _log_int(rng, 2, 148)
        return {"kind": kind, "type": rng.choice(["q4_0", "q4_0", "q8_0", "q8_0", "f16", "q4_1", "f32"]),
                "M": _log_int(rng, 1, 5184), "N": N, "K": K, "bias": rng.random() < 0.8}
    if kind == "attn":
        prec = rng.choice(["f16", "f32", "f32", "default"])
        form = rng.choice(["vit_window", "vit_global", "hiera_window", "hiera_pooled", "memory", "any"])
        layout = rng.choice(["heads", "vit", "tokens"])
        if form == "vit_window":
            D, B, nh, Nq = 64, rng.randint(1, 9), 16, rng.choice([576, 196, 64, rng.randint(50, 576)])
            Nkv = Nq
        elif form == "vit_global":
            D, B, nh, Nq = 64, 1, 16, _log_int(rng, 576, 5184)
            Nkv = Nq
        elif form == "hiera_window":
            D, B, nh = rng.choice([96, 56, 72]), rng.choice([1, 25, 64, 256]), rng.choice([1, 2, 4, 8])
            Nq = Nkv = rng.choice([64, 16, 196, 49])
        elif form == "hiera_pooled":
            D, B, nh = rng.choice([96, 56, 72]), rng.choice([25, 64, 256]), rng.choice([2, 4, 8])
            Nkv = rng.choice([64, 16, 196])
            Nq = Nkv // 4
        elif form == "memory":
            D, B, nh, Nq, Nkv = 256, 1, 1, _log_int(rng, 256, 4096), _log_int(rng, 1000, 28736)
            prec = "f16" if prec == "f16" else "default"
        else:
            D, B, nh = 4 * rng.randint(8, 32), rng.randint(1, 3), rng.randint(1, 8)
            Nq, Nkv = _log_int(rng, 1, 2000), _log_int(rng, 1, 2000)
        return {"kind": kind, "prec": prec, "D": D, "B": B, "nh": nh, "Nq": Nq, "Nkv": Nkv, "layout": layout}
    if kind == "layer_norm":
        return {"kind": kind, "rows": _log_int(rng, 1, 20736), "n": rng.choice([1024, 256, 96, 192, 384, 768, 224, 448,
                                                                                 896, 32 * rng.randint(1, 64)])}
    if kind == "preprocess":
        w, h = rng.choice([(1920, 1080), (1280, 720), (640, 480), (3840, 2160),
                           (_log_int(rng, 200, 4000), _log_int(rng, 200, 3000))])
        return {"kind": kind, "w": w, "h": h, "size": rng.choice([1008, 1024, 32 * rng.randint(8, 32)]),
                "norm": rng.randint(0, 1)}
    if kind == "neck":
        return {"kind": kind, "type": rng.choice(["q8_0", "f16", "f32"]), "img": rng.choice([1008, 672, 336])}
    if kind == "mem_attn":
        return {"kind": kind, "type": rng.choice(["q8_0", "f16", "q4_0"]), "side": rng.randint(12, 64),
                "frames": rng.randint(1, 7), "ptr": 4 * rng.randint(0, 16)}
    if kind == "hiera":
        return {"kind": kind, "variant": rng.choice(["hiera_t", "hiera_s", "hiera_b+", "hiera_l"]),
                "type": rng.choice(["f16", "q8_0", "q4_0"]), "img": rng.choice([1024, 512, 32 * rng.randint(12, 31)])}
    return {"kind": "sam3", "type": rng.choice(["q8_0", "f16", "q4_1"]), "neck": rng.randint(1, 2)}


# ---- what a program holds before the call ----------------------------------
_held = {}


def _ctx():
    if "ctx" not in _held:
        _held["ctx"] = s3e.Context(0)
    return _held["ctx"]


def _state(key, write):
    """The loaded model and the state of a model file that `write` makes; one per model, as a program keeps them."""
    if key not in _held:
        with tempfile.TemporaryDirectory() as folder:
            path = os.path.join(folder, "model.ggml")
            write(path)
            model = s3e.Model(_ctx(), path)
        _held[key] = s3e.State(_ctx(), model, key[-1] if key[0] == "hiera" else 0)
    return _held[key]


def _buf(t):
    return s3e.DeviceView(t.data_ptr(), t.numel() * t.element_size())


class _OnDevice:
    """A state tensor's memory, for torch to read where it lies."""

    def __init__(self, view):
        self.view = view
        self.__cuda_array_interface__ = {"shape": (view.nbytes // 4,), "typestr": "<f4", "data": (view.ptr, False),
                                         "version": 2}


def _tensors(state, names):
    return {n: torch.as_tensor(_OnDevice(state.device_view(n)), device=DEV) for n in names}


def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device=DEV, dtype=torch.float32)


def _weight_codes(kind, W):
    """Block codes of weights W [N][K] as the reference quantizers choose them: (codes [N][K/32][32] from 0 or signed,
    fp16 scales [N][K/32], fp16 minima or None)."""
    b = W.reshape(W.shape[0], -1, 32)
    if kind == "q8_0":
        d = b.abs().amax(-1) / 127
        inv = torch.where(d > 0, 1 / d, torch.zeros_like(d))
        return torch.round(b * inv[..., None]), d.half(), None
    if kind == "q4_0":
        m = torch.gather(b, -1, b.abs().argmax(-1, keepdim=True))[..., 0]
        d = m / -8
        inv = torch.where(d != 0, 1 / d, torch.zeros_like(d))
        return torch.clamp(torch.floor(b * inv[..., None] + 8.5), max=15), d.half(), None
    lo, hi = b.amin(-1), b.amax(-1)
    d = (hi - lo) / 15
    inv = torch.where(d > 0, 1 / d, torch.zeros_like(d))
    return torch.clamp(torch.floor((b - lo[..., None]) * inv[..., None] + 0.5), max=15), d.half(), lo.half()


def _ggml_bytes(kind, W):
    if kind == "f32":
        return W.cpu().numpy()
    if kind == "f16":
        return W.half().cpu().numpy()
    q, d, m = _weight_codes(kind, W)
    parts = [x[..., None].view(torch.uint8) for x in (d, m) if x is not None]
    if kind == "q8_0":
        parts.append(q.to(torch.int8).view(torch.uint8))
    else:
        q = q.to(torch.uint8)
        parts.append(q[..., :16] | (q[..., 16:] << 4))
    return torch.cat(parts, -1).reshape(W.shape[0], -1).contiguous().cpu().numpy()


def _linear_inputs(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    X = _randn(gen, case["M"], case["K"])
    W = _randn(gen, case["N"], case["K"]) * 0.02
    return X, W, _randn(gen, case["N"]) * 0.1 if case["bias"] else None


def _attn_inputs(case, seed):
    """q, k, v as [B][nh][N][D] views of the memory layout a graph has them in: "heads" all contiguous, "vit" V a view of
    [B][N][nh][D] rows, "tokens" all three such views."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    B, nh, D = case["B"], case["nh"], case["D"]
    out = []
    for i, n in enumerate((case["Nq"], case["Nkv"], case["Nkv"])):
        by_token = case["layout"] == "tokens" or (case["layout"] == "vit" and i == 2)
        t = _randn(gen, B, n, nh, D).transpose(1, 2) if by_token else _randn(gen, B, nh, n, D)
        out.append(t.half() if case["prec"] == "f16" else t)
    return out


def _image(seed, h, w):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    # blocks of colour with noise on top, as a camera frame has both
    coarse = torch.randint(0, 256, (1, 3, (h + 31) // 32, (w + 31) // 32), generator=gen, device=DEV).float()
    img = torch.nn.functional.interpolate(coarse, size=(h, w), mode="bilinear")[0].permute(1, 2, 0)
    return (img + 12 * _randn(gen, h, w, 3)).clamp(0, 255).to(torch.uint8).contiguous()


def _sinusoid(n, d):
    pos = torch.arange(n, device=DEV, dtype=torch.float32)[:, None]
    i = torch.arange(d, device=DEV)
    ang = pos / torch.pow(torch.tensor(10000.0, device=DEV), (i // 2 * 2).float() / d)
    return torch.where(i % 2 == 0, ang.sin(), ang.cos())


def _axial_rope(d, side):
    """Axial RoPE table [side²][d/2][2] (cos, sin), theta 10000: x angles, then y angles."""
    f = 1.0 / torch.pow(torch.tensor(10000.0, device=DEV), torch.arange(d // 4, device=DEV).float() * 4 / d)
    i = torch.arange(side * side, device=DEV)
    ang = torch.cat([(i % side).float()[:, None] * f, (i // side).float()[:, None] * f], 1)
    return torch.stack([ang.cos(), ang.sin()], -1).contiguous()


def prepare(case, seed):
    kind = case["kind"]
    ctx = _ctx()
    s = {"case": case}
    gen = torch.Generator(device=DEV).manual_seed(seed)
    if kind == "linear":
        X, W, bias = _linear_inputs(case, seed)
        s["w"] = ctx.weight(TYPES[case["type"]], case["K"], case["N"], _ggml_bytes(case["type"], W))
        s["X"], s["bias"] = X, bias
        s["Y"] = torch.empty(case["M"], case["N"], device=DEV)
    elif kind == "attn":
        s["qkv"] = _attn_inputs(case, seed)
        s["O"] = torch.empty(case["B"], case["Nq"], case["nh"], case["D"], device=DEV)
    elif kind == "layer_norm":
        n = case["n"]
        s["x"] = _randn(gen, case["rows"], n) * 2 + 0.3
        s["w"], s["b"] = 1 + 0.1 * _randn(gen, n), 0.1 * _randn(gen, n)
        s["y"] = torch.empty_like(s["x"])
    elif kind == "preprocess":
        s["img"] = _image(seed, case["h"], case["w"])
        s["chw"] = torch.empty(3, case["size"], case["size"], device=DEV)
    elif kind == "neck":
        img = case["img"]
        s["st"] = _state(("neck", case["type"], img), lambda p: s3e.synth_write(
            p, img_size=img, window=24 if img > 336 else 8, depth=1, global_idx=(), ftype=case["type"]))
        s["x"] = _randn(gen, (img // 14) ** 2, 1024)
    elif kind == "mem_attn":
        s["st"] = _state(("mem_attn", case["type"]), lambda p: s3e.synth_write_sam2(
            p, "hiera_t", img_size=64, ftype=case["type"], mem_attn_layers=4, embed_dim=32, stages=(1, 1, 1, 1),
            global_idx=(), window_spec=(4, 4, 2, 2), bkg=(2, 2)))
        h, frames, ptr = case["side"], case["frames"], case["ptr"]
        N, M = h * h, frames * h * h + ptr
        s["curr"], s["pos"] = _randn(gen, N, 256), _sinusoid(N, 256)
        s["prompt"] = _randn(gen, M, 64)
        s["ppos"] = torch.cat([_sinusoid(N, 64) + 0.1 * _randn(gen, 64) for _ in range(frames)] + [0.1 * _randn(gen, ptr, 64)])
        s["rope_q"] = _axial_rope(256, h)
        s["rope_k"] = s["rope_q"].repeat(frames, 1, 1)
        s["out"] = torch.empty(N, 256, device=DEV)
    elif kind == "hiera":
        s["st"] = _state(("hiera", case["variant"], case["type"], case["img"]), lambda p: s3e.synth_write_sam2(
            p, case["variant"], img_size=1024, ftype=case["type"]))
        s["chw"] = _chw(_image(seed, case["img"], case["img"]), imagenet=True)
    else:
        s["st"] = _state(("sam3", case["type"], case["neck"]), lambda p: s3e.synth_write(
            p, ftype=case["type"], neck=case["neck"]))
        s["chw"] = _chw(_image(seed, 1008, 1008), imagenet=False)
    # the engine's stream is not torch's: what torch made must be there before the first call
    torch.cuda.synchronize()
    return s


def _chw(img, imagenet):
    v = img.float() / 255
    if imagenet:
        v = (v - torch.tensor([0.485, 0.456, 0.406], device=DEV)) / torch.tensor([0.229, 0.224, 0.225], device=DEV)
    else:
        v = (v - 0.5) / 0.5
    return v.permute(2, 0, 1).contiguous()


# ---- one call ----------------------------------------------------------------
def run(s):
    case, ctx = s["case"], _ctx()
    kind = case["kind"]
    if kind == "linear":
        ctx.mul_mat(s["w"], _buf(s["X"]), case["M"], _buf(s["Y"]), None if s["bias"] is None else _buf(s["bias"]))
        return s["Y"]
    if kind == "attn":
        q, k, v = s["qkv"]
        nb = [(1, t.stride(2), t.stride(1), t.stride(0)) for t in (q, k, v)]
        args = (_buf(q), nb[0], _buf(k), nb[1], _buf(v), nb[2], case["D"], case["Nq"], case["Nkv"], case["nh"],
                case["B"], 1 / math.sqrt(case["D"]), _buf(s["O"]))
        if case["prec"] == "f16":
            ctx.flash_attn_ext_f16(*args)
        else:
            ctx.flash_attn_ext(*args, prec=s3e.PREC_F32 if case["prec"] == "f32" else s3e.PREC_DEFAULT)
        return s["O"]
    if kind == "layer_norm":
        ctx.layer_norm(_buf(s["x"]), case["rows"], case["n"], 1e-5, _buf(s["w"]), _buf(s["b"]), _buf(s["y"]))
        return s["y"]
    if kind == "preprocess":
        ctx.preprocess_image(_buf(s["img"]), case["w"], case["h"], case["size"], case["norm"], _buf(s["chw"]))
        return s["chw"]
    if kind == "neck":
        s["st"].run_neck(_buf(s["x"]))
        return _tensors(s["st"], ["neck_trk_%d" % i for i in range(4)])
    if kind == "mem_attn":
        N, M = s["curr"].shape[0], s["prompt"].shape[0]
        s["st"].mem_attn(_buf(s["curr"]), _buf(s["pos"]), N, _buf(s["prompt"]), _buf(s["ppos"]), M, case["ptr"],
                         _buf(s["rope_q"]), _buf(s["rope_k"]), _buf(s["out"]))
        return s["out"]
    s["st"].encode_chw(_buf(s["chw"]))
    if kind == "hiera":
        return _tensors(s["st"], ["neck_trk_%d" % i for i in range(3)] + ["hiera_stage_3"])
    names = ["vit_output"] + ["neck_trk_%d" % i for i in range(4)]
    return _tensors(s["st"], names + (["neck_det_%d" % i for i in range(4)] if case["neck"] == 2 else []))


# ---- what the call cannot do without -----------------------------------------
def _neck_work(img, type_):
    T, E, D, side = (img // 14) ** 2, 1024, 256, img // 14
    T3 = ((side - 2) // 2 + 1) ** 2
    macs = T * E * 4 * 512 + 4 * T * 512 * 4 * D + 16 * T * D * D + 16 * T * D * 9 * D  # 4x level
    macs += T * E * 4 * 512 + 4 * T * 512 * D + 4 * T * D * 9 * D  # 2x
    macs += T * E * D + T * D * 9 * D + T3 * E * D + T3 * D * 9 * D  # 1x and 0.5x
    weights = 2 * (2 * E * 4 * 512 + 512 * 4 * D) + 4 * (D * D + 512 * D + 2 * E * D + 4 * 9 * D * D)
    return {"bytes": 4 * T * E + weights + 4 * D * (16 * T + 4 * T + T + T3), "flops": 2 * macs}


def _hiera_work(variant, type_, img):
    v = s3e.HIERA_VARIANTS[variant]
    dim, side, i, macs, weights = v["embed_dim"], img // 4, 0, 147 * v["embed_dim"] * (img // 4) ** 2, 0
    for st, blocks in enumerate(v["stages"]):
        for b in range(blocks):
            # at a stage change the block pools its queries and doubles its width
            enter = st > 0 and b == 0
            d_in = dim // 2 if enter else dim
            tin = (side * 2) ** 2 if enter else side ** 2
            tout = side ** 2
            win = v["window_spec"][st - 1 if enter else st]
            keys = tin if i in v["global_idx"] else win * win
            macs += tin * d_in * 3 * dim + (tin * d_in * dim if enter else 0) + 2 * tout * keys * dim + tout * dim * 9 * dim
            weights += d_in * 3 * dim + (d_in * dim if enter else 0) + 9 * dim * dim
            i += 1
        macs += side ** 2 * dim * 256
        weights += dim * 256
        if st < 3:
            dim, side = dim * 2, side // 2
    out = sum((img // k) ** 2 * 256 * 4 for k in (4, 8, 16)) + (img // 32) ** 2 * dim * 4
    return {"bytes": 12 * img * img + weights * BYTES_PER_WEIGHT[type_] + out, "flops": 2 * macs}


def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": N * K * BYTES_PER_WEIGHT[case["type"]] + 4 * M * (K + N) + (4 * N if case["bias"] else 0),
                "flops": 2 * M * N * K}
    if kind == "attn":
        heads, size = case["B"] * case["nh"] * case["D"], 2 if case["prec"] == "f16" else 4
        return {"bytes": heads * (size * (case["Nq"] + 2 * case["Nkv"]) + 4 * case["Nq"]),
                "flops": 4 * heads * case["Nq"] * case["Nkv"]}
    if kind == "layer_norm":
        return {"bytes": 8 * case["rows"] * case["n"] + 8 * case["n"], "flops": 8 * case["rows"] * case["n"]}
    if kind == "preprocess":
        S, w, h = case["size"], case["w"], case["h"]
        return {"bytes": 3 * min(w, 2 * S) * min(h, 2 * S) + 12 * S * S, "flops": 3 * 12 * S * S}
    if kind == "neck":
        return _neck_work(case["img"], case["type"])
    if kind == "mem_attn":
        N, D, MD, F = case["side"] ** 2, 256, 64, 2048
        M = case["frames"] * N + case["ptr"]
        macs = 4 * (N * D * 4 * D + N * D * 2 * D + 2 * M * MD * D + 2 * N * D * F + 2 * N * (N + M) * D)
        weights = 4 * (6 * D * D + 2 * MD * D + 2 * D * F)
        return {"bytes": weights * BYTES_PER_WEIGHT[case["type"]] + 4 * (3 * N * D + 2 * M * MD + N * D + M * D), "flops": 2 * macs}
    if kind == "hiera":
        return _hiera_work(case["variant"], case["type"], case["img"])
    T, E, mlp = 5184, 1024, 4736
    macs = 32 * T * E * (4 * E + 2 * mlp) + 2 * T * E * (28 * 576 + 4 * T) + T * E * 588
    neck = _neck_work(1008, case["type"])
    return {"bytes": 12 * 1008 * 1008 + 32 * E * (4 * E + 2 * mlp) * BYTES_PER_WEIGHT[case["type"]] + 4 * T * E
            + case["neck"] * (neck["bytes"] - 4 * T * E), "flops": 2 * macs + case["neck"] * neck["flops"]}


def tolerance(case):
    kind = case["kind"]
    if kind == "linear":
        # the same quantized operands on both sides: sums of fp32 products, in another order 1e-7 to 3e-7
        return {"rel": 2e-6, "max": 1e-4}
    if kind == "attn":
        # f32 attention: 4e-7 in other orders; fp16 operands and probabilities: 3e-4 to 5e-4 off the exact quotient
        return {"rel": 2e-6, "max": 1e-4} if case["prec"] == "f32" else {"rel": 2e-3}
    if kind == "layer_norm":
        return {"rel": 5e-7}
    if kind == "preprocess":
        return "exact"  # the reference's bytes, normalised by two correctly rounded operations
    if kind == "neck":
        # F32 convolutions on either side of fp16 deconvolution inputs (one-ulp flips); F16 files round every input
        return {"rel": 3e-4 if case["type"] == "f16" else 4e-5}
    # whole calls: a last-bit difference in one layer flips fp16 roundings (F16 files) or Q8 codes (quantized files)
    # in all that follow; two of ggml's own evaluation orders differ by 1.6e-2 over the 32 quantized ViT blocks
    if kind == "mem_attn":
        return {"rel": 4e-3 if case["type"] == "f16" else 0.02}
    return {"rel": 4e-3 if case["type"] == "f16" else 0.03}


# ---- the same in 64 bits -------------------------------------------------------
def _q8_activations(X):
    """ggml's from_float of the rows: codes, fp16 scales, fp16 block sums, all as float64."""
    b = X.reshape(X.shape[0], -1, 32)
    amax = b.abs().amax(-1)
    top = torch.full_like(amax, 127)  # tensors: divided as IEEE does, not by a reciprocal
    inv = torch.where(amax > 0, top / amax, torch.zeros_like(amax))
    q = torch.round(b * inv[..., None])
    d = amax / top
    return q.double(), d.half().double(), (d * q.sum(-1)).half().double()


def _linear_exact(case, seed):
    X, W, bias = _linear_inputs(case, seed)
    t = case["type"]
    if t in ("f32", "f16"):
        x, w = (X.double(), W.double()) if t == "f32" else (X.half().double(), W.half().double())
        Y = x @ w.T
    else:
        q, d, m = _weight_codes(t, W)
        if t == "q4_0":
            q = q - 8
        w = (q.double() * d.double()[..., None]).reshape(W.shape)
        xq, xd, xs = _q8_activations(X)
        Y = (xq * xd[..., None]).reshape(X.shape) @ w.T
        if m is not None:
            Y += xs @ m.double().T
    return Y if bias is None else Y + bias.double()


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        return _linear_exact(case, seed)
    if kind == "attn":
        q, k, v = _attn_inputs(case, seed)
        B, nh, D = case["B"], case["nh"], case["D"]
        O = torch.empty(B, case["Nq"], nh, D, device=DEV, dtype=torch.float64)
        for b in range(B):
            for h in range(nh):
                p = torch.softmax(q[b, h].double() @ k[b, h].double().T / math.sqrt(D), -1)
                O[b, :, h] = p @ v[b, h].double()
        return O
    if kind == "layer_norm":
        gen = torch.Generator(device=DEV).manual_seed(seed)
        x = (_randn(gen, case["rows"], case["n"]) * 2 + 0.3).double()
        w, b = 1 + 0.1 * _randn(gen, case["n"]), 0.1 * _randn(gen, case["n"])
        c = x - x.mean(-1, keepdim=True)
        return c / torch.sqrt(c.square().mean(-1, keepdim=True) + 1e-5) * w.double() + b.double()
    if kind == "preprocess":
        return _preprocess_exact(_image(seed, case["h"], case["w"]).double(), case["size"], case["norm"])
    return None


def _preprocess_exact(img, S, norm):
    h, w, _ = img.shape
    if (h, w) != (S, S):
        taps = []
        for n in (h, w):
            f = ((torch.arange(S, device=DEV, dtype=torch.float64) + 0.5) * (n / S) - 0.5).clamp(min=0)
            i0 = f.floor().long()
            taps.append((i0, (i0 + 1).clamp(max=n - 1), f - i0))
        (y0, y1, wy), (x0, x1, wx) = taps
        wy, wx = wy[:, None, None], wx[None, :, None]
        top = (1 - wx) * img[y0][:, x0] + wx * img[y0][:, x1]
        bottom = (1 - wx) * img[y1][:, x0] + wx * img[y1][:, x1]
        img = torch.floor((1 - wy) * top + wy * bottom + 0.5).clamp(0, 255)
    v = img / 255
    if norm:
        v = (v - torch.tensor([0.485, 0.456, 0.406], device=DEV, dtype=torch.float64)) / torch.tensor(
            [0.229, 0.224, 0.225], device=DEV, dtype=torch.float64)
    else:
        v = (v - 0.5) / 0.5
    return v.permute(2, 0, 1).contiguous()
