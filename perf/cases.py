"""The work whose speed this library is judged by, through its public entry points.

Each case is one call that a program built on this library makes: whole transformer blocks (Flux.1 joint and single,
Wan, the SD 1.5 / SDXL UNet), the projections around them that run with few rows, LoRA on a palettized base, attention
over a joint text + image sequence, and the dequantizing read of a palettized weight.  `listed()` names the points
that are always measured, `draw()` samples the ranges they stand for.

A case is a dict of plain values; "kind" selects the path:

  dense        Dense over palettized or plain fp16 weights, any rows / widths       rows 1 .. 8192, K 64 .. 5120
  lora         LoRADense, the pair in fp16 or (high precision) in fp32              rows 64 .. 4608, rank 4 .. 128
  unet         BasicTransformerBlock, fp16 stream                                   256 .. 4096 tokens x batch 1 .. 2
  flux_joint   JointTransformerBlock, text + image streams, 24 x 128 heads          256 .. 4096 image tokens
  flux_single  SingleTransformerBlock                                               512 .. 4608 tokens
  wan          WanAttentionBlock, 40 x 128 heads                                    1024 .. 32760 tokens
  attention    sdpa_segments over text + image segments, norm and RoPE fused        Sq 256 .. 4608, D 40 .. 128
  dequantize   QxTensor.dequantize                                                  2^18 .. 2^26 weights
"""
import importlib
import math

import torch

_dt = importlib.import_module("draw-things-community_amd")
_flux1 = importlib.import_module("draw-things-community_amd.flux1")
_wan = importlib.import_module("draw-things-community_amd.wan")
_unet = importlib.import_module("draw-things-community_amd.unet")

_CODEC_BITS = {"f16": 16.0, "q4p": 4.5, "q5p": 5.5, "q6p": 6.25, "q7p": 7.25, "q8p": 8.25}  # per weight, palettes included


def listed():
    return [
        # the smallest call: the six modulation vectors of one block from one conditioning row (adaLN weights ship as
        # q8p), bound by reading the weights
        {"name": "dense_one_row", "kind": "dense", "m": 1, "k": 3072, "n": 3072, "weights": 6, "codec": "q8p", "act": "none"},
        # keys and values of the text context for a video block's cross-attention, once per generation
        {"name": "dense_context_kv", "kind": "dense", "m": 512, "k": 5120, "n": 5120, "weights": 2, "codec": "q5p", "act": "none"},
        # no size a multiple of a tile: three prompts of 77 text rows through a projection of generic odd widths
        {"name": "dense_ragged", "kind": "dense", "m": 231, "k": 1000, "n": 1001, "weights": 1, "codec": "q8p", "act": "gelu"},
        # LoRA on the out-projection of a 1024 x 1024 image's token stream, as most LoRA files come (rank 16, fp16)
        {"name": "lora_fp16", "kind": "lora", "m": 4608, "k": 3072, "n": 3072, "rank": 16, "codec": "q6p", "high": False},
        # the same with the pair kept in fp32
        {"name": "lora_fp32", "kind": "lora", "m": 4608, "k": 3072, "n": 3072, "rank": 32, "codec": "q6p", "high": True},
        # first-level UNet block, both halves of classifier-free guidance, 512 x 512 image
        {"name": "unet_4096", "kind": "unet", "head": 40, "heads": 8, "batch": 2, "grid_h": 64, "grid_w": 64, "text": 77,
         "context": 768, "codec": "q6p"},
        # deeper and wider UNet block on a non-square image, plain fp16 weights
        {"name": "unet_1008", "kind": "unet", "head": 64, "heads": 20, "batch": 2, "grid_h": 28, "grid_w": 36, "text": 77,
         "context": 2048, "codec": "f16"},
        # the benchmark's block: 1024 x 1024 image, 512 text tokens
        {"name": "flux_joint_4608", "kind": "flux_joint", "text": 512, "grid_h": 64, "grid_w": 64, "codec": "q6p"},
        # single-stream block of a small non-square image with a short prompt
        {"name": "flux_single_1376", "kind": "flux_single", "text": 256, "grid_h": 40, "grid_w": 28, "codec": "q8p"},
        # the largest: 81 video frames at 480 x 832
        {"name": "wan_32760", "kind": "wan", "frames": 21, "grid_h": 30, "grid_w": 52, "text": 512, "codec": "q5p"},
        # joint attention with the norms and the rotation applied on the way in, lengths no multiple of a tile
        {"name": "attention_joint", "kind": "attention", "batch": 1, "heads": 24, "kv_heads": 24, "head": 128, "text": 333,
         "image": 2304, "fused": True},
        # a feed-forward weight read without keeping it packed
        {"name": "dequantize_q6p", "kind": "dequantize", "n": 12288, "k": 3072, "codec": "q6p"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dense", "dense", "dense", "lora", "lora", "unet", "unet", "flux_joint", "flux_single", "wan",
                       "attention", "attention", "dequantize"])
    codec = rng.choice(["q4p", "q5p", "q6p", "q6p", "q8p", "q8p"])
    if kind == "dense":
        m = _log_int(rng, 1, 8192)
        if rng.random() < 0.25:  # widths off the 64-wide grid that model widths lie on
            m = min(m, 1024)
            k, n = _log_int(rng, 64, 2560), _log_int(rng, 64, 2560)
        else:
            k, n = 64 * _log_int(rng, 1, 80), 64 * _log_int(rng, 1, 80)
        return {"kind": kind, "m": m, "k": k, "n": n, "weights": rng.choice([1, 1, 2, 3, 6]),
                "codec": rng.choice([codec, codec, "f16"]), "act": rng.choice(["none", "none", "gelu"])}
    if kind == "lora":
        return {"kind": kind, "m": _log_int(rng, 64, 4608), "k": 64 * _log_int(rng, 5, 80), "n": 64 * _log_int(rng, 5, 80),
                "rank": rng.choice([4, 8, 16, 32, 64, 128]), "codec": codec, "high": rng.random() < 0.4}
    if kind == "unet":
        head, heads = rng.choice([(40, 8), (80, 8), (64, 10), (64, 20)])
        return {"kind": kind, "head": head, "heads": heads, "batch": rng.choice([1, 2]), "grid_h": rng.randint(16, 64),
                "grid_w": rng.randint(16, 64), "text": 77 * rng.choice([1, 1, 2]), "context": rng.choice([768, 1024, 2048]),
                "codec": rng.choice(["f16", "q6p", "q8p"])}
    if kind == "flux_joint":
        return {"kind": kind, "text": rng.choice([77, 128, 256, 333, 512]), "grid_h": rng.randint(16, 64),
                "grid_w": rng.randint(16, 64), "codec": codec}
    if kind == "flux_single":
        return {"kind": kind, "text": rng.choice([256, 333, 512]), "grid_h": rng.randint(16, 64),
                "grid_w": rng.randint(16, 64), "codec": codec}
    if kind == "wan":
        gh, gw = rng.randint(12, 30), rng.randint(20, 52)
        return {"kind": kind, "frames": max(1, min(21, round(_log_int(rng, 1024, 32760) / (gh * gw)))), "grid_h": gh, "grid_w": gw,
                "text": rng.choice([226, 512]), "codec": codec}
    if kind == "attention":
        head = rng.choice([40, 64, 128, 128])
        heads = rng.choice([8, 12, 24])
        return {"kind": kind, "batch": rng.choice([1, 1, 2]), "heads": heads, "kv_heads": rng.choice([heads, heads, heads // 4]),
                "head": head, "text": rng.choice([77, 154, 256, 333, 512]), "image": _log_int(rng, 256, 4096),
                "fused": rng.random() < 0.5}
    return {"kind": kind, "n": _log_int(rng, 512, 16384), "k": 64 * _log_int(rng, 8, 64), "codec": codec}


# ---- inputs ------------------------------------------------------------------------------------------------------

class _Source:
    """Everything random of one state, from one seed, made on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.float16):
        return torch.randn(shape, generator=self.g, device="cuda").mul_(std).add_(mean).to(dtype)

    def weight(self, n, k, codec):
        """A [n, k] weight: palettes ~ N(0, 0.02) and uniform indices, packed as the store hands them out."""
        if codec == "f16":
            return _dt.QxTensor(self.normal(n, k, std=0.02), 16, 0, (n, k))
        q, nib = _dt.CODEC[codec]
        count = n * k
        total = _dt.qx_bytes(q, nib, count)
        buf = torch.zeros((total + 15) // 16 * 16, dtype=torch.uint8, device="cuda")
        buf[:total] = torch.randint(0, 256, (total,), generator=self.g, device="cuda", dtype=torch.uint8)
        pal, stride, full = 2 << q, (2 << q) + nib * q // 8, count // nib
        if full:
            p = self.normal(full, 1 << q, std=0.02).view(torch.uint8)
            buf[:full * stride].view(full, stride)[:, :pal] = p
        if count % nib:
            buf[full * stride:full * stride + pal] = self.normal(1 << q, std=0.02).view(torch.uint8)
        return _dt.QxTensor(buf, q, nib, (n, k))

    def weights(self, names, shapes, codec):
        return {name: self.weight(*shapes(name), codec) for name in names}

    def table(self, rows):
        return torch.from_numpy(rows).to("cuda", torch.float16).contiguous()


def prepare(case, seed):
    s, kind, codec = _Source(seed), case["kind"], case.get("codec")
    if kind == "dense":
        m, k, n = case["m"], case["k"], case["n"]
        return {"kind": kind, "x": s.normal(m, k), "w": [s.weight(n, k, codec) for _ in range(case["weights"])],
                "b": [s.normal(n, std=0.1) for _ in range(case["weights"])], "act": case["act"]}
    if kind == "lora":
        m, k, n, r = case["m"], case["k"], case["n"], case["rank"]
        op = _dt.LoRADense(n, _dt.LoRANetworkConfiguration(r, 0.75, case["high"]))
        op.weight, op.bias = s.weight(n, k, codec), s.normal(n, std=0.1)
        dtype = torch.float32 if case["high"] else torch.float16
        op.down = _dt.QxTensor(s.normal(r, k, std=0.02, dtype=dtype), 16, 0, (r, k))
        op.up = _dt.QxTensor(s.normal(n, r, std=0.05, dtype=dtype), 16, 0, (n, r))
        return {"kind": kind, "op": op, "x": s.normal(1, m, k)}
    if kind == "unet":
        c, hw, cw = case["head"] * case["heads"], case["grid_h"] * case["grid_w"], case["context"]
        block = _unet.BasicTransformerBlock(case["head"], case["heads"], case["batch"], hw, case["text"])
        shapes = {"tokeys2": (c, cw), "tovalues2": (c, cw), "fc10": (4 * c, c), "fc11": (4 * c, c), "fc2": (c, 4 * c)}
        block.weight = s.weights(_unet.DENSE_NAMES, lambda name: shapes.get(name, (c, c)), codec)
        block.bias = {name: s.normal(shapes.get(name, (c, c))[0], std=0.1) for name in _unet.DENSE_NAMES if name not in _unet.NO_BIAS}
        block.norm = {name: (s.normal(c, std=0.1, mean=1.0), s.normal(c, std=0.1)) for name in _unet.NORM_NAMES}
        return {"kind": kind, "op": block, "x": s.normal(case["batch"], hw, c), "c": s.normal(case["batch"], case["text"], cw)}
    if kind in ("flux_joint", "flux_single"):
        h, k, t, gh, gw = 24, 128, case["text"], case["grid_h"], case["grid_w"]
        c, hw = h * k, gh * gw
        wide = lambda name: (4 * c, c) if "linear1" in name else (c, 4 * c) if "out_proj" in name else (c, c)
        rot = s.table(_dt.Flux1RotaryPositionEmbedding(gh, gw, t, channels=k))
        # shift, scale (with its + 1), gate
        chunks = lambda n: [s.normal(c, std=0.3, mean=1.0 if i % 3 == 1 else 0.0) for i in range(n)]
        joint = kind == "flux_joint"
        block = _flux1.JointTransformerBlock(k, h, t, hw) if joint else _flux1.SingleTransformerBlock(k, h, t + hw)
        names, norms = ((_flux1.DENSE_NAMES, _flux1.NORM_NAMES) if joint else
                        (_flux1.SINGLE_DENSE_NAMES, _flux1.SINGLE_NORM_NAMES))
        block.weight = s.weights(names, wide, codec)
        block.bias = {name: s.normal(wide(name)[0], std=0.1) for name in names}
        block.norm = {name: s.normal(k, std=0.1, mean=1.0) for name in norms}
        if not joint:
            return {"kind": kind, "op": block, "x": s.normal(1, t + hw, c, dtype=torch.float32), "rot": rot, "chunks": chunks(3)}
        return {"kind": kind, "op": block, "c": s.normal(1, t, c, dtype=torch.float32), "x": s.normal(1, hw, c, dtype=torch.float32),
                "rot": rot, "c_chunks": chunks(6), "x_chunks": chunks(6)}
    if kind == "wan":
        h, k, ff = 40, 128, 13824
        c, hw = h * k, case["frames"] * case["grid_h"] * case["grid_w"]
        block = _wan.WanAttentionBlock(k, h, hw, ff)
        wide = lambda name: (ff, c) if name == "x_linear1" else (c, ff) if name == "x_out_proj" else (c, c)
        block.weight = s.weights(_wan.DENSE_NAMES, wide, codec)
        block.bias = {name: s.normal(wide(name)[0], std=0.1) for name in _wan.DENSE_NAMES}
        block.norm = {name: s.normal(c, std=0.1, mean=1.0) for name in _wan.ROW_NORM_NAMES}
        f32 = dict(dtype=torch.float32)
        block.norm3_weight, block.norm3_bias = s.normal(c, std=0.1, mean=1.0, **f32), s.normal(c, std=0.1, **f32)
        block.modulation = [s.normal(c, std=0.1, **f32) for _ in range(6)]
        rot = s.table(_dt.WanRotaryPositionEmbedding(case["grid_h"], case["grid_w"], case["frames"], channels=k))
        return {"kind": kind, "op": block, "x": s.normal(1, hw, c, **f32), "rot": rot,
                "c": [s.normal(c, std=0.3, **f32) for _ in range(6)], "ck": s.normal(1, case["text"], h, k),
                "cv": s.normal(1, case["text"], h, k)}
    if kind == "attention":
        b, h, hk, d, t, n = (case[key] for key in ("batch", "heads", "kv_heads", "head", "text", "image"))
        state = {"kind": kind, "q": [s.normal(b, t, h, d), s.normal(b, n, h, d)], "k": [s.normal(b, t, hk, d), s.normal(b, n, hk, d)],
                 "v": [s.normal(b, t, hk, d), s.normal(b, n, hk, d)], "scale": 1.0 / math.sqrt(d), "more": {}}
        if case["fused"]:
            gamma = lambda: [s.normal(d, std=0.1, mean=1.0) for _ in range(2)]
            angle = torch.arange(t + n, device="cuda")[:, None] * torch.pow(1e4, -torch.arange(d // 2, device="cuda") / (d // 2))[None]
            rot = torch.stack([angle.cos(), angle.sin()], dim=-1).reshape(t + n, d).half()
            state["more"] = {"gamma_q": gamma(), "gamma_k": gamma(), "rot_q": rot, "rot_k": rot}
        return state
    return {"kind": kind, "w": s.weight(case["n"], case["k"], codec)}


def run(state):
    kind = state["kind"]
    if kind == "dense":
        if state["act"] == "gelu":
            return _dt.dense_post(state["x"], state["w"], state["b"], [_dt.DensePost(_dt.ACT_GELU_TANH)] * len(state["w"]))
        return _dt.dense_multi(state["x"], state["w"], state["b"])
    if kind == "lora":
        return state["op"](state["x"])
    if kind == "unet":
        return state["op"](state["x"], state["c"])
    if kind == "flux_joint":
        return state["op"](state["c"], state["x"], state["rot"], state["c_chunks"], state["x_chunks"])
    if kind == "flux_single":
        return state["op"](state["x"], state["rot"], state["chunks"])
    if kind == "wan":
        return state["op"](state["x"], state["rot"], state["c"], state["ck"], state["cv"])
    if kind == "attention":
        return _dt.sdpa_segments(state["q"], state["k"], state["v"], state["scale"], **state["more"])
    return state["w"].dequantize()


# ---- what a pass cannot do without ---------------------------------------------------------------------------------

def _sdpa_flops(b, h, sq, skv, d):
    return 4.0 * b * h * sq * skv * d


def work(case):
    """Every input read once, every output written once (intermediate tensors of a block are neither)."""
    kind = case["kind"]
    bits = _CODEC_BITS[case.get("codec", "f16")] / 8
    if kind == "dense":
        m, k, n, w = case["m"], case["k"], case["n"], case["weights"]
        return {"bytes": 2 * m * k + w * (bits * n * k + 2 * n + 2 * m * n), "flops": 2.0 * m * n * k * w}
    if kind == "lora":
        m, k, n, r = case["m"], case["k"], case["n"], case["rank"]
        pair = (4 if case["high"] else 2) * r * (k + n)
        return {"bytes": 2 * m * k + bits * n * k + 2 * n + pair + 2 * m * n, "flops": 2.0 * m * (n * k + r * (k + n))}
    if kind == "unet":
        c, hw, b, t, cw = case["head"] * case["heads"], case["grid_h"] * case["grid_w"], case["batch"], case["text"], case["context"]
        weights = 18 * c * c + 2 * c * cw
        flops = 2.0 * b * (hw * 18 * c * c + t * 2 * c * cw) + _sdpa_flops(b, case["heads"], hw, hw + t, case["head"])
        return {"bytes": bits * weights + 2 * b * (2 * hw * c + t * cw), "flops": flops}
    if kind in ("flux_joint", "flux_single"):
        c, s = 3072, case["text"] + case["grid_h"] * case["grid_w"]
        n_weights = (24 if kind == "flux_joint" else 12) * c * c
        return {"bytes": bits * n_weights + 8 * s * c + 2 * s * 128, "flops": 24.0 * s * c * c + _sdpa_flops(1, 24, s, s, 128)}
    if kind == "wan":
        c, ff, hw, t = 5120, 13824, case["frames"] * case["grid_h"] * case["grid_w"], case["text"]
        flops = 2.0 * hw * (6 * c * c + 2 * c * ff) + _sdpa_flops(1, 40, hw, hw + t, 128)
        return {"bytes": bits * (6 * c * c + 2 * c * ff) + 8 * hw * c + 4 * t * c + 2 * hw * 128, "flops": flops}
    if kind == "attention":
        b, h, hk, d, s = case["batch"], case["heads"], case["kv_heads"], case["head"], case["text"] + case["image"]
        return {"bytes": 4 * b * s * (h + hk) * d + (2 * s * d if case["fused"] else 0), "flops": _sdpa_flops(b, h, s, s, d)}
    return {"bytes": (bits + 2) * case["n"] * case["k"], "flops": 0}


def tolerance(case):
    """About four times the distance of each path from itself with float64 sums and the same fp16 roundings between its
    operations: what another order of the sums does is to move single values by one fp16 rounding (max 2e-3).  Measured
    as rel: 2e-6 .. 2e-5 for the projections (one such value among 64 weighs up to 1e-4), 1e-4 .. 3.4e-4 for attention
    and the blocks, whose probabilities are fp16.  A dequantized weight is a table lookup and has to be exact."""
    kind = case["kind"]
    if kind == "dequantize":
        return "exact"
    if kind in ("dense", "lora"):
        return {"rel": 2e-4, "max": 8e-3}
    return {"rel": 1.3e-3, "max": 1.2e-2}
