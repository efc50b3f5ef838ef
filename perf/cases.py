"""The work a user of the INT8 engine has it do, as cases to be timed.

A diffusion transformer is a stack of linear layers between attention kernels: modulation projections of one
conditioning vector per image, projections of a few dozen to a few thousand tokens, and the blocks those make up.
LoRAs are merged into the int8 weights when a workflow changes.  Every case is one such piece of work through the
package's public entry points: `Int8TensorwiseOps.Linear`, `forward_fanout`, `forward_pair` and the LoRA adapters.

    listed()          the named cases
    draw(rng)         one more case of the same ranges
    prepare(case, s)  what a program holds before the call: layers, activations, vectors, LoRA factors
    run(state)        one pass
    work(case)        bytes and operations the pass cannot do without
    tolerance(case)   how far another correct implementation may be
"""
from __future__ import annotations

import torch

from __graft_entry__ import load_package

pkg = load_package()
ops = pkg.Int8TensorwiseOps
L = pkg._lib

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


# About four times what the same pass differs by when it is evaluated in 64 bits between the tensors a program sees (each
# still rounded to its dtype): one rounding of the output for the small-batch layers, that and a second rounding with the
# bias for the int8 layers, and in the blocks a few int8 activations one step apart.  The merges: shares of the weights in
# which a delta of another summation order falls on the other side of its random number.
TOLERANCES = {
    "vector": {"rel": 7e-3, "max": 0.016}, "linear": {"rel": 1.2e-2, "max": 0.09}, "fanout": {"rel": 1.2e-2, "max": 0.1},
    "mlp": {"rel": 1.1e-2, "max": 0.3}, "double": {"rel": 1.4e-2, "max": 0.15}, "single": {"rel": 1.2e-2, "max": 0.2},
    "merge": {"rel": 1e-4, "max": 0.06, "differ": 3e-6}, "stack": {"rel": 1e-4, "max": 0.06, "differ": 3e-6},
}


# --------------------------------------------------------------------------- the cases
def listed():
    return [
        # The smallest call: a layer of the timestep or guidance embedder on the vectors of four images, weights rotated.
        {"name": "vector_4x3072_3072_rotated", "kind": "vector", "rows": 4, "width": 3072, "outs": 3072, "layers": 1,
         "dtype": "fp16", "rotate": True},
        # The modulation projections of both streams of a double-stream block, one image: a read of 113 MB of weights.
        {"name": "modulation_1x3072_18432_pair", "kind": "vector", "rows": 1, "width": 3072, "outs": 18432, "layers": 2,
         "dtype": "bf16", "rotate": False},
        # The modulation projection of a batch of images (image batches, or conditional and unconditional together).
        {"name": "modulation_12x3840_15360", "kind": "vector", "rows": 12, "width": 3840, "outs": 15360, "layers": 1,
         "dtype": "bf16", "rotate": False},
        # A text encoder's 77 tokens through one projection of a checkpoint with one scale per weight.
        {"name": "text_77x3072_3072_one_scale", "kind": "linear", "rows": 77, "width": 3072, "outs": 3072, "dtype": "bf16",
         "rotate": False, "row_scale": False, "rank": 0},
        # Widths that fit no tile and rows that fill none: pruned or custom layers.
        {"name": "odd_333x1160_1001", "kind": "linear", "rows": 333, "width": 1160, "outs": 1001, "dtype": "bf16",
         "rotate": False, "row_scale": True, "rank": 0},
        # The text stream's feed-forward half of an adaLN block: norm, modulation, up, GELU, down, gate, residual.
        {"name": "mlp_512x3072_12288", "kind": "mlp", "rows": 512, "width": 3072, "hidden": 12288, "dtype": "bf16"},
        # A small image's tokens (ragged) through a layer with an un-merged LoRA of rank 32.
        {"name": "dynamic_lora_1357x3072_9216_r32", "kind": "linear", "rows": 1357, "width": 3072, "outs": 9216, "dtype": "bf16",
         "rotate": False, "row_scale": True, "rank": 32},
        # Separate q, k and v projections of one normalised tensor, rotated weights, width 3840.
        {"name": "qkv_4096x3840_rotated", "kind": "fanout", "rows": 4096, "width": 3840, "outs": 3840, "layers": 3,
         "dtype": "fp16", "rotate": True},
        # The linear layers of a double-stream block: 4096 image and 512 text tokens, width 3072.
        {"name": "double_block_4096+512x3072", "kind": "double", "rows": 4096, "text": 512, "width": 3072, "dtype": "bf16"},
        # A single-stream block on a large image with its text (ragged): the two wide layers around attention.
        {"name": "single_block_9729x3072", "kind": "single", "rows": 9729, "width": 3072, "dtype": "bf16"},
        # One LoRA merged into an int8 weight by stochastic rounding.
        {"name": "lora_merge_12288x3072_r32", "kind": "merge", "outs": 12288, "width": 3072, "ranks": "32"},
        # A stack of three LoRAs merged into an int8 weight in one rounding step.
        {"name": "lora_stack_9216x3072_r16_r32_r64", "kind": "stack", "outs": 9216, "width": 3072, "ranks": "16 32 64"},
    ]


def _log_int(rng, lo, hi, step=1):
    """A multiple of `step` between lo and hi, spread over the logarithm."""
    v = lo * (hi / lo) ** rng.random()
    return min(hi // step * step, max(step, round(v / step) * step))


def _cost(case):
    """Seconds of the pass at rates near the card's, to keep drawn cases within the largest listed one."""
    w = work(case)
    rate = 5e12 if _has_odd_widths(case) else 2.5e15
    return w["flops"] / rate + w["bytes"] / 4e12


def _has_odd_widths(case):
    return case["kind"] == "linear" and (case["width"] % 16 != 0 or case["outs"] % 8 != 0)


def draw(rng):
    limit = max(_cost(c) for c in listed() if not _has_odd_widths(c))
    while True:
        case = _draw_one(rng)
        if _cost(case) <= limit:
            return case


def _draw_one(rng):
    kind = rng.choice(["vector", "vector", "linear", "linear", "linear", "odd", "mlp", "fanout", "double", "single", "merge", "stack"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "vector":
        rotate = rng.random() < 0.4
        width = _log_int(rng, 256, 6144, 128 if rotate else 16)
        return {"kind": "vector", "rows": rng.randint(1, 16), "width": width, "outs": _log_int(rng, 512, 24576, 8),
                "layers": rng.choice([1, 1, 2]), "dtype": dtype, "rotate": rotate}
    if kind == "odd":
        return {"kind": "linear", "rows": _log_int(rng, 17, 512), "width": _log_int(rng, 100, 1500), "outs": _log_int(rng, 100, 1500),
                "dtype": dtype, "rotate": False, "row_scale": rng.random() < 0.7, "rank": 0}
    if kind == "linear":
        rotate = rng.random() < 0.3
        rank = rng.choice([0, 0, 0, 4, 16, 32, 64])
        width = _log_int(rng, 384, 13824, 128 if rotate or rank else 16)
        return {"kind": "linear", "rows": _log_int(rng, 17, 16384), "width": width, "outs": _log_int(rng, 384, 13824, 8),
                "dtype": dtype, "rotate": rotate, "row_scale": rng.random() < 0.8, "rank": rank}
    if kind == "mlp":
        width = _log_int(rng, 1024, 5120, 64)
        return {"kind": "mlp", "rows": _log_int(rng, 64, 8192), "width": width, "hidden": width * rng.choice([3, 4]) // 64 * 64, "dtype": dtype}
    if kind == "fanout":
        width = _log_int(rng, 1024, 5120, 128)
        return {"kind": "fanout", "rows": _log_int(rng, 64, 8192), "width": width, "outs": width, "layers": rng.choice([2, 3]),
                "dtype": dtype, "rotate": rng.random() < 0.7}
    if kind == "double":
        return {"kind": "double", "rows": _log_int(rng, 512, 9216), "text": _log_int(rng, 32, 1024), "width": _log_int(rng, 1024, 4096, 128),
                "dtype": "bf16"}
    if kind == "single":
        return {"kind": "single", "rows": _log_int(rng, 256, 9729), "width": _log_int(rng, 1024, 3072, 128), "dtype": "bf16"}
    if kind == "merge":
        return {"kind": "merge", "outs": _log_int(rng, 1024, 18432, 8), "width": _log_int(rng, 1024, 12288, 16),
                "ranks": str(rng.choice([4, 8, 16, 32, 64, 128]))}
    return {"kind": "stack", "outs": _log_int(rng, 1024, 12288, 8), "width": _log_int(rng, 1024, 6144, 16),
            "ranks": " ".join(str(rng.choice([4, 8, 16, 32, 64])) for _ in range(rng.choice([2, 3])))}


# --------------------------------------------------------------------------- inputs
class _Draws:
    """Everything a state is made of, from one seed."""

    def __init__(self, seed, dtype="bf16"):
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.gen = torch.Generator(device=self.dev).manual_seed(seed)
        self.dtype = DTYPES[dtype]

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.gen, device=self.dev) * std

    def tokens(self, rows, width):
        """Activations of a transformer: N(0, 1) with one channel in a hundred twenty times as large."""
        x = self.normal(1, rows, width)
        loud = torch.randperm(width, generator=self.gen, device=self.dev)[: max(1, width // 100)]
        x[..., loud] *= 20.0
        return x.to(self.dtype)

    def vectors(self, width, std=0.3):
        return self.normal(1, 1, width, std=std).to(self.dtype)

    def layer(self, width, outs, rotate=False, row_scale=True, bias=True):
        """A quantised layer as a pre-quantised checkpoint gives it, on the GPU."""
        w = self.normal(outs, width, std=0.02)
        if row_scale:
            q, s = pkg.hip_quantize_rowwise(w, rotate=rotate)
        else:
            q, s = pkg.quantize_int8_tensorwise(L.rotate128(w) if rotate else w)
        lin = ops.Linear(width, outs, bias=bias, device="meta")
        sd = {"weight": q, "weight_scale": s}
        if bias:
            sd["bias"] = self.normal(outs, std=0.01).to(self.dtype)
        lin._load_from_state_dict(sd, "", {}, True, [], [], [])
        lin._use_quarot = rotate
        return lin

    def lora(self, outs, width, rank):
        """The weights of a LoRA file for one layer: (up, down, alpha, mid, dora_scale, reshape)."""
        return (self.normal(outs, rank, std=0.01), self.normal(rank, width, std=0.01), float(rank), None, None, None)


def prepare(case, seed):
    d = _Draws(seed, case.get("dtype", "bf16"))
    kind = case["kind"]
    st = {"kind": kind}
    if kind == "vector":
        st["x"] = d.normal(case["rows"], case["width"]).to(d.dtype)
        st["layers"] = [d.layer(case["width"], case["outs"], case["rotate"]) for _ in range(case["layers"])]
    elif kind == "linear":
        st["x"] = d.tokens(case["rows"], case["width"])
        lin = st["layer"] = d.layer(case["width"], case["outs"], case["rotate"], case["row_scale"])
        if case["rank"]:   # as the dynamic LoRA hook leaves it on the layer: the strength inside lora_A
            lin.lora_A = d.normal(case["rank"], case["width"], std=0.02).to(d.dtype)
            lin.lora_B = d.normal(case["outs"], case["rank"], std=0.02).to(d.dtype)
    elif kind == "fanout":
        st["x"] = d.tokens(case["rows"], case["width"])
        st["norm_weight"] = (1.0 + d.normal(case["width"], std=0.2)).to(d.dtype)
        st["scale"] = d.vectors(case["width"])
        st["layers"] = [d.layer(case["width"], case["outs"], case["rotate"], bias=False) for _ in range(case["layers"])]
    elif kind == "mlp":
        st["x"] = d.tokens(case["rows"], case["width"])
        st["up"], st["down"] = d.layer(case["width"], case["hidden"]), d.layer(case["hidden"], case["width"])
        st["scale"], st["shift"], st["gate"] = (d.vectors(case["width"]) for _ in range(3))
    elif kind == "double":
        w, streams = case["width"], (case["rows"], case["text"])
        st["vec"] = d.normal(1, w).to(d.dtype)
        for name, k, n in (("mod", w, 6 * w), ("qkv", w, 3 * w), ("proj", w, w), ("up", w, 4 * w), ("down", 4 * w, w)):
            st[name] = [d.layer(k, n) for _ in streams]
        # what the model's attention and elementwise kernels hand to each projection, and the residual streams
        st["x"], st["attn_in"], st["attn_out"], st["mlp_in"] = ([d.tokens(m, w) for m in streams] for _ in range(4))
        st["hidden"] = [torch.nn.functional.gelu(d.normal(1, m, 4 * w), approximate="tanh").to(d.dtype) for m in streams]
    elif kind == "single":
        w = case["width"]
        st["x"], st["attn"] = d.tokens(case["rows"], w), d.normal(1, case["rows"], w).to(d.dtype)
        st["linear1"], st["linear2"] = d.layer(w, 7 * w), d.layer(5 * w, w)
        st["scale"], st["shift"], st["gate"] = (d.vectors(w) for _ in range(3))
    else:
        n, k = case["outs"], case["width"]
        st["weight"], scale = pkg.hip_quantize_rowwise(d.normal(n, k, std=0.02))
        loras = [d.lora(n, k, int(r)) for r in case["ranks"].split()]
        if kind == "merge":
            st["adapter"] = pkg.INT8LoRAPatchAdapter(set(), loras[0], scale, seed=seed & 0xFFFF)
        else:
            parts = [(pkg.INT8LoRAPatchAdapter(set(), w, scale), 1.0 - 0.25 * i) for i, w in enumerate(loras)]
            st["adapter"] = pkg.INT8MergedLoRAPatchAdapter(parts, scale, seed=seed & 0xFFFF)
    return st


# --------------------------------------------------------------------------- one pass
@torch.no_grad()
def run(st):
    kind = st["kind"]
    if kind == "vector":
        if len(st["layers"]) == 1:
            return [st["layers"][0](st["x"])]
        return pkg.forward_fanout(st["layers"], st["x"])
    if kind == "linear":
        return [st["layer"](st["x"])]
    if kind == "fanout":
        return pkg.forward_fanout(st["layers"], st["x"], prologue=L.PRO_RMS_NORM, mod_scale=st["scale"], norm_weight=st["norm_weight"], eps=1e-5)
    if kind == "mlp":
        h = st["up"](st["x"], prologue=L.PRO_NORM_MODULATE, mod_scale=st["scale"], mod_shift=st["shift"])
        return [st["down"](h, prologue=L.PRO_GELU_TANH, gate=st["gate"], residual=st["x"])]
    if kind == "double":
        mods = pkg.forward_fanout(st["mod"], st["vec"])
        parts = [m[:, None, :].chunk(6, dim=-1) for m in mods]
        qkv = pkg.forward_pair(st["qkv"], st["attn_in"])
        x = pkg.forward_pair(st["proj"], st["attn_out"], gates=[p[2] for p in parts], residuals=st["x"])
        up = pkg.forward_pair(st["up"], st["mlp_in"])
        out = pkg.forward_pair(st["down"], st["hidden"], gates=[p[5] for p in parts], residuals=x)
        return [*mods, *qkv, *up, *out]
    if kind == "single":
        w = st["x"].shape[-1]
        y = st["linear1"](st["x"], prologue=L.PRO_NORM_MODULATE, mod_scale=st["scale"], mod_shift=st["shift"])
        qkv, mlp = y.split((3 * w, 4 * w), dim=-1)
        return [qkv, st["linear2"](st["attn"], prologue=L.PRO_CONCAT_GELU, mod_scale=mlp, gate=st["gate"], residual=st["x"])]
    return [st["adapter"].calculate_weight(st["weight"], "", 1.0, 1.0, None, None)]


# --------------------------------------------------------------------------- what a pass cannot do without
def _layer_bytes(width, outs):
    return width * outs + 6 * outs   # int8 weight, binary32 scale and 16-bit bias of each row


def work(case):
    kind = case["kind"]
    if kind in ("merge", "stack"):   # weight in and out, factors; the random numbers are the pass's own
        n, k, ranks = case["outs"], case["width"], [int(r) for r in case["ranks"].split()]
        return {"bytes": 2 * n * k + 4 * n + 4 * sum(ranks) * (n + k), "flops": 2 * n * k * sum(ranks)}
    m, w = case["rows"], case["width"]
    if kind == "vector":
        n, c = case["outs"], case["layers"]
        return {"bytes": 2 * m * w + c * (_layer_bytes(w, n) + 2 * m * n), "flops": 2 * c * m * w * n}
    if kind == "linear":
        n, r = case["outs"], case["rank"]
        return {"bytes": 2 * m * w + _layer_bytes(w, n) + 2 * m * n + 2 * r * (w + n), "flops": 2 * m * w * n + 2 * m * r * (w + n)}
    if kind == "fanout":
        n, c = case["outs"], case["layers"]
        return {"bytes": 2 * m * w + c * (_layer_bytes(w, n) + 2 * m * n), "flops": 2 * c * m * w * n}
    if kind == "mlp":   # (the hidden activations stay inside the pass)
        h = case["hidden"]
        return {"bytes": 4 * m * w + _layer_bytes(w, h) + _layer_bytes(h, w), "flops": 4 * m * w * h}
    if kind == "double":
        # in: the four inputs and the residual of each token; out: qkv, up and the residual stream
        per_token = 2 * (4 * w + 4 * w + 3 * w + 4 * w + w)
        layers = _layer_bytes(w, 6 * w) + _layer_bytes(w, 3 * w) + _layer_bytes(w, w) + _layer_bytes(w, 4 * w) + _layer_bytes(4 * w, w)
        t = m + case["text"]
        return {"bytes": t * per_token + 2 * layers, "flops": 2 * t * w * 12 * w + 2 * 2 * w * 6 * w}
    # single: x, attn and (inside) the activations; out: qkv and x
    return {"bytes": 2 * m * (2 * w + 3 * w + w) + _layer_bytes(w, 7 * w) + _layer_bytes(5 * w, w), "flops": 2 * m * w * 12 * w}


def tolerance(case):
    return TOLERANCES[case["kind"]]
