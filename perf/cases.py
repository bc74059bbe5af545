"""The performance cases of the fused attention library: what a program has it do, through the
compiled module `fused_attn`, from the smallest call to the largest.

`listed()` names twelve calls, `draw(rng)` gives more from the same ranges; `prepare` makes the
tensors a program holds before the call, `run` is one call, `work` the bytes and operations the
call cannot do without and `tolerance` the error another correct implementation would show.

Keys of a case:
  op       "attention", "projection" (the QKV projection), or "block" (the projection, then causal
           attention on three views of its packed output, with no copy in between)
  B R L H  batch, heads, sequence length, head_dim
  F_in     input features of the projection (0 for plain attention)
  dtype    "fp16" or "bf16"
  mask     "none", "causal" (the flag), "padding" (additive [B, L, L], 0 where the key exists and
           -inf behind the end of its sequence) or "bias" (additive, a finite value per score)
  layout   "blf" ([B, L, R*H]), "bhld" ([B, R, L, H]) or "packed" (three slices of [B, L, 3, R*H])
  lse      the log-sum-exp of every row is returned as well (what a backward pass keeps)
  rope     the projection applies a rotary position encoding to q and k
  std      standard deviation of q, k and v: 1, or 3 for large scores
"""
import math

import torch

import fused_attn

# Scores of the largest listed case (B1 R32 L16384); a drawn case has no more, nor a larger projection
# than 0.55 TFLOP.
MOST_SCORES = 32 * 16384 * 16384
MOST_PROJECTION_FLOPS = 5.5e11

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _case(name, op, B, R, L, H, F_in=0, dtype="fp16", mask="none", layout="blf", lse=False, rope=False, std=1.0):
    case = {"op": op, "B": B, "R": R, "L": L, "H": H, "F_in": F_in, "dtype": dtype, "mask": mask,
            "layout": layout, "lse": lse, "rope": rope, "std": std}
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # one short prompt, few heads: the call's latency and its host path
        _case("smoke", "attention", 1, 4, 256, 64),
        # a batch of short sequences with narrow heads (compact encoders, set and patch models)
        _case("narrow_heads", "attention", 16, 8, 512, 32),
        # an encoder layer of twelve 64-wide heads on full sequences
        _case("encoder", "attention", 8, 12, 1024, 64),
        # the same layer on sequences padded to the longest of the batch, an odd length
        _case("encoder_padded", "attention", 16, 12, 381, 64, mask="padding"),
        # a relative position bias added to every score, the rows of the bias 16-byte aligned
        _case("position_bias", "attention", 2, 12, 2048, 64, dtype="bf16", mask="bias"),
        # a ragged length and scores of a wide spread
        _case("ragged_large_scores", "attention", 2, 8, 3073, 64, std=3.0),
        # long sequences, the headline configuration
        _case("long", "attention", 4, 16, 4096, 64),
        # training forward of a decoder: causal, [B, R, L, H] tensors, the log-sum-exp kept
        _case("long_causal", "attention", 4, 16, 4096, 64, dtype="bf16", mask="causal", layout="bhld", lse=True),
        # forty 128-wide heads, the configuration of the reference's own benchmark
        _case("wide_heads", "attention", 4, 40, 2048, 128),
        # one very long sequence, 128-wide heads
        _case("very_long", "attention", 1, 32, 16384, 128),
        # the QKV projection of the headline configuration, with bias and rotary encoding
        _case("projection", "projection", 4, 16, 4096, 64, F_in=1024, rope=True),
        # prefill of one prompt in a decoder of forty 128-wide heads: projection, then causal attention
        _case("prefill", "block", 1, 40, 512, 128, F_in=5120, dtype="bf16", mask="causal", layout="packed", rope=True),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _length(rng, low, high):
    """A sequence length, spread over the logarithm: as it falls, or a multiple of 64."""
    L = _log_int(rng, low, high)
    return L if rng.random() < 0.5 else max(64, L // 64 * 64)


def draw(rng):
    op = rng.choice(["attention"] * 6 + ["projection", "block"])
    dtype = rng.choice(["fp16", "bf16"])
    H = rng.choice([16, 32, 64, 64, 64, 128, 128])
    R = rng.choice([4, 8, 12, 16, 20, 32, 40])
    if op != "attention":
        H = max(H, 32)
        L = _length(rng, 64, 4096)
        F_in = rng.choice([1, 1, 2]) * R * H if R * H <= 2560 else R * H
        most_rows = min(16384, MOST_PROJECTION_FLOPS / (6.0 * F_in * R * H))
        L = min(L, max(64, int(most_rows)))
        B = max(1, min(_log_int(rng, 1, 16), int(most_rows // L)))
        block = op == "block"
        return _case(None, op, B, R, L, H, F_in=F_in, dtype=dtype, mask="causal" if block else "none",
                     layout="packed" if block else "blf", rope=rng.random() < 0.6)
    mask = rng.choice(["none", "none", "none", "causal", "causal", "padding", "bias"])
    L = _length(rng, 32, 4096 if mask in ("padding", "bias") else 16384)
    B = _log_int(rng, 1, 32)
    B = max(1, min(B, MOST_SCORES // (R * L * L)))
    if mask in ("padding", "bias"):
        B = max(1, min(B, (1 << 28) // (L * L)))      # a mask of half a gigabyte at most
    R = max(1, min(R, MOST_SCORES // (B * L * L)))
    layout = rng.choice(["blf", "blf", "bhld", "packed"])
    return _case(None, "attention", B, R, L, H, dtype=dtype, mask=mask, layout=layout, lse=rng.random() < 0.3,
                 std=rng.choice([1.0, 1.0, 1.0, 3.0]))


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]
    B, R, L, H, F = case["B"], case["R"], case["L"], case["H"], case["R"] * case["H"]

    def normal(*shape, std=1.0):
        return torch.randn(shape, generator=gen, device=dev, dtype=dtype).mul_(std)

    if case["op"] != "attention":
        F_in = case["F_in"]
        cos = sin = None
        if case["rope"]:
            inv = 10000.0 ** (-torch.arange(0, H, 2, device=dev, dtype=torch.float32) / H)
            angle = torch.arange(L, device=dev, dtype=torch.float32)[:, None] * inv[None, :]
            cos, sin = angle.cos(), angle.sin()
        return {"case": case, "hidden": normal(B, L, F_in), "weight": normal(F_in, 3 * F, std=1.0 / math.sqrt(F_in)),
                "bias": normal(3 * F, std=0.1), "cos": cos, "sin": sin}

    std = case["std"]
    if case["layout"] == "packed":
        qkv = normal(B, L, 3, F, std=std)
        q, k, v = qkv[:, :, 0], qkv[:, :, 1], qkv[:, :, 2]
    else:
        shape = (B, R, L, H) if case["layout"] == "bhld" else (B, L, F)
        q, k, v = (normal(*shape, std=std) for _ in range(3))
    mask = None
    if case["mask"] == "padding":
        # lengths spread over the upper half, the longest sequence fills the batch's length
        lengths = L - torch.randint(0, L // 2 + 1, (B,), generator=gen, device=dev)
        lengths[0] = L
        keys = torch.zeros(B, 1, L, device=dev, dtype=dtype)
        keys.masked_fill_(torch.arange(L, device=dev)[None, None, :] >= lengths[:, None, None], -math.inf)
        mask = keys.expand(B, L, L).contiguous()
    elif case["mask"] == "bias":
        mask = normal(B, L, L)
    return {"case": case, "q": q, "k": k, "v": v, "mask": mask}


def run(state):
    case = state["case"]
    H = case["H"]
    if case["op"] != "attention":
        qkv = fused_attn.qkv_projection(state["hidden"], state["weight"], state["bias"], case["R"], H, state["cos"],
                                        state["sin"])
        if case["op"] == "projection":
            return qkv
        return qkv, fused_attn.attention_forward_ex(qkv[:, :, 0], qkv[:, :, 1], qkv[:, :, 2], H, causal=True)
    q, k, v, mask = state["q"], state["k"], state["v"], state["mask"]
    if case["dtype"] == "fp16" and case["layout"] == "blf" and case["mask"] != "causal" and not case["lse"]:
        return fused_attn.attention_forward(H, min(128, 2 * H), q, k, v, mask)
    layout = "bhld" if case["layout"] == "bhld" else "blf"
    return fused_attn.attention_forward_ex(q, k, v, H, mask=mask, causal=case["mask"] == "causal",
                                           return_lse=case["lse"], layout=layout)


def work(case):
    B, R, L, H, F, F_in = case["B"], case["R"], case["L"], case["H"], case["R"] * case["H"], case["F_in"]
    nbytes = flops = 0.0
    if case["op"] != "attention":
        flops += 6.0 * B * L * F_in * F
        nbytes += 2.0 * (B * L * F_in + 3 * F_in * F + 3 * F + 3 * B * L * F)
        nbytes += 4.0 * L * H if case["rope"] else 0.0
    if case["op"] != "projection":
        share = 1.0
        if case["mask"] == "causal":
            share = (L + 1) / (2.0 * L)
        elif case["mask"] == "padding":
            share = (1.0 + 0.75 * (B - 1)) / B         # the keys that exist, on average
        flops += 4.0 * B * R * L * L * H * share
        # behind a projection q, k and v are its output: written once, counted above
        nbytes += 2.0 * B * L * F * (1 if case["op"] == "block" else 4)
        nbytes += 2.0 * B * L * L if case["mask"] in ("padding", "bias") else 0.0
        nbytes += 4.0 * B * R * L if case["lse"] else 0.0
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # one rounding of each result and, in attention, of each softmax weight, to 11 (fp16) or 8 (bf16)
    # significant bits; with large scores a few keys carry a row and the roundings do not average out
    if case["dtype"] == "fp16":
        return {"rel": 2e-3, "max": 2e-2}
    return {"rel": 1e-2, "max": 1e-1}
