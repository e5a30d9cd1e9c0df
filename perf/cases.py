"""The work that a user of the library has it do, as cases that can be timed and checked.

Every case goes through the Python binding of the C ABI, on the current stream, with inputs and
weights resident on the GPU as a denoising program holds them. `listed()` names twelve calls from
one denoise step of the joint audio-video transformer and from preparing its checkpoint; `draw()`
gives more of the same ranges.

Paths:
  linear   one quantized linear (`linear_q`, or `linear_q_noalloc` for callers that capture)
  ffn      the feed-forward pair: up with GELU-tanh fused, then down
  lora     a quantized linear with a low-rank adapter (`linear_q_lora`)
  dense    a bf16 linear of an unquantized tensor (`linear`)
  i8       a quantized linear under the int8 tier (`set_i8_gemm`)
  pack     quantizing a float weight into the packed format, and expanding it to bf16
"""
import importlib.util
import math
import os
import sys

import torch

ROOT = os.getcwd()


def _package():
    name = "vpipe_ltx25_amd"
    if name not in sys.modules:
        # the package directory's name is no Python identifier: it is loaded by its path
        spec = importlib.util.spec_from_file_location(
            name, os.path.join(ROOT, "vpipe-ltx-2.5_amd", "__init__.py"))
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


def _case(path, M, K, N, bits=8, group=64, bias="none", gelu=False, rank=0, noalloc=False, **name):
    return dict(name, path=path, M=M, K=K, N=N, bits=bits, group=group, bias=bias, gelu=gelu,
                rank=rank, noalloc=noalloc)


def listed():
    return [
        # An audio token projection (attention out, cross q and out: six of a block's linears):
        # the smallest call, a few microseconds of work.
        _case("linear", 126, 2048, 2048, bias="f32", name="audio_proj"),
        # The audio feed-forward; the reduction over 8192 is split between workgroups.
        _case("ffn", 126, 2048, 8192, bias="bf16", name="audio_ffn"),
        # The packed key / value projection of the 1024 prompt tokens (video cross-attention).
        _case("linear", 1024, 4096, 8192, bias="bf16", name="prompt_kv"),
        # One linear at a few hundred tokens, as in a short clip or a preview.
        _case("linear", 320, 4096, 4096, bias="f32", name="short_clip_proj"),
        # A video projection at the full token count (eight of a block's linears).
        _case("linear", 8160, 4096, 4096, bias="bf16", name="video_proj"),
        # The video feed-forward, most of a denoise step's time: the largest call.
        _case("ffn", 8160, 4096, 16384, name="video_ffn"),
        # The upscaler's rank-32 adapter on the feed-forward widening, at 128 tokens.
        _case("lora", 128, 4096, 16384, bias="bf16", gelu=True, rank=32, name="upscaler_lora"),
        # The distilled adapter (rank 450) on a video projection.
        _case("lora", 8160, 4096, 4096, bias="bf16", rank=450, name="distilled_lora"),
        # A 4-bit checkpoint's fused query / key / value projection, a quarter of the tokens.
        _case("linear", 2040, 4096, 12288, bits=4, group=32, bias="bf16", name="w4_qkv"),
        # The per-head gate logits, kept dense in a quantized checkpoint: 32 columns out.
        _case("dense", 8160, 4096, 32, bits=16, bias="bf16", name="gate_logits"),
        # A video projection on the int8 tier.
        _case("i8", 8160, 4096, 4096, bias="bf16", name="i8_proj"),
        # Packing a float weight to w8g64 when a checkpoint is made, and its bf16 expansion.
        _case("pack", 1, 4096, 16384, name="pack_weight"),
    ]


# The largest listed case's operations and bytes: no drawn case goes over either.
_MOST_FLOPS = 4.0 * 8160 * 4096 * 16384
_MOST_BYTES = 1.2e9


def _spread(rng, lo, hi):
    """A whole number, spread evenly over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        path = rng.choice(["linear", "linear", "linear", "ffn", "lora", "lora", "dense", "i8", "pack"])
        bits, group = rng.choice([(8, 64), (8, 64), (8, 32), (4, 64), (4, 32)])
        M = _spread(rng, 1, 8192)
        K = 64 * _spread(rng, 8, 256)
        N = 16 * _spread(rng, 4, 1024)
        if rng.random() < 0.15:
            N += rng.randint(1, 15)   # an output width that is no multiple of 16
        c = dict(bits=bits, group=group, bias=rng.choice(["none", "bf16", "f32"]))
        if path == "linear":
            c.update(gelu=rng.random() < 0.3, noalloc=rng.random() < 0.2)
        elif path == "ffn":
            # the hidden width is the wider one, and the down projection's reduction
            K, N = sorted((K, 64 * max(1, N // 64)))
        elif path == "lora":
            c.update(gelu=rng.random() < 0.3, rank=_spread(rng, 4, 512))
        elif path == "dense":
            c.update(bits=16, group=64)
        elif path == "i8":
            # the tier's own floors; under them it declines
            M, K = max(M, 1024), 128 * max(8, K // 128)
            c.update(gelu=rng.random() < 0.3)
        else:
            M = 1
            c.update(bias="none")
        case = _case(path, M, K, N, **c)
        w = work(case)
        if w["flops"] <= _MOST_FLOPS and w["bytes"] <= _MOST_BYTES:
            return case


# ---- inputs ---------------------------------------------------------------------------

def _randn(gen, *shape):
    return torch.randn(shape, device="cuda", generator=gen)


def _quantized(gen, N, K, bits, group):
    """A weight as a checkpoint holds it: normal values, group-affine codes (little-endian
    bytes, low bits first), bf16 scales and zero points."""
    w = (_randn(gen, N, K) * 0.02).view(N, K // group, group)
    lo, hi = w.amin(2, keepdim=True), w.amax(2, keepdim=True)
    qmax = (1 << bits) - 1
    scale = ((hi - lo) / qmax).to(torch.bfloat16)
    zero = lo.to(torch.bfloat16)
    q = ((w - zero.float()) / scale.float()).round_().clamp_(0, qmax).to(torch.uint8).view(N, K)
    if bits == 4:
        q = q[:, 0::2] | (q[:, 1::2] << 4)
    return q.contiguous(), scale.view(N, -1).contiguous(), zero.view(N, -1).contiguous()


def _bias(gen, n, kind):
    b = _randn(gen, n) * 0.02
    return None if kind == "none" else b.to(torch.bfloat16) if kind == "bf16" else b


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    M, K, N = case["M"], case["K"], case["N"]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1000003 * int(seed) + 17)
    s = {}
    if case["path"] == "pack":
        s["w"] = _randn(gen, N, K) * 0.02
        return s
    s["x"] = _randn(gen, M, K).to(torch.bfloat16)
    if case["path"] == "dense":
        s["w"] = (_randn(gen, N, K) * 0.02).to(torch.bfloat16)
    else:
        s["q"] = _quantized(gen, N, K, case["bits"], case["group"])
    s["bias"] = _bias(gen, N, case["bias"])
    if case["path"] == "ffn":
        s["q2"] = _quantized(gen, K, N, case["bits"], case["group"])
        s["bias2"] = _bias(gen, K, case["bias"])
    if case["path"] == "lora":
        s["a"] = (_randn(gen, case["rank"], K) * 0.02).to(torch.bfloat16)
        s["b"] = (_randn(gen, N, case["rank"]) * 0.02).to(torch.bfloat16)
    return s


def prepare(case, seed):
    pkg = _package()
    pkg.load()
    s = _inputs(case, seed)
    M, K, N = case["M"], case["K"], case["N"]

    def out(rows, cols):
        return torch.empty((rows, cols), dtype=torch.bfloat16, device="cuda")

    s["pkg"], s["case"] = pkg, case
    s["epilogue"] = pkg.EPI_GELU_TANH if case["gelu"] else pkg.EPI_NONE
    if case["path"] == "pack":
        bits, group = case["bits"], case["group"]
        s["codes"] = torch.empty((N, K * bits // 8), dtype=torch.uint8, device="cuda")
        s["scales"], s["zeros"] = out(N, K // group), out(N, K // group)
        s["qw"] = pkg.QWeight(s["codes"], s["scales"], s["zeros"], bits, group)
        s["expanded"] = out(N, K)
        return s
    for name in ("q", "q2"):
        if name in s:
            s[name + "w"] = pkg.QWeight(*s[name], case["bits"], case["group"])
    s["y"] = out(M, K if case["path"] == "ffn" else N)
    if case["path"] == "ffn":
        s["h"] = out(M, N)
    return s


def run(state):
    s, pkg = state, state["pkg"]
    c = s["case"]
    M, K, N = c["M"], c["K"], c["N"]
    if c["path"] == "linear":
        linear = pkg.linear_q_noalloc if c["noalloc"] else pkg.linear_q
        linear(s["x"], s["qw"], s["bias"], s["y"], M, K, N, s["epilogue"])
    elif c["path"] == "ffn":
        pkg.linear_q(s["x"], s["qw"], s["bias"], s["h"], M, K, N, pkg.EPI_GELU_TANH)
        pkg.linear_q(s["h"], s["q2w"], s["bias2"], s["y"], M, N, K)
    elif c["path"] == "lora":
        pkg.linear_q_lora(s["x"], s["qw"], s["bias"], s["a"], s["b"], c["rank"], s["y"], M, K, N,
                          s["epilogue"])
    elif c["path"] == "dense":
        pkg.linear(s["x"], s["w"], s["bias"], s["y"], M, K, N)
    elif c["path"] == "i8":
        # the switch is process-wide, so a program that mixes tiers sets it around its calls
        pkg.set_i8_gemm(True)
        pkg.linear_q(s["x"], s["qw"], s["bias"], s["y"], M, K, N, s["epilogue"])
        pkg.set_i8_gemm(False)
    else:
        pkg.quantize_affine(s["w"], s["codes"], s["scales"], s["zeros"], N, K, c["bits"],
                            c["group"])
        pkg.dequant(s["qw"], s["expanded"], N, K)
        return {"codes": s["codes"], "scales": s["scales"], "zeros": s["zeros"],
                "expanded": s["expanded"]}
    return s["y"]


# ---- what a pass cannot do without ------------------------------------------------------

def work(case):
    M, K, N, r = case["M"], case["K"], case["N"], case["rank"]
    bits = case["bits"]
    weight = 2.0 * N * K if bits == 16 else N * K * bits / 8 + 4.0 * N * K / case["group"]
    if case["path"] == "pack":
        # the float weight in; codes, scales and zero points out; the bf16 expansion out
        return {"bytes": 4.0 * N * K + weight + 2.0 * N * K, "flops": 4.0 * N * K}
    bias = {"none": 0, "bf16": 2, "f32": 4}[case["bias"]]
    if case["path"] == "ffn":
        return {"bytes": 2 * weight + bias * (N + K) + 4.0 * M * K, "flops": 4.0 * M * N * K}
    return {"bytes": weight + bias * N + 2.0 * M * (K + N) + 2.0 * r * (K + N),
            "flops": 2.0 * M * N * K + 2.0 * M * r * (K + N)}


# bf16 outputs: over the listed cases and two dozen drawn ones a pass is 1.7e-3 to 3.6e-3 (2-norm)
# and up to 1.8e-2 at one value off the products in 64 bits, mostly by the rounding of the weight,
# the hidden activations and the output to bf16. Summed in another order, values near a rounding
# boundary move by a bf16 ulp: up to 2.2e-4, and 1.2e-2 at one value. The int8 tier's quantization
# is fixed, so two implementations differ by output roundings alone. The packed format is bytes,
# and its expansion one rounding of an exact value.
def tolerance(case):
    if case["path"] == "pack":
        return "exact"
    return {"rel": 1e-2, "max": 6e-2}


# ---- the same in 64 bits ----------------------------------------------------------------

def _weight64(q, bits, group):
    codes, scale, zero = q
    if bits == 4:
        codes = torch.stack((codes & 15, codes >> 4), 2).flatten(1)
    n, k = codes.shape
    w = codes.view(n, k // group, group).double()
    return (w * scale.double()[:, :, None] + zero.double()[:, :, None]).view(n, k)


def exact(case, seed):
    if case["path"] == "pack":
        return None   # bytes and single roundings, defined in 32 bits step by step
    s = _inputs(case, seed)
    bits, group = case["bits"], case["group"]
    gelu = lambda v: torch.nn.functional.gelu(v, approximate="tanh")  # noqa: E731

    def linear(x, w, bias):
        y = x @ w.t()
        return y if bias is None else y.add_(bias.double())

    w = s["w"].double() if case["path"] == "dense" else _weight64(s["q"], bits, group)
    w2 = _weight64(s["q2"], bits, group) if case["path"] == "ffn" else None
    rows = []
    for x in s["x"].split(2048):   # a few rows at a time, for the memory of 64-bit copies
        x = x.double()
        y = linear(x, w, s["bias"])
        if case["path"] == "lora":
            y += (x @ s["a"].double().t()) @ s["b"].double().t()
        if case["path"] == "ffn":
            y = linear(gelu(y), w2, s["bias2"])
        rows.append(gelu(y) if case["gelu"] else y)
    return torch.cat(rows)
