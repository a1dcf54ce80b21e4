"""Workloads of the MXFP attention path: what is timed when its performance is worked on.

A case is a dict of plain values.  ``kind`` says which public entry points a pass goes through:

  attn    one call of ``ours.mxfp_attn.mxfp_attn`` on 16-bit q, k, v (self-attention with and without the causal mask,
          grouped heads, cross attention, routed precision, tile skipping)
  linear  a linear layer with MX weights: the activations are quantized (``quantize_mx``) and multiplied with weights that
          were quantized once (``block_scaled_matmul``)
  gemm    both operands quantized and multiplied (``quantize_block_scaled_from_tensor`` + ``block_scaled_matmul``)
  scores  the call sequence of code written against the reference: quantizer with one code per byte, scales in the packed
          layout, operand packaging, batched score product
"""

import math
import os
import sys

import torch

# the package of the tree that is the working folder
sys.path.insert(0, os.path.join(os.getcwd(), "mp-sparse-attn_amd"))

from ours import _lib  # noqa: E402
from ours.batched_block_scaled_matmul import block_scaled_batched_matmul  # noqa: E402
from ours.block_scaled_matmul import (block_scaled_matmul, make_configs, pack_scale_5d,  # noqa: E402
                                      quantize_block_scaled_from_tensor)
from ours.mxfp_attn import mxfp_attn  # noqa: E402
from ours.mxfp_attn_kernel import initialize_block_scaled_batched_from_tensor  # noqa: E402
from ours.quant_mxint8 import quant_mxfp4, quant_mxfp8e5, quantize_mx  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
LARGEST_FLOPS = 2.0 * 32 * 131072 ** 2 * 128


def _attn(name, **kw):
    case = {"name": name, "kind": "attn", "B": 1, "Hq": 32, "Hkv": 8, "Nq": 0, "Nk": 0, "D": 128, "causal": True, "dtype": "bf16",
            "layout": "HND", "type": "diag", "tile": 128, "smooth_k": False, "skip_thresh": 0.0, "route_thresh": 0.0,
            "values": "outliers"}
    case.update(kw)
    case["Nq"] = case["Nq"] or case["Nk"]
    return case


def listed():
    return [
        # prefill of a chat turn: every layer of a Llama-style model makes this call, and at this length a call is latency
        _attn("prompt_160", Nk=160),
        # a page or two of prompt, a length that is no multiple of a tile
        _attn("prompt_1000", Nk=1000),
        # the headline configuration: Llama-3-8B-shaped prefill
        _attn("prompt_8192", Nk=8192),
        # long-context prefill, the largest configuration
        _attn("prompt_131072", Nk=131072),
        # the small configuration: 64-wide heads, 64 x 64 tiles, the entry point's default smoothing of K
        _attn("heads64_1024", Hq=8, Hkv=8, Nk=1024, D=64, tile=64, smooth_k=True, values="plain"),
        # cross attention of an image or video transformer to its text tokens: fp16, [B,N,H,D] layout, two samples (guidance)
        _attn("cross_4096x333", B=2, Hq=16, Hkv=16, Nq=4096, Nk=333, causal=False, dtype="fp16", layout="NHD", type="mxfp8",
              smooth_k=True, values="plain"),
        # video-DiT self-attention, precision chosen per tile by the router
        _attn("dit_32760_routed", Hq=40, Hkv=40, Nk=32760, causal=False, type="routed", route_thresh=0.97, smooth_k=True,
              values="frames"),
        # the same sequence with the reference's tile skipping, one rank's share of the heads
        _attn("dit_32760_skip", Hq=8, Hkv=8, Nk=32760, causal=False, type="mxfp4", skip_thresh=1.1, values="frames"),
        # decode: a linear layer on the new tokens of a batch of 16 sequences
        {"name": "linear_16x4096x4096", "kind": "linear", "M": 16, "N": 4096, "K": 4096, "type": "mxfp4", "dtype": "bf16"},
        # prefill of 1000 tokens through a wide layer, 8-bit activations and 4-bit weights
        {"name": "linear_1000x14336x4096", "kind": "linear", "M": 1000, "N": 14336, "K": 4096, "type": "mixed", "dtype": "bf16"},
        # the quantize + multiply configuration
        {"name": "gemm_8192", "kind": "gemm", "M": 8192, "N": 8192, "K": 8192, "type": "mxfp4", "packed": True, "dtype": "bf16"},
        # score product through the reference's own sequence of calls
        {"name": "scores_2048", "kind": "scores", "B": 1, "Hq": 16, "Hkv": 16, "N": 2048, "type": "mxfp4", "dtype": "fp16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    pick = rng.choice(["prompt", "prompt", "prompt", "small", "dense", "cross", "routed", "skip", "linear", "linear", "linear", "gemm", "scores"])
    if pick == "prompt":            # causal prefill, a few hundred to some ten thousand tokens
        hkv = rng.choice([1, 2, 4, 8])
        case = _attn("", B=rng.choice([1, 1, 1, 2, 4]), Hkv=hkv, Hq=hkv * rng.choice([1, 4, 4, 8]), Nk=_log(rng, 128, 49152),
                     type=rng.choice(["diag", "diag", "mxfp4", "mxfp8", "mixed"]), dtype=rng.choice(["bf16", "bf16", "fp16"]),
                     layout=rng.choice(["HND", "NHD"]), smooth_k=rng.random() < 0.3)
    elif pick == "small":           # 64-wide heads
        h = rng.choice([4, 8, 12, 16, 32])
        case = _attn("", B=rng.choice([1, 2, 4]), Hq=h, Hkv=h, Nk=_log(rng, 128, 16384), D=64, tile=rng.choice([64, 128]),
                     causal=rng.random() < 0.6, type=rng.choice(["diag", "mxfp4", "mxfp8"]), dtype=rng.choice(["bf16", "fp16"]),
                     layout=rng.choice(["HND", "NHD"]), smooth_k=True, values="plain")
    elif pick == "dense":           # image / video self-attention without a mask
        h = rng.choice([8, 16, 24, 40])
        case = _attn("", B=rng.choice([1, 1, 2]), Hq=h, Hkv=h, Nk=_log(rng, 256, 32768), causal=False,
                     type=rng.choice(["diag", "mxfp4", "mxfp8", "mixed"]), dtype=rng.choice(["bf16", "fp16"]),
                     layout=rng.choice(["HND", "NHD"]), smooth_k=rng.random() < 0.5, values="frames")
    elif pick == "cross":
        h = rng.choice([8, 16, 24])
        case = _attn("", B=rng.choice([1, 2]), Hq=h, Hkv=h, Nq=_log(rng, 256, 32768), Nk=_log(rng, 77, 1024), causal=False,
                     type=rng.choice(["mxfp4", "mxfp8"]), dtype=rng.choice(["bf16", "fp16"]), layout=rng.choice(["HND", "NHD"]),
                     smooth_k=rng.random() < 0.5, values="plain")
    elif pick in ("routed", "skip"):
        h = rng.choice([4, 8, 16, 40])
        case = _attn("", Hq=h, Hkv=h, Nk=_log(rng, 1024, 32768), causal=False, type="routed" if pick == "routed" else rng.choice(["mxfp4", "mxfp8"]),
                     route_thresh=rng.choice([0.95, 0.97, 0.99]) if pick == "routed" else 0.0,
                     skip_thresh=rng.choice([0.9, 1.0, 1.1]) if pick == "skip" else 0.0, smooth_k=pick == "routed", values="frames")
    elif pick == "linear":
        case = {"kind": "linear", "M": _log(rng, 1, 8192), "N": 128 * _log(rng, 8, 128), "K": 128 * _log(rng, 8, 112),
                "type": rng.choice(["mxfp4", "mixed", "mxfp8"]), "dtype": rng.choice(["bf16", "bf16", "fp16"])}
    elif pick == "gemm":
        size = lambda: 128 * _log(rng, 2, 64)  # noqa: E731
        case = {"kind": "gemm", "M": size(), "N": size(), "K": size(), "type": rng.choice(["mxfp4", "mxfp8", "mixed"]),
                "packed": rng.random() < 0.5, "dtype": "bf16"}
    else:
        hkv = rng.choice([4, 8, 16])
        case = {"kind": "scores", "B": 1, "Hq": hkv * rng.choice([1, 2]), "Hkv": hkv, "N": 128 * _log(rng, 1, 32),
                "type": rng.choice(["mxfp4", "mxfp8e5"]), "dtype": "fp16"}
    case.pop("name", None)
    while work(case)["flops"] > LARGEST_FLOPS / 2:
        case["Nq"] = case["Nk"] = case["Nk"] * 3 // 4
    return case


def _randn(gen, dtype, *shape):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32).to(dtype)


def _qkv(case, gen):
    """q, k, v as the model hands them over: [B,N,H,D] memory for "NHD", [B,H,N,D] for "HND".  ``values``: "plain" N(0,1);
    "outliers": one channel per head of q and of k is 20 times as large, as in language models; "frames": sigma 0.5 and an
    offset per frame and channel on q and k, as in video transformers."""
    dt, D = DTYPES[case["dtype"]], case["D"]
    out = []
    for name, H, N in (("q", case["Hq"], case["Nq"]), ("k", case["Hkv"], case["Nk"]), ("v", case["Hkv"], case["Nk"])):
        x = torch.empty(case["B"], H, N, D, device="cuda", dtype=dt)
        if case["values"] == "frames":
            x.normal_(0.0, 0.5, generator=gen)
            if name != "v":
                frames = 21
                off = 0.5 * torch.randn(frames, D, generator=gen, device="cuda")
                x += off[torch.arange(N, device="cuda") * frames // N].to(dt)
        else:
            x.normal_(0.0, 1.0, generator=gen)
            if case["values"] == "outliers" and name != "v":
                channel = torch.randint(0, D, (1, H, 1, 1), generator=gen, device="cuda")
                x *= torch.ones(1, H, 1, D, device="cuda").scatter_(3, channel, 20.0).to(dt)
        out.append(x.transpose(1, 2).contiguous() if case["layout"] == "NHD" else x)
    return out


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    state = {"case": case}
    if case["kind"] == "attn":
        state["q"], state["k"], state["v"] = _qkv(case, gen)
    elif case["kind"] == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        state["configs"] = configs = make_configs(case["type"])
        state["fmt_x"] = _lib.FMT_E2M1 if configs["ELEM_PER_BYTE_A"] == 2 else _lib.FMT_E4M3
        weight = _randn(gen, dt, N, K) * 0.02
        codes, scales = quantize_mx(weight[None, None], 1.0, _lib.FMT_E2M1 if configs["ELEM_PER_BYTE_B"] == 2 else _lib.FMT_E4M3)
        state["w"], state["ws"] = codes[0, 0], scales[0, 0]
        state["x"] = _randn(gen, dt, M, K)
    elif case["kind"] == "gemm":
        state["a"], state["b"] = _randn(gen, dt, case["M"], case["K"]), _randn(gen, dt, case["N"], case["K"])
    else:
        B, N = case["B"], case["N"]
        state["q"], state["k"] = _randn(gen, dt, B, case["Hq"], N, 128), _randn(gen, dt, B, case["Hkv"], N, 128)
    return state


def run(state):
    case = state["case"]
    dt = DTYPES[case["dtype"]]
    if case["kind"] == "attn":
        skip = case["skip_thresh"] or None
        return mxfp_attn(state["q"], state["k"], state["v"], is_causal=case["causal"], smooth_k=case["smooth_k"],
                         tensor_layout=case["layout"], output_dtype=dt, return_sparsity=skip is not None, skip_thresh=skip,
                         block_scale_type=case["type"], BLKQ=case["tile"], route_thresh=case["route_thresh"] or None)
    if case["kind"] == "linear":
        codes, scales = quantize_mx(state["x"][None, None], 1.0, state["fmt_x"])
        return block_scaled_matmul(codes[0, 0], scales[0, 0], state["w"], state["ws"], dt, case["M"], case["N"], case["K"], state["configs"])
    if case["kind"] == "gemm":
        a, sa, b, sb, configs = quantize_block_scaled_from_tensor(state["a"], state["b"], case["type"], packed_scales=case["packed"])
        c = block_scaled_matmul(a, sa, b, sb, dt, case["M"], case["N"], case["K"], configs)
        return {"c": c, "a": a, "sa": sa, "b": b, "sb": sb}
    if case["type"] == "mxfp4":
        qc, qs, kc, ks = quant_mxfp4(state["q"], state["k"], packed=False)
    else:
        qc, qs, kc, ks = quant_mxfp8e5(state["q"], state["k"])
    a, sa, b, sb, configs, _ = initialize_block_scaled_batched_from_tensor(qc, kc, pack_scale_5d(qs), pack_scale_5d(ks), case["type"])
    return block_scaled_batched_matmul(a, sa, b, sb, dt, case["B"], case["Hq"], case["N"], case["N"], 128, configs)


def work(case):
    if case["kind"] == "attn":
        B, Hq, Hkv, Nq, Nk, D = (case[x] for x in ("B", "Hq", "Hkv", "Nq", "Nk", "D"))
        pairs = Nq * (Nq + 1) / 2 if case["causal"] else Nq * Nk
        # tile skipping: every score is needed for its tile's statistic, P.V only where a tile is kept (about half)
        flops = (3.0 if case["skip_thresh"] else 4.0) * B * Hq * D * pairs
        return {"bytes": 2.0 * B * D * (2 * Hq * Nq + 2 * Hkv * Nk), "flops": flops}
    if case["kind"] == "scores":
        B, Hq, Hkv, N = (case[x] for x in ("B", "Hq", "Hkv", "N"))
        return {"bytes": 2.0 * B * (Hq + Hkv) * N * 128 + 2.0 * B * Hq * N * N, "flops": 2.0 * B * Hq * N * N * 128}
    M, N, K = case["M"], case["N"], case["K"]
    configs = make_configs(case["type"])
    width = lambda epb: 1.0 / epb + 1.0 / 32  # noqa: E731  bytes per quantized element
    if case["kind"] == "linear":
        moved = 2.0 * M * K + N * K * width(configs["ELEM_PER_BYTE_B"]) + 2.0 * M * N
    else:
        moved = M * K * (2.0 + width(configs["ELEM_PER_BYTE_A"])) + N * K * (2.0 + width(configs["ELEM_PER_BYTE_B"])) + 2.0 * M * N
    return {"bytes": moved, "flops": 2.0 * M * N * K}


def tolerance(case):
    # results are rounded to 16 bits, and so is P in front of the P.V product; codes and scale bytes are exact
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3}
