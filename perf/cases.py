"""Performance cases: the attention-forward and fp16-GEMM calls a user of this framework makes.

Every case goes through a public Python entry point (`flash_atten.flash_attention` on a tuner's launch
spec, `flash_atten.attention`, `flash_atten.sdpa`, `mma._matmul_contiguous_kernel`, `mma.matmul`). Sizes
are those of the benchmark, the tests and the decode and TTFT harnesses, and generic odd ones.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parent.parent / "flash-attn-economical-gpu_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import flash_atten  # noqa: E402
import mma  # noqa: E402
import tuner  # noqa: E402

_DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
_TUNERS = {
    "basic": tuner.FlashAttentionTuner,
    "optimized": tuner.FlashAttentionOptimizeSharedMemTuner,
    "sliced": tuner.FlashAttentionBlockDNomaskTuner,
}


def _attn(name, op, variant, dtype, B, H, H_kv, M, N, D, causal=False, lse=False):
    case = {"op": op, "variant": variant, "dtype": dtype, "B": B, "H": H, "H_kv": H_kv, "M": M, "N": N, "D": D,
            "causal": causal, "lse": lse}
    return case if name is None else {"name": name, **case}


def _gemm(name, op, M, N, K):
    case = {"op": op, "M": M, "N": N, "K": K}
    return case if name is None else {"name": name, **case}


def listed():
    return [
        # the benchmark's headline: long non-causal attention, tuned spec launched in a loop (the largest call)
        _attn("opt_f16_d128_8k", "spec", "optimized", "f16", 4, 32, 32, 8192, 8192, 128),
        # a training-length causal forward that keeps the log-sum-exp (its backward would need it)
        _attn("opt_f16_d128_2k_causal_lse", "spec", "optimized", "f16", 4, 32, 32, 2048, 2048, 128, True, True),
        # the benchmark's large-head-dimension configuration, bf16, split-KV variant
        _attn("sliced_bf16_d256_2k", "spec", "sliced", "bf16", 2, 16, 16, 2048, 2048, 256),
        # the reference's own pipeline case (one sequence, 28 heads) through its default kernel
        _attn("basic_f16_28h_8k", "spec", "basic", "f16", 1, 28, 28, 8192, 8192, 128),
        # the smallest attention configuration (latency and launch cost)
        _attn("opt_f16_d64_512", "spec", "optimized", "f16", 1, 4, 4, 512, 512, 64),
        # prefill of one 4096-token prompt in a grouped-query decoder: strided projection views
        _attn("prefill_bf16_gqa_4k", "sdpa", "sliced", "bf16", 1, 12, 2, 4096, 4096, 128, True),
        # cross-attention of odd lengths, head dim 64, called without keeping a launch spec
        _attn("odd_bf16_d64_777x1283", "attention", "optimized", "bf16", 2, 16, 16, 777, 1283, 64, False, True),
        # decode step of a single sequence: one query row against an 8k KV cache
        _attn("decode_bf16_b1_8k", "sdpa", "sliced", "bf16", 1, 32, 8, 1, 8192, 128),
        # decode step of a serving batch with long caches (bandwidth)
        _attn("decode_bf16_b8_32k", "sdpa", "sliced", "bf16", 8, 32, 8, 1, 32768, 128),
        # a product of odd sizes (no tile divides it; rows of B are not 16-byte multiples)
        _gemm("gemm_1000x1004x1000", "matmul", 1000, 1004, 1000),
        # the reference's own GEMM test and chart shape: short K, the C write dominates
        _gemm("gemm_8192x8192x256", "kernel", 8192, 8192, 256),
        # the benchmark's square GEMM
        _gemm("gemm_8192", "kernel", 8192, 8192, 8192),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _step(x, step):
    return max(step, x // step * step)


_MAX_PAIRS = 4 * 32 * 8192 * 8192 * 128  # B H M N D of the largest listed attention case


def draw(rng):
    kind = rng.choice(["spec", "spec", "prefill", "odd", "decode", "gemm", "matmul"])
    if kind in ("spec", "odd"):
        D = rng.choice([64, 128, 128, 256])
        dtype = rng.choice(["f16", "bf16"])
        H_kv = rng.choice([2, 4, 8, 16])
        H = H_kv * rng.choice([1, 1, 2, 4])
        B = rng.choice([1, 1, 2, 4])
        causal = rng.random() < 0.5
        N = _log_uniform(rng, 256, 16384)
        while B * H * N * N * D > _MAX_PAIRS:
            N //= 2
        if kind == "spec":
            N = _step(N, 64)
            return _attn(None, "spec", rng.choice(["basic", "optimized", "optimized", "sliced"]), dtype, B, H, H_kv, N,
                         N, D, causal, rng.random() < 0.5)
        M = N if causal else max(17, int(N * rng.uniform(0.2, 1.0)))
        return _attn(None, "attention", "optimized", dtype, B, H, H_kv, M, N, D, causal, True)
    if kind == "prefill":
        H, H_kv, D = rng.choice([(12, 2, 128), (32, 8, 128), (28, 4, 128), (16, 2, 64), (16, 16, 256)])
        N = _log_uniform(rng, 128, 16384)
        return _attn(None, "sdpa", "sliced", rng.choice(["f16", "bf16"]), rng.choice([1, 1, 2]), H, H_kv, N, N, D, True)
    if kind == "decode":
        H, H_kv, D = rng.choice([(32, 8, 128), (12, 2, 128), (16, 2, 64), (16, 16, 128), (8, 1, 256)])
        B = rng.choice([1, 1, 4, 8, 16, 32])
        N = _log_uniform(rng, 512, 131072)
        while B * H_kv * N * D > 8 * 8 * 65536 * 128:
            N //= 2
        return _attn(None, "sdpa", "sliced", rng.choice(["f16", "bf16", "bf16"]), B, H, H_kv, rng.choice([1, 1, 1, 4]), N, D)
    sizes = [_log_uniform(rng, 64, 8192) for _ in range(3)]
    if kind == "gemm":
        return _gemm(None, "kernel", _step(sizes[0], 128), _step(sizes[1], 64), _step(sizes[2], 32))
    return _gemm(None, "matmul", sizes[0], _step(sizes[1], 4), _step(sizes[2], 8))


def _inputs(case, seed):
    """q, k, v (or a, b) of one case: the same values for prepare() and exact()."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    if case["op"] in ("kernel", "matmul"):
        M, N, K = case["M"], case["N"], case["K"]
        a = torch.rand(M, K, device=dev, generator=gen) * 2 - 1
        b = torch.rand(K, N, device=dev, generator=gen) * 2 - 1
        return a.half(), b.half()
    B, H, H_kv, M, N, D = (case[x] for x in ("B", "H", "H_kv", "M", "N", "D"))
    dtype = _DTYPES[case["dtype"]]
    sigma = 0.5 if D == 256 else 1.0
    if case["op"] == "sdpa" and M > 8:
        # projection outputs [B, S, heads, D], seen by the layer as [B, heads, S, D]
        shapes = [(B, M, H, D), (B, N, H_kv, D), (B, N, H_kv, D)]
        return tuple((torch.randn(s, device=dev, generator=gen, dtype=dtype) * sigma).transpose(1, 2) for s in shapes)
    shapes = [(B, H, M, D), (B, H_kv, N, D), (B, H_kv, N, D)]
    return tuple(torch.randn(s, device=dev, generator=gen, dtype=dtype) * sigma for s in shapes)


def prepare(case, seed):
    x = _inputs(case, seed)
    state = {"case": case, "in": x}
    if case["op"] == "spec":
        q, k, v = x
        state["spec"] = _TUNERS[case["variant"]](
            tuple(q.shape), tuple(k.shape), tuple(v.shape), q.element_size(), causal=case["causal"],
            return_lse=case["lse"]).build_flash_attention_launch_spec(q, k, v)
    elif case["op"] == "kernel":
        M, N, K = case["M"], case["N"], case["K"]
        bm, bn, bk, group_m, waves, stages = mma._select_2d_contiguous_config(M, N, K)
        state["c"] = torch.empty(M, N, device=x[0].device, dtype=torch.float16)
        state["grid"] = (-(-M // bm) * -(-N // bn),)
        state["meta"] = {"BLOCK_M": bm, "BLOCK_N": bn, "BLOCK_K": bk, "GROUP_M": group_m, "num_warps": waves,
                         "num_stages": stages,
                         "USE_CACHE_EVICTION_HINTS": mma._supports_contiguous_cache_eviction_hints(x[0].device)}
    return state


def run(state):
    case, x = state["case"], state["in"]
    op = case["op"]
    if op == "spec":
        out = flash_atten.flash_attention(state["spec"])
        if case["variant"] == "sliced" and case["lse"]:  # that layout returns only o; the lse is a keyword argument
            return out, state["spec"].kernel_kwargs["lse"]
        return out
    if op == "attention":
        return flash_atten.attention(*x, causal=case["causal"], return_lse=case["lse"], variant=case["variant"])
    if op == "sdpa":
        return flash_atten.sdpa(*x, is_causal=case["causal"], variant=case["variant"])
    if op == "matmul":
        return mma.matmul(*x)
    mma._matmul_contiguous_kernel[state["grid"]](*x, state["c"], case["M"], case["N"], case["K"], **state["meta"])
    return state["c"]


def work(case):
    if case["op"] in ("kernel", "matmul"):
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 2 * (M * K + K * N + M * N), "flops": 2 * M * N * K}
    B, H, H_kv, M, N, D = (case[x] for x in ("B", "H", "H_kv", "M", "N", "D"))
    pairs = N * (N + 1) // 2 if case["causal"] else M * N  # causal cases have M == N
    return {"bytes": 2 * (2 * B * H * M * D + 2 * B * H_kv * N * D) + (4 * B * H * M if case["lse"] else 0),
            "flops": 4 * B * H * pairs * D}


def tolerance(case):
    # Four times the distance from the 64-bit result that was measured. Attention: P and O are rounded to the
    # input type. GEMM: fp32 sums, one rounding to binary16 (2.1e-4 relative in the 2-norm).
    if case["op"] in ("kernel", "matmul"):
        return {"rel": 1e-3}
    return {"rel": 1.2e-3} if case["dtype"] == "f16" else {"rel": 1e-2}


def exact(case, seed):
    x = [t.double() for t in _inputs(case, seed)]
    if case["op"] in ("kernel", "matmul"):
        return x[0] @ x[1]
    q, k, v = x
    B, H, M, D = q.shape
    H_kv, N = k.shape[1], k.shape[2]
    out = torch.empty(B, H, M, D, device=q.device, dtype=torch.float64)
    lse = torch.empty(B, H, M, device=q.device, dtype=torch.float64)
    rows = 4096
    col = torch.arange(N, device=q.device)
    for b in range(B):
        for h in range(H):
            kt, vh = k[b, h // (H // H_kv)].t().contiguous(), v[b, h // (H // H_kv)].contiguous()
            for r in range(0, M, rows):
                s = (q[b, h, r:r + rows].contiguous() @ kt).mul_(D ** -0.5)
                if case["causal"]:
                    s.masked_fill_(col[None, :] > torch.arange(r, r + s.shape[0], device=q.device)[:, None], -math.inf)
                top = s.amax(dim=1, keepdim=True)
                s.sub_(top).exp_()
                total = s.sum(dim=1, keepdim=True)
                out[b, h, r:r + rows] = (s @ vh) / total
                lse[b, h, r:r + rows] = (top + total.log())[:, 0]
    return (out, lse) if case["lse"] else out
