"""A call whose form (shapes, strides, types, flags) was seen before is launched from a kept argument
block: with other tensors, other scales, flags and strides in between, every call has to give what the
C ABI gives for its own arguments, bit for bit."""
from __future__ import annotations

import pytest
import torch

import flash_atten
import hip_lib
import oracle
import tuner
from helpers import ATOL, make_qkv, max_abs, to_device

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16


def _direct(q, k, v, causal, scale, tile, variant, lse=False, splits=1):
    o = torch.empty_like(q)
    x = torch.empty(q.shape[:3], dtype=torch.float32, device=q.device) if lse else None
    need = hip_lib.workspace_bytes(*q.shape, splits)
    ws = torch.empty(need, dtype=torch.uint8, device=q.device) if need else None
    hip_lib.fa_fwd(q, k, v, o, x, sm_scale=scale, causal=causal, variant=variant, tile=hip_lib.make_tile(*tile, splits),
                   workspace=ws)
    return o, x


def _qkv(seed, B, H, Hk, M, N, D, dtype):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(s, device="cuda", generator=g).to(dtype) for s in ((B, H, M, D), (B, Hk, N, D), (B, Hk, N, D))]


@pytest.mark.parametrize("variant", ["basic", "optimized", "sliced"])
def test_repeated_forms_with_other_values(gpu, variant):
    code = {"basic": 0, "optimized": 1, "sliced": 2}[variant]
    forms = [(1, 4, 4, 96, 160, 64, torch.float16, False, None), (1, 4, 2, 96, 160, 64, torch.float16, True, 0.3),
             (1, 4, 2, 96, 160, 64, torch.float16, False, 0.3), (2, 4, 4, 96, 96, 128, torch.bfloat16, True, None),
             (1, 8, 2, 1, 2000, 128, torch.bfloat16, False, None)]
    for seed in (1, 2, 3):
        for B, H, Hk, M, N, D, dtype, causal, scale in forms:
            q, k, v = _qkv(seed, B, H, Hk, M, N, D, dtype)
            print(f"[plans] {variant} seed={seed} {B},{H},{Hk},{M},{N},{D} causal={causal}", flush=True)
            spec = {"basic": tuner.FlashAttentionTuner, "optimized": tuner.FlashAttentionOptimizeSharedMemTuner,
                    "sliced": tuner.FlashAttentionBlockDNomaskTuner}[variant](
                tuple(q.shape), tuple(k.shape), tuple(v.shape), 2, causal=causal,
                return_lse=True).build_flash_attention_launch_spec(q, k, v, sm_scale=scale)
            kw = spec.kernel_kwargs
            tile = (kw["BLOCK_M"], kw["BLOCK_N"], kw["num_warps"], kw["num_stages"])
            o_ref, lse_ref = _direct(q, k, v, causal, D ** -0.5 if scale is None else scale, tile, code, True,
                                     kw.get("SPLITS", 1))
            o, lse = flash_atten.attention(q, k, v, causal=causal, sm_scale=scale, return_lse=True, variant=variant)
            assert torch.equal(o, o_ref) and torch.equal(lse, lse_ref)
            assert torch.equal(flash_atten.attention(q, k, v, causal=causal, sm_scale=scale, variant=variant), o_ref)
            out = flash_atten.flash_attention(spec)
            assert torch.equal(out[0] if isinstance(out, tuple) else out, o_ref)
            spec.update_data((q, v, k))  # other tensors of the same form
            flash_atten.flash_attention(spec)
            swapped, _ = _direct(q, v, k, causal, D ** -0.5 if scale is None else scale, tile, code, False,
                                 kw.get("SPLITS", 1))
            assert torch.equal(spec.kernel_args[3], swapped)
            for layout in (lambda t: t, lambda t: t.transpose(1, 2).contiguous().transpose(1, 2)):
                got = flash_atten.sdpa(layout(q), layout(k), layout(v), is_causal=causal, scale=scale, variant=variant)
                assert torch.equal(got, o_ref)
                assert got.stride() == torch.empty(B, M, H, D).transpose(1, 2).stride()


def test_strides_that_are_not_the_tensors_own(gpu):
    """The strided layout takes its strides from the arguments: a launch that gives others than the
    tensor's must not meet the plan of the tensor's own."""
    q, k, v = _qkv(9, 1, 2, 2, 64, 64, 64, torch.float16)
    spec = tuner.FlashAttentionOptimizeSharedMemTuner(tuple(q.shape), tuple(k.shape), tuple(v.shape), 2, causal=False,
                                                      return_lse=False).build_flash_attention_launch_spec(q, k, v)
    kernel = flash_atten.flash_attention_kernel_mapping[spec.function_name]
    flash_atten.flash_attention(spec)
    plain = spec.kernel_args[3].clone()
    args = list(spec.kernel_args)
    args[10] = 0  # both heads read kv head 0
    args[14] = 0
    kernel[spec.grid](*args, **spec.kernel_kwargs)
    shared = spec.kernel_args[3].clone()
    want = flash_atten.attention(q, k[:, :1].expand(1, 2, 64, 64), v[:, :1].expand(1, 2, 64, 64))
    assert torch.equal(shared, want) and not torch.equal(shared, plain)
    args[10] = 1 << 40  # beyond the storage: refused, as before
    with pytest.raises(RuntimeError):
        kernel[spec.grid](*args, **spec.kernel_kwargs)


@pytest.mark.parametrize("case", [
    (1, 2, 2, 128, 700, 128, BF16, False), (1, 4, 2, 200, 2500, 64, F16, False), (2, 2, 1, 333, 333, 128, BF16, True),
    (1, 1, 1, 1500, 1283, 128, F16, True), (1, 4, 4, 300, 1100, 256, BF16, False), (1, 1, 1, 129, 40000, 64, BF16, False),
], ids=lambda c: "x".join(map(str, c[:6])) + f"_c{int(c[7])}")
def test_prefill_splits_against_the_oracle(gpu, case):
    """Sliced prefill shapes whose keys are split over the grid, contiguous and from [B, S, H, D] storage."""
    B, H, Hkv, M, N, D, dtype, causal = case
    print(f"[launch_plans] prefill splits {case}", flush=True)
    q, k, v = make_qkv(4100 + M + N, B, H, Hkv, M, N, D, dtype)
    o_ref, lse_ref = oracle.attention(q, k, v, causal=causal)
    qd, kd, vd = (to_device(x, dtype, "cuda:0") for x in (q, k, v))
    o, lse = flash_atten.attention(qd, kd, vd, causal=causal, return_lse=True, variant="sliced")
    assert max_abs(o.float().cpu().numpy(), o_ref) <= ATOL[dtype]
    assert max_abs(lse.cpu().numpy(), lse_ref) <= 1e-3
    qt, kt, vt = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (qd, kd, vd))
    o = flash_atten.sdpa(qt, kt, vt, is_causal=causal, variant="sliced")
    assert max_abs(o.float().cpu().numpy(), o_ref) <= ATOL[dtype]
