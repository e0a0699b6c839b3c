"""Host logic of the drop-in surface (no GPU): tune-argument validation, tuner validation, launch
layouts, config selection, resource errors, and the resource report. Restates the reference's
rules (tuner.py:72-157, 252-339, 563-590, 597-734; mma.py:63-81; exceptions.py:633-757)."""
from __future__ import annotations

import functools
import itertools

import pytest
import torch

import exceptions
import flash_atten
import gfx950_configs as cfgs
import hip_lib
import mma
import tuner
from tuner import (
    FlashAttenTuneArguments,
    FlashAttentionBlockDNomaskTuner,
    FlashAttentionOptimizeSharedMemTuner,
    FlashAttentionTuner,
)

# ---- FlashAttenTuneArguments (tuner.py:82-108) ----------------------------------------------------


@pytest.mark.parametrize(
    "kwargs,message",
    [
        ({"BLOCK_N": 0}, "BLOCK_N must be positive when provided"),
        ({"BLOCK_M": -4}, "BLOCK_M must be positive when provided"),
        ({"BLOCK_M": 96}, "BLOCK_M must be a power of 2 when provided"),
        ({"BLOCK_N_PAD": 0}, "BLOCK_N_PAD must be positive when provided"),
        ({"BLOCK_N_PAD": 48}, "BLOCK_N_PAD must be a power of 2 when provided"),
        ({"BLOCK_DMODEL": 0}, "BLOCK_DMODEL must be positive when provided"),
        ({"BLOCK_DMODEL": 80}, "BLOCK_DMODEL must be a power of 2 when provided"),
        ({"BLOCK_DMODEL_OUTER": -1}, "BLOCK_DMODEL_OUTER must be positive when provided"),
        ({"BLOCK_DMODEL_OUTER": 24}, "BLOCK_DMODEL_OUTER must be a power of 2 when provided"),
        ({"NUM_WARPS": 0}, "NUM_WARPS must be positive when provided"),
        ({"NUM_STAGES": 0}, "NUM_STAGES must be positive when provided"),
    ],
)
def test_tune_argument_validation(kwargs, message):
    with pytest.raises(ValueError, match=message):
        FlashAttenTuneArguments(**kwargs)


def test_tune_arguments_accept_non_power_of_two_block_n():
    assert FlashAttenTuneArguments(BLOCK_N=48).BLOCK_N == 48  # only BLOCK_N skips the power-of-2 rule


# ---- tuner constructor (tuner.py:132-157) ----------------------------------------------------------

Q = (1, 4, 256, 64)


@pytest.mark.parametrize(
    "shapes,tune,message",
    [
        (((1, 4, 256), Q, Q), None, "must all be 4D"),
        ((Q, (2, 4, 256, 64), Q), None, "Batch and head dimensions must match"),
        ((Q, (1, 3, 256, 64), (1, 3, 256, 64)), None, "Batch and head dimensions must match"),
        ((Q, (1, 2, 256, 64), (1, 4, 256, 64)), None, "Batch and head dimensions must match"),
        ((Q, (1, 4, 256, 32), Q), None, "Last dimension must match"),
        ((Q, (1, 4, 128, 64), Q), None, "sequence lengths must match"),
        ((Q, Q, Q), FlashAttenTuneArguments(BLOCK_DMODEL=32), "BLOCK_DMODEL must be >= D"),
        ((Q, Q, Q), FlashAttenTuneArguments(BLOCK_N=128, BLOCK_N_PAD=64), "BLOCK_N cannot exceed BLOCK_N_PAD"),
        ((Q, Q, Q), FlashAttenTuneArguments(NUM_WARPS=64), "NUM_WARPS must be <= 16"),
    ],
)
def test_tuner_validation(shapes, tune, message):
    with pytest.raises(ValueError, match=message):
        FlashAttentionTuner(*shapes, 2, causal=False, return_lse=False, tune_args=tune)


def test_gqa_shapes_accepted_and_sliced_allows_small_block_dmodel():
    FlashAttentionTuner(Q, (1, 2, 300, 64), (1, 2, 300, 64), 2, causal=True, return_lse=True)
    FlashAttentionBlockDNomaskTuner(Q, Q, Q, 2, causal=False, return_lse=False,
                                    tune_args=FlashAttenTuneArguments(BLOCK_DMODEL=32))


# ---- launch layouts (tuner.py:264-305, 639-658) ------------------------------------------------------


def _cpu_qkv(B=1, H=4, M=256, N=256, D=64, Hkv=None, dtype=torch.float16):
    Hkv = H if Hkv is None else Hkv
    return (torch.zeros(B, H, M, D, dtype=dtype), torch.zeros(B, Hkv, N, D, dtype=dtype),
            torch.zeros(B, Hkv, N, D, dtype=dtype))


@pytest.mark.parametrize("cls", [FlashAttentionTuner, FlashAttentionOptimizeSharedMemTuner])
@pytest.mark.parametrize("return_lse", [False, True])
def test_strided_launch_layout(cls, return_lse):
    q, k, v = _cpu_qkv()
    spec = cls(tuple(q.shape), tuple(k.shape), tuple(v.shape), 2, causal=True, return_lse=return_lse
               ).build_flash_attention_launch_spec(q, k, v)
    assert spec.function_name == cls.KERNEL_NAME
    assert len(spec.kernel_args) == 29
    assert spec.kernel_args[24:28] == (4, 256, 256, 64)
    assert spec.kernel_args[28] == pytest.approx(64 ** -0.5)
    assert spec.kernel_args[5:9] == q.stride()
    assert isinstance(spec.kernel_args[4], torch.Tensor) == return_lse
    assert set(spec.kernel_kwargs) == {"causal", "HAS_LSE", "BLOCK_M", "BLOCK_N", "BLOCK_N_PAD", "BLOCK_DMODEL",
                                       "num_warps", "num_stages"}
    assert spec.kernel_kwargs["causal"] is True and spec.kernel_kwargs["HAS_LSE"] is return_lse
    assert spec.grid == (-(-256 // spec.kernel_kwargs["BLOCK_M"]), 4)
    assert spec.tune_args.BLOCK_M == spec.kernel_kwargs["BLOCK_M"]
    assert spec.input_shapes["q"] == (1, 4, 256, 64)
    assert spec.input_shapes["lse"] == ((1, 4, 256) if return_lse else None)
    ctx = spec.launch_context
    assert ctx["compiled_shared_memory_bytes_per_block"] <= ctx["available_shared_memory_bytes_per_sm"]


def test_sliced_launch_layout_and_update_data():
    q, k, v = _cpu_qkv(M=128, N=512, D=128, Hkv=2)
    spec = FlashAttentionBlockDNomaskTuner(tuple(q.shape), tuple(k.shape), tuple(v.shape), 2, causal=False,
                                           return_lse=False).build_flash_attention_launch_spec(q, k, v, sm_scale=0.5)
    assert len(spec.kernel_args) == 9
    assert spec.kernel_args[4:] == (4, 128, 512, 128, 0.5)
    assert {"BLOCK_M", "BLOCK_N", "BLOCK_DMODEL", "BLOCK_DMODEL_OUTER", "num_warps", "num_stages"} <= set(
        spec.kernel_kwargs)
    o = spec.kernel_args[3]
    q2, k2, v2 = _cpu_qkv(M=128, N=512, D=128, Hkv=2)
    spec.update_data((q2, k2, v2))
    assert spec.kernel_args[0] is q2 and spec.kernel_args[3] is o  # o reused (tuner.py:56-69)
    assert spec.launch_context["kv_splits"] == spec.kernel_kwargs["SPLITS"]


def test_config_cache_is_per_class_and_reused():
    q, k, v = _cpu_qkv()
    a = FlashAttentionTuner(tuple(q.shape), tuple(k.shape), tuple(v.shape), 2, causal=False, return_lse=False)
    spec1 = a.build_flash_attention_launch_spec(q, k, v)
    spec2 = a.build_flash_attention_launch_spec(q, k, v)
    assert spec1.kernel_kwargs == spec2.kernel_kwargs
    b = FlashAttentionOptimizeSharedMemTuner(tuple(q.shape), tuple(k.shape), tuple(v.shape), 2, causal=False,
                                             return_lse=False)
    assert b._cache_key(q) != a._cache_key(q)


def test_tune_args_are_hints_with_recorded_relaxation():
    q, k, v = _cpu_qkv(D=128)
    ta = FlashAttenTuneArguments(BLOCK_N=64, BLOCK_M=128, BLOCK_N_PAD=64, BLOCK_DMODEL=128, NUM_WARPS=8,
                                 NUM_STAGES=1)
    spec = FlashAttentionTuner(tuple(q.shape), tuple(k.shape), tuple(v.shape), 2, causal=False, return_lse=False,
                               tune_args=ta).build_flash_attention_launch_spec(q, k, v)
    assert spec.kernel_kwargs["BLOCK_M"] == 128 and spec.kernel_kwargs["BLOCK_N"] == 64
    assert spec.kernel_kwargs["num_stages"] == 1
    assert "NUM_WARPS" in spec.launch_context.get("tune_args_relaxed", "")


def test_unknown_kernel_name_raises_name_error():
    q, k, v = _cpu_qkv()
    spec = FlashAttentionTuner(tuple(q.shape), tuple(k.shape), tuple(v.shape), 2, causal=False,
                               return_lse=False).build_flash_attention_launch_spec(q, k, v)
    bad = tuner.FlashAttentionLaunchSpec(grid=spec.grid, kernel_args=spec.kernel_args,
                                         kernel_kwargs=spec.kernel_kwargs, launch_context={},
                                         function_name="_no_such_kernel", tune_args=spec.tune_args,
                                         input_shapes=spec.input_shapes)
    with pytest.raises(NameError, match="No such kernel named _no_such_kernel"):
        flash_atten.flash_attention(bad)


def test_unsupported_head_dim_and_dtype():
    q, k, v = _cpu_qkv(D=96)
    with pytest.raises(ValueError, match="not built"):
        FlashAttentionTuner(tuple(q.shape), tuple(k.shape), tuple(v.shape), 2, causal=False,
                            return_lse=False).build_flash_attention_launch_spec(q, k, v)
    q, k, v = _cpu_qkv(dtype=torch.float32)
    with pytest.raises(ValueError, match="dtype"):
        FlashAttentionTuner(tuple(q.shape), tuple(k.shape), tuple(v.shape), 4, causal=False,
                            return_lse=False).build_flash_attention_launch_spec(q, k, v)


# ---- resource errors are host-forcible (exceptions.py:695-757, tuner.py:519-554) -------------------------


def _fake_limits(lds):
    def provider():
        lim = exceptions.gfx950_static_limits()
        lim["available_shared_memory_bytes_per_sm"] = lds
        return lim

    return provider


def test_out_of_resources_with_detail_when_lds_too_small():
    exceptions.set_device_limits_provider(_fake_limits(1024))
    FlashAttentionTuner._config_cache.clear()  # the class cache is keyed on shapes, not limits
    try:
        q, k, v = _cpu_qkv()
        with pytest.raises(exceptions.OutOfResourcesWithDetail) as info:
            FlashAttentionTuner(tuple(q.shape), tuple(k.shape), tuple(v.shape), 2, causal=False,
                                return_lse=False).build_flash_attention_launch_spec(q, k, v)
        err = info.value
        assert err.name == "shared memory" and err.limit == 1024 and err.required > 1024
        assert err.kernel_name == "_flash_attn_fwd_kernel_basic"
        text = str(err)
        assert "Kernel: _flash_attn_fwd_kernel_basic." in text and "LDS" in text
    finally:
        exceptions.set_device_limits_provider(None)
        FlashAttentionTuner._config_cache.clear()


def test_out_of_resources_registers_when_register_file_too_small():
    def provider():
        lim = exceptions.gfx950_static_limits()
        lim["vgprs_per_simd_lane"] = 64
        return lim

    exceptions.set_device_limits_provider(provider)
    FlashAttentionTuner._config_cache.clear()
    try:
        q, k, v = _cpu_qkv()
        with pytest.raises(exceptions.OutOfResourcesWithDetail) as info:
            FlashAttentionOptimizeSharedMemTuner(tuple(q.shape), tuple(k.shape), tuple(v.shape), 2, causal=False,
                                                 return_lse=False).build_flash_attention_launch_spec(q, k, v)
        assert info.value.name == "registers"
    finally:
        exceptions.set_device_limits_provider(None)
        FlashAttentionTuner._config_cache.clear()


def test_out_of_resources_from_base_and_pickle():
    import pickle

    base = exceptions.OutOfResources(10, 5, "shared memory")
    detail = exceptions.OutOfResourcesWithDetail.from_out_of_resources(base, kernel_name="k",
                                                                       launch_context={"a": 1})
    assert detail.original_exception is base and detail.launch_context == {"a": 1}
    assert pickle.loads(pickle.dumps(base)).required == 10


def test_resource_usage_summary_format():
    ctx = {"compiled_shared_memory_bytes_per_block": 100, "available_shared_memory_bytes_per_sm": 200,
           "attempted_register_file_size_bytes_per_block": 3, "available_register_file_size_bytes_per_sm": 4,
           "attempted_registers_per_block": 5, "available_registers_per_sm": 6}
    text = exceptions._resource_usage_summary("kern", ctx, tune_args=FlashAttenTuneArguments(BLOCK_M=64),
                                               input_shapes={"q": (1, 2), "lse": None})
    assert text.startswith("kern tuner resources: \nshared=100/200 bytes per block/SM, ")
    assert "register_file=3/4" in text and "registers=5/6" in text
    assert "tune_args=BLOCK_M=64" in text and "input_shapes=q=(1, 2)" in text
    assert exceptions._format_tune_args(None) is None and exceptions._format_input_shapes({"x": None}) is None


# ---- GEMM config selection (mma.py:63-81) ----------------------------------------------------------


def _reference_accepts(m, n, k):
    if k % 32:
        return False
    return (m % 128 == 0 and n % 64 == 0) or (m % 64 == 0 and n % 256 == 0)


def test_gemm_selector_accepts_exactly_the_reference_shapes():
    sizes = [64, 96, 128, 192, 256, 320, 512, 768, 1024]
    for m, n, k in itertools.product(sizes, sizes, [32, 48, 64, 256]):
        if _reference_accepts(m, n, k):
            bm, bn, bk, group_m, warps, stages = mma._select_2d_contiguous_config(m, n, k)
            assert m % bm == 0 and n % bn == 0 and k % bk == 0 and group_m >= 1 and stages == 2
        else:
            with pytest.raises(ValueError):
                mma._select_2d_contiguous_config(m, n, k)


def test_gemm_selector_prefers_large_tiles_and_hints():
    assert mma._select_2d_contiguous_config(8192, 8192, 8192)[:3] in [(256, 256, 64), (256, 256, 32),
                                                                     (256, 128, 64), (128, 256, 64)]
    assert cfgs.choose_gemm_tile(1024, 1024, 256, hint=(128, 128, 64))[:3] == (128, 128, 64)
    # block sizes + wave count narrow the candidates; a wave count that is not built keeps the sizes
    assert cfgs.choose_gemm_tile(8192, 8192, 8192, hint=(256, 256, 64, 4))[:4] == (256, 256, 64, 4)
    assert cfgs.choose_gemm_tile(8192, 8192, 8192, hint=(256, 256, 64, 8))[:4] == (256, 256, 64, 8)
    assert cfgs.choose_gemm_tile(8192, 8192, 8192, hint=(256, 256, 64, 2))[:3] == (256, 256, 64)


def test_gemm_launch_hints_keep_the_tuned_tile():
    """BLOCK_* hints equal to the tuned tile's sizes (what _select_2d_contiguous_config returns and
    test_mma.py passes back) must launch the tuned tile, wave count included."""
    bm, bn, bk, group_m, warps, _ = mma._select_2d_contiguous_config(8192, 8192, 8192)
    assert cfgs.choose_gemm_tile(8192, 8192, 8192, hint=(bm, bn, bk))[:4] == (bm, bn, bk, warps)
    assert cfgs.choose_gemm_tile(8192, 8192, 8192, hint=(bm, bn, bk, warps))[:4] == (bm, bn, bk, warps)


@pytest.mark.parametrize("M,N,K,tiles", [
    # a large C of a short K: its write is the time, the 256x256 tiles' smaller grid makes it longer
    (7808, 7104, 64, [(128, 64, 32, 4)]), (6912, 2624, 192, [(128, 64, 32, 4)]), (7168, 4032, 96, [(128, 64, 32, 4)]),
    (4096, 576, 2976, [(128, 64, 32, 4)]),
])
def test_gemm_model_keeps_small_tiles_for_large_c(M, N, K, tiles):
    tile = cfgs.choose_gemm_tile(M, N, K)[:4]
    assert tile in tiles and cfgs.choose_gemm_splits(M, N, K, tile) == (tile, 1)


def test_gemm_choice_takes_empty_products():
    """K = 0 reaches the launch, which refuses it; M = 0 and N = 0 are launches of nothing."""
    for M, N, K in ((128, 64, 0), (64, 64, 0), (1, 4, 0), (0, 64, 64), (64, 0, 64)):
        tile = cfgs.choose_gemm_tile_any(M, N, K)
        assert cfgs.choose_gemm_splits(M, N, K, tile[:4]) == (tile[:4], 1)
    assert cfgs.choose_gemm_tile(128, 64, 0)[:4] in cfgs.gemm_candidates()


def test_cache_eviction_hint_false_without_gpu():
    assert mma._supports_contiguous_cache_eviction_hints() is torch.cuda.is_available()


# ---- gfx950 selection helpers ---------------------------------------------------------------------------


def test_filter_by_hints_relaxes_minimally():
    cands = [cfgs.FaTileChoice(128, 64, 4, 1), cfgs.FaTileChoice(256, 64, 8, 1)]
    got, relaxed = cfgs.filter_by_hints(cands, {"BLOCK_M": 128, "NUM_WARPS": 8, "NUM_STAGES": 1})
    assert relaxed == ["NUM_WARPS"] and got == [cands[0]]
    got, relaxed = cfgs.filter_by_hints(cands, {"BLOCK_M": 256, "NUM_WARPS": 8})
    assert relaxed == [] and got == [cands[1]]
    got, relaxed = cfgs.filter_by_hints(cands, {"BLOCK_M": 512})
    assert relaxed == ["BLOCK_M"] and got == cands


def test_choose_splits():
    assert cfgs.choose_splits(4, 32, 8192, 8192, 256, 64) == 1  # grid already fills the GPU
    # prefill-shaped grids (full query tiles) split only below a quarter of the CUs
    assert cfgs.choose_splits(1, 12, 4096, 4096, 256, 64) == 1  # 192 workgroups
    assert cfgs.choose_splits(1, 28, 1024, 1024, 128, 64) == 1  # 224 workgroups
    assert cfgs.choose_splits(1, 2, 256, 65536, 256, 64) == cfgs.PREFILL_SPLIT_CUS // 2
    s = cfgs.choose_splits(1, 4, 512, 8192, 128, 64)              # 16 workgroups
    assert s == cfgs.PREFILL_SPLIT_CUS // 16
    # decode-shaped grids (a few rows per tile) split up to the resident capacity
    assert cfgs.choose_splits(1, 1, 1, 100000, 256, 64) == cfgs.MAX_SPLITS
    assert cfgs.choose_splits(8, 32, 1, 32768, 128, 64) == 2  # 256 single-row tiles, 2 per CU
    assert cfgs.choose_splits(1, 1, 64, 128, 256, 64) == 1  # too few KV tiles to split


def test_prefill_splits():
    """Prefill-shaped grids: one workgroup per CU at most, only where the serial steps saved outweigh the
    partials; a causal block's steps end at its diagonal, so short-M causal launches stay whole."""
    for B, H, M, N, block_m, causal in itertools.product((1, 3), (1, 5, 16), (128, 777, 4096), (64, 300, 2048, 40000),
                                                         (128, 256), (False, True)):
        base = B * H * -(-M // block_m)
        s = cfgs.prefill_splits(base, M, N, block_m, 64, causal)
        assert 1 <= s <= max(1, -(-N // 64) // 2) and (s == 1 or s * base <= cfgs.NUM_CUS)
        assert (s - 1) * -(-(-(-N // 64)) // s) < -(-N // 64) or N == 0  # the last split has keys
    assert cfgs.prefill_splits(32, 1024, 8192, 128, 64, False) == 8
    assert cfgs.prefill_splits(32, 1024, 8192, 128, 64, True) == 1
    assert cfgs.prefill_splits(128, 2048, 2048, 128, 64, True) == 1
    assert cfgs.prefill_splits(128, 16384, 16384, 128, 64, True) == 2
    assert cfgs.prefill_splits(18, 288, 572, 128, 32, False, 256) > 1  # D = 256: a step takes longer
    assert cfgs.choose_splits(1, 1, 328, 328, 256, 64, causal=True, D=64) == 1  # as its 128-row blocks


def test_prefill_tiles_of_sliced_shapes_between_the_buckets():
    """Sliced prefill shapes take no tile of a decode bucket; short splits take the four-wave tile."""
    def tile(dtype, D, causal, B, H, M, N):
        t = cfgs.choose_fa_tile(hip_lib.FA_VARIANT_SLICED, dtype, D, causal, B, H, M, N,
                                cfgs.fa_candidates(hip_lib.FA_VARIANT_SLICED, dtype, D))
        return t.block_m, t.block_n, t.waves, t.stages
    for dtype in (torch.float16, torch.bfloat16):
        assert tile(dtype, 128, False, 1, 32, 3000, 3000)[3] in (8, 9)
        assert tile(dtype, 128, False, 1, 4, 1024, 8192) == cfgs.KEY_GROUP_TILE
        assert tile(dtype, 128, False, 1, 2, 128, 700) == cfgs.SPLIT_TILE
    assert tile(torch.bfloat16, 128, False, 1, 32, 1, 8192)[2] == 4  # decode keeps its buckets' tiles


@pytest.mark.parametrize("D,causal,BH,M,N,stages", [
    (64, False, 8, 10814, 11518, (10, 6)),    # 344 blocks: a second round of 88 on 256 CUs
    (128, True, 51, 4000, 4000, (8,)),     # 16 blocks a head: the fixed sequences stack heavy ones
    (128, True, 20, 5000, 5000, (10,)),
    (128, False, 14, 8000, 8000, (8, 9)),  # 448 blocks, nearly two whole rounds
    (64, True, 1, 65793, 65793, (10,)),    # 258 blocks of 256 rows, not dealt by XCD: half the serial steps
])
def test_full_grid_tiles_follow_the_schedule(D, causal, BH, M, N, stages):
    for best in [t for t, us in cfgs.GRID_STEP_US.items() if (D, causal) in us]:
        assert cfgs.choose_full_grid_tile(True, D, causal, BH, M, N, best)[3] in stages


def test_full_grid_tiles_keep_the_bucket_beyond_the_model():
    best = cfgs.PERSISTENT_TILE
    assert cfgs.choose_full_grid_tile(True, 96, False, 64, 4096, 4096, best) == best
    assert cfgs.choose_full_grid_tile(True, 128, True, 4096, 4096, 4096, best) == best  # too many blocks
    assert cfgs.choose_full_grid_tile(True, 128, True, 1, 1 << 21, 4096, best) == best  # one head alone has too many
    # no keys: the kernel whose launch and blocks cost least
    assert cfgs.choose_full_grid_tile(True, 128, False, 300, 200, 0, best) == (128, 64, 4, 6)


def _reference_steps(rows, per_step, order, block_steps, BH, M, N, causal):
    """fa_grid_steps of one block to a CU, block by block: the persistent kernel's rounds as its item order
    deals them, else the CUs of each XCD's four engines, served in turn and in order."""
    nb = -(-M // rows)
    total = nb * BH

    def cost(mb):
        keys = min(N, (mb + 1) * rows) if causal else N
        half = 0.7 if M - mb * rows <= rows // 2 else 1.0
        return block_steps * half + -(-(-(-keys // 64)) // per_step)

    def block(pid):
        return nb - 1 - pid % nb if causal else pid % nb

    if order == hip_lib.GRID_PERSISTENT:
        G = min(total, 256)
        by_xcd = total % 8 == 0 and G % 8 == 0
        S, per = (G // 8, total // 8) if by_xcd else (G, total)
        end = 0.0
        for w in range(G):
            x, slot = (w & 7, w >> 3) if by_xcd else (0, w)
            ks = (r * S + (S - 1 - slot if r & 1 else slot) for r in range(-(-per // S)))
            end = max(end, sum(cost(block(x * per + k)) for k in ks if k < per))
        return end
    end = 0.0
    for x in range(8):
        free = [[0.0] * 8 for _ in range(4)]
        start = 0.0
        for i, wg in enumerate(range(x, total, 8)):
            if order == hip_lib.GRID_HEAVIEST_FIRST and causal:
                mb = nb - 1 - wg // BH
            else:
                mb = block(wg % 8 * (total // 8) + wg // 8 if total % 8 == 0 else wg)
            engine = free[i % 4]
            cu = engine.index(min(engine))
            start = max(start, engine[cu])
            engine[cu] = start + cost(mb)
            end = max(end, engine[cu])
    return end


@pytest.mark.parametrize("BH,M,N", [(1, 300, 300), (3, 100, 900), (8, 2048, 2048), (66, 4200, 4200), (51, 4000, 4000),
                                    (43, 1500, 777), (2, 3103, 3103), (144, 961, 961), (64, 2048, 4096)])
@pytest.mark.parametrize("causal", [False, True])
def test_grid_steps_against_a_block_by_block_reference(BH, M, N, causal):
    """One block, less than a round, whole rounds, counts that are no multiple of the XCDs, blocks per head
    that divide the engines' turn, a reversed second round."""
    for rows, per_step, order in ((256, 1, hip_lib.GRID_HEAD_MAJOR), (256, 1, hip_lib.GRID_PERSISTENT),
                                  (128, 2, hip_lib.GRID_HEAVIEST_FIRST)):
        got = hip_lib.grid_steps(rows, per_step, order, 1, 2.5, 1.0, BH, M, N, causal)
        assert got == pytest.approx(_reference_steps(rows, per_step, order, 2.5, BH, M, N, causal), rel=1e-12)


def test_grid_steps_of_shared_cus_and_refusals():
    steps = functools.partial(hip_lib.grid_steps, 128, 1, hip_lib.GRID_HEAD_MAJOR)
    alone = steps(2, 3.0, 0.6, 16, 2048, 1024, False)  # 256 blocks, one to a CU
    assert 0.6 * 19 * 0.95 <= alone <= 0.6 * 19 * 1.05
    shared = steps(2, 3.0, 0.6, 32, 2048, 1024, False)  # 512, two to a CU
    assert 19 * 0.95 <= shared <= 19 * 1.05
    assert shared + alone * 0.9 < steps(2, 3.0, 0.6, 48, 2048, 1024, False) <= 2 * shared  # half a round more
    assert steps(4, 3.0, 0.6, 64, 2048, 1024, False) > shared  # three and four to a CU are slower each
    for bad in ((0, 3.0, 0.6, 1, 64, 64, False), (5, 3.0, 0.6, 1, 64, 64, False), (1, 3.0, 0.6, 0, 64, 64, False),
                (1, 3.0, 0.6, 1, 0, 64, False), (1, 3.0, 0.6, 1, 64, -1, False), (1, 3.0, 0.6, 4097, 128, 64, False)):
        assert steps(*bad) == -1


@pytest.mark.parametrize("variant,dtype,D,causal,BH,M,tiles", [
    # inside a swept bucket, off its corner: the persistent kernel stacks heavy blocks
    (1, torch.float16, 128, True, 66, 4200, [(256, 64, 8, 8)]), (1, torch.float16, 128, True, 113, 4000, [(256, 64, 8, 8)]),
    (1, torch.float16, 128, True, 120, 2100, [(256, 64, 8, 8)]), (1, torch.bfloat16, 128, True, 15, 9000, [(128, 64, 8, 10)]),
    (1, torch.float16, 128, True, 128, 4096, [(256, 64, 8, 9)]),  # the corner keeps its timing
    # many heads of few rows: a second round of key-group blocks costs more than 256-row ones
    (1, torch.bfloat16, 64, True, 100, 268, [(256, 64, 8, 8), (128, 64, 4, 6)]),
    (1, torch.float16, 128, True, 116, 304, [(256, 64, 8, 8)]), (2, torch.bfloat16, 128, False, 96, 157, [(256, 64, 8, 8), (128, 64, 4, 6)]),
    # basic: 128 rows where 256 leave CUs idle, the dispatched body where the sequences stack
    (0, torch.float16, 128, False, 4, 1024, [(128, 64, 4, 1)]), (0, torch.bfloat16, 128, True, 37, 4273, [(256, 64, 8, 8)]),
    (0, torch.float16, 128, True, 128, 2048, [(256, 64, 8, 1)]),
], ids=lambda v: "x".join(map(str, v[0])) if isinstance(v, list) else str(v).replace("torch.", ""))
def test_tiles_follow_the_schedule_of_the_shape(variant, dtype, D, causal, BH, M, tiles):
    got = cfgs.choose_fa_tile(variant, dtype, D, causal, 1, BH, M, M, cfgs.fa_launch_candidates(variant, dtype, D))
    assert (got.block_m, got.block_n, got.waves, got.stages) in tiles


@pytest.mark.parametrize("variant,D,tile", [(1, 64, (128, 64, 4, 5)), (1, 128, (128, 64, 4, 3)), (2, 64, (128, 32, 4, 6)),
                                            (0, 128, (128, 128, 4, 1)), (1, 256, (128, 32, 4, 6)), (1, 64, (256, 64, 8, 9)),
                                            (0, 64, (256, 64, 8, 1)), (0, 128, (256, 64, 8, 1)), (0, 128, (256, 64, 8, 8))])
@pytest.mark.parametrize("causal", [False, True])
def test_a_hinted_tile_is_kept(variant, D, tile, causal):
    """Hints that leave one tile get it, whether the schedule model knows it and its kind was timed or not."""
    for dtype in (torch.float16, torch.bfloat16):
        for BH, M in ((1, 129), (1, 4000), (64, 2048), (100, 300)):
            kw = dict(zip(("BLOCK_M", "BLOCK_N", "num_warps", "num_stages"), tile))
            got = flash_atten._tile_for(variant, dtype, D, causal, 1, BH, M, 4000, kw)
            assert (got.block_m, got.block_n, got.waves, got.stages) == tile


def test_a_new_length_asks_nothing_of_the_library(monkeypatch):
    """A length not seen before: the built tiles and the parsed table are those of earlier calls."""
    args = (hip_lib.FA_VARIANT_SLICED, torch.bfloat16, 128)
    flash_atten._tile_for(*args, False, 1, 32, 1, 5000, {})
    index = cfgs._bucket_index(cfgs.load_tune_table()["fa"])
    monkeypatch.setattr(hip_lib, "fa_fwd_supported", lambda *a: pytest.fail("the library was asked again"))
    for M, N, causal in ((1, 5001, False), (1, 70001, False), (777, 777, True), (3001, 3001, True)):
        flash_atten._tile_for(*args, causal, 1, 32, M, N, {})
    assert cfgs._bucket_index(cfgs.load_tune_table()["fa"]) is index


def test_split_residency_follows_the_resource_table():
    # D=128 4-wave split kernels keep two workgroups per CU; the D=256 pipelined kernel (one wave
    # per SIMD) and 8-wave kernels keep one
    assert cfgs.split_residency(torch.float16, 128, 128, 64, 4, 3) == 2
    assert cfgs.split_residency(torch.bfloat16, 256, 128, 32, 4, 3) == 1
    assert cfgs.split_residency(torch.float16, 128, 256, 128, 8, 2) == 1
    # decode shapes fill the resident capacity: 128 single-row tiles split in two when one split
    # workgroup fits a CU, in four when two do
    assert cfgs.choose_splits(1, 128, 1, 32768, 128, 32, resident_per_cu=1) == 2
    assert cfgs.choose_splits(1, 128, 1, 32768, 128, 32, resident_per_cu=2) == 4


def test_every_candidate_has_compiled_resources():
    for variant in (0, 1, 2):
        for dtype in (torch.float16, torch.bfloat16):
            for D in (64, 128, 256):
                cands = cfgs.fa_candidates(variant, dtype, D)
                assert cands, (variant, dtype, D)
                for c in cands:
                    res = cfgs.fa_resources(variant, dtype, D, c)
                    assert res is not None and res["lds_bytes"] <= 160 * 1024
                    # the resources are those of the candidate's own pipeline
                    sym = hip_lib.fwd_kernel_symbol(variant, dtype, D, c.to_c())
                    if c.stages >= 6:  # the 16x16x32-MFMA kernels: PIPE 0, 1, 2 (stages 6, 7, 8)
                        assert "fa_fwd16_kernel" in sym and f"ELi{c.waves}ELi{c.block_n}ELi{c.stages - 6}ELb" in sym, (
                            sym, c)
                    else:
                        assert f"ELi{c.block_n}ELi{c.stages}ELb" in sym, (sym, c)
    for t in cfgs.gemm_candidates():
        assert cfgs.gemm_resources(t) is not None


def test_refine_reranks_the_top_candidates_by_interleaved_medians(monkeypatch):
    """gfx950_tune._refine re-times only the fastest three of a first pass, in interleaved rounds,
    and ranks them by their medians (a one-pass outlier does not win the table)."""
    import gfx950_tune
    first = {"a": 1.00, "b": 1.01, "c": 1.02, "d": 1.50}
    later = {"a": [1.10, 1.09, 1.11, 1.10, 1.30], "b": [1.00, 1.01, 1.00, 0.99, 1.00], "c": [1.05] * 5}
    calls = []

    def fake_time(fn, warmup, iters, batch_ms=1.0):
        key = fn()
        calls.append(key)
        return later[key][sum(1 for k in calls if k == key) - 1]

    monkeypatch.setattr(gfx950_tune, "_time", fake_time)
    fns = {k: (lambda k=k: k) for k in first}
    refined = gfx950_tune._refine(fns, first)
    assert set(refined) == {"a", "b", "c"} and "d" not in calls
    assert calls[:3] == ["a", "b", "c"]  # interleaved, not candidate after candidate
    assert min(refined, key=refined.get) == "b" and refined["a"] == 1.10
    assert gfx950_tune._refine({"a": fns["a"]}, {"a": 1.0}) == {}
