// Host-visible kernel parameter blocks and registries shared between the kernel translation units
// and the C ABI (fa_abi.hip).
#pragma once

#include <stdint.h>

namespace fa {

// One attention-forward launch. Pointers are device pointers; strides are in elements.
struct FwdParams {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* o;
  float* lse;     // nullable: fp32 [B,H,M] natural-log sum-exp of the scaled logits
  float* ws_o;    // split partials [splits][B*H][M][D] fp32 (SPLIT kernels only)
  float* ws_lse;  // split partial lse [splits][B*H][M] fp32 (SPLIT kernels only)
  int64_t sq0, sq1, sq2;
  int64_t sk0, sk1, sk2;
  int64_t sv0, sv1, sv2;
  int64_t so0, so1, so2;
  int64_t sl0, sl1, sl2;
  int32_t B, H, Hkv, M, N;
  int32_t group;            // H / Hkv
  int32_t pack;             // 1, or group: the query heads of a kv head share one row space
                            // (row r = head offset r / M, position r % M); grid over (b, kv head)
  float c;                  // sm_scale * log2(e): exp(x*sm_scale) == exp2(x*c)
  float sm_scale;
  int32_t causal;
  int32_t splits;           // KV splits (1 when not splitting)
  int32_t tiles_per_split;  // KV tiles (of block_n rows) per split
  int32_t m_blocks;         // ceil(M / block_m)
  int32_t total_blocks;     // m_blocks * B * H * splits
  int32_t grid;             // workgroups launched (the persistent kernel's; total_blocks otherwise)
};

struct MergeParams {
  const float* ws_o;
  const float* ws_lse;
  uint16_t* o;
  float* lse;
  int64_t so0, so1, so2;
  int64_t sl0, sl1, sl2;
  int32_t B, H, M, splits;
  int32_t waves_per_row;  // 1, 2 or 4: the waves of a workgroup that share one row's splits
};

typedef void (*FwdKernelFn)(FwdParams);
typedef void (*MergeKernelFn)(MergeParams);

struct FaKernelEntry {
  int32_t stages;  // 1 = basic, 2 = double-buffered K/V LDS (optimized), 3-5 = LDS-DMA pipelines
                   // (32x32x16 MFMAs), 6-10 = 16x16x32 MFMA kernels: 6 lean, 7 software-pipelined,
                   // 8 ping-pong, 9 persistent ping-pong, 10 key groups (fa_fwd16.hip)
  int32_t dtype;   // FA_DTYPE_*
  int32_t D;
  int32_t waves;
  int32_t rows_per_wave;
  int32_t block_n;
  int32_t split;   // writes fp32 partials for the LSE merge
  const void* fn;
  const char* symbol;  // mangled kernel name (the key of the build's resource table)
  // The basic kernels of fa_fwd16.hip run the body of another stages number: its launch rules apply
  // (addressing limits, grid), and its KV tile may be smaller than the block_n the tile names.
  int32_t body_stages = 0;
  int32_t body_block_n = 0;
  int32_t pipeline() const { return body_stages ? body_stages : stages; }
  int32_t kv_tile() const { return body_block_n ? body_block_n : block_n; }
};

struct FaMergeEntry {
  int32_t dtype;
  int32_t D;
  const void* fn;
};

const FaKernelEntry* fa_fwd_registry(int* count);
const FaKernelEntry* fa_fwd16_registry(int* count);
const FaMergeEntry* fa_merge_registry(int* count);

struct GemmParams {
  const uint16_t* a;
  const uint16_t* b;
  uint16_t* c;
  int32_t M, N, K;
  int64_t lda, ldb, ldc;
  int32_t group_m;
  int32_t tiles_m, tiles_n;
  int32_t region_m;  // 0: flat grouped order; else XCD regions in region_m rows x (8 / region_m) columns
  int32_t grid;      // workgroups launched (the persistent kernel walks tiles with this stride)
  // split K over the grid (gemm_f16_part_kernel, gemm_f16_reduce_kernel)
  float* ws;                // fp32 partial products [ksplits][M][N]
  int32_t ksplits;
  int32_t slabs_per_split;  // K slabs (of block_k) per split
};

struct GemmKernelEntry {
  int32_t block_m, block_n, block_k, waves;
  const void* fn;          // default slab ring (as deep as fits in 128 KiB, up to 4)
  const void* fn_shallow;  // shallow ring for short K (nullptr when it would be the same)
  const char* symbol;      // mangled name of `fn`
  const void* fn_persist;  // persistent short-K kernel (nullptr when not built for the tile)
  const void* fn_part = nullptr;  // split-K kernel (nullptr when not built for the tile)
};

// K slabs up to which a tile's shallow-ring kernel is launched (more workgroups per CU beat a
// deeper prefetch when the whole K loop is this short).
constexpr int kGemmShallowMaxSlabs = 8;
// K slabs for which a tile's persistent kernel is launched (when built and the shape divides into
// whole tiles): at least the slab steps over which it stores a tile's C, and few enough that the C
// write is a large share of the time.
constexpr int kGemmPersistMinSlabs = 4;
constexpr int kGemmPersistMaxSlabs = 16;
// Waves the persistent kernel adds to the tile's compute waves to write C (one per SIMD).
constexpr int kGemmPersistStoreWaves = 4;

const GemmKernelEntry* gemm_registry(int* count);
const void* gemm_reduce_fn();

// Resources of one kernel as the compiler reported them (-Rpass-analysis=kernel-resource-usage).
// The table is generated by build_lib.py after the kernels are compiled and linked into the
// library (_build/kernel_resource_table.cpp).
struct KernelResourceRow {
  const char* symbol;
  int32_t vgprs, agprs, sgprs, lds_bytes, scratch_bytes, occupancy;
};
extern const KernelResourceRow kKernelResourceRows[];
extern const int kKernelResourceRowCount;

}  // namespace fa
