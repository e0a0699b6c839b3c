// Attention forward with v_mfma_f32_16x16x32 tiles (stages=6): the lean one-KV-tile-per-step
// pipeline (stages=5) rebuilt around 16x16 MFMA tiles.
//
// Same algorithm as fa_fwd.hip (reference flash_atten.py:14-50 / 136-172 / 261-275: online
// softmax over KV tiles in the exp2 domain with a lazily moved row offset, P rounded to the input
// dtype before P V, O normalised by the row sum at the end; causal top-left; GQA by head index;
// split-KV partials + LSE merge for the sliced variant). What changes is the matrix-core shape:
//  * 16x16x32 MFMAs move half the accumulator registers per flop of 32x32x16 ones. The attention
//    kernels run at the chip's power cap (MFMA busy ~0.6 at 1.5-1.7 GHz); in the GEMM the same
//    switch raised the clock of the power-capped 8-wave tiles from ~1.5 to ~1.8 GHz.
//  * Scores are S^T = K Q^T per 16-key x 16-query tile: lane l holds query (l & 15) and keys
//    4 (l >> 4) + 0..3, so a query's row max / sum spans the four 16-lane rows of the wave (two
//    permlane swaps). Each wave owns 32 query rows as two 16-query tiles.
//  * P feeds P V straight from the score registers. For 32 keys (score tiles 2c, 2c+1) a lane holds
//    keys {4g .. 4g+3} and {16+4g .. 16+4g+3} (g = l >> 4) of its query: those 8 values are its B
//    operand (MFMA k index 8g + e), and the V^T A operand is built to match: two transposing reads
//    whose 16-lane group g addresses rows 4g.. and 16+4g.. of the 32-key chunk.
//  * The pipelined binary16 kernels take the row sum l from P V itself: one more MFMA per 32-key
//    chunk and query tile, with an all-ones A operand, leaves every lane its query's sum.
//  * K and V tiles reach LDS by LDS-DMA in fragment-major order (every 1 KiB block is exactly what
//    one read instruction of the wave reads), into a 2-slot ring, as in stages=5.
#include <type_traits>

#include "fa_common.h"
#include "fa_kernels.h"
#include "../../include/fa_gfx950.h"

namespace fa {

// PIPE 0 (stages=6): one KV tile per step. PIPE 1 (stages=7): the stages=3 software pipeline --
// the QK MFMAs of tile u+1 beside the exp / pack VALU work of tile u, then the PV MFMAs of tile u
// beside the row max of tile u+1.
template <typename Tag, int D, int WAVES, int BN, int PIPE, bool SPLIT>
struct Fwd16 {
  static constexpr int THREADS = WAVES * 64;
  static constexpr int QT = 2;            // 16-query tiles per wave
  static constexpr int ROWS = 16 * QT;    // query rows per wave
  static constexpr int KG = PIPE == 4 ? 2 : 1;  // groups of waves that share the rows and split the keys
  static constexpr int BM = WAVES / KG * ROWS;
  static constexpr int DC = D / 32;       // 32-deep d chunks of Q K^T
  static constexpr int DTL = D / 16;      // 16-row d tiles of O^T
  static constexpr int JT = BN / 16;      // 16-key score tiles
  static constexpr int KC = BN / 32;      // 32-key chunks of P V
  static constexpr int NKB = JT * DC;     // 1 KiB K blocks per tile
  static constexpr int NVB = KC * DTL;    // 1 KiB V blocks per tile
  static constexpr int KT_ELEMS = NKB * 512;
  static constexpr int VT_ELEMS = NVB * 512;
  static constexpr int NKW = NKB / WAVES;  // DMA blocks per wave per tile
  static constexpr int NVW = NVB / WAVES;
  static constexpr float THRESH = 8.0f;    // lazy-rescale threshold (log2 units)
  static constexpr bool kSumRounded = __is_same(Tag, f16_t);
  // Pipelined binary16 kernels: the row sum l comes from one more MFMA per (32-key chunk, query
  // tile) whose A operand is all ones, so every lane ends with its query's full sum of the rounded
  // P (the same sum the VALU dot2 path forms) and the step's VALU work loses 16 ops. bfloat16 keeps
  // the fp32 sum of the unrounded P.
  static constexpr bool kSumMfma = PIPE && __is_same(Tag, f16_t);
  static_assert(D % 32 == 0 && BN % 32 == 0, "tile shape");
  static_assert(NKB % WAVES == 0 && NVB % WAVES == 0, "tile blocks must split evenly over waves");
  static_assert(DC % NKW == 0 && DTL % NVW == 0, "a wave's DMA blocks stay in one key group");
  static_assert(BM % BN == 0, "causal tile bound assumes block_m % block_n == 0");
  // Workgroups per CU the launch bounds ask for: the one-tile-per-step kernel with 32-key tiles at
  // D <= 128 fits three (LDS and registers), the others two (the pipelined kernel holds two score
  // tiles).
  static constexpr int kBlocksPerCu = PIPE >= 2 ? 1 : (!PIPE && BN == 32 && D <= 128) ? 3 : 2;
  static_assert(KT_ELEMS == VT_ELEMS, "one ring offset serves K and V");
  static_assert(PIPE < 2 || WAVES == 8, "the ping-pong kernels run two groups of four waves");
  // Q fragments of the workgroup's rows in LDS (persistent kernel): block (wave, qt, cc) of 1 KiB
  // holds, at byte 16 l, Q[row wave*ROWS + 16 qt + (l & 15)][32 cc + 8 (l >> 4) .. +7] -- lane l's qf.
  static constexpr int QB_ELEMS = PIPE == 3 ? WAVES * QT * DC * 512 : 0;
  static constexpr int kQChunks = 4;  // steps over which the persistent kernel prefetches the next Q
  // O leaves in 64-byte row pieces (pack_o_wide) except from the kernels held to three workgroups
  // per CU, whose register cap the extra swap registers would exceed (they spilled).
  static constexpr bool kWideO = !SPLIT && kBlocksPerCu < 3;
  static constexpr bool kScalarIds = BN == 64 && PIPE != 1;

  typedef DT<Tag> T;
  typedef floatx4 STile[JT][QT];
  typedef floatx4 OAcc[DTL][QT];

  // S^T tiles of one KV tile from its fragment-major K slot: block (jt, cc) holds, at byte 16 l,
  // K[jt*16 + (l & 15)][cc*32 + 8 (l >> 4) .. +7] (the MFMA A operand of lane l).
  __device__ static inline void qk(STile& s, const u32x4 (&qf)[QT][DC], const uint16_t* kslot_lane) {
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int cc = 0; cc < DC; ++cc) {
#pragma unroll
      for (int jt = 0; jt < JT; ++jt) {
        const u32x4 kf = *reinterpret_cast<const u32x4*>(kslot_lane + (jt * DC + cc) * 512);
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) s[jt][qt] = T::mfma16(kf, qf[qt][cc], cc == 0 ? zero : s[jt][qt]);
      }
    }
  }

  // O^T += V^T P^T from the fragment-major V slot: block (kc, dt) holds the two transposing reads of
  // that (32-key chunk, 16-column d tile); in read `half` lane L's 8 bytes (at 8 L) are
  // V[kc*32 + 16 half + 4 (L >> 4) + ((L & 15) >> 2)][dt*16 + 4 (L & 3) .. +3].
  __device__ static inline void pv(OAcc& acc, const u32x4 (&pk)[KC][QT], const uint16_t* vslot_lane,
                                   floatx4 (&lsum)[QT]) {
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) {
      if constexpr (kSumMfma) {
        constexpr uint32_t one2 = __is_same(Tag, f16_t) ? 0x3c003c00u : 0x3f803f80u;
        const u32x4 ones = {one2, one2, one2, one2};
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) lsum[qt] = T::mfma16(ones, pk[kc][qt], lsum[qt]);
      }
#pragma unroll
      for (int dt = 0; dt < DTL; ++dt) {
        const uint16_t* base = vslot_lane + (kc * DTL + dt) * 512;
        const u32x2 lo = lds_read_tr16(base);
        const u32x2 hi = lds_read_tr16(base + 256);
        const u32x4 vf = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) acc[dt][qt] = T::mfma16(vf, pk[kc][qt], acc[dt][qt]);
      }
    }
  }

  // Keys past N, and (causal) keys after the query row, get score -inf. Wave-uniform test first.
  __device__ static inline bool tile_needs_mask(int n0, int wrow0, const FwdParams& p) {
    return (n0 + BN > p.N) || (p.causal && n0 + BN - 1 > wrow0);
  }
  // First tile of the range starting at tile t_begin (counted from it) that needs the mask: the test
  // above holds from there on, so a loop over tiles compares its index with this one number.
  __device__ static inline int first_masked_tile(int t_begin, int wrow0, const FwdParams& p) {
    int first = p.N / BN;
    if (p.causal) first = min(first, (wrow0 + 1) / BN);
    return __builtin_amdgcn_readfirstlane(first - t_begin);
  }
  // KV tiles, of the ntiles from t_begin on, that the ROWS rows from wrow0 attend to (0 without rows). A
  // wave multiplies no tile past them: its P would be all zeros there, and 0 times an infinity or NaN
  // in such a V row is NaN.
  __device__ static inline int wave_tile_count(bool has_rows, int wrow0, int t_begin, int ntiles, const FwdParams& p) {
    int n = has_rows ? ntiles : 0;
    if (p.causal) n = min(n, (wrow0 + ROWS - 1) / BN + 1 - t_begin);
    return __builtin_amdgcn_readfirstlane(n);
  }
  // Key j of query i is kept when j < lim_i = N (or min(N, i + 1) causal). Each element takes a
  // sign-bit mask and a bitfield select -- vector ALU only: per-element compares would each hold a
  // scalar register pair, and the scheduler hoists all 32 of them.
  __device__ static inline void mask_tile(STile& s, int n0, int wrow0, int q16, int g, const FwdParams& p) {
    mask_tile(s, n0, wrow0, q16, g, p.N, p.causal != 0);
  }
  __device__ static inline void mask_tile(STile& s, int n0, int wrow0, int q16, int g, int n_lim, bool causal) {
    const uint32_t ninf = __float_as_uint(FA_NEG_INF);
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const int i = wrow0 + qt * 16 + q16;
      const int lim = causal ? min(n_lim, i + 1) : n_lim;
#pragma unroll
      for (int jt = 0; jt < JT; ++jt) {
        const int rel = lim - (n0 + jt * 16 + 4 * g);  // keys r < rel of this lane are kept
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const uint32_t keep = (uint32_t)((r - rel) >> 31);  // all ones when r < rel
          s[jt][qt][r] = __uint_as_float((__float_as_uint(s[jt][qt][r]) & keep) | (ninf & ~keep));
        }
      }
    }
  }

  // Max of a score tile over this lane's keys of each query (a quarter of the row: the row's max
  // over the four lane rows is formed only when the offset moves, in rescale). A chain that takes
  // two scores per step (v_max3_f32): 4·JT/2 ops per query tile, where a tree per key tile costs more.
  __device__ static inline void tile_max(const STile& s, float (&mx)[QT]) {
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      float m = fmaxf(s[0][qt][0], s[0][qt][1]);
      m = fmaxf(fmaxf(m, s[0][qt][2]), s[0][qt][3]);
#pragma unroll
      for (int jt = 1; jt < JT; ++jt) {
        m = fmaxf(fmaxf(m, s[jt][qt][0]), s[jt][qt][1]);
        m = fmaxf(fmaxf(m, s[jt][qt][2]), s[jt][qt][3]);
      }
      mx[qt] = m;
    }
  }

  // O and l of query tile qt times alpha.
  __device__ static inline void scale_row(int qt, float alpha, OAcc& acc, float (&l_i)[QT], floatx4 (&lsum)[QT]) {
    if constexpr (kSumMfma) {
#pragma unroll
      for (int r = 0; r < 4; ++r) lsum[qt][r] *= alpha;
    } else {
      l_i[qt] *= alpha;
    }
#pragma unroll
    for (int dt = 0; dt < DTL; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[dt][qt][r] *= alpha;
  }
  // Exponent offsets of a wave's QT query tiles: m in score units (-inf before the first tile),
  // and two values derived from it: mc(c) = m c (0 while m is -inf), the offset every score's FMA
  // subtracts, and thr(c) = m + THRESH / c, the bound of the rescale test. The ping-pong kernels,
  // whose softmax phase is VALU-bound, keep both and update them only when the offset moves
  // (rare; measured 0.4-0.7% faster non-causal); the others take them per step (the 256-dimension
  // kernel at its register cap ran 4.5% slower keeping them).
  static constexpr bool kCachedOff = PIPE >= 2;
  struct RowOff {
    float m[QT], mc_[kCachedOff ? QT : 1], thr_[kCachedOff ? QT : 1];
    __device__ inline void reset() {
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        m[qt] = FA_NEG_INF;
        if constexpr (kCachedOff) {
          mc_[qt] = 0.f;
          thr_[qt] = FA_NEG_INF;
        }
      }
    }
    __device__ inline void set(int qt, float m_new, float c) {
      m[qt] = m_new;
      if constexpr (kCachedOff) {
        mc_[qt] = (m_new == FA_NEG_INF) ? 0.f : m_new * c;
        thr_[qt] = m_new + THRESH / c;
      }
    }
    __device__ inline float mc(int qt, float c) const {
      if constexpr (kCachedOff) return mc_[qt];
      else return (m[qt] == FA_NEG_INF) ? 0.f : m[qt] * c;
    }
    __device__ inline float thr(int qt, float c) const {
      if constexpr (kCachedOff) return thr_[qt];
      else return m[qt] + THRESH / c;
    }
  };

  // Lazy rescale: move the exponent offset (and rescale O and l) only when some lane of the wave
  // sees a score more than THRESH (log2 units) above it; the moved offset is the row max over the
  // four lane rows, so the lanes of a query keep one offset. One ballot over all query tiles guards
  // the per-tile tests, so a step that moves no offset (the common case) takes a single branch.
  __device__ static inline void rescale(const float (&mx)[QT], OAcc& acc, RowOff& ro, float (&l_i)[QT],
                                        floatx4 (&lsum)[QT], float c) {
    bool need[QT], any = false;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      need[qt] = mx[qt] > ro.thr(qt, c);
      any |= need[qt];
    }
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(any) == 0, 1)) return;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      if (__builtin_amdgcn_ballot_w64(need[qt]) != 0) {
        const float m_new = fmaxf(ro.m[qt], xquad_max(mx[qt]));
        const float alpha = (ro.m[qt] == FA_NEG_INF) ? 0.f : fast_exp2((ro.m[qt] - m_new) * c);
        ro.set(qt, m_new, c);
        scale_row(qt, alpha, acc, l_i, lsum);
      }
    }
  }

  // Online softmax of one score tile that needs no mask: row max, lazy rescale, then P.
  __device__ static inline void softmax_unmasked(const STile& s, u32x4 (&pk)[KC][QT], OAcc& acc, RowOff& ro,
                                                 float (&l_i)[QT], floatx4 (&lsum)[QT], float c) {
    float mx[QT];
    tile_max(s, mx);
    rescale(mx, acc, ro, l_i, lsum, c);
    exp_pack(s, pk, ro, l_i, c);
  }

  // The same for a tile that may need one.
  __device__ static inline void softmax(STile& s, u32x4 (&pk)[KC][QT], OAcc& acc, RowOff& ro,
                                        float (&l_i)[QT], floatx4 (&lsum)[QT], bool masked, int n0, int wrow0, int q16,
                                        int g, const FwdParams& p) {
    if (masked) mask_tile(s, n0, wrow0, q16, g, p);
    softmax_unmasked(s, pk, acc, ro, l_i, lsum, p.c);
  }

  // P = exp2(S c - m c) rounded to the input dtype and packed as the B operand of P V; the row
  // sum l accumulates the same P.
  __device__ static inline void exp_pack(const STile& s, u32x4 (&pk)[KC][QT], const RowOff& ro,
                                         float (&l_i)[QT], float c) {
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const float mc = ro.mc(qt, c);
      float l0 = 0.f, l1 = 0.f;
#pragma unroll
      for (int kc = 0; kc < KC; ++kc)
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            const floatx4& t = s[2 * kc + half][qt];
            const float e0 = fast_exp2(__builtin_fmaf(t[2 * w], c, -mc));
            const float e1 = fast_exp2(__builtin_fmaf(t[2 * w + 1], c, -mc));
            const uint32_t pw = T::pack2(e0, e1);
            pk[kc][qt][2 * half + w] = pw;
            if (kSumMfma) {
              // l comes from the ones-row MFMA in pv
            } else if (kSumRounded) {
              // binary16 P: summing the rounded pair moves l by <= 2^-12 relative
              if (w) l1 = dot2_sum<Tag>(pw, l1);
              else l0 = dot2_sum<Tag>(pw, l0);
            } else {
              // bfloat16 P is too coarse for l: sum the fp32 values
              if (w) l1 += e0 + e1;
              else l0 += e0 + e1;
            }
          }
      if (!kSumMfma) l_i[qt] += l0 + l1;
    }
  }

  // Scheduling hints: LDS fragment reads a few MFMAs ahead of their use.
  __device__ static inline void qk_schedule() {
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);  // DS read
#pragma unroll
    for (int i = 0; i < DC * JT; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, QT, 0);  // MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // DS read
    }
  }
  __device__ static inline void pv_schedule() {
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 1);
#pragma unroll
    for (int i = 0; i < KC * DTL; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, QT, 1);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
    }
  }
  // Between the phases of a ping-pong step that has no branch: without it the scheduler moves the
  // softmax's packs past the barrier into the matrix phase and the DMA into the softmax (4% slower).
  __device__ static inline void phase_fence() { __builtin_amdgcn_sched_barrier(0); }
  // Ping-pong matrix block (QK of the next tile, then PV of this one, one scheduling region): AHEAD
  // LDS reads first, then the remaining K and V fragment reads spread evenly over the MFMA groups.
  template <int I, int G, int NR>
  __device__ static inline void m_schedule_groups() {
    if constexpr (I < G) {
      __builtin_amdgcn_sched_group_barrier(0x008, QT, 3);
      constexpr int r = (NR * (I + 1)) / G - (NR * I) / G;
      if constexpr (r > 0) __builtin_amdgcn_sched_group_barrier(0x100, r, 3);
      m_schedule_groups<I + 1, G, NR>();
    }
  }
  template <int AHEAD>
  __device__ static inline void m_schedule() {
    constexpr int reads = DC * JT + 2 * KC * DTL;
    __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 3);
    m_schedule_groups<0, DC * JT + KC * DTL, reads - AHEAD>();
  }
  // Pipelined step, first half: the next tile's QK MFMAs with this tile's exp / pack / sum VALU work
  // (FMA + exp per score, pack + sum per pair), a few VALU ops per group of QT MFMAs.
  static constexpr int kExpValu = QT * JT * (4 * 2 + 2 * (kSumMfma ? 1 : 2));
  static constexpr int kXValuPerMfma = (kExpValu + DC * JT - 1) / (DC * JT);
  __device__ static inline void x_schedule() {
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 2);
#pragma unroll
    for (int i = 0; i < DC * JT; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, QT, 2);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 2);
      __builtin_amdgcn_sched_group_barrier(0x002, kXValuPerMfma, 2);
    }
  }
  // Second half: this tile's PV MFMAs with the next tile's row max.
  __device__ static inline void y_schedule() {
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 2);
#pragma unroll
    for (int i = 0; i < KC * DTL; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, QT, 2);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 2);
      __builtin_amdgcn_sched_group_barrier(0x002, 2, 2);
    }
  }

  // Epilogue of one work item of the persistent kernel (the same code as the end of run(), which
  // keeps its copy inline: called there, even always-inlined, it pushed the 32-key one-tile-per-step
  // kernel past its 168-VGPR cap into scratch). l over the four lane rows, O = acc / l; lane holds
  // d = 16 dt + 4 g .. +3. The output parameters are read from the kernel-argument segment (scalar
  // loads at the point of use); fa_fwd16_kernel takes FwdParams as its only argument (checked there).
  __device__ __attribute__((always_inline)) static inline void store_out(const OAcc& acc, const RowOff& ro, const float (&l_i)[QT],
                                          const floatx4 (&lsum)[QT], int wrow0, int q16, int g, int rows, int b, int h,
                                          int split_u) {
    const auto pe = kernarg_params<FwdParams>();
    constexpr float kLn2 = 0.69314718055994530942f;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const float l = kSumMfma ? lsum[qt][0] : xquad_sum(l_i[qt]);
      const int i = wrow0 + qt * 16 + q16;
      const float inv = (l > 0.f) ? 1.f / l : 0.f;
      const float lse_val = (l > 0.f) ? (ro.m[qt] * pe->c + __builtin_amdgcn_logf(l)) * kLn2 : FA_NEG_INF;
      u32x4 wide[DTL / 2];
      if constexpr (kWideO) pack_o_wide(acc, qt, inv, wide);  // cross-lane: before the row test
      if (i < rows) {
        const int hr = pe->pack > 1 ? h + i / pe->M : h;
        const int mr = pe->pack > 1 ? i % pe->M : i;
        if (SPLIT) {
          const int64_t wrow = (int64_t)(split_u * pe->B + b) * pe->H + hr;  // [split][b][h][m] rows
          float* wo = pe->ws_o + (wrow * pe->M + mr) * D;
#pragma unroll
          for (int dt = 0; dt < DTL; ++dt) {
            floatx4 val = {acc[dt][qt][0] * inv, acc[dt][qt][1] * inv, acc[dt][qt][2] * inv, acc[dt][qt][3] * inv};
            *reinterpret_cast<floatx4*>(wo + dt * 16 + 4 * g) = val;
          }
          if (g == 0) pe->ws_lse[wrow * pe->M + mr] = lse_val;
        } else {
          uint16_t* orow = pe->o + (int64_t)b * pe->so0 + (int64_t)hr * pe->so1 + (int64_t)mr * pe->so2;
          if constexpr (kWideO) {
#pragma unroll
            for (int pp = 0; pp < DTL / 2; ++pp)
              *reinterpret_cast<u32x4*>(orow + 32 * pp + wide_col(g)) = wide[pp];
          } else {
#pragma unroll
            for (int dt = 0; dt < DTL; ++dt) {
              u32x2 val = {T::pack2(acc[dt][qt][0] * inv, acc[dt][qt][1] * inv),
                           T::pack2(acc[dt][qt][2] * inv, acc[dt][qt][3] * inv)};
              *reinterpret_cast<u32x2*>(orow + dt * 16 + 4 * g) = val;
            }
          }
          float* lse = pe->lse;
          if (lse != nullptr && g == 0)
            lse[(int64_t)b * pe->sl0 + (int64_t)hr * pe->sl1 + (int64_t)mr * pe->sl2] = lse_val;
        }
      }
    }
  }

  // O of query tile qt (times inv), rounded, as 16-byte lane chunks. The accumulator gives lane row g
  // (lanes 16 g .. 16 g + 15) columns d = 16 dt + 4 g .. +3 of each d tile, so a store per tile
  // writes 32 bytes of each of 16 rows, and every such half line is an L2 request of its own. One
  // v_permlane16_swap per dword of tiles 2 pp and 2 pp + 1 (it swaps the odd 16-lane rows of one
  // operand with the even rows of the other) leaves lane row g holding 8 consecutive columns of the
  // pair, starting at 32 pp + wide_col(g): each store then writes 64 contiguous bytes of each row,
  // half the store instructions and L2 requests. Cross-lane: call with every lane active.
  __device__ static inline void pack_o_wide(const OAcc& acc, int qt, float inv, u32x4 (&wide)[DTL / 2]) {
    static_assert(DTL % 2 == 0, "d tiles pair up");
#pragma unroll
    for (int pp = 0; pp < DTL / 2; ++pp) {
      const floatx4& a = acc[2 * pp][qt];
      const floatx4& b = acc[2 * pp + 1][qt];
      const auto lo = __builtin_amdgcn_permlane16_swap(T::pack2(a[0] * inv, a[1] * inv), T::pack2(b[0] * inv, b[1] * inv),
                                                       false, false);
      const auto hi = __builtin_amdgcn_permlane16_swap(T::pack2(a[2] * inv, a[3] * inv), T::pack2(b[2] * inv, b[3] * inv),
                                                       false, false);
      wide[pp] = (u32x4){lo[0], hi[0], lo[1], hi[1]};
    }
  }
  // First column, within a pair of d tiles, of lane row g's chunk: rows 0..3 hold tile 2 pp's
  // columns 0..7, tile 2 pp + 1's 0..7, tile 2 pp's 8..15, tile 2 pp + 1's 8..15.
  __device__ static inline int wide_col(int g) { return 8 * (((g & 1) << 1) | (g >> 1)); }

  // ---- persistent ping-pong (stages=9) ----------------------------------------------------------
  // One workgroup per CU walks a fixed sequence of work items (the logical blocks of run()). The
  // sequence is a snake over the XCD's slots: item k of XCD x goes to slot k % S in round k / S,
  // slots reversed in odd rounds, so that with heaviest-first causal blocks each slot's rounds pair
  // a heavy block with a light one. Within an item the schedule is run()'s ping-pong; across items
  // the K/V rings keep running: the last two steps of an item fetch the next item's K_0, K_1 and
  // V_0 into the slots the ring frees, and its first steps fetch the next item's Q into an LDS
  // buffer (each wave's own fragments, in kQChunks pieces), so an item starts without waiting on
  // memory.
  // A work item: its batch, query head, kv head and split, first query row and KV tile range.
  struct Item {
    int b, h, hk, split, m0, t_begin, ntiles;
  };
  // Buffer descriptors of an item's K and V rows (its (batch, kv head)) and Q rows (batch, head).
  template <class P>
  __device__ static inline u32x4 k_rsrc(const Item& d, const P& p) {
    return make_rsrc(p.k + (int64_t)d.b * p.sk0 + (int64_t)d.hk * p.sk1, (uint32_t)p.N * (uint32_t)p.sk2 * 2u);
  }
  template <class P>
  __device__ static inline u32x4 v_rsrc(const Item& d, const P& p) {
    return make_rsrc(p.v + (int64_t)d.b * p.sv0 + (int64_t)d.hk * p.sv1, (uint32_t)p.N * (uint32_t)p.sv2 * 2u);
  }
  template <class P>
  __device__ static inline u32x4 q_rsrc(const Item& d, const P& p) {
    return make_rsrc(p.q + (int64_t)d.b * p.sq0 + (int64_t)d.h * p.sq1, (uint32_t)p.M * (uint32_t)p.sq2 * 2u);
  }
  // Logical block of round r for workgroup w of G, or -1 past the end of its sequence.
  __device__ static inline int item_pid(int r, int w, int G, int total) {
    int x = 0, slot = w, S = G, per = total;
    if ((total & 7) == 0 && (G & 7) == 0) {  // XCD x = w % 8 walks logical blocks [x per, (x+1) per)
      x = w & 7;
      slot = w >> 3;
      S = G >> 3;
      per = total >> 3;
    }
    const int k = r * S + ((r & 1) ? S - 1 - slot : slot);
    return k < per ? x * per + k : -1;
  }
  template <class P>
  __device__ static inline Item make_item(int pid, const P& p) {
    // the divisions run on the vector ALU; their results are uniform
    Item it;
    const int rest = pid / p.m_blocks, bh = rest / p.splits;
    int mb = pid % p.m_blocks;
    if (p.causal) mb = p.m_blocks - 1 - mb;  // heaviest query blocks first, as run()
    it.m0 = __builtin_amdgcn_readfirstlane(mb) * BM;
    it.split = __builtin_amdgcn_readfirstlane(rest % p.splits);
    it.b = __builtin_amdgcn_readfirstlane(bh / p.H);
    it.h = __builtin_amdgcn_readfirstlane(bh % p.H);
    it.hk = __builtin_amdgcn_readfirstlane(it.h / p.group);
    it.t_begin = it.split * p.tiles_per_split;
    int n_end = (it.t_begin + p.tiles_per_split) * BN;
    if (n_end > p.N) n_end = p.N;
    if (p.causal && n_end > it.m0 + BM) n_end = it.m0 + BM;
    const int t_end = (n_end + BN - 1) / BN;
    it.ntiles = __builtin_amdgcn_readfirstlane(t_end > it.t_begin ? t_end - it.t_begin : 0);
    return it;
  }

  template <int GRP>
  __device__ static void persistent_group(const FwdParams& p, uint16_t* smem, int lane, int wave, int first_pid) {
    // lane-derived values are computed inside each group's copy of the loop: shared ones, hoisted
    // above the group branch, stayed live across group 0's loop and spilled
    asm volatile("" : "+v"(lane));
    const int q16 = lane & 15, g = lane >> 4;
    // workgroup id and count from the builtin and the host (blockIdx / gridDim go through library
    // calls that this build does not inline, whose results the compiler cannot prove uniform)
    const int G = p.grid, w = (int)__builtin_amdgcn_workgroup_id_x();
    // per-lane DMA offsets (item-independent): K, V as run(); Q rows of this wave within an item
    uint32_t koff, voff;
    {
      const int blk = wave * NKW, jt = blk / DC, cc = blk % DC;
      const uint32_t row = jt * 16 + (lane & 15), c0 = cc * 32 + 8 * (lane >> 4);
      koff = (row * (uint32_t)p.sk2 + c0) * 2u;
    }
    {
      const int blk = wave * NVW, kc = blk / DTL, dt = blk % DTL;
      const int m = lane;
      const uint32_t row = kc * 32 + 16 * (m >> 5) + 4 * ((m & 31) >> 3) + ((m & 7) >> 1);
      const uint32_t c0 = dt * 16 + 8 * (m & 1);
      voff = (row * (uint32_t)p.sv2 + c0) * 2u;
    }
    uint32_t qoff[QT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
      qoff[qt] = ((uint32_t)(wave * ROWS + qt * 16 + q16) * (uint32_t)p.sq2 + 8 * g) * 2u;
    uint16_t* kring = smem;
    uint16_t* vring = smem + 2 * KT_ELEMS;
    const uint16_t* qbuf = smem + 2 * (KT_ELEMS + VT_ELEMS);
    const uint32_t kring_lds = lds_address(smem), vring_lds = kring_lds + 2 * KT_ELEMS * 2;
    const uint32_t qbuf_lds = kring_lds + 2 * (KT_ELEMS + VT_ELEMS) * 2;
    const uint16_t* klane = kring + lane * 8;
    const uint16_t* vlane = vring + lane * 4;
    const uint16_t* qlane = qbuf + (wave * QT * DC) * 512 + lane * 8;

    // bytes between consecutive KV tiles of K and of V (the host keeps them below 2^32); a tile's
    // offset moves the buffer resource (slab_rsrc), so the lanes' offsets koff / voff stay fixed
    const uint32_t kstep = (uint32_t)BN * (uint32_t)p.sk2 * 2u, vstep = (uint32_t)BN * (uint32_t)p.sv2 * 2u;
    // Item-level parameters (pointers, strides, grid shape) are read through a fresh kernel-
    // argument pointer at each item boundary rather than held in scalar registers across the KV
    // loop: held there, they pushed the loop's own scalars out, and the compiler re-read strides
    // with scalar loads inside the loop, whose waits (lgkmcnt, shared with LDS reads) then
    // serialised every LDS fragment read.
    Item cur = make_item(first_pid, *kernarg_params<FwdParams>());
    int par = 0;              // ring slot of the current item's tile 0
    bool prefetched = false;  // its Q, K_0, K_1, V_0 were fetched by the previous item
    for (int r = 0;; ++r) {
      const auto pi = kernarg_params<FwdParams>();
      const int pid_n = item_pid(r + 1, w, pi->grid, pi->total_blocks);
      Item nxt;
      if (pid_n >= 0) {
        nxt = make_item(pid_n, *pi);
      } else {
        nxt = cur;
        nxt.ntiles = 0;
      }
      const int ntiles = cur.ntiles;
      const u32x4 krs = k_rsrc(cur, *pi), vrs = v_rsrc(cur, *pi);
      const int wrow0 = cur.m0 + wave * ROWS;
      const bool wave_has_rows = wrow0 < p.M;
      const int mask_from = first_masked_tile(cur.t_begin, wrow0, p);
      const int wtiles = wave_tile_count(wave_has_rows, wrow0, cur.t_begin, ntiles, p);
      // Tile u of the current item, or tile u - ntiles of the next one (K up to the next item's
      // tile 1, V up to its tile 0), into ring slot (par + u) & 1.
      // (The next item's branch builds its descriptors there, in the two steps per item that take
      // it; the empty asm keeps the compiler from merging the two branches' loads into one, which
      // would build those descriptors on every step.)
      auto issue_k = [&](int u) {
        const uint32_t slot = kring_lds + (uint32_t)((par + u) & 1) * (KT_ELEMS * 2) + wave * NKW * 1024;
        if (__builtin_expect(u < ntiles, 1)) {
          buffer_load16_to_lds_blocks<NKW, 64>(slab_rsrc(krs, (uint32_t)(cur.t_begin + u) * kstep, true), koff, slot);
        } else if (u - ntiles < nxt.ntiles) {
          asm volatile("");
          const uint32_t toff = (uint32_t)(nxt.t_begin + u - ntiles) * kstep;
          const auto pn = kernarg_params<FwdParams>();
          buffer_load16_to_lds_blocks<NKW, 64>(slab_rsrc(k_rsrc(nxt, *pn), toff, true), koff, slot);
        }
      };
      auto issue_v = [&](int u) {
        const uint32_t slot = vring_lds + (uint32_t)((par + u) & 1) * (VT_ELEMS * 2) + wave * NVW * 1024;
        if (__builtin_expect(u < ntiles, 1)) {
          buffer_load16_to_lds_blocks<NVW, 32>(slab_rsrc(vrs, (uint32_t)(cur.t_begin + u) * vstep, true), voff, slot);
        } else if (u - ntiles < nxt.ntiles) {
          asm volatile("");
          const uint32_t toff = (uint32_t)(nxt.t_begin + u - ntiles) * vstep;
          const auto pn = kernarg_params<FwdParams>();
          buffer_load16_to_lds_blocks<NVW, 32>(slab_rsrc(v_rsrc(nxt, *pn), toff, true), voff, slot);
        }
      };
      auto issue_q = [&](const Item& it) {
        const auto pq = kernarg_params<FwdParams>();
        const uint32_t moff = (uint32_t)it.m0 * (uint32_t)pq->sq2 * 2u;
        const u32x4 qrs = q_rsrc(it, *pq);
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
          buffer_load16_to_lds_blocks<DC, 64>(qrs, qoff[qt] + moff, qbuf_lds + ((wave * QT + qt) * DC) * 1024);
      };
      // Chunk c (of kQChunks) of this wave's QT * DC Q blocks of item `it`. Every workgroup starts
      // its items at about the same time, so the whole chip's next-item Q fetch issued in one step
      // (64 KiB per workgroup) made that step wait on HBM; in chunks over the item's first steps
      // it hides behind their K/V traffic (measured 1-4% faster; 8 chunks were slower than 4).
      auto issue_q_chunk = [&](const Item& it, int c) {
        const auto pq = kernarg_params<FwdParams>();
        const uint32_t moff = (uint32_t)it.m0 * (uint32_t)pq->sq2 * 2u;
        const u32x4 qrs = q_rsrc(it, *pq);
#pragma unroll
        for (int bq = 0; bq < QT * DC; ++bq) {
          if (bq * kQChunks / (QT * DC) == c) {
            const int qt = bq / DC, cc = bq % DC;
            buffer_load16_to_lds(qrs, qoff[qt] + moff + cc * 64, qbuf_lds + ((wave * QT + qt) * DC + cc) * 1024);
          }
        }
      };
      auto kslot = [&](int u) { return klane + ((par + u) & 1) * KT_ELEMS; };

      OAcc acc;
      RowOff ro;
      ro.reset();
      float l_i[QT];
      floatx4 lsum[QT];
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        l_i[qt] = 0.f;
        lsum[qt] = (floatx4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int dt = 0; dt < DTL; ++dt) acc[dt][qt] = (floatx4){0.f, 0.f, 0.f, 0.f};
      }
      if (ntiles > 0) {
        // DMA over an item of T tiles: K 0..T+1 and V 0..T (tiles past T - 1 are the next item's).
        // The previous item fetched this one's K_0, V_0 and, when T >= 2, K_1; with T == 1 this
        // item's K_1 is the next item's K_0, fetched here.
        if (!prefetched) {
          issue_q(cur);
          issue_k(0);
          wait_vm_lds_barrier<0>();
          issue_k(1);  // K_1 (or the next item's K_0) and V_0 land by the end of phase 2
          issue_v(0);
        } else if (ntiles == 1) {
          issue_k(1);
        }
        u32x4 qf[QT][DC];
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
#pragma unroll
          for (int cc = 0; cc < DC; ++cc) qf[qt][cc] = *reinterpret_cast<const u32x4*>(qlane + (qt * DC + cc) * 512);
        STile s;
        u32x4 pk[KC][QT];
        // Step j: S = Q K_j^T (ring offset tog), O += P_{j-1} V_{j-1} (the other slot)
        auto mma_block = [&](uint32_t tog) __attribute__((always_inline)) {
          // in the last step the QK reads the slot holding the next item's K_0 (landed one step
          // earlier; the step's DMA fills the other slot) and its S is never used: one
          // straight-line block, as in run()
          __builtin_amdgcn_s_setprio(1);
          qk(s, qf, klane + tog / 2);
          pv(acc, pk, vlane + (KT_ELEMS - tog / 2), lsum);
          m_schedule<8>();
          __builtin_amdgcn_s_setprio(0);
        };
        auto softmax_block = [&](int t) __attribute__((always_inline)) {
          if (t < wtiles) softmax(s, pk, acc, ro, l_i, lsum, t >= mask_from, (cur.t_begin + t) * BN, wrow0, q16, g, p);
        };
        if (GRP == 0 && wave_has_rows) {
          qk(s, qf, kslot(0));
          qk_schedule();
        }
        wait_vm_lds_barrier<63>();
        if (wave_has_rows) {
          if (GRP == 0) {
            softmax_block(0);
          } else {
            qk(s, qf, kslot(0));
            qk_schedule();
          }
        }
        // A prefetched item's Q, K_0, K_1 and V_0 landed by the previous item's last wait; what is
        // still in flight here is that item's O stores and (T == 1) the next item's K_0, which
        // only step 1's discarded QK reads before step 1's own wait. So the barrier need not
        // wait for memory (the O stores then drain during step 1).
        if (prefetched) wait_vm_lds_barrier<63>();
        else wait_vm_lds_barrier<0>();
        // Steps that take chunks of the next item's Q: 1 .. min(kQChunks, T) (none without a next item).
        const int q_last = __builtin_amdgcn_readfirstlane(nxt.ntiles > 0 ? min(kQChunks, ntiles) : 0);
        // Ring offset of K_j and V_j and the resources of step j's fetches, carried from step to step
        uint32_t tog = (uint32_t)((par + 1) & 1) * (KT_ELEMS * 2);
        u32x4 kr = slab_rsrc(krs, (uint32_t)(cur.t_begin + 2) * kstep, true);
        u32x4 vr = slab_rsrc(vrs, (uint32_t)(cur.t_begin + 1) * vstep, true);
        const uint32_t kdst = kring_lds + wave * NKW * 1024 + KT_ELEMS * 2, vdst = vring_lds + wave * NVW * 1024;
        auto advance = [&]() __attribute__((always_inline)) {
          tog = KT_ELEMS * 2 - tog;
          kr = slab_rsrc(kr, kstep, true);
          vr = slab_rsrc(vr, vstep, true);
        };
        auto fast_dma = [&]() __attribute__((always_inline)) {  // K_{j+1} and V_j, both of this item
          buffer_load16_to_lds_blocks<NKW, 64>(kr, koff, kdst - tog);
          buffer_load16_to_lds_blocks<NVW, 32>(vr, voff, vdst + tog);
        };
        // Steps fast_begin .. fast_end - 1 take no chunk of Q, no fetch across the item's end and no
        // masked tile: they run in a loop that tests nothing but its own end. The scalar tests and
        // offsets of a step sit between its barriers, where every cycle is the step's: with the loop,
        // and the item's divisions done once per item, B4 H32 D64 causal N=2048 went from 103 to 92 us,
        // D128 causal N=1024 from 50.0 to 48.3 and N=4096 from 530 to 523.
        const int fast_begin = q_last + 1;
        const int fast_end = wave_has_rows ? min(ntiles - 1, GRP == 0 ? mask_from : mask_from + 1) : 0;
        for (int j = 1; j <= ntiles; ++j) {
          if (j == fast_begin) {
            for (; j < fast_end; ++j) {
              fast_dma();
              if (GRP == 0) mma_block(tog);
              else softmax_unmasked(s, pk, acc, ro, l_i, lsum, p.c);
              phase_fence();
              wait_vm_lds_barrier<63>();
              phase_fence();
              if (GRP == 0) softmax_unmasked(s, pk, acc, ro, l_i, lsum, p.c);
              else mma_block(tog);
              phase_fence();
              advance();
              wait_vm_lds_barrier<0>();
              phase_fence();
            }
          }
          if (j + 1 < ntiles) {
            fast_dma();
          } else {
            issue_k(j + 1);
            issue_v(j);
          }
          // every wave read its Q fragments before the barriers above: the buffer takes the next
          // item's Q, chunk c at step min(c + 1, T), so all of it has landed by the item's last wait
          if (j <= q_last) {
#pragma unroll
            for (int c = 0; c < kQChunks; ++c)
              if (j == min(c + 1, ntiles)) issue_q_chunk(nxt, c);
          }
          if (j <= wtiles) {
            if (GRP == 0) mma_block(tog);
            else softmax_block(j - 1);
          }
          wait_vm_lds_barrier<63>();
          if (j <= wtiles) {
            if (GRP == 0) softmax_block(j);
            else mma_block(tog);
          }
          advance();
          wait_vm_lds_barrier<0>();
        }
      }
      {
        const auto pe = kernarg_params<FwdParams>();
        store_out(acc, ro, l_i, lsum, wrow0, q16, g, pe->M, cur.b, cur.h, cur.split);
      }
      if (pid_n < 0) break;
      prefetched = ntiles > 0 && nxt.ntiles > 0;
      par = (par + ntiles) & 1;
      cur = nxt;
    }
  }

  __device__ static void run_persistent(const FwdParams& p) {
    __shared__ __attribute__((aligned(16))) uint16_t smem[2 * (KT_ELEMS + VT_ELEMS) + QB_ELEMS];
    const int tid = (int)__builtin_amdgcn_workitem_id_x();
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int pid0 = item_pid(0, (int)__builtin_amdgcn_workgroup_id_x(), p.grid, p.total_blocks);
    if (pid0 < 0) return;  // workgroup-uniform: more workgroups than blocks
    if (wave < 4) persistent_group<0>(p, smem, lane, wave, pid0);
    else persistent_group<1>(p, smem, lane, wave, pid0);
  }

  // SKIP: a wave multiplies no tile past its rows' last key (wave_tile_count). The test per step, which
  // the compiler cannot take out of the loop, costs the 256-dimension kernel 1-2% (bf16 B1 H12 causal
  // N=1973 69.5 -> 70.7 us), so there only the basic variant makes it; elsewhere it costs nothing, and
  // the skipped products make causal grids 1-3% faster.
  template <bool SKIP = (D <= 128)>
  __device__ static void run(const FwdParams& p) {
    __shared__ __attribute__((aligned(16))) uint16_t smem[2 * (KT_ELEMS + VT_ELEMS)];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q16 = lane & 15, g = lane >> 4;

    // Logical block id: XCD-local, then (bh, split, m-block), m-block fastest; packed GQA rows for
    // decode shapes (row r = query head h + r / M, position r % M), as in fa_fwd.hip.
    const int pid = xcd_remap(blockIdx.x, p.total_blocks);
    int mb = pid % p.m_blocks;
    const int rest = pid / p.m_blocks;
    const int split = rest % p.splits;
    const int bh = rest / p.splits;
    if (p.causal) mb = p.m_blocks - 1 - mb;  // heaviest query blocks first
    int b, h, hk;
    if (p.pack > 1) {
      b = bh / p.Hkv;
      hk = bh % p.Hkv;
      h = hk * p.group;
    } else {
      b = bh / p.H;
      h = bh % p.H;
      hk = h / p.group;
    }
    // The integer divisions above run on the vector ALU, though their results are workgroup-
    // uniform. Declaring them uniform puts the tile bounds, and the loop's branches on them, in
    // scalar registers: measured 1-3% faster for the 64-key kernels; the 32-key ones lose (their
    // register allocation grows by 30-60 VGPRs), so they keep vector copies.
    if constexpr (kScalarIds) {
      mb = __builtin_amdgcn_readfirstlane(mb);
      b = __builtin_amdgcn_readfirstlane(b);
      h = __builtin_amdgcn_readfirstlane(h);
      hk = __builtin_amdgcn_readfirstlane(hk);
    }
    const int split_u = kScalarIds ? __builtin_amdgcn_readfirstlane(split) : split;
    const int rows = p.M * p.pack;
    const int m0 = mb * BM;
    const int wrow0 = m0 + wave * ROWS;
    const bool wave_has_rows = wrow0 < rows;
    auto row_head = [&](int r) { return p.pack > 1 ? h + r / p.M : h; };
    auto row_pos = [&](int r) { return p.pack > 1 ? r % p.M : r; };

    // Q^T fragments (B operand of Q K^T): lane holds query row wrow0 + 16 qt + q16 at
    // d = 32 cc + 8 g .. +7.
    u32x4 qf[QT][DC];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const int row = wrow0 + qt * 16 + q16;
      const uint16_t* qrow =
          p.q + (int64_t)b * p.sq0 + (int64_t)row_head(row) * p.sq1 + (int64_t)row_pos(row) * p.sq2;
#pragma unroll
      for (int cc = 0; cc < DC; ++cc) {
        u32x4 val = {0u, 0u, 0u, 0u};
        if (row < rows) val = *reinterpret_cast<const u32x4*>(qrow + cc * 32 + g * 8);
        qf[qt][cc] = val;
      }
    }

    // KV tiles of this split, clipped by the causal diagonal.
    const int t_begin = split_u * p.tiles_per_split;
    int n_end = (t_begin + p.tiles_per_split) * BN;
    if (n_end > p.N) n_end = p.N;
    if (p.causal && n_end > m0 + BM) n_end = m0 + BM;
    const int t_end = (n_end + BN - 1) / BN;
    const int ntiles = t_end > t_begin ? t_end - t_begin : 0;
    const int wtiles = wave_tile_count(wave_has_rows, wrow0, t_begin, ntiles, p);

    OAcc acc;
    RowOff ro;
    ro.reset();
    float l_i[QT];
    floatx4 lsum[QT];  // row sums of the ones-row MFMA (kSumMfma)
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      l_i[qt] = 0.f;
      lsum[qt] = (floatx4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int dt = 0; dt < DTL; ++dt) acc[dt][qt] = (floatx4){0.f, 0.f, 0.f, 0.f};
    }

    // LDS-DMA sources: the buffer range is the (b, kv-head) rows [0, N) of K and of V, so rows past
    // N read as zero (the host keeps (N + block_n) * row stride * 2 bytes below 2^32). Lane m of a
    // K block (jt, cc) moves K[jt*16 + (m & 15)][cc*32 + 8 (m >> 4) .. +7]; a wave's next block is
    // the next d chunk (+64 bytes). Lane m of a V block (kc, dt) moves the 16 bytes of transposing-
    // read lanes L = 2 (m & 31), L + 1 of read m >> 5: V[kc*32 + 16 (m >> 5) + 4 ((m & 31) >> 3)
    // + ((m & 7) >> 1)][dt*16 + 8 (m & 1) .. +7]; a wave's next block is the next d tile (+32 bytes).
    const auto krs = make_rsrc(p.k + (int64_t)b * p.sk0 + (int64_t)hk * p.sk1, (uint32_t)p.N * (uint32_t)p.sk2 * 2u);
    const auto vrs = make_rsrc(p.v + (int64_t)b * p.sv0 + (int64_t)hk * p.sv1, (uint32_t)p.N * (uint32_t)p.sv2 * 2u);
    uint32_t koff, voff;
    {
      const int blk = wave * NKW, jt = blk / DC, cc = blk % DC;
      const uint32_t row = jt * 16 + (lane & 15), c0 = cc * 32 + 8 * (lane >> 4);
      koff = (row * (uint32_t)p.sk2 + c0) * 2u;
    }
    {
      const int blk = wave * NVW, kc = blk / DTL, dt = blk % DTL;
      const int m = lane;
      const uint32_t row = kc * 32 + 16 * (m >> 5) + 4 * ((m & 31) >> 3) + ((m & 7) >> 1);
      const uint32_t c0 = dt * 16 + 8 * (m & 1);
      voff = (row * (uint32_t)p.sv2 + c0) * 2u;
    }
    uint16_t* kring = smem;
    uint16_t* vring = smem + 2 * KT_ELEMS;
    const uint32_t kring_lds = lds_address(smem), vring_lds = kring_lds + 2 * KT_ELEMS * 2;
    auto issue_k = [&](int u) {
      if (u >= ntiles) return;
      const uint32_t toff = (uint32_t)((t_begin + u) * BN) * (uint32_t)p.sk2 * 2u;
      const uint32_t slot = kring_lds + (uint32_t)(u & 1) * (KT_ELEMS * 2);
      // uniform tile offset (64-key kernels): it moves the resource, the lanes' offsets stay fixed
      if constexpr (kScalarIds)
        buffer_load16_to_lds_blocks<NKW, 64>(slab_rsrc(krs, toff, true), koff, slot + wave * NKW * 1024);
      else
        buffer_load16_to_lds_blocks<NKW, 64>(krs, koff + toff, slot + wave * NKW * 1024);
    };
    auto issue_v = [&](int u) {
      if (u >= ntiles) return;
      const uint32_t toff = (uint32_t)((t_begin + u) * BN) * (uint32_t)p.sv2 * 2u;
      const uint32_t slot = vring_lds + (uint32_t)(u & 1) * (VT_ELEMS * 2);
      if constexpr (kScalarIds)
        buffer_load16_to_lds_blocks<NVW, 32>(slab_rsrc(vrs, toff, true), voff, slot + wave * NVW * 1024);
      else
        buffer_load16_to_lds_blocks<NVW, 32>(vrs, voff + toff, slot + wave * NVW * 1024);
    };
    const uint16_t* klane = kring + lane * 8;  // this lane's 16 bytes in every K block
    const uint16_t* vlane = vring + lane * 4;  // this lane's 8 bytes in every V half-block

    if constexpr (PIPE == 2) {
      // Ping-pong: waves 0-3 (group 0) and 4-7 (group 1) run the same sequence of blocks, group 1
      // one phase behind, with a workgroup barrier between phases. Blocks alternate between matrix
      // work and softmax work -- block 0: S = Q K_0^T; block 2u+1: softmax of tile u (mask, row
      // max, rescale, P_u); block 2u+2: S = Q K_{u+1}^T (u+1 < n) and O += P_u V_u -- so in every
      // phase one group issues MFMAs while the other, on the same SIMDs, issues the exp/pack VALU
      // work, and the two streams overlap instead of taking turns inside one wave.
      // K_t and V_t live in slot t & 1 of two-slot rings. K_t is read in phases 2t (group 0) and
      // 2t+1 (group 1), V_t in phases 2t+2 and 2t+3; phase 2s (s >= 1) refills with K_{s+1} and
      // V_s (their slots' previous tiles were last read in phase 2s-1) and every wave waits for its
      // own refills before the barrier that ends phase 2s+1, two phases before their first reader.
      STile s;
      u32x4 pk[KC][QT];
      const int mask_from = first_masked_tile(t_begin, wrow0, p);
      auto mma_block = [&](const uint16_t* kj, const uint16_t* vp) {  // S = Q K_j^T, O += P_{j-1} V_{j-1}
        // past the last tile the QK reads a stale K slot and its S is never used: one straight-line
        // block lets the V reads start during the QK MFMAs
        // the matrix group issues first: its MFMAs then wait for no VALU op of the softmax group
        __builtin_amdgcn_s_setprio(1);
        qk(s, qf, kj);
        pv(acc, pk, vp, lsum);
        m_schedule<8>();
        __builtin_amdgcn_s_setprio(0);
      };
      auto softmax_block = [&](int t) {
        softmax(s, pk, acc, ro, l_i, lsum, t >= mask_from, (t_begin + t) * BN, wrow0, q16, g, p);
      };
      // Group G's sequence; phases 2j and 2j+1 form iteration j. The branches on G and on
      // wave_has_rows are wave-uniform, and every wave runs the same barriers.
      auto run_group = [&](auto G) {
        constexpr int grp = decltype(G)::value;
        issue_k(0);
        wait_vm_lds_barrier<0>();
        issue_k(1);  // K_1 and V_0 land by the end of phase 1
        issue_v(0);
        if (grp == 0 && wave_has_rows) {
          qk(s, qf, klane);
          qk_schedule();
        }
        wait_vm_lds_barrier<63>();
        if (wave_has_rows) {
          if (grp == 0) {
            softmax_block(0);
          } else {
            qk(s, qf, klane);
            qk_schedule();
          }
        }
        wait_vm_lds_barrier<0>();
        int j = 1;
        if (wave_has_rows) {
          // The steps without a masked tile or a fetch past the last one, in a loop that tests nothing
          // but its own end, its ring offset and resources carried along (scalar ops between the
          // barriers lengthen a step): fp16 B4 H32 D128 N=8192 3.52 -> 3.44 ms, bf16 N=4096 901 -> 882
          // us, D64 N=4096 564 -> 541.
          const int fast_end = min(ntiles - 1, grp == 0 ? mask_from : mask_from + 1);
          const uint32_t kstep = (uint32_t)BN * (uint32_t)p.sk2 * 2u, vstep = (uint32_t)BN * (uint32_t)p.sv2 * 2u;
          const uint32_t kdst = kring_lds + wave * NKW * 1024 + KT_ELEMS * 2, vdst = vring_lds + wave * NVW * 1024;
          uint32_t tog = KT_ELEMS * 2;  // slot offset of K_j and V_j
          u32x4 kr = slab_rsrc(krs, (uint32_t)(t_begin + 2) * kstep, true);
          u32x4 vr = slab_rsrc(vrs, (uint32_t)(t_begin + 1) * vstep, true);
          for (; j < fast_end; ++j) {
            buffer_load16_to_lds_blocks<NKW, 64>(kr, koff, kdst - tog);
            buffer_load16_to_lds_blocks<NVW, 32>(vr, voff, vdst + tog);
            phase_fence();
            if (grp == 0) mma_block(klane + tog / 2, vlane + (KT_ELEMS - tog / 2));
            else softmax_unmasked(s, pk, acc, ro, l_i, lsum, p.c);
            phase_fence();
            wait_vm_lds_barrier<63>();
            phase_fence();
            if (grp == 0) softmax_unmasked(s, pk, acc, ro, l_i, lsum, p.c);
            else mma_block(klane + tog / 2, vlane + (KT_ELEMS - tog / 2));
            phase_fence();
            tog = KT_ELEMS * 2 - tog;
            kr = slab_rsrc(kr, kstep, true);
            vr = slab_rsrc(vr, vstep, true);
            wait_vm_lds_barrier<0>();
            phase_fence();
          }
        }
        // Iterations with work for this wave. Worked out here and tested once per block: kept across the
        // fast loop, and tested inside the softmax blocks too, it made long steps 0.2-1% slower (fp16 B4
        // H32 D64 N=4096 560 -> 554 us, D128 N=8192 3557 -> 3552).
        const int last = wave_tile_count(wave_has_rows, wrow0, t_begin, ntiles, p);
        for (; j <= ntiles; ++j) {
          issue_k(j + 1);
          issue_v(j);
          const uint16_t *kj = klane + (j & 1) * KT_ELEMS, *vp = vlane + ((j - 1) & 1) * VT_ELEMS;
          if (j <= last) {
            if (grp == 0) mma_block(kj, vp);
            else softmax_block(j - 1);
          }
          wait_vm_lds_barrier<63>();
          if (grp == 0 ? j < last : j <= last) {
            if (grp == 0) softmax_block(j);
            else mma_block(kj, vp);
          }
          wait_vm_lds_barrier<0>();
        }
      };
      if (ntiles > 0) {
        if (wave < 4) run_group(std::integral_constant<int, 0>{});
        else run_group(std::integral_constant<int, 1>{});
      }
    } else if constexpr (PIPE) {
      // Step u reads K_{u+1} and V_u: K runs one tile ahead of V. 2-slot rings: step u issues
      // K_{u+2} into K_u's slot and V_{u+1} into V_{u-1}'s (both read in step u-1) and waits for
      // them at the end of the step. Before step u the wave holds S_u and its unmasked row max.
      STile sa, sb;
      float mxa[QT], mxb[QT];
      if (ntiles > 0) {
        issue_k(0);
        issue_v(0);
        issue_k(1);
        wait_vm_lds_barrier<0>();
        if (wave_has_rows) {
          qk(sa, qf, klane);
          qk_schedule();
          tile_max(sa, mxa);
        }
        wait_vm_lds_barrier<0>();  // every wave is done with K slot 0 before step 0 refills it
      }
      // Masks for tile u (rare: sequence end, causal diagonal) and the row max they change.
      auto fix_masked = [&](STile& cur, float (&mx_cur)[QT], int u) {
        const int n0 = (t_begin + u) * BN;
        if (tile_needs_mask(n0, wrow0, p)) {
          mask_tile(cur, n0, wrow0, q16, g, p);
          tile_max(cur, mx_cur);
        }
      };
      auto step = [&](STile& cur, float (&mx_cur)[QT], STile& nxt, float (&mx_nxt)[QT], int u) {
        issue_k(u + 2);
        issue_v(u + 1);
        if (u < wtiles) {  // waves without rows or keys here still move their share of K/V
          fix_masked(cur, mx_cur, u);
          rescale(mx_cur, acc, ro, l_i, lsum, p.c);
          u32x4 pk[KC][QT];
          exp_pack(cur, pk, ro, l_i, p.c);
          qk(nxt, qf, klane + ((u + 1) & 1) * KT_ELEMS);
          x_schedule();
          pv(acc, pk, vlane + (u & 1) * VT_ELEMS, lsum);
          tile_max(nxt, mx_nxt);
          y_schedule();
        }
        wait_vm_lds_barrier<0>();
      };
      auto last = [&](STile& cur, float (&mx_cur)[QT], int u) {
        if (u >= wtiles) return;
        fix_masked(cur, mx_cur, u);
        rescale(mx_cur, acc, ro, l_i, lsum, p.c);
        u32x4 pk[KC][QT];
        exp_pack(cur, pk, ro, l_i, p.c);
        pv(acc, pk, vlane + (u & 1) * VT_ELEMS, lsum);
        pv_schedule();
      };
      if (ntiles > 0) {
        int u = 0;
        for (; u + 2 < ntiles; u += 2) {
          step(sa, mxa, sb, mxb, u);
          step(sb, mxb, sa, mxa, u + 1);
        }
        if (u + 1 < ntiles) {
          step(sa, mxa, sb, mxb, u);
          last(sb, mxb, u + 1);
        } else {
          last(sa, mxa, u);
        }
      }
    } else {
    // One KV tile per step: step u issues tile u+1 into the slot tile u-1 left (read in step u-1)
    // and waits for it at the end of the step.
    if (ntiles > 0) {
      issue_k(0);
      issue_v(0);
      wait_vm_lds_barrier<0>();
    }
    for (int u = 0; u < ntiles; ++u) {
      issue_k(u + 1);
      issue_v(u + 1);
      if (SKIP ? u < wtiles : wave_has_rows) {  // waves without rows or keys here still move their share of K/V
        STile s;
        u32x4 pk[KC][QT];
        qk(s, qf, klane + (u & 1) * KT_ELEMS);
        qk_schedule();
        softmax(s, pk, acc, ro, l_i, lsum, tile_needs_mask((t_begin + u) * BN, wrow0, p), (t_begin + u) * BN, wrow0, q16, g,
                p);
        pv(acc, pk, vlane + (u & 1) * VT_ELEMS, lsum);
        pv_schedule();
      }
      wait_vm_lds_barrier<0>();
    }
    }

    // Epilogue: l over the four lane rows, O = acc / l; lane holds d = 16 dt + 4 g .. +3. The
    // output parameters are read again from the kernel-argument segment (scalar loads) rather than
    // kept in scalar registers across the loop, where they would crowd out its own; fa_fwd16_kernel
    // takes FwdParams as its only argument (checked there), so the segment starts with it.
    const auto pe = kernarg_params<FwdParams>();
    constexpr float kLn2 = 0.69314718055994530942f;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const float l = kSumMfma ? lsum[qt][0] : xquad_sum(l_i[qt]);
      const int i = wrow0 + qt * 16 + q16;
      const float inv = (l > 0.f) ? 1.f / l : 0.f;
      const float lse_val = (l > 0.f) ? (ro.m[qt] * pe->c + __builtin_amdgcn_logf(l)) * kLn2 : FA_NEG_INF;
      u32x4 wide[DTL / 2];
      if constexpr (kWideO) pack_o_wide(acc, qt, inv, wide);  // cross-lane: before the row test
      if (i < rows) {
        const int hr = pe->pack > 1 ? h + i / pe->M : h;
        const int mr = pe->pack > 1 ? i % pe->M : i;
        if (SPLIT) {
          const int64_t wrow = (int64_t)(split_u * pe->B + b) * pe->H + hr;  // [split][b][h][m] rows
          float* wo = pe->ws_o + (wrow * pe->M + mr) * D;
#pragma unroll
          for (int dt = 0; dt < DTL; ++dt) {
            floatx4 val = {acc[dt][qt][0] * inv, acc[dt][qt][1] * inv, acc[dt][qt][2] * inv, acc[dt][qt][3] * inv};
            *reinterpret_cast<floatx4*>(wo + dt * 16 + 4 * g) = val;
          }
          if (g == 0) pe->ws_lse[wrow * pe->M + mr] = lse_val;
        } else {
          uint16_t* orow = pe->o + (int64_t)b * pe->so0 + (int64_t)hr * pe->so1 + (int64_t)mr * pe->so2;
          if constexpr (kWideO) {
#pragma unroll
            for (int pp = 0; pp < DTL / 2; ++pp)
              *reinterpret_cast<u32x4*>(orow + 32 * pp + wide_col(g)) = wide[pp];
          } else {
#pragma unroll
            for (int dt = 0; dt < DTL; ++dt) {
              u32x2 val = {T::pack2(acc[dt][qt][0] * inv, acc[dt][qt][1] * inv),
                           T::pack2(acc[dt][qt][2] * inv, acc[dt][qt][3] * inv)};
              *reinterpret_cast<u32x2*>(orow + dt * 16 + 4 * g) = val;
            }
          }
          float* lse = pe->lse;
          if (lse != nullptr && g == 0)
            lse[(int64_t)b * pe->sl0 + (int64_t)hr * pe->sl1 + (int64_t)mr * pe->sl2] = lse_val;
        }
      }
    }
  }

  // ---- key groups (stages=10) ---------------------------------------------------------------------
  // The ping-pong schedule for grids too small to fill the chip with 256-row blocks: a block is 128
  // query rows, and its two groups of four waves hold the same rows and take alternate KV tiles
  // (group 0 tiles 0, 2, ..., group 1 tiles 1, 3, ...), one phase apart as in run(). Twice the blocks
  // with half the serial steps each, at twice the K/V fetch per step (a ring slot holds a pair of
  // tiles); the two partial results meet through LDS at the end, so there is no workspace and no
  // second launch. What bounds the small grids it is for is the longest block's chain of steps: bf16
  // B1 H12/2 D128 causal N=4096 94 -> 70 us (740 TFLOP/s), B2 H16 D64 777x1283 26 -> 19, fp16 B1 H28
  // D128 N=1024 29 -> 22. A step has a ping-pong step's products and takes 1.23 (D64) to 1.43 (D128) of
  // its time, so grids that fill the chip stay there.
  __device__ static void run_key_groups(const FwdParams& p) {
    static_assert(PIPE != 4 || (WAVES == 8 && BN == 64 && KG == 2), "two groups of four waves");
    constexpr uint32_t kPairK = 2 * KT_ELEMS * 2, kPairV = 2 * VT_ELEMS * 2;  // bytes of a ring slot
    __shared__ __attribute__((aligned(16))) uint16_t smem[4 * (KT_ELEMS + VT_ELEMS)];
    const int tid = (int)__builtin_amdgcn_workitem_id_x();
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q16 = lane & 15, g = lane >> 4;

    // Causal: heaviest query blocks of all heads first, heads fastest (with a multiple of 8 heads a
    // head's blocks stay on one XCD), so the last blocks to start are the short ones. Otherwise
    // neighbouring blocks of a head on one XCD, as run().
    int mb, rest;
    const int wg = (int)__builtin_amdgcn_workgroup_id_x();
    if (p.causal) {
      const int heads = p.total_blocks / p.m_blocks;
      mb = p.m_blocks - 1 - wg / heads;
      rest = wg % heads;
    } else {
      const int pid = xcd_remap(wg, p.total_blocks);
      mb = pid % p.m_blocks;
      rest = pid / p.m_blocks;
    }
    mb = __builtin_amdgcn_readfirstlane(mb);
    const int split = __builtin_amdgcn_readfirstlane(rest % p.splits);
    const int bh = rest / p.splits;
    const int bheads = p.pack > 1 ? p.Hkv : p.H;
    const int b = __builtin_amdgcn_readfirstlane(bh / bheads);
    const int hi = bh % bheads;
    const int h = __builtin_amdgcn_readfirstlane(p.pack > 1 ? hi * p.group : hi);
    const int hk = __builtin_amdgcn_readfirstlane(h / p.group);
    const int rows = p.M * p.pack;
    const int m0 = mb * BM;
    const int wrow0 = m0 + (wave & 3) * ROWS;
    const bool wave_has_rows = wrow0 < rows;

    u32x4 qf[QT][DC];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const int row = wrow0 + qt * 16 + q16;
      const int hr = p.pack > 1 ? h + row / p.M : h, mr = p.pack > 1 ? row % p.M : row;
      const uint16_t* qrow = p.q + (int64_t)b * p.sq0 + (int64_t)hr * p.sq1 + (int64_t)mr * p.sq2;
#pragma unroll
      for (int cc = 0; cc < DC; ++cc) {
        u32x4 val = {0u, 0u, 0u, 0u};
        if (row < rows) val = *reinterpret_cast<const u32x4*>(qrow + cc * 32 + g * 8);
        qf[qt][cc] = val;
      }
    }

    const int t_begin = split * p.tiles_per_split;
    int n_end = min((t_begin + p.tiles_per_split) * BN, p.N);
    if (p.causal) n_end = min(n_end, m0 + BM);
    n_end = __builtin_amdgcn_readfirstlane(n_end);
    const int ntiles = max((n_end + BN - 1) / BN - t_begin, 0);
    const int nsteps = (ntiles + 1) / 2;

    OAcc acc;
    RowOff ro;
    ro.reset();
    float l_i[QT];
    floatx4 lsum[QT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      l_i[qt] = 0.f;
      lsum[qt] = (floatx4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int dt = 0; dt < DTL; ++dt) acc[dt][qt] = (floatx4){0.f, 0.f, 0.f, 0.f};
    }

    // DMA sources and ring as run(); a slot holds the K (V) tiles of both groups. Keys past N read
    // zeros; a pair's second tile past the range's end is not multiplied.
    const u32x4 krs = make_rsrc(p.k + (int64_t)b * p.sk0 + (int64_t)hk * p.sk1, (uint32_t)p.N * (uint32_t)p.sk2 * 2u);
    const u32x4 vrs = make_rsrc(p.v + (int64_t)b * p.sv0 + (int64_t)hk * p.sv1, (uint32_t)p.N * (uint32_t)p.sv2 * 2u);
    uint32_t koff, voff;
    {
      const int blk = wave * NKW, jt = blk / DC, cc = blk % DC;
      koff = ((uint32_t)(jt * 16 + q16) * (uint32_t)p.sk2 + cc * 32 + 8 * g) * 2u;
    }
    {
      const int blk = wave * NVW, kc = blk / DTL, dt = blk % DTL;
      const uint32_t row = kc * 32 + 16 * (lane >> 5) + 4 * ((lane & 31) >> 3) + ((lane & 7) >> 1);
      voff = (row * (uint32_t)p.sv2 + dt * 16 + 8 * (lane & 1)) * 2u;
    }
    const uint32_t kring_lds = lds_address(smem), vring_lds = kring_lds + 2 * kPairK;
    const uint32_t ktile = (uint32_t)BN * (uint32_t)p.sk2 * 2u, vtile = (uint32_t)BN * (uint32_t)p.sv2 * 2u;
    // A tile that starts past N has no valid byte: its resource gets range 0 (slab_rsrc needs an
    // offset within the range).
    auto issue_k = [&](int u) __attribute__((always_inline)) {
      if (u >= nsteps) return;
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const int t = t_begin + 2 * u + x;
        const bool live = t * BN < p.N;
        buffer_load16_to_lds_blocks<NKW, 64>(slab_rsrc(krs, live ? (uint32_t)t * ktile : 0u, live), koff,
                                             kring_lds + (uint32_t)(u & 1) * kPairK + x * (KT_ELEMS * 2) + wave * NKW * 1024);
      }
    };
    auto issue_v = [&](int u) __attribute__((always_inline)) {
      if (u >= nsteps) return;
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const int t = t_begin + 2 * u + x;
        const bool live = t * BN < p.N;
        buffer_load16_to_lds_blocks<NVW, 32>(slab_rsrc(vrs, live ? (uint32_t)t * vtile : 0u, live), voff,
                                             vring_lds + (uint32_t)(u & 1) * kPairV + x * (VT_ELEMS * 2) + wave * NVW * 1024);
      }
    };

    auto run_group = [&](auto G) __attribute__((always_inline)) {
      constexpr int grp = decltype(G)::value;
      STile s;
      u32x4 pk[KC][QT];
      const uint16_t* klane = smem + grp * KT_ELEMS + lane * 8;
      const uint16_t* vlane = smem + 4 * KT_ELEMS + grp * VT_ELEMS + lane * 4;
      // first step of this group whose tile needs the mask
      int first = n_end / BN;
      if (p.causal) first = min(first, (wrow0 + 1) / BN);
      const int mask_from = __builtin_amdgcn_readfirstlane(max(first - t_begin - grp + 1, 0) / 2);
      // steps whose tile is in the range and, for some row of this wave, before the diagonal
      const int wsteps = max(wave_tile_count(wave_has_rows, wrow0, t_begin, ntiles, p) - grp + 1, 0) / 2;
      auto mma_block = [&](uint32_t tog) __attribute__((always_inline)) {  // S = Q K_j^T, O += P_{j-1} V_{j-1}
        __builtin_amdgcn_s_setprio(1);
        qk(s, qf, klane + tog * (2 * KT_ELEMS));
        pv(acc, pk, vlane + (1 - tog) * (2 * VT_ELEMS), lsum);
        m_schedule<8>();
        __builtin_amdgcn_s_setprio(0);
      };
      auto softmax_block = [&](int u) __attribute__((always_inline)) {
        if (u >= wsteps) return;
        const int n0 = (t_begin + 2 * u + grp) * BN;
        if (u >= mask_from) mask_tile(s, n0, wrow0, q16, g, n_end, p.causal != 0);
        softmax_unmasked(s, pk, acc, ro, l_i, lsum, p.c);
      };
      issue_k(0);
      wait_vm_lds_barrier<0>();
      issue_k(1);
      issue_v(0);
      if (grp == 0 && wave_has_rows) {
        qk(s, qf, klane);
        qk_schedule();
      }
      wait_vm_lds_barrier<63>();
      if (wave_has_rows) {
        if (grp == 0) {
          softmax_block(0);
        } else {
          qk(s, qf, klane);
          qk_schedule();
        }
      }
      wait_vm_lds_barrier<0>();
      int j = 1;
      if (wave_has_rows) {
        // unmasked inner steps, as run(): both tiles of the fetched pairs are inside [0, N)
        const int fast_end = min(min(nsteps - 1, (n_end / BN - t_begin) / 2 - 1), grp == 0 ? mask_from : mask_from + 1);
        const uint32_t kstep = 2 * ktile, vstep = 2 * vtile;
        uint32_t tog = 1;  // ring slot of K_j and V_j
        u32x4 kr = slab_rsrc(krs, (uint32_t)(t_begin + 4) * ktile, true);
        u32x4 vr = slab_rsrc(vrs, (uint32_t)(t_begin + 2) * vtile, true);
        const uint32_t kdst = kring_lds + wave * NKW * 1024, vdst = vring_lds + wave * NVW * 1024;
        for (; j < fast_end; ++j) {
#pragma unroll
          for (int x = 0; x < 2; ++x)
            buffer_load16_to_lds_blocks<NKW, 64>(slab_rsrc(kr, x * ktile, true), koff,
                                                 kdst + (1 - tog) * kPairK + x * (KT_ELEMS * 2));
#pragma unroll
          for (int x = 0; x < 2; ++x)
            buffer_load16_to_lds_blocks<NVW, 32>(slab_rsrc(vr, x * vtile, true), voff,
                                                 vdst + tog * kPairV + x * (VT_ELEMS * 2));
          phase_fence();
          if (grp == 0) mma_block(tog);
          else softmax_unmasked(s, pk, acc, ro, l_i, lsum, p.c);
          phase_fence();
          wait_vm_lds_barrier<63>();
          phase_fence();
          if (grp == 0) softmax_unmasked(s, pk, acc, ro, l_i, lsum, p.c);
          else mma_block(tog);
          phase_fence();
          tog = 1 - tog;
          kr = slab_rsrc(kr, kstep, true);
          vr = slab_rsrc(vr, vstep, true);
          wait_vm_lds_barrier<0>();
          phase_fence();
        }
      }
      for (; j <= nsteps; ++j) {
        issue_k(j + 1);
        issue_v(j);
        if (j <= wsteps) {
          if (grp == 0) mma_block(j & 1);
          else softmax_block(j - 1);
        }
        wait_vm_lds_barrier<63>();
        if (j <= wsteps) {
          if (grp == 0) softmax_block(j);
          else mma_block(j & 1);
        }
        wait_vm_lds_barrier<0>();
      }
      // The groups' halves meet: each keeps one half of the d tiles and gets the other group's sums of
      // them through LDS (the ring is free after the last barrier), with its row offset and row sum.
      constexpr int HT = DTL / 2, keep0 = grp * HT, give0 = (1 - grp) * HT;
      float* const ex = reinterpret_cast<float*>(smem);
      constexpr int kStats = 8 * HT * QT * 256;  // floats before the (m, l) pairs
      static_assert((kStats + 8 * QT * 128) * 4 <= 4 * (KT_ELEMS + VT_ELEMS) * 2, "exchange fits the ring");
      float l[QT];
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        l[qt] = kSumMfma ? lsum[qt][0] : xquad_sum(l_i[qt]);
#pragma unroll
        for (int i = 0; i < HT; ++i)
          *reinterpret_cast<floatx4*>(ex + ((wave * HT + i) * QT + qt) * 256 + lane * 4) = acc[give0 + i][qt];
        ex[kStats + (wave * QT + qt) * 128 + lane] = ro.m[qt];
        ex[kStats + (wave * QT + qt) * 128 + 64 + lane] = l[qt];
      }
      __syncthreads();
      const int peer = wave ^ 4;
      constexpr float kLn2 = 0.69314718055994530942f;
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        const float m1 = ex[kStats + (peer * QT + qt) * 128 + lane], l1 = ex[kStats + (peer * QT + qt) * 128 + 64 + lane];
        const float m = fmaxf(ro.m[qt], m1);
        const float a0 = ro.m[qt] == FA_NEG_INF ? 0.f : fast_exp2((ro.m[qt] - m) * p.c);
        const float a1 = m1 == FA_NEG_INF ? 0.f : fast_exp2((m1 - m) * p.c);
        const float lt = l[qt] * a0 + l1 * a1;
        const float inv = lt > 0.f ? 1.f / lt : 0.f;
        const float lse_val = lt > 0.f ? (m * p.c + __builtin_amdgcn_logf(lt)) * kLn2 : FA_NEG_INF;
        floatx4 out[HT];
#pragma unroll
        for (int i = 0; i < HT; ++i) {
          const floatx4 x = *reinterpret_cast<const floatx4*>(ex + ((peer * HT + i) * QT + qt) * 256 + lane * 4);
#pragma unroll
          for (int r = 0; r < 4; ++r) out[i][r] = (acc[keep0 + i][qt][r] * a0 + x[r] * a1) * inv;
        }
        u32x4 wide[HT / 2];
        if constexpr (!SPLIT) {  // 64-byte row pieces, as pack_o_wide; cross-lane: before the row test
#pragma unroll
          for (int pp = 0; pp < HT / 2; ++pp) {
            const floatx4 &a = out[2 * pp], &c = out[2 * pp + 1];
            const auto lo = __builtin_amdgcn_permlane16_swap(T::pack2(a[0], a[1]), T::pack2(c[0], c[1]), false, false);
            const auto hi2 = __builtin_amdgcn_permlane16_swap(T::pack2(a[2], a[3]), T::pack2(c[2], c[3]), false, false);
            wide[pp] = (u32x4){lo[0], hi2[0], lo[1], hi2[1]};
          }
        }
        const int i = wrow0 + qt * 16 + q16;
        if (i < rows) {
          const int hr = p.pack > 1 ? h + i / p.M : h, mr = p.pack > 1 ? i % p.M : i;
          if constexpr (SPLIT) {
            const int64_t wrow = (int64_t)(split * p.B + b) * p.H + hr;
            float* wo = p.ws_o + (wrow * p.M + mr) * D + keep0 * 16 + 4 * g;
#pragma unroll
            for (int d = 0; d < HT; ++d) *reinterpret_cast<floatx4*>(wo + d * 16) = out[d];
            if (grp == 0 && g == 0) p.ws_lse[wrow * p.M + mr] = lse_val;
          } else {
            uint16_t* orow = p.o + (int64_t)b * p.so0 + (int64_t)hr * p.so1 + (int64_t)mr * p.so2 + keep0 * 16;
#pragma unroll
            for (int pp = 0; pp < HT / 2; ++pp) *reinterpret_cast<u32x4*>(orow + 32 * pp + wide_col(g)) = wide[pp];
            if (p.lse != nullptr && grp == 0 && g == 0)
              p.lse[(int64_t)b * p.sl0 + (int64_t)hr * p.sl1 + (int64_t)mr * p.sl2] = lse_val;
          }
        }
      }
    };
    if (wave < 4) run_group(std::integral_constant<int, 0>{});
    else run_group(std::integral_constant<int, 1>{});
  }
};

template <typename Tag, int D, int WAVES, int BN, int PIPE, bool SPLIT>
__global__ __launch_bounds__(WAVES * 64, (Fwd16<Tag, D, WAVES, BN, PIPE, SPLIT>::kBlocksPerCu)) void fa_fwd16_kernel(
    FwdParams p) {
  static_assert(kernel_has_sole_arg<FwdParams>(&fa_fwd16_kernel<Tag, D, WAVES, BN, PIPE, SPLIT>),
                "the epilogues read FwdParams from kernel-argument offset 0: it must stay the only argument");
  if constexpr (PIPE == 4)
    Fwd16<Tag, D, WAVES, BN, PIPE, SPLIT>::run_key_groups(p);
  else if constexpr (PIPE == 3)
    Fwd16<Tag, D, WAVES, BN, PIPE, SPLIT>::run_persistent(p);
  else
    Fwd16<Tag, D, WAVES, BN, PIPE, SPLIT>::run(p);
}

// The basic variant's kernels (stages=1): the bodies above under the basic tiles. 256 rows and 8 waves run
// the persistent ping-pong (a tile of stages=8 the dispatched one instead, whose kernel is the registry's
// own), 128 rows and 4 waves the software pipeline, D = 256 the lean pipeline on 32-key tiles. The
// kernels they replace kept one K/V buffer, filled through registers, with two
// barriers per tile and 32x32x16 MFMAs: fp16 B4 H32 D128 N=8192 4.29 -> 3.41 ms, causal N=2048 209 -> 143
// us, bf16 B2 H16 D256 N=2048 180 -> 120 us.
template <typename Tag, int D, int WAVES, int BN, int STAGES, bool SPLIT>
__global__ __launch_bounds__(WAVES * 64, WAVES == 8 ? 1 : 2) void fa_basic_kernel(FwdParams p) {
  static_assert(kernel_has_sole_arg<FwdParams>(&fa_basic_kernel<Tag, D, WAVES, BN, STAGES, SPLIT>),
                "the epilogues read FwdParams from kernel-argument offset 0: it must stay the only argument");
  static_assert(STAGES == 1 && BN == 64 && !SPLIT, "basic tiles");
  if constexpr (WAVES == 8)
    Fwd16<Tag, D, 8, 64, 3, false>::run_persistent(p);
  else if constexpr (D <= 128)
    Fwd16<Tag, D, 4, 64, 1, false>::run(p);
  else
    Fwd16<Tag, D, 4, 32, 0, false>::template run<true>(p);
}

// Registry (stages=6: PIPE 0, stages=7: PIPE 1, stages=8: PIPE 2 and stages=9: PIPE 3 with 8 waves;
// 32 query rows per wave).
#define FA16_SYM_TAG_f16_t "5f16_t"
#define FA16_SYM_TAG_bf16_t "6bf16_t"
#define FA16_SYMBOL(TAG, D, W, BN, PI, SP)                                                                    \
  "_ZN2fa15fa_fwd16_kernelINS_" FA16_SYM_TAG_##TAG "ELi" #D "ELi" #W "ELi" #BN "ELi" #PI "ELb" #SP \
  "EEEvNS_9FwdParamsE"
#define FA16_ENTRY(TAG, DTYPE, D, W, BN, PI, SP)                                                         \
  {6 + PI, DTYPE, D, W, 32, BN, SP, (const void*)&fa_fwd16_kernel<TAG, D, W, BN, PI, (SP != 0)>, \
   FA16_SYMBOL(TAG, D, W, BN, PI, SP)}
#define FA16_PAIR(TAG, DTYPE, D, BN, PI) FA16_ENTRY(TAG, DTYPE, D, 4, BN, PI, 0), FA16_ENTRY(TAG, DTYPE, D, 4, BN, PI, 1)
#define FA16_PAIR8(TAG, DTYPE, D, BN, PI) FA16_ENTRY(TAG, DTYPE, D, 8, BN, PI, 0), FA16_ENTRY(TAG, DTYPE, D, 8, BN, PI, 1)
// key groups: 8 waves on 128 rows
#define FA16_KG_ENTRY(TAG, DTYPE, D, SP)                                                                    \
  {10, DTYPE, D, 8, 16, 64, SP, (const void*)&fa_fwd16_kernel<TAG, D, 8, 64, 4, (SP != 0)>, \
   FA16_SYMBOL(TAG, D, 8, 64, 4, SP)}
#define FA16_KG_PAIR(TAG, DTYPE, D) FA16_KG_ENTRY(TAG, DTYPE, D, 0), FA16_KG_ENTRY(TAG, DTYPE, D, 1)
#define FA16_ENTRIES(TAG, DTYPE, D)                                                             \
  FA16_PAIR(TAG, DTYPE, D, 64, 0), FA16_PAIR(TAG, DTYPE, D, 32, 0), FA16_PAIR(TAG, DTYPE, D, 64, 1), \
      FA16_PAIR(TAG, DTYPE, D, 32, 1), FA16_PAIR8(TAG, DTYPE, D, 64, 2), FA16_PAIR8(TAG, DTYPE, D, 64, 3), \
      FA16_KG_PAIR(TAG, DTYPE, D)

#define FA16_BASIC(TAG, DTYPE, D, W, BODY, BODY_BN)                                                    \
  {1, DTYPE, D, W, 32, 64, 0, (const void*)&fa_basic_kernel<TAG, D, W, 64, 1, false>,                 \
   "_ZN2fa15fa_basic_kernelINS_" FA16_SYM_TAG_##TAG "ELi" #D "ELi" #W "ELi64ELi1ELb0EEEvNS_9FwdParamsE", BODY, BODY_BN}
#define FA16_BASICS(TAG, DTYPE)                                                                 \
  FA16_BASIC(TAG, DTYPE, 64, 8, 9, 64), FA16_BASIC(TAG, DTYPE, 64, 4, 7, 64), FA16_BASIC(TAG, DTYPE, 128, 8, 9, 64), \
      FA16_BASIC(TAG, DTYPE, 128, 4, 7, 64), FA16_BASIC(TAG, DTYPE, 256, 4, 6, 32)

static const FaKernelEntry kFwd16Entries[] = {
    FA16_BASICS(f16_t, FA_DTYPE_F16),             FA16_BASICS(bf16_t, FA_DTYPE_BF16),
    FA16_ENTRIES(f16_t, FA_DTYPE_F16, 64),        FA16_ENTRIES(f16_t, FA_DTYPE_F16, 128),
    FA16_ENTRIES(bf16_t, FA_DTYPE_BF16, 64),      FA16_ENTRIES(bf16_t, FA_DTYPE_BF16, 128),
    // D = 256: one tile per step only (the pipelined kernel's two score tiles do not fit beside O
    // and Q in 256 registers)
    FA16_PAIR(f16_t, FA_DTYPE_F16, 256, 32, 0),   FA16_PAIR(bf16_t, FA_DTYPE_BF16, 256, 32, 0),
};

const FaKernelEntry* fa_fwd16_registry(int* count) {
  *count = (int)(sizeof(kFwd16Entries) / sizeof(kFwd16Entries[0]));
  return kFwd16Entries;
}

}  // namespace fa
