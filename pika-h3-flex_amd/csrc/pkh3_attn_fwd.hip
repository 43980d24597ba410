// Non-causal flash-style attention forward for gfx950 (CDNA4), head dim 128.
//
// Work split.  A workgroup is 12 waves (dense; three per SIMD) or 8 waves (block-sparse; two per SIMD);
// each wave owns 32 queries of one (batch, head) and keeps for them, in VGPRs, the Q operand images, the
// running row max / row sum and the fp32 output accumulator O^T (128 x 32, sixteen 16x16 blocks).  All waves share every 64-key
// K/V tile, which is copied HBM/L2 -> LDS with direct-to-LDS loads into a 3-slot ring, two tiles ahead of
// the math.  Several waves per SIMD is what overlaps the softmax VALU work of one wave with the MFMAs of
// another; the whole per-wave state stays in VGPRs (<= 168 dense, <= 256 sparse) so no accumulator ever
// moves between register files.  Q is read in place: RMSNorm, rotation and fp8 quantisation of the Q rows
// happen in registers while the first K/V tiles are in flight.
//
// Math per tile, all on the 16x16 MFMA shapes (see pkh3_common.h for the operand images and why these shapes):
//   S^T = K' Q'^T      A = K image (LDS), B = Q image (VGPR)      -> lane l holds queries l%16 and 16 + l%16, 4 keys
//                      per 16-key block (bf16: 32 x 16x16x32, Q' carries softmax_scale * log2(e) so S^T is in the
//                      log2 domain; fp8: 8 x 16x16x128 on e4m3 images, S^T rescaled by the per-64-row-block
//                      dequantisation scales in the softmax multiply)
//   softmax            bounded-logit path (the usual one): |q_i| * max_j |k_j| bounds every logit of the wave's
//                      queries; when that bound is small, exp2(logit) needs no maximum at all.  Otherwise the
//                      online form: row max in-lane over the keys + two row swaps across the four lane groups,
//                      raised only when exceeded by 2^8 so the O^T rescale is rare.  Row sum kept per lane group,
//                      merged once at the end.
//   O^T += V^T P^T     A = V image (LDS), B = P packed to bf16 straight from the S^T registers (32 x 16x16x32)
// The transposed formulation keeps every per-query quantity (max, sum, rescale factor) a per-lane
// scalar: no cross-lane traffic in the rescale, none between the two GEMMs.  O leaves through LDS, turned
// around into whole 256-byte rows.
//
// Other forms of the dense kernel (see attn_fwd_body): the short-key form (few key tiles, or few queries: 4 waves per
// workgroup, 32-key half tiles, three workgroups per CU), the narrow form (fewer queries still: one 32-query block per
// workgroup, its waves share the keys out; attn_fwd_narrow_kernel), the relay form (many queries, few to some dozens of key tiles: a workgroup
// per CU goes from one block of queries to the next; attn_fwd_relay_kernel), and the long form with the key tiles of a unit shared out
// among several workgroups that merge through global scratch, for a thinly filled last round of a long call.
//
// Block-sparse variant.  A workgroup covers 4 query row-blocks (64 queries each, a wave pair per row-block).
// Phase 1 walks the key tiles all four row-blocks keep, exactly like the dense kernel.  Phase 2 walks the
// remaining tiles per row-block: every iteration gives each wave pair one 32-key half of a tile of its own
// list in its own LDS area, so all 8 waves stay busy.  The lists are made on
// the device by the first workgroups of the K/V pass, for calls on prepared keys by a launch of their own (pkh3_plan.h).
#include <float.h>
#include <limits.h>
#include <math.h>

#include <atomic>
#include <type_traits>

#include "pkh3_common.h"
#include "pkh3_index.h"
#include "pkh3_internal.h"

namespace pkh3 {

constexpr int kDenseWaves = 12;  // dense kernel: three waves per SIMD (<= 168 VGPRs each), 384 queries per workgroup
constexpr int kShortWaves = 4;   // short-key dense kernel: three 4-wave workgroups per CU
constexpr int kMaxParts = 8;     // long dense form: most workgroups a unit's key tiles are shared out among ...
constexpr int kMinPartTiles = 24;  // ... and fewest key tiles such a workgroup is worth starting for
constexpr int kSparseWaves = 2 * kSparseRows;  // block-sparse: a wave pair per row-block; one such workgroup on a CU (96 to 128 KiB of LDS)
constexpr int kRing = 3;               // LDS ring depth (tiles)
constexpr int kStages2 = 2;            // block-sparse phase 2: stages of row-private half tiles
constexpr int kPipeRing = 4;           // ... of the pipelined short-key form (32-key halves)
constexpr float kRescaleSlack = 8.0f;  // the running max is only raised when exceeded by 2^8
// The running max before the first key.  Finite: keys whose logits are all -inf then weigh exp2(-inf - max) = 0, wherever
// among a wave's keys they lie, and two shares without a key meet as exp2(0) times a row sum of 0.
constexpr float kNoMax = -FLT_MAX;
constexpr float kStaticMaxLimit = 48.0f;  // rows whose |logit| bound is below this skip the running max (terms 2^-48 .. 2^48)

#define PKH3_SGB(mask, n) __builtin_amdgcn_sched_group_barrier(mask, n, 0)
// Each tile loop ends on an MFMA into the O^T accumulators.  The compiler was seen to place the register
// copies that merge the two loop variants (v_mov_b64 reading the accumulator's last registers) four scalar
// instructions after that MFMA, before its result is written back; the block-sparse kernel then returned a stale
// O^T block.  32 idle issue cycles after every loop let the last MFMA retire whatever follows.  The accumulators
// are operands of the statement, so every read or copy of them the compiler emits after the loop is ordered
// after the idle cycles.
#define PKH3_MFMA_DRAIN(W)                                                                                               \
  asm volatile("s_nop 15\n\ts_nop 15"                                                                                    \
               : "+v"((W).o[0][0]), "+v"((W).o[0][1]), "+v"((W).o[1][0]), "+v"((W).o[1][1]), "+v"((W).o[2][0]),          \
                 "+v"((W).o[2][1]), "+v"((W).o[3][0]), "+v"((W).o[3][1]), "+v"((W).o[4][0]), "+v"((W).o[4][1]),          \
                 "+v"((W).o[5][0]), "+v"((W).o[5][1]), "+v"((W).o[6][0]), "+v"((W).o[6][1]), "+v"((W).o[7][0]),          \
                 "+v"((W).o[7][1])::"memory")
constexpr int kSgMfma = 0x008, kSgDsRead = 0x100;

__device__ __forceinline__ void lds_dma16(const char* g, unsigned lane_off, char* l) {
  // 64 lanes x 16 B, global -> LDS without passing through VGPRs: lane i copies g[lane_off_i .. +16) to
  // l + i*16.  `g` and `l` are wave-uniform (the address arithmetic stays on the scalar unit), `lane_off` is
  // the per-lane byte offset.
  // Issued through inline assembly on purpose: once the compiler sees a direct-to-LDS load it stops trusting
  // the in-order LDS counter and turns every later wait on an LDS read into lgkmcnt(0), which serialises the
  // operand image reads.  Completion is tracked by hand: the s_waitcnt vmcnt(0) at the top of each tile loop.
  const unsigned lds_addr = (unsigned)(size_t)(__attribute__((address_space(3))) char*)l;
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(lane_off), "s"(g), "s"(lds_addr)
               : "memory", "m0");
}

// Wave-uniform reads of tables earlier kernels wrote (tile lists, fp8 scales): through the scalar cache, so
// they count on lgkmcnt and never make the wave wait for its outstanding HBM->LDS copies (vmcnt).
template <typename T>
__device__ __forceinline__ T uniform_load(const T* p, int i) {
  return ((const __attribute__((address_space(4))) T*)p)[i];
}

// Stores and loads that are coherent across the whole device (all XCDs) one by one: they go past the caches that
// are not, so data handed from one workgroup to another needs no cache write-back or invalidation around it --
// only the writer's wait for its stores before it signals, and the reader's signal check before its loads.
__device__ __forceinline__ void store_device(float* p, f32x4 v) {
  const unsigned long long lo = ((unsigned long long)__float_as_uint(v[1]) << 32) | __float_as_uint(v[0]);
  const unsigned long long hi = ((unsigned long long)__float_as_uint(v[3]) << 32) | __float_as_uint(v[2]);
  __hip_atomic_store((unsigned long long*)p, lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store((unsigned long long*)p + 1, hi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_device(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ f32x4 load_device4(const float* p) {
  const unsigned long long lo = __hip_atomic_load((const unsigned long long*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const unsigned long long hi = __hip_atomic_load((const unsigned long long*)p + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return f32x4{__uint_as_float((unsigned)lo), __uint_as_float((unsigned)(lo >> 32)), __uint_as_float((unsigned)hi),
               __uint_as_float((unsigned)(hi >> 32))};
}
__device__ __forceinline__ float load_device(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Per-wave state.  Lane (c = l % 16, g = l / 16) works for the two queries 16*qb + c, qb = 0, 1, of the wave's 32.
template <bool FP8>
struct WaveState {
  bf16x8 qf[FP8 ? 1 : 2][FP8 ? 1 : 4];  // bf16 Q images (qb, ks): Q'[16*qb + c][32*ks + 8*g + j]
  i32x8 q8[FP8 ? 2 : 1];                // fp8 Q images (qb): bytes 8*ks + j = element 32*ks + 8*g + j
  f32x4 s[4][2];                        // S^T of the tile (kb, qb): keys 16*kb + 4*g + i
  f32x4 o[8][2];                        // O^T accumulators (db, qb): head-dim rows 16*db + 4*g + i
  bf16x8 vf[8];                         // V images of the first 32 keys, fetched while QK^T finishes
  float m[2], l[2];                     // per query block: running row max (scaled, log2 domain), this lane group's row sum
  int qe;                               // fp8 with power-of-two scales: exponent byte (E8M0) of the Q block's scale
};

// One 16-row block of queries with its rotation tables, as they lie in memory.  Rows past the end are the last one again: what is made of
// them is not stored, and neither the largest magnitude of their 64 queries nor any bound is another for it.
struct QRows {
  Rows16 q, cos, sin;
};
template <typename Params>
__device__ __forceinline__ void ask_q_rows(QRows& r, const Params& p, int b, int h, int first, int lane) {
  ask_rows16(r.q, (const char*)p.q + ((int64_t)b * p.q_sb + (int64_t)h * p.q_sh) * 2, p.q_ss * 2, first, p.Sq - 1, lane);
  if (p.q_rope_mode != 0) {
    ask_rows16(r.cos, (const char*)p.q_cos, kD / 2 * sizeof(float), first, p.Sq - 1, lane);
    ask_rows16(r.sin, (const char*)p.q_sin, kD / 2 * sizeof(float), first, p.Sq - 1, lane);
  }
}
// RMSNorm, rotation and `factor` of such a block, through 4 KiB of LDS of the wave's own: lane (c, g) gets its 32 elements of row c
template <typename Params>
__device__ __forceinline__ void q_rows_ready(float (&x)[32], const QRows& r, const Params& p, const NormLanes& norm, float factor, char* lds, int lane) {
  bf16x8 raw[4];
  turn_elements(r.q, raw, lds, lane);
  RopeQuarter rope;
  if (p.q_rope_mode != 0) {
    turn_table(r.cos, rope.c, p.q_rope_mode, lds, lane);
    turn_table(r.sin, rope.s, p.q_rope_mode, lds, lane);
  }
  norm_row(x, raw, p.q_norm_w != nullptr, p.q_eps, norm, factor);
  rope_row(x, p.q_rope_mode, rope);
}

// Consecutive MFMAs share an operand where they can: the two query blocks of an image come in turn (0 1, 1 0, 0 1 ..), so that only
// one of the operands changes from one to the next.  Less toggles in the matrix unit, at a clock that is set by power: 480p 19.82 ->
// 19.66 ms, 768p 130.1 -> 128.9, 14,830 + 512 rows 2,149 -> 2,138 us, with the projection's GEMMs (the same) a block of them 3,168 -> 3,145
// (means of two comparisons on one card); fp8 and short calls the same.
#define PKH3_MFMA16(A, B, C) __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, B, C, 0, 0, 0)
// format codes 0/0 = e4m3 x e4m3; scale operands 0 select the unscaled form of the instruction
#define PKH3_MFMA16_F8(A, B, C) __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(A, B, C, 0, 0, 0, 0, 0, 0)
// the scaled form: the product is multiplied by 2^(EA - 127) * 2^(EB - 127), EA / EB = byte 0 of each lane's scale
// operand (every lane passes the same exponents: one scale per 64-row block, not per 32 elements)
#define PKH3_MFMA16_F8S(A, B, C, EA, EB) __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(A, B, C, 0, 0, 0, EA, 0, EB)

// S^T = K' Q'^T for the 64 keys of one tile: image i of the K tile is (half, ks, kb2) = (i >> 3, (i >> 1) & 3, i & 1)
// and feeds the two query blocks, so four accumulators rotate inside each half.  LDS reads run 8 images ahead of
// the MFMAs that consume them; the tail of the MFMA chain covers the first V image reads.
// LEAN (three waves per SIMD, 168 VGPRs): the reads run only 4 images ahead and V is left to the P.V loop.
// AHEAD: images the LEAN reads run ahead (the copies of the loop that run once per workgroup take 2 and fit the registers)
// POW2 (fp8): the block scales are powers of two and go into the MFMA as its scale operands (`ke`: exponent byte of
// this K tile's scale), so S^T leaves the MFMA dequantised.
// MASKED (lean bf16 form): the sums start from -inf instead of 0 for keys from `lim` on, which costs the softmax nothing.
template <bool FP8, bool LEAN, int AHEAD = 4, bool POW2 = false, bool MASKED = false>
__device__ __forceinline__ void qk_tile(WaveState<FP8>& w, const char* kbuf, const char* vbuf, int lane, int ke = 0, int lim = 0) {
  static_assert(!MASKED || (!FP8 && LEAN), "the forms that ask for it");
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  if constexpr (MASKED) {
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) w.s[kb][0][i] = w.s[kb][1][i] = 16 * kb + 4 * (lane >> 4) + i >= lim ? -INFINITY : 0.f;
  }
  if constexpr (!FP8 && LEAN) {
    bf16x8 kf[16];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) kf[i] = *(const bf16x8*)(kbuf + (i * 64 + lane) * 16);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int ks = (i >> 1) & 3, kb = 2 * (i >> 3) + (i & 1);
#pragma unroll
      for (int q = 0, qb = i & 1; q < 2; ++q, qb ^= 1) w.s[kb][qb] = PKH3_MFMA16(kf[i], w.qf[qb][ks], ks == 0 && !MASKED ? zero : w.s[kb][qb]);
      if (i + AHEAD < 16) kf[i + AHEAD] = *(const bf16x8*)(kbuf + ((i + AHEAD) * 64 + lane) * 16);
    }
    PKH3_SGB(kSgDsRead, AHEAD);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      PKH3_SGB(kSgMfma, 2);
      if (i + AHEAD < 16) PKH3_SGB(kSgDsRead, 1);
    }
  } else if constexpr (!FP8) {
    bf16x8 kf[16];
#pragma unroll
    for (int i = 0; i < 8; ++i) kf[i] = *(const bf16x8*)(kbuf + (i * 64 + lane) * 16);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int ks = (i >> 1) & 3, kb = 2 * (i >> 3) + (i & 1);
#pragma unroll
      for (int q = 0, qb = i & 1; q < 2; ++q, qb ^= 1) w.s[kb][qb] = PKH3_MFMA16(kf[i], w.qf[qb][ks], ks == 0 ? zero : w.s[kb][qb]);
      if (i < 8)
        kf[i + 8] = *(const bf16x8*)(kbuf + ((i + 8) * 64 + lane) * 16);
      else
        w.vf[i - 8] = *(const bf16x8*)(vbuf + ((i - 8) * 64 + lane) * 16);
    }
    PKH3_SGB(kSgDsRead, 8);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      PKH3_SGB(kSgMfma, 2);
      PKH3_SGB(kSgDsRead, 1);
    }
  } else {
    i32x4 kc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) kc[i] = *(const i32x4*)(kbuf + (i * 64 + lane) * 16);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const i32x4 a0 = kc[2 * kb], a1 = kc[2 * kb + 1];
      const i32x8 a = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
        w.s[kb][qb] = POW2 ? PKH3_MFMA16_F8S(a, w.q8[qb], zero, ke, w.qe) : PKH3_MFMA16_F8(a, w.q8[qb], zero);
      // the MFMA chain covers the first V image reads: 8 images, or 4 where registers are short (LEAN)
      if constexpr (LEAN) {
        w.vf[kb] = *(const bf16x8*)(vbuf + (kb * 64 + lane) * 16);
      } else {
        w.vf[2 * kb] = *(const bf16x8*)(vbuf + ((2 * kb) * 64 + lane) * 16);
        w.vf[2 * kb + 1] = *(const bf16x8*)(vbuf + ((2 * kb + 1) * 64 + lane) * 16);
      }
    }
  }
}

// exp2 of one logit.  bf16 path, and fp8 with power-of-two scales: Q' already carries softmax_scale * log2(e) (and the
// MFMA applied the scales), so S^T is in the log2 domain and `c` is unused; fp8 with absmax scales (MUL): `c` carries
// that factor times the dequantisation scales.  STATIC: the logits are bounded in magnitude (see kStaticMaxLimit), so
// no maximum is subtracted at all.
template <bool MUL, bool STATIC>
__device__ __forceinline__ float softmax_numerator(float s, float c, float m) {
  if constexpr (MUL) return __builtin_amdgcn_exp2f(STATIC ? s * c : fmaf(s, c, -m));
  else return __builtin_amdgcn_exp2f(STATIC ? s : s - m);
}

// Softmax numerators of NKB key blocks of w.s (a whole tile: 4, a 32-key half: 2), from block AT on, into the P^T operands of
// the P.V MFMAs: operand (half, qb) takes, for lane group g, the keys v_image_key(g, j) of its half, i.e. registers
// 0..3 of key block 2*half and of key block 2*half + 1 -- P never leaves its lane.  Also the running max / rescale
// of the online path and the row sums.  `lim` = keys of these blocks that exist (only read when MASKED).
// STATIC: w.m is not used: every logit is bounded (|q_i| * max_j |k_j| * c), small enough that exp2(logit) is a
// normal number; the running max, its exchange across the lane groups and the O^T rescale are then not needed at
// all, and the numerators of the first 32 keys do not wait for the second half of S^T.
// FIRST: nothing has been summed up yet.
template <bool FP8, bool STATIC, bool MASKED, int NKB, bool POW2 = false, int AT = 0, bool FIRST = false>
__device__ __forceinline__ void softmax_blocks(WaveState<FP8>& w, bf16x8 (&pf)[NKB / 2][2], float c, int lim, int lane) {
  constexpr bool MUL = FP8 && !POW2;  // the logits still need their dequantisation scales
  const int g = lane >> 4;
  if (MASKED) {
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (16 * kb + 4 * g + i >= lim) {
          w.s[AT + kb][0][i] = -INFINITY;
          w.s[AT + kb][1][i] = -INFINITY;
        }
  }
  float m_new[2] = {w.m[0], w.m[1]}, alpha[2] = {1.0f, 1.0f};
  if constexpr (!STATIC) {
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      float mx = w.s[AT][qb][0];
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, w.s[AT + kb][qb][i]);
      mx = max_across_groups(mx) * (MUL ? c : 1.0f);
      m_new[qb] = (mx > w.m[qb] + kRescaleSlack) ? mx : w.m[qb];
      alpha[qb] = __builtin_amdgcn_exp2f(w.m[qb] - m_new[qb]);
      w.m[qb] = m_new[qb];
    }
    if (!FIRST && __any(alpha[0] != 1.0f || alpha[1] != 1.0f)) {
#pragma unroll
      for (int db = 0; db < 8; ++db)
#pragma unroll
        for (int qb = 0; qb < 2; ++qb)
#pragma unroll
          for (int i = 0; i < 4; ++i) w.o[db][qb][i] *= alpha[qb];
    }
  }
  const bf16x2 one2 = {(__bf16)1.0f, (__bf16)1.0f};
  float rsum[2] = {0.f, 0.f};
#pragma unroll
  for (int half = 0; half < NKB / 2; ++half)
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      bf16x8 pk;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        pk[j] = (__bf16)softmax_numerator<MUL, STATIC>(w.s[AT + 2 * half + (j >> 2)][qb][j & 3], c, m_new[qb]);
      // row sum over the bf16-rounded values, the same numbers the P.V MFMA consumes
#pragma unroll
      for (int j = 0; j < 8; j += 2) {
        const bf16x2 pr = {pk[j], pk[j + 1]};
        rsum[qb] = __builtin_amdgcn_fdot2_f32_bf16(pr, one2, rsum[qb], false);
      }
      pf[half][qb] = pk;
    }
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) w.l[qb] = FIRST ? rsum[qb] : STATIC ? w.l[qb] + rsum[qb] : w.l[qb] * alpha[qb] + rsum[qb];
}

// Softmax of w.s, then O^T += V^T P^T for one tile: V image i is (half, db) = (i >> 3, i & 7) and feeds the two
// query blocks, sixteen accumulators in rotation.  `c` = softmax scale * log2(e) (times the fp8 dequantisation
// scales of this tile); `lim` = keys of this tile that exist (only read when MASKED).
template <bool FP8, bool STATIC, bool LEAN, bool MASKED, bool POW2 = false, bool FIRST = false>
__device__ __forceinline__ void softmax_pv_tile(WaveState<FP8>& w, const char* vbuf, float c, int lim, int lane) {
  static_assert(!FIRST || LEAN, "the forms that ask for it");
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  bf16x8 pf[2][2];
  softmax_blocks<FP8, STATIC, MASKED, 4, POW2, 0, FIRST>(w, pf, c, lim, lane);
  if constexpr (LEAN) {
    bf16x8 vg[16];
#pragma unroll
    for (int i = 0; i < 4; ++i) vg[i] = FP8 ? w.vf[i] : *(const bf16x8*)(vbuf + (i * 64 + lane) * 16);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
#pragma unroll
      for (int q = 0, qb = i & 1; q < 2; ++q, qb ^= 1) w.o[i & 7][qb] = PKH3_MFMA16(vg[i], pf[i >> 3][qb], FIRST && i < 8 ? zero : w.o[i & 7][qb]);
      if (i + 4 < 16) vg[i + 4] = *(const bf16x8*)(vbuf + ((i + 4) * 64 + lane) * 16);
    }
  } else {
    bf16x8 vg[8];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
#pragma unroll
      for (int q = 0, qb = i & 1; q < 2; ++q, qb ^= 1) w.o[i & 7][qb] = PKH3_MFMA16(i < 8 ? w.vf[i] : vg[i - 8], pf[i >> 3][qb], w.o[i & 7][qb]);
      if (i < 8) vg[i] = *(const bf16x8*)(vbuf + ((i + 8) * 64 + lane) * 16);
    }
  }
}

// ---- 32-key half tiles: the short-key form of the dense kernel, phase 2 of the block-sparse one ----
// S^T (32 keys x 32 queries) into w.s[AT..AT + 1]; kbuf/vbuf point at this half's K images (8 bf16 / 4 fp8 chunks)
// and V images (8).
// LEAN (three waves per SIMD): the K reads run 4 images ahead and only the fp8 path prefetches V (4 images).
template <bool FP8, bool LEAN = false, bool POW2 = false, int AT = 0>
__device__ __forceinline__ void qk_half(WaveState<FP8>& w, const char* kbuf, const char* vbuf, int lane, int ke = 0) {
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  if constexpr (!FP8 && LEAN) {
    bf16x8 kf[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) kf[i] = *(const bf16x8*)(kbuf + (i * 64 + lane) * 16);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
      for (int q = 0, qb = i & 1; q < 2; ++q, qb ^= 1) w.s[AT + (i & 1)][qb] = PKH3_MFMA16(kf[i], w.qf[qb][i >> 1], i < 2 ? zero : w.s[AT + (i & 1)][qb]);
      if (i + 4 < 8) kf[i + 4] = *(const bf16x8*)(kbuf + ((i + 4) * 64 + lane) * 16);
    }
  } else if constexpr (!FP8) {
    bf16x8 kf[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) kf[i] = *(const bf16x8*)(kbuf + (i * 64 + lane) * 16);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
      for (int q = 0, qb = i & 1; q < 2; ++q, qb ^= 1) w.s[AT + (i & 1)][qb] = PKH3_MFMA16(kf[i], w.qf[qb][i >> 1], i < 2 ? zero : w.s[AT + (i & 1)][qb]);
      w.vf[i] = *(const bf16x8*)(vbuf + (i * 64 + lane) * 16);
    }
  } else {
    i32x4 kc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) kc[i] = *(const i32x4*)(kbuf + (i * 64 + lane) * 16);
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      const i32x4 a0 = kc[2 * kb], a1 = kc[2 * kb + 1];
      const i32x8 a = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
        w.s[AT + kb][qb] = POW2 ? PKH3_MFMA16_F8S(a, w.q8[qb], zero, ke, w.qe) : PKH3_MFMA16_F8(a, w.q8[qb], zero);
#pragma unroll
      for (int i = 0; i < (LEAN ? 2 : 4); ++i) {
        const int v = (LEAN ? 2 : 4) * kb + i;
        w.vf[v] = *(const bf16x8*)(vbuf + (v * 64 + lane) * 16);
      }
    }
  }
}

// Softmax numerators of w.s[AT..AT + 1] and O^T += V^T P^T for one half tile (V images already in w.vf).
// `lim` = keys of this half that exist (<= 0: none; only read when < 32).
// LEAN: the V images (beyond the 4 the fp8 path prefetched) are read here, 4 ahead of their MFMAs, from vbuf.
// FULL: the caller guarantees lim == 32, no masking code at all.
template <bool FP8, bool STATIC, bool LEAN = false, bool FULL = false, bool POW2 = false, int AT = 0>
__device__ __forceinline__ void softmax_pv_half(WaveState<FP8>& w, float c, int lim, int lane, const char* vbuf = nullptr) {
  bf16x8 pf[1][2];
  // the running-max form always takes the masking copy (two copies of it do not fit the registers of some variants)
  if (!FULL && (!STATIC || lim < 32)) softmax_blocks<FP8, STATIC, true, 2, POW2, AT>(w, pf, c, lim, lane);
  else softmax_blocks<FP8, STATIC, false, 2, POW2, AT>(w, pf, c, lim, lane);
  if constexpr (LEAN) {
    bf16x8 vg[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) vg[i] = FP8 ? w.vf[i] : *(const bf16x8*)(vbuf + (i * 64 + lane) * 16);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
      for (int q = 0, qb = i & 1; q < 2; ++q, qb ^= 1) w.o[i][qb] = PKH3_MFMA16(vg[i], pf[0][qb], w.o[i][qb]);
      if (i + 4 < 8) vg[i + 4] = *(const bf16x8*)(vbuf + ((i + 4) * 64 + lane) * 16);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int q = 0, qb = i & 1; q < 2; ++q, qb ^= 1) w.o[i][qb] = PKH3_MFMA16(w.vf[i], pf[0][qb], w.o[i][qb]);
  }
}

// The largest K' row norm of a (batch, head) over its `n` 32-key halves, in two parts: the first 256 halves are asked for ahead of
// time (`first`), the wave's lanes meet where the number is needed.
template <typename Params>
__device__ __forceinline__ f32x4 ask_key_norms(const Params& p, int bh, int lane) {
  return *(const f32x4*)(p.knorm + (int64_t)bh * p.knorm_stride + min(kNormFirst + 4 * lane, p.knorm_stride - 4));
}
// AT_ONCE: steps of the walk behind them that are on their way together.  One after the other they cost a block of 64 queries against 500,000
// keys (narrow form) 1.5 %; in the long form, where they are nothing beside a unit, four made the code around them 0.5 % slower.
template <int AT_ONCE = 1, typename Params>
__device__ __forceinline__ float largest_key_norm(const Params& p, int bh, int n, f32x4 first, int lane) {
  const float* norms = p.knorm + (int64_t)bh * p.knorm_stride;
  const float known = uniform_load(norms, 0);   // prepared keys
  if (known >= 0.f) return known;
  norms += kNormFirst;
  float top = 0.f;
  auto take = [&](const f32x4& v, int at) {   // places past the valid keys may never have been written
#pragma unroll
    for (int j = 0; j < 4; ++j) top = at + j < n ? fmaxf(top, v[j]) : top;
  };
  take(first, 4 * lane);
  if constexpr (AT_ONCE == 1) {
    for (int at = 4 * lane + 256; at < n; at += 256) take(*(const f32x4*)(norms + at), at);
  } else {
#pragma unroll 1
    for (int at = 4 * lane + 256; at < n; at += 256 * AT_ONCE) {
      f32x4 v[AT_ONCE];
#pragma unroll
      for (int i = 0; i < AT_ONCE; ++i) v[i] = *(const f32x4*)(norms + min(at + 256 * i, (n - 1) & ~3));
#pragma unroll
      for (int i = 0; i < AT_ONCE; ++i) take(v[i], at + 256 * i);
    }
  }
  return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(wave_max(top))));
}

// O = O^T * inv in bf16, out of one wave.  A lane holds 4 consecutive d of a query per accumulator, which would make 8-byte
// stores scattered over 16 rows; instead the wave turns its 32 x 128 block around in 8 KiB of LDS of its own (`stage`;
// 16-byte chunks XOR-swizzled by the row so both directions are conflict-free) and stores whole 256-byte rows, 16 bytes per
// lane.  A block whose 32 rows all exist is eight stores of every lane.
template <bool FP8, typename Params>
__device__ __forceinline__ void store_output(const Params& p, const WaveState<FP8>& w, const float (&inv)[2], char* stage, int b, int h, int q32,
                                             int lane) {
  const int c16 = lane & 15, g4 = lane >> 4;
#pragma unroll
  for (int qb = 0; qb < 2; ++qb)
#pragma unroll
    for (int db = 0; db < 8; ++db) {
      bf16x4 wv;
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) wv[rr] = (__bf16)(w.o[db][qb][rr] * inv[qb]);
      // elements d = 16*db + 4*g .. +3 of row 16*qb + c16: 16-byte chunk 2*db + g/2, its half g%2
      const int chunk = (2 * db + (g4 >> 1)) ^ c16;
      *(bf16x4*)(stage + (16 * qb + c16) * 256 + chunk * 16 + 8 * (g4 & 1)) = wv;
    }
  // same wave wrote and reads: the LDS counter orders the two, no barrier
  if (p.o_images) {
    // operand images of the out-projection GEMM: image (16-row block, k-step h*4 + ks) holds, in lane (c = l % 16,
    // g = l / 16), elements 32*ks + 8*g .. +7 of this head for row c of the block -- one 1 KiB store per image
    if (q32 * 32 >= p.Sq) return;  // a block without rows: the buffer may end before it
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const int r = 16 * rb + c16;
      const bool live = q32 * 32 + r < p.Sq;
      char* img = (char*)p.o + (int64_t)(q32 * 2 + rb) * p.o_img_blk_stride + (int64_t)h * (kD / 32) * 1024;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        bf16x8 v = *(const bf16x8*)(stage + r * 256 + (((4 * ks + g4) ^ (r & 15)) * 16));
        if (!live) v = bf16x8{};
        *(bf16x8*)(img + (ks * 64 + lane) * 16) = v;
      }
    }
    return;
  }
  __bf16* ob = (__bf16*)p.o + (int64_t)b * p.o_sb + (int64_t)h * p.o_sh;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = 4 * i + (lane >> 4), c = lane & 15;
    const bf16x8 v = *(const bf16x8*)(stage + row * 256 + ((c ^ (row & 15)) * 16));
    const int q = q32 * 32 + row;
    if (q < p.Sq) *(bf16x8*)(ob + (int64_t)q * p.o_ss + 8 * c) = v;
  }
}

// The loop of the pipelined short-key form.  A pass runs S^T of the next half beside the softmax of this one, for waves that
// have their SIMD to themselves or share it with one other.  A half takes 0.48 us with one
// workgroup on a CU and 0.41 with two, of which 512 cycles are MFMAs.  (Measured, the same: P.V of half i, softmax of i + 1 and
// S^T of i + 2 in one pass; six passes of lookahead instead of two.)  K of half i + 1 and V of half i are used,
// half i + 2 is on its way and half i + 3 takes the slot of half i - 1 (past the end: the last half once more, into a slot that is
// not read again, which leaves the pass without a branch).
template <bool FP8, bool STATIC, bool POW2, typename Copy>
__device__ __forceinline__ void pipe_loop(WaveState<FP8>& w, char* ring, int n, int sk, const float* kscale, float c, int lane, const Copy& copy) {
  constexpr int kKHalf = (FP8 ? kK8TileBytes : kKTileBytes) / 2, kHalf = kKHalf + kVTileBytes / 2;
  constexpr int kCopies = kHalf / 1024 / kShortWaves;    // of a half, by each wave
  static_assert(kPipeRing == 4, "slots by the low bits of the half");
  auto slot = [&](int i) { return ring + (i & 3) * kHalf; };
  auto scale = [&](int i) { return FP8 ? uniform_load(kscale, min(i, n - 1) >> 1) : 1.0f; };
  auto arrived = [&]() {                                 // all halves but the newest, for every wave
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kCopies) : "memory");
    __syncthreads();
  };
  if (n == 0) return;
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kCopies) : "memory");
  __syncthreads();
  float ks = scale(0);
  qk_half<FP8, false, POW2>(w, slot(0), slot(0) + kKHalf, lane, e8m0_of(ks));
  auto pass = [&](auto at, auto full, int i) {
    constexpr int AT = decltype(at)::value;
    constexpr bool FULL = decltype(full)::value;
    arrived();
    const float ks_next = scale(i + 1);
    qk_half<FP8, false, POW2, 2 - AT>(w, slot(i + 1), slot(i) + kKHalf, lane, e8m0_of(ks_next));
    copy(min(i + 3, n - 1), (i + 3) & 3);
    softmax_pv_half<FP8, STATIC, false, FULL, POW2, AT>(w, (FP8 && !POW2) ? c * ks : c, sk - 32 * i, lane);
    ks = ks_next;
  };
  // the last half has no next one, and is the one that may be partial: its pass computes S^T of nothing that is used
  const std::integral_constant<int, 0> even;
  const std::integral_constant<int, 2> odd;
  int i = 0;
#pragma unroll 1
  for (; i + 2 < n; i += 2) {
    pass(even, std::true_type{}, i);
    pass(odd, std::true_type{}, i + 1);
  }
  if (i + 1 < n) {
    pass(even, std::true_type{}, i);
    pass(odd, std::false_type{}, i + 1);
  } else {
    pass(even, std::false_type{}, i);
  }
  PKH3_MFMA_DRAIN(w);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the spare copies: the epilogue uses the LDS
}

// WAVES == kShortWaves selects the short-key form of the dense kernel: 4 waves (one per SIMD, <= 168 VGPRs) and a
// ring of 32-key half tiles in 48 KiB of LDS, so three workgroups share a CU and the Q load and O store of one
// run under the tiles of the others.  With few key tiles that overlap is worth more than the three-fold K/V
// copies cost (the K/V of such calls sit in L2).
// PARTS (long dense form only): `parts` workgroups share a unit's queries and walk 1/parts of the key tiles each, so
// such a workgroup lasts 1/parts as long as a whole one: the way a call's last, thinly filled round of workgroups is
// cut into pieces that fill the chip (see launch_fp).  Each wave leaves its partial result (un-normalised O^T, row
// sums, row maxima) in global scratch; the wave that arrives last of the `parts` adds the others' to its own and
// writes the output.
constexpr int kMergeBytes = kPartialBytes;  // one wave's partial result in fp32

// workgroups of `blocks` 32-query blocks a (batch, head) needs
__host__ __device__ constexpr int units_per_head(int Sq, int blocks) { return ((Sq + 31) / 32 + blocks - 1) / blocks; }

// Where the waves turn their queries around before the loops: behind the tiles that are on their way by then, all of the ring but its last
// slot, which is not written before every wave has its queries.
constexpr int kTurnBytes = 16 * kD * 2;
template <bool FP8, bool SPARSE, int WAVES, bool PIPE = false>
constexpr int fwd_turn_offset() {
  constexpr int kTileBytes = (FP8 ? kK8TileBytes : kKTileBytes) + kVTileBytes;
  return !SPARSE && WAVES == kShortWaves ? ((PIPE ? kPipeRing : kRing) - 1) * (kTileBytes / 2) : (kRing - 1) * kTileBytes;
}

// bytes of LDS a form of the kernel needs
template <bool FP8, bool SPARSE, int WAVES, bool PIPE = false>
constexpr int fwd_lds_bytes() {
  constexpr bool HALFMODE = !SPARSE && WAVES == kShortWaves;
  constexpr int kTileBytes = (FP8 ? kK8TileBytes : kKTileBytes) + kVTileBytes;
  constexpr int kHalfBytes = kTileBytes / 2;
  constexpr int kStageBytes = 32 * kD * 2;    // one wave's 32 x 128 bf16 output block, staged for the row-wise store
  // dense / phase 1: ring of kRing whole tiles; sparse phase 2: kStages2 stages of row-private half tiles
  constexpr int kPhase2Bytes = SPARSE ? kStages2 * kSparseRows * kHalfBytes : 0;
  constexpr int kRingBytes = HALFMODE ? (PIPE ? kPipeRing : kRing) * kHalfBytes
                             : (kPhase2Bytes > kRing * kTileBytes ? kPhase2Bytes : kRing * kTileBytes);
  constexpr int kAfterBytes = WAVES * kStageBytes;  // LDS use after the loops
  constexpr int kBeforeBytes = fwd_turn_offset<FP8, SPARSE, WAVES, PIPE>() + WAVES * kTurnBytes;   // ... and before them
  constexpr int kBytes = kRingBytes > kAfterBytes ? kRingBytes : kAfterBytes;
  return kBytes > kBeforeBytes ? kBytes : kBeforeBytes;
}

// POW2 (fp8 only): power-of-two block scales, applied by the scaled MFMA; softmax_scale * log2(e) rides in Q' before
// it is quantised, so the softmax has no multiply left (the instruction count of the bf16 form).
// One workgroup's work.  `blk`: index of the workgroup inside its section of the launch; the section covers the
// units [unit0, unit0 + units), a unit being one workgroup's block of queries (`parts` workgroups per unit; their
// partial results start at slot `part_base` of the scratch, their counters at unit slot `cnt_base`).
// Block-sparse with work queues: returns the next position of the home queue, taken (thread 0) while the output is stored.
template <bool FP8, bool SPARSE, int WAVES, bool POW2, bool PIPE = false, typename Params>
__device__ __forceinline__ int attn_fwd_body(const Params& p, int blk, int unit0, int units, int parts, int part_base,
                                              int cnt_base, char* lds_raw, int fetched = -1) {
  static_assert(!SPARSE || WAVES == kSparseWaves, "block-sparse layout: a wave pair per row-block of the plan");
  static_assert(FP8 || !POW2, "power-of-two scales belong to the fp8 form");
  constexpr bool SHORT = !SPARSE && WAVES == kShortWaves;
  constexpr bool LEAN = !SPARSE;                        // dense long-key form: three waves per SIMD, lean read-ahead
  constexpr int kAhead = kRing - 1;                     // tiles in flight ahead of the one being used
  constexpr bool HALFMODE = SHORT;                      // ring of 32-key half tiles
  constexpr bool kAskFirst = SPARSE || PIPE;            // (their registers hold both blocks' rows and tables)
  constexpr bool PARTS = !SPARSE && !SHORT;             // the long dense form: the key tiles may be shared out (`parts`)
  constexpr int kKBytes = FP8 ? kK8TileBytes : kKTileBytes;
  constexpr int kTileBytes = kKBytes + kVTileBytes;
  constexpr int kChunks = kTileBytes / 1024;  // 1 KiB pieces of a tile, dealt round-robin to the waves
  constexpr int kHalfBytes = kTileBytes / 2;  // K and V images of 32 keys
  constexpr int kStageBytes = 32 * kD * 2;    // one wave's 32 x 128 bf16 output block, staged for the row-wise store
  char(*lds)[kTileBytes] = (char(*)[kTileBytes])lds_raw;
  int lane = threadIdx.x & 63;
  // (what is made of the lane is made again for every unit: kept across the units, it does not fit the registers)
  if constexpr (SPARSE) asm volatile("" : "+v"(lane));
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  // Workgroups are handed to the 8 XCDs round-robin; give each XCD one contiguous run of
  // (batch, head, query tile) so the 32 CUs behind one L2 stream the same K/V at the same time.
  // (Every section of a launch starts at a workgroup index that is a multiple of 8.)
  // (`fetched` >= 0: the unit came from the work queues instead, see attn_fwd_dense_kernel.)
  const int total = units * parts;
  const int per_xcd = (total + 7) / 8;
  const int lin = fetched >= 0 ? fetched : (blk & 7) * per_xcd + (blk >> 3);
  if (lin >= total) return 0;
  // unit inside the section, and which share of its keys: share-major, so that the workgroups an XCD runs at the
  // same time walk the same key tiles of (mostly) the same head, as the whole units before them do
  const int part = lin / units, ul = lin % units;
  const int unit = unit0 + ul;
  const int wq = wave;                                    // which 32-query block of the unit
  const int nQt = SPARSE ? p.nQ64 / kSparseRows : units_per_head(p.Sq, WAVES);  // units per (batch, head)
  const int bh = unit / nQt, qt = unit % nQt;
  const int q32 = qt * WAVES + wq;
  const int b = bh / p.H, h = bh % p.H;

  QRows q_rows[2];
  NormLanes q_norm;
  const f32x4 first_norms = ask_key_norms(p, bh, lane);
  int q_lane = lane;                                      // (places in LDS that the output uses as well are not kept until then)
  asm volatile("" : "+v"(q_lane));
  auto load_q = [&](int qb) { ask_q_rows(q_rows[qb], p, b, h, q32 * 32 + 16 * qb, q_lane); };
  // The block-sparse form has one workgroup per CU and nothing to run beside this: rows, tables and weights are asked for before
  // anything else of the unit is known, so that they cost one trip to memory between them and the plan's look-ups and the first
  // key copies run beside it (14,907 rows, fp8: the call 691 -> 679 us; 48,360, bf16: 6,880 -> 6,800).  So does the pipelined short-key form.
  // Where a third wave per SIMD runs beside it, it gave nothing.  (The turn through LDS did: against loads in the order of the images in the long form
  // alone, 124,992 rows 128.74 -> 127.18 ms, 48,360 19.68 -> 19.54, 15,342 2.093 -> 2.078, 48,360 in fp8 the same.)
  if constexpr (kAskFirst) load_q(0), load_q(1);
  load_norm_lanes(q_norm, p.q_norm_w, lane);

  const int sk = p.row_cnt ? uniform_load(p.row_cnt, b) : p.Sk;
  const int nkt = (sk + kTileKeys - 1) / kTileKeys;
  // sparse: [tiles every row-block of this workgroup keeps | tiles only row-block 0 keeps | ... 1 | ...]
  const int* plan = SPARSE ? p.plan + (int64_t)qt * p.plan_stride : nullptr;
  const int* plan_cnt = SPARSE ? p.plan_cnt + qt * kSparseLists : nullptr;
  const int nt = SPARSE ? uniform_load(plan_cnt, 0) : nkt;  // tiles all the waves walk together
  // the tiles [t_begin, t_end) of those are this workgroup's share
  // (32-bit arithmetic: at most 2^18 tiles times kMaxParts; the results address the tile copies from scalar registers)
  const int t_begin = PARTS ? __builtin_amdgcn_readfirstlane(part * nt / parts) : 0;
  const int t_end = PARTS ? __builtin_amdgcn_readfirstlane((part + 1) * nt / parts) : nt;

  // this wave's pieces of every [K|V] tile record: 1 KiB chunks wave, wave + WAVES, ...
  const char* kv_w = p.kv + (int64_t)bh * p.kv_bh_stride + wave * 1024;
  const unsigned lane_off = lane * 16;
  auto dma = [&](int tile, int slot) {
    const char* g = kv_w + (int64_t)tile * p.kv_tile_stride;
    char* d = lds[slot] + wave * 1024;
#pragma unroll
    for (int i = 0; i < (kChunks + WAVES - 1) / WAVES; ++i) {
      if ((i + 1) * WAVES <= kChunks) lds_dma16(g + i * WAVES * 1024, lane_off, d + i * WAVES * 1024);
      else if (i * WAVES + wave < kChunks) lds_dma16(g + i * WAVES * 1024, lane_off, d + i * WAVES * 1024);
    }
  };
  auto entry = [&](int i) { return SPARSE ? uniform_load(plan, i) : i; };  // i-th shared tile

  // half-tile form: [K half | V half] per ring slot, every wave copies the same share
  constexpr int kKHalfB = kKBytes / 2, kVHalfB = kVTileBytes / 2;
  const int n_half = (sk + 31) / 32;
  const int h_begin = 0, n_mine = n_half;
  char* ring = lds_raw;
  auto dma_short = [&](int half, int slot) {
    static_assert((kKHalfB / 1024) % kShortWaves == 0 && (kVHalfB / 1024) % kShortWaves == 0, "equal shares");
    const char* g = p.kv + (int64_t)bh * p.kv_bh_stride + (int64_t)(half >> 1) * p.kv_tile_stride;
    char* d = ring + slot * kHalfBytes;
    const int kb = half & 1;
#pragma unroll
    for (int i = 0; i < kKHalfB / 1024 / kShortWaves; ++i) {
      const int ch = wq * (kKHalfB / 1024 / kShortWaves) + i;
      lds_dma16(g + kb * kKHalfB + ch * 1024, lane_off, d + ch * 1024);
    }
#pragma unroll
    for (int i = 0; i < kVHalfB / 1024 / kShortWaves; ++i) {
      const int ch = wq * (kVHalfB / 1024 / kShortWaves) + i;
      lds_dma16(g + kKBytes + kb * kVHalfB + ch * 1024, lane_off, d + kKHalfB + ch * 1024);
    }
  };

  WaveState<FP8> w;
  if constexpr (PIPE) {
    if (n_half > 0) {
#pragma unroll
      for (int i = 0; i < kPipeRing - 1; ++i) dma_short(min(i, n_half - 1), i);
    }
  } else if constexpr (HALFMODE) {
    if (n_mine > 0) dma_short(h_begin, 0);
    if (n_mine > 1) dma_short(h_begin + 1, 1);
  } else if (t_end > t_begin) {
    dma(entry(t_begin), 0);
    if (t_end > t_begin + 1) dma(entry(t_begin + 1), 1);
  }
  // Q, fused with QK-RMSNorm, rotation and (fp8) quantisation, in the layout of the MFMA B images themselves:
  // lane (c, g) gets, for each of the wave's two 16-query blocks qb, the 32 elements d = 32*ks + 8*g + j of query
  // row q32*32 + 16*qb + c (four lanes per row), so the operand images are formed in the lane
  // that uses them and Q' never exists in memory.
  float qscale = 1.0f;
  float qn2 = 0.f;  // largest squared norm of this lane's Q' rows as the MFMAs take them
  {
    float x[2][32];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      if constexpr (!kAskFirst) load_q(qb);
      // softmax_scale * log2(e) rides in Q' (bf16, and fp8 with power-of-two scales), so S^T comes out of the MFMAs in the log2 domain
      q_rows_ready(x[qb], q_rows[qb], p, q_norm, FP8 && !POW2 ? 1.0f : p.c, lds_raw + fwd_turn_offset<FP8, SPARSE, WAVES, PIPE>() + wave * kTurnBytes, q_lane);
    }
    if constexpr (!FP8) {
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        float n2[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          bf16x8 t;
#pragma unroll
          for (int j = 0; j < 8; ++j) t[j] = (__bf16)x[qb][ks * 8 + j];
          w.qf[qb][ks] = t;
          n2[ks] = add_squares(t, 0.f);
        }
        qn2 = fmaxf(qn2, wave_sum_groups((n2[0] + n2[1]) + (n2[2] + n2[3])));
      }
    } else {
      // one absmax scale per 64-query block = this wave and its neighbour (wave ^ 1)
      __shared__ float q_amax[WAVES];
      float amax = 0.f;
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
#pragma unroll
        for (int i = 0; i < 32; ++i) amax = fmaxf(amax, fabsf(x[qb][i]));
      amax = wave_max(amax);
      if (lane == 0) q_amax[wave] = amax;
      __syncthreads();
      amax = fmaxf(amax, q_amax[wave ^ 1]);
      qscale = fp8_block_scale(amax, POW2);
      w.qe = e8m0_of(qscale);
      const float inv = 1.0f / qscale;
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        float n2 = 0.f;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          const i32x2 q = quant_fp8_piece(x[qb] + 8 * ks, inv);   // bytes 8*ks + j of the image = element 32*ks + 8*g + j
          w.q8[qb][2 * ks] = q[0];
          w.q8[qb][2 * ks + 1] = q[1];
#pragma unroll
          for (int wd = 0; wd < 2; ++wd) {
            const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8(q[wd], false);
            const auto hi = __builtin_amdgcn_cvt_pk_f32_fp8(q[wd], true);
            n2 += lo[0] * lo[0] + lo[1] * lo[1] + hi[0] * hi[0] + hi[1] * hi[1];
          }
        }
        qn2 = fmaxf(qn2, wave_sum_groups(n2) * qscale * qscale);
      }
    }
  }
#pragma unroll
  for (int db = 0; db < 8; ++db)
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
      for (int i = 0; i < 4; ++i) w.o[db][qb][i] = 0.f;
  w.m[0] = w.m[1] = kNoMax;
  w.l[0] = w.l[1] = 0.f;
  const float c = POW2 ? 1.0f : p.c * qscale;  // what the softmax still multiplies the logits by (fp8 absmax form only)
  const float* kscale = FP8 ? p.kscale + (int64_t)bh * p.nKt : nullptr;
  const int tail = sk & (kTileKeys - 1);  // keys in the last tile when it is partial

  // Upper bound of the magnitude of this query's logits (log2 domain): |q_i| * max_j |k_j| * c.  When it is
  // small for the whole wave, exp2(logit) is a normal number in fp32 and in bf16 whatever the data, and so are
  // the row sums and O^T (at most 2^bound * keys * |v|), so no running max is needed at all.
  bool static_max = false;
  if (HALFMODE ? n_half > 0 : nt > 0) {
    // margins: K' is rounded to bf16 (relative step 2^-9; fp8: to e4m3, relative step 2^-4) after its norms were taken
    const float bound = sqrtf(qn2) * largest_key_norm(p, bh, n_half, first_norms, lane) * (FP8 ? (POW2 ? 1.08f : p.c * 1.08f) : 1.01f);
    static_max = __all(bound <= kStaticMaxLimit);
  }

  int slot = 0, slot_prev = kRing - 1;  // ring slots of tile i and of tile i-1 (which takes the newest copy)
  // Only the last key tile can be partial.  It is peeled off the loop so that the loop body has no masking
  // branch between S^T and the softmax, which lets the numerators of the first 32 keys be scheduled under
  // the MFMAs of the second 32.
  const int n_masked = (tail && t_end > t_begin && entry(t_end - 1) == nkt - 1) ? 1 : 0;
  float ks_next = (FP8 && !HALFMODE && t_end > t_begin) ? uniform_load(kscale, entry(t_begin)) : 1.0f;
#define PKH3_TILE_LOOP(STATIC, MASKED, FROM, TO)                                                        \
  for (int i = FROM; i < TO; ++i) {                                                                     \
    /* tile i (and, with a ring of three, i+1) is in LDS for every wave (own slices: vmcnt, the others': */ \
    /* barrier), and every wave is past tile i-1, whose slot takes the newest copy */                   \
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                                                    \
    __syncthreads();                                                                                    \
    const char* kbuf = lds[slot];                                                                       \
    /* the K scale of this tile was asked for an iteration ago (with power-of-two scales the first MFMA */ \
    /* needs it); the one of the next tile is asked for now */                                          \
    const float ks = ks_next;                                                                           \
    if (FP8) ks_next = uniform_load(kscale, entry(min(i + 1, t_end - 1)));                              \
    qk_tile<FP8, LEAN, (MASKED) ? 2 : 4, POW2>(w, kbuf, kbuf + kKBytes, lane, e8m0_of(ks));             \
    /* the copies of the tile two ahead are issued under the MFMAs of S^T, not in front of them: right */ \
    /* after the barrier their scalar address chain would run in every wave at once with the pipe idle */ \
    /* (power-of-two fp8 form: issued without a branch, a spare copy of the last tile at the end, which leaves */ \
    /* the tile body one straight run of code; that schedule measured 2.4 % faster there and 1 - 3 % slower in */ \
    /* the other forms) */                                                                              \
    if (POW2) dma(entry(min(i + kAhead, t_end - 1)), slot_prev);                                        \
    else if (i + kAhead < t_end) dma(entry(i + kAhead), slot_prev);                                     \
    slot_prev = slot;                                                                                   \
    slot = slot == kRing - 1 ? 0 : slot + 1;                                                            \
    const float ct = (FP8 && !POW2) ? c * ks : c;                                                       \
    softmax_pv_tile<FP8, STATIC, LEAN, MASKED, POW2>(w, kbuf + kKBytes, ct, tail, lane);                \
  }
  // Half-tile loop.  The leading full halves take the copy of the code without masking; the one partial half at the
  // very end of the keys, if any, takes the general copy.
#define PKH3_SHORT_LOOP(STATIC, FULL, FROM, TO)                                                         \
  for (int i = FROM; i < TO; ++i) {                                                                     \
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                                                    \
    __syncthreads();                                                                                    \
    const char* hbuf = ring + slot * kHalfBytes;                                                        \
    const int half = h_begin + i;                                                                       \
    const bool live = FULL || i < n_mine;                                                               \
    const float ks = (FP8 && live) ? uniform_load(kscale, half >> 1) : 1.0f;                            \
    if (live) qk_half<FP8, true, POW2>(w, hbuf, hbuf + kKHalfB, lane, e8m0_of(ks));                     \
    /* copies of the half two ahead: under the MFMAs of S^T (see the whole-tile loop) */               \
    if (i + 2 < n_mine) dma_short(h_begin + i + 2, slot_prev);                                          \
    slot_prev = slot;                                                                                   \
    slot = slot == kRing - 1 ? 0 : slot + 1;                                                            \
    if (live) {                                                                                         \
      const float ct = (FP8 && !POW2) ? c * ks : c;                                                     \
      softmax_pv_half<FP8, STATIC, true, FULL, POW2>(w, ct, sk - 32 * half, lane, hbuf + kKHalfB);      \
    }                                                                                                   \
  }
  if constexpr (PIPE) {
    static_assert(HALFMODE, "32-key halves");
    if (static_max) pipe_loop<FP8, true, POW2>(w, ring, n_half, sk, kscale, c, lane, dma_short);
    else pipe_loop<FP8, false, POW2>(w, ring, n_half, sk, kscale, c, lane, dma_short);
  } else if constexpr (HALFMODE) {
    const int n_iter = n_half;
    const int n_lead = sk / 32;  // leading full halves
    if (static_max) {
      PKH3_SHORT_LOOP(true, true, 0, n_lead)
      PKH3_SHORT_LOOP(true, false, n_lead, n_iter)
      PKH3_MFMA_DRAIN(w);
    } else {
      PKH3_SHORT_LOOP(false, true, 0, n_lead)
      PKH3_SHORT_LOOP(false, false, n_lead, n_iter)
      PKH3_MFMA_DRAIN(w);
    }
  } else if (static_max) {
    PKH3_TILE_LOOP(true, false, t_begin, t_end - n_masked)
    PKH3_TILE_LOOP(true, true, t_end - n_masked, t_end)
    PKH3_MFMA_DRAIN(w);
  } else {
    PKH3_TILE_LOOP(false, false, t_begin, t_end - n_masked)
    PKH3_TILE_LOOP(false, true, t_end - n_masked, t_end)
    PKH3_MFMA_DRAIN(w);
  }
#undef PKH3_TILE_LOOP
#undef PKH3_SHORT_LOOP

  if constexpr (SPARSE) {
    // Phase 2: the tiles that only some row-blocks keep.  Each row-block (a wave pair) walks its own list in
    // 32-key halves; an iteration gives every pair one half tile in its own LDS area, so all 8 waves stay
    // busy whichever rows a tile belongs to.  Two stages, the next half tile is copied while this one is used.
    const int r = wave >> 1;  // row-block of this wave inside the workgroup
    const int* mine = plan + (1 + r) * p.nKt;
    const int n_mine = uniform_load(plan_cnt, 1 + r);
    int n_longest = 0;  // every wave runs as many iterations as the longest list needs, so the barriers match
#pragma unroll
    for (int rr = 0; rr < kSparseRows; ++rr) n_longest = max(n_longest, uniform_load(plan_cnt, 1 + rr));
    const int n_iter = 2 * n_longest;
    constexpr int kKHalf = kKBytes / 2, kVHalf = kVTileBytes / 2;
    // this wave copies half of its pair's K half (and V half): K images are 1 KiB x (8 bf16 | 4 fp8) per half
    auto dma_half = [&](int it, int stage) {
      const int tile = uniform_load(mine, it >> 1);
      const int kb = it & 1;
      const char* g = p.kv + (int64_t)bh * p.kv_bh_stride + (int64_t)tile * p.kv_tile_stride;
      char* d = lds_raw + (stage * kSparseRows + r) * kHalfBytes;
      const int sub = wave & 1;
#pragma unroll
      for (int i = 0; i < kKHalf / 2048; ++i)
        lds_dma16(g + kb * kKHalf + (sub * (kKHalf / 2048) + i) * 1024, lane_off, d + (sub * (kKHalf / 2048) + i) * 1024);
#pragma unroll
      for (int i = 0; i < kVHalf / 2048; ++i)
        lds_dma16(g + kKBytes + kb * kVHalf + (sub * (kVHalf / 2048) + i) * 1024, lane_off,
                  d + kKHalf + (sub * (kVHalf / 2048) + i) * 1024);
    };
    __syncthreads();  // every wave is done with the phase-1 ring
    // kStages2 - 1 half tiles ahead: half tile `it` lives in stage it % kStages2
#pragma unroll
    for (int a = 0; a < kStages2 - 1; ++a)
      if (a < 2 * n_mine) dma_half(a, a);
    int st2 = 0, st2_free = kStages2 - 1;  // stage of half tile `it`, and the one the newest copy goes to
    // list entry and K scale of the half tile an iteration uses are asked for an iteration ahead
    int tile_next = n_mine > 0 ? uniform_load(mine, 0) : 0;
    float ks2_next = (FP8 && n_mine > 0) ? uniform_load(kscale, tile_next) : 1.0f;
#define PKH3_HALF_LOOP(STATIC)                                                                          \
  for (int it = 0; it < n_iter; ++it) {                                                                 \
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                                                    \
    __syncthreads();                                                                                    \
    const char* hbuf = lds_raw + (st2 * kSparseRows + r) * kHalfBytes;                                  \
    const int st2_write = st2_free;                                                                     \
    st2_free = st2;                                                                                     \
    st2 = st2 == kStages2 - 1 ? 0 : st2 + 1;                                                            \
    if (it >= 2 * n_mine) continue; /* wave-uniform: this row-block has run out of tiles (and of copies) */ \
    const int tile = tile_next;                                                                         \
    const float ks = ks2_next;                                                                          \
    tile_next = uniform_load(mine, min(it + 1, 2 * n_mine - 1) >> 1);                                   \
    if (FP8) ks2_next = uniform_load(kscale, tile_next);                                                \
    /* the running-max copy needs registers for the rescale: it takes the lean read-ahead (4 images) */ \
    qk_half<FP8, !STATIC, POW2>(w, hbuf, hbuf + kKHalf, lane, e8m0_of(ks));                             \
    /* copies of the next half tile of this row-block: under the MFMAs of S^T (see the whole-tile loop) */ \
    if (it + kStages2 - 1 < 2 * n_mine) dma_half(it + kStages2 - 1, st2_write);                         \
    const float ct = (FP8 && !POW2) ? c * ks : c;                                                       \
    const int lim = (tail && tile == nkt - 1) ? tail - 32 * (it & 1) : 32;                              \
    softmax_pv_half<FP8, STATIC, !STATIC, false, POW2>(w, ct, lim, lane, hbuf + kKHalf);                \
  }
    if (static_max) {
      PKH3_HALF_LOOP(true)
      PKH3_MFMA_DRAIN(w);
    } else {
      PKH3_HALF_LOOP(false)
      PKH3_MFMA_DRAIN(w);
    }
#undef PKH3_HALF_LOOP
  }

  int next_pos = 0;
  if constexpr (SPARSE) {
    if (p.queue_next && threadIdx.x == 0) next_pos = take_position(p.queue_next + (blockIdx.x & (kQueues - 1)));
  }

  __syncthreads();  // every wave is done reading K/V tiles: the LDS becomes staging space
  if constexpr (PARTS) {
    if (parts > 1) {
      // `parts` workgroups hold a share of this unit's result each.  Every wave leaves its partial result in global
      // scratch and counts itself in; the wave that finds all the others counted adds their partials to its own and
      // goes on to write the output, the others are done.  Partials and counter move through device-coherent
      // stores, loads and atomics: a wave counts itself in only after its stores have completed, and reads the
      // others' partials only after it has seen their counts.
      const int64_t wslot = kMergeBytes / 4;   // floats per wave
      float* mine = p.split_scratch + ((int64_t)(part_base + ul * parts + part) * WAVES + wave) * wslot;
#pragma unroll
      for (int db = 0; db < 8; ++db)
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) store_device(mine + ((db * 2 + qb) * 64 + lane) * 4, w.o[db][qb]);
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        store_device(mine + 64 * 64 + qb * 64 + lane, w.l[qb]);
        store_device(mine + 64 * 64 + 128 + qb * 64 + lane, w.m[qb]);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      int arrived = 0;
      if (lane == 0)
        arrived = __hip_atomic_fetch_add(p.split_cnt + (cnt_base + ul) * WAVES + wave, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      arrived = __builtin_amdgcn_readfirstlane(arrived);
      if (arrived != parts - 1) return 0;
      // The partials are added up in the order of the shares, whichever wave does it (its own comes back from the
      // scratch like the others), so the result does not depend on which workgroup finished last.
#pragma unroll 1
      for (int src = 0; src < parts; ++src) {
        const float* theirs = p.split_scratch + ((int64_t)(part_base + ul * parts + src) * WAVES + wave) * wslot;
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
          const float l2 = load_device(theirs + 64 * 64 + qb * 64 + lane), m2 = load_device(theirs + 64 * 64 + 128 + qb * 64 + lane);
          // On the bounded-logit path nothing was subtracted, so numerators and row sums just add; on the
          // running-max path each side is first brought to the common maximum.  Share 0 starts the sum.
          float a1 = src == 0 ? 0.0f : 1.0f, a2 = 1.0f;
          if (!static_max && src != 0) {
            const float mn = fmaxf(w.m[qb], m2);
            a1 = __builtin_amdgcn_exp2f(w.m[qb] - mn);
            a2 = __builtin_amdgcn_exp2f(m2 - mn);
            w.m[qb] = mn;
          } else if (src == 0) {
            w.m[qb] = m2;
          }
          w.l[qb] = src == 0 ? l2 : w.l[qb] * a1 + l2 * a2;
#pragma unroll
          for (int db = 0; db < 8; ++db) {
            const f32x4 v4 = load_device4(theirs + ((db * 2 + qb) * 64 + lane) * 4);
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) w.o[db][qb][rr] = src == 0 ? v4[rr] : w.o[db][qb][rr] * a1 + v4[rr] * a2;
          }
        }
      }
    }
  }
  float inv[2];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const float lt = wave_sum_groups(w.l[qb]);
    inv[qb] = lt > 0.f ? 1.0f / lt : 0.f;
  }
  store_output(p, w, inv, lds_raw + wq * kStageBytes, b, h, q32, lane);
  return next_pos;
}

// The block-sparse kernel and the short-key dense kernel (the block-sparse one takes its units from the work queues
// when the launch has them: they differ in length with the tile lists on top of the XCDs' clocks).
template <bool FP8, bool SPARSE, int WAVES, bool POW2, bool PIPE = false>
__global__ __launch_bounds__(64 * WAVES, (SPARSE ? 8 / WAVES : PIPE ? 2 : 3)) void attn_fwd_kernel(FwdParams p) {
  __shared__ __attribute__((aligned(1024))) char lds_raw[fwd_lds_bytes<FP8, SPARSE, WAVES, PIPE>()];
  if constexpr (!SPARSE) {
    attn_fwd_body<FP8, SPARSE, WAVES, POW2, PIPE>(p, blockIdx.x, 0, p.sec_units[0], 1, 0, 0, lds_raw);
  } else {
    __shared__ int fetched_unit;
    int next_pos = 0;
    if (p.queue_next && threadIdx.x == 0) next_pos = take_position(p.queue_next + (blockIdx.x & (kQueues - 1)));
    // A workgroup per CU takes units until the queues are empty (each pass takes a position, so the loop ends); without queues it
    // does the unit of its index.  A workgroup per unit, dealt out by the hardware, left CUs idle for 15 us between two units and
    // up to a quarter of them while a few long units ran on others (rows that keep every tile last four times as long): with
    // 14,907 rows (fp8, density 0.28) 117 of 787 us a CU, now 40.  The call 727 -> 688 us; at 48,360 rows the same.  Handing out
    // the longest units first gave nothing on top of this (689).
#pragma unroll 1
    do {
      int fetched = -1;
      if (p.queue_next) {   // wave-uniform
        // (every wave has left the last unit's LDS when it comes to this barrier)
        if (threadIdx.x == 0) fetched_unit = fetch_unit(p.queue_next, blockIdx.x & (kQueues - 1), p.sec_units[0], next_pos);
        __syncthreads();
        fetched = __builtin_amdgcn_readfirstlane(fetched_unit);
        if (fetched < 0) return;
      }
      // The arguments are read again for every unit, from where the kernel got them: kept across the loop, what is made of them
      // does not fit the scalar registers.
      unsigned at = 0;
      asm volatile("" : "+s"(at));
      typedef const __attribute__((address_space(4))) char* KernargBytes;
      const auto& again = *(const __attribute__((address_space(4))) FwdParams*)((KernargBytes)__builtin_amdgcn_kernarg_segment_ptr() + at);
      next_pos = attn_fwd_body<FP8, SPARSE, WAVES, POW2>(again, blockIdx.x, 0, again.sec_units[0], 1, 0, 0, lds_raw, fetched);
    } while (p.queue_next);
  }
}

// The long dense kernel: a launch of up to kSections sections, handed out in this order as CUs fall free.  Section 0
// holds whole units (one workgroup each); the later ones the units of a thinly filled last round, each shared out
// among sec_parts[] workgroups.  When the launch has work queues, every section's work is taken from queues of its own.
template <bool FP8, bool POW2>
__global__ __launch_bounds__(64 * kDenseWaves, 1) void attn_fwd_dense_kernel(FwdParams p) {
  __shared__ __attribute__((aligned(1024))) char lds_raw[fwd_lds_bytes<FP8, false, kDenseWaves>()];
  __shared__ int fetched_unit;
  static_assert(kSections == 3 && kSections * kQueues <= kQueueSlots, "the section look-up below is written out for three");
  const int bid = blockIdx.x, b0 = p.sec_blocks[0], b1 = p.sec_blocks[1];
  const int sec = (bid >= b0 ? 1 : 0) + (bid >= b0 + b1 ? 1 : 0);
  const int blk = bid - (sec >= 1 ? b0 : 0) - (sec >= 2 ? b1 : 0);
  const int unit0 = (sec >= 1 ? p.sec_units[0] : 0) + (sec >= 2 ? p.sec_units[1] : 0);
  const int units = sec == 0 ? p.sec_units[0] : sec == 1 ? p.sec_units[1] : p.sec_units[2];
  const int parts = sec == 0 ? p.sec_parts[0] : sec == 1 ? p.sec_parts[1] : p.sec_parts[2];
  // partial results and counters of section 2 lie behind those of section 1 (section 0 has none)
  const bool behind = sec == 2 && p.sec_parts[1] > 1;
  const int part_base = behind ? p.sec_units[1] * p.sec_parts[1] : 0, cnt_base = behind ? p.sec_units[1] : 0;
  int fetched = -1;
  if (p.queue_next) {   // wave-uniform; every section has queues of its own over its workgroups' work
    if (threadIdx.x == 0) fetched_unit = fetch_unit(p.queue_next + sec * kQueues, blk & (kQueues - 1), units * parts);
    __syncthreads();
    fetched = __builtin_amdgcn_readfirstlane(fetched_unit);
    if (fetched < 0) return;
  }
  attn_fwd_body<FP8, false, kDenseWaves, POW2>(p, blk, unit0, units, parts, part_base, cnt_base, lds_raw, fetched);
}

// The narrow form, for calls whose 32-query blocks hardly outnumber the CUs: a workgroup is one block of 32 queries, and its
// 4 waves share the keys out in runs of 32-key half tiles.  No two waves of a workgroup read the same images, and an image
// is exactly what a lane of the MFMA wants, so they go from the L2 straight into registers: no LDS ring and no barrier in
// the loop, the next K images on their way under the softmax, the V images under S^T.  The partial results meet in LDS,
// where every wave adds up its share of the 16-row blocks of O^T, in the order of the key shares.
// Bound by the CU's 64 bytes per clock of vector loads (16 KiB for 32 MFMAs: twice what the matrix units need for them) and,
// for few keys, by the start and the merge of a workgroup; two workgroups of 4 waves share a CU, so that those of one run
// under the loads of the other (one of 8 waves: the same up to 256 blocks, 8 x 2000 rows 28.0 against 23.9 us).  Kernel times
// (launches back to back) against the form that took these calls before: 4 heads x 1,024 rows 23.2 -> 10.3 us, 2 x 3,000 88 -> 18.5,
// 24 x 256 rows and 2,048 keys 61 -> 14.7, 8 x 2,000 62 -> 24 (fp8 57 -> 21), 1 x 15,000 404 -> 138.
constexpr int kNarrowWaves = 4;

// The tiles a query block walks: all of them, or (block-sparse) the two lists of the plan it belongs to.
template <bool SPARSE>
struct TileWalk {
  const int* shared;   // tiles its whole plan entry keeps ...
  int n_shared;
  const int* own;      // ... and those its row-block keeps besides
  __device__ __forceinline__ int operator()(int e) const {
    if constexpr (!SPARSE) return e;
    else return e < n_shared ? uniform_load(shared, e) : uniform_load(own, e - n_shared);
  }
};

template <bool FP8, bool POW2, bool SPARSE, bool STATIC>
__device__ __forceinline__ void narrow_loop(WaveState<FP8>& w, i32x4 (&kf)[FP8 ? 4 : 8], const char* kv, int tile_stride, const float* kscale,
                                            const TileWalk<SPARSE>& walk, int h0, int h1, int sk, float c, int lane) {
  constexpr int kKBytes = FP8 ? kK8TileBytes : kKTileBytes;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  int tile = h0 < h1 ? walk(h0 >> 1) : 0;
#pragma unroll 1
  for (int i = h0; i < h1; ++i) {
    // (the last iteration asks for its own K images again: the loads need no branch)
    const int n = min(i + 1, h1 - 1);
    const int tile_next = walk(n >> 1);
    const char* v = kv + (int64_t)tile * tile_stride + kKBytes + (i & 1) * (kVTileBytes / 2);
    const float ks = FP8 ? uniform_load(kscale, tile) : 1.0f;
    // (a sparse list may go on behind the short last tile, whose second half then holds no key: lim <= 0, probabilities of 0)
    const int lim = sk - 64 * tile - 32 * (i & 1);
#pragma unroll
    for (int j = 0; j < 8; ++j) w.vf[j] = *(const bf16x8*)(v + (j * 64 + lane) * 16);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!FP8) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int qb = 0; qb < 2; ++qb)
          w.s[j & 1][qb] = PKH3_MFMA16(__builtin_bit_cast(bf16x8, kf[j]), w.qf[qb][j >> 1], j < 2 ? zero : w.s[j & 1][qb]);
    } else {
      const int ke = e8m0_of(ks);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const i32x4 a0 = kf[2 * kb], a1 = kf[2 * kb + 1];
        const i32x8 a = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
#pragma unroll
        for (int qb = 0; qb < 2; ++qb)
          w.s[kb][qb] = POW2 ? PKH3_MFMA16_F8S(a, w.q8[qb], zero, ke, w.qe) : PKH3_MFMA16_F8(a, w.q8[qb], zero);
      }
    }
    const char* k = kv + (int64_t)tile_next * tile_stride + (n & 1) * (kKBytes / 2);
#pragma unroll
    for (int j = 0; j < (FP8 ? 4 : 8); ++j) kf[j] = *(const i32x4*)(k + (j * 64 + lane) * 16);
    __builtin_amdgcn_sched_barrier(0);
    softmax_pv_half<FP8, STATIC, false, false, POW2>(w, (FP8 && !POW2) ? c * ks : c, lim, lane);
    tile = tile_next;
  }
  PKH3_MFMA_DRAIN(w);
}

// MASKED (key mask: how many keys are valid is known on the device only).  The start and the merge of every block of 32 queries are
// worth it for long walks alone.  The launch holds the workgroups of both forms, and where fewer than p.few_halves half tiles are
// valid it is the short-key ones (128 queries each, in front) that do the work.  24 heads x 1,558 rows, 23 of
// 2,526 keys valid: 16.1 -> 8.9 us; 4 x 24 heads x 87 rows, 29 of 446: 7.2 -> 6.0.
template <bool FP8, bool POW2, bool SPARSE, bool MASKED = false>
__global__ __launch_bounds__(64 * kNarrowWaves, 2) void attn_fwd_narrow_kernel(FwdParams p) {
  static_assert(!MASKED || (!FP8 && !SPARSE), "key masks are taken by dense bf16 calls only");
  constexpr int NW = kNarrowWaves;
  constexpr int kKBytes = FP8 ? kK8TileBytes : kKTileBytes;
  constexpr int kSlot = 64 * 64 * 4;                       // one wave's O^T in fp32
  __shared__ __attribute__((aligned(1024))) char part[NW * kSlot];
  __shared__ __attribute__((aligned(1024))) char rows[32 * kD * 2];   // the Q images, later the output rows
  __shared__ float part_l[NW][2][16], part_m[NW][2][16];
  __shared__ float s_n2[2], s_amax[4];
  const int lane = threadIdx.x & 63, c16 = lane & 15, g4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int nth = blockIdx.x >> 3;                               // of the workgroups of this XCD
  if constexpr (MASKED) {
    static_assert(kNarrowWaves == kShortWaves && fwd_lds_bytes<false, false, kShortWaves>() <= (int)sizeof(part), "a workgroup of the short-key form");
    const int per_xcd4 = (p.sec_units[1] + 7) / 8;
    if (nth < per_xcd4) {
      const int unit = (blockIdx.x & 7) * per_xcd4 + nth;
      if (unit >= p.sec_units[1] || (p.row_cnt[unit / units_per_head(p.Sq, kShortWaves) / p.H] + 31) / 32 >= p.few_halves) return;
      attn_fwd_body<false, false, kShortWaves, false>(p, 0, 0, p.sec_units[1], 1, 0, 0, part, unit);
      return;
    }
    nth -= per_xcd4;
  }
  const int per_xcd = (p.sec_units[0] + 7) / 8;            // a contiguous run of (batch, head, query block) per XCD
  const int lin = (blockIdx.x & 7) * per_xcd + nth;
  if (nth >= per_xcd || lin >= p.sec_units[0]) return;
  const int nq = units_per_head(p.Sq, 1);
  const int bh = lin / nq, q32 = lin % nq;
  const int b = bh / p.H, h = bh % p.H;
  const int sk = p.row_cnt ? p.row_cnt[b] : p.Sk;
  TileWalk<SPARSE> walk{};
  int n_half = (sk + 31) / 32;
  if (MASKED && n_half < p.few_halves) return;
  if constexpr (SPARSE) {
    // plan entry of this block's 256 queries, row-block of its 64 (the lists of attn_fwd_body, walked in the same order)
    const int entry = q32 / (2 * kSparseRows), r = (q32 / 2) % kSparseRows;
    walk.shared = p.plan + (int64_t)entry * p.plan_stride;
    walk.own = walk.shared + (1 + r) * p.nKt;
    walk.n_shared = uniform_load(p.plan_cnt + entry * kSparseLists, 0);
    const int n = walk.n_shared + uniform_load(p.plan_cnt + entry * kSparseLists, 1 + r);
    // a last tile of at most 32 keys has one half tile: a full map is shared out as the dense call is
    const bool short_end = n > 0 && (n_half & 1) && walk(n - 1) == p.nKt - 1;
    n_half = 2 * n - (short_end ? 1 : 0);
  }
  const int h0 = wave * n_half / NW, h1 = (wave + 1) * n_half / NW;
  const char* kv = p.kv + (int64_t)bh * p.kv_bh_stride;

  WaveState<FP8> w;
  i32x4 kf[FP8 ? 4 : 8];
  if (h0 < h1) {
    const char* k = kv + (int64_t)walk(h0 >> 1) * p.kv_tile_stride + (h0 & 1) * (kKBytes / 2);
#pragma unroll
    for (int j = 0; j < (FP8 ? 4 : 8); ++j) kf[j] = *(const i32x4*)(k + (j * 64 + lane) * 16);
  }
  const f32x4 first_norms = ask_key_norms(p, bh, lane);
  // The queries, a 16-row block per wave for all waves (as in attn_fwd_body).  fp8: one scale
  // per 64 queries, so four waves look at the four blocks this block's 64 queries consist of, and two of them are it.
  const int mine = FP8 ? wave - 2 * (q32 & 1) : wave;      // which of the two 16-query blocks, if 0 or 1
  const bool prepares = (unsigned)mine < 2u;
  float x[32];
  float qscale = 1.0f;
  if (FP8 || prepares) {
    QRows in;
    NormLanes norm;
    ask_q_rows(in, p, b, h, q32 * 32 + 16 * mine, lane);
    load_norm_lanes(norm, p.q_norm_w, lane);
    q_rows_ready(x, in, p, norm, FP8 && !POW2 ? 1.0f : p.c, part + wave * kSlot, lane);
    if constexpr (FP8) {
      float amax = 0.f;
#pragma unroll
      for (int i = 0; i < 32; ++i) amax = fmaxf(amax, fabsf(x[i]));
      amax = wave_max(amax);
      if (lane == 0) s_amax[wave] = amax;
    }
  }
  if constexpr (FP8) {
    __syncthreads();
    qscale = fp8_block_scale(fmaxf(fmaxf(s_amax[0], s_amax[1]), fmaxf(s_amax[2], s_amax[3])), POW2);
    w.qe = e8m0_of(qscale);
  }
  if (prepares) {
    float n2 = 0.f;
    if constexpr (!FP8) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        bf16x8 t;
#pragma unroll
        for (int j = 0; j < 8; ++j) t[j] = (__bf16)x[ks * 8 + j];
        n2 = add_squares(t, n2);
        *(bf16x8*)(rows + ((mine * 4 + ks) * 64 + lane) * 16) = t;
      }
    } else {
      const float inv = 1.0f / qscale;
#pragma unroll
      for (int c2 = 0; c2 < 2; ++c2) {
        const i32x2 q0 = quant_fp8_piece(x + 16 * c2, inv), q1 = quant_fp8_piece(x + 16 * c2 + 8, inv);
        const i32x4 q = {q0[0], q0[1], q1[0], q1[1]};
#pragma unroll
        for (int wd = 0; wd < 4; ++wd) {
          const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8(q[wd], false);
          const auto hi = __builtin_amdgcn_cvt_pk_f32_fp8(q[wd], true);
          n2 += lo[0] * lo[0] + lo[1] * lo[1] + hi[0] * hi[0] + hi[1] * hi[1];
        }
        *(i32x4*)(rows + ((mine * 2 + c2) * 64 + lane) * 16) = q;
      }
      n2 *= qscale * qscale;
    }
    n2 = wave_max(fmaxf(wave_sum_groups(n2), 0.f));
    if (lane == 0) s_n2[mine] = n2;
  }
#pragma unroll
  for (int db = 0; db < 8; ++db)
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) w.o[db][qb] = f32x4{0.f, 0.f, 0.f, 0.f};
  w.m[0] = w.m[1] = kNoMax;
  w.l[0] = w.l[1] = 0.f;
  __syncthreads();
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    if constexpr (!FP8) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) w.qf[qb][ks] = *(const bf16x8*)(rows + ((qb * 4 + ks) * 64 + lane) * 16);
    } else {
      const i32x4 a0 = *(const i32x4*)(rows + ((qb * 2) * 64 + lane) * 16), a1 = *(const i32x4*)(rows + ((qb * 2 + 1) * 64 + lane) * 16);
      w.q8[qb] = i32x8{a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
    }
  }
  // The bound of attn_fwd_body: small enough, and no running maximum is needed.  As there, block-sparse rows without a tile that all of their
  // plan entry keeps run the maximum all the same: their largest weights are then 1 and carry no rounding.
  const float margin = FP8 ? (POW2 ? 1.08f : p.c * 1.08f) : 1.01f;
  const bool static_max = (SPARSE ? walk.n_shared : n_half) > 0 &&
                          __all(sqrtf(fmaxf(s_n2[0], s_n2[1])) * largest_key_norm<4>(p, bh, (sk + 31) / 32, first_norms, lane) * margin <= kStaticMaxLimit);
  const float* kscale = FP8 ? p.kscale + (int64_t)bh * p.nKt : nullptr;
  const float c = POW2 ? 1.0f : p.c * qscale;   // what the softmax still multiplies the logits by (fp8 absmax form only)
  if (static_max) narrow_loop<FP8, POW2, SPARSE, true>(w, kf, kv, p.kv_tile_stride, kscale, walk, h0, h1, sk, c, lane);
  else narrow_loop<FP8, POW2, SPARSE, false>(w, kf, kv, p.kv_tile_stride, kscale, walk, h0, h1, sk, c, lane);

#pragma unroll
  for (int db = 0; db < 8; ++db)
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) *(f32x4*)(part + wave * kSlot + ((db * 2 + qb) * 64 + lane) * 16) = w.o[db][qb];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const float l = wave_sum_groups(w.l[qb]);
    if (g4 == 0) part_l[wave][qb][c16] = l, part_m[wave][qb][c16] = w.m[qb];
  }
  __syncthreads();
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    float top = kNoMax, l = 0.f, a[NW];
    if (!static_max) {
#pragma unroll
      for (int j = 0; j < NW; ++j) top = fmaxf(top, part_m[j][qb][c16]);
    }
#pragma unroll
    for (int j = 0; j < NW; ++j) {
      a[j] = static_max ? 1.0f : __builtin_amdgcn_exp2f(part_m[j][qb][c16] - top);
      l += a[j] * part_l[j][qb][c16];
    }
    const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
    for (int i = 0; i < 8 / NW; ++i) {
      const int db = wave + i * NW;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NW; ++j) {
        const f32x4 t = *(const f32x4*)(part + j * kSlot + ((db * 2 + qb) * 64 + lane) * 16);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] += a[j] * t[r];
      }
      bf16x4 o;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = (__bf16)(acc[r] * inv);
      // elements d = 16*db + 4*g .. +3 of row 16*qb + c, chunks XOR-swizzled by the row as in attn_fwd_body
      *(bf16x4*)(rows + (16 * qb + c16) * 256 + (((2 * db + (g4 >> 1)) ^ c16) * 16) + 8 * (g4 & 1)) = o;
    }
  }
  __syncthreads();
  if (p.o_images) {
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const int ks = wave, r = 16 * rb + c16;
      bf16x8 v = *(const bf16x8*)(rows + r * 256 + (((4 * ks + g4) ^ c16) * 16));
      if (q32 * 32 + r >= p.Sq) v = bf16x8{};
      *(bf16x8*)((char*)p.o + (int64_t)(q32 * 2 + rb) * p.o_img_blk_stride + ((int64_t)h * (kD / 32) + ks) * 1024 + lane * 16) = v;
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 32 / (4 * NW); ++i) {
    const int row = (threadIdx.x >> 4) + i * 4 * NW;
    const bf16x8 v = *(const bf16x8*)(rows + row * 256 + ((c16 ^ (row & 15)) * 16));
    if (q32 * 32 + row < p.Sq)
      *(bf16x8*)((__bf16*)p.o + (int64_t)b * p.o_sb + (int64_t)h * p.o_sh + (int64_t)(q32 * 32 + row) * p.o_ss + 8 * c16) = v;
  }
}

// The relay form (bf16), for calls of many queries against few to some dozens of key tiles: one workgroup per CU for the whole call, twelve waves
// (three groups of four) that walk the tiles of a (batch, head) round and round.  A round is three units, a unit 128 queries, a group a unit.
// The ring of two tiles never drains: behind the last tile of a round comes the first of the next, already on its way under the
// last one's work.  The next queries come to LDS while the tiles are walked, each wave's to a place of its own, which
// the output goes through on its way out.
//
// What it is for: a workgroup of the other dense forms lasts a few tiles, and its start (the launch, keys known, queries, first tiles: one
// trip to memory behind the other) and its end cost as much as five of them.  Here a round costs 3.9 us and 2.1 to 2.2 a tile,
// short-key workgroups (three to a CU) 9 and 2.3, long ones 13 and 2.0.  Kernel, us, before / with it: 24 heads x 49,640 queries against
// 302 of 512 keys 249 / 228, 1,024 keys 543 / 505; x 14,830 against 1,536 keys 242 / 228; x 9,000 against 2,048 219 / 185 (rounds of
// long workgroups that are nearly empty at the end).  What bounds it now, by counters of 49,640 x 302: vector work.  A SIMD's MFMAs take 46 % of the
// cycles and its other vector instructions 54 %, at the same time 11 %; memory alone would take half of the time.  Between two rounds stores and
// queries of all CUs (8 KiB of each a wave: 96 KiB a CU) come at once.
// Queries are copied four neighbouring lanes to 64 bytes: lanes in the order of the operand images, neighbours in different rows, keep a CU's
// vector-memory path busy four times as long (16 against 60 bytes a clock, one workgroup alone; stores the same).
// Measured and not kept: the three groups a third of a round apart, each handing over while the others walk tiles (302 keys 243 against
// 237, one key tile 160 / 140: every step lasts as long as its slowest wave), and staggered CUs (1 to 2 %, as much as the stagger costs).
constexpr int kRelayWaves = 12, kRelayGroups = 3;

// The lane's number, made where it is used: kept from round to round, what is made of it does not fit the registers.
__device__ __forceinline__ int lane_here() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}

// The units [at, end) of this workgroup: equal shares of all units or, where a key mask leaves the entries of a batch unequal keys (which the
// device alone knows), of their weights (relay_weight): in equal shares half of the CUs may have the short entry and wait for the other
// half.  us, long form (whose queues even this out) / equal counts / by weight: 2 x 24 heads x 20,000 queries against 2,500 keys, 64 and 2,500 of
// them valid, 849 / 934 / 536, 625 and 2,500 852 / 937 / 629, all 961 / 958 / 950; x 14,830 against 1,500, 64 and 1,500 424 / 443 / 273; 8 x 12 x 4,000
// against 2,000, 250 to 2,000 290 / 339 / 227; x 49,640 against 512, 64 and 512 598 (short-key form) / 544 / 425.
struct RelayRun {
  int at, end;
};
template <bool ROPE>
__device__ __forceinline__ RelayRun relay_run(const FwdParams& p, int per_head) {
  const int wgs = gridDim.x, rank = (blockIdx.x & 7) * (wgs >> 3) + (blockIdx.x >> 3);   // a contiguous run per XCD and workgroup
  const int per_entry = p.H * per_head, all = p.B * per_entry;
  // (entries of fewer than four units: every run has some, and looking at all of them costs as much as it evens out)
  if (!p.row_cnt || p.B == 1 || per_entry < 4) return {relay_cut(rank, all, per_head, wgs, !ROPE), relay_cut(rank + 1, all, per_head, wgs, !ROPE)};
  // Every lane has B / 64 entries.  (64 at a time, with a prefix sum for each, took 4 us for 300 entries, 21 for 1,500.)
  const int lane = threadIdx.x & 63, each = (p.B + 63) / 64, first = min(lane * each, p.B), last = min(first + each, p.B);
  int w = 0;
  for (int b = first; b < last; ++b) w += relay_weight(p.row_cnt[b]);
  int sum = w;                                           // over this lane and those before it
#pragma unroll
  for (int d = 1; d < 64; d *= 2) {
    const int x = __shfl_up(sum, d, 64);
    if (lane >= d) sum += x;
  }
  const int total = __builtin_amdgcn_readlane(sum, 63);
  RelayRun run{all, all};                                // (no entry holds the end of the last run)
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    int into = (rank + i) * total - (sum - w) * wgs;     // (in 1 / wgs of a weight; 65,535 entries of at most 42 each)
    const unsigned long long here = __ballot(into >= 0 && into < w * wgs);
    if (here) {                                          // (one lane)
      int b = first, entry = 0;
      for (; b < last; ++b, into -= entry * wgs) {
        entry = each == 1 ? w : relay_weight(p.row_cnt[b]);
        if (into < entry * wgs) break;
      }
      const int unit = b * per_entry + relay_unit(into, max(entry, 1), wgs, per_entry);
      (i ? run.end : run.at) = __builtin_amdgcn_readlane(unit, __builtin_ctzll(here));
    }
  }
  return run;
}

template <bool ROPE>
__global__ __launch_bounds__(64 * kRelayWaves, 1) void attn_fwd_relay_kernel(FwdParams p) {
  constexpr int kTile = kKTileBytes + kVTileBytes;
  __shared__ __attribute__((aligned(1024))) char ring[2 * kTile];
  __shared__ __attribute__((aligned(1024))) char rows[kRelayWaves * kQBlkBytes];   // every wave's next 32 queries
  static_assert(sizeof(ring) + sizeof(rows) <= 163840, "all of a CU's LDS");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = wave / kShortWaves, wq = wave & (kShortWaves - 1);
  char* own = rows + wave * kQBlkBytes;
  const int per_head = units_per_head(p.Sq, kShortWaves);
  RelayRun run = relay_run<ROPE>(p, per_head);
  unsigned long long third;                              // lanes of a tile's third copy: it is 32 KiB, for twelve waves
  asm volatile("s_cmp_lt_i32 %1, %2\n\ts_cselect_b64 %0, -1, 0" : "=s"(third) : "s"(wave), "n"(kTile / 1024 - 2 * kRelayWaves) : "scc");
  const unsigned rows_lds = (unsigned)(size_t)(__attribute__((address_space(3))) char*)own;
  const unsigned ring_lds = (unsigned)(size_t)(__attribute__((address_space(3))) char*)ring;

  NormLanes norm;
  load_norm_lanes(norm, p.q_norm_w, lane);
  const float top_weight = wave_max(fmaxf(fabsf(norm.w[0]), fabsf(norm.w[1]))) * p.c;

#pragma unroll 1
  while (run.at < run.end) {
    // a stretch: the units of one (batch, head), three to a round
    WaveState<false> w;
    const int bh = run.at / per_head, first = run.at - bh * per_head, count = min(run.end - run.at, per_head - first);
    run.at += count;
    const int b = bh / p.H, h = bh % p.H;
    const int sk = p.row_cnt ? uniform_load(p.row_cnt, b) : p.Sk;
    const int n = (sk + kTileKeys - 1) / kTileKeys, ring_n = max(n, 1);
    const char* kv = p.kv + (int64_t)bh * p.kv_bh_stride + wave * 1024;
    const int l0 = lane_here();
    const float key_norm = n > 0 ? largest_key_norm(p, bh, (sk + 31) / 32, ask_key_norms(p, bh, l0), l0) : 0.f;
    // a normalised row is no longer than sqrt(D) times the largest weight, whatever the queries (tables may hold what they like: a rotated
    // one is looked at itself)
    const bool sure = !ROPE && p.q_norm_w && __all(sqrtf((float)kD) * top_weight * key_norm * 1.01f <= kStaticMaxLimit);
    int ahead = ring_n - 1, slot = 0;                    // the next tile to copy; slot of the tile in use (a round begins with the last tile)
    auto copy = [&](int to) {
      const char* g = kv + (int64_t)ahead * p.kv_tile_stride;
      char* d = ring + to * kTile + wave * 1024;
      lds_dma16(g, lane * 16, d);
      lds_dma16(g + kRelayWaves * 1024, lane * 16, d + kRelayWaves * 1024);
      asm volatile("s_mov_b32 m0, %2\n\ts_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1"
                   :
                   : "v"(lane * 16), "s"(g + 2 * kRelayWaves * 1024), "s"(ring_lds + to * kTile + (wave + 2 * kRelayWaves) * 1024), "s"(third)
                   : "memory", "m0");
      ahead = ahead + 1 == ring_n ? 0 : ahead + 1;
    };
    auto barrier = [&]() {
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    };
    // 16 of a block's 32 rows of queries into `own`, four neighbouring lanes to the 64 bytes of a row: piece g of row c of image ks comes to
    // lie at 4c + (g ^ c/4).  Rows past the end are the last one again.
    auto ask_rows = [&](int q32, int qb) {
      const int l = lane_here();
      const int row0 = min(q32 * 32 + 16 * qb, p.Sq - 1);
      const char* q = (const char*)p.q + ((int64_t)b * p.q_sb + (int64_t)h * p.q_sh + (int64_t)row0 * p.q_ss) * 2;
      const unsigned off = (unsigned)min(l >> 2, p.Sq - 1 - row0) * ((unsigned)p.q_ss * 2) + ((l ^ (l >> 4)) & 3) * 16;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                     :
                     : "v"(off), "s"(q + 64 * ks), "s"(rows_lds + (4 * qb + ks) * 1024)
                     : "memory", "m0");
    };
    auto q32_of = [&](int unit) { return (first + unit) * kShortWaves + wq; };
    bool static_max = sure;
    bf16x8 rows_now[2][4];
    auto read_rows = [&]() {
      const int l = lane_here(), c16 = l & 15;
#pragma unroll
      for (int i = 0; i < 8; ++i) rows_now[i >> 2][i & 3] = *(const bf16x8*)(own + i * 1024 + c16 * 64 + (((l >> 4) ^ (c16 >> 2)) * 16));
    };
    auto prepare = [&](int q32, int q32_next) {
      const int l = lane_here();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // nothing is read from `own` any more: the next rows may come
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        float x[32];
        norm_row(x, rows_now[qb], p.q_norm_w != nullptr, p.q_eps, norm, p.c);
        if constexpr (ROPE) {
          Rows16 cos, sin;
          RopeQuarter rope;
          ask_rows16(cos, (const char*)p.q_cos, kD / 2 * sizeof(float), q32 * 32 + 16 * qb, p.Sq - 1, l);
          ask_rows16(sin, (const char*)p.q_sin, kD / 2 * sizeof(float), q32 * 32 + 16 * qb, p.Sq - 1, l);
          turn_table(cos, rope.c, p.q_rope_mode, own, l);
          turn_table(sin, rope.s, p.q_rope_mode, own, l);
          rope_row(x, p.q_rope_mode, rope);
        }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          bf16x8 q;
#pragma unroll
          for (int j = 0; j < 8; ++j) q[j] = (__bf16)x[8 * ks + j];
          w.qf[qb][ks] = q;
        }
        __builtin_amdgcn_sched_barrier(0);
        if (!ROPE && q32_next >= 0) ask_rows(q32_next, qb);
      }
      // (behind the tables: the wait for those is one for everything before them, and they go through `own`)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (ROPE && q32_next >= 0) ask_rows(q32_next, 0), ask_rows(q32_next, 1);
      if (!sure) {
        // the bound of these queries themselves
        float n2[2][4];
#pragma unroll
        for (int i = 0; i < 8; ++i) n2[i >> 2][i & 3] = add_squares(w.qf[i >> 2][i & 3], 0.f);
        const float top = fmaxf(wave_sum_groups((n2[0][0] + n2[0][1]) + (n2[0][2] + n2[0][3])), wave_sum_groups((n2[1][0] + n2[1][1]) + (n2[1][2] + n2[1][3])));
        static_max = __all(sqrtf(top) * key_norm * 1.01f <= kStaticMaxLimit);
      }
      w.m[0] = w.m[1] = kNoMax;
    };
    auto no_keys = [&]() {
#pragma unroll
      for (int db = 0; db < 8; ++db)
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) w.o[db][qb] = f32x4{0.f, 0.f, 0.f, 0.f};
      w.l[0] = w.l[1] = 0.f;
    };
    // every wave is past the last stretch's ring, and its last copies have landed
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    barrier();
    if (grp < count) ask_rows(q32_of(grp), 0), ask_rows(q32_of(grp), 1);
    copy(0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    barrier();
    copy(1);
    // A step: its tile is in its slot for every wave (own copies: vmcnt, the others': barrier), and every wave is past the tile before, whose
    // slot takes the tile after this one.  The first step's tile, and the copies of the second's, were seen to at the end of the round before.
    // The step that begins the sums takes the last tile: its keys past the end start from -inf, and O^T and the row sums from nothing.
#define PKH3_RELAY_STEP(STATIC, FIRST, I)                                                               \
  {                                                                                                     \
    if (!(FIRST)) {                                                                                     \
      if ((I) == 1 && slack) asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)" ::: "memory");               \
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");                                  \
      barrier();                                                                                        \
    }                                                                                                   \
    const char* kbuf = ring + slot * kTile;                                                             \
    const int l = (FIRST) ? lane_here() : lane;                                                         \
    qk_tile<false, true, 4, false, FIRST>(w, kbuf, kbuf + kKTileBytes, l, 0, sk - kTileKeys * (n - 1)); \
    slot ^= 1;                                                                                          \
    if (!(FIRST)) copy(slot);                                                                           \
    softmax_pv_tile<false, STATIC, true, false, false, FIRST>(w, kbuf + kKTileBytes, 1.0f, 0, l);       \
  }
    auto round_ends = [&]() {
      // the next round's queries and first tile are there, and its second takes the place of the last tile
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      barrier();
      copy(slot ^ 1);
    };
    bool stored = false;
    if (grp < count) read_rows();
#pragma unroll 1
    for (int unit = grp; unit < count; unit += kRelayGroups) {
      const bool more = unit + kRelayGroups < count;
      prepare(q32_of(unit), more ? q32_of(unit + kRelayGroups) : -1);
      const bool slack = stored && more;                 // eight stores and eight loads were issued after the copies of the second tile
      if (n == 0) {
        no_keys();
      } else if (static_max) {
        PKH3_RELAY_STEP(true, true, 0)
#pragma unroll 1
        for (int i = 1; i < n; ++i) PKH3_RELAY_STEP(true, false, i)
      } else {
        PKH3_RELAY_STEP(false, true, 0)
#pragma unroll 1
        for (int i = 1; i < n; ++i) PKH3_RELAY_STEP(false, false, i)
      }
      PKH3_MFMA_DRAIN(w);
      round_ends();
      const int q32 = q32_of(unit);
      float inv[2];
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        const float lt = wave_sum_groups(w.l[qb]);
        inv[qb] = lt > 0.f ? 1.0f / lt : 0.f;
      }
      read_rows();                                       // (the next unit's, if there is one) before the output takes their place
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      const int l = lane_here();
      __builtin_amdgcn_sched_barrier(0);
      store_output(p, w, inv, own, b, h, q32, l);
      __builtin_amdgcn_sched_barrier(0);
      stored = q32 * 32 + 32 <= p.Sq;
    }
    if (count % kRelayGroups != 0 && grp >= count % kRelayGroups) {
      // the last round has no unit for this group: it copies and synchronises
#pragma unroll 1
      for (int i = 0; i < n; ++i) {
        if (i > 0) {
          asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
          barrier();
        }
        slot ^= 1;
        if (i > 0) copy(slot);
      }
      round_ends();
    }
#undef PKH3_RELAY_STEP
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // no copy may arrive after the workgroup has given its LDS back
}

static int blocks_of(int workgroups) { return (workgroups + 7) / 8 * 8; }

// How a long dense call ends.  One 12-wave workgroup per CU at a time: the call runs in rounds of `cus` workgroups, and
// `rest` units left for a last round leave CUs idle for a whole workgroup's duration.  Sharing each of those units out
// among P workgroups (1/P of the key tiles each) gives workgroups of 1/P of the duration that again run in rounds of
// `cus`; one or two such sections (P1 for the units that fill a round, P2 for what is left) end the call in
// 1/P1 + 1/P2 of a whole round.  The cheapest plan within the scratch (one partial result per workgroup) is taken.
struct TailPlan {
  int units[2], parts[2];
};
static TailPlan plan_tail(int rest, int cus, int n_tiles, int64_t max_workgroups) {
  TailPlan best{{rest, 0}, {1, 1}};
  if (rest <= 0 || cus <= 0) return best;
  const int pmax = max(1, min(kMaxParts, n_tiles / kMinPartTiles));
  double best_cost = 1.0;
  auto consider = [&](int u1, int p1, int u2, int p2) {
    const int64_t wgs = (p1 > 1 ? (int64_t)u1 * p1 : 0) + (p2 > 1 ? (int64_t)u2 * p2 : 0);
    if (wgs > max_workgroups) return;
    const double cost = 1.0 / p1 + (u2 > 0 ? 1.0 / p2 : 0.0);
    if (cost < best_cost - 1e-9) best_cost = cost, best = TailPlan{{u1, u2}, {p1, p2}};
  };
  const int p_all = min(pmax, cus / rest);     // every unit of the rest in one round of workgroups
  if (p_all > 1) consider(rest, p_all, 0, 1);
  for (int p1 = 2; p1 <= pmax; ++p1) {
    const int u1 = cus / p1;                   // units that fill one round at p1
    if (u1 <= 0 || u1 >= rest) continue;
    const int p2 = min(pmax, cus / (rest - u1));
    if (p2 >= 1) consider(u1, p1, rest - u1, p2);
  }
  return best;
}

// Whether a dense call runs in the relay form.  At least a round and a third per CU (with fewer the other forms' rounds come out as they do), and
// as long as a round's start and end weigh: to 40 key tiles.  Below 17, where the short-key form takes over from the long one, the gain is what
// the start cost: from 8 tiles on, and where the queries' tables are not read besides (each wave waits for them between two rounds).  Other form /
// relay, us, 24 heads, without rotation, 512, 1,024, 1,536, 2,048 and 3,072 keys: 6,000 rows 45.0 / 43.1, 75.3 / 70.9, 115 / 99, 145 / 127,
// 206 / 183; 9,000 61.0 / 61.0, 105.5 / 101.7, 173 / 143, 219 / 185, 296 / 269; 27,000 179 / 169, 299 / 282, 427 / 398, 534 / 517, 759 / 761; 49,640
// 327 / 300, 543 / 505, 744 / 727, 951 / 933, 1,367 / 1,361; 256 keys from 40.1 / 41.7 to 122 / 111.  With rotation: 14,830 rows
// 105 / 114 (512 keys), 175 / 178 (1,024), 262 / 245, 326 / 312; 4,000 rows (three units a CU) 74.7 / 77.2 against 1,536 keys.
// What the figures leave out, from 600 calls of other sizes (whole calls, us):
// - against the short-key form, about five units a CU where an XCD does not have whole heads (31 heads of 41 units x 896 keys 79 / 84, 33 of 40 x 704 71
//   / 76, 54 of 25 x 640 69 / 72.5, 45 of 34 x 640 71 / 74; 48 of 31 x 832 89 / 83, 24 of 51 to 63 0.98 to 1.05 times as fast, and from 6.5 units a CU on
//   0.98 to 1.07, whatever the heads), and heads of no more than eight units with fewer than ten a CU (210 of 6 x 512 63 / 69, 516 of 4 x 1,024
//   245 / 252; 400 of 7 x 838, eleven a CU, 233 / 227): of 354 calls that come here against few tiles, 6 are more than 2 % behind and 256 ahead;
// - with a key mask, which may leave one or two tiles of the few (24 heads, 512 keys, valid 64, 100, 190 and 302: 6,500 rows 25.7 / 28.1, 29.1 / 31.4, 32.4
//   / 34.8, 40.1 / 42.7; 14,830 41.1 / 43.1, 47.9 / 49.4, 56.3 / 56.6, 72.5 / 73.1; from 14 units a CU on only a single tile is behind: 49,640
//   143 / 147, 169 / 152, 197 / 173, 250 / 225);
// - against the long form, the keys of all heads being walked at once: where they do not fit the 256 MB cache behind the L2s and that form's
//   blocks of 384 rows are full (tiles of all heads, us: 7,696 561 / 588, 7,956 744 / 779, 10,791 592 / 626; 7,068 529 / 515, 5,874 615 / 603; blocks
//   full to 0.87 7,099 451 / 416, 7,917 522 / 486).
static bool relay_form(const FwdParams& p, int cus) {
  const int64_t per_head = units_per_head(p.Sq, kShortWaves), units = p.B * p.H * per_head;
  if (p.fp8 || p.plan || cus < 8 || units <= 4 * cus || p.nKt > 40 || p.q_ss > (1 << 26)) return false;   // (16 rows of queries lie within 32 bits of each other)
  if (p.nKt > kShortMaxTiles) return (int64_t)p.B * p.H * p.nKt <= 7168 || 10 * per_head < 27 * units_per_head(p.Sq, kDenseWaves);
  if (p.nKt < 8 || p.q_rope_mode || (p.row_cnt && units <= 14 * cus)) return false;
  return per_head > 8 ? 2 * units > 13 * (int64_t)cus || (p.B * p.H) % 8 == 0 : units > 10 * cus;
}

// Which form of the kernel a call takes.
AttnForm attn_form(const FwdParams& p, int cus) {
  if (p.long_key_kernel) return p.plan ? kFormSparse : kFormLong;
  cus = max(cus, 1);
  auto units = [&](int blocks) { return p.B * p.H * units_per_head(p.Sq, blocks); };
  const int n4 = units(kShortWaves), n32 = units(1), n_half = (p.Sk + 31) / 32;
  const int per_cu = (n4 + cus - 1) / cus;
  // A narrow workgroup of an fp8 call reads the 64 queries its scale is of and writes 32 of them: with the output in the queries' place it
  // could read rows its neighbour has written.  The other forms read no query but those they write.
  const bool narrow = !(p.fp8 && p.in_place);
  // Block-sparse calls of at most four 32-query blocks per CU take the narrow form, whatever their maps (the kept tiles are
  // known on the device only).  Narrow / 8-wave form, 24 heads, us, at densities 0.03, 0.1, 0.3 and 1 (with the diagonal): 641 rows (504
  // blocks) 8.5 / 12.6, 10.2 / 18.2, 11.0 / 19.2, 13.7 / 21.5; 900 rows (696) 13.4 / 14.1, 15.6 / 17.3, 17.2 / 27.1, 22.0 / 26.2; 1,300 rows
  // (984) 16.0 / 17.5, 17.7 / 21.3, 21.3 / 30.7, 32.5 / 33.4 (fp8 17.1 / 17.4, 18.7 / 20.7, 21.0 / 28.7, 28.9 / 32.1).  Behind on maps of one
  // tile a row-block alone, from three blocks per CU on: 15.0 / 11.5 at 1,300 rows.  From five blocks per CU on it is behind on more of
  // them: 1,500 rows (1,128) 17.6 / 18.6, 20.7 / 24.0, 26.6 / 40.8, 45.2 / 39.2; 1,700 (1,296) 19.5 / 15.9, 22.5 / 22.7, 29.1 / 39.5,
  // 55.4 / 41.9.  fp8 calls of many keys take it up to five blocks per CU: 10 heads x 4,000 rows (1,250), densities 0.03, 0.1,
  // 0.3, 0.6 and 1: 24.1 / 23.9, 30.1 / 36.5, 44.4 / 62.2, 58.2 / 75.7, 82.1 / 76.7.
  if (p.plan) return narrow && n32 <= (p.fp8 && n_half >= 96 ? 5 : 4) * cus ? kFormNarrow : kFormSparse;
  // Dense calls of at most two short-key workgroups per CU leave a long form's chip half empty, whatever the number of keys.  They
  // take the narrow form where it is estimated shorter, else the short-key form.  The estimates are straight lines through
  // kernel times in microseconds (bf16; fp8 lies within a tenth of them): the narrow form, a start and a merge and 0.135 per half tile
  // for every 32-query block a CU gets; the short-key form, a half tile per 0.60 with one workgroup on a CU and per 0.87
  // with two (the plain loop, as in the figures here; the pipelined one, which takes these calls, needs 0.48 and 0.82: the line has not been
  // moved with it).  Measured (narrow / short-key / long): 240 blocks x 10 half tiles 7.9 / 11.1 / 17.2, 504 x 63 23.9 / 41.9 / 62.9,
  // 768 x 64 34.8 / 43.4 / 63.7, 1,256 x 157 115 / 128 / 144; on the other side of the line 456 x 4 7.9 / 7.7 / 12.6,
  // 816 x 34 27.3 / 26.3 / 38.5, 1,504 x 94 86 / 81 / 90, 1,896 x 79 95 / 73 / 78.  With three short-key workgroups per CU the
  // long form is ahead as long as its own workgroups are no more than the CUs (2,256 x 94: 114 / 94), and behind when a few
  // are left over for a second round (3,000 x 125: 165 / 218).
  if (narrow && per_cu <= 2 && 3.2f + (n32 + cus - 1) / cus * (0.135f * n_half + 2.7f) < 5.0f + (per_cu == 1 ? 0.60f : 0.87f) * n_half) return kFormNarrow;
  if (relay_form(p, cus)) return kFormRelay;
  const bool few = per_cu <= 2 || (per_cu == 3 && units(kDenseWaves) > cus);
  return few || p.nKt <= kShortMaxTiles ? kFormShort : kFormLong;
}

// Half tiles of valid keys from which a masked call of `n32` blocks of 32 queries (`n4` of 128) is better off in the narrow form: where
// straight lines through kernel times in us meet.  Narrow: 5.9 while every CU has one block, then 2.6 and 4.2 for every round of two
// blocks per CU, and 0.125 per half tile for every block a CU gets; short-key: 5.5 and 0.585 per half tile with one
// workgroup on a CU, 8.0 and 0.80 with two.  Measured (narrow / short-key): 40 blocks x 1 half tile 6.0 / 5.9, x 2 6.1 / 6.4; 288 x 1
// 7.1 / 6.0, x 4 7.5 / 7.8; 504 x 1 7.4 / 6.3, x 4 7.9 / 8.1; 656 x 1 10.8 / 6.4, x 16 16.4 / 15.3, x 32 22.0 / 24.3; 1,056 x 1
// 15.4 / 8.6, x 16 22.9 / 21.0, x 32 33.2 / 33.2, x 75 59.4 / 64.7.
static int narrow_from(int n32, int n4, int cus) {
  const int per_cu = (n32 + cus - 1) / cus, rounds = (n32 + 2 * cus - 1) / (2 * cus);
  const bool one = n4 <= cus;
  const float start = (per_cu == 1 ? 5.9f : 2.6f + 4.2f * rounds) - (one ? 5.5f : 8.0f);
  const float gain = (one ? 0.585f : 0.80f) - 0.125f * per_cu;   // per half tile
  return gain > 0.f ? (int)ceilf(start / gain) : INT_MAX;
}

template <bool FP8, bool POW2 = false>
static hipError_t launch_fp(FwdParams p, int cus, hipStream_t st) {
  auto units = [&](int blocks) { return p.B * p.H * units_per_head(p.Sq, blocks); };
  for (int i = 0; i < kSections; ++i) p.sec_units[i] = p.sec_blocks[i] = 0, p.sec_parts[i] = 1;
  const AttnForm form = attn_form(p, cus);
  if (form == kFormNarrow) {
    const int n = units(1);
    p.queue_next = nullptr;
    p.sec_units[0] = n;
    const dim3 grid(blocks_of(n)), block(64 * kNarrowWaves);
    if (p.plan) {
      hipLaunchKernelGGL((attn_fwd_narrow_kernel<FP8, POW2, true>), grid, block, 0, st, p);
    } else if (!FP8 && p.row_cnt) {
      p.sec_units[1] = units(kShortWaves);
      p.few_halves = narrow_from(n, p.sec_units[1], cus);
      hipLaunchKernelGGL((attn_fwd_narrow_kernel<false, false, false, true>), dim3(blocks_of(p.sec_units[1]) + blocks_of(n)), block, 0, st, p);
    } else {
      hipLaunchKernelGGL((attn_fwd_narrow_kernel<FP8, POW2, false>), grid, block, 0, st, p);
    }
    return hipGetLastError();
  }
  if (form == kFormSparse) {
    const int n = p.B * p.H * (p.nQ64 / kSparseRows);
    p.sec_units[0] = n;
    int wgs = n;
    if (p.queue_next && cus > 0 && n >= cus) {
      // at least a round of workgroups: one per CU (the LDS of the form holds no second), units from the work queues
      hipError_t e = p.counters_clear ? hipSuccess : launch_fill_zero((unsigned*)p.queue_next, kQueues, st);
      if (e != hipSuccess) return e;
      wgs = cus;
    } else {
      p.queue_next = nullptr;
    }
    hipLaunchKernelGGL((attn_fwd_kernel<FP8, true, kSparseWaves, POW2>), dim3(blocks_of(wgs)), dim3(64 * kSparseWaves), 0, st, p);
    return hipGetLastError();
  }
  if constexpr (!FP8) {
    if (form == kFormRelay) {
      p.queue_next = nullptr;
      const dim3 grid(cus / 8 * 8), block(64 * kRelayWaves);
      if (p.q_rope_mode) hipLaunchKernelGGL(attn_fwd_relay_kernel<true>, grid, block, 0, st, p);
      else hipLaunchKernelGGL(attn_fwd_relay_kernel<false>, grid, block, 0, st, p);
      return hipGetLastError();
    }
  }
  if (form == kFormShort) {
    p.queue_next = nullptr;
    p.sec_units[0] = units(kShortWaves);
    // Up to two workgroups per CU: the pipelined loop, which needs the registers of three waves for two.  From the third on, three
    // to a CU overlap better (24 heads, us, plain / pipelined: 216 workgroups x 34 halves 27.8 / 22.8 and x 64 44.3 / 37.6, 168 x 25 20.5 / 18.3,
    // 384 x 63 57.4 / 54.8, 504 x 82 78.6 / 75.2; 960 x 16 38.9 / 38.0, 2,784 x 16 94.8 / 99.1, 9,312 x 10 249 / 264; fp8 alike).
    if (p.sec_units[0] <= 2 * cus) {
      hipLaunchKernelGGL((attn_fwd_kernel<FP8, false, kShortWaves, POW2, true>), dim3(blocks_of(p.sec_units[0])), dim3(64 * kShortWaves), 0, st, p);
      return hipGetLastError();
    }
    hipLaunchKernelGGL((attn_fwd_kernel<FP8, false, kShortWaves, POW2>), dim3(blocks_of(p.sec_units[0])), dim3(64 * kShortWaves), 0, st, p);
    return hipGetLastError();
  }
  const int n = units(kDenseWaves);
  const int whole = cus > 0 ? n / cus * cus : n, rest = n - whole;
  p.sec_units[0] = n;
  int shared = 0;   // units whose key tiles are shared out: they have arrival counters
  if (whole > 0 && rest > 0 && !p.long_key_kernel && p.split_cnt && p.split_scratch_bytes) {
    const int64_t cap = (int64_t)(p.split_scratch_bytes / ((size_t)kDenseWaves * kMergeBytes));
    const TailPlan t = plan_tail(rest, cus, p.nKt, cap);
    if (t.parts[0] > 1 || t.parts[1] > 1) {
      p.sec_units[0] = whole;
      p.sec_units[1] = t.units[0], p.sec_parts[1] = t.parts[0];
      p.sec_units[2] = t.units[1], p.sec_parts[2] = t.parts[1];
      shared = (t.parts[0] > 1 ? t.units[0] : 0) + (t.parts[1] > 1 ? t.units[1] : 0);
    }
  }
  // calls of at least one round of workgroups take their whole units from the work queues
  const bool queues = whole > 0 && !p.long_key_kernel && p.queue_next;
  if (!queues) p.queue_next = nullptr;
  if ((queues || shared > 0) && !p.counters_clear) {
    // queue positions and arrival counters start at zero (the arrival counters follow the queue slots)
    hipError_t e = launch_fill_zero((unsigned*)(p.split_cnt - kQueueSlots), kQueueSlots + shared * kDenseWaves, st);
    if (e != hipSuccess) return e;
  }
  int blocks = 0;
  for (int i = 0; i < kSections; ++i) {
    int wgs = p.sec_units[i] * p.sec_parts[i];
    // the spare workgroups of the faster XCDs: an eighth on top of the whole units; as many again for the shared
    // units of the call's end, where an XCD that is through early can take most of a slower one's share
    if (queues && wgs > 0) wgs += i == 0 ? max(kQueues, wgs / 8) : wgs;
    blocks += p.sec_blocks[i] = blocks_of(wgs);
  }
  hipLaunchKernelGGL((attn_fwd_dense_kernel<FP8, POW2>), dim3(blocks), dim3(64 * kDenseWaves), 0, st, p);
  return hipGetLastError();
}

// CUs of the current device, asked once per device; threads that race here store the same value
hipError_t device_cu_count(int* out) {
  static std::atomic<int> cu_count[64];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  int cus = 0;
  if (dev >= 0 && dev < 64) {
    cus = cu_count[dev].load(std::memory_order_relaxed);
    if (cus == 0) {
      e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
      if (e != hipSuccess) return e;
      cu_count[dev].store(cus, std::memory_order_relaxed);
    }
  }
  *out = cus;
  return hipSuccess;
}

hipError_t launch_attn_fwd(const FwdParams& p, hipStream_t st) {
  int cus = 0;
  hipError_t e = device_cu_count(&cus);
  if (e != hipSuccess) return e;
  if (p.fp8 && p.fp8_pow2) return launch_fp<true, true>(p, cus, st);
  if (p.fp8) return launch_fp<true>(p, cus, st);
  return launch_fp<false>(p, cus, st);
}

}  // namespace pkh3
