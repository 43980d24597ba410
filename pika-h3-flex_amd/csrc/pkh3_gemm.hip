// Projection GEMMs around the attention kernel (gfx950, bf16 MFMA 16x16x32, fp32 accumulation):
//   to_q / to_k / to_v  (+ LoRA)  from the modulated hidden states, with the K side's RMSNorm + rotation
//                       (+ fp8 quantisation) and the K / V operand-image layout done in the epilogue, so that
//                       K and V go from the accumulators straight into the records the attention kernel reads
//   to_out.0 (+ LoRA)   from the attention output, with bias, per-row gate and residual in the epilogue
//   LoRA down-projection x A^T, written as operand images for the second K segment of the GEMMs above
//
// Operands.  Both operands come as 1 KiB operand images (16 rows x 32 contraction elements, lane l holds row
// l%16, elements 8*(l/16)..+7 -- the shape of the attention kernel's K images): activations as [16-token
// block][k-step], weights as [16-feature block][k-step] (packed once when the weights are loaded).  They move
// HBM/L2 -> LDS -> VGPR as straight 16-byte copies, like the K/V tiles of the attention kernel: direct-to-LDS loads
// into a ring of three slots (four where a launch's tiles have a CU each), as many chunks ahead, one barrier per chunk.  Since the two MFMA operands have the same register
// form, one pair of images serves both orientations:
//   C^T = W x^T  (features down the accumulator registers, one token per lane)   Q, K, row-major outputs
//   C   = x W^T  (tokens down the registers, one feature per lane)               V images
// Weight rows are stored permuted inside each 128-feature head so that, in the C^T form, the 32 accumulator
// values a lane holds for a token are the four 8-element pieces p8 = 4*ks + g (elements 32*ks + 8*g .. +7) of that
// token's head row: exactly what lane (g, c) of the attention kernel's K images carries, so the K epilogue stores
// its accumulators (after norm and rotation) without any lane movement, and so do the row-major and the V epilogues.
//
// Work split.  Workgroup = 4 waves, one per SIMD = 256 features x 256, 192, 128 or 64 tokens; wave (fh, th) owns features
// fh*128..+127 (one head) x half of the tokens (TB = 8, 6, 4 or 2 blocks of 16).  Eight waves of
// 128 x 64 read 96 KiB of LDS for a 32-wide k-chunk; four of 128 x 128 read 64 KiB and need no second wave to cover their
// issue, but accumulators of 256 registers a lane, which live in the accumulator half of the register file.  What bounds it
// (counters, to_q/to_k/to_v, hidden size 3,072): in long launches the MFMAs, at the clock the part holds under them: pipe busy
// 68 % at 1.98 GHz at 48,360 tokens (eight waves: 63 % at 1.82), 75 % at 1.69 GHz at 15,342 (TB = 4), LDS busy 17 and 28 %; in
// short ones the CUs without a workgroup and, with one workgroup of TB = 2 alone on a CU, the wait for its copies at
// every chunk's barrier (MFMA 30 %, waiting 36 % of the time, LDS 19 %).  LoRA is a second K segment: k-chunks beyond the hidden size take their activation images from the
// down-projected rows (x A^T, scaled) and their weight images from B.
#include <type_traits>

#include "pkh3_common.h"
#include "pkh3_index.h"
#include "pkh3_internal.h"

namespace pkh3 {

constexpr int kGemmWaves = 4;                       // two 128-feature heads x two token halves
constexpr int kGemmFeatures = 256;                  // features per workgroup
constexpr int kGemmRing = 3;                        // ring slots (R; see launch_gemm): one 32-wide k-chunk of weight and activation images each
constexpr int kGemmWPieces = kGemmFeatures / 16;    // 1 KiB weight images of a chunk

// The two halves of a direct-to-LDS copy (see lds_dma16 in pkh3_attn_fwd.hip: wave-uniform base address, per-lane byte
// offset, tracked by vmcnt): where the next one goes, and the copy.  `lanes`: all or none -- past the last chunk
// the copies are still issued, so that the waits count the same, but move nothing.
__device__ __forceinline__ void dma_to(unsigned lds_addr) { asm volatile("s_mov_b32 m0, %0" ::"s"(lds_addr) : "m0"); }
__device__ __forceinline__ void dma_from(const char* g, unsigned lane_off, unsigned long long lanes) {
  asm volatile("s_mov_b64 exec, %2\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1"
               :
               : "v"(lane_off), "s"(g), "s"(lanes)
               : "memory");
}
// operand of s_waitcnt: at most `vm` copies and `lgkm` LDS reads still on their way
constexpr int waitcnt_vm_lgkm(int vm, int lgkm) { return (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | (lgkm << 8); }

// c += a b.  Written as an instruction because the compiler, left to place 256 accumulator registers itself, moves them
// between the two halves of the register file inside the loop (456 moves per 128 MFMAs).  AGPR: the accumulators lie in the
// accumulator half (TB = 8 and 6); the smaller forms keep them in the vector half, where the epilogue reads them in place.
// WAIT: the last of a chunk with 192 accumulators.  The compiler does not know these instructions for MFMAs; where two paths join it
// copied such an accumulator (it has registers to copy into) right behind its MFMA, before the result was there.  The other forms have been built
// without such a copy; a host test (test_nothing_touches_a_product_before_it_is_there) looks for one in every build.
template <bool AGPR, bool WAIT>
__device__ __forceinline__ void mfma_acc(f32x4& c, const bf16x8& a, const bf16x8& b) {
  if constexpr (AGPR && WAIT) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\ts_nop 13" : "+a"(c) : "v"(a), "v"(b));
  else if constexpr (AGPR) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}

// A 16-token block's accumulators in vector registers.  From the accumulator half by instructions that stay where they are
// written: the compiler would move all blocks first and spill.
template <bool AGPR>
__device__ __forceinline__ float acc_value(float a) {
  if constexpr (!AGPR) return a;
  float v;
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(a));
  return v;
}
template <bool AGPR>
__device__ __forceinline__ void acc_block(float (&x)[32], const f32x4 (&a)[8]) {
  static_for<8>([&](auto fc) {
    constexpr int fb = decltype(fc)::value;
    const f32x4 q = a[fb];
    x[4 * fb] = acc_value<AGPR>(q[0]), x[4 * fb + 1] = acc_value<AGPR>(q[1]);
    x[4 * fb + 2] = acc_value<AGPR>(q[2]), x[4 * fb + 3] = acc_value<AGPR>(q[3]);
  });
}

// Main loop: acc[t][fb] = the wave's 16-token block t x 16-feature block fb.  SWAP: tokens down the registers (V images).
template <int TB, int R, bool SWAP>
__device__ __forceinline__ void gemm_loop(const GemmParams& p, const GemmTarget& tg, int m_tile, int n_tile_in_target, bool head_live,
                                          char* lds_raw, f32x4 (&acc)[TB][8]) {
  constexpr int kStage = (kGemmWPieces + 2 * TB) * 1024;
  constexpr int kXPieces = TB / 2;                   // activation pieces of a chunk each wave copies (and 4 weight pieces)
  constexpr int PP = 4 + kXPieces;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fh = wave & 1, th = wave >> 1;
  const int nk1 = p.nk1, nk = __builtin_amdgcn_readfirstlane(p.nk1 + tg.nk2);

  // sources of this wave's pieces of the next chunk to copy: running pointers inside the current K segment, per-lane
  // offsets of the pieces behind them (consecutive 16-row blocks)
  const char* w_next = tg.w_img + (int64_t)(n_tile_in_target * kGemmWPieces + wave * 4) * tg.w_blk_stride;
  // (a tile of 192 tokens may reach past the blocks the images are padded to: those past the last token's are read as that one)
  const int x_blk = m_tile * 2 * TB + wave * kXPieces, x_last = (p.M - 1) / 16;
  auto x_at = [&](int i) { return TB == 6 ? min(x_blk + i, x_last) : x_blk + i; };
  const char* x_next = p.a_img + (int64_t)x_at(0) * p.a_blk_stride;
  unsigned w_off[4], x_off[kXPieces];
#pragma unroll
  for (int i = 0; i < 4; ++i) w_off[i] = lane * 16 + i * (unsigned)tg.w_blk_stride;
#pragma unroll
  for (int i = 0; i < kXPieces; ++i) x_off[i] = lane * 16 + (x_at(i) - x_at(0)) * (unsigned)p.a_blk_stride;
  int left = nk1;                                    // chunks not yet copied of the segment the pointers walk
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char*)lds_raw;
  unsigned long long lanes = ~0ull;                  // all lanes while chunks are left, then none
  int total_left = nk;
  // this wave's piece I of the next chunk, into ring slot `slot`; the last piece moves on to the chunk after it
  auto piece_to = [&](auto ic, int slot) {
    constexpr int i = decltype(ic)::value;
    dma_to(lds0 + slot * kStage + (i < 4 ? wave * 4 + i : kGemmWPieces + wave * kXPieces + i - 4) * 1024);
  };
  auto piece_from = [&](auto ic) {
    constexpr int i = decltype(ic)::value;
    if constexpr (i < 4) dma_from(w_next, w_off[i], lanes);
    else dma_from(x_next, x_off[i - 4], lanes);
    if constexpr (i == PP - 1) {
      w_next += 1024;
      x_next += 1024;
      --total_left;
      asm volatile("s_cmp_gt_i32 %1, 0\n\ts_cselect_b64 %0, -1, 0" : "=s"(lanes) : "s"(total_left) : "scc");
      if (--left == 0) {                             // on to the second segment (past the end: not read any more)
        w_next = tg.w2_img + (int64_t)(n_tile_in_target * kGemmWPieces + wave * 4) * tg.w2_blk_stride;
        x_next = tg.a2_img + (int64_t)x_at(0) * tg.a2_blk_stride;
#pragma unroll
        for (int j = 0; j < 4; ++j) w_off[j] = lane * 16 + j * (unsigned)tg.w2_blk_stride;
#pragma unroll
        for (int j = 0; j < kXPieces; ++j) x_off[j] = lane * 16 + (x_at(j) - x_at(0)) * (unsigned)tg.a2_blk_stride;
      }
    }
  };
  auto copy_chunk = [&](int slot) {
    static_for<PP>([&](auto ic) {
      piece_to(ic, slot);
      asm volatile("s_nop 0");
      piece_from(ic);
    });
  };

  // the bias is what the sums start from (launches with a bias have out_scale 1)
  static_for<8>([&](auto fc) {
    constexpr int fb = decltype(fc)::value;
    f32x4 start = {0.f, 0.f, 0.f, 0.f};
    if (tg.bias && head_live) {
      const float* bias = tg.bias + (n_tile_in_target * 2 + fh) * 128;
      const int g = lane >> 4, c = lane & 15;
      if constexpr (SWAP) {
        const float b = bias[16 * fb + c];
        start = f32x4{b, b, b, b};
      } else {
        start = *(const f32x4*)(bias + 32 * (fb >> 1) + 8 * g + 4 * (fb & 1));
      }
    }
    static_for<TB>([&](auto tc) { acc[decltype(tc)::value][fb] = start; });
  });

  bf16x8 wa[8], wb[8], xa[TB], xb[TB];               // operand images of this and of the next chunk, in turn
  const char* w_lds = lds_raw + lane * 16 + fh * 8 * 1024;
  const char* x_lds = lds_raw + lane * 16 + (kGemmWPieces + th * TB) * 1024;
  constexpr int kReads = 8 + TB;
  // (a plain load: it stays between the MFMAs it is written between, whose statements the compiler takes for accesses to memory)
  auto read_image = [&](auto ic, const char* w_at, const char* x_at, bf16x8 (&w)[8], bf16x8 (&x)[TB]) {
    constexpr int i = decltype(ic)::value;
    if constexpr (i < TB) x[i] = *(const bf16x8*)(x_at + i * 1024);
    else w[i - TB] = *(const bf16x8*)(w_at + (i - TB) * 1024);
  };
  // One chunk: the MFMAs on w, x with, between them, the reads of the next chunk's images (w2, x2) and the copies of the
  // chunk R ahead, which goes into the slot this chunk came from (its images are in every wave's registers).  A wave is
  // alone on its SIMD, so the pipe idles whenever something else takes longer to issue than the 12 cycles an MFMA leaves
  // free: at most one such instruction follows an MFMA.  15,342 tokens x 9,216 features, K 3,072: everything at the head
  // of the chunk 1.18 PFLOP/s, three or four at the head of each feature block 1.40, one at a time 1.51.
  auto chunk = [&](int read_slot, int dma_slot, bf16x8 (&w)[8], bf16x8 (&x)[TB], bf16x8 (&w2)[8], bf16x8 (&x2)[TB]) {
    const char *w_at = w_lds + read_slot * kStage, *x_at = x_lds + read_slot * kStage;
    constexpr int kEvery = TB > 4 ? TB : 4;          // MFMAs from copy to copy
    // this wave's pieces of the next chunk have landed, and so have the images it read for this one
    // (the builtin, which the compiler counts the images' arrival by: it then adds no waits of its own)
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm((R - 2) * PP, 0));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    static_for<8 * TB>([&](auto kc) {
      // (token blocks back and forth: from one MFMA to the next only one operand changes)
      constexpr int k = decltype(kc)::value, fb = k / TB, t = fb & 1 ? TB - 1 - k % TB : k % TB;
      if constexpr (SWAP) mfma_acc<(TB > 4), TB == 6 && k == 8 * TB - 1>(acc[t][fb], x[t], w[fb]);
      else mfma_acc<(TB > 4), TB == 6 && k == 8 * TB - 1>(acc[t][fb], w[fb], x[t]);
      if constexpr (TB > 2) {
        // reads after MFMAs 0, 2, 4 ..; a copy's target after 1 + i*kEvery, the copy itself two later
        static_assert(2 * kReads <= 8 * TB && kEvery * (PP - 1) + 3 < 8 * TB, "all of them fit between the MFMAs");
        if constexpr (k % 2 == 0 && k / 2 < kReads) read_image(std::integral_constant<int, k / 2>{}, w_at, x_at, w2, x2);
        if constexpr (k % kEvery == 1 && k / kEvery < PP) piece_to(std::integral_constant<int, k / kEvery>{}, dma_slot);
        if constexpr (k % kEvery == 3 && k / kEvery < PP) piece_from(std::integral_constant<int, k / kEvery>{});
      } else {
        static_assert(kReads + PP <= 16, "all of them fit between the MFMAs");
        if constexpr (k < kReads) {
          read_image(std::integral_constant<int, k>{}, w_at, x_at, w2, x2);
        } else if constexpr (k - kReads < PP) {
          piece_to(std::integral_constant<int, k - kReads>{}, dma_slot);
          piece_from(std::integral_constant<int, k - kReads>{});
        }
      }
    });
  };
  auto next = [](int slot) { return slot == R - 1 ? 0 : slot + 1; };

  // Ring: entering chunk kc, its images are in this wave's registers and chunks kc+1 .. kc+R-1 are on their way to LDS.
  // The barrier at its top makes chunk kc+1 visible (each wave has waited for its own pieces) and tells that every wave
  // holds chunk kc in registers, so its slot can be refilled.
#pragma unroll
  for (int i = 0; i < R; ++i) copy_chunk(i);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((R - 1) * PP) : "memory");
  __syncthreads();
  int slot = 0, kc = 0;
  if (!head_live) {
    // a head past the end of the target: this wave only copies and synchronises
    for (; kc < nk; ++kc) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((R - 2) * PP) : "memory");
      __builtin_amdgcn_s_barrier();
      copy_chunk(slot);
      slot = next(slot);
    }
    return;
  }
  static_for<kReads>([&](auto ic) { read_image(ic, w_lds, x_lds, wa, xa); });
  for (; kc + 2 <= nk; kc += 2) {
    const int s1 = next(slot), s2 = next(s1);
    chunk(s1, slot, wa, xa, wb, xb);
    chunk(s2, s1, wb, xb, wa, xa);
    slot = s2;
  }
  if (kc < nk) chunk(next(slot), slot, wa, xa, wb, xb);
  // the compiler does not know the instructions above for MFMAs: let the last one retire before anything reads the accumulators
  static_for<TB>([&](auto tc) {
    f32x4(&a)[8] = acc[decltype(tc)::value];
    if constexpr (TB > 4)
      asm volatile("s_nop 15\n\ts_nop 15"
                   : "+a"(a[0]), "+a"(a[1]), "+a"(a[2]), "+a"(a[3]), "+a"(a[4]), "+a"(a[5]),
                     "+a"(a[6]), "+a"(a[7])::"memory");
    else
      asm volatile("s_nop 15\n\ts_nop 15"
                   : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]),
                     "+v"(a[6]), "+v"(a[7])::"memory");
  });
}

// Lane (g, c) = feature 16*fb + c of the head, registers = tokens 4*g + i of a 16-token block: the V image (half, db = fb)
// wants, in that same lane, the tokens 16*(j/4) + 4*g + j%4 of its 32: blocks 2*half and 2*half + 1.
template <int TB>
__device__ __forceinline__ void epilogue_v(const GemmParams& p, const GemmTarget& tg, int head, int tok0, const f32x4 (&acc)[TB][8]) {
  const int lane = threadIdx.x & 63, g = lane >> 4;
  static_for<TB / 2>([&](auto tc) {
    constexpr int t2 = decltype(tc)::value;
    const int tok = tok0 + 32 * t2;
    if ((tok & ~63) >= p.M) return;                  // a tile past the last token has no record
    char* rec = tg.out + (int64_t)head * tg.out_head_stride + (int64_t)(tok >> 6) * tg.out_blk_stride + ((tok >> 5) & 1) * 8192;
    float x[2][32];
    acc_block<(TB > 4)>(x[0], acc[2 * t2]);
    acc_block<(TB > 4)>(x[1], acc[2 * t2 + 1]);
    bool live[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) live[j] = tok + v_image_key(g, j) < p.M;
#pragma unroll
    for (int fb = 0; fb < 8; ++fb) {
      bf16x8 img;
#pragma unroll
      for (int j = 0; j < 8; ++j) img[j] = live[j] ? (__bf16)x[j >> 2][4 * fb + (j & 3)] : (__bf16)0.0f;
      *(bf16x8*)(rec + (fb * 64 + lane) * 16) = img;
    }
  });
}

// In the other orientation lane (g, c) = token 16*t + c; its accumulators (t, fb) are elements 32*ks + 8*g + j of the head
// row with fb = 2*ks + j/4, i = j%4 (the weight-row permutation, see pack_rows_kernel), so acc_block() leaves piece ks of
// the row in x[8*ks .. 8*ks + 7].

// K tiles of the attention kernel: norm, rotation, largest row norm, (fp8) one scale per 64-token tile.  With fp8 the rows
// are formed twice, before and after the tile's scale is known: they do not fit the registers beside the accumulators.
template <int TB, int ROPE>
__device__ __forceinline__ void epilogue_k(const GemmParams& p, const GemmTarget& tg, int head, bool head_live, int tok0, char* lds,
                                           const f32x4 (&acc)[TB][8]) {
  // parts of the wave's tokens: whole 64-token tiles, or (TB == 2 and 6) the 32-token halves of tiles it may share with another wave
  constexpr int kTBlk = TB % 4 ? 2 : 4;              // 16-token blocks of a part
  constexpr int kParts = TB / kTBlk;
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int wave = threadIdx.x >> 6;
  const bool full = tok0 + 16 * TB <= p.M;           // (wave-uniform) no row of this wave lies past the end
  NormLanes norm;
  // Tables of the next blocks to form, asked for one or two blocks ahead (what the registers allow): one after the other,
  // every block would wait for a trip to memory.  They are asked for as they lie in memory and turned around in 4 KiB of the ring (`lds`, the wave's
  // own): in the lane order of the images each load took the CU's vector-memory path four times as long, 6 us of a workgroup of 192 tokens, on
  // which a launch of one tile a CU waits.  With the norm weights in two registers, block of 1,085 tokens 158.8 -> 156.4 us, of
  // 15,342 (one card) 0.9 % less, of 3,197 376 -> 365 together with the modulation's 6.
  constexpr int kAhead = TB <= 4 ? 1 : 2;
  struct { Rows16 cos, sin; } rope[kAhead];
  auto fetch_rope = [&](int t, auto& r) {
    if constexpr (ROPE != 0) {
      ask_rows16(r.cos, (const char*)tg.cos_t, kD / 2 * sizeof(float), tok0 + 16 * t, p.M - 1, lane);
      ask_rows16(r.sin, (const char*)tg.sin_t, kD / 2 * sizeof(float), tok0 + 16 * t, p.M - 1, lane);
    }
  };
  auto form_row = [&](float (&x)[32], auto tc, int t_next) {   // t_next: block kAhead later in the order they are formed in
    constexpr int t = decltype(tc)::value;
    acc_block<(TB > 4)>(x, acc[t]);
    if (!full) {
      const bool valid = tok0 + 16 * t + c < p.M;
#pragma unroll
      for (int i = 0; i < 32; ++i) x[i] = valid ? x[i] : 0.f;   // zero through norm and rotation as well
    }
    if (tg.norm_w) norm_lanes(x, tg.norm_eps, norm);
    if constexpr (TB <= 4) __builtin_amdgcn_sched_barrier(0);
    RopeQuarter now;
    if constexpr (ROPE != 0) {
      turn_table(rope[t % kAhead].cos, now.c, ROPE, lds, lane);
      turn_table(rope[t % kAhead].sin, now.s, ROPE, lds, lane);
    }
    if constexpr (TB <= 4) __builtin_amdgcn_sched_barrier(0);   // (the registers)
    rope_row(x, ROPE, now);
    if constexpr (TB <= 4) __builtin_amdgcn_sched_barrier(0);
    fetch_rope(t_next, rope[t % kAhead]);
  };
  load_norm_lanes(norm, tg.norm_w, lane);
#pragma unroll
  for (int i = 0; i < kAhead; ++i) fetch_rope(i, rope[i]);
  float amax[kParts];
  auto part_live = [&](int part) { return head_live && ((tok0 + 16 * kTBlk * part) & ~63) < p.M; };   // (wave-uniform) a tile past the last token has no record
  auto record = [&](int part) { return tg.out + (int64_t)head * tg.out_head_stride + (int64_t)((tok0 + 16 * kTBlk * part) >> 6) * tg.out_blk_stride; };
  int n_live = 0;                                    // 16-token blocks of the parts that are formed, which come first
#pragma unroll
  for (int i = 0; i < kParts; ++i) n_live += part_live(i) ? kTBlk : 0;
  static_for<kParts>([&](auto hc) {
    constexpr int part = decltype(hc)::value;
    const int first = tok0 + 16 * kTBlk * part;
    amax[part] = 0.f;
    if (!part_live(part)) return;
    char* rec = record(part);
    float nmax = 0.f;
    static_for<kTBlk>([&](auto tc) {
      constexpr int t = part * kTBlk + decltype(tc)::value;
      float x[32];
      // with fp8 the blocks of the parts that are formed come a second time
      form_row(x, std::integral_constant<int, t>{}, t + kAhead < n_live || !tg.fp8 ? min(t + kAhead, TB - 1) : t + kAhead - n_live);
      float ssq[4] = {0.f, 0.f, 0.f, 0.f};           // four running sums: one would be a chain of dependent instructions
      if (!tg.fp8) {
        // K tile image (half, ks, kb2) of 16-token block tb = 2*half + kb2: this lane's piece ks at its own place
        const int tb = ((first & 63) >> 4) + decltype(tc)::value;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          bf16x8 v;
#pragma unroll
          for (int j = 0; j < 8; ++j) v[j] = (__bf16)x[ks * 8 + j];
          // the row norm of the rounded values, two at a time
#pragma unroll
          for (int j = 0; j < 8; j += 2) ssq[j / 2] = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{v[j], v[j + 1]}, bf16x2{v[j], v[j + 1]}, ssq[j / 2], false);
          *(bf16x8*)(rec + ((((tb >> 1) * 4 + ks) * 2 + (tb & 1)) * 64 + lane) * 16) = v;
        }
      } else {
#pragma unroll
        for (int i = 0; i < 32; ++i) ssq[i & 3] += x[i] * x[i];
#pragma unroll
        for (int i = 0; i < 32; ++i) amax[part] = fmaxf(amax[part], fabsf(x[i]));
        asm volatile("" : "+v"(amax[part]));   // here, not where it is used: the rows of all blocks would have to live until then
      }
      nmax = fmaxf(nmax, wave_sum_groups((ssq[0] + ssq[1]) + (ssq[2] + ssq[3])));
    });
    nmax = sqrtf(wave_max(nmax));
    float* norms = tg.norm_out + (int64_t)head * tg.norm_stride + kNormFirst + (first >> 5);
    if (lane < kTBlk / 2) norms[lane] = nmax;        // the places of the part's 32-token halves
    if (first == 0 && lane == 0) norms[-kNormFirst] = -1.0f;
  });
  if (!tg.fp8) return;
#pragma unroll
  for (int i = 0; i < kParts; ++i) amax[i] = wave_max(amax[i]);
  if constexpr (kTBlk == 2) {
    // the scale of a tile is that of the larger magnitude of its halves, this wave's next one or the other wave's of this head
    __shared__ float half_amax[kGemmWaves][kParts];
    if (lane < kParts) {
      float mine = amax[0];
#pragma unroll
      for (int i = 1; i < kParts; ++i) mine = lane == i ? amax[i] : mine;
      half_amax[wave][lane] = mine;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kParts; ++i) {
      const int half = (wave >> 1) * kParts + i, other = half ^ 1;   // halves of the workgroup's tokens, a whole number of tiles
      amax[i] = fmaxf(amax[i], half_amax[(wave & 1) + 2 * (other / kParts)][other % kParts]);
    }
  }
  static_for<kParts>([&](auto hc) {
    constexpr int part = decltype(hc)::value;
    const int first = tok0 + 16 * kTBlk * part;
    if (!part_live(part)) return;
    char* rec = record(part);
    const float scale = fp8_block_scale(amax[part], tg.fp8_pow2 != 0);
    const float inv = 1.0f / scale;
    if (lane == 0 && (first & 63) == 0) tg.scale_out[(int64_t)head * tg.scale_head_stride + (first >> 6)] = scale;
    // fp8 K tile: key block tb is 2 KiB, chunk c2 of a lane holds its pieces ks = 2*c2 and 2*c2 + 1
    static_for<kTBlk>([&](auto tc) {
      constexpr int t = part * kTBlk + decltype(tc)::value;
      const int tb = ((first & 63) >> 4) + decltype(tc)::value;
      float x[32];
      form_row(x, std::integral_constant<int, t>{}, min(t + kAhead, TB - 1));
#pragma unroll
      for (int c2 = 0; c2 < 2; ++c2) {
        const i32x2 q0 = quant_fp8_piece(x + 16 * c2, inv), q1 = quant_fp8_piece(x + 16 * c2 + 8, inv);
        *(i32x4*)(rec + ((tb * 2 + c2) * 64 + lane) * 16) = i32x4{q0[0], q0[1], q1[0], q1[1]};
      }
    });
  });
}

// operand images of these GEMMs: [16-token block][k-step], this lane's piece ks at its own place in image ks; the tile's blocks past
// the last token are zeros, where the buffer has them
template <int TB>
__device__ __forceinline__ void epilogue_a(const GemmParams& p, const GemmTarget& tg, int head, int tok0, const f32x4 (&acc)[TB][8]) {
  const int lane = threadIdx.x & 63, c = lane & 15;
  static_for<TB>([&](auto tc) {
    constexpr int t = decltype(tc)::value;
    const int blk = tok0 + 16 * t;
    if (TB == 6 && !in_image_buffer(blk, p.M)) return;   // (wave-uniform)
    float x[32];
    acc_block<(TB > 4)>(x, acc[t]);
    const bool valid = blk + c < p.M;                  // rows past the end are zeros, whatever their activations held
    char* rec = tg.out + (int64_t)head * tg.out_head_stride + (int64_t)(blk >> 4) * tg.out_blk_stride;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      bf16x8 v;
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = valid ? (__bf16)(x[ks * 8 + j] * tg.out_scale) : (__bf16)0.0f;
      *(bf16x8*)(rec + (ks * 64 + lane) * 16) = v;
    }
  });
}

// row-major bf16 rows: y = residual + gate[row_index] * acc (the bias is in it); 16-byte pieces per lane.  The table rows
// of all blocks are asked for first and the gate and residual pieces one or two blocks ahead (what the registers allow):
// one after the other, each block would wait for two trips to memory.
template <int TB, bool GATE, bool RES>
__device__ __forceinline__ void epilogue_rows(const GemmParams& p, const GemmTarget& tg, int head, int tok0, const f32x4 (&acc)[TB][8]) {
  constexpr int kAhead = TB == 4 ? 1 : 2;
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int last = p.M - 1;                          // rows past the end read the last one and write nothing
  int rows[(TB + 3) / 4];                            // table rows of the wave's tokens, 64 to a register
  if constexpr (GATE) {
#pragma unroll
    for (int i = 0; i < (TB + 3) / 4; ++i) rows[i] = tg.row_index ? tg.row_index[min(tok0 + 64 * i + lane, last)] : 0;
  }
  struct Pieces { bf16x8 gate[4], res[4]; } even, odd;
  auto fetch = [&](int t, Pieces& f) {
    if constexpr (RES) {
      const __bf16* res = (const __bf16*)tg.residual + (int64_t)min(tok0 + 16 * t + c, last) * tg.res_row_stride + head * 128 + 8 * g;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) f.res[ks] = *(const bf16x8*)(res + 32 * ks);
    }
    if constexpr (GATE) {
      const int row = __shfl(rows[t / 4], 16 * (t & 3) + c, 64);
      const __bf16* gate = (const __bf16*)tg.gate + (int64_t)row * tg.gate_row_stride + head * 128 + 8 * g;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) f.gate[ks] = *(const bf16x8*)(gate + 32 * ks);
    }
  };
  auto block = [&](auto tc, Pieces& f) {
    constexpr int t = decltype(tc)::value;
    float x[32];
    acc_block<(TB > 4)>(x, acc[t]);
    const int token = tok0 + 16 * t + c;
    bf16x8 o[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float v = x[ks * 8 + j];
        if constexpr (GATE) v *= (float)f.gate[ks][j];
        if constexpr (RES) v += (float)f.res[ks][j];
        o[ks][j] = (__bf16)v;
      }
    if (t + kAhead < TB) fetch(t + kAhead, f);
    __bf16* orow = (__bf16*)tg.out + (int64_t)token * tg.out_row_stride + (int64_t)head * tg.out_head_elems + 8 * g;
    if (token < p.M) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) *(bf16x8*)(orow + 32 * ks) = o[ks];
    }
  };
  fetch(0, even);
  if constexpr (kAhead == 2) fetch(1, odd);
  static_for<TB>([&](auto tc) { block(tc, kAhead == 2 && (decltype(tc)::value & 1) ? odd : even); });
}

template <int TB, int R>
__global__ __launch_bounds__(64 * kGemmWaves, TB > 4 ? 1 : 2) void gemm_kernel(GemmParams p) {
  __shared__ __attribute__((aligned(1024))) char lds_raw[R * (kGemmWPieces + 2 * TB) * 1024];
  // Workgroups go to the 8 XCDs round-robin; each XCD takes one contiguous run of the tile order below, in which 32
  // consecutive tiles (the workgroups the 32 CUs behind one L2 run together) form a block of 4 token tiles x 8
  // feature tiles: every activation panel is then shared by 8 and every weight panel by 4 of them.
  constexpr int kBlockN = 8;
  const int total = p.m_tiles * p.n_tiles;
  const int per_xcd = (total + 7) / 8;
  int lin = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (p.queue_next) {
    // tiles from per-XCD work queues (see fetch_unit): the launch holds spare workgroups, and an XCD that is through
    // with its run early takes tiles off the slower ones
    __shared__ int fetched_tile;
    if (threadIdx.x == 0) fetched_tile = fetch_unit<kGemmQueueStride>(p.queue_next, blockIdx.x & (kQueues - 1), total);
    __syncthreads();
    lin = __builtin_amdgcn_readfirstlane(fetched_tile);
    if (lin < 0) return;
  }
  if (lin >= total) return;
  const int full = p.n_tiles / kBlockN * kBlockN;       // feature tiles in whole column blocks
  int m_tile, n_tile;
  if (lin < full * p.m_tiles) {
    const int nb = lin / (kBlockN * p.m_tiles), rem = lin % (kBlockN * p.m_tiles);
    m_tile = rem / kBlockN;
    n_tile = nb * kBlockN + rem % kBlockN;
  } else {
    const int rest = lin - full * p.m_tiles, width = p.n_tiles - full;
    m_tile = rest / width;
    n_tile = full + rest % width;
  }
  int t = 0;
  while (t + 1 < p.n_targets && n_tile >= p.tg[t].n_tiles) { n_tile -= p.tg[t].n_tiles; ++t; }
  const GemmTarget& tg = p.tg[t];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int head = n_tile * 2 + (wave & 1);             // 128-feature head inside the target
  const bool head_live = head * 128 < tg.n;
  const int tok0 = (m_tile * 2 + (wave >> 1)) * (16 * TB);   // first of the wave's tokens
  f32x4 acc[TB][8];
  if (tg.epi == kEpiVImg) {
    gemm_loop<TB, R, true>(p, tg, m_tile, n_tile, head_live, lds_raw, acc);
    // by the 64-token record, not by the wave's own tokens: with TB == 2 a wave holds half a record, and a half without tokens
    // is written as zeros (kernels that walk whole 64-key tiles multiply it by probabilities of 0)
    if (head_live && (tok0 & ~63) < p.M) epilogue_v<TB>(p, tg, head, tok0, acc);
    return;
  }
  gemm_loop<TB, R, false>(p, tg, m_tile, n_tile, head_live, lds_raw, acc);
  if (tg.epi == kEpiKImg) {
    __syncthreads();                                    // every wave has its images: the ring becomes space to turn tables around in
    char* lds = lds_raw + wave * 4096;
    if (tg.rope_mode == 1) epilogue_k<TB, 1>(p, tg, head, head_live, tok0, lds, acc);
    else if (tg.rope_mode == 2) epilogue_k<TB, 2>(p, tg, head, head_live, tok0, lds, acc);
    else epilogue_k<TB, 0>(p, tg, head, head_live, tok0, lds, acc);
    return;
  }
  if (!head_live || tok0 >= p.M) return;
  if (tg.epi == kEpiAImg) epilogue_a<TB>(p, tg, head, tok0, acc);
  else if (tg.gate && tg.residual) epilogue_rows<TB, true, true>(p, tg, head, tok0, acc);
  else if (tg.gate) epilogue_rows<TB, true, false>(p, tg, head, tok0, acc);
  else if (tg.residual) epilogue_rows<TB, false, true>(p, tg, head, tok0, acc);
  else epilogue_rows<TB, false, false>(p, tg, head, tok0, acc);
}

// The down-projections (x A^T: 128 features per adapter) of few tokens.  gemm_kernel gives them a workgroup per 64 tokens x 256
// features, which walks all of K while most CUs have none (1,085 tokens: 17 or 34 workgroups).  Here a workgroup is
// 32 tokens x 64 features and its eight waves share K out: no two of them read the same images, so the images go from the L2
// straight into the registers of the MFMAs, four chunks ahead, without LDS or barrier; the partial sums meet in LDS, in the
// order of the shares.  Bound by the CU's 64 bytes per clock of vector loads (6 KiB per 8 MFMAs), which is why the rule in
// launch_gemm leaves larger calls to the form that shares its copies.
// A block's two launches of them together (K 3,072; whole block before and after): 500 tokens 149 -> 116 us, 1,085 198 -> 164,
// 2,340 324 -> 307, 4,000 552 -> 530.
constexpr int kThinWaves = 8, kThinTokens = 32, kThinFeatures = 64;

__global__ __launch_bounds__(64 * kThinWaves, 2) void gemm_thin_kernel(GemmParams p, int n_tiles) {
  constexpr int kGroup = 4;                              // chunks asked for together
  __shared__ __attribute__((aligned(16))) char part[kThinWaves * 8 * 1024];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int total = (p.M + kThinTokens - 1) / kThinTokens * n_tiles;
  const int per_xcd = (total + 7) / 8;                   // a contiguous run of token tiles per XCD
  const int lin = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_xcd || lin >= total) return;
  const int m_tile = lin / n_tiles;
  int n_tile = lin % n_tiles, t = 0;
  while (t + 1 < p.n_targets && n_tile >= p.tg[t].n / kThinFeatures) n_tile -= p.tg[t].n / kThinFeatures, ++t;
  const GemmTarget& tg = p.tg[t];
  const char* x0 = p.a_img + (int64_t)(m_tile * 2) * p.a_blk_stride;
  const char* w0 = tg.w_img + (int64_t)(n_tile * 4) * tg.w_blk_stride;
  const int k0 = wave * p.nk1 / kThinWaves, k1 = (wave + 1) * p.nk1 / kThinWaves;
  struct Images { bf16x8 x[kGroup][2], w[kGroup][4]; };
  auto fetch = [&](Images& im, int kc) {                 // chunks past the share: its last one again, not used
#pragma unroll
    for (int u = 0; u < kGroup; ++u) {
      const int64_t at = (int64_t)min(kc + u, k1 - 1) * 1024 + lane * 16;
#pragma unroll
      for (int i = 0; i < 2; ++i) im.x[u][i] = *(const bf16x8*)(x0 + i * p.a_blk_stride + at);
#pragma unroll
      for (int i = 0; i < 4; ++i) im.w[u][i] = *(const bf16x8*)(w0 + i * tg.w_blk_stride + at);
    }
  };
  f32x4 acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int fb = 0; fb < 4; ++fb) acc[i][fb] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto use = [&](const Images& im, int kc) {
#pragma unroll
    for (int u = 0; u < kGroup; ++u) {
      if (kc + u >= k1) break;
#pragma unroll
      for (int fb = 0; fb < 4; ++fb)
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[i][fb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(im.w[u][fb], im.x[u][i], acc[i][fb], 0, 0, 0);
    }
  };
  if (k0 < k1) {
    Images a, b;
    fetch(a, k0);
#pragma unroll 1
    for (int kc = k0; kc < k1; kc += 2 * kGroup) {
      fetch(b, kc + kGroup);
      __builtin_amdgcn_sched_barrier(0);
      use(a, kc);
      __builtin_amdgcn_sched_barrier(0);
      if (kc + kGroup < k1) {
        fetch(a, kc + 2 * kGroup);
        __builtin_amdgcn_sched_barrier(0);
        use(b, kc + kGroup);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int fb = 0; fb < 4; ++fb) *(f32x4*)(part + wave * 8192 + ((i * 4 + fb) * 64 + lane) * 16) = acc[i][fb];
  __syncthreads();
  // wave (i, fb) adds up token block i, feature block fb: lane (g, c) = token c, elements 32*ks + 8*g + 4*(fb%2) .. +3 of the
  // head, ks = fb/2 of its 64-feature half: half of this lane's piece of image ks (see epilogue_a)
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < kThinWaves; ++j) sum += *(const f32x4*)(part + j * 8192 + (wave * 64 + lane) * 16);
  const int i = wave >> 2, fb = (n_tile & 1) * 4 + (wave & 3), blk = m_tile * 2 + i;
  const bool valid = blk * 16 + (lane & 15) < p.M;       // rows past the end are zeros, whatever their activations held
  bf16x4 o;
#pragma unroll
  for (int r = 0; r < 4; ++r) o[r] = valid ? (__bf16)(sum[r] * tg.out_scale) : (__bf16)0.0f;
  char* rec = tg.out + (int64_t)(n_tile >> 1) * tg.out_head_stride + (int64_t)blk * tg.out_blk_stride;
  *(bf16x4*)(rec + ((fb >> 1) * 64 + lane) * 16 + 8 * (fb & 1)) = o;
}

template <int TB, int R = kGemmRing>
static hipError_t launch_gemm_tb(GemmParams p, int cus, hipStream_t st) {
  p.m_tiles = (p.M + 32 * TB - 1) / (32 * TB);
  const int total = p.m_tiles * p.n_tiles;
  // launches of at least two rounds of workgroups take their tiles from per-XCD work queues, with an eighth more
  // workgroups than tiles, the spare ones for the XCDs that finish early
  if (total < 2 * cus * (TB > 4 ? 1 : 2)) p.queue_next = nullptr;
  if (p.queue_next) {
    hipError_t e = launch_fill_zero((unsigned*)p.queue_next, kQueueSlots, st);
    if (e != hipSuccess) return e;
  }
  const int wgs = p.queue_next ? total + (total / 8 > kQueues ? total / 8 : kQueues) : total;
  hipLaunchKernelGGL((gemm_kernel<TB, R>), dim3((wgs + 7) / 8 * 8), dim3(64 * kGemmWaves), 0, st, p);
  return hipGetLastError();
}

hipError_t launch_gemm(const GemmParams& p, hipStream_t st) {
  int cus = 0;
  hipError_t e = device_cu_count(&cus);
  if (e != hipSuccess) return e;
  if (cus <= 0) cus = 1;
  // Thin tiles for launches of down-projections only, up to three of them per CU: measured against the other form (whole block)
  // two 64-feature tiles a 32-token tile gain 15 us at 1,085 tokens, 22 at 4,000, 5 at 9,360 and nothing at 11,700; six gain 15 at
  // 1,085, nothing at 4,000 and lose 10 at 9,360.
  int thin_tiles = 0;
  for (int t = 0; t < p.n_targets; ++t) {
    const GemmTarget& tg = p.tg[t];
    if (tg.epi != kEpiAImg || tg.nk2 || tg.bias || tg.n % 128) { thin_tiles = -1; break; }
    thin_tiles += tg.n / kThinFeatures;
  }
  if (thin_tiles > 0) {
    const int64_t total = (int64_t)((p.M + kThinTokens - 1) / kThinTokens) * thin_tiles;
    if (total <= 3 * cus) {
      hipLaunchKernelGGL(gemm_thin_kernel, dim3((unsigned)(total + 7) / 8 * 8), dim3(64 * kThinWaves), 0, st, p, thin_tiles);
      return hipGetLastError();
    }
  }
  switch (gemm_token_blocks(p.M, p.n_tiles, p.nk1, cus)) {
    case 8: return launch_gemm_tb<8>(p, cus, st);
    case 6: return launch_gemm_tb<6>(p, cus, st);
    case 4: return launch_gemm_tb<4>(p, cus, st);
    default: break;
  }
  // 64 tokens with one workgroup on a CU: a chunk is done in 0.22 us, and three of them cover a copy's way where two do not.  Ring of
  // 3 / 4, K 3,072 x 3,072 features, us: 128 tokens 29.7 / 24.6, 500 31.2 / 26.0, 1,085 32.0 / 27.2 (of 5 to 7 the same); with a dozen workgroups on
  // the chip the way is short enough (64 tokens 23.0 / 23.6), and for few chunks the longer start costs as much (K 1,024 13.4 / 12.6 and
  // 11.7 / 12.0, 512 8.1 / 8.3).  From K 1,536 on 8 to 22 % in 53 of 56 calls of 32 to 216 tiles; 2 % slower: 44 tiles, K 1,536 13.8 / 14.1, and
  // 32 tiles of 256 features, K 1,536 20.5 / 20.9 and 2,048 24.0 / 24.4 (with an adapter; K 3,072 36.5 / 32.7).  The larger forms gain nothing from it.
  const int64_t tiles = (int64_t)((p.M + 63) / 64) * p.n_tiles;
  return tiles >= 24 && tiles <= cus && p.nk1 >= 48 ? launch_gemm_tb<2, 4>(p, cus, st) : launch_gemm_tb<2>(p, cus, st);
}

// ------------------------------------------------------------------------------------------------
// Rows -> operand images.
// One wave per row: lane l holds the 16-byte pieces l, l + 64, ... of the row.  Piece pc (elements 8*pc .. +7) of row r
// belongs to image (16-row block r/16, k-step pc/4), lane 16*(pc%4) + r%16: byte ((r/16)*(K/32) + pc/4)*1024 +
// (16*(pc%4) + r%16)*16.
// `head_perm`: the rows are weight rows (output features) and are stored permuted inside each 128-row head
// (see acc_block and epilogue_k): image row 16*fb + 4*g + i takes source row 32*(fb/2) + 8*g + 4*(fb%2) + i.
constexpr int kPackMaxPieces = 8;  // 16-byte pieces per lane: rows of up to 64 * 8 * 8 = 4096 elements

constexpr int kPackRows = 8;                                        // rows (waves) of a workgroup
constexpr int kPackPitch = kPackMaxPieces * 64 * 16 + 16;           // bytes between the rows staged in LDS (+16: no bank conflicts)

// the workgroup's 8 staged rows are one half of a 16-row block: piece pc of the 8 rows is 128 contiguous bytes of its image
__device__ __forceinline__ void store_images(const PackParams& p, const char* stage, int pitch) {
  const int row0 = blockIdx.x * kPackRows, pieces = p.K / 8;
  char* ob = p.out + (int64_t)(row0 >> 4) * p.out_blk_stride + (row0 & 15) * 16;
  for (int q = threadIdx.x; q < kPackRows * pieces; q += 64 * kPackRows) {
    const int rr = q & (kPackRows - 1), pc = q / kPackRows;
    const bf16x8 t = *(const bf16x8*)(stage + rr * pitch + pc * 16);
    *(bf16x8*)(ob + ((int64_t)(pc >> 2) * 64 + 16 * (pc & 3) + rr) * 16) = t;
  }
}

__global__ __launch_bounds__(64 * kPackRows) void pack_rows_kernel(PackParams p) {
  // the rows of the workgroup, as bf16 pieces, before they go out: in an image a row's pieces lie 256 bytes apart and
  // the same piece of 16 consecutive rows side by side, so whole cache lines only come from several rows together
  __shared__ __attribute__((aligned(16))) char stage[kPackRows * kPackPitch];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = blockIdx.x * kPackRows + wave;     // destination row (rows_padded is a multiple of 16: always inside)
  int src = row;
  if (p.head_perm) {
    const int in_head = row & 127, fb = in_head >> 4, g = (in_head >> 2) & 3, i = in_head & 3;
    src = (row & ~127) + 32 * (fb >> 1) + 8 * g + 4 * (fb & 1) + i;
  }
  const bool valid = src < p.rows;
  const int pieces = p.K / 8;                        // 16-byte pieces per row
#pragma unroll
  for (int c = 0; c < kPackMaxPieces; ++c) {
    const int pc = lane + 64 * c;
    if (pc >= pieces) continue;
    bf16x8 t = {};
    if (valid) t = *(const bf16x8*)((const __bf16*)p.x + (int64_t)src * p.row_stride + 8 * pc);
    *(bf16x8*)(stage + wave * kPackPitch + pc * 16) = t;
  }
  __syncthreads();
  store_images(p, stage, kPackPitch);
}

// Rows -> operand images through the AdaLN modulation of the block:
//   y = norm(x) * (1 + scale[row_index]) + shift[row_index]
// with norm = LayerNorm without affine parameters or RMSNorm without weight, statistics in fp32.  Rows, pieces and staging as
// above; NP: pieces of a lane, of which only the last may lie past the row's end (lanes there read the row's last piece and take zeros for it).
// Bound by the memory from some thousand rows on (2 bytes in and out per element: 48,360 x 3,072 at 5.5 TB/s), below by a row's chain of trips to
// memory (row, its table row's number, tables) and its two sums across the wave, with four waves a SIMD beside it.  So the tables' pieces are asked for all
// at once and before the sums.  Asked for piece by piece where they were used, behind a test each, with 1.6 times the instructions (what may
// not be there was looked after element by element) and sums through the LDS crossbar, us, before / now: K 3,072: 1,085 rows 8.0 / 6.4, 4,000
// 17.6 / 11.4, 15,342 57.0 / 36.2, 48,360 160.7 / 108.9; K 512: 128 rows 4.4 / 3.0, 15,342 23.9 / 9.4; K 4,096: 15,342 79.9 / 45.2.
template <int NORM, int NP>
__global__ __launch_bounds__(64 * kPackRows, 4) void modulate_rows_kernel(PackParams p) {
  constexpr int kPitch = NP * 1024 + 16;
  __shared__ __attribute__((aligned(16))) char stage[kPackRows * kPitch];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = blockIdx.x * kPackRows + wave;
  const int last = p.K / 8 - 1;                      // the row's last piece
  char* mine = stage + wave * kPitch;
  auto piece = [&](int c) { return c < NP - 1 ? lane + 64 * c : min(lane + 64 * c, last); };
  if (row < p.rows) {                                // (wave-uniform)
    bf16x8 x[NP], scale[NP], shift[NP];
    const __bf16* src = (const __bf16*)p.x + (int64_t)row * p.row_stride;
#pragma unroll
    for (int c = 0; c < NP; ++c) x[c] = *(const bf16x8*)(src + 8 * piece(c));
    const int64_t table = (p.row_index ? p.row_index[row] : 0) * p.table_stride;
    // (in the place of a table that is not there the row itself: no branches between these loads and the wait for those above)
    const __bf16* scale_row = p.scale ? (const __bf16*)p.scale + table : src;
    const __bf16* shift_row = p.shift ? (const __bf16*)p.shift + table : src;
#pragma unroll
    for (int c = 0; c < NP; ++c) {
      scale[c] = *(const bf16x8*)(scale_row + 8 * piece(c));
      shift[c] = *(const bf16x8*)(shift_row + 8 * piece(c));
    }
    __builtin_amdgcn_sched_barrier(0);
    // the row's values are formed anew for every pass where they do not fit the registers beside the tables
    auto anew = [&]() {
      if constexpr (NP > 6)
#pragma unroll
        for (int c = 0; c < NP; ++c) {
          i32x4 v = __builtin_bit_cast(i32x4, x[c]);
          asm volatile("" : "+v"(v));
          x[c] = __builtin_bit_cast(bf16x8, v);
        }
    };
    const bool there = lane + 64 * (NP - 1) <= last;
    // Two passes over the row held in registers: the mean first, then the sum of squared distances from it.  The
    // one-pass form E[x^2] - mean^2 cancels when a row's mean is large against its spread.
    const float inv_k = 1.0f / (float)p.K;
    float mean = 0.f;
    if constexpr (NORM == kNormLayer) {
      float sum[8] = {};
#pragma unroll
      for (int c = 0; c < NP; ++c)
#pragma unroll
        for (int j = 0; j < 8; ++j) sum[j] += c < NP - 1 || there ? (float)x[c][j] : 0.f;
      mean = wave_sum(((sum[0] + sum[1]) + (sum[2] + sum[3])) + ((sum[4] + sum[5]) + (sum[6] + sum[7]))) * inv_k;
      asm volatile("" : "+v"(mean));                 // rounded: as part of a fused x - sum / K it leaves a constant row something
    }
    anew();
    float ssq[8] = {};
#pragma unroll
    for (int c = 0; c < NP; ++c)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float d = c < NP - 1 || there ? (float)x[c][j] - mean : 0.f;
        ssq[j] = fmaf(d, d, ssq[j]);
      }
    // a constant row with eps == 0 comes out as zeros (plus shift) instead of 0 * inf
    const float ve = wave_sum(((ssq[0] + ssq[1]) + (ssq[2] + ssq[3])) + ((ssq[4] + ssq[5]) + (ssq[6] + ssq[7]))) * inv_k + p.eps;
    const float rs = ve > 0.f ? rsqrtf(ve) : 0.f;
    anew();
    if (!p.scale)
#pragma unroll
      for (int c = 0; c < NP; ++c) scale[c] = bf16x8{};
    if (!p.shift)
#pragma unroll
      for (int c = 0; c < NP; ++c) shift[c] = bf16x8{};
#pragma unroll
    for (int c = 0; c < NP; ++c) {
      bf16x8 t;
#pragma unroll
      for (int j = 0; j < 8; ++j) t[j] = (__bf16)fmaf(((float)x[c][j] - mean) * rs, 1.0f + (float)scale[c][j], (float)shift[c][j]);
      *(bf16x8*)(mine + (lane + 64 * c) * 16) = t;   // (what lies past the row's end is not read again)
    }
  } else {
#pragma unroll
    for (int c = 0; c < NP; ++c) *(bf16x8*)(mine + (lane + 64 * c) * 16) = bf16x8{};
  }
  __syncthreads();
  store_images(p, stage, kPitch);
}

template <int NORM, int NP = 1>
static void launch_modulate(const PackParams& p, hipStream_t st) {
  if constexpr (NP < kPackMaxPieces)
    if (p.K > NP * 512) return launch_modulate<NORM, NP + 1>(p, st);
  hipLaunchKernelGGL((modulate_rows_kernel<NORM, NP>), dim3(p.rows_padded / kPackRows), dim3(64 * kPackRows), 0, st, p);
}

hipError_t launch_pack_rows(const PackParams& p, hipStream_t st) {
  switch (p.norm) {
    case kNormLayer: launch_modulate<kNormLayer>(p, st); break;
    case kNormRms: launch_modulate<kNormRms>(p, st); break;
    default: hipLaunchKernelGGL(pack_rows_kernel, dim3(p.rows_padded / kPackRows), dim3(64 * kPackRows), 0, st, p); break;
  }
  return hipGetLastError();
}

// clears `n` 32-bit words (queue positions, arrival counters)
__global__ void fill_zero_kernel(unsigned* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

hipError_t launch_fill_zero(unsigned* p, int n, hipStream_t st) {
  hipLaunchKernelGGL(fill_zero_kernel, dim3((n + 255) / 256), dim3(256), 0, st, p, n);
  return hipGetLastError();
}

}  // namespace pkh3
