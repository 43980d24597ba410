// Shared device-side definitions for the gfx950 attention kernels: vector types, the operand-image
// layouts the prologue (or the projection GEMM's epilogue) writes and the attention kernel consumes,
// and small wave helpers.
//
// Operand images.  The attention kernel runs on the CDNA4 16x16 MFMA shapes (16x16x32 bf16, 16x16x128 fp8):
// at the same peak rate they move a quarter of the accumulator registers per instruction of the 32x32 shapes,
// and the part sustains about 10 % more of them per second on real data.  For those shapes lane l of a wave
// supplies row/column c = l % 16 of an operand and the 8 consecutive contraction elements selected by its group
// g = l / 16; the 16x16 fp32 result puts column c in lane l and rows 4*g + i in its 4 registers i.  K and V are
// stored in HBM already cut into 1 KiB images (64 lanes x 16 B) in exactly that order, so the attention kernel
// moves them HBM -> LDS -> VGPR as straight 16-byte copies with no shuffles and no LDS bank conflicts.
//
//   K tile (64 keys, bf16, 16 KiB): image (half, ks, kb2), half in 0..1, ks in 0..3, kb2 in 0..1, at byte
//       (((half*4 + ks)*2 + kb2)*64 + l)*16 holds K'[32*half + 16*kb2 + c][32*ks + 8*g + j], j = 0..7
//       (A operand of S^T = K' Q'^T; the 32-key halves are contiguous for the half-tile forms of the kernel)
//   Q block (32 queries, bf16, registers only): image (qb, ks) holds Q'[16*qb + c][32*ks + 8*g + j]
//       (B operand of S^T)
//   V tile (64 keys, bf16, 16 KiB): image (half, db), db in 0..7, at ((half*8 + db)*64 + l)*16 holds
//       V[32*half + 16*(j/4) + 4*g + j%4][16*db + c], j = 0..7      (A operand of O^T = V^T P^T)
//       -- the key order is the one the S^T result registers of key blocks 2*half and 2*half+1 already have,
//       so P goes from the softmax registers into the next MFMA without leaving the lane.
//   fp8 K tile (8 KiB): key block kb in 0..3 is 2 KiB, 32 B per lane as two 16-byte chunks c2 at
//       ((kb*2 + c2)*64 + l)*16; byte 8*(ks%2) + j of chunk c2 = ks/2 is element d = 32*ks + 8*g + j of row
//       16*kb + c -- the same lane-to-d assignment as the bf16 images; Q uses it alike, which is all the
//       contraction needs.
//
// Rows are prepared (RMSNorm, rotation, quantisation) in the layout of the images themselves, four lanes per row
// (norm_row and rope_row below): by the K prologue, by the K epilogue of the projection GEMM and by the attention
// kernel's Q load.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace pkh3 {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(8))) int i32x8;
typedef __attribute__((ext_vector_type(4))) int i32x4;
typedef __attribute__((ext_vector_type(2))) int i32x2;

// f(0) .. f(N - 1), the index as a constant
template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, I + 1>(f);
  }
}

constexpr int kD = 128;            // head dim (fixed)
constexpr int kTileKeys = 64;      // keys per K/V tile, also the block-sparse tile edge
constexpr int kKTileBytes = 16384; // bf16 K tile
constexpr int kK8TileBytes = 8192; // fp8 K tile
constexpr int kVTileBytes = 16384; // bf16 V tile
constexpr int kQBlkBytes = 8192;   // bf16 Q block of 32 queries
constexpr int kQ8BlkBytes = 4096;  // fp8 Q block of 32 queries
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kFp8Max = 448.0f;  // OCP e4m3fn

__device__ __forceinline__ float wave_sum_groups(float x) {
  // sum over the four lanes l % 16 == const (one per 16-lane group): two row swaps, no trip through the LDS crossbar
  const auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r16[0]) + __uint_as_float(r16[1]);
  const auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r32[0]) + __uint_as_float(r32[1]);
}

// maximum over the four lanes l % 16 == const (one per 16-lane group): two row swaps, no LDS crossbar
__device__ __forceinline__ float max_across_groups(float x) {
  const auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(r16[0]), __uint_as_float(r16[1]));
  const auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r32[0]), __uint_as_float(r32[1]));
}

// maximum over the wave, in every lane: pairs, quads and halves of the 16-lane rows by permutations that ride on the comparison,
// then across the rows (no trip through the LDS crossbar)
template <int CTRL>
__device__ __forceinline__ float max_with(float x) {
  const int v = __float_as_int(x);
  return fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false)));
}
__device__ __forceinline__ float wave_max(float x) {
  x = max_with<0xB1>(x);     // quad_perm 1 0 3 2
  x = max_with<0x4E>(x);     // quad_perm 2 3 0 1
  x = max_with<0x141>(x);    // row_half_mirror
  x = max_with<0x140>(x);    // row_mirror
  return max_across_groups(x);
}

// the sum of all lanes, the same way
template <int CTRL>
__device__ __forceinline__ float sum_with(float x) {
  const int v = __float_as_int(x);
  return x + __int_as_float(__builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float wave_sum(float x) {
  x = sum_with<0xB1>(x);
  x = sum_with<0x4E>(x);
  x = sum_with<0x141>(x);
  x = sum_with<0x140>(x);
  return wave_sum_groups(x);
}

// ---- four lanes per row: the layout of the 16x16 operand images themselves ----
// Lane (c = l % 16, g = l / 16) holds the pieces p8 = 4*ks + g of row c of a 16-row block, i.e. elements
// d = 32*ks + 8*g + j at x[8*ks + j]; the three other lane groups (lanes l ^ 16, l ^ 32, l ^ 48) hold the rest of the
// row, so the sum of squares needs two exchanges and both pairings of the rotation (interleaved (2i, 2i+1) /
// half-split (i, i+64): ks and ks + 2) stay inside the lane.  What a lane holds is exactly its 16 bytes of the four K
// images (ks = 0..3) of its 16-row block, so rows prepared this way are stored, or fed to the MFMA, without any lane
// movement.

// The rotation tables of one row as its lane group uses them (8 vectors of 4).  Interleaved: c[ks] = pairs
// 16*ks + 4*g .. +3 (elements 2jj, 2jj+1 of piece ks).  Half-split: c[2*ks], c[2*ks+1] = pairs 32*ks + 8*g .. +7
// (element j of piece ks with its partner in piece ks + 2), ks = 0, 1.
struct RopeQuarter {
  f32x4 c[4], s[4];
};

// the rotation of this lane's 32 elements of a row, with the row's tables already in registers
__device__ __forceinline__ void rope_row(float (&x)[32], int rope_mode, const RopeQuarter& r) {
  if (rope_mode == 1) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const float a0 = x[ks * 8 + 2 * jj], a1 = x[ks * 8 + 2 * jj + 1];
        x[ks * 8 + 2 * jj] = a0 * r.c[ks][jj] - a1 * r.s[ks][jj];
        x[ks * 8 + 2 * jj + 1] = a1 * r.c[ks][jj] + a0 * r.s[ks][jj];
      }
  } else if (rope_mode == 2) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float cj = r.c[2 * ks + (j >> 2)][j & 3], sj = r.s[2 * ks + (j >> 2)][j & 3];
        const float lo = x[ks * 8 + j], hi = x[(ks + 2) * 8 + j];
        x[ks * 8 + j] = lo * cj - hi * sj;
        x[(ks + 2) * 8 + j] = hi * cj + lo * sj;
      }
  }
}

// the sum of the squares of eight bf16 values on top of `sum`
__device__ __forceinline__ float add_squares(const bf16x8& v, float sum) {
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    const bf16x2 pr = {v[j], v[j + 1]};
    sum = __builtin_amdgcn_fdot2_f32_bf16(pr, pr, sum, false);
  }
  return sum;
}

// ---- rows on their way from memory to the layout above ----
// Sixteen rows of 256 bytes (a block's queries or keys of a head, or its cosines, or its sines).  Loaded in the layout above, neighbouring lanes lie
// in different rows, which keeps the CU's vector-memory path busy four times as long as whole rows do (one workgroup alone: 16
// against 60 bytes a clock).  So they are asked for as they lie in memory, lane l the 16-byte chunk l % 16 of row 4*i + l / 16, and
// turned around in 4 KiB of LDS of the wave's own, chunks XOR-swizzled by the row.  The start of a short-key workgroup with rotation took
// 30 % of its 20 us, most of it these loads: 3 x 8 heads x 777 rows (the call) 32.7 -> 31.4 us; block-sparse calls, whose workgroups begin
// anew every 70 to 350 us, 14,907 rows 658 -> 648, 4 x 24 heads x 1,000 rows with rotation 1 to 3 %.
struct Rows16 {
  i32x4 v[4];
};
// base: the first byte of row 0 of the table or head; rows past `last` are that one again
__device__ __forceinline__ void ask_rows16(Rows16& r, const char* base, int64_t row_bytes, int first, int last, int lane) {
#pragma unroll
  for (int i = 0; i < 4; ++i) r.v[i] = *(const i32x4*)(base + (int64_t)min(first + 4 * i + (lane >> 4), last) * row_bytes + (lane & 15) * 16);
}
// the rows src[i] of this lane
__device__ __forceinline__ void ask_rows16(Rows16& r, const char* base, int64_t row_bytes, const int (&src)[4], int lane) {
#pragma unroll
  for (int i = 0; i < 4; ++i) r.v[i] = *(const i32x4*)(base + (int64_t)src[i] * row_bytes + (lane & 15) * 16);
}
// chunk(j): which chunk of its row c = l % 16 the lane wants as its j-th
template <class F>
__device__ __forceinline__ void turn_rows16(const Rows16& r, i32x4 (&out)[4], char* lds, int lane, F&& chunk) {
  const int c = lane & 15;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 4 * i + (lane >> 4);
    *(i32x4*)(lds + row * 256 + ((c ^ row) * 16)) = r.v[i];
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) out[j] = *(const i32x4*)(lds + c * 256 + ((chunk(j) ^ c) * 16));
}
// a row's elements, as norm_row takes them
__device__ __forceinline__ void turn_elements(const Rows16& r, bf16x8 (&raw)[4], char* lds, int lane) {
  i32x4 out[4];
  turn_rows16(r, out, lds, lane, [&](int j) { return 4 * j + (lane >> 4); });
#pragma unroll
  for (int j = 0; j < 4; ++j) raw[j] = __builtin_bit_cast(bf16x8, out[j]);
}
// a row's cosines or sines, as RopeQuarter holds them
__device__ __forceinline__ void turn_table(const Rows16& r, f32x4 (&table)[4], int rope_mode, char* lds, int lane) {
  const int g = lane >> 4;
  i32x4 out[4];
  turn_rows16(r, out, lds, lane, [&](int j) { return rope_mode == 1 ? 4 * j + g : 8 * (j >> 1) + 2 * g + (j & 1); });
#pragma unroll
  for (int j = 0; j < 4; ++j) table[j] = __builtin_bit_cast(f32x4, out[j]);
}

// The RMSNorm weights in two registers: lane (c, g) has those of the elements 32*(c/8) + 8*g + c%8 and 64 further on, of which its row of
// 16 lanes needs all; the multiplication takes them from there.
struct NormLanes {
  float w[2];
};
__device__ __forceinline__ void load_norm_lanes(NormLanes& n, const float* norm_w, int lane) {
#pragma unroll
  for (int i = 0; i < 2; ++i) n.w[i] = norm_w ? norm_w[64 * i + 32 * ((lane & 15) >> 3) + 8 * (lane >> 4) + (lane & 7)] : 1.0f;
}
// `factor` times the value that lane N of this lane's row of 16 holds.  (`x` must not come from the two vector instructions before this one, and the
// compiler puts no wait states in front of assembly: see settle.)
template <int N>
__device__ __forceinline__ float times_row_lane(float x, float factor) {
  float y;
  asm("v_mul_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "=v"(y) : "v"(x), "v"(factor), "n"(N));
  return y;
}

// where the weights were kept elsewhere, they have been back for as long as it takes
__device__ __forceinline__ void settle(NormLanes& n) { asm volatile("s_nop 1" : "+v"(n.w[0]), "+v"(n.w[1])); }

// RMSNorm (if `normed`) and `factor` of this lane's 32 elements of a row as they are in memory: the squares are summed up two at a
// time before the elements are unpacked, and the factor (the softmax scale and log2 e of the queries) rides with the norm's.
__device__ __forceinline__ void norm_row(float (&x)[32], const bf16x8 (&raw)[4], bool normed, float eps, NormLanes n, float factor) {
  if (normed) {
    float part[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) part[ks] = add_squares(raw[ks], 0.f);
    // an all-zero row with eps == 0 stays all zero instead of 0 * inf
    const float ms = wave_sum_groups((part[0] + part[1]) + (part[2] + part[3])) * (1.0f / kD) + eps;
    factor *= ms > 0.f ? rsqrtf(ms) : 0.f;
  }
  settle(n);
  static_for<32>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    x[i] = times_row_lane<i & 15>(n.w[i >> 4], factor);
  });
#pragma unroll
  for (int i = 0; i < 32; ++i) x[i] *= (float)raw[i >> 3][i & 7];
}
// RMSNorm of this lane's 32 elements of a row
__device__ __forceinline__ void norm_lanes(float (&x)[32], float eps, NormLanes& n) {
  float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 32; ++i) part[i & 3] += x[i] * x[i];
  // an all-zero row with eps == 0 stays all zero instead of 0 * inf
  const float ms = wave_sum_groups((part[0] + part[1]) + (part[2] + part[3])) * (1.0f / kD) + eps;
  const float rs = ms > 0.f ? rsqrtf(ms) : 0.f;
  settle(n);
  static_for<32>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    x[i] *= times_row_lane<i & 15>(n.w[i >> 4], rs);
  });
}

// eight values -> eight fp8 e4m3 bytes
__device__ __forceinline__ i32x2 quant_fp8_piece(const float* x, float inv) {
  i32x2 t;
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    int v = 0;
    v = __builtin_amdgcn_cvt_pk_fp8_f32(x[4 * w] * inv, x[4 * w + 1] * inv, v, false);
    v = __builtin_amdgcn_cvt_pk_fp8_f32(x[4 * w + 2] * inv, x[4 * w + 3] * inv, v, true);
    t[w] = v;
  }
  return t;
}

// key (inside its 32-key half) that element j of lane group g carries in a V image / in the P operand
__device__ __forceinline__ int v_image_key(int g, int j) { return 16 * (j >> 2) + 4 * g + (j & 3); }

// Dequantisation scale of an fp8 block whose largest magnitude is `amax`: amax / 448, or, with `pow2`, the smallest
// power of two that is at least that (the form the scaled MFMA takes as an operand: an 8-bit exponent).  The product
// amax * fl(1/448) is rounded to float32 first and the power of two is taken of that number.  A block of zeros gets 1.
__device__ __forceinline__ float fp8_block_scale(float amax, bool pow2) {
  if (!(amax > 0.f)) return 1.0f;
  const float s = amax * (1.0f / kFp8Max);
  if (!pow2) return s;
  const unsigned bits = __float_as_uint(s);
  unsigned e = (bits >> 23) & 0xffu;
  if (bits & 0x7fffffu) ++e;
  e = e < 1u ? 1u : (e > 254u ? 254u : e);
  return __uint_as_float(e << 23);
}

// the 8-bit exponent (E8M0: value 2^(e - 127)) of a power-of-two scale, as the scaled MFMA takes it
__device__ __forceinline__ int e8m0_of(float pow2_scale) { return (int)((__float_as_uint(pow2_scale) >> 23) & 0xffu); }

constexpr int kQueues = 8;       // work queues of a launch: one per XCD

// Work queues of a launch's units.  The XCDs of one part hold different clocks under the power cap
// (a few per cent apart), and the hardware deals workgroups to them round-robin, an eighth each whatever their speed,
// so with a fixed workgroup -> unit map the call lasts as long as its slowest XCD needs for its eighth.  Instead every
// XCD has a queue (a counter) over its contiguous run of units: a workgroup takes the next unit of its own XCD's queue
// and, when that is empty, of the queue with the most units left.  Launches of a workgroup per unit hold an eighth more workgroups than
// units, so an XCD that is through early keeps getting workgroups, which take units off the slower ones; in the block-sparse form a
// workgroup per CU takes one unit after the other.  A workgroup that finds every queue empty exits.  Returns the unit (index inside the section) or -1.
// `taken`: a position of the home queue that the caller has taken ahead (take_position), or -1.
// STRIDE: ints between the queues' positions.  The accesses of all XCDs to one stretch of 32 bytes are served one after the
// other, which is the rate of a launch of short workgroups whose positions share one (see gemm_kernel).
__device__ __forceinline__ int take_position(int* next) { return __hip_atomic_fetch_add(next, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

template <int STRIDE = 1>
__device__ __forceinline__ int fetch_unit(int* queue_next, int home, int units, int taken = -1) {
  const int per = (units + kQueues - 1) / kQueues;
  int q = home;
  if (taken >= 0 && taken < min(per, units - home * per)) return home * per + taken;
  // Every pass either takes a unit, or finds all queues empty, or lost a unit to another workgroup (which is
  // progress of the launch as a whole: the positions only grow), so the loop ends.
#pragma unroll 1
  for (;;) {
    const int size = max(0, min(per, units - q * per));
    // a look first: a queue that is empty stays empty, no need to count it further up
    if (__hip_atomic_load(queue_next + q * STRIDE, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < size) {
      const int i = take_position(queue_next + q * STRIDE);
      if (i < size) return q * per + i;
    }
    int best = -1, most = 0;
    for (int j = 0; j < kQueues; ++j) {
      const int left = max(0, min(per, units - j * per)) - __hip_atomic_load(queue_next + j * STRIDE, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (left > most) most = left, best = j;
    }
    if (best < 0) return -1;
    q = best;
  }
}

}  // namespace pkh3
