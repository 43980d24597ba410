// Prologue kernels: everything that touches each Q/K/V row exactly once before the S x S work.
//   - key-mask compaction (prefix sum of the padding mask -> list of valid key rows)
//   - QK-RMSNorm + rotary embedding (+ optional fp8 e4m3 quantisation with per-64-row absmax scales),
//     written as MFMA operand images
//   - V re-laid out as the A-operand images of O^T = V^T P^T
//   - rotary cos/sin tables from the float64 position grid
// All of it is HBM-bound streaming work (a few hundred MB per layer call against ~29 TFLOP of attention).
#include "pkh3_common.h"
#include "pkh3_index.h"
#include "pkh3_internal.h"
#include "pkh3_plan.h"

namespace pkh3 {

// ------------------------------------------------------------------------------------------------
// Key-mask compaction in front of the K/V pass, where the pass does not do it itself (kv_pass_reads_mask): idx[b][slot] = key index of the slot-th valid key, cnt[b] = number of valid keys.
// One workgroup of 1024 threads per batch walks the mask in chunks, carrying the running count.
__global__ __launch_bounds__(1024) void mask_compact_kernel(const uint8_t* __restrict__ mask, int Sk,
                                                            int* __restrict__ idx, int* __restrict__ cnt) {
  __shared__ int wave_tot[16];
  __shared__ int carry;
  const int b = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint8_t* m = mask + (int64_t)b * Sk;
  int* out = idx + (int64_t)b * Sk;
  if (tid == 0) carry = 0;
  __syncthreads();
  for (int base = 0; base < Sk; base += 1024) {
    const int key = base + tid;
    const bool on = key < Sk && m[key] != 0;
    const unsigned long long bal = __ballot(on);
    const int before = __popcll(bal & ((1ull << lane) - 1ull));
    if (lane == 0) wave_tot[wave] = __popcll(bal);
    __syncthreads();
    int off = carry;
    for (int w = 0; w < wave; ++w) off += wave_tot[w];
    if (on) out[off + before] = key;
    __syncthreads();
    if (tid == 0) {
      int t = carry;
      for (int w = 0; w < 16; ++w) t += wave_tot[w];
      carry = t;
    }
    __syncthreads();
  }
  if (tid == 0) cnt[b] = carry;
}

static hipError_t launch_mask_compact(const uint8_t* mask, int B, int Sk, int* idx, int* cnt, hipStream_t st) {
  hipLaunchKernelGGL(mask_compact_kernel, dim3(B), dim3(1024), 0, st, mask, Sk, idx, cnt);
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------
// The K/V pass: one workgroup takes one 64-key tile of `heads_per_wg` consecutive heads, its K rows (RMSNorm, rotation,
// fp8 quantisation -> operand images; the Q side does the same math inside the attention kernel) or its V rows
// (-> operand images), by the parity of blockIdx.x: both sides of a tile in one launch, so that the streaming V waves
// run beside the K waves' arithmetic.
//
// Bound by HBM and, before that, by the CU's load path: the rotation tables and the norm weights of a row are 1 KiB,
// the row of one head 256 B.  So a wave keeps them in registers and walks the heads, with the rows of the next head on
// their way while it works on one; 16 rows per wave (a quarter of a tile) leaves the registers for three waves per SIMD.
// Against a K and a V launch of one wave per tile and head: 48,360 rows x 24 heads 293 -> 241 us (4.9 TB/s), fp8 285 -> 215;
// 15,342 rows 127 -> 85 us.

// K: lane (c = l%16, g = l/16) of wave kb gets the 32 elements d = 32*ks + 8*g + j of row 16*kb + c -- its own 16 bytes
// of the block's four K images, so norm and rotation need two cross-lane exchanges (the sum of squares), and every store
// instruction writes one whole 1 KiB image.  Rows and tables are asked for as they lie in memory (four whole rows a load) and
// turned around in 4 KiB of LDS a wave: asked for in the order of the images, 64 B of 16 rows a load, the CU's load path gives
// a quarter of its rate.  That against this: 48,360 rows x 24 heads 218 -> 209 us, fp8 204 -> 196; 15,342 rows 70 -> 64.5;
// 3 x 8 heads x 777 rows with a mask (with the shorter look through it below) 12.3 -> 8.6; 2 x 4 heads x 200 rows 5.0 -> 4.6.
template <bool FP8>
__device__ __forceinline__ void k_tile(const QkPrologueParams& p, int tile, int b, int h0, int n_heads, int rows, const int* source,
                                       unsigned* s_norm, unsigned* s_amax, char* turn) {
  const int lane = threadIdx.x & 63, kb = threadIdx.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  const bool valid = tile * 64 + kb * 16 + c < rows;
  int src[4];                                            // rows of the block as they are asked for
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int in_tile = kb * 16 + 4 * i + g;
    src[i] = tile * 64 + in_tile < rows ? (source ? source[in_tile] : tile * 64 + in_tile) : 0;
  }
  const char* xr = (const char*)p.x + ((int64_t)b * p.sb + (int64_t)h0 * p.sh) * 2;
  Rows16 next, cos, sin;
  ask_rows16(next, xr, p.ss * 2, src, lane);
  NormLanes norm;
  load_norm_lanes(norm, p.norm_w, lane);
  RopeQuarter rope;
  if (p.rope_mode != 0) {
    ask_rows16(cos, (const char*)p.cos_t, kD / 2 * sizeof(float), src, lane);
    ask_rows16(sin, (const char*)p.sin_t, kD / 2 * sizeof(float), src, lane);
    turn_table(cos, rope.c, p.rope_mode, turn, lane);
    turn_table(sin, rope.s, p.rope_mode, turn, lane);
  }
  char* ob = p.out + (int64_t)(b * p.H + h0) * p.out_bh_stride + (int64_t)tile * p.out_blk_stride;
#pragma unroll 1
  for (int hi = 0; hi < n_heads; ++hi, ob += p.out_bh_stride) {
    bf16x8 raw[4];
    float x[32];
    turn_elements(next, raw, turn, lane);
    if (hi + 1 < n_heads) ask_rows16(next, xr + (int64_t)(hi + 1) * p.sh * 2, p.ss * 2, src, lane);
    norm_row(x, raw, p.norm_w != nullptr, p.eps, norm, 1.0f);
    rope_row(x, p.rope_mode, rope);
    if (tile * 64 + 64 > rows) {                         // rows past the end are zero, whatever row 0 and its rotation hold
#pragma unroll
      for (int i = 0; i < 32; ++i) x[i] = valid ? x[i] : 0.f;
    }
    float part[4] = {0.f, 0.f, 0.f, 0.f};   // four running sums: one would be a chain of 32 dependent instructions
#pragma unroll
    for (int i = 0; i < 32; ++i) part[i & 3] += x[i] * x[i];
    const float ssq = wave_sum_groups((part[0] + part[1]) + (part[2] + part[3]));
    if (g == 0) atomicMax(s_norm + hi, __float_as_uint(fmaxf(ssq, 0.f)));   // a NaN row counts as none
    if constexpr (!FP8) {
      // image (half, ks, kb2) of the tile, half = kb / 2, kb2 = kb % 2: this lane's piece ks at its own place
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        bf16x8 t;
#pragma unroll
        for (int j = 0; j < 8; ++j) t[j] = (__bf16)x[ks * 8 + j];
        *(bf16x8*)(ob + ((((kb >> 1) * 4 + ks) * 2 + (kb & 1)) * 64 + lane) * 16) = t;
      }
    } else {
      // one scale per 64-row tile: the largest magnitude of the workgroup's four waves
      float amax = 0.f;
#pragma unroll
      for (int i = 0; i < 32; ++i) amax = fmaxf(amax, fabsf(x[i]));
      amax = max_across_groups(amax);
      if (g == 0) atomicMax(s_amax + hi, __float_as_uint(amax));
      __syncthreads();
      const float scale = fp8_block_scale(__uint_as_float(s_amax[hi]), p.fp8_pow2 != 0);
      const float inv = 1.0f / scale;
      if (threadIdx.x == 0) p.scale_out[(int64_t)(b * p.H + h0 + hi) * p.nBlk64 + tile] = scale;
      // key block kb is 2 KiB, chunk c2 of a lane holds its pieces ks = 2*c2 and 2*c2 + 1
#pragma unroll
      for (int c2 = 0; c2 < 2; ++c2) {
        const i32x2 q0 = quant_fp8_piece(x + 16 * c2, inv), q1 = quant_fp8_piece(x + 16 * c2 + 8, inv);
        *(i32x4*)(ob + ((kb * 2 + c2) * 64 + lane) * 16) = i32x4{q0[0], q0[1], q1[0], q1[1]};
      }
    }
  }
  // largest row norm of the tile in each head, after norm and rotation: an upper bound for every logit is |q_i| * max_j |k_j|,
  // which lets the attention kernel drop the running max when the bound is small.  Every tile has places of its own (one
  // for each 32 rows, as the projection's K epilogue fills them): one word a head, raised by all its tiles, was what a call of few
  // heads and tiles waited for -- atomics of eight XCDs on one line, 3 x 8 heads x 13 tiles 15.4 us against 8.0 (with
  // rotation 17.5 against 11.8), and a launch to clear the words besides.
  __syncthreads();
  if ((int)threadIdx.x < n_heads) {
    const float top = sqrtf(__uint_as_float(s_norm[threadIdx.x]));
    float* row = p.norm_out + (int64_t)(b * p.H + h0 + threadIdx.x) * p.norm_stride;
    *(f32x2*)(row + kNormFirst + 2 * tile) = f32x2{top, top};
    if (tile == 0) row[0] = -1.0f;
  }
}

// V: wave (half, odd) takes 32 keys of the even or odd heads.  Whole 16-byte pieces of rows go through 8 KiB of LDS of
// its own and come back transposed: lane (c, g) of image (half, db) needs V[32*half + v_image_key(g, j)][16*db + c], and
// one ds_read_b64_tr_b16 gives every 16-lane group g four rows x 16 columns that way round (lane 4*r + m of the group
// names the row r's columns 4*m .. +3, lane c receives column c).  The 32-byte pieces of a row are XOR-swizzled by the row
// so that 8 rows of the same columns lie in different banks.
__device__ __forceinline__ void v_tile(const VPrologueParams& p, int tile, int b, int h0, int n_heads, int rows, const int* source, char* lds) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = wave & 1, first = wave >> 1;
  const int row0 = tile * 64 + half * 32;
  char* mine = lds + wave * 8192;
  const int chunk = lane & 15, r4 = lane >> 4;        // 16-byte chunk of row 4*i + r4, i = 0..7
  const __bf16* vr[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = row0 + 4 * i + r4;
    int src = 0;
    if (row < rows) src = source ? source[row - tile * 64] : row;
    vr[i] = (const __bf16*)p.v + (int64_t)b * p.sb + (int64_t)src * p.ss + 8 * chunk;
  }
  auto fetch = [&](bf16x8 (&raw)[8], int hi) {
#pragma unroll
    for (int i = 0; i < 8; ++i) raw[i] = *(const bf16x8*)(vr[i] + (int64_t)(h0 + hi) * p.sh);
  };
  if (first >= n_heads) return;
  bf16x8 next[8];
  fetch(next, first);
  char* ob = p.out + (int64_t)(b * p.H + h0 + first) * p.out_bh_stride + (int64_t)tile * p.out_tile_stride + half * 8192;
  const int g = lane >> 4, c = lane & 15;
#pragma unroll 1
  for (int hi = first; hi < n_heads; hi += 2, ob += 2 * p.out_bh_stride) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = 4 * i + r4;
      *(bf16x8*)(mine + r * 256 + ((chunk ^ (2 * (r & 7))) * 16)) = next[i];
    }
    if (hi + 2 < n_heads) fetch(next, hi + 2);
#pragma unroll
    for (int db = 0; db < 8; ++db) {
      bf16x8 img;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const int r = 16 * kb + 4 * g + (c >> 2);      // the row this lane names, columns 16*db + 4*(c%4) .. +3
        const auto t = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
            (__attribute__((address_space(3))) bf16x4*)(mine + r * 256 + ((db ^ (r & 7)) * 32) + 8 * (c & 3)));
#pragma unroll
        for (int j = 0; j < 4; ++j) img[4 * kb + j] = row0 + 16 * kb + 4 * g + j < rows ? t[j] : (__bf16)0.0f;
      }
      *(bf16x8*)(ob + (db * 64 + lane) * 16) = img;
    }
  }
}

// Key mask of one batch entry: the number of valid keys, and the source rows of this tile's 64 (where it has them) in `source`, for all
// four waves after the next barrier.  Every workgroup looks at the whole mask: a few bytes a thread, asked for at
// once, where a launch of its own in front of this one cost the call 3 to 4 us (3 x 8 heads x 777 rows 39.9 -> 36.5).
// kMost: 64-key pieces of a wave.  What it costs is instructions that a wave issues one by one, so short masks take a
// form with 4 pieces rather than 16, and a piece none of whose keys is the tile's is not placed.
template <int kMost>
__device__ __forceinline__ int compact_mask(const uint8_t* mask, int S, int tile, int* source) {
  __shared__ int wave_tot[4];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pieces = (S + 255) / 256;
  const int key0 = wave * pieces * 64 + lane;
  uint8_t m[kMost];
#pragma unroll
  for (int i = 0; i < kMost; ++i) m[i] = i < pieces && key0 + 64 * i < S ? mask[key0 + 64 * i] : 0;
  unsigned long long on[kMost];
  int total = 0;
#pragma unroll
  for (int i = 0; i < kMost; ++i) {
    on[i] = __ballot(m[i] != 0);
    total += __popcll(on[i]);
  }
  if (lane == 0) wave_tot[wave] = total;
  __syncthreads();
  int at = -64 * tile, all = 0;                         // place of the next valid key, counted from the tile's first
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const int n = wave_tot[w];
    if (w < wave) at += n;
    all += n;
  }
#pragma unroll
  for (int i = 0; i < kMost; ++i) {
    const int here = __popcll(on[i]);
    if (at < 64 && at + here > 0) {                     // (wave-uniform) some of these 64 keys may be the tile's
      const int place = at + __popcll(on[i] & ((1ull << lane) - 1ull));
      if (m[i] != 0 && place >= 0 && place < 64) source[place] = key0 + 64 * i;
    }
    at += here;
  }
  return all;
}

template <bool FP8>
__global__ __launch_bounds__(256, 3) void kv_prologue_kernel(QkPrologueParams k, VPrologueParams v, SparsePlanParams plan, int heads_per_wg,
                                                             int groups) {
  __shared__ __attribute__((aligned(16))) char lds[4 * 8192];
  static_assert(kPlanChunk <= (int)sizeof(lds), "the masks of a plan entry");
  if ((int)blockIdx.x < plan.n) {
    if (blockIdx.y == 0) plan_entry(plan, blockIdx.x, (unsigned char*)lds);
    return;
  }
  const int bid = blockIdx.x - plan.n;
  // head groups vary fastest across workgroups: neighbours read neighbouring pieces of the same [S, H, D] rows
  const int tile = bid / (2 * groups), in_tile = bid % (2 * groups), b = blockIdx.y;
  const int h0 = (in_tile >> 1) * heads_per_wg, n = min(heads_per_wg, k.H - h0);
  if (k.clear_n > 0) {
    const int64_t word = word_to_clear(blockIdx.y, gridDim.x - plan.n, bid, threadIdx.x);
    if (word < k.clear_n) k.clear[word] = 0u;
  }
  __shared__ int source[64];                            // source row of each row of the tile (key mask)
  int rows = k.S;
  if (k.row_cnt) {
    const uint8_t* mask = k.mask + (int64_t)b * k.S;
    rows = !k.mask ? k.row_cnt[b] : k.S <= 1024 ? compact_mask<4>(mask, k.S, tile, source) : compact_mask<kOwnMaskKeys / 256>(mask, k.S, tile, source);
    if (k.mask && tile == 0 && in_tile == 0 && threadIdx.x == 0) k.row_cnt[b] = rows;
    if (tile * 64 >= rows) return;                      // no valid key in this tile: nothing reads its record
    if (!k.mask && threadIdx.x < 64 && tile * 64 + threadIdx.x < rows) source[threadIdx.x] = k.gather_idx[(int64_t)b * k.S + tile * 64 + threadIdx.x];
    __syncthreads();
  }
  const int* src = k.row_cnt ? source : nullptr;
  if (in_tile & 1) {
    v_tile(v, tile, b, h0, n, rows, src, lds);
    return;
  }
  unsigned* s_norm = (unsigned*)lds;
  unsigned* s_amax = s_norm + kKvMaxHeads;
  if (threadIdx.x < 2 * kKvMaxHeads) s_norm[threadIdx.x] = 0u;
  __syncthreads();
  k_tile<FP8>(k, tile, b, h0, n, rows, src, s_norm, s_amax, lds + 8192 + (threadIdx.x >> 6) * 4096);
}

hipError_t launch_kv_prologue(QkPrologueParams k, const VPrologueParams& v, const SparsePlanParams& plan, hipStream_t st) {
  int cus = 0;
  hipError_t e = device_cu_count(&cus);
  if (e != hipSuccess) return e;
  cus = max(cus, 1);
  const KvSplit split = kv_split(k.nBlk64, k.B, k.H, cus, k.rope_mode != 0, k.mask != nullptr);
  const int64_t workgroups = (int64_t)2 * split.groups * k.nBlk64 * k.B;
  if (k.mask && !kv_pass_reads_mask(k.S, workgroups, cus)) {
    if ((e = launch_mask_compact(k.mask, k.B, k.S, k.gather_idx, k.row_cnt, st)) != hipSuccess) return e;
    k.mask = nullptr;
  }
  // The entries of a block-sparse plan ride in front: each is a chain of short steps, so they end under the tiles' loads.  A launch
  // of their own costs a call 3 us (24 heads x 14,907 rows in fp8: 683.9 -> 680.4 us; 48,360 in bf16: 6,876 -> 6,873).
  const dim3 grid((unsigned)(2 * split.groups) * k.nBlk64 + plan.n, k.B), block(256);
  if (k.fp8) hipLaunchKernelGGL(kv_prologue_kernel<true>, grid, block, 0, st, k, v, plan, split.heads, split.groups);
  else hipLaunchKernelGGL(kv_prologue_kernel<false>, grid, block, 0, st, k, v, plan, split.heads, split.groups);
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void sparse_plan_kernel(SparsePlanParams p) {
  __shared__ unsigned char mask[kPlanChunk];
  plan_entry(p, blockIdx.x, mask);
}

hipError_t launch_sparse_plan(const SparsePlanParams& p, hipStream_t st) {
  hipLaunchKernelGGL(sparse_plan_kernel, dim3(p.n), dim3(256), 0, st, p);
  return hipGetLastError();
}

// The largest norm of every head in front of its norms, for keys that many calls will use: their workgroups then read one word
// each (24 heads x 16,366 queries against 512 prepared keys 103.2 -> 102.0 us).  A head's 4,096 norms (131,072 keys) are asked for at
// once: bound by that one trip to memory.
__global__ __launch_bounds__(256) void fold_norms_kernel(QkPrologueParams p) {
  __shared__ float wave_top[4];
  const int bh = blockIdx.x, lane = threadIdx.x & 63;
  const int n = ((p.row_cnt ? p.row_cnt[bh / p.H] : p.S) + 31) / 32;
  float* row = p.norm_out + (int64_t)bh * p.norm_stride;
  float top = 0.f;
  for (int i0 = 4 * threadIdx.x; i0 < n; i0 += 4096) {
    f32x4 v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = *(const f32x4*)(row + kNormFirst + min(i0 + 1024 * j, (n - 1) & ~3));
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) top = i0 + 1024 * j + e < n ? fmaxf(top, v[j][e]) : top;   // (places past the last may never have been written)
  }
  top = wave_max(top);
  if (lane == 0) wave_top[threadIdx.x >> 6] = top;
  __syncthreads();
  if (threadIdx.x == 0) row[0] = fmaxf(fmaxf(wave_top[0], wave_top[1]), fmaxf(wave_top[2], wave_top[3]));
}

hipError_t launch_fold_norms(const QkPrologueParams& k, hipStream_t st) {
  hipLaunchKernelGGL(fold_norms_kernel, dim3((unsigned)(k.B * k.H)), dim3(256), 0, st, k);
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------
// cos/sin tables from the [S,3] float64 position grid.  Pair p of the D/2 = 64 pairs belongs to the
// axis whose slice contains it; inside its slice of n = axis_dims[a]/2 pairs, pair i rotates by
// pos[a] * theta^(-2i / axis_dims[a]).  Computed in float64, stored fp32.
__global__ void rope_tables_kernel(const double* __restrict__ pos, int S, int d0, int d1, int d2, double log_theta,
                                   float* __restrict__ cos_out, float* __restrict__ sin_out) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= (int64_t)S * (kD / 2)) return;
  const int s = (int)(gid / (kD / 2)), pr = (int)(gid % (kD / 2));
  int a, i, dim;
  if (pr < d0 / 2) { a = 0; i = pr; dim = d0; }
  else if (pr < (d0 + d1) / 2) { a = 1; i = pr - d0 / 2; dim = d1; }
  else { a = 2; i = pr - (d0 + d1) / 2; dim = d2; }
  const double freq = exp(-log_theta * (2.0 * i) / (double)dim);
  const double ang = pos[(int64_t)s * 3 + a] * freq;
  cos_out[gid] = (float)cos(ang);
  sin_out[gid] = (float)sin(ang);
}

hipError_t launch_rope_tables(const double* pos, int S, const int* axis_dims, double theta, float* cos_out,
                              float* sin_out, hipStream_t st) {
  const int64_t n = (int64_t)S * (kD / 2);
  hipLaunchKernelGGL(rope_tables_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, pos, S, axis_dims[0],
                     axis_dims[1], axis_dims[2], log(theta), cos_out, sin_out);
  return hipGetLastError();
}

}  // namespace pkh3
