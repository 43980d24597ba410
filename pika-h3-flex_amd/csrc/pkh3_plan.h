// The block-sparse plan, made beside the K/V pass of a call (pkh3_prologue.hip) or, on prepared keys, by a launch of its own.
#pragma once
#include "pkh3_common.h"
#include "pkh3_internal.h"

namespace pkh3 {

// Block-sparse plan.  For each workgroup (kSparseRows consecutive 64-query row-blocks) 1 + kSparseRows ascending
// tile lists, each `nKt` ints apart: [0] the key tiles every one of its row-blocks keeps (walked by all its waves
// together), [1+r] the tiles row-block r keeps that are not in [0] (walked by that row-block's wave pair).  One
// workgroup per attention workgroup merges the CSR rows through an LDS mask array, key tiles in chunks.
constexpr int kPlanChunk = 8192;   // bytes of LDS for the masks
__device__ __forceinline__ void plan_entry(const SparsePlanParams& p, int qt, unsigned char* mask) {
  __shared__ int wave_tot[4];
  __shared__ int carry[kSparseLists];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nKt = p.nKt;
  int* out = p.plan + (int64_t)qt * p.plan_stride;
  const int rows_here = max(0, min(kSparseRows, p.nRow64 - qt * kSparseRows));
  const int full = (1 << rows_here) - 1;
  if (tid < kSparseLists) carry[tid] = 0;
  for (int base = 0; base < nKt; base += kPlanChunk) {
    for (int i = tid; i < kPlanChunk; i += 256) mask[i] = 0;
    __syncthreads();
    for (int r = 0; r < rows_here; ++r) {
      const int row = qt * kSparseRows + r;
      const int beg = p.row_ptr[row], end = p.row_ptr[row + 1];
      for (int j = beg + tid; j < end; j += 256) {
        const int col = p.col_idx[j] - base;
        // within one r two threads touch the same byte only when the row repeats a column, and then both store the
        // same value; columns outside [0, nKt) are ignored; a row whose end lies before its start is empty
        if (col >= 0 && col < kPlanChunk && col + base < nKt) mask[col] |= (unsigned char)(1 << r);
      }
      __syncthreads();
    }
    for (int list = 0; list < kSparseLists; ++list) {
      for (int c0 = 0; c0 < kPlanChunk && base + c0 < nKt; c0 += 256) {
        const int col = c0 + tid;
        const int mk = (base + col < nKt) ? mask[col] : 0;
        const bool take = list == 0 ? (mk == full && full != 0) : (((mk >> (list - 1)) & 1) && mk != full);
        const unsigned long long bal = __ballot(take);
        const int before = __popcll(bal & ((1ull << lane) - 1ull));
        if (lane == 0) wave_tot[wave] = __popcll(bal);
        __syncthreads();
        int off = carry[list];
        for (int wv = 0; wv < wave; ++wv) off += wave_tot[wv];
        if (take) out[list * nKt + off + before] = base + col;
        __syncthreads();
        if (tid == 0) carry[list] += wave_tot[0] + wave_tot[1] + wave_tot[2] + wave_tot[3];
        __syncthreads();
      }
    }
  }
  if (tid < kSparseLists) p.plan_cnt[qt * kSparseLists + tid] = carry[tid];
}

}  // namespace pkh3
