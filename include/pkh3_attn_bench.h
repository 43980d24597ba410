/*
 * pkh3_attn_bench.h -- measurement and test hooks of libpkh3attn.so.  Not part of the product interface
 * (include/pkh3_attn.h): pkh3_attn_time_kernel is the one export that synchronises with the device, and only
 * benchmark harnesses and tests call them.  They replace nothing in the reference, which publishes no kernel
 * timings (it records wall-clock per pipeline stage, src/pika_h3/pipeline.py:91-93,168).
 */
#ifndef PKH3_ATTN_BENCH_H
#define PKH3_ATTN_BENCH_H

#include "pkh3_attn.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Runs `iters` back-to-back launches of ONLY the attention kernel of the given call (the prologue
   that normalises/rotates/lays out K and V runs once before), brackets them with HIP events on
   `stream`, and returns the mean milliseconds per launch in *ms_out.  Synchronises. */
int pkh3_attn_time_kernel(const pkh3_attn_args* a, void* stream, int iters, float* ms_out);

/* The form of the attention kernel the call takes on a device of `cus` compute units (of shapes and options alone, nothing is
   launched and no GPU is needed), or a negative PKH3_E* code. */
enum {
  PKH3_FORM_LONG = 0,   /* dense, 12 waves of 32 queries per workgroup */
  PKH3_FORM_SHORT = 1,  /* dense, 4 waves of 32 queries, half tiles of 32 keys */
  PKH3_FORM_NARROW = 2, /* dense or block-sparse, one block of 32 queries, 4 waves share its keys out */
  PKH3_FORM_SPARSE = 3, /* block-sparse, 8 waves of 32 queries */
  PKH3_FORM_RELAY = 4   /* dense bf16, a workgroup of 12 waves per CU that goes from one 128 queries to the next */
};
int pkh3_attn_form(const pkh3_attn_args* a, int cus);

#ifdef __cplusplus
}
#endif
#endif
