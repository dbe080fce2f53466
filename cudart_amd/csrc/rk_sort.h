// The radix sort as the builders and traces use it (rk_sort.hip): a plan of
// its passes and buffers, so that the kernel that makes the keys can write them
// where the first pass reads them and count the first digits as it goes.
#pragma once

#include "rk_device.h"

// A stable LSD sort of n keys (and values) on their low bits.
template <typename K>
struct RkSortPlan {
  uint32_t n = 0, tiles = 0, copies = 0;
  int passes = 0;              // of 8 bits
  int items = 0;               // keys per lane of the scatter kernel
  bool one = false;            // one workgroup sorts everything in LDS
  uint32_t* head = nullptr;    // [0] error word, then copies x passes x 256 counts
  uint32_t* status = nullptr;  // look-back words
  size_t head_words = 0, status_words = 0;  // status_words: of the first pass
  K* src = nullptr;            // where the unsorted keys and values go
  uint32_t* vsrc = nullptr;
  K* dst = nullptr;            // where the sorted ones end up (the caller's arrays)
  uint32_t* vdst = nullptr;
  K* alt = nullptr;
  uint32_t* valt = nullptr;
};

// Plans a sort of n keys (vals may be NULL) on their low 'bits' bits, into
// keys and vals; anywhere: the unsorted keys may be put where the plan says
// (src, vsrc), else they are in keys and vals. The first word of ws is the
// error word. RK_ERROR_WORKSPACE when ws is too small.
template <typename K>
rk_status rk_sort_plan(uint32_t n, int bits, bool anywhere, K* keys, uint32_t* vals, void* ws, size_t ws_bytes,
                       RkSortPlan<K>& plan);
// Zeroes what the counts of a fused key kernel, and the first pass, need
// (the error word too), and 'info' (RK_INFO_WORDS, may be NULL).
template <typename K>
rk_status rk_sort_clear(hipStream_t st, const RkSortPlan<K>& plan, uint32_t* info);
// Runs it. counted: the digits are counted already (after rk_sort_clear).
// err (may be NULL: the error word): receives RK_FLAG_SPIN_LIMIT.
template <typename K>
rk_status rk_sort_run(hipStream_t st, const RkSortPlan<K>& plan, bool counted, uint32_t* err);

// Digit counts in a key kernel: a workgroup counts into LDS (rk_count_digits),
// then adds its counts to the copy of its block index (rk_flush_digits).
template <typename K, int kPasses>
__device__ __forceinline__ void rk_count_digits(uint32_t* s_hist, K key) {
#pragma unroll
  for (int p = 0; p < kPasses; ++p) atomicAdd(&s_hist[p * 256 + (int)((key >> (8 * p)) & 0xFFu)], 1u);
}
template <int kPasses, int kThreads>
__device__ __forceinline__ void rk_flush_digits(const uint32_t* s_hist, uint32_t* __restrict__ counts,
                                                uint32_t copies) {
  uint32_t* g = counts + (size_t)(blockIdx.x % copies) * (kPasses * 256);
  for (int i = threadIdx.x; i < kPasses * 256; i += kThreads) {
    const uint32_t c = s_hist[i];
    if (c) atomicAdd(&g[i], c);
  }
}
