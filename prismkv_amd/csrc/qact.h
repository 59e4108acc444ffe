// Selection by query activations (router "q_activation", core.py:131-139),
// shared by prismkv_route_qact and the fused step of that router: each head's
// 16 largest activations (value descending, bucket ascending: the stable
// descending argsort) out of kQaParts lists, weights val / max(sum val, 1e-20) / 4
// with the sum taken in rank order; score[bucket] = the weights of the bucket
// summed in head order; the selection = the buckets of positive score and
// nonzero size, by score descending and bucket ascending, up to 64.
#pragma once

#include "select.h"

namespace prismkv {
namespace {

constexpr int kQaParts = 24;             // bucket ranges of qact_part_kernel
constexpr int kQaBuckets = kF / kQaParts;  // 125
constexpr int kQaSel = kHq * kTop;       // 64
static_assert(kQaBuckets * kQaParts == kF && kQaParts * kTop % 64 == 0, "whole ranges, whole 64-key sets");

// Head h's 16 best candidates of group g, rank j in lane j of every row (one wave).
__device__ __forceinline__ unsigned long long qact_head_top(const unsigned long long* cand, int g, int h) {
  constexpr int kSets = kQaParts * kTop / 64;
  unsigned long long v[kSets];
#pragma unroll
  for (int k = 0; k < kSets; ++k)
    v[k] = cand[((size_t)g * kHq + h) * kQaParts * kTop + 64 * k + (threadIdx.x & 63)];
  return sorted_rows_top16<kSets>(v);  // each 16-lane row is one part's ranked list
}

__device__ __forceinline__ bool qact_infinite(unsigned long long key) { return (unsigned)(key >> 12) == 0x7f800000u; }

// A head's weights: val / max(sum of the 16 in rank order, 1e-20) / 4, for the
// wave that holds its list (lane r, rank r).
__device__ __forceinline__ float qact_weight(unsigned long long key) {
  const float val = __uint_as_float((unsigned)(key >> 12));
  float s = 0.f;
#pragma unroll
  for (int r = 0; r < kTop; ++r) s += lane_bcast(val, r);
  return (val / fmaxf(s, 1e-20f)) / (float)kHq;
}

// One wave: entry e = 16 h + r (lane e) is head h's rank-r activation, top[e].
// Returns the selection's sorted keys (lane r: rank r, 0 past the last) and, of
// the lane's own entry, its bucket, the bucket's score and whether the entry is
// the bucket's first.
__device__ __forceinline__ unsigned long long qact_rank(const unsigned long long* top, const int* counts, int& bucket,
                                                        float& score, bool& first) {
  const int lane = threadIdx.x & 63, h = lane >> 4;
  const unsigned long long key = top[lane];  // never 0: every part holds at least 16 real buckets
  const float val = __uint_as_float((unsigned)(key >> 12));
  bucket = key ? key_bucket(key) : 0;
  const int size = counts[bucket];
  float s = 0.f;
#pragma unroll
  for (int r = 0; r < kTop; ++r) s += __uint_as_float((unsigned)(top[kTop * h + r] >> 12));
  s = fmaxf(s, 1e-20f);
  const float c = (val / s) / (float)kHq;
  // the bucket's score: its entries' weights added in entry order, from 0
  float sc = 0.f;
  first = true;
#pragma unroll
  for (int e = 0; e < kQaSel; ++e) {
    const bool same = __builtin_amdgcn_readlane(bucket, e) == bucket;
    sc += same ? lane_bcast(c, e) : 0.f;
    first = first && !(same && e < lane);
  }
  score = sc;
  return wave_sort_desc(first && sc > 0.f && size > 0 ? make_key(sc, bucket) : 0ull);
}

}  // namespace
}  // namespace prismkv
