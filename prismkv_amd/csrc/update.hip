// Stage 4 -- the index update (append_index) and the prefill index build
// (build_index): encode keys with the group's SAE, take the exact batch-wide
// positive Top-k of the activations, set the members' bitmap bits and
// (re)compute the bucket moments.
//
// Semantics: src/prismkv/core.py:186-201 (append_index) on top of
//   build_index  core.py:92-103  center = keys.float().mean(0) unless given
//                                (append: the ORIGINAL center);
//                                x = (k - center) / key_scale;
//                                a = relu(x W^T + b) (SharedSAE.dense,
//                                core.py:47-48);
//   positive_global_topk core.py:13-26  budget N * key_mean over the keys
//                                indexed: keep a > tau and a > 0, then, if
//                                tau > 0, values == tau in ascending flat
//                                index (token * F + feature) up to the budget;
//   summarize    core.py:76-89   per-bucket mean / population variance of
//                                the ORIGINAL keys (two-pass);
//   the merge    core.py:190-199 mean = (a m_a + b m_b) / max(a+b, 1),
//                                var = (a v_a + b v_b) / max(a+b, 1)
//                                      + a b / max(a+b, 1)^2 (m_a - m_b)^2,
//                                in fp32 and in that operation order;
//   lists        core.py:200     new members are tokens H + t: here bits
//                                H + t of the bucket's bitmap row
//                                (kernels/ppu_8b/pack.cu:5 bit order).
//
// Launches of one update (all G groups at once; the update runs every
// `interval` tokens, its cost is amortised):
//   sample   W as pairs of f16 in the encode's operand order, and a histogram
//            (13 bits) of the positive activations of a few hundred tokens;
//   encode   the GEMM on the f16 matrix cores (in fp32 for rows and buckets that
//            this would not serve), 512 buckets x 16 tokens per workgroup and
//            step, a = relu(...): the values at or above a floor
//            read off the sample (about twice the budget of them) go to the
//            group's candidate list as (flat index, value), and, where the
//            caller reads them, all of them to [G][N][F];
//   split    finds the digit of the candidates' values that holds tau, the
//            budget-th largest (the encode has counted them): the candidates
//            above it are members, whose bitmap bits it sets, those in it go to
//            a short list;
//   select   one workgroup per group finds tau in that list and, when ties at
//            tau overflow the budget, the flat index of the last one taken, and
//            sets the rest of the bits (many, where they read the activations);
//   moments  per 32-bucket tile: new members from the bitmap, two-pass
//            moments of their keys, merge, counts += new.
// The sample decides only how long the list is.  Where it misjudged (fewer
// candidates than the budget, or more than the list holds) the same kernels
// read the dense activations instead, and the result is the same.
// Keys are the model's bf16 K cache or fp32 rows (the `_f32` entry points):
// the kernels that read keys take the element type as a template argument
// and widen every key to fp32 at the load, so both compute the same fp32 /
// double arithmetic on the values they are given.
// The build runs the same selection over all H keys of a group (in batches
// of groups, so the activations of one batch fit the workspace) after a
// center pass and a bitmap clear, with select's work spread over many
// workgroups for long histories (histogram / digit / refine, three levels, emit),
// and computes every bucket's moments from scratch (build_moments: one
// workgroup per bucket, any member count).  Unless the caller keeps them, a
// build never writes its activations (12 KB per key) at all.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"

namespace prismkv {
namespace {

constexpr int kUT = 256;
constexpr int kFT = 64;        // buckets per encode tile
constexpr int kFTiles = (kF + kFT - 1) / kFT;  // 47
constexpr int kBins = 2048;
constexpr int kRep = 4;        // global histogram replicas
constexpr int kLevels = 3;
constexpr int kRefineBlocks = 256;  // workgroups per group of a pass over a
constexpr int kMaxTieBlocks = 4096;  // contiguous ranges of a per group for the ordered ties
constexpr int kTieMinLen = 65536;    // values per range at least (multiple of 4 * kUT)
constexpr int kTieGrid = 256;        // workgroups per group of the tie kernels
constexpr int kCenterParts = 64;     // row ranges of the center sum
constexpr unsigned kListSlack = 1u << 18;  // list entries beyond kListPerKey per key
constexpr int kListPerKey = 48;
constexpr int kSampleShift = 18, kSampleBins = 1 << (31 - kSampleShift);  // 13-bit digits of positive floats: 3.1% each
constexpr int kSelectMax = 4096;  // keys up to which one workgroup per group selects
constexpr int kFineShift = 12;     // the candidates' own digits: 2^12 bit patterns each (0.05%), kBins of them from the floor on
constexpr int kMaxBuild = 1 << 20;   // keys per group of a build (N * F < 2^32 flat indices)
constexpr int kBuildCenter = 1;      // prismkv_build flag: compute the center (else it is an input)
constexpr int kBuildNoAct = 4;       // prismkv_build flag: the activations need not be left in the workspace

// ctl words per group
enum { kMode = 0, kPrefix, kRem, kTau, kNeed, kTies, kOrdered, kCount, kFloor, kListLen, kCut, kTieLen, kArrived, kCtl = 16 };
enum { kModeTopK = 0, kModeAllPositive = 1 };

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x2 load_f2(__amdgpu_buffer_rsrc_t r, unsigned byte_offset, int base) {
  const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, byte_offset, base, 0);
  return f32x2{__uint_as_float(v[0]), __uint_as_float(v[1])};
}

// Key loads of the two key element types: 2 or 8 consecutive dims as the
// raw loaded bits (kept packed while in flight) and their fp32 values.
template <typename KT>
struct KeyLoad;

template <>
struct KeyLoad<uint16_t> {  // bf16
  typedef uint32_t Raw2;
  static __device__ __forceinline__ Raw2 load2(__amdgpu_buffer_rsrc_t r, unsigned byte_offset, int base = 0) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, byte_offset, base, 0);
  }
  static __device__ __forceinline__ float lo(Raw2 r) { return bf16_lo(r); }
  static __device__ __forceinline__ float hi(Raw2 r) { return bf16_hi(r); }
  typedef u32x4 Raw8;
  static __device__ __forceinline__ Raw8 raw8(const uint16_t* p) { return *reinterpret_cast<const u32x4*>(p); }
  static __device__ __forceinline__ float at(const Raw8& r, int j) { return j & 1 ? bf16_hi(r[j >> 1]) : bf16_lo(r[j >> 1]); }
  static __device__ __forceinline__ void load8(const uint16_t* p, float (&x)[8]) {
    const Raw8 v = raw8(p);
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = at(v, j);
  }
};

template <>
struct KeyLoad<float> {
  typedef unsigned Raw2 __attribute__((ext_vector_type(2)));
  static __device__ __forceinline__ Raw2 load2(__amdgpu_buffer_rsrc_t r, unsigned byte_offset, int base = 0) {
    return __builtin_amdgcn_raw_buffer_load_b64(r, byte_offset, base, 0);
  }
  static __device__ __forceinline__ float lo(Raw2 r) { return __uint_as_float(r[0]); }
  static __device__ __forceinline__ float hi(Raw2 r) { return __uint_as_float(r[1]); }
  struct Raw8 {
    u32x4 a, b;
  };
  static __device__ __forceinline__ Raw8 raw8(const float* p) {
    return Raw8{reinterpret_cast<const u32x4*>(p)[0], reinterpret_cast<const u32x4*>(p)[1]};
  }
  static __device__ __forceinline__ float at(const Raw8& r, int j) { return __uint_as_float(j < 4 ? r.a[j & 3] : r.b[j & 3]); }
  static __device__ __forceinline__ void load8(const float* p, float (&x)[8]) {
    const Raw8 v = raw8(p);
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = at(v, j);
  }
};

struct UpdateArgs {
  const void* k;      // K rows (bf16 or fp32); the block is rows [H, H+N) of each group
  int64_t ks;         // group stride (elements)
  const float* W;     // [G][F][128]
  const float* b;     // [G][F]
  const float* center;  // [G][128]
  const float* scale;   // [G]
  uint32_t* bits;
  int64_t row_words;
  int* counts;     // [G][kFP]
  float* moments;  // [G][kChunks][256][32]
  float* act;      // [G][N][F]
  _Float16* wsplit;  // [G][kFTiles][kWTile] W split for the encode
  unsigned* hist;  // [G][kLevels][kRep][kBins]
  unsigned* ctl;   // [G][kCtl]
  unsigned* tcount;  // [G][tie_blocks] ties per contiguous range of a
  unsigned* sample;  // [G][kSampleBins] histogram of the sample tokens' positive values
  uint2* list;       // [G][list_cap] candidates: (flat index, value bits) of the values at or above the floor
  unsigned* ties;    // [G][list_cap] flat indices of the values equal to tau, when they overflow the budget
  unsigned list_cap;  // entries per group
  unsigned target;    // sample values at or above the floor, at least
  int listed;         // whether the call collects candidates
  int fine;           // whether the encode counts them in fine digits (hist level 0), for split_kernel
  int H, N;          // first key row / bitmap column, keys indexed
  long long budget;  // N * key_mean
  int tie_blocks;
  long long tie_len;  // values per range, a multiple of 4 * kUT
};

__device__ __forceinline__ unsigned budget_of(const UpdateArgs& a) {
  const long long n = (long long)a.N * kF;
  return (unsigned)(a.budget < n ? a.budget : n);
}

// Whether the group's candidate list holds every value the selection can take
// (after the collecting encode): it did not overflow, and it has the budget's
// number of values or every positive one.
__device__ __forceinline__ bool list_ok(const UpdateArgs& a, int g) {
  if (!a.listed) return false;
  const unsigned* ctl = a.ctl + (size_t)g * kCtl;
  const unsigned len = ctl[kListLen];
  return len <= a.list_cap && (len >= budget_of(a) || ctl[kFloor] <= 1u);
}

__device__ __forceinline__ unsigned* hist_of(const UpdateArgs& a, int g, int level) {
  return a.hist + ((size_t)g * kLevels + level) * kRep * kBins;
}

__device__ __forceinline__ unsigned fine_digit(unsigned u, unsigned floor) {
  return min((u - floor) >> kFineShift, (unsigned)kBins - 1u);
}

// ---------------------------------------------------------------------------
// The encode's products run on the f16 matrix cores as a split: an fp32 value
// v times a power of two is hi + lo, hi = f16(v), lo = f16(v - hi), and
//   x . w = x_hi . w_hi + x_hi . w_lo + x_lo . w_hi
// in fp32 accumulators (three f16 MFMAs of 32 dims instead of eight fp32 ones
// of 4).  hi + lo is within 2^-22 of v at most and 2^-24.8 rms, x_lo . w_lo
// (left out) 2^-24.7 rms of its product: not v itself, but over many dims less
// than the roundings of an fp32 chain.  Against 64 bits the activations of dense
// rows are within 1.4e-7 (2-norm over a block) where the fp32 MFMA chain has
// 2.1e-7; the fewer products of a sum are not 0, the shorter the chain's error
// (1.0e-7 at 32 of them, 2.5e-8 at one), while the split's stays (0.8 to 1.0e-7).
// The power of two, per key row and per bucket, brings the largest magnitude
// to [2^14, 2^15), so nothing overflows f16 and what underflows is below 2^-39
// of that largest one.  A row or bucket is not split, its values being computed
// by fp32 MFMA (fp32_products), if
//   - it is not finite, or its largest magnitude lies outside 2^+-60 (the
//     scales' products would leave fp32);
//   - fewer than kMinDims of its dims are at least 2^-16 of the largest one (a
//     key dim 2^18 above the others under a zero weight: 2.4e-7 split, 2.0e-7
//     by the chain).  A split row and a split bucket then share 32 such dims at
//     least, where the split is the closer one.  An all-zero one is split.
//
// The split W of tile ft (64 buckets) is 32 fragments of 1 KB,
// [kb (4)][hi, lo][j (4)], lane (i, q) = (l % 16, l / 16) of a fragment holding
// bucket 64 ft + 16 j + i, dims 32 kb + 8 q .. + 7 (an MFMA A operand), then
// the buckets' biases and inverse scales.  It is made once per call, by the
// sample kernel, and not in each encode workgroup: that takes it off the
// encode's VALU, which its epilogue already fills.
// ---------------------------------------------------------------------------
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
constexpr int kScaleExp = 14;   // scaled rows have their largest magnitude in [2^14, 2^15)
constexpr int kMaxScale = 60;   // |exponent| of a row's or bucket's largest magnitude, at most
constexpr int kMinDims = 80;    // significant dims of a row or bucket that is split, at least
constexpr float kSignificant = 0x1p-16f;  // of the largest magnitude, at least
constexpr int kWTile = kFT * kD * 2 + kFT * 4;  // f16 words of a split W tile: the fragments, 64 biases, 64 inverse scales (fp32)
constexpr int kKB = kD / 32;          // MFMA dim blocks

// The power of two that scales a row of largest magnitude m, and its inverse;
// inverse 0 marks a row that is not split.
__device__ __forceinline__ float2 row_scale(float m) {
  if (m == 0.f) return make_float2(1.f, 1.f);
  const int e = (int)(__float_as_uint(m) >> 23) - 127;  // 128 for infinities and NaN, -127 for subnormals
  if (!(e >= -kMaxScale && e <= kMaxScale)) return make_float2(0.f, 0.f);
  const int k = kScaleExp - e;
  return make_float2(__uint_as_float((unsigned)(127 + k) << 23), __uint_as_float((unsigned)(127 - k) << 23));
}

// The larger, or the sum, of lane l's and lane l ^ M's value, M = 8, 16 or 32, by vector
// instructions alone: after a swap the two stand in some order in r[0] and r[1].
template <int M>
__device__ __forceinline__ float max_xor(float v) {
  if constexpr (M == 8) {
    return fmaxf(v, xor8(v));
  } else {
    const unsigned u = __float_as_uint(v);
    const auto r = M == 16 ? __builtin_amdgcn_permlane16_swap(u, u, false, false)
                           : __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
}
template <int M>
__device__ __forceinline__ int add_xor(int v) {
  if constexpr (M == 8) {
    return v + __float_as_int(xor8(__int_as_float(v)));
  } else {
    const auto r = M == 16 ? __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false)
                           : __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
    return (int)(r[0] + r[1]);
  }
}

// Whether at least kMinDims of a row's 128 magnitudes are significant.  The
// calling lane holds N of them, the row's lanes are M = 8 or 16 apart; m
// is the row's largest.  Every row of the wave answers at once: nearly always by
// the lanes' minima alone (a N(0, 1) row has a smaller value once in 250).
template <int M, int N>
__device__ __forceinline__ bool enough_dims(const float (&x)[N], float m) {
  const float least = m * kSignificant;
  float lo = fabsf(x[0]);
#pragma unroll
  for (int i = 1; i < N; ++i) lo = fminf(lo, fabsf(x[i]));
  if (!__any(lo < least)) return true;  // uniform
  int n = 0;
#pragma unroll
  for (int i = 0; i < N; ++i) n += fabsf(x[i]) >= least ? 1 : 0;
  if constexpr (M == 8) n = add_xor<8>(n);
  return add_xor<32>(add_xor<16>(n)) >= kMinDims;
}

template <typename Fn>
__device__ __forceinline__ void split8(const float (&x)[8], Fn scaled, half8& hi, half8& lo) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float v = scaled(x[j]);
    hi[j] = (_Float16)v;
    lo[j] = (_Float16)(v - (float)hi[j]);
  }
}

constexpr int kET = 512;                          // sample and encode workgroups
constexpr int kSampleFew = kET / 64 * 16;         // sample tokens per workgroup at 16 per wave (128); at 32, twice as many
constexpr int kWLoads = kFT * kD * 4 / 16 / kET;  // 16-byte words of a W tile's fragments per thread (4)
constexpr int kWRows = kWTile * 2 / 16;           // 16-byte words of a tile
constexpr int kJ = kFT / 16;                      // 16-bucket columns of a tile (4)

// The wave's key rows and its center, as loaded: lane (i, q) takes dims
// 32 kb + 8 q .. + 7 of its own tokens.  All of it is requested before any is
// used, so the split below waits for one memory round trip.
template <typename KT, int kTB>
struct RowsRaw {
  typename KeyLoad<KT>::Raw8 k[kTB][kKB];
  f32x4 c[kKB][2];
  float scale;
  __device__ __forceinline__ void load(const UpdateArgs& a, int g, const int (&tok)[kTB]) {
    const int lq = (threadIdx.x >> 4) & 3;
    const KT* kg = static_cast<const KT*>(a.k) + (size_t)g * a.ks + 8 * lq;
    const float* cg = a.center + (size_t)g * kD + 8 * lq;
#pragma unroll
    for (int tb = 0; tb < kTB; ++tb)
#pragma unroll
      for (int kb = 0; kb < kKB; ++kb)
        k[tb][kb] = KeyLoad<KT>::raw8(kg + (size_t)(a.H + tok[tb]) * kD + 32 * kb);
#pragma unroll
    for (int kb = 0; kb < kKB; ++kb) {
      c[kb][0] = *reinterpret_cast<const f32x4*>(cg + 32 * kb);
      c[kb][1] = *reinterpret_cast<const f32x4*>(cg + 32 * kb + 4);
    }
    scale = a.scale[g];
  }
};

// d / s in fp32, rounded to nearest, for many d (Markstein, "Computation of elementary
// functions on the IBM RISC System/6000 processor", 1990): r = 1 / s (rounded), one
// product, its remainder and one correction, which round as the division does
// while nothing leaves the normal range (8e8 random pairs, none differs); an
// infinite or NaN d gives NaN, a row that the split does not serve.
__device__ __forceinline__ float divide_by(float d, float s, float r) {
  const float q = d * r;
  return fmaf(fmaf(-q, s, d), r, q);
}

// d / s by divide_by for any d and a finite s >= 1: where d is infinite or NaN
// (an infinite key, squares past fp32) the division's own result, which the
// remainder would make NaN, by one more instruction.
__device__ __forceinline__ float quotient(float d, float s, float r) {
  return __builtin_amdgcn_div_fixupf(divide_by(d, s, r), s, d);
}

// The split x = (k - center) / key_scale (fp32, core.py:98) of the wave's
// tokens.  xinv: the inverse of each row's scale; returns whether a row of the
// wave is not split.
template <typename KT, int kTB>
__device__ __forceinline__ bool split_rows(const RowsRaw<KT, kTB>& raw, half8 (&xh)[kTB][kKB], half8 (&xl)[kTB][kKB],
                                           float (&xinv)[kTB]) {
  const float s = raw.scale, rs = 1.0f / s;
  // (the scale's own range bounds what divide_by may meet)
  bool bad = !(fabsf(s) >= 0x1p-60f && fabsf(s) <= 0x1p60f);
#pragma unroll
  for (int tb = 0; tb < kTB; ++tb) {
    float x[kKB][8], m = 0.f;
#pragma unroll
    for (int kb = 0; kb < kKB; ++kb)
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const float d = KeyLoad<KT>::at(raw.k[tb][kb], t) - raw.c[kb][t >> 2][t & 3];
        m = fmaxf(m, fabsf(d));  // NaN is passed over: its sums are NaN either way
        x[kb][t] = divide_by(d, s, rs);
      }
    m = max_xor<32>(max_xor<16>(m));
    const float2 s2 = row_scale(fabsf(divide_by(m, s, rs)));  // the largest |x|; NaN for an infinite m
    xinv[tb] = s2.y;
    bad |= s2.y == 0.f;
#pragma unroll
    for (int kb = 0; kb < kKB; ++kb) split8(x[kb], [&](float v) { return v * s2.x; }, xh[tb][kb], xl[tb][kb]);
  }
  return __any(bad);
}

// The sample's products.  acc[tb][j] = those of the wave's 16 kTB tokens (16 or 32,
// kTB of them a lane's column) with a split W tile in LDS:
// v_mfma_f32_16x16x32_f16, lane (i, q) feeding A[i][8 q + t] and B[8 q + t][i],
// t = 0..7, and holding D[4 q + r][i].  A is W (bucket rows), B is x (token
// columns), so lane (i, q) ends with buckets 16 j + 4 q + r of token i.
template <int kTB>
__device__ __forceinline__ void tile_products(const u32x4* ws, const half8 (&xh)[kTB][kKB], const half8 (&xl)[kTB][kKB],
                                              f32x4 (&acc)[kTB][kJ]) {
  const half8* wt = reinterpret_cast<const half8*>(ws) + (threadIdx.x & 63);
#pragma unroll
  for (int tb = 0; tb < kTB; ++tb)
#pragma unroll
    for (int j = 0; j < kJ; ++j) acc[tb][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kb = 0; kb < kKB; ++kb) {
    half8 wh[kJ], wl[kJ];
#pragma unroll
    for (int j = 0; j < kJ; ++j) {
      wh[j] = wt[((kb * 2 + 0) * kJ + j) * 64];
      wl[j] = wt[((kb * 2 + 1) * kJ + j) * 64];
    }
    // eight accumulators interleaved: no MFMA waits on the one before it
#pragma unroll
    for (int tb = 0; tb < kTB; ++tb)
#pragma unroll
      for (int j = 0; j < kJ; ++j)
        acc[tb][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wl[j], xh[tb][kb], acc[tb][j], 0, 0, 0);
#pragma unroll
    for (int tb = 0; tb < kTB; ++tb)
#pragma unroll
      for (int j = 0; j < kJ; ++j)
        acc[tb][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[j], xl[tb][kb], acc[tb][j], 0, 0, 0);
#pragma unroll
    for (int tb = 0; tb < kTB; ++tb)
#pragma unroll
      for (int j = 0; j < kJ; ++j)
        acc[tb][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[j], xh[tb][kb], acc[tb][j], 0, 0, 0);
  }
}

// A byte offset as a vector register, whatever it is the sum of.
__device__ __forceinline__ unsigned vector_offset(unsigned o) {
  asm("" : "+v"(o));
  return o;
}

// The lane's number, found again where it is rarely needed: what the compiler derives
// from it is then not kept in registers of a loop that has none to spare (a spilled
// word's reload awaits the activations' stores).
__device__ __forceinline__ int lane_again() {
  unsigned zero = 0u;
  asm volatile("" : "+s"(zero));
  return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, zero));
}

// The products of 16 tokens (`tok`, the lane's) with the buckets f0 .. f0 + 63 in
// fp32, for rows and buckets that the split does not serve: v_mfma_f32_16x16x4f32
// (lane (i, q) feeding A[i][q] and B[q][i], and holding D[4 q + r][i]), four dims
// 16 kb + 4 q .. of its row per block.  Straight from memory: W comes from L2 for
// each 16 tokens, 32 KB per wave against 128 MFMAs of 32 cycles, which the MFMAs
// still bound.  (One fp32 chain per lane and value: a 64-token append whose tile
// held one infinite key took 822 us, and 63 without it.)
template <typename KT>
__device__ __forceinline__ void fp32_products(const UpdateArgs& a, int g, int tok, int f0, f32x4 (&acc)[kJ]) {
  const int l = lane_again(), li = l & 15, lq = l >> 4;
  // (as buffers: one offset register each, and zeros for buckets past F)
  const __amdgpu_buffer_rsrc_t kr = raw_buffer(static_cast<const KT*>(a.k) + (size_t)g * a.ks + (size_t)a.H * kD,
                                               a.N * kD * (int)sizeof(KT));
  const __amdgpu_buffer_rsrc_t cr = raw_buffer(a.center + (size_t)g * kD, kD * (int)sizeof(float));
  const __amdgpu_buffer_rsrc_t wr = raw_buffer(a.W + (size_t)g * kF * kD, kF * kD * (int)sizeof(float));
  const unsigned ko = ((unsigned)tok * kD + 4 * lq) * (unsigned)sizeof(KT);
  const unsigned co = 4 * lq * (unsigned)sizeof(float), wo = ((unsigned)(f0 + li) * kD + 4 * lq) * (unsigned)sizeof(float);
  const float s = a.scale[g];
#pragma unroll
  for (int j = 0; j < kJ; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int e = 0; e < kD / 8; ++e) {  // two of the block's four dims at a time
    const int d = 16 * (e >> 1) + 2 * (e & 1);
    f32x2 wv[kJ];
#pragma unroll
    for (int j = 0; j < kJ; ++j) wv[j] = load_f2(wr, wo, (16 * j * kD + d) * (int)sizeof(float));
    const f32x2 m = load_f2(cr, co, d * (int)sizeof(float));
    const typename KeyLoad<KT>::Raw2 r = KeyLoad<KT>::load2(kr, ko, d * (int)sizeof(KT));
    const float x[2] = {(KeyLoad<KT>::lo(r) - m[0]) / s, (KeyLoad<KT>::hi(r) - m[1]) / s};
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < kJ; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[j][t], x[t], acc[j], 0, 0, 0);
  }
}

// fp32_products with the tile's W in the wave's registers, as f32x4 words: w[e][j]
// is lane (i, q)'s dims 16 e + 4 q .. + 3 of bucket 16 j + i.  The same products in
// the same order.
template <typename KT>
__device__ __forceinline__ void fp32_products(const UpdateArgs& a, int g, int tok, const half8 (&w)[kD / 16][kJ],
                                              f32x4 (&acc)[kJ]) {
  const int lq = (threadIdx.x >> 4) & 3;
  const __amdgpu_buffer_rsrc_t kr = raw_buffer(static_cast<const KT*>(a.k) + (size_t)g * a.ks + (size_t)a.H * kD,
                                               a.N * kD * (int)sizeof(KT));
  const __amdgpu_buffer_rsrc_t cr = raw_buffer(a.center + (size_t)g * kD, kD * (int)sizeof(float));
  const unsigned ko = ((unsigned)tok * kD + 4 * lq) * (unsigned)sizeof(KT), co = 4 * lq * (unsigned)sizeof(float);
  const float s = a.scale[g];
#pragma unroll
  for (int j = 0; j < kJ; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int e = 0; e < kD / 8; ++e) {  // two of the block's four dims at a time
    const int d = 16 * (e >> 1) + 2 * (e & 1);
    const f32x2 m = load_f2(cr, co, d * (int)sizeof(float));
    const typename KeyLoad<KT>::Raw2 r = KeyLoad<KT>::load2(kr, ko, d * (int)sizeof(KT));
    const float x[2] = {(KeyLoad<KT>::lo(r) - m[0]) / s, (KeyLoad<KT>::hi(r) - m[1]) / s};
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < kJ; ++j) {
        const f32x4 wv = __builtin_bit_cast(f32x4, w[e >> 1][j]);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[2 * (e & 1) + t], x[t], acc[j], 0, 0, 0);
      }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The sample's values of one bucket tile for the wave's 16 kTB tokens, after the products
// (made again in fp32 where a row or bucket is not split): four(tb, j, v) gets
// lane (i, q)'s pre-relu sums of buckets 16 j + 4 q .. + 3.  `tok` is the lane's
// kTB tokens; sg the tile's biases, then its inverse bucket scales.
template <typename KT, int kTB, typename Four>
__device__ __forceinline__ void tile_values(const UpdateArgs& a, int g, int f0, const int (&tok)[kTB],
                                            const float (&xinv)[kTB], bool bad_rows, const float* sg,
                                            f32x4 (&acc)[kTB][kJ], Four four) {
  const int lq = (threadIdx.x >> 4) & 3;
  float4 bias[kJ], winv[kJ];
  bool bad = bad_rows;
#pragma unroll
  for (int j = 0; j < kJ; ++j) {
    const int o = 16 * j + 4 * lq;
    bias[j] = *reinterpret_cast<const float4*>(sg + o);
    winv[j] = *reinterpret_cast<const float4*>(sg + kFT + o);
    bad |= winv[j].x == 0.f || winv[j].y == 0.f || winv[j].z == 0.f || winv[j].w == 0.f;
  }
  bad = __any(bad);
#pragma unroll
  for (int tb = 0; tb < kTB; ++tb) {
    if (bad) fp32_products<KT>(a, g, tok[tb], f0, acc[tb]);  // uniform
#pragma unroll
    for (int j = 0; j < kJ; ++j) {
      const float b4[4] = {bias[j].x, bias[j].y, bias[j].z, bias[j].w};
      const float s4[4] = {winv[j].x, winv[j].y, winv[j].z, winv[j].w};
      float v[4];
      // the scales are powers of two: one rounding, that of the sum with the bias
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = bad ? acc[tb][j][r] + b4[r] : fmaf(acc[tb][j][r] * xinv[tb], s4[r], b4[r]);
      four(tb, j, v);
    }
  }
}

// Token of sample row r of S (a.N tokens): one of each N / S consecutive ones,
// at a place that r decides, so that no period of the text meets the sample's.
__device__ __forceinline__ int sample_token(int r, int S, int N) {
  if (S == N) return r;
  const unsigned step = (unsigned)N / (unsigned)S;
  return (int)((long long)r * N / S) + (int)((((unsigned)r * 0x9E3779B9u) >> 8) % step);
}

// Where the histogram keeps a bin: 37 words from its neighbour's, so that the
// bins of an octave, which every workgroup adds to, lie in lines of their own
// (the atomics of a line are serial); and the inverse of 37 mod 8192.
constexpr unsigned kPlace = 37u, kPlaceInverse = 7085u;
static_assert((kPlace * kPlaceInverse) % kSampleBins == 1u, "inverse places");
__device__ __forceinline__ unsigned sample_place(unsigned bin) { return bin * kPlace % kSampleBins; }

// ---------------------------------------------------------------------------
// sample: grid (max(ceil(S / (128 kTB)), 1), kFTiles, G) x 512.  Splits bucket tile
// ft of W (the first token tile's workgroups write it for the encode), and adds
// to the group's histogram, for each of S sample tokens and each 16 buckets of
// the tile (a lane's), the largest activation if it is positive.  Around tau a
// token's 16 buckets hold 0.04 values, so that counts all but 4% of them; a
// token that outweighs the others (a hundred times the memberships) counts
// for 188 at most, and the floor stays one that serves the others.  S = 0 only
// splits.
// ---------------------------------------------------------------------------
template <typename KT, int kTB>
__global__ __launch_bounds__(kET) void sample_kernel(UpdateArgs a, int S) {
  const int y = blockIdx.x, ft = blockIdx.y, g = blockIdx.z, tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  __shared__ __align__(16) u32x4 ws[kWRows];
  __shared__ __align__(16) unsigned hist[kSampleBins];
  const int r0 = y * kSampleFew * kTB + w * 16 * kTB;  // the wave's first sample row
  const bool live = r0 < S;                      // uniform per wave
  int tok[kTB];
  RowsRaw<KT, kTB> raw;
  if (live) {
#pragma unroll
    for (int tb = 0; tb < kTB; ++tb) tok[tb] = sample_token(min(r0 + 16 * tb + (lane & 15), S - 1), S, a.N);
    raw.load(a, g, tok);
  }
  if (w < kJ) {  // wave j splits the tile's column j
    const int f = ft * kFT + 16 * w + (lane & 15);
    float x[kKB][8], m = 0.f;
#pragma unroll
    for (int kb = 0; kb < kKB; ++kb) {
      float4 u = make_float4(0.f, 0.f, 0.f, 0.f), v = u;
      if (f < kF) {
        const float4* row = reinterpret_cast<const float4*>(a.W + ((size_t)g * kF + f) * kD + 32 * kb + 8 * (lane >> 4));
        u = row[0];
        v = row[1];
      }
      x[kb][0] = u.x; x[kb][1] = u.y; x[kb][2] = u.z; x[kb][3] = u.w;
      x[kb][4] = v.x; x[kb][5] = v.y; x[kb][6] = v.z; x[kb][7] = v.w;
#pragma unroll
      for (int t = 0; t < 8; ++t) m = fmaxf(m, fabsf(x[kb][t]));
    }
    m = max_xor<32>(max_xor<16>(m));
    const float2 sc = row_scale(m);
    // (the sample itself, which only places the floor, uses any split there is)
    const bool enough = enough_dims<16>(reinterpret_cast<const float (&)[kKB * 8]>(x), m);
    half8* lds = reinterpret_cast<half8*>(ws) + lane;
    half8* out = reinterpret_cast<half8*>(a.wsplit + ((size_t)g * kFTiles + ft) * kWTile) + lane;
#pragma unroll
    for (int kb = 0; kb < kKB; ++kb) {
      half8 hi, lo;
      split8(x[kb], [&](float v) { return v * sc.x; }, hi, lo);
      lds[((kb * 2 + 0) * kJ + w) * 64] = hi;
      lds[((kb * 2 + 1) * kJ + w) * 64] = lo;
      if (y == 0) {
        out[((kb * 2 + 0) * kJ + w) * 64] = hi;
        out[((kb * 2 + 1) * kJ + w) * 64] = lo;
      }
    }
    if (lane < 16) {
      float* tail = reinterpret_cast<float*>(ws + kET * kWLoads) + 16 * w + lane;
      tail[0] = f < kF ? a.b[(size_t)g * kF + f] : 0.f;
      tail[kFT] = sc.y;
      if (y == 0) {
        float* t = reinterpret_cast<float*>(a.wsplit + ((size_t)g * kFTiles + ft) * kWTile + kFT * kD * 2) + 16 * w + lane;
        t[0] = tail[0];
        t[kFT] = enough ? sc.y : 0.f;
      }
    }
  }
  if (y == 0 && ft == 0 && tid == 0) {
    a.ctl[(size_t)g * kCtl + kListLen] = 0u;
    a.ctl[(size_t)g * kCtl + kTieLen] = 0u;
    a.ctl[(size_t)g * kCtl + kArrived] = 0u;
  }
  if (S == 0) return;  // uniform
  for (int i = tid; i < kSampleBins; i += kET) hist[i] = 0u;
  half8 xh[kTB][kKB], xl[kTB][kKB];
  float xinv[kTB];
  bool bad_rows = false;
  if (live) bad_rows = split_rows<KT, kTB>(raw, xh, xl, xinv);
  __syncthreads();
  if (live) {
    f32x4 acc[kTB][kJ];
    tile_products(ws, xh, xl, acc);
    float most[kTB];
#pragma unroll
    for (int tb = 0; tb < kTB; ++tb) most[tb] = 0.f;
    tile_values<KT, kTB>(a, g, ft * kFT, tok, xinv, bad_rows, reinterpret_cast<const float*>(ws + kET * kWLoads), acc,
                    [&](int tb, int j, const float (&v)[4]) {
      most[tb] = fmaxf(most[tb], fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])));
    });
#pragma unroll
    for (int tb = 0; tb < kTB; ++tb)
      if (r0 + 16 * tb + (lane & 15) < S && most[tb] > 0.f)
        atomicAdd(&hist[__float_as_uint(most[tb]) >> kSampleShift], 1u);
  }
  __syncthreads();
  unsigned* sh = a.sample + (size_t)g * kSampleBins;
#pragma unroll
  for (int u = 0; u < kSampleBins / 4 / kET; ++u) {
    const int i = 4 * (tid + kET * u);
    const u32x4 c = *reinterpret_cast<const u32x4*>(&hist[i]);
    if (c[0] | c[1] | c[2] | c[3]) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c[e]) atomicAdd(&sh[sample_place(i + e)], c[e]);
    }
  }
}

// ---------------------------------------------------------------------------
// encode: grid (G, 6, R) x 512.  Workgroup (g, part, y) takes range y of the
// group's tokens, whole 16-token steps, and wave w the bucket tile 8 part + w,
// whose split W it holds in registers (128 of them) from start to end; the 47
// tiles leave the last part's last wave to the splitting only.  The keys go
// through LDS: 64 tokens at a time (a stage) are loaded, made x = (k - center) /
// key_scale, split and written as MFMA operands, double-buffered, and every wave
// multiplies the stage's four steps by its tile.  A group's workgroups lie 8
// blocks apart, with 8 groups on one XCD, whose L2 then holds that group's W.
//
// The other way round (x in registers, W tiles streamed through LDS, a barrier
// per tile) every wave read 32 KB of LDS per 96 MFMAs; here it is 16 KB, a
// barrier per 192, and no load of the loop but the next stage's rows.  1024 /
// 4096 keys with the activations stored: 38 / 121 us then, 37 / 113 now; 65536
// without: 1.33 ms, now 1.18 (2.07 GHz under this load, 1.03 PFLOP/s; the
// products alone took 0.90 ms, and a large f16 library product runs at 1.2).
// Neither a higher priority for some of the waves nor the epilogue's values
// placed one by one between the next step's products changed that.
//
// kCollect: the values at or above the group's floor, the lower edge of the
// sample histogram's bin that holds the target-th largest value, go to the
// candidate list: each wave gathers its own in LDS (places from a ballot, no
// atomics) and moves them to a range of the list that it reserves with one
// atomic; the workgroup's rest goes out together at the end.  An LDS histogram
// of every positive value instead took longer than the products.
// kStore: every activation is written, one 16-byte store per lane and column.
// Without kCollect the kernel is the dense path of a call that collects no
// candidates, or whose list turned out unusable (else it returns at once).
// ---------------------------------------------------------------------------
constexpr int kEW = kET / 64;                           // waves, a bucket tile each
constexpr int kEParts = (kFTiles + kEW - 1) / kEW;      // 6
constexpr int kStage = 64;                              // tokens split at a time
constexpr int kSteps = kStage / 16;
constexpr int kWaveBuf = 512;  // candidates a wave gathers

template <typename KT, bool kStore, bool kCollect>
__global__ __launch_bounds__(kET) void encode_kernel(UpdateArgs a) {
  const int g = blockIdx.x, part = blockIdx.y, y = blockIdx.z, ranges = gridDim.z, tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 15, lq = lane >> 4;
  __shared__ __align__(16) half8 xs[2][kSteps * kKB * 2 * 64];  // [buffer][step][dim block][hi, lo][lane]
  __shared__ __align__(16) float xinv[2][kStage];               // inverse scales; 0: a row that is not split
  __shared__ __align__(16) float center[kD];
  __shared__ uint2 cand[kCollect ? kEW : 1][kCollect ? kWaveBuf + 64 : 1];  // the wave's, and a dump per lane
  __shared__ unsigned fine[kCollect ? kBins : 1];  // the candidates' fine digits
  __shared__ unsigned wsum[kEW], floor_s, base_s;
  unsigned* ctl = a.ctl + (size_t)g * kCtl;
  if constexpr (!kCollect)
    if (list_ok(a, g)) return;  // uniform
  // the workgroup's tokens, the wave's bucket tile
  const int blocks = (a.N + 15) / 16;
  const int t0 = 16 * (int)((long long)blocks * y / ranges), t1 = min(a.N, 16 * (int)((long long)blocks * (y + 1) / ranges));
  const int ft = part * kEW + w, f0 = ft * kFT + 4 * lq;
  const bool live = ft < kFTiles;  // uniform per wave: the last part's last wave only splits rows
  // rows of a stage: thread (row 8 w + l % 8, dims 16 (l / 8) .. + 15)
  const KT* kg = static_cast<const KT*>(a.k) + (size_t)g * a.ks;
  const float scale = a.scale[g], rscale = 1.0f / scale;
  // (the scale's own range bounds what divide_by may meet)
  const bool scaled = fabsf(scale) >= 0x1p-60f && fabsf(scale) <= 0x1p60f;
  typename KeyLoad<KT>::Raw8 raw[2];
  auto load_rows = [&](int t) {
    const int l = lane_again(), sr = 8 * w + (l & 7), sp = l >> 3;
    const KT* p = kg + (size_t)(a.H + min(t + sr, a.N - 1)) * kD + 16 * sp;
    raw[0] = KeyLoad<KT>::raw8(p);
    raw[1] = KeyLoad<KT>::raw8(p + 8);
  };
  auto split_rows = [&](int buf) {
    const int l = lane_again(), sr = 8 * w + (l & 7), sp = l >> 3;
    float x[2][8], m = 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x4 c0 = *reinterpret_cast<const f32x4*>(center + 16 * sp + 8 * h);
      const f32x4 c1 = *reinterpret_cast<const f32x4*>(center + 16 * sp + 8 * h + 4);
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        x[h][t] = KeyLoad<KT>::at(raw[h], t) - (t < 4 ? c0[t & 3] : c1[t & 3]);
        m = fmaxf(m, fabsf(x[h][t]));  // NaN is passed over: its sums are NaN either way
      }
    }
    m = max_xor<32>(max_xor<16>(max_xor<8>(m)));
    const float2 s2 = row_scale(fabsf(divide_by(m, scale, rscale)));  // the largest |x|; NaN for an infinite m
    const bool enough = enough_dims<8>(reinterpret_cast<const float (&)[16]>(x), m);
    // (d / s) times the row's power of two: the quotient and its remainder scale exactly
    const float rs = rscale * s2.x, ss = scale * s2.y;
    half8* out = &xs[buf][((sr >> 4) * kKB + (sp >> 1)) * 2 * 64 + (2 * (sp & 1)) * 16 + (sr & 15)];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      half8 hi, lo;
      split8(x[h], [&](float d) { return divide_by(d, ss, rs); }, hi, lo);
      out[16 * h] = hi;
      out[64 + 16 * h] = lo;
    }
    // (a quotient's remainder stays in the normal range)
    if (sp == 0) xinv[buf][sr] = scaled && enough && fabsf(ss) >= 0x1p-100f ? s2.y : 0.f;
  };
  load_rows(t0);
  if (tid < kD) center[tid] = a.center[(size_t)g * kD + tid];
  const _Float16* wt = a.wsplit + ((size_t)g * kFTiles + min(ft, kFTiles - 1)) * kWTile;
  // The tile's W, split ([2 kb + hi, lo][column]), or in fp32 (fp32_products).
  static_assert(2 * kKB == kD / 16, "both forms take 128 registers");
  half8 wf[2 * kKB][kJ];
#pragma unroll
  for (int e = 0; e < 2 * kKB; ++e)
#pragma unroll
    for (int j = 0; j < kJ; ++j) wf[e][j] = reinterpret_cast<const half8*>(wt)[(e * kJ + j) * 64 + lane];
  f32x4 bias[kJ], winv[kJ];
  bool bad_w = false;
#pragma unroll
  for (int j = 0; j < kJ; ++j) {
    const float* tail = reinterpret_cast<const float*>(wt + kFT * kD * 2) + 16 * j + 4 * lq;
    bias[j] = *reinterpret_cast<const f32x4*>(tail);
    winv[j] = *reinterpret_cast<const f32x4*>(tail + kFT);
#pragma unroll
    for (int r = 0; r < 4; ++r) bad_w |= winv[j][r] == 0.f;
  }
  bad_w = __any(bad_w);
  float least = 0.f;  // the floor
  if constexpr (kCollect) {
    // every workgroup reads the same histogram and puts its bins in order, in
    // the buffer of the second stage; then thread t has the 16 bins below 8192 - 16 t
    constexpr int kPer = kSampleBins / kET;
    static_assert(kSampleBins * sizeof(unsigned) <= sizeof(xs[1]), "room for the histogram");
    const uint4* sh = reinterpret_cast<const uint4*>(a.sample + (size_t)g * kSampleBins);
    unsigned* ordered = reinterpret_cast<unsigned*>(xs[1]);
    uint4 h[kPer / 4];
#pragma unroll
    for (int u = 0; u < kPer / 4; ++u) h[u] = sh[tid + kET * u];
#pragma unroll
    for (int u = 0; u < kPer / 4; ++u) {
      const unsigned at = 4u * (unsigned)(tid + kET * u);
      ordered[at * kPlaceInverse % kSampleBins] = h[u].x;
      ordered[(at + 1u) * kPlaceInverse % kSampleBins] = h[u].y;
      ordered[(at + 2u) * kPlaceInverse % kSampleBins] = h[u].z;
      ordered[(at + 3u) * kPlaceInverse % kSampleBins] = h[u].w;
    }
    __syncthreads();
    unsigned c[kPer], tot = 0u;
#pragma unroll
    for (int u = 0; u < kPer / 4; ++u) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(&ordered[kSampleBins - kPer * (tid + 1) + 4 * u]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        c[4 * u + i] = v[i];
        tot += v[i];
      }
    }
    if (tid == 0) floor_s = 1u;  // too few positive values in the sample: every one is collected
    for (int i = tid; i < kBins; i += kET) fine[i] = 0u;
    unsigned run = block_incl_scan<kET>(tot, wsum) - tot;
    if (run < a.target && run + tot >= a.target) {
#pragma unroll
      for (int u = kPer - 1; u >= 0; --u) {
        if (run < a.target && run + c[u] >= a.target)
          floor_s = max(1u, (unsigned)(kSampleBins - kPer * (tid + 1) + u) << kSampleShift);
        run += c[u];
      }
    }
    __syncthreads();
    if (y == 0 && part == 0 && tid == 0) ctl[kFloor] = floor_s;
    least = __uint_as_float(floor_s);
  } else {
    __syncthreads();
  }
  split_rows(0);
  __syncthreads();
  // fp32 products throughout, W in registers, for a tile with a bucket that is not
  // split, and where half of the first stage's steps have a row that is not; a lone
  // such step takes its W from L2 (the build of 65536 keys with an encoder of 6 of 128
  // weights: 15.4 ms with every step's W from there, 6.4 from registers)
  const unsigned long long odd = __ballot(xinv[0][lane] == 0.f);
  const int odd_steps = (int)((odd & 0xffffull) != 0) + (int)((odd >> 16 & 0xffffull) != 0) +
                        (int)((odd >> 32 & 0xffffull) != 0) + (int)(odd >> 48 != 0);
  const bool whole = __builtin_amdgcn_readfirstlane(bad_w || odd_steps >= 2 ? 1 : 0) != 0;  // uniform, as a scalar
  if (__builtin_expect(whole, 0)) {
    const __amdgpu_buffer_rsrc_t wr = raw_buffer(a.W + (size_t)g * kF * kD, kF * kD * (int)sizeof(float));  // 0 past F
    const unsigned o = ((unsigned)(ft * kFT + li) * kD + 4 * lq) * (unsigned)sizeof(float);
#pragma unroll
    for (int e = 0; e < kD / 16; ++e)
#pragma unroll
      for (int j = 0; j < kJ; ++j)
        wf[e][j] = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(
            wr, o, (16 * j * kD + 16 * e) * (int)sizeof(float), 0));
  }
  // W is awaited here: left pending into the loop, its first use there waited in every
  // step for the stores of the step before
#pragma unroll
  for (int e = 0; e < 2 * kKB; ++e)
#pragma unroll
    for (int j = 0; j < kJ; ++j) asm volatile("" ::"v"(wf[e][j]));
#pragma unroll
  for (int j = 0; j < kJ; ++j) asm volatile("" ::"v"(bias[j]), "v"(winv[j]));
  uint2* list = a.list + (size_t)g * a.list_cap;
  unsigned n = 0u;  // the wave's gathered candidates (uniform)
  auto put = [&](unsigned at, unsigned i) {
    const uint2 e = cand[kCollect ? w : 0][i];
    if (at + i < a.list_cap) list[at + i] = e;
    if (a.fine) atomicAdd(&fine[kCollect ? fine_digit(e.y, floor_s) : 0u], 1u);
  };
  auto place = [&](unsigned long long m) {
    return n + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
  };
  auto gather = [&](bool in, unsigned flat, float v) {
    const unsigned long long m = __ballot(in);
    if (m) {  // uniform
      if (in) cand[kCollect ? w : 0][place(m)] = make_uint2(flat, __float_as_uint(v));
      n += (unsigned)__popcll(m);
    }
  };
  int collect_to = t1;  // the first token of which nothing is collected (uniform)
  auto flush = [&]() {
    if (n <= kWaveBuf - 256) return;  // uniform
    __builtin_amdgcn_wave_barrier();
    unsigned at = 0u;
    if (lane == 0) at = atomicAdd(&ctl[kListLen], n);
    at = (unsigned)__builtin_amdgcn_readfirstlane((int)at);
    if (at >= a.list_cap) collect_to = 0;  // the list overflowed and is of no use: no more of it
    for (unsigned i = lane; i < n; i += 64) put(at, i);
    __builtin_amdgcn_wave_barrier();
    n = 0u;
  };
  const unsigned flat0 = (unsigned)li * kF + (unsigned)f0;
  // The lane's offsets in a step's rows; 2^31 is outside.  The step's own part is
  // added to them, by vector_offset where the compiler can't take it apart again, and
  // not given as the instruction's scalar offset: four-word stores with one lost their
  // last word to the vector instruction that followed, which the compiler takes to
  // need no wait.
  static_assert(kF - (kFTiles - 1) * kFT > 16 * (kJ - 1) && kF % 4 == 0, "of the last tile only the last column ends early");
  const unsigned column = flat0 * (unsigned)sizeof(float);
  const unsigned last_column = f0 + 16 * (kJ - 1) < kF ? column + 64u * (kJ - 1) : 1u << 31;
  int buf = 0;
  auto tokens = [&](auto in_fp32) {
    constexpr bool kWhole = decltype(in_fp32)::value;
    for (int t = t0; t < t1; t += kStage) {  // uniform
      const bool more = t + kStage < t1;
      if (more) load_rows(t + kStage);  // in flight while this stage is multiplied
      // the stage's activation rows; stores past them (rows past the block, buckets
      // past F) carry an offset outside the resource and are dropped
      const __amdgpu_buffer_rsrc_t ar = raw_buffer(a.act + ((size_t)g * a.N + t) * kF,
                                                   kStore ? min(kStage, t1 - t) * kF * (int)sizeof(float) : 0);
      if (live) {
#pragma unroll 1
        for (int s = 0; s < kSteps && t + 16 * s < t1; ++s) {  // uniform
          const int tok = t + 16 * s + li;
          const half8* x = &xs[buf][s * kKB * 2 * 64 + lane];
          half8 xh = x[0], xl = x[64];
          const float inv = xinv[buf][16 * s + li];
          f32x4 acc[kJ];
          if constexpr (!kWhole) {
#pragma unroll
            for (int j = 0; j < kJ; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kb = 0; kb < kKB; ++kb) {
              // the next dim block's rows are requested before this one's products
              const half8 yh = x[(kb + 1) % kKB * 2 * 64], yl = x[((kb + 1) % kKB * 2 + 1) * 64];
              __builtin_amdgcn_sched_barrier(0);
#pragma unroll
              for (int j = 0; j < kJ; ++j)
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[2 * kb + 1][j], xh, acc[j], 0, 0, 0);
#pragma unroll
              for (int j = 0; j < kJ; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[2 * kb][j], xl, acc[j], 0, 0, 0);
#pragma unroll
              for (int j = 0; j < kJ; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[2 * kb][j], xh, acc[j], 0, 0, 0);
              __builtin_amdgcn_sched_barrier(0);
              xh = yh;
              xl = yl;
            }
          } else {
            fp32_products<KT>(a, g, min(tok, a.N - 1), wf, acc);
          }
          const unsigned flat = flat0 + (unsigned)(t + 16 * s) * kF;
          if (kWhole || __builtin_expect(__any(inv == 0.f), 0)) {  // uniform
            if constexpr (!kWhole) fp32_products<KT>(a, g, min(tok, a.N - 1), ft * kFT, acc);
#pragma unroll
            for (int j = 0; j < kJ; ++j) acc[j] += bias[j];
          } else {
            // the scales are powers of two: one rounding, that of the sum with the bias
#pragma unroll
            for (int j = 0; j < kJ; ++j)
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[j][r] = fmaf(acc[j][r] * inv, winv[j][r], bias[j][r]);
          }
          const unsigned at_step = 16u * s * kF * (unsigned)sizeof(float);
          float most = -INFINITY;
          unsigned hits = 0u;
          // NaN (nothing is collected) for rows past the range; a bucket past F has a
          // zero row and bias: its 0 is below every floor
          const float from = tok < collect_to ? least : __builtin_nanf("");
#pragma unroll
          for (int j = 0; j < kJ; ++j) {
            u32x4 p;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float v = acc[j][r];
              p[r] = __float_as_uint(v > 0.f ? v : 0.f);  // relu; NaN is not positive
              // hits = 2 hits + (v >= from), in two instructions
              if constexpr (kCollect)
                asm("v_cmp_ge_f32_e32 vcc, %1, %2\n\tv_addc_co_u32_e32 %0, vcc, %0, %0, vcc" : "+v"(hits) : "v"(v), "v"(from) : "vcc");
              most = fmaxf(most, v);
            }
            if constexpr (kStore)
              __builtin_amdgcn_raw_buffer_store_b128(
                  p, ar, j < kJ - 1 ? vector_offset(column + at_step) + 64u * j : vector_offset(last_column + at_step), 0, 0);
          }
          if constexpr (kCollect) {
            // a lane's one candidate is its largest value
            const bool one = hits != 0u && (hits & (hits - 1u)) == 0u;
            const unsigned long long m = __ballot(one);
            const unsigned e = (unsigned)__clz((int)hits) & 15u;  // bit 15 is the first value
            cand[w][one ? place(m) : kWaveBuf + lane] = make_uint2(flat + 4u * (e & 12u) + (e & 3u), __float_as_uint(most));
            n += (unsigned)__popcll(m);
            const bool several = hits != 0u && !one;
            if (__any(several)) {  // uniform
#pragma unroll
              for (int j = 0; j < kJ; ++j) {
                flush();
#pragma unroll
                for (int r = 0; r < 4; ++r)
                  gather(several && (hits >> (15 - 4 * j - r) & 1u), flat + (unsigned)(16 * j + r), acc[j][r]);
              }
            }
            flush();
          }
        }
      }
      if (more) {
        split_rows(buf ^ 1);  // last read before the previous barrier
        __syncthreads();
        buf ^= 1;
      }
    }
  };
  if (__builtin_expect(whole, 0))
    tokens(std::true_type{});
  else
    tokens(std::false_type{});
  if constexpr (kCollect) {  // the rest of the 8 waves, one reservation
    __syncthreads();
    if (lane == 0) wsum[w] = n;
    __syncthreads();
    if (tid == 0) {
      unsigned total = 0u;
      for (int i = 0; i < kEW; ++i) total += wsum[i];
      base_s = total ? atomicAdd(&ctl[kListLen], total) : 0u;
    }
    __syncthreads();
    unsigned at = base_s;
    for (int i = 0; i < w; ++i) at += wsum[i];
    for (unsigned i = lane; i < n; i += 64) put(at, i);
    if (a.fine) {  // uniform
      __syncthreads();
      unsigned* hg = hist_of(a, g, 0);
      for (int i = tid; i < kBins; i += kET)
        if (fine[i]) atomicAdd(&hg[i], fine[i]);
    }
  }
}

// ---------------------------------------------------------------------------
// digit: grid G x 256.  Level L consumes hist level L (all replicas, then
// zeroes them for the next update) and narrows the threshold prefix.
// Level widths: 11 bits (30..20), 11 bits (19..9), 9 bits (8..0); positive
// floats order like their bit patterns, so the prefix after level 2 is the
// exact bit pattern of tau, the budget-th largest value.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kUT) void digit_kernel(UpdateArgs a, int level) {
  const int g = blockIdx.x, tid = threadIdx.x;
  __shared__ unsigned wsum[kUT / 64];
  __shared__ unsigned found_digit, found_rem, found_ties;
  unsigned* ctl = a.ctl + (size_t)g * kCtl;
  unsigned* h = hist_of(a, g, level);
  constexpr int kPer = kBins / kUT;  // 8 bins per thread, descending digits
  unsigned c[kPer], tot = 0;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int d = kBins - 1 - (tid * kPer + u);
    unsigned s = 0;
#pragma unroll
    for (int r = 0; r < kRep; ++r) {
      s += h[r * kBins + d];
      h[r * kBins + d] = 0;
    }
    c[u] = s;
    tot += s;
  }
  if (level == 0 && a.listed)
    for (int i = tid; i < kSampleBins; i += kUT) a.sample[(size_t)g * kSampleBins + i] = 0u;
  const unsigned count = budget_of(a);
  const unsigned incl = block_incl_scan<kUT>(tot, wsum);
  unsigned rem, prefix_in;
  if (level == 0) {
    // wsum holds the per-wave totals: their sum is the number of positive values
    const unsigned npos = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    if (npos < count || count == 0) {
      // fewer positives than the budget: tau = 0 and every positive value is
      // kept (core.py:22-26); an empty budget keeps nothing
      if (tid == 0) {
        ctl[kMode] = count == 0 ? kModeTopK : kModeAllPositive;
        ctl[kPrefix] = 0;
        ctl[kRem] = 0;
        ctl[kTau] = count == 0 ? 0x7f800000u : 0u;
        ctl[kNeed] = 0;
        ctl[kTies] = 0;
        ctl[kOrdered] = 0;
        ctl[kCut] = 0;
        ctl[kCount] = count;
      }
      return;
    }
    rem = count;
    prefix_in = 0;
  } else {
    if (ctl[kMode] != kModeTopK || ctl[kTau] == 0x7f800000u) return;
    rem = ctl[kRem];
    prefix_in = ctl[kPrefix];
  }
  const int width = level < 2 ? 11 : 9;
  unsigned run = incl - tot;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int d = kBins - 1 - (tid * kPer + u);
    if (d < (1 << width) && run < rem && run + c[u] >= rem) {
      found_digit = (unsigned)d;
      found_rem = rem - run;
      found_ties = c[u];
    }
    run += c[u];
  }
  __syncthreads();
  if (tid == 0) {
    const unsigned prefix = (prefix_in << width) | found_digit;
    ctl[kMode] = kModeTopK;
    ctl[kPrefix] = prefix;
    ctl[kRem] = found_rem;
    ctl[kCount] = count;
    if (level == kLevels - 1) {
      // prefix is the exact tau; found_rem of its found_ties ties are taken
      ctl[kTau] = prefix;
      ctl[kNeed] = found_rem;
      ctl[kTies] = found_ties;
      ctl[kOrdered] = found_ties > found_rem;
      ctl[kCut] = ~0u;  // every tie is taken, unless the tie kernels find the last one
      ctl[kTieLen] = 0u;
    } else {
      ctl[kTau] = 0;
    }
  }
}

// The values a pass over a group reads: its candidate list (listed), or the
// dense activations.  fn(value bits, flat index) is called for each, by NT
// threads of `blocks` workgroups, kU loads in flight per thread.
template <int NT, typename Fn>
__device__ __forceinline__ void each_value(const UpdateArgs& a, int g, bool listed, int block, int blocks, Fn fn) {
  constexpr int kU = 8;
  if (listed) {
    const uint2* list = a.list + (size_t)g * a.list_cap;
    const unsigned len = a.ctl[(size_t)g * kCtl + kListLen], step = (unsigned)(NT * blocks);
    for (unsigned i0 = (unsigned)(block * NT) + threadIdx.x; i0 < len; i0 += kU * step) {
      uint2 e[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) e[u] = list[i0 + u * step < len ? i0 + u * step : i0];
#pragma unroll
      for (int u = 0; u < kU; ++u)
        if (i0 + u * step < len) fn(e[u].y, e[u].x);
    }
  } else {
    const size_t n4 = (size_t)a.N * kF / 4, step = (size_t)NT * blocks;
    const float4* ag = reinterpret_cast<const float4*>(a.act + (size_t)g * a.N * kF);
    for (size_t i0 = (size_t)block * NT + threadIdx.x; i0 < n4; i0 += kU * step) {
      float4 v[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) v[u] = ag[i0 + u * step < n4 ? i0 + u * step : i0];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const size_t i = i0 + u * step;
        if (i >= n4) break;
        const float vv[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (vv[j] > 0.f) fn(__float_as_uint(vv[j]), (unsigned)(4 * i + j));
      }
    }
  }
}

// ---------------------------------------------------------------------------
// hist0 / refine: grid (kRefineBlocks, G) x 256; histogram of the first digit
// of the positive values, and of the next digit of those whose higher bits
// equal the prefix.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void level_hist(const UpdateArgs& a, int level, int shift_hi, unsigned prefix, int shift,
                                           unsigned dmask) {
  const int g = blockIdx.y, tid = threadIdx.x;
  __shared__ unsigned hist[kBins];
  for (int i = tid; i < kBins; i += kUT) hist[i] = 0;
  __syncthreads();
  each_value<kUT>(a, g, list_ok(a, g), blockIdx.x, gridDim.x, [&](unsigned u, unsigned) {
    if ((u >> shift_hi) == prefix) atomicAdd(&hist[(u >> shift) & dmask], 1u);
  });
  __syncthreads();
  unsigned* hg = hist_of(a, g, level) + (blockIdx.x % kRep) * kBins;
  for (int i = tid; i < kBins; i += kUT)
    if (hist[i]) atomicAdd(&hg[i], hist[i]);
}

__global__ __launch_bounds__(kUT) void hist0_kernel(UpdateArgs a) { level_hist(a, 0, 31, 0u, 20, 0x7ffu); }

__global__ __launch_bounds__(kUT) void refine_kernel(UpdateArgs a, int level) {
  const unsigned* ctl = a.ctl + (size_t)blockIdx.y * kCtl;
  if (ctl[kMode] != kModeTopK || ctl[kTau] == 0x7f800000u) return;
  level_hist(a, level, level == 1 ? 20 : 9, ctl[kPrefix], level == 1 ? 9 : 0, level == 1 ? 0x7ffu : 0x1ffu);
}

// One level of a radix search in LDS: the digit of the rem-th largest key among
// the `bins` counted ones; rem becomes its rank inside the digit's bin, whose
// count is returned in `ties`.  NT threads; the result is uniform.
struct Found {
  unsigned digit, rem, ties;
};
template <int NT>
__device__ __forceinline__ Found find_digit(const unsigned* hist, int bins, unsigned rem, unsigned* wsum, Found* out) {
  const int tid = threadIdx.x, per = (bins + NT - 1) / NT;
  unsigned tot = 0u;
  for (int u = 0; u < per; ++u) {
    const int d = bins - 1 - (tid * per + u);
    tot += d >= 0 ? hist[d] : 0u;
  }
  unsigned run = block_incl_scan<NT>(tot, wsum) - tot;
  if (run < rem && run + tot >= rem)
    for (int u = 0; u < per; ++u) {
      const int d = bins - 1 - (tid * per + u);
      const unsigned c = d >= 0 ? hist[d] : 0u;
      if (run < rem && run + c >= rem) *out = Found{(unsigned)d, rem - run, c};
      run += c;
    }
  __syncthreads();
  const Found f = *out;
  __syncthreads();
  return f;
}

__device__ __forceinline__ void set_member(const UpdateArgs& a, int g, unsigned flat) {
  const int tok = (int)(flat / kF), f = (int)(flat % kF);
  const int t = a.H + tok;
  atomicOr(a.bits + ((size_t)g * kF + f) * a.row_words + (t >> 5), 1u << (t & 31));
}

// ---------------------------------------------------------------------------
// Calls of up to kSelectMax keys take their members in two launches: split and
// select.  The encode has counted the candidates in fine digits, so split, grid
// (kSplitBlocks, G) x 256, knows the digit of tau: the candidates above it are
// members, whose bits it sets, and the few in it (0.4% of the budget where
// activations are normal) go to a list of their own.  select, grid G x 1024, finds
// tau and the cut of its ties among those, in LDS, and sets the rest of the bits.
// (One workgroup that read the whole list twice and an emit launch: 18.5 us at
// 1024 keys, 41.5 at 4096, bound by its one CU; now 12.5 and 22.  64 or
// 128 split workgroups per group were no faster: 8 and 9 us for 7, 16 and 18 for 16.)
// A digit that does not fit (ties by the thousand) or that the counts do not
// reach: select takes all of it, by passes over the list.  Beyond kSelectMax those
// would be too long for one workgroup, and hist0 / digit / refine and the tie
// kernels, over 256 workgroups per group, are the better ones.
//
// A list that cannot be used (the sample misjudged): both launches read the dense
// activations, over all their workgroups.  split counts the positive values in
// 13-bit digits; select's workgroups, which otherwise leave at once, set the bits of
// the values above tau's digit and list those in it, and the last of them to end
// finds tau and the cut among these.  Where even they are more than the list holds
// (one value millions of times) they are counted by their other 18 bits, and the
// last workgroup takes the ties in one ordered pass.  (Appends of 600 / 4096 keys with
// every value tied: 0.23 / 0.56 ms; 8.1 / 49 with all of it in one workgroup per group.)
// ---------------------------------------------------------------------------
constexpr int kST = 1024;
constexpr int kSelBuf = 8192;
constexpr int kSplitBlocks = 32;
constexpr int kSelectBlocks = 32;
constexpr int kLowBins = 1 << kSampleShift;  // the values of one 13-bit digit

// The fine digit of the budget-th largest candidate; false if split and select
// cannot work with it.
template <int NT>
__device__ __forceinline__ bool find_fine(const UpdateArgs& a, int g, unsigned* wsum, Found* out, Found& f) {
  if (threadIdx.x == 0) *out = Found{(unsigned)kBins - 1u, 0u, ~0u};
  f = find_digit<NT>(hist_of(a, g, 0), kBins, budget_of(a), wsum, out);
  return list_ok(a, g) && f.digit < (unsigned)kBins - 1u && f.ties <= (unsigned)kSelBuf;
}

// Adds to a histogram, a thread's run of equal bins at once: where one value comes
// by the million its counter would take an atomic for each.
struct RunCount {
  unsigned bin = 0u, n = 0u;
  __device__ __forceinline__ void add(unsigned* hist, unsigned d) {
    if (d != bin) flush(hist);
    bin = d;
    ++n;
  }
  __device__ __forceinline__ void flush(unsigned* hist) {
    if (n) atomicAdd(&hist[bin], n);
    n = 0u;
  }
  // The whole wave's runs, equal bins joined (a counter in memory takes 10 ns for each).
  __device__ __forceinline__ void flush_wave(unsigned* hist) {
    for (unsigned long long left = __ballot(n != 0u); left; left = __ballot(n != 0u)) {  // uniform
      const int lead = (int)__builtin_ctzll(left);
      const unsigned b = (unsigned)__builtin_amdgcn_readlane((int)bin, lead);
      const bool same = n != 0u && bin == b;
      const int total = wave_sum_i(same ? (int)n : 0);
      if ((int)(threadIdx.x & 63) == lead) atomicAdd(&hist[b], (unsigned)total);
      if (same) n = 0u;
    }
  }
};

// The 13-bit counts of a group whose list cannot be used: in the levels of the
// histogram that calls of up to kSelectMax keys have no other use for.
__device__ __forceinline__ unsigned* dense_hist(const UpdateArgs& a, int g) {
  static_assert(2 * kRep * kBins >= kSampleBins, "room in levels 1 and 2");
  return hist_of(a, g, 1);
}

__global__ __launch_bounds__(kUT) void split_kernel(UpdateArgs a) {
  const int g = blockIdx.y, tid = threadIdx.x;
  __shared__ unsigned wsum[kUT / 64];
  __shared__ unsigned dense[kSampleBins];
  __shared__ Found found;
  unsigned* ctl = a.ctl + (size_t)g * kCtl;
  Found f;
  if (!find_fine<kUT>(a, g, wsum, &found, f)) {  // uniform
    if (list_ok(a, g)) return;
    for (int i = tid; i < kSampleBins; i += kUT) dense[i] = 0u;
    unsigned* low = a.ties + (size_t)g * a.list_cap;
    for (int i = (int)blockIdx.x * kUT + tid; i < kLowBins; i += kSplitBlocks * kUT) low[i] = 0u;
    __syncthreads();
    RunCount run;
    each_value<kUT>(a, g, false, blockIdx.x, gridDim.x, [&](unsigned u, unsigned) { run.add(dense, u >> kSampleShift); });
    run.flush(dense);
    __syncthreads();
    unsigned* hg = dense_hist(a, g);
    for (int i = tid; i < kSampleBins; i += kUT)
      if (dense[i]) atomicAdd(&hg[i], dense[i]);
    return;
  }
  const unsigned floor = ctl[kFloor];
  uint2* ties = reinterpret_cast<uint2*>(a.ties + (size_t)g * a.list_cap);
  each_value<kUT>(a, g, true, blockIdx.x, gridDim.x, [&](unsigned u, unsigned flat) {
    const unsigned d = fine_digit(u, floor);
    if (d > f.digit) set_member(a, g, flat);
    if (d == f.digit) ties[atomicAdd(&ctl[kTieLen], 1u)] = make_uint2(flat, u);
  });
}

// The flat index of the `rem`-th of the ties at `tau` in ascending order, by a radix
// search over the complements of what each(fn(value, flat)) goes through.
template <typename Each>
__device__ __forceinline__ unsigned tie_cut(unsigned tau, unsigned rem, unsigned* hist, unsigned* wsum, Found* found,
                                            Each each) {
  unsigned key = 0u;
  const int width[3] = {11, 11, 10};
  int shift = 32;
  for (int l = 0; l < 3; ++l) {
    shift -= width[l];
    const unsigned mask = (1u << width[l]) - 1u;
    const int hi = shift + width[l];
    for (int i = threadIdx.x; i < (1 << width[l]); i += kST) hist[i] = 0u;
    __syncthreads();
    each([&](unsigned u, unsigned flat) {
      const unsigned c = ~flat;
      if (u == tau && (hi == 32 || (c >> hi) == key)) atomicAdd(&hist[(c >> shift) & mask], 1u);
    });
    __syncthreads();
    const Found f = find_digit<kST>(hist, 1 << width[l], rem, wsum, found);
    key = (key << width[l]) | f.digit;
    rem = f.rem;
  }
  return ~key;
}

// tau, given its 13-bit digit and its rank f.rem among that digit's values, from
// passes over them; f becomes that of tau's own ties.
template <typename Each>
__device__ __forceinline__ unsigned find_tau(unsigned top, Found& f, unsigned* hist, unsigned* wsum, Found* found,
                                             Each each) {
  unsigned prefix = top;
  for (int shift = 9; shift >= 0; shift -= 9) {
    for (int i = threadIdx.x; i < 512; i += kST) hist[i] = 0u;
    __syncthreads();
    each([&](unsigned u, unsigned) {
      if ((u >> (shift + 9)) == prefix) atomicAdd(&hist[(u >> shift) & 511u], 1u);
    });
    __syncthreads();
    f = find_digit<kST>(hist, 512, f.rem, wsum, found);
    prefix = (prefix << 9) | f.digit;
  }
  return prefix;
}

struct SelectLds {
  unsigned hist[kSampleBins];
  uint2 bin[kSelBuf];
  unsigned wsum[kST / 64], nbin, base;
  Found found;
};

// select of a group whose list cannot be used, by workgroup x of kSelectBlocks.
__device__ __forceinline__ void select_dense(const UpdateArgs& a, int g, int x, SelectLds& L) {
  const int tid = threadIdx.x;
  unsigned* ctl = a.ctl + (size_t)g * kCtl;
  const unsigned count = budget_of(a);
  unsigned npos = 0u;
  for (int i = tid; i < kSampleBins; i += kST) {
    L.hist[i] = dense_hist(a, g)[i];
    npos += L.hist[i];
  }
  block_incl_scan<kST>(npos, L.wsum);
  npos = 0u;
  for (int i = 0; i < kST / 64; ++i) npos += L.wsum[i];
  __syncthreads();
  const bool all = npos < count;  // fewer positives than the budget: every one is kept (core.py:22-26)
  Found f{0u, 0u, 0u};
  if (!all) f = find_digit<kST>(L.hist, kSampleBins, count, L.wsum, &L.found);
  const unsigned top = f.digit;
  const bool gathered = f.ties <= a.list_cap;
  uint2* list = a.list + (size_t)g * a.list_cap;  // (what the encode left there serves nothing)
  unsigned* low = a.ties + (size_t)g * a.list_cap;
  RunCount run;
  each_value<kST>(a, g, false, x, kSelectBlocks, [&](unsigned u, unsigned flat) {
    const unsigned d = u >> kSampleShift;
    if (all || d > top)
      set_member(a, g, flat);
    else if (d == top && gathered) {
      const unsigned i = atomicAdd(&L.nbin, 1u);
      uint2* to = i < (unsigned)kSelBuf ? L.bin + i : list + atomicAdd(&ctl[kTieLen], 1u);
      *to = make_uint2(flat, u);
    } else if (d == top)
      run.add(low, u & (kLowBins - 1u));
  });
  run.flush_wave(low);
  __syncthreads();
  const unsigned mine = min(L.nbin, (unsigned)kSelBuf);
  if (tid == 0) L.base = mine ? atomicAdd(&ctl[kTieLen], mine) : 0u;
  __syncthreads();
  for (unsigned i = tid; i < mine; i += kST) list[L.base + i] = L.bin[i];
  // the last workgroup to come here goes on
  __threadfence();
  __syncthreads();
  if (tid == 0) L.base = atomicAdd(&ctl[kArrived], 1u);
  __syncthreads();
  if (L.base != kSelectBlocks - 1) return;  // uniform
  __threadfence();
  for (int i = tid; i < kSampleBins; i += kST) dense_hist(a, g)[i] = 0u;  // for the next call
  if (all) return;
  if (gathered) {
    const unsigned n = f.ties;
    const bool in_lds = n <= (unsigned)kSelBuf;
    if (in_lds) {
      for (unsigned i = tid; i < n; i += kST) L.bin[i] = list[i];
      __syncthreads();
    }
    auto each = [&](auto fn) {
      for (unsigned i = tid; i < n; i += kST) {
        const uint2 e = in_lds ? L.bin[i] : list[i];
        fn(e.y, e.x);
      }
    };
    const unsigned tau = find_tau(top, f, L.hist, L.wsum, &L.found, each);
    const unsigned cut = f.ties > f.rem ? tie_cut(tau, f.rem, L.hist, L.wsum, &L.found, each) : ~0u;
    each([&](unsigned u, unsigned flat) {
      if (u > tau || (u == tau && flat <= cut)) set_member(a, g, flat);
    });
    return;
  }
  // tau from the counts of the digit's 2^18 values, 256 of them (a wave's load) at first
  constexpr int kPer = kLowBins / kST;
  static_assert(kPer == 4 * 64, "a wave's 16-byte words");
  const unsigned in_digit = f.rem;
  constexpr int kLoads = 8;
  for (int i0 = tid / 64 * 64; i0 < tid / 64 * 64 + 64; i0 += kLoads) {
    uint4 v[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) v[i] = reinterpret_cast<const uint4*>(low + kPer * (i0 + i))[tid & 63];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int c = wave_sum_i((int)(v[i].x + v[i].y + v[i].z + v[i].w));
      if ((tid & 63) == 0) L.hist[i0 + i] = (unsigned)c;
    }
  }
  __syncthreads();
  f = find_digit<kST>(L.hist, kST, f.rem, L.wsum, &L.found);
  const unsigned high = f.digit;
  if (tid < kPer) L.hist[tid] = low[kPer * high + tid];
  __syncthreads();
  f = find_digit<kST>(L.hist, kPer, f.rem, L.wsum, &L.found);
  const unsigned tau = (top << kSampleShift) | (kPer * high + f.digit);
  const unsigned above = in_digit - f.rem, need = f.rem;  // the digit's members beside tau's ties, and those
  // the activations in flat order until both are complete
  constexpr int kU = 8;
  const size_t n4 = (size_t)a.N * kF / 4;
  const float4* ag = reinterpret_cast<const float4*>(a.act + (size_t)g * a.N * kF);
  unsigned taken = 0u, over = 0u;
  for (size_t base = 0; base < n4 && (taken < need || over < above); base += kU * kST) {  // uniform
    auto value = [&](int u) {
      const size_t i = base + (size_t)u * kST + tid;
      return i < n4 ? ag[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    };
    auto bits = [](float x) { return x > 0.f ? __float_as_uint(x) : 0u; };
    auto in = [&](unsigned b) { return b >= tau && (b >> kSampleShift) == top; };
    bool any = false;
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const float4 v = value(u);
      any |= in(bits(v.x)) || in(bits(v.y)) || in(bits(v.z)) || in(bits(v.w));
    }
    if (!__syncthreads_or(any)) continue;
#pragma unroll 1
    for (int u = 0; u < kU; ++u) {
      const unsigned flat = 4u * (unsigned)(base + (size_t)u * kST + tid);
      const float4 v = value(u);
      const unsigned b[4] = {bits(v.x), bits(v.y), bits(v.z), bits(v.w)};
      unsigned k = 0u;  // ties, and in the upper half the larger ones
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        k += b[j] == tau ? 1u : 0u;
        if (b[j] > tau && in(b[j])) {
          set_member(a, g, flat + j);
          k += 1u << 16;
        }
      }
      unsigned rank = taken + ((block_incl_scan<kST>(k, L.wsum) - k) & 0xffffu);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (b[j] == tau && rank++ < need) set_member(a, g, flat + j);
      unsigned total = 0u;
      for (int i = 0; i < kST / 64; ++i) total += L.wsum[i];
      taken += total & 0xffffu;
      over += total >> 16;
      __syncthreads();  // wsum is rewritten by the next scan
    }
  }
}

// Grid (G, kSelectBlocks) x 1024.
__global__ __launch_bounds__(kST) void select_kernel(UpdateArgs a) {
  const int g = blockIdx.x, tid = threadIdx.x;
  if (blockIdx.y && list_ok(a, g)) return;  // uniform
  __shared__ SelectLds L;
  unsigned* ctl = a.ctl + (size_t)g * kCtl;
  const unsigned count = budget_of(a);
  if (blockIdx.y == 0)
    for (int i = tid; i < kSampleBins; i += kST) a.sample[(size_t)g * kSampleBins + i] = 0u;  // for the next call
  if (tid == 0) L.nbin = 0u;
  Found f;
  const bool split = blockIdx.y == 0 && find_fine<kST>(a, g, L.wsum, &L.found, f);  // uniform
  if (blockIdx.y == 0)
    for (int i = tid; i < kBins; i += kST) hist_of(a, g, 0)[i] = 0u;  // for the next call
  if (!split && !list_ok(a, g)) {
    select_dense(a, g, blockIdx.y, L);
    return;
  }
  unsigned prefix;
  if (split) {
    const uint2* ties = reinterpret_cast<const uint2*>(a.ties + (size_t)g * a.list_cap);
    for (unsigned i = tid; i < f.ties; i += kST) L.bin[i] = ties[i];
    if (tid == 0) L.nbin = f.ties;
    for (int i = tid; i < (1 << kFineShift); i += kST) L.hist[i] = 0u;
    __syncthreads();
    const unsigned base = ctl[kFloor] + (f.digit << kFineShift);
    for (unsigned i = tid; i < L.nbin; i += kST) atomicAdd(&L.hist[L.bin[i].y - base], 1u);
    __syncthreads();
    f = find_digit<kST>(L.hist, 1 << kFineShift, f.rem, L.wsum, &L.found);
    prefix = base + f.digit;
    auto each = [&](auto fn) {
      for (unsigned i = tid; i < L.nbin; i += kST) fn(L.bin[i].y, L.bin[i].x);
    };
    const unsigned cut = f.ties > f.rem ? tie_cut(prefix, f.rem, L.hist, L.wsum, &L.found, each) : ~0u;
    each([&](unsigned u, unsigned flat) {
      if (u > prefix || (u == prefix && flat <= cut)) set_member(a, g, flat);
    });
    return;
  }
  // The listed values lie within a few octaves above the floor, 32 digits each,
  // so they are counted in kRel digits from the floor's on, 8 replicas of each
  // (64 lanes meet in some 25 digits: one replica took 15 us of atomics for the
  // list of 4096 keys); where tau lies beyond them, in all 8192.
  auto listed_values = [&](auto fn) { each_value<kST>(a, g, true, 0, 1, fn); };
  constexpr unsigned kRel = kSampleBins / 8;
  unsigned npos = 0u;
  for (bool rel = true;; rel = false) {  // uniform
    const unsigned base = rel ? ctl[kFloor] >> kSampleShift : 0u;
    __syncthreads();
    for (int i = tid; i < kSampleBins; i += kST) L.hist[i] = 0u;
    __syncthreads();
    listed_values([&](unsigned u, unsigned) {
      const unsigned d = (u >> kSampleShift) - base;
      atomicAdd(&L.hist[rel ? 8u * min(d, kRel - 1u) + (tid & 7) : d], 1u);
    });
    __syncthreads();
    if (rel) {
      unsigned c = 0u;
      if (tid < (int)kRel)
#pragma unroll
        for (int r = 0; r < 8; ++r) c += L.hist[8 * tid + r];
      __syncthreads();
      if (tid < (int)kRel) L.hist[tid] = c;
      __syncthreads();
    }
    const int bins = rel ? (int)kRel : kSampleBins;
    npos = 0u;
    for (int i = tid; i < bins; i += kST) npos += L.hist[i];
    block_incl_scan<kST>(npos, L.wsum);
    npos = 0u;
    for (int i = 0; i < kST / 64; ++i) npos += L.wsum[i];
    __syncthreads();
    if (npos < count) {  // fewer positives than the budget: every one is kept (core.py:22-26)
      listed_values([&](unsigned, unsigned flat) { set_member(a, g, flat); });
      return;
    }
    f = find_digit<kST>(L.hist, bins, count, L.wsum, &L.found);
    if (!rel) break;
    if (f.digit < kRel - 1u) {
      f.digit += base;
      break;
    }
  }
  const unsigned top = f.digit;
  const bool gathered = f.ties <= (unsigned)kSelBuf;
  if (gathered) {
    listed_values([&](unsigned u, unsigned flat) {
      if ((u >> kSampleShift) == top) L.bin[atomicAdd(&L.nbin, 1u)] = make_uint2(flat, u);
    });
    __syncthreads();
  }
  auto each = [&](auto fn) {
    if (gathered)
      for (unsigned i = tid; i < L.nbin; i += kST) fn(L.bin[i].y, L.bin[i].x);
    else
      listed_values(fn);
  };
  prefix = find_tau(top, f, L.hist, L.wsum, &L.found, each);
  const unsigned cut = f.ties > f.rem ? tie_cut(prefix, f.rem, L.hist, L.wsum, &L.found, each) : ~0u;
  listed_values([&](unsigned u, unsigned flat) {
    if (u > prefix || (u == prefix && flat <= cut)) set_member(a, g, flat);
  });
}

// ---------------------------------------------------------------------------
// emit: grid (blocks, G) x 256: the bit of every value above tau and of the ties
// up to the cut.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kUT) void emit_kernel(UpdateArgs a) {
  const int g = blockIdx.y;
  const unsigned* ctl = a.ctl + (size_t)g * kCtl;
  const unsigned tau = ctl[kTau], cut = ctl[kCut];
  each_value<kUT>(a, g, list_ok(a, g), blockIdx.x, gridDim.x, [&](unsigned u, unsigned flat) {
    if (u > tau || (u == tau && flat <= cut)) set_member(a, g, flat);
  });
}

// ---------------------------------------------------------------------------
// ties, only when the ties at tau overflow the budget: the flat index of the
// last of the first `need` in ascending flat index (core.py:23-24).
// tie_count_kernel, grid (blocks, G) x 256: gathers the ties' flat indices from
// the list, or counts the ties of each contiguous range [r L, (r + 1) L) of the
// dense activations.  tie_cut_kernel, grid G x 1024: a radix search over the
// gathered indices, or the range that holds the need-th tie and a scan of it.
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool ordered_ties(const UpdateArgs& a, int g) {
  const unsigned* ctl = a.ctl + (size_t)g * kCtl;
  return ctl[kMode] == kModeTopK && ctl[kOrdered];
}

__global__ __launch_bounds__(kUT) void tie_count_kernel(UpdateArgs a) {
  const int g = blockIdx.y, tid = threadIdx.x;
  if (!ordered_ties(a, g)) return;
  __shared__ unsigned wsum[kUT / 64];
  unsigned* ctl = a.ctl + (size_t)g * kCtl;
  if (list_ok(a, g)) {
    const unsigned tau = ctl[kTau];
    unsigned* ties = a.ties + (size_t)g * a.list_cap;
    each_value<kUT>(a, g, true, blockIdx.x, gridDim.x, [&](unsigned u, unsigned flat) {
      if (u == tau) ties[atomicAdd(&ctl[kTieLen], 1u)] = flat;
    });
    return;
  }
  const float tau = __uint_as_float(ctl[kTau]);
  const size_t n = (size_t)a.N * kF;
  const float4* ag = reinterpret_cast<const float4*>(a.act + (size_t)g * n);
  for (int r = blockIdx.x; r < a.tie_blocks; r += gridDim.x) {  // uniform
    const size_t lo = min(n, (size_t)r * a.tie_len), hi = min(n, lo + a.tie_len);
    unsigned c = 0;
    constexpr int kU = 8;  // loads in flight per thread
    for (size_t i0 = lo / 4 + tid; i0 < hi / 4; i0 += kU * kUT) {
      float4 v[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const size_t i = i0 + (size_t)u * kUT;
        v[u] = ag[i < hi / 4 ? i : i0];  // a repeated value is not counted twice below
      }
#pragma unroll
      for (int u = 0; u < kU; ++u)
        if (i0 + (size_t)u * kUT < hi / 4)
          c += (unsigned)(v[u].x == tau) + (unsigned)(v[u].y == tau) + (unsigned)(v[u].z == tau) +
               (unsigned)(v[u].w == tau);
    }
    block_incl_scan<kUT>(c, wsum);
    if (tid == 0) a.tcount[(size_t)g * a.tie_blocks + r] = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    __syncthreads();  // wsum is rewritten by the next range's scan
  }
}

__global__ __launch_bounds__(kST) void tie_cut_kernel(UpdateArgs a) {
  const int g = blockIdx.x, tid = threadIdx.x;
  if (!ordered_ties(a, g)) return;
  __shared__ unsigned hist[kBins], wsum[kST / 64], range_s, below_s;
  __shared__ Found found;
  unsigned* ctl = a.ctl + (size_t)g * kCtl;
  const unsigned need = ctl[kNeed];  // >= 1
  if (list_ok(a, g)) {
    const unsigned* ties = a.ties + (size_t)g * a.list_cap;
    const unsigned len = ctl[kTieLen];
    unsigned key = 0u, rem = need;
    const int width[3] = {11, 11, 10};
    int shift = 32;
    for (int l = 0; l < 3; ++l) {
      shift -= width[l];
      const unsigned mask = (1u << width[l]) - 1u;
      const int hi = shift + width[l];
      for (int i = tid; i < kBins; i += kST) hist[i] = 0u;
      __syncthreads();
      for (unsigned i = tid; i < len; i += kST) {
        const unsigned c = ~ties[i];
        if (hi == 32 || (c >> hi) == key) atomicAdd(&hist[(c >> shift) & mask], 1u);
      }
      __syncthreads();
      const Found f = find_digit<kST>(hist, 1 << width[l], rem, wsum, &found);
      key = (key << width[l]) | f.digit;
      rem = f.rem;
    }
    if (tid == 0) ctl[kCut] = ~key;
    return;
  }
  const float tau = __uint_as_float(ctl[kTau]);
  constexpr int kPer = kMaxTieBlocks / kST;
  unsigned c[kPer], tot = 0u;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int r = tid * kPer + u;
    c[u] = r < a.tie_blocks ? a.tcount[(size_t)g * a.tie_blocks + r] : 0u;
    tot += c[u];
  }
  unsigned run = block_incl_scan<kST>(tot, wsum) - tot;
  if (run < need && run + tot >= need)
    for (int u = 0; u < kPer; ++u) {
      if (run < need && run + c[u] >= need) {
        range_s = (unsigned)(tid * kPer + u);
        below_s = run;
      }
      run += c[u];
    }
  __syncthreads();
  const size_t n = (size_t)a.N * kF;
  const size_t lo = min(n, (size_t)range_s * a.tie_len), hi = min(n, lo + a.tie_len);
  const float4* ag = reinterpret_cast<const float4*>(a.act + (size_t)g * n);
  unsigned taken = below_s;
  for (size_t base = lo / 4; base < hi / 4 && taken < need; base += kST) {  // uniform condition
    const size_t i = base + tid;
    const float4 v = i < hi / 4 ? ag[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    const bool h[4] = {v.x == tau, v.y == tau, v.z == tau, v.w == tau};
    const unsigned k = (unsigned)h[0] + (unsigned)h[1] + (unsigned)h[2] + (unsigned)h[3];
    const unsigned incl = block_incl_scan<kST>(k, wsum);
    unsigned rank = taken + incl - k;  // rank of this thread's first tie among all ties
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (h[j] && ++rank == need) ctl[kCut] = (unsigned)(4 * i + j);
    for (int j = 0; j < kST / 64; ++j) taken += wsum[j];
    __syncthreads();  // wsum is rewritten by the next scan
  }
}

// ---------------------------------------------------------------------------
// moments: grid (kChunks, G) x 512.  Wave w handles buckets 32c + 4w + j:
// members from the bitmap, two-pass moments of their keys; then the tile
// merge, thread = (dim k, bucket col) pairs of mean row k and var row 128+k.
// Bound by memory round trips, by the 49 MB of moments read and rewritten (8
// groups) and by the fetching of its own instructions, so the buckets are a
// loop that 24 waves per CU run side by side, not one unrolled over a wave's
// buckets (171 registers, 35 us at 1024 keys).  Lane l owns dims 2l, 2l + 1
// of every member, so no sum crosses lanes, and the first 8 members of a
// bucket (at a budget of 8 per key, 3 at 1024 keys and 11 at 4096 on average)
// are requested together and kept for the second pass; the tile's old moments
// are requested before the first of them.  15.9 us at 1024 keys, 40 at 4096
// (16 members kept: 22 and 46, registers spilled at 6 waves per SIMD).
// ---------------------------------------------------------------------------
constexpr int kMaxBlock = 4096;  // new tokens per update
constexpr int kMT = 512;
constexpr int kMomSlot = 512;    // members listed at once: 16 bitmap words hold no more
constexpr int kMomRound = 8;     // member key words requested at once
constexpr int kMomCols = kChunk / (kMT / 64);  // buckets per wave (4)

// The update's merge (core.py:194-199) for bucket sizes a (old) and b (block),
// den = max(a + b, 1): every rounding of (a x + b y) / den + ..., with the
// quotients by quotient().
__device__ __forceinline__ float merge_mean(float a, float b, float den, float rden, float ma, float mb) {
#pragma clang fp contract(off)
  return quotient(a * ma + b * mb, den, rden);
}
__device__ __forceinline__ float merge_var(float a, float b, float den, float rden, float ab, float ma, float mb, float va,
                                           float vb) {
#pragma clang fp contract(off)
  const float v = quotient(a * va + b * vb, den, rden);
  const float d = ma - mb;
  return v + ab * (d * d);
}

template <typename KT>
__global__ __launch_bounds__(kMT, 6) void moments_kernel(UpdateArgs a) {
  const int c = blockIdx.x, g = blockIdx.y, tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  __shared__ float nm[kChunk][kD + 1], nv[kChunk][kD + 1];
  __shared__ int nb[kChunk];
  __shared__ uint16_t toks_all[kMT / 64][kMomSlot];  // tokens of the block, from its first word's on
  uint16_t* toks = toks_all[w];
  typedef KeyLoad<KT> KL;
  const int w_lo = a.H >> 5, w_hi = (a.H + a.N - 1) >> 5;
  // the block's key rows, from its first bitmap word's token on (32-bit offsets)
  constexpr unsigned kRowBytes = kD * sizeof(KT);
  const __amdgpu_buffer_rsrc_t kr =
      raw_buffer(static_cast<const KT*>(a.k) + (size_t)g * a.ks + (size_t)w_lo * 32 * kD,
                 (int)((unsigned)(a.H + a.N - 32 * w_lo) * kRowBytes));
  const unsigned at_dims = 2u * lane * (unsigned)sizeof(KT);
  const int f0 = c * kChunk + w * kMomCols;
  const uint32_t* rows = a.bits + ((size_t)g * kF + f0) * a.row_words;
  // Word wd of the wave's bucket j, tokens of the block only.
  auto word = [&](int j, int wd) {
    uint32_t m = f0 + j < kF && wd <= w_hi ? rows[(size_t)j * a.row_words + wd] : 0u;
    if (wd == w_lo) m &= ~0u << (a.H & 31);                                      // tokens before H
    if (wd == w_hi && ((a.H + a.N) & 31)) m &= (1u << ((a.H + a.N) & 31)) - 1u;  // tokens past H + N
    return m;
  };
  uint32_t next = word(0, w_lo + lane);
  float* tile = a.moments + (size_t)(g * kChunks + c) * kRow * kChunk;
  const int col = tid & (kChunk - 1), f = c * kChunk + col;
  constexpr int kRowsPerThread = kD / (kMT / kChunk);  // 8
  float ma[kRowsPerThread], va[kRowsPerThread];
#pragma unroll
  for (int i = 0; i < kRowsPerThread; ++i) {
    const int k = (tid >> 5) + (kMT / kChunk) * i;
    ma[i] = tile[k * kChunk + col];
    va[i] = tile[(kD + k) * kChunk + col];
  }
  const int na = a.counts[(size_t)g * kFP + f];
#pragma unroll 1
  for (int j = 0; j < kMomCols; ++j) {
    const uint32_t head = next;  // the bucket's first 64 words: the whole block up to 2017 tokens
    if (j + 1 < kMomCols) next = word(j + 1, w_lo + lane);
    // members of words [w0, w0 + 64) in ascending order to toks[n ..], up to kMomSlot; n grows by their number
    auto list_words = [&](uint32_t m, int w0, int n) {
      const int incl = (int)wave_incl_scan((unsigned)__popc(m));
      int at = n + incl - __popc(m);
      __builtin_amdgcn_wave_barrier();
      for (; m && at < kMomSlot; m &= m - 1u) toks[at++] = (uint16_t)((w0 + lane - w_lo) * 32 + (int)__builtin_ctz(m));
      __builtin_amdgcn_wave_barrier();
      return n + __builtin_amdgcn_readlane(incl, 63);
    };
    // two-pass moments of the ORIGINAL keys (core.py:84-88)
    float m0 = 0.f, m1 = 0.f, v0 = 0.f, v1 = 0.f;
    auto sum = [&](typename KL::Raw2 r) {
      m0 += KL::lo(r);
      m1 += KL::hi(r);
    };
    auto dev = [&](typename KL::Raw2 r) {
      const float d0 = KL::lo(r) - m0, d1 = KL::hi(r) - m1;
      v0 += d0 * d0;
      v1 += d1 * d1;
    };
    auto pass = [&](int i0, int n, auto add) {
      for (; i0 < n; i0 += kMomRound) {  // uniform
        typename KL::Raw2 r[kMomRound];
#pragma unroll
        for (int u = 0; u < kMomRound; ++u) r[u] = KL::load2(kr, toks[min(i0 + u, n - 1)] * kRowBytes + at_dims);
#pragma unroll
        for (int u = 0; u < kMomRound; ++u)
          if (i0 + u < n) add(r[u]);
      }
    };
    int b = list_words(head, w_lo, 0);
    for (int w0 = w_lo + 64; w0 <= w_hi; w0 += 64) b = list_words(word(j, w0 + lane), w0, b);
    if (b <= kMomSlot) {  // uniform: the list is whole
      if (b > 0) {
        typename KL::Raw2 kept[kMomRound];
#pragma unroll
        for (int u = 0; u < kMomRound; ++u) kept[u] = KL::load2(kr, toks[min(u, b - 1)] * kRowBytes + at_dims);
        const float n = (float)b, rn = 1.0f / n;
#pragma unroll
        for (int u = 0; u < kMomRound; ++u)
          if (u < b) sum(kept[u]);
        pass(kMomRound, b, sum);
        m0 = quotient(m0, n, rn);
        m1 = quotient(m1, n, rn);
#pragma unroll
        for (int u = 0; u < kMomRound; ++u)
          if (u < b) dev(kept[u]);
        pass(kMomRound, b, dev);
        v0 = quotient(v0, n, rn);
        v1 = quotient(v1, n, rn);
      }
    } else {  // 16 words (at most 512 members) at a time, once for each pass
      b = 0;
      for (int w0 = w_lo; w0 <= w_hi; w0 += 16) {
        const int n = list_words(lane < 16 ? word(j, w0 + lane) : 0u, w0, 0);
        pass(0, n, sum);
        b += n;
      }
      if (b > 0) {
        const float n = (float)b, rn = 1.0f / n;
        m0 = quotient(m0, n, rn);
        m1 = quotient(m1, n, rn);
        for (int w0 = w_lo; w0 <= w_hi; w0 += 16) 
          pass(0, list_words(lane < 16 ? word(j, w0 + lane) : 0u, w0, 0), dev);
        v0 = quotient(v0, n, rn);
        v1 = quotient(v1, n, rn);
      }
    }
    const int o = w * kMomCols + j;
    nm[o][2 * lane] = m0;
    nm[o][2 * lane + 1] = m1;
    nv[o][2 * lane] = v0;
    nv[o][2 * lane + 1] = v1;
    if (lane == 0) nb[o] = b;
  }
  __syncthreads();
  if (f >= kF) return;  // padding columns stay zero
  const int nbn = nb[col];
  const float fa = (float)na, fb = (float)nbn;
  const float total = fa + fb, den = total < 1.f ? 1.f : total, rden = 1.0f / den, ab = (fa * fb) / (den * den);
#pragma unroll
  for (int i = 0; i < kRowsPerThread; ++i) {
    const int k = (tid >> 5) + (kMT / kChunk) * i;
    const float mb = nm[col][k], vb = nv[col][k];
    tile[k * kChunk + col] = merge_mean(fa, fb, den, rden, ma[i], mb);
    tile[(kD + k) * kChunk + col] = merge_var(fa, fb, den, rden, ab, ma[i], mb, va[i], vb);
  }
  if (tid < kChunk) a.counts[(size_t)g * kFP + f] = na + nbn;
}

// ---------------------------------------------------------------------------
// Build-only kernels.
// center (build without a given center, core.py:95): keys.float().mean(0)
// over K rows [H, H + N).  center_part_kernel: grid (kCenterParts, G) x 256,
// part p sums rows [p R, (p + 1) R), R = ceil(N / kCenterParts), in double
// (thread = row step tid >> 4 of 16, dims 8 (tid & 15) ..);
// center_final_kernel: grid G x 128 adds the parts in order, divides by N.
// ---------------------------------------------------------------------------
template <typename KT>
__global__ __launch_bounds__(kUT) void center_part_kernel(UpdateArgs a, double* part) {
  const int p = blockIdx.x, g = blockIdx.y, tid = threadIdx.x;
  __shared__ double red[kUT / 16][kD];
  const int R = (a.N + kCenterParts - 1) / kCenterParts;
  const int lo = min(a.N, p * R), hi = min(a.N, lo + R);
  const int r = tid >> 4, d0 = (tid & 15) * 8;
  const KT* kg = static_cast<const KT*>(a.k) + (size_t)g * a.ks + (size_t)a.H * kD;
  double acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = 0.0;
  for (int t = lo + r; t < hi; t += kUT / 16) {
    float x[8];
    KeyLoad<KT>::load8(kg + (size_t)t * kD + d0, x);
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] += x[j];
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) red[r][d0 + j] = acc[j];
  __syncthreads();
  if (tid < kD) {
    double t = 0.0;
#pragma unroll
    for (int i = 0; i < kUT / 16; ++i) t += red[i][tid];
    part[((size_t)g * kCenterParts + p) * kD + tid] = t;
  }
}

__global__ __launch_bounds__(kD) void center_final_kernel(UpdateArgs a, const double* part, float* center) {
  const int g = blockIdx.x, d = threadIdx.x;
  double t = 0.0;
  for (int p = 0; p < kCenterParts; ++p) t += part[((size_t)g * kCenterParts + p) * kD + d];
  center[(size_t)g * kD + d] = (float)(t / (double)a.N);
}

// clear: grid (blocks, G) x 256 zeroes the group's F bitmap rows (row_words
// is a multiple of 4 words and the rows are 16-byte aligned).
__global__ __launch_bounds__(kUT) void clear_bits_kernel(UpdateArgs a) {
  const int g = blockIdx.y;
  const size_t n4 = (size_t)kF * a.row_words / 4;
  uint4* bg = reinterpret_cast<uint4*>(a.bits + (size_t)g * kF * a.row_words);
  for (size_t i = (size_t)blockIdx.x * kUT + threadIdx.x; i < n4; i += (size_t)gridDim.x * kUT)
    bg[i] = make_uint4(0u, 0u, 0u, 0u);
}

// ---------------------------------------------------------------------------
// build_moments: grid (F, G) x NT, one workgroup per bucket f, any member
// count.  Members are the set bits of the bucket's bitmap row below N (a
// build indexes K rows = bitmap columns [0, N)).  The row is compacted into an
// LDS token list, 2048 words (64K keys) requested at once; a list of more than
// kList tokens is rebuilt 64 words at a time in each pass.  Workgroup x takes
// bucket 375 (x % 8) + x / 8: consecutive workgroups go to the 8 XCDs in turn,
// so each XCD works through consecutive buckets and its L2 joins their 4-byte
// columns of the moment tiles before they are written back.  Thread = (member
// slot tid >> 4, dims 8 (tid & 15) ..), double accumulation, fixed order: the
// slots of a wave by shuffles, then the waves.  The first 192 members of 256
// threads (a 64K build has 175 on average; 96 of fp32) are requested together and
// kept packed in registers, so the second pass reads no memory.  Up to kSmallBuild keys a workgroup is one wave (four member slots,
// a list of 512 tokens): a bucket then has so few members that the launch is
// bound by the chain of its 24,000 workgroups' loads, and four times as many of
// them are in flight; longer buckets are left to build_moments_rest_kernel.  256
// against 64 threads, 8 groups: 136 / 52 us at 6000 keys, 158 / 87 at 16384, 190
// / 159 at 32768, 282 / 331 at 65536 (and the other launch).
// mean = sum / n rounded to fp32; var = sum (x - mean)^2 / n
// with that rounded mean; empty bucket -> 0 (core.py:84-88).  Counts and
// moments are written, not merged.
// ---------------------------------------------------------------------------
constexpr int kList = 2048;
constexpr int kSmallBuild = 32768;  // keys up to which a bucket is one wave's
template <typename KT>
constexpr int kKeep = sizeof(KT) == 2 ? 12 : 6;  // members per slot kept in registers (48 of them)

template <int NT>
struct BuildMomentsLds {
  static constexpr int kLen = NT == 64 ? kList / 4 : kList;  // of the token list
  int toks[kLen];
  double red[NT / 64][kD];
  unsigned wsum[NT / 64];
  float mean[kD];
};

// Members among words [w0, w0 + NT W) of the row below word w1, W consecutive
// words per thread (8: the row is 16-byte aligned, as a build's is and a
// caller's of summarize need not be) ->
// toks[at ..] when they all fit below kLen.  Returns their count (uniform);
// the caller barriers before the list is read and before the next chunk.
template <int NT, int W>
__device__ __forceinline__ unsigned compact_chunk(const uint32_t* row, int w0, int w1, int N, int* toks, unsigned at,
                                                  unsigned* wsum) {
  const int wd = w0 + W * (int)threadIdx.x, nw = (N + 31) >> 5;
  uint32_t m[W];
#pragma unroll
  for (int i = 0; i < W; ++i) m[i] = 0u;
  if constexpr (W == 8) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
      if (wd + 4 * h < w1) {  // (row_words is a multiple of 4)
        const uint4 v = *reinterpret_cast<const uint4*>(row + wd + 4 * h);
        m[4 * h] = v.x; m[4 * h + 1] = v.y; m[4 * h + 2] = v.z; m[4 * h + 3] = v.w;
      }
  } else if (wd < w1) {
    m[0] = row[wd];
  }
  unsigned pc = 0u;
#pragma unroll
  for (int i = 0; i < W; ++i) {
    if (wd + i >= nw) m[i] = 0u;
    if (wd + i == nw - 1 && (N & 31)) m[i] &= (1u << (N & 31)) - 1u;
    pc += (unsigned)__popc(m[i]);
  }
  const unsigned incl = block_incl_scan<NT>(pc, wsum);
  unsigned total = 0u;
#pragma unroll
  for (int i = 0; i < NT / 64; ++i) total += wsum[i];
  if (at + total <= (unsigned)BuildMomentsLds<NT>::kLen) {
    unsigned p = at + incl - pc;
#pragma unroll
    for (int i = 0; i < W; ++i)
      for (; m[i]; m[i] &= m[i] - 1u) toks[p++] = (wd + i) * 32 + (int)__builtin_ctz(m[i]);
  }
  return total;
}

// v of lane l ^ M, M = 16 or 32.
template <int M>
__device__ __forceinline__ double xor_d(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
  const unsigned x = M == 16 ? xor16_u(lo) : xor32_u(lo), y = M == 16 ? xor16_u(hi) : xor32_u(hi);
  return __longlong_as_double((long long)(((unsigned long long)y << 32) | x));
}

// One pass's order-fixed sum over the slots, into red[0].
template <int NT>
__device__ __forceinline__ void slot_sum(BuildMomentsLds<NT>& L, double (&acc)[8]) {
  const int tid = threadIdx.x, lane = tid & 63;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    acc[j] += xor_d<16>(acc[j]);
    acc[j] += xor_d<32>(acc[j]);
  }
  if (lane < 16)
#pragma unroll
    for (int j = 0; j < 8; ++j) L.red[tid >> 6][8 * lane + j] = acc[j];
  __syncthreads();
  if constexpr (NT > 64) {
    static_assert(NT == 256, "four waves");
    if (tid < kD) L.red[0][tid] = (L.red[0][tid] + L.red[1][tid]) + (L.red[2][tid] + L.red[3][tid]);
    __syncthreads();
  }
}

template <typename KT, int NT>
__device__ __forceinline__ void bucket_moments(const UpdateArgs& a, int g, int f, BuildMomentsLds<NT>& L) {
  constexpr int kSlots = NT / 16, kLen = BuildMomentsLds<NT>::kLen;
  const int tid = threadIdx.x, slot = tid >> 4, d0 = (tid & 15) * 8;
  typedef KeyLoad<KT> KL;
  const uint32_t* row = a.bits + ((size_t)g * kF + f) * a.row_words;
  const KT* kg = static_cast<const KT*>(a.k) + (size_t)g * a.ks + d0;
  const int nw = (a.N + 31) >> 5;
  // count the members, keeping the list while it fits
  unsigned n = 0;
  bool listed = true;
  const bool wide = ((a.row_words & 3) | (int64_t)(reinterpret_cast<uintptr_t>(a.bits) & 15u)) == 0;
  for (int w0 = 0; w0 < nw; w0 += wide ? 8 * NT : NT) {  // uniform
    const unsigned c = wide ? compact_chunk<NT, 8>(row, w0, nw, a.N, L.toks, n, L.wsum)
                            : compact_chunk<NT, 1>(row, w0, nw, a.N, L.toks, n, L.wsum);
    listed = listed && n + c <= (unsigned)kLen;
    __syncthreads();
    n += c;
  }
  if (tid == 0) a.counts[(size_t)g * kFP + f] = (int)n;
  if constexpr (NT == 64)
    if (!listed) return;  // uniform: build_moments_rest_kernel's
  auto key_row = [&](unsigned i) { return KL::raw8(kg + (size_t)L.toks[i] * kD); };
  typename KL::Raw8 kept[kKeep<KT>];
  if (listed)
#pragma unroll
    for (int u = 0; u < kKeep<KT>; ++u)
      if (kSlots * u < (int)n) kept[u] = key_row(min((unsigned)(slot + kSlots * u), n - 1u));  // uniform
  double acc[8];
  auto each_member = [&](auto add) {
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = 0.0;
    if (listed) {
#pragma unroll
      for (int u = 0; u < kKeep<KT>; ++u)
        if (slot + kSlots * u < (int)n) add(kept[u]);
#pragma unroll 4
      for (unsigned i = slot + kSlots * kKeep<KT>; i < n; i += kSlots) add(key_row(i));
    } else {
      for (int w0 = 0; w0 < nw; w0 += kLen / 32) {
        __syncthreads();  // the previous chunk's list has been read
        const unsigned c = compact_chunk<NT, 1>(row, w0, min(nw, w0 + kLen / 32), a.N, L.toks, 0u, L.wsum);  // always fits
        __syncthreads();
#pragma unroll 4
        for (unsigned i = slot; i < c; i += kSlots) add(key_row(i));
      }
    }
  };
  each_member([&](const typename KL::Raw8& r) {
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] += (double)KL::at(r, j);
  });
  slot_sum(L, acc);
  for (int d = tid; d < kD; d += NT) L.mean[d] = n ? (float)(L.red[0][d] / (double)n) : 0.f;
  __syncthreads();
  float m[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) m[j] = L.mean[d0 + j];
  each_member([&](const typename KL::Raw8& r) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const double t = (double)KL::at(r, j) - (double)m[j];
      acc[j] += t * t;
    }
  });
  slot_sum(L, acc);
  float* tile = a.moments + (size_t)(g * kChunks + f / kChunk) * kRow * kChunk;
  const int col = f % kChunk;
  for (int d = tid; d < kD; d += NT) {
    tile[d * kChunk + col] = L.mean[d];
    tile[(kD + d) * kChunk + col] = n ? (float)(L.red[0][d] / (double)n) : 0.f;
  }
}

__device__ __forceinline__ int moment_bucket(unsigned x) {
  static_assert(kF % 8 == 0, "buckets in 8 equal runs");
  return (int)(x & 7u) * (kF / 8) + (int)(x >> 3);
}

template <typename KT, int NT>
__global__ __launch_bounds__(NT, 4) void build_moments_kernel(UpdateArgs a) {
  __shared__ BuildMomentsLds<NT> L;
  bucket_moments<KT, NT>(a, blockIdx.y, moment_bucket(blockIdx.x), L);
}

// After it, grid (F, G) x 256: the buckets of more members than a one-wave
// workgroup lists.  A workgroup each, as any number of them may be (a dense bitmap,
// a budget of many per key): 64 workgroups for all took 22.9 ms for one group of
// 32768 keys with half of them in every bucket, 1000 took 2.1, now 1.9 (one launch
// of 256 threads: 1.7); where there is none, 8 groups' launch takes 7.5 us.
template <typename KT>
__global__ __launch_bounds__(kUT, 4) void build_moments_rest_kernel(UpdateArgs a) {
  __shared__ BuildMomentsLds<kUT> L;
  const int g = blockIdx.y, f = moment_bucket(blockIdx.x);
  if (a.counts[(size_t)g * kFP + f] > BuildMomentsLds<64>::kLen) bucket_moments<KT, kUT>(a, g, f, L);  // uniform
}

// ---------------------------------------------------------------------------
// positive_global_topk on a given [N][F] fp32 matrix (core.py:13-26), for
// callers of the Python surface: the same threshold kernels (digit / refine)
// after a level-0 histogram, then the flat indices in the reference's order
// -- every strict value (a > tau and a > 0; every positive one when fewer
// than the budget are positive) in ascending flat index, then the first
// `need` values equal to tau in ascending flat index.  The matrix is cut
// into the contiguous ranges of the tie kernels; flat_count_kernel counts
// each range's strict values and ties (tcount[2r], tcount[2r + 1]),
// flat_emit_kernel writes them after the lower ranges' ones.
// ---------------------------------------------------------------------------
struct FlatRule {
  float tau;
  bool all_pos, ties;
  __device__ bool strict(float v) const { return all_pos ? v > 0.f : (v > tau && v > 0.f); }
  __device__ bool tie(float v) const { return ties && v == tau; }
};

__device__ __forceinline__ FlatRule flat_rule(const UpdateArgs& a, int g) {
  const unsigned* ctl = a.ctl + (size_t)g * kCtl;
  FlatRule r;
  r.tau = __uint_as_float(ctl[kTau]);  // +inf (nothing) for an empty budget
  r.all_pos = ctl[kMode] == kModeAllPositive;
  r.ties = !r.all_pos && r.tau > 0.f && ctl[kTau] != 0x7f800000u;
  return r;
}

__global__ __launch_bounds__(kUT) void flat_count_kernel(UpdateArgs a) {
  const int g = blockIdx.y, tid = threadIdx.x;
  __shared__ unsigned wsum[kUT / 64];
  const FlatRule rule = flat_rule(a, g);
  const size_t n = (size_t)a.N * kF;
  const float4* ag = reinterpret_cast<const float4*>(a.act + (size_t)g * n);
  for (int r = blockIdx.x; r < a.tie_blocks; r += gridDim.x) {  // uniform
    const size_t lo = min(n, (size_t)r * a.tie_len), hi = min(n, lo + a.tie_len);
    unsigned cs = 0, ct = 0;
    for (size_t i = lo / 4 + tid; i < hi / 4; i += kUT) {
      const float4 v = ag[i];
      const float vv[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        cs += rule.strict(vv[j]);
        ct += rule.tie(vv[j]);
      }
    }
    block_incl_scan<kUT>(cs, wsum);
    if (tid == 0) a.tcount[((size_t)g * a.tie_blocks + r) * 2] = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    __syncthreads();
    block_incl_scan<kUT>(ct, wsum);
    if (tid == 0) a.tcount[((size_t)g * a.tie_blocks + r) * 2 + 1] = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    __syncthreads();
  }
}

__global__ __launch_bounds__(kUT) void flat_emit_kernel(UpdateArgs a, int64_t* out, int* out_len) {
  const int g = blockIdx.y, tid = threadIdx.x;
  __shared__ unsigned wsum[kUT / 64];
  const FlatRule rule = flat_rule(a, g);
  const unsigned need = rule.ties ? a.ctl[(size_t)g * kCtl + kNeed] : 0u;
  const unsigned* tc = a.tcount + (size_t)g * a.tie_blocks * 2;
  // all strict values come first: their total over every range
  unsigned all_s = 0, all_t = 0;
  for (int j = tid; j < a.tie_blocks; j += kUT) {
    all_s += tc[2 * j];
    all_t += tc[2 * j + 1];
  }
  block_incl_scan<kUT>(all_s, wsum);
  const unsigned strict_total = wsum[0] + wsum[1] + wsum[2] + wsum[3];
  __syncthreads();
  block_incl_scan<kUT>(all_t, wsum);
  const unsigned ties_total = wsum[0] + wsum[1] + wsum[2] + wsum[3];
  __syncthreads();
  if (blockIdx.x == 0 && tid == 0) out_len[g] = (int)(strict_total + min(ties_total, need));
  const size_t n = (size_t)a.N * kF;
  const float4* ag = reinterpret_cast<const float4*>(a.act + (size_t)g * n);
  for (int r = blockIdx.x; r < a.tie_blocks; r += gridDim.x) {  // uniform
    unsigned bs = 0, bt = 0;
    for (int j = tid; j < r; j += kUT) {
      bs += tc[2 * j];
      bt += tc[2 * j + 1];
    }
    block_incl_scan<kUT>(bs, wsum);
    unsigned at_s = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    __syncthreads();
    block_incl_scan<kUT>(bt, wsum);
    unsigned at_t = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    __syncthreads();
    const size_t lo = min(n, (size_t)r * a.tie_len), hi = min(n, lo + a.tie_len);
    for (size_t base = lo / 4; base < hi / 4; base += kUT) {  // uniform
      const size_t i = base + tid;
      const float4 v = i < hi / 4 ? ag[i] : make_float4(0.f, 0.f, 0.f, 0.f);
      const float vv[4] = {v.x, v.y, v.z, v.w};
      bool hs[4], ht[4];
      unsigned cs = 0, ct = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        hs[j] = i < hi / 4 && rule.strict(vv[j]);
        ht[j] = i < hi / 4 && rule.tie(vv[j]);
        cs += hs[j];
        ct += ht[j];
      }
      const unsigned is = block_incl_scan<kUT>(cs, wsum);
      const unsigned ts = wsum[0] + wsum[1] + wsum[2] + wsum[3];
      __syncthreads();
      const unsigned it = block_incl_scan<kUT>(ct, wsum);
      const unsigned tt = wsum[0] + wsum[1] + wsum[2] + wsum[3];
      __syncthreads();
      unsigned ks = at_s + is - cs, kt = at_t + it - ct;  // ranks of this thread's first strict value / tie
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int64_t flat = (int64_t)(4 * i + j);
        if (hs[j]) out[ks++] = flat;
        if (ht[j]) {
          if (kt < need) out[strict_total + kt] = flat;
          ++kt;
        }
      }
      at_s += ts;
      at_t += tt;
    }
  }
}

}  // namespace
}  // namespace prismkv

using namespace prismkv;

// Work layout (bytes) for `groups` groups and blocks of N keys: the regions
// that must start at zero (histograms, control words) and the other scratch
// first, at offsets that depend on the group count only, then the block's
// activations [groups][N][3000] f32 and the compact candidate list
// [groups][list_cap] (sized by N).  A workspace sized for the largest block
// therefore serves every smaller block: no call finds another call's
// activations or list where it expects zeroed histograms.
struct UpdateLayout {
  size_t hist, ctl, tcount, part, wsplit, sample, act, list, ties, total;
  unsigned list_cap;
  UpdateLayout(int groups, int N) {
    size_t o = 0;
    auto take = [&](size_t n) { const size_t at = o; o += (n + 255) & ~(size_t)255; return at; };
    hist = take((size_t)groups * kLevels * kRep * kBins * sizeof(unsigned));
    ctl = take((size_t)groups * kCtl * sizeof(unsigned));
    tcount = take((size_t)groups * kMaxTieBlocks * 2 * sizeof(unsigned));
    part = take((size_t)groups * kCenterParts * kD * sizeof(double));
    wsplit = take((size_t)groups * kFTiles * kWTile * sizeof(_Float16));
    sample = take((size_t)groups * kSampleBins * sizeof(unsigned));
    act = take((size_t)groups * N * kF * sizeof(float));
    // the candidate list: six times the 8 N budget of an index build, at least 2^19
    list_cap = N > 0 ? std::max(1u << 19, (unsigned)kListPerKey * (unsigned)N + kListSlack) : 0u;
    list = take((size_t)groups * list_cap * sizeof(uint2));
    ties = take((size_t)groups * list_cap * sizeof(unsigned));
    total = o;
  }
};

static UpdateArgs make_args(uint64_t k, uint64_t W, uint64_t b, uint64_t center, uint64_t scale, uint64_t bits,
                            uint64_t counts, uint64_t moments, uint64_t work, int groups, int H, int N, int key_mean,
                            int64_t ks, int64_t row_words, const UpdateLayout& L) {
  char* w = reinterpret_cast<char*>(work);
  UpdateArgs a;
  a.k = reinterpret_cast<const void*>(k);
  a.ks = ks;
  a.W = reinterpret_cast<const float*>(W);
  a.b = reinterpret_cast<const float*>(b);
  a.center = reinterpret_cast<const float*>(center);
  a.scale = reinterpret_cast<const float*>(scale);
  a.bits = reinterpret_cast<uint32_t*>(bits);
  a.row_words = row_words;
  a.counts = reinterpret_cast<int*>(counts);
  a.moments = reinterpret_cast<float*>(moments);
  a.act = reinterpret_cast<float*>(w + L.act);
  a.wsplit = reinterpret_cast<_Float16*>(w + L.wsplit);
  a.hist = reinterpret_cast<unsigned*>(w + L.hist);
  a.ctl = reinterpret_cast<unsigned*>(w + L.ctl);
  a.tcount = reinterpret_cast<unsigned*>(w + L.tcount);
  a.list = reinterpret_cast<uint2*>(w + L.list);
  a.list_cap = L.list_cap;
  a.sample = reinterpret_cast<unsigned*>(w + L.sample);
  a.ties = reinterpret_cast<unsigned*>(w + L.ties);
  a.listed = 0;
  a.fine = 0;
  a.target = 0;
  a.H = H;
  a.N = N;
  a.budget = (long long)N * key_mean;
  // ordered-tie ranges: at most kMaxTieBlocks per group, each a multiple of 4 * kUT values
  const long long n = (long long)N * kF;
  long long len = std::max<long long>(kTieMinLen, (n + kMaxTieBlocks - 1) / kMaxTieBlocks);
  len = (len + 4 * kUT - 1) / (4 * kUT) * (4 * kUT);
  a.tie_len = len;
  a.tie_blocks = (int)((n + len - 1) / len);
  (void)groups;
  return a;
}

// Token ranges R of an encode: one workgroup runs per CU, so a launch takes
// rounds of 256 of its 6 G R workgroups, each its 16-token steps plus about six
// steps' time to load its W, find the floor and split its first rows; of the
// R that fill 1 .. 8 rounds the one of the least total.
static int encode_ranges(int N, int groups) {
  const long long blocks = (N + 15) / 16, per = (long long)groups * kEParts;
  long long best = 1, least = -1;
  for (int q = 1; q <= 8; ++q) {
    const long long r = std::min(blocks, std::max(1ll, 256ll * q / per));
    const long long cost = (per * r + 255) / 256 * ((blocks + r - 1) / r + 6);
    if (least < 0 || cost < least) {
      least = cost;
      best = r;
    }
  }
  return (int)best;
}

// Sample tokens of a call over N keys: every key up to 128, 128 of up to 4096
// (the count at the floor is then good to a few percent, whatever N is), 256 of
// up to 16384, 1/64 beyond, at most 2048.
static int sample_tokens(int N) {
  if (N <= kSelectMax) return std::min(N, kSampleFew);
  return std::min(2048, std::max(2 * kSampleFew, N / 64 / (2 * kSampleFew) * (2 * kSampleFew)));
}

// sample .. emit: the exact batch-wide positive Top-k of the N keys' activations
// and their bitmap bits.  `keep`: the activations are left in the workspace.
template <typename KT>
static void launch_selection(UpdateArgs a, int groups, bool keep, hipStream_t s) {
  // Candidates are collected when the list holds three times the budget and what
  // the floor is expected to let through: it aims at 2 (select) or 1.5 times the
  // budget, with up to 28% of a bin's width on top, but counts one value of each 16
  // buckets: at p values per bucket a token counts 188 (1 - (1 - p)^16) of its 3000 p.
  // (1024 keys at 100 memberships each: a floor that no sample reaches, every positive
  // value collected and the list of no use, 1812 us; without candidates 189.)
  const double aim = (a.N <= kSelectMax ? 2.0 : 1.5) * (double)(a.budget / a.N), lanes = kF / 16.0;
  const double expected = aim < 0.8 * lanes ? 1.15 * kF * (1.0 - std::pow(1.0 - aim / lanes, 1.0 / 16)) * a.N : INFINITY;
  a.listed = 3 * a.budget <= (long long)a.list_cap && expected <= (double)a.list_cap;
  const int S = a.listed ? sample_tokens(a.N) : 0;
  const bool one = a.listed && a.N <= kSelectMax;
  a.fine = one;
  a.target = (unsigned)((one ? 4 : 3) * ((long long)S * (a.budget / a.N)) / 2);
  const dim3 grid(groups, kEParts, encode_ranges(a.N, groups));
  // 16 tokens per wave while that is one workgroup per tile: all 8 waves share the
  // rows' splitting, where 32 left it to four (1024 keys: 19.5 us, now 14); beyond,
  // 32, as every workgroup splits its W tile again
  if (S <= kSampleFew)
    hipLaunchKernelGGL((sample_kernel<KT, 1>), dim3(1, kFTiles, groups), dim3(kET), 0, s, a, S);
  else
    hipLaunchKernelGGL((sample_kernel<KT, 2>), dim3((S + 2 * kSampleFew - 1) / (2 * kSampleFew), kFTiles, groups), dim3(kET),
                       0, s, a, S);
  if (a.listed && keep) {
    hipLaunchKernelGGL((encode_kernel<KT, true, true>), grid, dim3(kET), 0, s, a);
  } else {
    if (a.listed) hipLaunchKernelGGL((encode_kernel<KT, false, true>), grid, dim3(kET), 0, s, a);
    hipLaunchKernelGGL((encode_kernel<KT, true, false>), grid, dim3(kET), 0, s, a);
  }
  if (one) {
    hipLaunchKernelGGL(split_kernel, dim3(kSplitBlocks, groups), dim3(kUT), 0, s, a);
    hipLaunchKernelGGL(select_kernel, dim3(groups, kSelectBlocks), dim3(kST), 0, s, a);
  } else {
    hipLaunchKernelGGL(hist0_kernel, dim3(kRefineBlocks, groups), dim3(kUT), 0, s, a);
    hipLaunchKernelGGL(digit_kernel, dim3(groups), dim3(kUT), 0, s, a, 0);
    for (int level = 1; level < kLevels; ++level) {
      hipLaunchKernelGGL(refine_kernel, dim3(kRefineBlocks, groups), dim3(kUT), 0, s, a, level);
      hipLaunchKernelGGL(digit_kernel, dim3(groups), dim3(kUT), 0, s, a, level);
    }
    hipLaunchKernelGGL(tie_count_kernel, dim3(kTieGrid, groups), dim3(kUT), 0, s, a);
    hipLaunchKernelGGL(tie_cut_kernel, dim3(groups), dim3(kST), 0, s, a);
    hipLaunchKernelGGL(emit_kernel, dim3(kRefineBlocks, groups), dim3(kUT), 0, s, a);
  }
}

template <typename KT>
static void launch_build_moments(const UpdateArgs& a, int groups, hipStream_t s) {
  // a budget that fills most buckets past a wave's list goes to whole workgroups at once
  // (64 per key of 32768: 4.34 ms, 4.59 by way of the other two launches)
  if (a.N <= kSmallBuild && a.budget <= (long long)kF * BuildMomentsLds<64>::kLen) {
    hipLaunchKernelGGL((build_moments_kernel<KT, 64>), dim3(kF, groups), dim3(64), 0, s, a);
    hipLaunchKernelGGL(build_moments_rest_kernel<KT>, dim3(kF, groups), dim3(kUT), 0, s, a);
  } else
    hipLaunchKernelGGL((build_moments_kernel<KT, kUT>), dim3(kF, groups), dim3(kUT), 0, s, a);
}

template <typename KT>
static bool aligned16(uint64_t p, int64_t stride_elems) {
  return ((p | (uint64_t)(stride_elems * (int64_t)sizeof(KT))) & 15u) == 0;
}

template <typename KT>
static int update_impl(uint64_t k, uint64_t W, uint64_t b, uint64_t center, uint64_t scale, uint64_t bits,
                       uint64_t counts, uint64_t moments, uint64_t work, int groups, int H, int N, int key_mean,
                       int64_t ks, int64_t row_words, size_t work_bytes, uint64_t stream) {
  if (groups < 1 || groups > 65535 || H < 0 || N < 1 || N > kMaxBlock || key_mean < 1 || key_mean > kF)
    return kBadSize;
  if (ks < (int64_t)(H + N) * kD || row_words < (H + N + 31) / 32) return kBadSize;
  if (!k || !W || !b || !center || !scale || !bits || !counts || !moments || !work) return kBadSize;
  if (!aligned16<KT>(k, ks) || ((W | b) & 15u)) return kBadSize;
  const UpdateLayout L(groups, N);
  if (work_bytes < L.total) return kBadSize;  // prismkv_update_work_bytes(groups, N)
  const UpdateArgs a = make_args(k, W, b, center, scale, bits, counts, moments, work, groups, H, N, key_mean, ks,
                                 row_words, L);
  hipStream_t s = (hipStream_t)stream;
  launch_selection<KT>(a, groups, true, s);
  hipLaunchKernelGGL(moments_kernel<KT>, dim3(kChunks, groups), dim3(kMT), 0, s, a);
  return (int)hipGetLastError();
}

template <typename KT>
static int build_impl(uint64_t k, uint64_t W, uint64_t b, uint64_t center, uint64_t scale, uint64_t bits,
                      uint64_t counts, uint64_t moments, uint64_t work, int groups, int batch, int H, int key_mean,
                      int flags, int64_t ks, int64_t row_words, size_t work_bytes, uint64_t stream) {
  if (groups < 1 || groups > 65535 || batch < 1 || batch > groups || H < 1 || H > kMaxBuild || key_mean < 1 ||
      key_mean > kF)
    return kBadSize;
  if (flags & ~(kBuildCenter | kBuildNoAct)) return kBadMode;
  if (ks < (int64_t)H * kD || row_words < (H + 31) / 32 || (row_words & 3)) return kBadSize;
  if (!k || !W || !b || !center || !scale || !bits || !counts || !moments || !work) return kBadSize;
  if (!aligned16<KT>(k, ks) || ((bits | W | b) & 15u)) return kBadSize;
  const UpdateLayout L(batch, H);
  if (work_bytes < L.total) return kBadSize;  // prismkv_build_work_bytes(batch, H)
  hipStream_t s = (hipStream_t)stream;
  for (int g0 = 0; g0 < groups; g0 += batch) {
    const int nb = std::min(batch, groups - g0);
    const uint64_t kg = k + (uint64_t)g0 * ks * sizeof(KT);
    const uint64_t cg = center + (uint64_t)g0 * kD * sizeof(float);
    UpdateArgs a = make_args(kg, W + (uint64_t)g0 * kF * kD * sizeof(float), b + (uint64_t)g0 * kF * sizeof(float),
                             cg, scale + (uint64_t)g0 * sizeof(float),
                             bits + (uint64_t)g0 * kF * row_words * sizeof(uint32_t),
                             counts + (uint64_t)g0 * kFP * sizeof(int),
                             moments + (uint64_t)g0 * kChunks * kRow * kChunk * sizeof(float), work, nb, 0, H,
                             key_mean, ks, row_words, L);
    if (flags & kBuildCenter) {
      double* part = reinterpret_cast<double*>(reinterpret_cast<char*>(work) + L.part);
      hipLaunchKernelGGL(center_part_kernel<KT>, dim3(kCenterParts, nb), dim3(kUT), 0, s, a, part);
      hipLaunchKernelGGL(center_final_kernel, dim3(nb), dim3(kD), 0, s, a, (const double*)part,
                         reinterpret_cast<float*>(cg));
    }
    hipLaunchKernelGGL(clear_bits_kernel, dim3(512, nb), dim3(kUT), 0, s, a);
    launch_selection<KT>(a, nb, !(flags & kBuildNoAct), s);
    launch_build_moments<KT>(a, nb, s);
  }
  return (int)hipGetLastError();
}

template <typename KT>
static int summarize_impl(uint64_t k, uint64_t bits, uint64_t center, uint64_t counts, uint64_t moments,
                          uint64_t work, int groups, int H, int flags, int64_t ks, int64_t row_words,
                          size_t work_bytes, uint64_t stream) {
  if (groups < 1 || groups > 65535 || H < 1 || H > kMaxBuild) return kBadSize;
  if (flags & ~kBuildCenter) return kBadMode;
  if (ks < (int64_t)H * kD || row_words < (H + 31) / 32) return kBadSize;
  if (!k || !bits || !center || !counts || !moments || !work || !aligned16<KT>(k, ks)) return kBadSize;
  const UpdateLayout L(groups, 0);
  if (work_bytes < L.total) return kBadSize;  // prismkv_summarize_work_bytes(groups)
  const UpdateArgs a = make_args(k, 0, 0, center, 0, bits, counts, moments, work, groups, 0, H, 1, ks, row_words, L);
  hipStream_t s = (hipStream_t)stream;
  if (flags & kBuildCenter) {
    double* part = reinterpret_cast<double*>(reinterpret_cast<char*>(work) + L.part);
    hipLaunchKernelGGL(center_part_kernel<KT>, dim3(kCenterParts, groups), dim3(kUT), 0, s, a, part);
    hipLaunchKernelGGL(center_final_kernel, dim3(groups), dim3(kD), 0, s, a, (const double*)part,
                       reinterpret_cast<float*>(center));
  }
  launch_build_moments<KT>(a, groups, s);
  return (int)hipGetLastError();
}

extern "C" {

size_t prismkv_update_work_bytes(int groups, int max_block) {
  if (groups < 1 || groups > 65535 || max_block < 1 || max_block > kMaxBlock) return 0;
  return UpdateLayout(groups, max_block).total;
}

size_t prismkv_update_act_offset(int groups) {
  if (groups < 1 || groups > 65535) return 0;
  return UpdateLayout(groups, 0).act;
}

int prismkv_update(uint64_t k, uint64_t W, uint64_t b, uint64_t center, uint64_t scale, uint64_t bits,
                   uint64_t counts, uint64_t moments, uint64_t work, int groups, int H, int N, int key_mean,
                   int64_t ks, int64_t row_words, size_t work_bytes, uint64_t stream) {
  return update_impl<uint16_t>(k, W, b, center, scale, bits, counts, moments, work, groups, H, N, key_mean, ks,
                               row_words, work_bytes, stream);
}

int prismkv_update_f32(uint64_t k, uint64_t W, uint64_t b, uint64_t center, uint64_t scale, uint64_t bits,
                       uint64_t counts, uint64_t moments, uint64_t work, int groups, int H, int N, int key_mean,
                       int64_t ks, int64_t row_words, size_t work_bytes, uint64_t stream) {
  return update_impl<float>(k, W, b, center, scale, bits, counts, moments, work, groups, H, N, key_mean, ks,
                            row_words, work_bytes, stream);
}

size_t prismkv_build_work_bytes(int batch, int H) {
  if (batch < 1 || batch > 65535 || H < 1 || H > kMaxBuild) return 0;
  return UpdateLayout(batch, H).total;
}

int prismkv_build(uint64_t k, uint64_t W, uint64_t b, uint64_t center, uint64_t scale, uint64_t bits,
                  uint64_t counts, uint64_t moments, uint64_t work, int groups, int batch, int H, int key_mean,
                  int flags, int64_t ks, int64_t row_words, size_t work_bytes, uint64_t stream) {
  return build_impl<uint16_t>(k, W, b, center, scale, bits, counts, moments, work, groups, batch, H, key_mean, flags,
                              ks, row_words, work_bytes, stream);
}

int prismkv_build_f32(uint64_t k, uint64_t W, uint64_t b, uint64_t center, uint64_t scale, uint64_t bits,
                      uint64_t counts, uint64_t moments, uint64_t work, int groups, int batch, int H, int key_mean,
                      int flags, int64_t ks, int64_t row_words, size_t work_bytes, uint64_t stream) {
  return build_impl<float>(k, W, b, center, scale, bits, counts, moments, work, groups, batch, H, key_mean, flags,
                           ks, row_words, work_bytes, stream);
}

size_t prismkv_topk_work_bytes(void) { return UpdateLayout(1, 0).total; }

int prismkv_topk(uint64_t act, uint64_t out, uint64_t out_len, uint64_t work, int N, int64_t count,
                 size_t work_bytes, uint64_t stream) {
  if (N < 1 || N > kMaxBuild || count < 0) return kBadSize;
  if (!act || !out || !out_len || !work || (act & 15u)) return kBadSize;
  const UpdateLayout L(1, 0);
  if (work_bytes < L.total) return kBadSize;  // prismkv_topk_work_bytes()
  const int64_t n = (int64_t)N * kF;
  UpdateArgs a = make_args(0, 0, 0, 0, 0, 0, 0, 0, work, 1, 0, N, 1, 0, 0, L);
  a.act = reinterpret_cast<float*>(act);  // read only here
  a.budget = count < n ? count : n;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(hist0_kernel, dim3(kRefineBlocks, 1), dim3(kUT), 0, s, a);
  hipLaunchKernelGGL(digit_kernel, dim3(1), dim3(kUT), 0, s, a, 0);
  for (int level = 1; level < kLevels; ++level) {
    hipLaunchKernelGGL(refine_kernel, dim3(kRefineBlocks, 1), dim3(kUT), 0, s, a, level);
    hipLaunchKernelGGL(digit_kernel, dim3(1), dim3(kUT), 0, s, a, level);
  }
  const int grid = std::min(a.tie_blocks, kTieGrid);
  hipLaunchKernelGGL(flat_count_kernel, dim3(grid, 1), dim3(kUT), 0, s, a);
  hipLaunchKernelGGL(flat_emit_kernel, dim3(grid, 1), dim3(kUT), 0, s, a, reinterpret_cast<int64_t*>(out),
                     reinterpret_cast<int*>(out_len));
  return (int)hipGetLastError();
}

size_t prismkv_summarize_work_bytes(int groups) {
  if (groups < 1 || groups > 65535) return 0;
  return UpdateLayout(groups, 0).total;
}

int prismkv_summarize(uint64_t k, uint64_t bits, uint64_t center, uint64_t counts, uint64_t moments, uint64_t work,
                      int groups, int H, int flags, int64_t ks, int64_t row_words, size_t work_bytes,
                      uint64_t stream) {
  return summarize_impl<uint16_t>(k, bits, center, counts, moments, work, groups, H, flags, ks, row_words, work_bytes,
                                  stream);
}

int prismkv_summarize_f32(uint64_t k, uint64_t bits, uint64_t center, uint64_t counts, uint64_t moments,
                          uint64_t work, int groups, int H, int flags, int64_t ks, int64_t row_words,
                          size_t work_bytes, uint64_t stream) {
  return summarize_impl<float>(k, bits, center, counts, moments, work, groups, H, flags, ks, row_words, work_bytes,
                               stream);
}

}  // extern "C"
