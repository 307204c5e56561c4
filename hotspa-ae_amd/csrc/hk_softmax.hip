// Softmax forward / backward for gfx950.
//
// Last-dimension softmax keeps the row in registers (one HBM read, one write), whatever its length and alignment:
// lanes of one wavefront agree on the row's maximum and then its sum (DPP); where a row takes a workgroup, every
// thread folds its elements into a (max, sum-of-exp) pair and the pairs are merged online across wavefronts (LDS).
// The stored exponentials are rescaled on the way out, so exp is evaluated once per element.
// Bound by HBM: what a row costs is its bytes and, for ragged rows, the extra cache lines of misaligned accesses
// (192 x 577 x 577 bf16, forward + backward: 508 us with element-wise passes, 118 us with vectors counted from the row's start,
// 107 us with those of odd rows on 4-byte boundaries; stored through the cache, 110).
#include "hk_common.h"

#include <algorithm>

namespace hk {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegInf = -__builtin_huge_valf();

struct SoftmaxRows {
  const void* x;    // forward: input;  backward: y
  const void* dy;   // backward only
  void* out;        // forward: y;      backward: dx
  int64_t rows;
  int64_t x_pitch, dy_pitch, out_pitch;   // elements between row starts (== cols for a dense array)
  int64_t n0, n1, n2;                     // rows on several levels in walk order (see LevelSteps); one level: n0 = rows
  LevelSteps x_lv, dy_lv, out_lv;
  int cols;
  int nvec;
  int spare;        // see RaggedRow
};
// What the kernels take of it (see kCheapArgs).  Steps below 2^31 elements; what lies further apart goes out in several launches.
// What a row's loads wait for lies in the first 64 bytes, one line of the scalar cache, and takes few scalar instructions: every
// workgroup passes through them before its loads are under way.  Forward and backward, us, steps and counts of 64 bits / of 32 signed bits
// in any order / so: bf16 4 x 1024 x 4096 31.7 / 32.05 / 31.3, 16 x 512 x 1024 17.45 / 18.1 / 17.45, 16 x 577 x 577 14.67 / 14.76 / 14.31, fp32 32 x
// 256 x 256 10.67 / 10.45 / 10.2.
struct SoftmaxArgs {
  const void* x;
  const void* dy;
  int n0, nvec, cols;
  uint32_t x_pitch, dy_pitch;
  ShortLevelSteps x_lv, dy_lv;
  uint16_t threads;   // of a workgroup
  uint16_t spare;
  void* out;
  uint32_t out_pitch;
  ShortLevelSteps out_lv;
};
static_assert(sizeof(SoftmaxArgs) <= kCheapArgs, "");

template <typename T, int NV, int LPR, bool RAGGED>
__global__ __launch_bounds__(LPR ? 256 : 1024)
void softmax_fwd_kernel(SoftmaxArgs a) {
  constexpr int VEC = VecIO<T>::N;
  using Lanes = RowLanes<LPR>;
  __shared__ float red[kMaxWaves * 2];
  const int tpr = Lanes::count(a.threads), t = Lanes::lane();
  const int64_t row = Lanes::row();
  if (LPR && row >= a.n0) return;   // row counts within the innermost level

  const T* xr = static_cast<const T*>(a.x) + row * a.x_pitch + outer_level_offset(a.x_lv);
  // slots past the row's end hold -inf, which changes neither the maximum nor the sum; in a ragged row they hold
  // elements of the row a second time, which the maximum may see and the sum leaves out
  [[maybe_unused]] const RaggedRow<T, true> odd(xr, a.cols, a.spare);
  u32x4 raw[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int v = i * tpr + t;
    if constexpr (RAGGED) {
      raw[i] = ld16_any<T>(xr + odd.column(v));
    } else if ((i + 1) * tpr <= a.nvec) {       // uniform: every thread's slot i is inside the row
      raw[i] = ld16(xr + v * VEC);
    } else {
      raw[i] = neg_inf_vec<T>();
      if (v < a.nvec) raw[i] = ld16(xr + v * VEC);
    }
  }
  float e[NV * VEC];
#pragma unroll
  for (int i = 0; i < NV; ++i) VecIO<T>::unpack(raw[i], &e[i * VEC]);
  static_assert((NV * VEC) % 2 == 0, "pairs of elements per max3");
  float m = fmaxf(e[0], e[1]);
#pragma unroll
  for (int k = 2; k < NV * VEC; k += 2) m = max3(m, e[k], e[k + 1]);
  // ml: the maximum in the log2 domain, rounded once (see OnlineSoftmaxTuple).  Lanes of one wavefront agree on the
  // row's maximum first: its butterfly is cheaper than merging (maximum, sum) pairs, whose every step takes two
  // exponentials, and an element held twice then comes out the same twice.  Across wavefronts each thread keeps its
  // own maximum and the pairs are merged, which costs one barrier instead of two.
  if constexpr (LPR > 0) m = Lanes::allreduce(MaxTuple{{m}}, red, a.threads).v[0];
  // A row whose maximum lies at the type's lowest values (scores masked with it) or at its highest would overflow in the
  // log2 domain: two different values out there are so far apart that any base gives 1 at the maximum and 0 elsewhere, so
  // lanes that agree on the row's maximum take base 2 for such a row.  A whole workgroup's threads have maxima of their
  // own, kept finite by log2_of_max(), and the row is counted below.
  const float k = (LPR > 0 && fabsf(m) > 2.3e38f) ? 1.0f : kLog2e;
  const float ml = LPR > 0 ? m * k : log2_of_max(m);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    [[maybe_unused]] const int skip = odd.skip(i * tpr + t);   // elements of earlier vectors (ragged)
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      float& x = e[i * VEC + j];
      x = __builtin_amdgcn_exp2f(fmaf(x, k, -ml));
      s += (RAGGED && j < skip) ? 0.f : x;
    }
  }
  T* yr = static_cast<T*>(a.out) + row * a.out_pitch + outer_level_offset(a.out_lv);
  float scale;
  if constexpr (LPR > 0) {
    scale = 1.0f / Lanes::allreduce(SumTuple<1>{{s}}, red, a.threads).v[0];
  } else {
    MaxSumTuple p;
    p.v[0] = ml; p.v[1] = s;
    p = Lanes::allreduce(p, red, a.threads);
    if (past_log2_range(p.v[0])) {   // uniform
      float M;
      const float n = row_max_count<T>(xr, a.cols, t, tpr, [&](auto v) {
        __syncthreads();   // red may still be read
        return Lanes::allreduce(v, red, a.threads);
      }, M);
      const float inv = 1.0f / (M == kNegInf ? __builtin_nanf("") : n);   // nothing but -inf has no softmax
      for (int c = t; c < a.cols; c += tpr) Cvt<T>::store(yr + c, (Cvt<T>::load(xr + c) == M ? 1.f : 0.f) * inv);
      return;
    }
    scale = __builtin_amdgcn_exp2f(ml - p.v[0]) / p.v[1];
  }

#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int v = i * tpr + t;
    if (RAGGED ? odd.live(v) : v < a.nvec) {
#pragma unroll
      for (int j = 0; j < VEC; ++j) e[i * VEC + j] *= scale;
      if constexpr (RAGGED) odd.template store<(LPR > 0)>(yr, v, &e[i * VEC]);
      else st16_stream(yr + v * VEC, VecIO<T>::pack(&e[i * VEC]));
    }
  }
}

template <typename T, int NV, int LPR, bool RAGGED>
__global__ __launch_bounds__(LPR ? 256 : 1024)
void softmax_bwd_kernel(SoftmaxArgs a) {
  constexpr int VEC = VecIO<T>::N;
  using Lanes = RowLanes<LPR>;
  __shared__ float red[kMaxWaves];
  const int tpr = Lanes::count(a.threads), t = Lanes::lane();
  const int64_t row = Lanes::row();
  if (LPR && row >= a.n0) return;   // row counts within the innermost level

  const T* yr = static_cast<const T*>(a.x) + row * a.x_pitch + outer_level_offset(a.x_lv);
  const T* dyr = static_cast<const T*>(a.dy) + row * a.dy_pitch + outer_level_offset(a.dy_lv);
  [[maybe_unused]] const RaggedRow<T, true> odd(yr, a.cols, a.spare);
  u32x4 ry[NV], rdy[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int v = i * tpr + t;
    if constexpr (RAGGED) {
      const int c = odd.column(v);
      ry[i] = ld16_any<T>(yr + c);
      rdy[i] = ld16_any<T>(dyr + c);
    } else {
      ry[i] = u32x4{0, 0, 0, 0};
      rdy[i] = u32x4{0, 0, 0, 0};
      if (v < a.nvec) { ry[i] = ld16(yr + v * VEC); rdy[i] = ld16(dyr + v * VEC); }
    }
  }
  SumTuple<1> s;
  s.v[0] = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    float y[VEC], d[VEC];
    VecIO<T>::unpack(ry[i], y);
    VecIO<T>::unpack(rdy[i], d);
    [[maybe_unused]] const int skip = odd.skip(i * tpr + t);
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      if constexpr (RAGGED) s.v[0] = j < skip ? s.v[0] : fmaf(y[j], d[j], s.v[0]);
      else s.v[0] = fmaf(y[j], d[j], s.v[0]);   // padding is zero
    }
  }
  s = Lanes::allreduce(s, red, a.threads);
  const float dot = s.v[0];
  T* dxr = static_cast<T*>(a.out) + row * a.out_pitch + outer_level_offset(a.out_lv);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int v = i * tpr + t;
    if (RAGGED ? odd.live(v) : v < a.nvec) {
      float y[VEC], d[VEC];
      VecIO<T>::unpack(ry[i], y);
      VecIO<T>::unpack(rdy[i], d);
#pragma unroll
      for (int j = 0; j < VEC; ++j) d[j] = y[j] * (d[j] - dot);
      if constexpr (RAGGED) odd.template store<true>(dxr, v, d);
      else st16_stream(dxr + v * VEC, VecIO<T>::pack(d));
    }
  }
}

// Softmax along a dimension other than the last, [outer, dim, inner].  A lane holds one 16-byte vector of neighbouring
// inner positions; the dimension is cut into slices of NK entries, LX lanes per slice, so that the whole column stays in
// registers: one read, one write.  Slices agree on the maximum and the sum through LDS.  The partial last vector of a
// plane is read as its last whole one, its own elements are stored one by one (in place, a neighbour may have replaced
// the others before they were read).
// Bound by HBM, by how many workgroups a compute unit has under way (one loads while another stores: hence at most 512
// threads a workgroup where the plan does not say otherwise) and, on odd planes, by the cache lines that neighbouring
// workgroups share: runs of 8 or 16 of them stay on one XCD, whose L2 then sees each line whole.  Forward / backward, us:
// 8 x 21 x 263169 fp32 66 / 94 (5.4 and 5.6 TB/s), 263168 62 / 89; 232 x 21 x 16384 bf16 52.6 / 75.5 (6.1 and 6.4 TB/s).
// AGAIN: the compiler keeps what it has formed of the vectors, exponentials or unpacked elements in fp32, from one step to the next.
// That is the faster program while it fits (10 entries of bf16 forward 118 registers, of which 40 hold them as loaded; 32 x 150 x
// 16384 56 us kept, 60 formed again).  Past it, it costs a compute unit its second workgroup or spills (12 forward 136 registers, 16
// backward 256 and 41 spilled), and what is needed again is formed again: forward 25 x 256 x 12101 87 -> 77, backward 19 x 256 x 16384
// 152 -> 85, 38 x 128 x 16384 87 -> 81.
constexpr int kDimVecs = 8;      // most entries per lane of a wavefront's run; of half a wavefront's, 16
// f[0..N): this lane's values; on return the slices' maximum or sum (in slice order) of each, the same in every slice.
// lds: [slices + 1][LX * N].  A thread merges the slices of one value (every thread merging all of its lane's values
// takes slices * N steps: 65 entries of 355 bf16 positions 9.0 us, so 5.5); calls may follow one another.
template <int N, int LX> __device__ __forceinline__ void slices_share(float* f, float* lds, int slices, bool take_max) {
  u32x4* mine = reinterpret_cast<u32x4*>(lds + (int(threadIdx.y) * LX + int(threadIdx.x)) * N);
#pragma unroll
  for (int q = 0; q < N / 4; ++q) mine[q] = u32x4{f2u(f[4 * q]), f2u(f[4 * q + 1]), f2u(f[4 * q + 2]), f2u(f[4 * q + 3])};
  __syncthreads();
  float* merged = lds + slices * LX * N;
  for (int i = int(threadIdx.y) * LX + int(threadIdx.x); i < LX * N; i += slices * LX) {
    float r = lds[i];
#pragma unroll 4
    for (int s = 1; s < slices; ++s) {
      const float o = lds[s * LX * N + i];
      r = take_max ? fmaxf(r, o) : r + o;
    }
    merged[i] = r;
  }
  __syncthreads();
  const u32x4* got = reinterpret_cast<const u32x4*>(merged + int(threadIdx.x) * N);
#pragma unroll
  for (int q = 0; q < N / 4; ++q) {
    const u32x4 o = got[q];
#pragma unroll
    for (int j = 0; j < 4; ++j) f[4 * q + j] = u2f(o[j]);
  }
}

// The same for few slices: every thread merges its own lane's values, without a second barrier and without the merged copy, in
// the same order (4 x 5 x 5904 bf16 forward 3.7 -> 3.0 us).
// lds: [slices][N / 4][LX] 16-byte vectors; a call that follows another takes an area of its own.
template <int N, int LX> __device__ __forceinline__ void few_slices_share(float* f, float* lds, int slices, bool take_max) {
  u32x4* area = reinterpret_cast<u32x4*>(lds) + int(threadIdx.x);
#pragma unroll
  for (int q = 0; q < N / 4; ++q)
    area[(int(threadIdx.y) * (N / 4) + q) * LX] = u32x4{f2u(f[4 * q]), f2u(f[4 * q + 1]), f2u(f[4 * q + 2]), f2u(f[4 * q + 3])};
  __syncthreads();
#pragma unroll
  for (int q = 0; q < N / 4; ++q) {
    const u32x4 o = area[q * LX];
#pragma unroll
    for (int j = 0; j < 4; ++j) f[4 * q + j] = u2f(o[j]);
  }
  for (int s = 1; s < slices; ++s) {
#pragma unroll
    for (int q = 0; q < N / 4; ++q) {
      const u32x4 o = area[(s * (N / 4) + q) * LX];
#pragma unroll
      for (int j = 0; j < 4; ++j) f[4 * q + j] = take_max ? fmaxf(f[4 * q + j], u2f(o[j])) : f[4 * q + j] + u2f(o[j]);
    }
  }
}
constexpr int kFewSlices = 6;
// LDS of a workgroup, in floats: the forward shares twice
template <int N, int LX, bool FEW, bool BWD>
static inline size_t share_floats(int slices) {
  return size_t(FEW ? (BWD ? slices : 2 * slices) : slices + 1) * LX * N;
}
template <int N, int LX, bool FEW>
__device__ __forceinline__ void share(float* f, float* lds, int slices, bool take_max, int call) {
  if (slices <= 1) return;   // uniform
  if constexpr (FEW) few_slices_share<N, LX>(f, lds + call * slices * LX * N, slices, take_max);
  else slices_share<N, LX>(f, lds, slices, take_max);
}

struct SoftmaxDimArgs {
  const void* x;       // forward: input;  backward: y
  const void* dy;
  void* out;
  int64_t inner, total;   // total: vectors of all planes, outer * run_vecs
  int dim, run_vecs, slices;
  int blocks;             // of the launch
};
static_assert(sizeof(SoftmaxDimArgs) <= kCheapArgs, "");
// What is formed from these vectors after this point is formed from them again, not kept in registers since before it.
template <int N>
__device__ __forceinline__ void form_again(u32x4 (&raw)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k) asm volatile("" : "+v"(raw[k]));
}
// this lane's column: element offset of its vector in entry 0 of the plane, its place in the run, whether it exists
template <typename T, int LX>
struct DimColumn {
  int64_t base;
  int v, first, count;
  bool live;
  __device__ __forceinline__ DimColumn(const SoftmaxDimArgs& a, int nk) {
    const int64_t id = xcd_run_block<LX == 256 ? 8 : 16>(blockIdx.x, uint32_t(a.blocks)) * LX + int(threadIdx.x);
    live = id < a.total;
    const uint32_t i = uint32_t(live ? id : a.total - 1), o = i / uint32_t(a.run_vecs);
    v = int(i - o * uint32_t(a.run_vecs));
    base = int64_t(o) * a.dim * a.inner + vec_column<T, true>(v, int(a.inner));
    // a slice of whole wavefronts: its entries' addresses are scalar
    first = (LX >= kWave ? __builtin_amdgcn_readfirstlane(int(threadIdx.y)) : int(threadIdx.y)) * nk;
    count = min(nk, a.dim - first);        // entries of this slice, at least one
  }
};

template <typename T, int NK, int LX, bool PLAIN, bool FEW, int MAXT, bool AGAIN>
__global__ __launch_bounds__(MAXT)
void softmax_fwd_dim_kernel(SoftmaxDimArgs a) {
  constexpr int VEC = VecIO<T>::N;
  extern __shared__ __align__(16) float shared[];   // share_floats
  const DimColumn<T, LX> c(a, NK);
  const T* xp = static_cast<const T*>(a.x) + c.base;
  u32x4 raw[NK];
  // entries past the slice's end are its last one again: no change to the maximum, left out of the sum
#pragma unroll
  for (int k = 0; k < NK; ++k) raw[k] = ld16_any<T>(xp + int64_t(c.first + min(k, c.count - 1)) * a.inner);
  float m[VEC];
  VecIO<T>::unpack(raw[0], m);
#pragma unroll
  for (int k = 1; k < NK; k += 2) {
    float f[VEC], g[VEC];
    VecIO<T>::unpack(raw[k], f);
    VecIO<T>::unpack(raw[k + 1 < NK ? k + 1 : k], g);
#pragma unroll
    for (int j = 0; j < VEC; ++j) m[j] = max3(m[j], f[j], g[j]);
  }
  share<VEC, LX, FEW>(m, shared, a.slices, true, 0);
  if constexpr (AGAIN) form_again(raw);
  float base2[VEC], ml[VEC], s[VEC];
#pragma unroll
  for (int j = 0; j < VEC; ++j) {
    base2[j] = fabsf(m[j]) > 2.3e38f ? 1.0f : kLog2e;   // lowest or highest values, as in softmax_fwd_kernel
    ml[j] = m[j] * base2[j];
    s[j] = 0.f;
  }
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    float f[VEC];
    VecIO<T>::unpack(raw[k], f);
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const float e = __builtin_amdgcn_exp2f(fmaf(f[j], base2[j], -ml[j]));
      s[j] += k < c.count ? e : 0.f;
    }
  }
  share<VEC, LX, FEW>(s, shared, a.slices, false, 1);
  if constexpr (AGAIN) form_again(raw);
  if (!c.live) return;
#pragma unroll
  for (int j = 0; j < VEC; ++j) s[j] = 1.0f / s[j];
  T* yp = static_cast<T*>(a.out) + c.base - vec_column<T, true>(c.v, int(a.inner));   // the run's start
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    if (k < c.count) {
      float f[VEC];
      VecIO<T>::unpack(raw[k], f);
#pragma unroll
      for (int j = 0; j < VEC; ++j) f[j] = __builtin_amdgcn_exp2f(fmaf(f[j], base2[j], -ml[j])) * s[j];
      store_row_vec<T, true, false, PLAIN>(yp + int64_t(c.first + k) * a.inner, c.v, f, int(a.inner));
    }
  }
}

template <typename T, int NK, int LX, bool PLAIN, bool FEW, int MAXT, bool AGAIN>
__global__ __launch_bounds__(MAXT)
void softmax_bwd_dim_kernel(SoftmaxDimArgs a) {
  constexpr int VEC = VecIO<T>::N;
  extern __shared__ __align__(16) float shared[];   // share_floats
  const DimColumn<T, LX> c(a, NK);
  const T* yp = static_cast<const T*>(a.x) + c.base;
  const T* dyp = static_cast<const T*>(a.dy) + c.base;
  u32x4 ry[NK], rd[NK];
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    const int64_t at = int64_t(c.first + min(k, c.count - 1)) * a.inner;
    ry[k] = ld16_any<T>(yp + at);
    rd[k] = ld16_any<T>(dyp + at);
  }
  float dot[VEC] = {};
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    float y[VEC], d[VEC];
    VecIO<T>::unpack(ry[k], y);
    VecIO<T>::unpack(rd[k], d);
#pragma unroll
    for (int j = 0; j < VEC; ++j) dot[j] = k < c.count ? fmaf(y[j], d[j], dot[j]) : dot[j];
  }
  share<VEC, LX, FEW>(dot, shared, a.slices, false, 0);
  if constexpr (AGAIN) { form_again(ry); form_again(rd); }
  if (!c.live) return;
  T* dxp = static_cast<T*>(a.out) + c.base - vec_column<T, true>(c.v, int(a.inner));
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    if (k < c.count) {
      float y[VEC], d[VEC];
      VecIO<T>::unpack(ry[k], y);
      VecIO<T>::unpack(rd[k], d);
#pragma unroll
      for (int j = 0; j < VEC; ++j) d[j] = y[j] * (d[j] - dot[j]);
      store_row_vec<T, true, false, PLAIN>(dxp + int64_t(c.first + k) * a.inner, c.v, d, int(a.inner));
    }
  }
}

// Softmax along a dimension of extent `dim` with element stride `inner`: longer dimensions than the kernels above take,
// shorter planes, those that softmax_strided_typed leaves to it, and fp64; for inner == 1, rows longer than a
// workgroup's registers hold or shorter than a vector, and fp64.
// One thread walks one (outer, inner) position, threads of a wave sit on
// neighbouring inner positions; for inner == 1 one workgroup takes one row.
template <typename T, typename CT>
struct SmIO {
  static __device__ __forceinline__ CT ld(const T* p) { return CT(Cvt<T>::load(p)); }
  static __device__ __forceinline__ void st(T* p, CT v) { Cvt<T>::store(p, v); }
};

template <typename CT> __device__ __forceinline__ CT exp_ct(CT v);
template <> __device__ __forceinline__ float exp_ct<float>(float v) { return __builtin_amdgcn_exp2f(v * kLog2e); }
template <> __device__ __forceinline__ double exp_ct<double>(double v) { return exp(v); }

template <typename T, typename CT>
__global__ __launch_bounds__(256)
void softmax_fwd_strided_kernel(const T* x, T* y, int64_t outer, int64_t dim, int64_t inner) {
  const int64_t pos = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (pos >= outer * inner) return;
  const int64_t o = pos / inner, in = pos - o * inner;
  const T* xp = x + o * dim * inner + in;
  T* yp = y + o * dim * inner + in;
  CT m = -__builtin_huge_val(), s = 0;
  for (int64_t k = 0; k < dim; ++k) {
    const CT v = SmIO<T, CT>::ld(xp + k * inner);
    m = v > m ? v : m;
  }
  for (int64_t k = 0; k < dim; ++k) s += exp_ct<CT>(SmIO<T, CT>::ld(xp + k * inner) - m);
  const CT inv = CT(1) / s;
  for (int64_t k = 0; k < dim; ++k)
    SmIO<T, CT>::st(yp + k * inner, exp_ct<CT>(SmIO<T, CT>::ld(xp + k * inner) - m) * inv);
}

template <typename T, typename CT>
__global__ __launch_bounds__(256)
void softmax_bwd_strided_kernel(const T* y, const T* dy, T* dx, int64_t outer, int64_t dim,
                                int64_t inner) {
  const int64_t pos = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (pos >= outer * inner) return;
  const int64_t o = pos / inner, in = pos - o * inner;
  const int64_t base = o * dim * inner + in;
  CT dot = 0;
  for (int64_t k = 0; k < dim; ++k)
    dot += SmIO<T, CT>::ld(y + base + k * inner) * SmIO<T, CT>::ld(dy + base + k * inner);
  for (int64_t k = 0; k < dim; ++k) {
    const CT yv = SmIO<T, CT>::ld(y + base + k * inner);
    SmIO<T, CT>::st(dx + base + k * inner, yv * (SmIO<T, CT>::ld(dy + base + k * inner) - dot));
  }
}

template <typename CT>
__device__ __forceinline__ CT block_reduce_generic(CT v, CT* lds, bool is_max) {
  const int tid = threadIdx.x;
  lds[tid] = v;
  __syncthreads();
  for (int s = 256 >> 1; s > 0; s >>= 1) {
    if (tid < s) lds[tid] = is_max ? (lds[tid] > lds[tid + s] ? lds[tid] : lds[tid + s])
                                   : lds[tid] + lds[tid + s];
    __syncthreads();
  }
  CT r = lds[0];
  __syncthreads();
  return r;
}

template <typename T, typename CT>
__global__ __launch_bounds__(256)
void softmax_fwd_longrow_kernel(const T* x, T* y, int64_t cols, int64_t x_pitch, int64_t y_pitch) {
  __shared__ CT lds[256];
  const T* xr = x + int64_t(blockIdx.x) * x_pitch;
  T* yr = y + int64_t(blockIdx.x) * y_pitch;
  CT m = -__builtin_huge_val();
  for (int64_t c = threadIdx.x; c < cols; c += 256) {
    const CT v = SmIO<T, CT>::ld(xr + c);
    m = v > m ? v : m;
  }
  m = block_reduce_generic<CT>(m, lds, true);
  CT s = 0;
  for (int64_t c = threadIdx.x; c < cols; c += 256) s += exp_ct<CT>(SmIO<T, CT>::ld(xr + c) - m);
  s = block_reduce_generic<CT>(s, lds, false);
  const CT inv = CT(1) / s;
  for (int64_t c = threadIdx.x; c < cols; c += 256)
    SmIO<T, CT>::st(yr + c, exp_ct<CT>(SmIO<T, CT>::ld(xr + c) - m) * inv);
}

template <typename T, typename CT>
__global__ __launch_bounds__(256)
void softmax_bwd_longrow_kernel(const T* y, const T* dy, T* dx, int64_t cols, int64_t y_pitch,
                                int64_t dy_pitch, int64_t dx_pitch) {
  __shared__ CT lds[256];
  const T* yr = y + int64_t(blockIdx.x) * y_pitch;
  const T* dyr = dy + int64_t(blockIdx.x) * dy_pitch;
  T* dxr = dx + int64_t(blockIdx.x) * dx_pitch;
  CT dot = 0;
  for (int64_t c = threadIdx.x; c < cols; c += 256)
    dot += SmIO<T, CT>::ld(yr + c) * SmIO<T, CT>::ld(dyr + c);
  dot = block_reduce_generic<CT>(dot, lds, false);
  for (int64_t c = threadIdx.x; c < cols; c += 256) {
    const CT yv = SmIO<T, CT>::ld(yr + c);
    SmIO<T, CT>::st(dxr + c, yv * (SmIO<T, CT>::ld(dyr + c) - dot));
  }
}

static inline int pow2_ceil_sm(int v) {
  int p = 1;
  while (p < v) p <<= 1;
  return p;
}

// lanes per row (threads of a workgroup per row when above 64) / vectors per lane for a row of nvec 16-byte vectors
// (aligned: whole vectors on 16-byte boundaries; odd: rows on odd 2-byte boundaries)
static bool pick_softmax_shape(int nvec, bool aligned, bool odd, int max_nv, bool bwd, int* threads, int* nv) {
  const int forced = tune_get(TUNE_SOFTMAX_THREADS);
  // measured on MI355X at 2048 bf16 columns: forward is fastest with two
  // vectors per thread (128 threads per row), backward with one (256 threads)
  const int want = bwd ? 1 : 2;
  // a forced width is rounded up to one that exists; a wavefront's lanes hold up to four vectors each
  if (forced > 0 && forced <= 64) {
    const int lanes = std::max(8, pow2_ceil_sm(forced)), n = (nvec + lanes - 1) / lanes;
    if (n <= 4) {
      *threads = lanes; *nv = n;
      return true;
    }
  }
  if (forced > 0) {
    int t = std::min(1024, std::max(128, (forced + 63) / 64 * 64));
    int n = pow2_ceil_sm((nvec + t - 1) / t);
    if (n > max_nv) return false;
    *threads = t; *nv = n;
    return true;
  }
  const bool whole_lines = aligned && nvec % 8 == 0;
  // Short rows share a wavefront: one to itself leaves most lanes of a short row idle, and the launch is then bound by
  // waves, not bytes.  Measured on arrays of 600 MB, bf16, forward / backward GB/s, one row per wavefront -> this
  // choice: 32 columns 680 / 1055 -> 4710 / 5150, 64: 1300 / 1990 -> 6500 / 6490, 128: 2390 / 3720 -> 6540 / 6470,
  // 256: 4440 / 5070 -> 6390 / 6490, 512: 6440 / 6440 -> 6380 / 6440.  What decides between the shapes:
  //  - the backward streams best with one vector of each operand per lane (1024 columns, 128 lanes x 1: 6560, 64 x 2:
  //    6180; 256 columns, 32 x 1: 6490, 16 x 2: 6200), the forward with two as long as no lane idles;
  //  - two vectors in half the lanes cover a short row forward only where it ends on a 128-byte line (200 columns
  //    5220 as 16 x 2, 5720 as 32 x 1);
  //  - rows on odd 2-byte boundaries, whose every access straddles lines, want a wavefront of their own up to 256
  //    vectors (2047 columns 5550 / 5950 against 5470 / 5410 with a workgroup); other backward rows do only where a
  //    workgroup of one vector per lane would leave two fifths of its lanes idle (300 fp32 columns 6110 against 5400).
  if (nvec <= 64) {
    *threads = nvec <= 8 ? 8 : (nvec <= 16 || (nvec <= 32 && whole_lines && !bwd)) ? 16
             : (nvec <= 40 || !bwd) ? 32 : 64;
    *nv = (nvec + *threads - 1) / *threads;
    return true;
  }
  if (nvec <= (odd ? 256 : bwd ? 76 : 192)) {
    *threads = 64;
    *nv = (nvec + 63) / 64;
    return true;
  }
  for (int n = want; n <= max_nv; n <<= 1) {
    int t = ((nvec + n - 1) / n + 63) / 64 * 64;
    if (t <= 1024) { *threads = t; *nv = n; return true; }
  }
  return false;
}

template <typename T, bool BWD, int LPR, bool RAGGED>
static int launch_softmax_nv(const SoftmaxArgs& a, int nv, dim3 grid, dim3 block, hipStream_t s) {
#define HK_SM_CASE(N)                                                                      \
  case N:                                                                                  \
    if constexpr (BWD) HK_LAUNCH((softmax_bwd_kernel<T, N, LPR, RAGGED>), grid, block, 0, s, a); \
    else HK_LAUNCH((softmax_fwd_kernel<T, N, LPR, RAGGED>), grid, block, 0, s, a);   \
    break;
  profile_before(s);
  switch (nv) {
    HK_SM_CASE(1) HK_SM_CASE(2) HK_SM_CASE(4)
    case 3:
      if constexpr (LPR > 0) {
        if constexpr (BWD) HK_LAUNCH((softmax_bwd_kernel<T, 3, LPR, RAGGED>), grid, block, 0, s, a);
        else HK_LAUNCH((softmax_fwd_kernel<T, 3, LPR, RAGGED>), grid, block, 0, s, a);
        break;
      }
      [[fallthrough]];
    case 8:
      if constexpr (!BWD && LPR == 0) {
        if (nv == 8) {
          HK_LAUNCH((softmax_fwd_kernel<T, 8, LPR, RAGGED>), grid, block, 0, s, a);
          break;
        }
      }
      [[fallthrough]];
    case 16:
      if constexpr (VecIO<T>::N == 4 && !BWD && LPR == 0) {
        if (nv == 16) {
          HK_LAUNCH((softmax_fwd_kernel<T, 16, LPR, RAGGED>), grid, block, 0, s, a);
          break;
        }
      }
      [[fallthrough]];
    default:
      set_last_error("softmax: no kernel for %d vectors per thread", nv);
      return HK_ERR_UNSUPPORTED;
  }
#undef HK_SM_CASE
  profile_after(s);
  return launch_check(BWD ? "softmax_bwd_kernel" : "softmax_fwd_kernel");
}

template <typename T, bool BWD, bool RAGGED>
static int launch_softmax(const SoftmaxRows& r, int threads, int nv, hipStream_t s) {
  const int64_t dy0 = BWD ? r.dy_pitch : 0, dy1 = BWD ? r.dy_lv.p1 : 0, dy2 = BWD ? r.dy_lv.p2 : 0;
  const bool far0 = far_level(r.n0, {r.x_pitch, dy0, r.out_pitch}), far1 = far_level(r.n1, {r.x_lv.p1, dy1, r.out_lv.p1}),
             far2 = far_level(r.n2, {r.x_lv.p2, dy2, r.out_lv.p2});
  if (far0 || far1 || far2) {
    return each_near_part(r, far0, far1, far2, [&](SoftmaxRows part, int64_t i, int64_t j, int64_t k) {
      const auto at = [&](int64_t pitch, const LevelSteps& l) { return i * pitch + j * l.p1 + k * l.p2; };
      part.x = static_cast<const T*>(r.x) + at(r.x_pitch, r.x_lv);
      if constexpr (BWD) part.dy = static_cast<const T*>(r.dy) + at(r.dy_pitch, r.dy_lv);
      part.out = static_cast<T*>(r.out) + at(r.out_pitch, r.out_lv);
      return launch_softmax<T, BWD, RAGGED>(part, threads, nv, s);
    });
  }
  const int rows_per_block = threads > 64 ? 1 : 256 / threads;
  const dim3 grid(unsigned((r.n0 + rows_per_block - 1) / rows_per_block), unsigned(r.n1), unsigned(r.n2));
  const dim3 block(threads > 64 ? unsigned(threads) : 256u);
  SoftmaxArgs a{};   // (a step of a level of one row is not taken)
  a.x = r.x; a.dy = r.dy; a.out = r.out; a.n0 = int(r.n0);
  if (r.n0 > 1) { a.x_pitch = uint32_t(r.x_pitch); a.dy_pitch = uint32_t(dy0); a.out_pitch = uint32_t(r.out_pitch); }
  if (r.n1 > 1) { a.x_lv.p1 = int(r.x_lv.p1); a.dy_lv.p1 = int(dy1); a.out_lv.p1 = int(r.out_lv.p1); }
  if (r.n2 > 1) { a.x_lv.p2 = int(r.x_lv.p2); a.dy_lv.p2 = int(dy2); a.out_lv.p2 = int(r.out_lv.p2); }
  a.cols = r.cols; a.nvec = r.nvec; a.spare = uint16_t(r.spare); a.threads = uint16_t(block.x);
  switch (threads) {
    case 8: return launch_softmax_nv<T, BWD, 8, RAGGED>(a, nv, grid, block, s);
    case 16: return launch_softmax_nv<T, BWD, 16, RAGGED>(a, nv, grid, block, s);
    case 32: return launch_softmax_nv<T, BWD, 32, RAGGED>(a, nv, grid, block, s);
    case 64: return launch_softmax_nv<T, BWD, 64, RAGGED>(a, nv, grid, block, s);
    default: return launch_softmax_nv<T, BWD, 0, RAGGED>(a, nv, grid, block, s);
  }
}

template <typename T, bool BWD>
static int softmax_lastdim_typed(SoftmaxRows a, hipStream_t s) {
  constexpr int VEC = VecIO<T>::N;
  auto steps_ok = [](int64_t pitch, const LevelSteps& l) { return pitch % VEC == 0 && l.p1 % VEC == 0 && l.p2 % VEC == 0; };
  const bool vec_ok = a.cols % VEC == 0 && aligned16(a.x) && aligned16(a.dy) && aligned16(a.out) &&
                      steps_ok(a.x_pitch, a.x_lv) && steps_ok(a.out_pitch, a.out_lv) &&
                      (!BWD || steps_ok(a.dy_pitch, a.dy_lv));
  // forward keeps NV*VEC exponentials per thread: at most 64 floats
  // backward holds y and dy: at most 4 vectors of each per thread
  const int max_nv = BWD ? 4 : 64 / VEC;
  int threads = 0, nv = 0;
  const uintptr_t boundary = reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.dy) |
                             reinterpret_cast<uintptr_t>(a.out) | uintptr_t(a.x_pitch * int64_t(sizeof(T))) |
                             uintptr_t(a.out_pitch * int64_t(sizeof(T)));
  a.nvec = (a.cols + VEC - 1) / VEC;
  const auto shape = [&](int nvec, int* t, int* n) {
    return pick_softmax_shape(nvec, vec_ok, (boundary & 3) != 0, max_nv, BWD, t, n);
  };
  const bool shaped = shape(a.nvec, &threads, &nv);
  if (shaped && !vec_ok) {
    const bool odd = ((reinterpret_cast<uintptr_t>(a.x) | uintptr_t(a.x_pitch * int64_t(sizeof(T)))) & 3) != 0;
    // The vector more is for free where the lanes are there.  Past a wavefront the backward, whose two operands pay for
    // accesses off 4 bytes, is the better for it, the forward only in a wavefront and where few wide threads hold the row.
    // bf16 us without / with it, forward: 40000 x 64 4.1 / 5.3, x 192 9.4 / 8.5, 4096 x 1024 5.8 / 5.3, 12288 x 2048 19.5 /
    // 22.6, 4096 x 4096 16 / 17, x 8192 28.7 / 30.4, x 16384 60 / 54; backward: 40000 x 64 4.9 / 6.3, x 192 12.0 / 10.4,
    // x 512 22.0 / 22.9, 4096 x 4096 22.0 / 18.9, x 8192 42.6 / 33.4, 1000 x 32768 (no workgroup holds a vector more) 47 / 124.
    a.spare = plan_spare<T>(a.cols, odd, a.nvec, threads, nv, shape, [&](int t, int n) {
      return a.nvec <= 64 ? t == threads && n == nv : BWD || t == 64 || threads == 1024 || nv == 8;
    });
  }
  if (vec_ok && shaped) return launch_softmax<T, BWD, false>(a, threads, nv, s);
  if (a.n0 != a.rows) {
    set_last_error("softmax: rows on several levels need 16-byte aligned rows and steps");
    return HK_ERR_UNSUPPORTED;
  }
  // any other length or alignment, down to rows of one vector
  if (shaped && a.cols >= VEC) return launch_softmax<T, BWD, true>(a, threads, nv, s);
  if constexpr (BWD) {
    HK_LAUNCH((softmax_bwd_longrow_kernel<T, float>), dim3(unsigned(a.rows)), dim3(256), 0, s,
                       static_cast<const T*>(a.x), static_cast<const T*>(a.dy), static_cast<T*>(a.out),
                       int64_t(a.cols), a.x_pitch, a.dy_pitch, a.out_pitch);
    return launch_check("softmax_bwd_longrow_kernel");
  } else {
    HK_LAUNCH((softmax_fwd_longrow_kernel<T, float>), dim3(unsigned(a.rows)), dim3(256), 0, s,
                       static_cast<const T*>(a.x), static_cast<T*>(a.out), int64_t(a.cols), a.x_pitch, a.out_pitch);
    return launch_check("softmax_fwd_longrow_kernel");
  }
}

// FEW: up to kFewSlices slices.  MAXT: the most threads that its plans have.  LEAST, MOST: the entries per lane that they give (of
// 16-bit types from 8 on even numbers, backward 14 and 16).  LEAST_AGAIN: from how many on AGAIN; 14 backward just fit without
template <typename T, bool BWD, int LX, bool PLAIN, bool FEW, int MAXT, int LEAST, int MOST, int LEAST_AGAIN = 17>
static int launch_softmax_dim(SoftmaxDimArgs a, int nk, hipStream_t s) {
  const auto built = [](int n) {
    return n >= LEAST && n <= MOST && (n <= kDimVecs || VecIO<T>::N == 4 || (n % 2 == 0 && (!BWD || n >= 14)));
  };
  if (!built(nk) || a.slices * LX > MAXT) {
    set_last_error("softmax: no kernel for %d entries per lane", nk);
    return HK_ERR_UNSUPPORTED;
  }
  a.blocks = int((a.total + LX - 1) / LX);
  const dim3 grid{unsigned(a.blocks)}, block{unsigned(LX), unsigned(a.slices)};
  const size_t lds = a.slices > 1 ? share_floats<VecIO<T>::N, LX, FEW, BWD>(a.slices) * sizeof(float) : 0;
#define HK_DIM_CASE(NK)                                                             \
  case NK:                                                                          \
    if constexpr (built(NK)) {                                                      \
      constexpr bool AGAIN = NK >= LEAST_AGAIN && !(BWD && NK == 14);               \
      if constexpr (BWD) HK_LAUNCH((softmax_bwd_dim_kernel<T, NK, LX, PLAIN, FEW, MAXT, AGAIN>), grid, block, lds, s, a); \
      else HK_LAUNCH((softmax_fwd_dim_kernel<T, NK, LX, PLAIN, FEW, MAXT, AGAIN>), grid, block, lds, s, a); \
    }                                                                               \
    break;
  profile_before(s);
  switch (nk) {
    HK_DIM_CASE(1) HK_DIM_CASE(2) HK_DIM_CASE(3) HK_DIM_CASE(4) HK_DIM_CASE(5) HK_DIM_CASE(6) HK_DIM_CASE(7) HK_DIM_CASE(8)
    HK_DIM_CASE(9) HK_DIM_CASE(10) HK_DIM_CASE(11) HK_DIM_CASE(12) HK_DIM_CASE(13) HK_DIM_CASE(14) HK_DIM_CASE(15) HK_DIM_CASE(16)
  }
#undef HK_DIM_CASE
  profile_after(s);
  return launch_check("softmax_dim_kernel");
}

template <typename T, typename CT, bool BWD>
static int softmax_strided_typed(const void* x, const void* dy, void* out, int64_t outer, int64_t dim,
                                 int64_t inner, int64_t x_pitch, int64_t dy_pitch, int64_t out_pitch,
                                 hipStream_t s) {
  if (inner == 1) {
    if constexpr (BWD) {
      HK_LAUNCH((softmax_bwd_longrow_kernel<T, CT>), dim3(unsigned(outer)), dim3(256), 0, s,
                         static_cast<const T*>(x), static_cast<const T*>(dy), static_cast<T*>(out), dim, x_pitch,
                         dy_pitch, out_pitch);
    } else {
      HK_LAUNCH((softmax_fwd_longrow_kernel<T, CT>), dim3(unsigned(outer)), dim3(256), 0, s,
                         static_cast<const T*>(x), static_cast<T*>(out), dim, x_pitch, out_pitch);
    }
    return launch_check("softmax_longrow_kernel");
  }
  if constexpr (!std::is_same<T, double>::value) {
    constexpr int VEC = VecIO<T>::N;
    // One thread per position stays the faster one (GPU us, one thread per position / the kernels above)
    //  - where the device has positions enough for it and planes are so short that every lane's vector has a cache line
    //    to itself: 32000 x 64 x 8 bf16 40.9 / 82.9, backward 37.8 / 113.3, and 8000 x 64 x 8 17.1 / 27.8 (one vector a
    //    plane: sooner); 32000 x 64 x 8 fp32 61.6 / 69.8 and 50.6 / 102.4; 16000 x 64 x 16 bf16 53.9 / 36.4 and 43.9 /
    //    47.1.  Odd planes, 28444 x 64 x 9 bf16, 63 / 50 and 70 / 69, and fewer positions, 2000 x 64 x 8 bf16 half the
    //    time with the kernels above, do not belong to them;
    //  - for a few positions of two to four entries on planes that share cache lines, where it is the shorter program:
    //    1306 x 2 x 49 bf16 2.9 / 3.45 and 2.75 / 3.3, 64 x 2 x 1000 2.8 / 3.2 (64 positions a plane 2.9 / 2.9).
    const int64_t positions = outer * inner, cus = device_cu_count(), bytes = inner * int64_t(sizeof(T));
    const bool short_planes = inner % 4 == 0 && (BWD ? bytes < 64 : inner < 16) &&
                              positions > cus * (BWD && bytes == 16 ? 192 : 512);
    const bool few_narrow = positions <= cus * 512 && bytes % 128 != 0 && dim <= 4;
    if (inner >= VEC && inner <= 0x7fffffff && dim <= 32 * kDimVecs && !short_planes && !few_narrow) {
      SoftmaxDimArgs a{};
      a.x = x; a.dy = dy; a.out = out; a.inner = inner; a.dim = int(dim);
      a.run_vecs = int((inner + VEC - 1) / VEC);
      a.total = outer * a.run_vecs;
      // A problem that leaves most wavefront slots empty takes 2 entries a lane, in workgroups of half a wavefront's
      // vectors (a quarter's, up to 64 slices, for the longer dimensions of the smallest): its time is one lane's chain
      // of instructions.  GPU us, forward / backward, with 6 to 8 entries in a wavefront's and so: 4 x 65 x 355 bf16
      // 8.6 / 7.5 and 4.4 / 3.6, 2 x 250 x 200 fp32 9.4 / 10.7 and 5.8 / 5.9, 3 x 57 x 5877 fp32 5.8 / 6.3 and 4.5 / 4.4,
      // 4 x 100 x 10000 bf16 10.1 / 8.0 and 7.8 / 6.8; at 2 x 128 x 16384 fp32 they meet, 8.9 / 11.1 and 9.9 / 10.8.
      const bool few = a.total <= cus * 64 && a.total * dim <= cus * 3072;
      const bool odd = bytes % 128 != 0;   // planes share cache lines
      const int64_t array = a.total * dim * 16;
      // More entries than that: runs of half a wavefront's vectors in up to 16 slices; forward, of the longest dimensions of 16-bit
      // entries, a quarter's in up to 32 where planes are whole lines or the array is small.  A workgroup then has at most 512
      // threads and several share a compute unit (runs of 64 lanes in up to 16 slices of 8 or 6 entries, as before, / 32 / 16
      // lanes; forward, bf16: 122 x 40 x 16384 66 / 54 / 54, 76 x 64 61 / 55 / 55, 55 x 88 72 / 54 / 56, 38 x 128 72 / 57 / 55, 32 x
      // 150 73 / 56 / 56, 26 x 182 71 / 60 / 56, 19 x 256 73 / 69 / 58; odd planes, 75 x 88 x 12101 81 / 69 / 72, 36 x 182 90 / 75 / 80,
      // 25 x 256 89 / 77 / 86; backward: 76 x 64 x 16384 90 / 76 / 78, 55 x 88 89 / 78 / 78, 4 x 224 x 12288 13.5 / 12.2 / 14.4, 19 x 256 147 / 85 /
      // 85, 3 x 256 x 12288 21 / 15 / 15).  Odd planes of up to
      // 48 entries keep their runs longer (300 x 33 x 8191 forward 65 / 73).  In the 16-bit backward of 129 to 192 entries (5 x 182 x
      // 12288, 6 entries in 31 slices 12.1, 12 in 16 12.7) and of fp32 (13 x 167 x 3648 forward 11.7 / 12.1), slices are the 32 that a
      // workgroup can have; fp32 up to 128 entries stays with runs of 64 lanes, up to 16 slices (64 / 32 lanes, 4 x 60 x 263169 115 / 132
      // and 168 / 196, 39 x 70 x 3264 forward 12.6 / 13.9, 38 x 64 x 16384 56 / 55).
      const bool many = !few && dim > (VEC == 4 ? 128 : odd ? 48 : 32);
      const bool tall = many && dim > 128 && (VEC == 4 || (BWD && dim <= 192));
      const bool quarter = VEC == 8 && !BWD && dim > 160 && many && (!odd || array < (int64_t(48) << 20));
      const int lx = few ? (a.total <= cus * 16 && dim > 64 ? 16 : 32) : quarter ? 16 : 32;
      const int most_slices = (few || tall ? 1024 : 512) / lx, fewest = int((dim + most_slices - 1) / most_slices);
      int nk;
      if (many) {
        // (up to 80 entries forward 8 or a little less: 12 x 52 x 40554 22.5 us, of 5 entries 24.8)
        nk = std::max(tall ? (VEC == 4 ? 8 : 6) : BWD ? 4 : dim <= 80 ? int((dim + (dim + 7) / 8 - 1) / ((dim + 7) / 8)) : 5, fewest);
        if (nk > kDimVecs) nk = (nk + 1) / 2 * 2;
        if (BWD && nk > kDimVecs) nk = std::max(nk, 14);
      } else {
        // the 16-bit backward of small arrays and of odd planes takes as few as 6 (22 x 8 x 20059 6.4 / 7.0 us, 310 x 46 x 3005 53 / 64)
        const int full = VEC == 8 && BWD && (array < (int64_t(48) << 20) || odd) ? 6 : kDimVecs;
        const int most = few ? std::max(2, fewest) : full, slices = int((dim + most - 1) / most);
        nk = int((dim + slices - 1) / slices);
      }
      a.slices = int((dim + nk - 1) / nk);
      if (a.total <= 0x7fffffffLL) {
        // fp32 planes that fill the device many times over take longer runs, which share fewer lines: 9 to 24 entries, on odd planes
        // of 256 KiB 32, two slices of 128 lanes; fewer one of 128 forward, 256 backward on odd planes.  Time of slices of up to 8
        // entries of 64 lanes over that of the two, forward and backward, geometric means of 9 to 24 entries: odd planes of 5001
        // to 263169, by vectors per compute unit, 300 0.94 and 0.93, 500 0.99 and 1.00, 780 1.00 and 1.00, 1030 to 1170 1.02 and 1.03, 1550 1.03 and
        // 1.05, 2100 1.03 and 1.06, 7800 1.05 and 1.10; planes of whole lines 1030 to 1150 0.99 and 1.00, 1550 1.00 and 1.01, 2100 1.00 and 1.02,
        // 4700 1.01 and 1.02.  28 and 32 entries: odd planes of 5001 at 2100 0.96 and 0.98, of 20001 at 1130 1.00 and 0.99, 2100 0.98 and
        // 0.99, of 100003 at 780 0.99 and 0.99, 1170 1.00 and 1.00, 2100 1.01 and 1.02, of 263169 at 1030 1.07 and 1.07, 2100 1.11 and 1.12; whole
        // lines, 128 x 32 x 16384, 0.98 and 0.96.
        // Runs of 64 lanes are as good for few entries on planes of whole lines (16 x 2 x 1048576 42.3 / 44.3 and 60.9 / 62.7 us) and
        // better for 16-bit entries (8 x 21 x 263169 35.3 / 37.8 / 48.1 and 50.3 / 51.0 / 55.8).
        const bool wide = VEC == 4 && (dim <= kDimVecs ? odd && a.total >= cus * 2048
                                       : dim <= 24     ? a.total >= cus * (odd ? 1024 : 2048)
                                                       : dim <= 32 && odd && bytes >= (256 << 10) && a.total >= cus * 1024);
        if (wide && dim > kDimVecs) { nk = int((dim + 1) / 2); a.slices = 2; }
        // PLAIN: stored through the cache, where lines that two workgroups share meet and a call that follows may find them.  Larger arrays
        // and planes of whole lines are streamed (streamed / so, bf16 forward: 60 x 5 x 263169 56.9 / 58.7, 413 x 5 x 12101 20.9 / 19.8, 1322 x 5 x 12101 61.1 / 63.5,
        // 232 x 21 x 16384 52.6 / 57.4, 18 x 16 x 263169 55.7 / 58.7, 13 x 220 x 4093 15.5 / 16, 13 x 150 x 12101 25.6 / 25.1, 44 x 150 x 12101
        // 73.7 / 69.7, 30 x 220 x 12101 89 / 85, planes of less than 4 KiB, 1567813 x 4 x 17, 188 / 180, 3043 x 26 x 1033 77 / 68; backward: 976 x 5 x 16384
        // 74 / 80, 232 x 21 x 16384 75.5 / 82, 15 x 19 x 44480 15.6 / 15.0, 98 x 21 x 12101 29 / 28, 51 x 128 x 12101 98.6 / 103,
        // 214 x 2 x 1427 3.55 / 3.1, 17 x 11 x 52027 13.0 / 12.5, 5 x 153 x 10427 12.5 / 13.1; fp32, 2 x 193 x 21456 forward 13.0 / 14.8,
        // 5 x 98 x 12304 backward 13.0 / 15.2, planes of less than 4 KiB, 6614 x 187 x 29, 87 / 75 and 135 / 121).
        // Odd planes whose forward and backward follow one another, three sets of buffers in turn: 18 to 48 entries at 35 to 62 MiB 1.00 to
        // 1.08 of the speed with the forward streamed, at 128 to 176 MiB 1.01 to 1.09 with both streamed (13 x 21 x 271110 132 / 124, 30 x 9 x 263349 122 /
        // 117); by itself a forward of 32 to 64 MiB takes up to 10 % longer so, and both directions up to 8 % past 128 MiB.
        const auto mib = [&](int n) { return int64_t(n) << 20; };
        const bool plain = VEC == 8 && BWD && tall                            ? false
                           : odd && bytes < 4096 && (BWD || array >= mib(24)) ? true
                           : VEC == 4                                         ? false
                           : BWD && !many                                     ? odd || array < mib(48)
                                                                              : odd && array >= mib(24) && (!BWD || array < mib(128));
        // Up to kFewSlices slices every thread merges its own values, GPU us, with slices_share / so: 64 x 10 x 12544 bf16 (2
        // slices) forward 8.3 / 7.2, 32 x 12 x 40000 11.7 / 11.1, 4 x 5 x 5904 (3) 3.7 / 3.0, 32 x 40 x 6401 (5) 10.4 / 10.2, 4 x 12 x 5904 (6) 3.6 /
        // 3.35, 16 x 60 x 30001 (8) 25.9 / 27.3.
        // What nk can be.  64 slices: 2 to 4, for 65 to 256 entries.  The few in 32: up to 6, because at 192 entries and past 16
        // vectors per compute unit they are no longer few; 1 or 2 in few slices.  32 slices of a quarter's run: 6 to 8; of half
        // one 8, in the 16-bit backward 6.  16 of half one: forward 6 to 16, streamed,
        // which odd planes of 24 MiB and more are not, 10, backward 4 to 8, 14 and 16.  fp32 in more than
        // six slices of 64 lanes: 7 or 8; the 16-bit backward of 37 to 48 entries on odd planes: 6.  Of those in few slices
        // through the cache, the 16-bit backward's are on odd planes or small, the fp32 forward's of 24 MiB and more in less
        // than 2048 vectors per compute unit.
        constexpr int kLeastPlain = VEC == 4 && !BWD ? 3 : 1, kMostPlain = VEC == 8 && BWD ? 6 : kDimVecs;
        constexpr int kLeast = BWD ? 4 : 6, kLeastAgain = BWD ? 7 : 12;
        if (few) {
          if (lx == 16) return launch_softmax_dim<T, BWD, 16, true, false, 1024, 2, 4>(a, nk, s);
          if (a.slices <= kFewSlices) return launch_softmax_dim<T, BWD, 32, true, true, 1024, 1, 2>(a, nk, s);
          return launch_softmax_dim<T, BWD, 32, true, false, 1024, 2, 6>(a, nk, s);
        }
        if constexpr (VEC == 8 && !BWD) {
          if (quarter) return launch_softmax_dim<T, BWD, 16, false, false, 512, 6, 8>(a, nk, s);
        }
        if constexpr (VEC == 4) {
          if (tall && plain) return launch_softmax_dim<T, BWD, 32, true, false, 1024, kDimVecs, kDimVecs>(a, nk, s);
          if (tall) return launch_softmax_dim<T, BWD, 32, false, false, 1024, kDimVecs, kDimVecs>(a, nk, s);
        } else if constexpr (BWD) {
          if (tall) return launch_softmax_dim<T, BWD, 32, false, false, 1024, 6, 6>(a, nk, s);
        }
        if constexpr (BWD && VEC == 8) {
          // (24 MB / 64 MB of 128 entries 16.6 / 35.9 formed again, 15.4 / 36.8 kept; 160 MB 81.5 / 87.4)
          if (many && nk <= kDimVecs && array < (int64_t(48) << 20)) {
            if (plain) return launch_softmax_dim<T, BWD, 32, true, false, 512, kLeast, kDimVecs>(a, nk, s);
            return launch_softmax_dim<T, BWD, 32, false, false, 512, kLeast, kDimVecs>(a, nk, s);
          }
        }
        if constexpr (VEC == 8) {
          if (many && plain) return launch_softmax_dim<T, BWD, 32, true, false, 512, kLeast, 16, kLeastAgain>(a, nk, s);
          if (many) return launch_softmax_dim<T, BWD, 32, false, false, 512, kLeast, (BWD ? 16 : 10), kLeastAgain>(a, nk, s);
        }
        if constexpr (VEC == 4) {
          if (wide && a.slices == 2) return launch_softmax_dim<T, BWD, 128, false, true, 256, 5, 16>(a, nk, s);
          if (wide) return launch_softmax_dim<T, BWD, (BWD ? 256 : 128), false, true, 256, 1, kDimVecs>(a, nk, s);
          if (a.slices > kFewSlices) return launch_softmax_dim<T, BWD, 64, false, false, 1024, kDimVecs - 1, kDimVecs>(a, nk, s);
        }
        if constexpr (VEC == 8 && BWD) {
          if (a.slices > kFewSlices) return launch_softmax_dim<T, BWD, 64, true, false, 512, 6, 6>(a, nk, s);   // odd planes
        }
        if (plain) return launch_softmax_dim<T, BWD, 64, true, true, 512, kLeastPlain, kMostPlain>(a, nk, s);
        return launch_softmax_dim<T, BWD, 64, false, true, 512, 1, kDimVecs>(a, nk, s);
      }
    }
  }
  const int64_t npos = outer * inner;
  const int64_t blocks = (npos + 255) / 256;
  if constexpr (BWD) {
    HK_LAUNCH((softmax_bwd_strided_kernel<T, CT>), dim3(unsigned(blocks)), dim3(256), 0, s,
                       static_cast<const T*>(x), static_cast<const T*>(dy), static_cast<T*>(out), outer,
                       dim, inner);
  } else {
    HK_LAUNCH((softmax_fwd_strided_kernel<T, CT>), dim3(unsigned(blocks)), dim3(256), 0, s,
                       static_cast<const T*>(x), static_cast<T*>(out), outer, dim, inner);
  }
  return launch_check("softmax_strided_kernel");
}

// x_pitch / dy_pitch / out_pitch: elements between the starts of consecutive rows when inner == 1 (0: dense, the
// row's own length); a dimension other than the last (inner > 1) only exists for dense arrays.
struct SoftmaxLevels {
  int64_t n0, n1, n2;          // in walk order
  int64_t x_pitch, dy_pitch, out_pitch;
  LevelSteps x, dy, out;
};

template <bool BWD>
static int softmax_dispatch(int dtype, const void* x, const void* dy, void* out, int64_t outer,
                            int64_t dim, int64_t inner, int64_t x_pitch, int64_t dy_pitch, int64_t out_pitch,
                            hipStream_t s, const char* who, const SoftmaxLevels* levels = nullptr) {
  HK_REQUIRE(outer >= 0 && dim >= 0 && inner >= 0, HK_ERR_INVALID, "%s: negative extent", who);
  if (outer == 0 || dim == 0 || inner == 0) return HK_OK;
  HK_REQUIRE(x && out && (!BWD || dy), HK_ERR_INVALID, "%s: null input/output", who);
  if (x_pitch == 0) x_pitch = dim;
  if (dy_pitch == 0) dy_pitch = dim;
  if (out_pitch == 0) out_pitch = dim;
  HK_REQUIRE((levels && levels->n0 == 1) || (x_pitch >= dim && out_pitch >= dim && dy_pitch >= dim), HK_ERR_INVALID,
             "%s: a row pitch is smaller than the %lld columns of a row", who, (long long)dim);
  HK_REQUIRE(inner == 1 || (x_pitch == dim && dy_pitch == dim && out_pitch == dim), HK_ERR_INVALID,
             "%s: row pitches only apply to the last dimension", who);
  HK_REQUIRE(outer <= 0x7fffffffLL && (outer * inner + 255) / 256 <= 0x7fffffffLL, HK_ERR_INVALID,
             "%s: too many rows", who);
  if (inner == 1 && dim <= 0x3fffffff && dtype != HK_FLOAT64) {
    SoftmaxRows a{};
    a.x = x; a.dy = dy; a.out = out; a.rows = outer; a.cols = int(dim);
    a.x_pitch = x_pitch; a.dy_pitch = dy_pitch; a.out_pitch = out_pitch;
    a.n0 = outer; a.n1 = a.n2 = 1;
    if (levels) {
      a.n0 = levels->n0; a.n1 = levels->n1; a.n2 = levels->n2;
      a.x_lv = levels->x; a.dy_lv = levels->dy; a.out_lv = levels->out;
    }
    switch (dtype) {
      case HK_FLOAT32: return softmax_lastdim_typed<float, BWD>(a, s);
      case HK_BFLOAT16: return softmax_lastdim_typed<bf16, BWD>(a, s);
      case HK_FLOAT16: return softmax_lastdim_typed<fp16, BWD>(a, s);
      default: break;
    }
  }
  if (levels && levels->n0 != outer) {
    set_last_error("%s: rows on several levels are not implemented for dtype %d", who, dtype);
    return HK_ERR_UNSUPPORTED;
  }
  switch (dtype) {
    case HK_FLOAT32: return softmax_strided_typed<float, float, BWD>(x, dy, out, outer, dim, inner, x_pitch, dy_pitch, out_pitch, s);
    case HK_BFLOAT16: return softmax_strided_typed<bf16, float, BWD>(x, dy, out, outer, dim, inner, x_pitch, dy_pitch, out_pitch, s);
    case HK_FLOAT16: return softmax_strided_typed<fp16, float, BWD>(x, dy, out, outer, dim, inner, x_pitch, dy_pitch, out_pitch, s);
    case HK_FLOAT64: return softmax_strided_typed<double, double, BWD>(x, dy, out, outer, dim, inner, x_pitch, dy_pitch, out_pitch, s);
    default:
      set_last_error("%s: not implemented for dtype %d", who, dtype);
      return HK_ERR_UNSUPPORTED;
  }
}

} // namespace hk

using namespace hk;

extern "C" {

int hk_softmax_fwd(int dtype, const void* x, void* y, int64_t outer, int64_t dim, int64_t inner,
                   hkStream_t stream) {
  return softmax_dispatch<false>(dtype, x, nullptr, y, outer, dim, inner, 0, 0, 0, as_hip(stream), "hk_softmax_fwd");
}

int hk_softmax_fwd_pitched(int dtype, const void* x, int64_t x_pitch, void* y, int64_t y_pitch, int64_t rows,
                           int64_t cols, hkStream_t stream) {
  HK_REQUIRE(x_pitch > 0 && y_pitch > 0, HK_ERR_INVALID, "hk_softmax_fwd_pitched: a row pitch must be positive");
  return softmax_dispatch<false>(dtype, x, nullptr, y, rows, cols, 1, x_pitch, x_pitch, y_pitch, as_hip(stream),
                                 "hk_softmax_fwd_pitched");
}

static int softmax_levels(const int64_t level_rows[3], const int64_t* x_steps, const int64_t* dy_steps,
                          const int64_t* out_steps, SoftmaxLevels* lv, int64_t* rows, const char* who) {
  HK_REQUIRE(level_rows && x_steps && out_steps, HK_ERR_INVALID, "%s: null level_rows / steps", who);
  const int64_t n0 = level_rows[0], n1 = level_rows[1], n2 = level_rows[2];
  HK_REQUIRE(n0 >= 0 && n1 >= 0 && n2 >= 0, HK_ERR_INVALID, "%s: negative level count", who);
  *rows = 0;
  if (n0 == 0 || n1 == 0 || n2 == 0) return HK_OK;
  HK_REQUIRE(n0 <= 0x7fffffffLL && n0 * n1 <= 0x7fffffffLL && n0 * n1 * n2 <= 0x7fffffffLL, HK_ERR_INVALID,
             "%s: too many rows", who);
  *rows = n0 * n1 * n2;
  int64_t key[3] = {0, 0, 0};
  for (int k = 0; k < 3; ++k) key[k] = x_steps[k] + out_steps[k] + (dy_steps ? dy_steps[k] : 0);
  const RowWalk w = plan_row_walk(level_rows, key, /*on_grid=*/true);
  HK_REQUIRE(walk_fits_grid(w), HK_ERR_UNSUPPORTED,
             "%s: two of the three levels must hold at most 65535 rows each (got %lld, %lld, %lld)", who,
             (long long)n0, (long long)n1, (long long)n2);
  lv->n0 = w.n[0]; lv->n1 = w.n[1]; lv->n2 = w.n[2];
  walk_steps(w, x_steps, &lv->x_pitch, &lv->x);
  walk_steps(w, out_steps, &lv->out_pitch, &lv->out);
  lv->dy_pitch = lv->x_pitch;
  lv->dy = lv->x;
  if (dy_steps) walk_steps(w, dy_steps, &lv->dy_pitch, &lv->dy);
  return HK_OK;
}

int hk_softmax_fwd_strided_rows(int dtype, const void* x, const int64_t x_steps[3], void* y, const int64_t y_steps[3],
                                const int64_t level_rows[3], int64_t cols, hkStream_t stream) {
  const char* who = "hk_softmax_fwd_strided_rows";
  SoftmaxLevels lv{};
  int64_t rows = 0;
  int rc = softmax_levels(level_rows, x_steps, nullptr, y_steps, &lv, &rows, who);
  if (rc != HK_OK || rows == 0) return rc;
  return softmax_dispatch<false>(dtype, x, nullptr, y, rows, cols, 1, lv.x_pitch, lv.dy_pitch, lv.out_pitch,
                                 as_hip(stream), who, &lv);
}

int hk_softmax_bwd_strided_rows(int dtype, const void* y, const int64_t y_steps[3], const void* dy,
                                const int64_t dy_steps[3], void* dx, const int64_t dx_steps[3],
                                const int64_t level_rows[3], int64_t cols, hkStream_t stream) {
  const char* who = "hk_softmax_bwd_strided_rows";
  HK_REQUIRE(dy_steps, HK_ERR_INVALID, "%s: null steps", who);
  SoftmaxLevels lv{};
  int64_t rows = 0;
  int rc = softmax_levels(level_rows, y_steps, dy_steps, dx_steps, &lv, &rows, who);
  if (rc != HK_OK || rows == 0) return rc;
  return softmax_dispatch<true>(dtype, y, dy, dx, rows, cols, 1, lv.x_pitch, lv.dy_pitch, lv.out_pitch,
                                as_hip(stream), who, &lv);
}

int hk_softmax_bwd(int dtype, const void* y, const void* dy, void* dx, int64_t outer, int64_t dim,
                   int64_t inner, hkStream_t stream) {
  return softmax_dispatch<true>(dtype, y, dy, dx, outer, dim, inner, 0, 0, 0, as_hip(stream), "hk_softmax_bwd");
}

int hk_softmax_bwd_pitched(int dtype, const void* y, int64_t y_pitch, const void* dy, int64_t dy_pitch, void* dx,
                           int64_t dx_pitch, int64_t rows, int64_t cols, hkStream_t stream) {
  HK_REQUIRE(y_pitch > 0 && dy_pitch > 0 && dx_pitch > 0, HK_ERR_INVALID,
             "hk_softmax_bwd_pitched: a row pitch must be positive");
  return softmax_dispatch<true>(dtype, y, dy, dx, rows, cols, 1, y_pitch, dy_pitch, dx_pitch, as_hip(stream),
                                "hk_softmax_bwd_pitched");
}

} // extern "C"
