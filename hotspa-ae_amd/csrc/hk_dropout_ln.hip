// Dropout-add-LayerNorm / RMSNorm with every feature of the interface: dropout,
// per-row and per-column scaling, row subsets, mixed input / residual / weight
// types and the parallel-residual form.  Calls that use none of these are handed
// to the plain norm kernels; this file is the general path.
//
// Work split: a thread owns chunks of 8 consecutive columns (one 16-byte vector
// of a 16-bit type, two of fp32).  Forward: one group of threads per row, the row
// in registers, statistics as in the plain kernel (Welford / Chan for LayerNorm,
// two sums for RMSNorm).  Backward: a persistent grid of column-owner groups
// keeps up to five per-column sums in registers and writes one fp32 partial row
// per group; a second kernel folds the partial rows.
//
// Dropout mask: element e of the input draws word e % 4 of Philox4x32-10 (key =
// seed, counter = (2 * (e / 4) + input number, offset)), so the mask does not
// depend on the launch shape.
#include "hk_common.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace hk {

// ---------------------------------------------------------------------------
// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11)
// ---------------------------------------------------------------------------
// (bitop3 with the truth table of a ^ b ^ c; the compiler makes two instructions of the expression)
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
  return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}
__device__ __forceinline__ void philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                              uint32_t k0, uint32_t k1, uint32_t out[4]) {
  constexpr uint32_t kM0 = 0xD2511F53u, kM1 = 0xCD9E8D57u, kW0 = 0x9E3779B9u, kW1 = 0xBB67AE85u;
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint64_t p0 = uint64_t(kM0) * c0;
    const uint64_t p1 = uint64_t(kM1) * c2;
    const uint32_t n0 = xor3(uint32_t(p1 >> 32), c1, k0);
    const uint32_t n2 = xor3(uint32_t(p0 >> 32), c3, k1);
    c1 = uint32_t(p1);
    c3 = uint32_t(p0);
    c0 = n0;
    c2 = n2;
    k0 += kW0;
    k1 += kW1;
  }
  out[0] = c0; out[1] = c1; out[2] = c2; out[3] = c3;
}

struct DropArgs {
  uint32_t seed_lo, seed_hi, off_lo, off_hi;
  uint32_t keep_max;
};

// The 8 elements [e0, e0 + 8) of input number `which` (e0 is a multiple of 8): is element e0 + j kept?  A draw is
// float(bits) * 2^-32 + 2^-33 in (0, 1], kept when <= keep probability; it grows with its bits, so they are compared with the
// largest that is kept (keep_max()).  The rounds run beside the row's loads and are felt all the same: the comparison of the
// bits, and one exclusive or of three operands, took the forward of 16384 x 4096 bf16 from 113.0 to 108.1 us, of 1190 x 1104
// from 6.4 to 5.9.
struct Keep8 {
  bool k[8];
};
__device__ __forceinline__ Keep8 keep8(int64_t e0, int which, const DropArgs& d) {
  const uint64_t g2 = (uint64_t(e0) >> 1) + uint64_t(which);   // 2 * (e0 / 4) + which
  Keep8 keep;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint64_t g = g2 + uint64_t(2 * h);
    uint32_t r[4];
    philox4x32_10(uint32_t(g), uint32_t(g >> 32), d.off_lo, d.off_hi, d.seed_lo, d.seed_hi, r);
#pragma unroll
    for (int j = 0; j < 4; ++j) keep.k[4 * h + j] = r[j] <= d.keep_max;
  }
  return keep;
}
// the largest 32 random bits whose draw is at most keep_p (> 0)
inline uint32_t keep_max(float keep_p) {
  const auto draw = [](uint32_t bits) { return std::fmaf(float(bits), 2.3283064365386963e-10f, 1.1641532182693481e-10f); };
  uint32_t low = 0, high = 0xffffffffu;   // draw(0) = 2^-33 is below the smallest keep_p, 2^-24
  while (low < high) {
    const uint32_t mid = high - (high - low) / 2;
    if (draw(mid) <= keep_p) low = mid; else high = mid - 1;
  }
  return low;
}

// 8 mask bytes (0 / 1) as one 8-byte store / load
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void store_mask8(uint8_t* p, const Keep8& keep) {
  uint32_t w0 = 0, w1 = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    w0 |= keep.k[j] ? 1u << (8 * j) : 0u;
    w1 |= keep.k[4 + j] ? 1u << (8 * j) : 0u;
  }
  *reinterpret_cast<u32x2*>(p) = u32x2{w0, w1};
}
__device__ __forceinline__ uint32_t load_mask8(const uint8_t* p) {
  const u32x2 w = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(p));
  uint32_t bits = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    bits |= (((w.x >> (8 * j)) & 0xffu) ? 1u : 0u) << j;
    bits |= (((w.y >> (8 * j)) & 0xffu) ? 1u : 0u) << (4 + j);
  }
  return bits;
}

// 8 consecutive elements of T <-> 8 floats
template <typename T>
__device__ __forceinline__ void load8(const T* p, float* f) {
  VecIO<T>::unpack(ld16(p), f);
  if constexpr (VecIO<T>::N == 4) VecIO<T>::unpack(ld16(p + 4), f + 4);
}
template <typename T>
__device__ __forceinline__ void load8_keep(const T* p, float* f) {
  VecIO<T>::unpack(ld16_keep(p), f);
  if constexpr (VecIO<T>::N == 4) VecIO<T>::unpack(ld16_keep(p + 4), f + 4);
}
// STREAM is a template argument on purpose: with the choice as a run-time flag the compiler merges the two
// branches into one plain store and the non-temporal hint is lost.
template <typename T, bool STREAM>
__device__ __forceinline__ void store8(T* p, const float* f) {
  if constexpr (STREAM) {
    st16_stream(p, VecIO<T>::pack(f));
    if constexpr (VecIO<T>::N == 4) st16_stream(p + 4, VecIO<T>::pack(f + 4));
  } else {
    st16(p, VecIO<T>::pack(f));
    if constexpr (VecIO<T>::N == 4) st16(p + 4, VecIO<T>::pack(f + 4));
  }
}

constexpr int kChunk = 8;

// 1-based row number of a subset entry, 0 when it names no row or lies outside [0, numrows]
__device__ __forceinline__ int64_t subset_row(const int32_t* subset, int64_t row, int64_t numrows) {
  const int64_t v = subset[row];
  return (v < 0 || v > numrows) ? 0 : v;
}

// ===========================================================================
// forward
// ===========================================================================
// threads per row of nchunks chunks, nc to a thread
__host__ __device__ __forceinline__ int dal_fwd_threads(int nchunks, int nc) {
  return int((uint32_t(nchunks + nc - 1) / uint32_t(nc) + 63u) / 64u * 64u);
}
struct DalFwdArgs {
  const void* x0;
  const void* x1;
  const void* residual;
  const void* gamma;
  const void* beta;
  const void* gamma1;
  const void* beta1;
  const void* rowscale;
  const void* colscale;
  const int32_t* x0_subset;
  const int32_t* z_subset;
  void* z;
  void* z1;
  void* x;
  uint8_t* dmask;
  uint8_t* dmask1;
  float* mu;
  float* rs;
  int64_t rows, x0_numrows, z_numrows;
  int cols, nchunks, tpr;
  float eps, inv_cols, scale, rowscale_const;
  int is_rms, dropout;
  DropArgs drop;
  template <int NC> __device__ __forceinline__ DalFwdArgs args() const { return *this; }
};
// The same with one input and one affine pair, no scaling and no subsets (see kCheapArgs: 1528 x 1104 fp16, forward and backward,
// 17.2 -> 16.3 us, the fold of the partial rows among it)
struct DalFwdFlat {
  const void* x0;
  const void* residual;
  const void* gamma;
  const void* beta;
  void* z;
  void* x;
  uint8_t* dmask;
  float* mu;
  float* rs;
  uint32_t rows, cols;   // the highest bits: is_rms, dropout
  float eps, inv_cols, scale;
  DropArgs drop;
  static bool holds(const DalFwdArgs& a) {
    return !a.x1 && !a.gamma1 && !a.beta1 && !a.rowscale && !a.colscale && !a.x0_subset && !a.z_subset && !a.z1 && !a.dmask1;
  }
  explicit DalFwdFlat(const DalFwdArgs& a)
      : x0(a.x0), residual(a.residual), gamma(a.gamma), beta(a.beta), z(a.z), x(a.x), dmask(a.dmask), mu(a.mu), rs(a.rs),
        rows(uint32_t(a.rows) | (a.is_rms ? 0x80000000u : 0u)), cols(uint32_t(a.cols) | (a.dropout ? 0x80000000u : 0u)),
        eps(a.eps), inv_cols(a.inv_cols), scale(a.scale), drop(a.drop) {}
  template <int NC>
  __device__ __forceinline__ DalFwdArgs args() const {
    DalFwdArgs a{};
    a.x0 = x0; a.residual = residual; a.gamma = gamma; a.beta = beta; a.z = z; a.x = x; a.dmask = dmask; a.mu = mu; a.rs = rs;
    a.rows = a.x0_numrows = a.z_numrows = rows & 0x7fffffffu;
    a.cols = int(cols & 0x7fffffffu);
    a.nchunks = int(uint32_t(a.cols) / uint32_t(kChunk));
    a.tpr = dal_fwd_threads(a.nchunks, NC);
    a.eps = eps; a.inv_cols = inv_cols; a.scale = scale; a.is_rms = int(rows >> 31); a.dropout = int(cols >> 31);
    a.drop = drop;
    return a;
  }
};
static_assert(sizeof(DalFwdFlat) <= kCheapArgs, "");

// IT / RT / WT: input, residual and weight element types; NC: chunks per thread.  A block holds
// blockDim.x / tpr row groups; every group takes part in the (block-wide) reduction barrier, a group
// past the last row works on a copy of the last row and stores nothing.
// DROP == false, built for one chunk: nothing is dropped.  Without the kept elements' lane masks 8 wavefronts fit a SIMD (60
// scalar registers instead of 103; 40000 x 256 bf16 with an fp32 weight 30.7 -> 25.4 us, with an fp32 residual 33.4 -> 30.2).
// Asked for 8 of them with the masks, the compiler spills scalars: 1190 x 1104 bf16 7.5 against 6.8 us, 16384 x 1024 37.1
// against 35.0, and only 6578 x 512 with an fp32 residual 12.2 against 12.6.
// A: DalFwdArgs, or DalFwdFlat where that holds the arguments.
template <typename IT, typename RT, typename WT, int NC, bool DROP, typename A>
__global__ __launch_bounds__(256)
void dal_fwd_kernel(A given) {
  const DalFwdArgs a = given.template args<NC>();
  __shared__ float red[kMaxWaves * 3];
  const int tpr = a.tpr;
  const int group = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / tpr);
  const int t = int(threadIdx.x) - group * tpr;
  const int rpb = max(1, 256 / tpr);
  const int wpg = tpr >> 6;
  const int64_t row_raw = int64_t(blockIdx.x) * rpb + group;
  const bool row_ok = row_raw < a.rows;
  const int64_t row = row_ok ? row_raw : a.rows - 1;

  const bool subset = a.x0_subset != nullptr;
  float rowscale_val = 1.f;
  int64_t row_x0 = row + 1, row_z = row + 1;
  if (subset) {
    rowscale_val = a.rowscale_const;
    row_x0 = subset_row(a.x0_subset, row, a.x0_numrows);
    row_z = subset_row(a.z_subset, row, a.z_numrows);
  } else if (a.rowscale) {
    rowscale_val = Cvt<IT>::load(static_cast<const IT*>(a.rowscale) + row);
  }
  const bool load_x0 = row_x0 > 0;
  const bool dropout = DROP && a.dropout != 0;

  // Every load of the row is issued before the first one is waited for (the optional operands sit behind
  // uniform branches; unpacking inside those branches would serialise the loads).  A thread past the row's
  // end shadows chunk 0 and contributes nothing.
  constexpr int NI = kChunk / VecIO<IT>::N;
  constexpr int NR = kChunk / VecIO<RT>::N;
  u32x4 raw0[NC][NI], raw1[NC][NI], rawr[NC][NR];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
#pragma unroll
    for (int k = 0; k < NI; ++k) { raw0[i][k] = u32x4{0, 0, 0, 0}; raw1[i][k] = u32x4{0, 0, 0, 0}; }
#pragma unroll
    for (int k = 0; k < NR; ++k) rawr[i][k] = u32x4{0, 0, 0, 0};
  }
  if (load_x0) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = i * tpr + t;
      const IT* p = static_cast<const IT*>(a.x0) + (row_x0 - 1) * int64_t(a.cols) + (c < a.nchunks ? c : 0) * kChunk;
#pragma unroll
      for (int k = 0; k < NI; ++k) raw0[i][k] = ld16(p + k * VecIO<IT>::N);
    }
  }
  if (a.x1) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = i * tpr + t;
      const IT* p = static_cast<const IT*>(a.x1) + row * int64_t(a.cols) + (c < a.nchunks ? c : 0) * kChunk;
#pragma unroll
      for (int k = 0; k < NI; ++k) raw1[i][k] = ld16(p + k * VecIO<IT>::N);
    }
  }
  if (a.residual) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = i * tpr + t;
      const RT* p = static_cast<const RT*>(a.residual) + row * int64_t(a.cols) + (c < a.nchunks ? c : 0) * kChunk;
#pragma unroll
      for (int k = 0; k < NR; ++k) rawr[i][k] = ld16(p + k * VecIO<RT>::N);
    }
  }

  float xf[NC * kChunk];
  int cnt = 0;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = i * tpr + t;
    float* v = &xf[i * kChunk];
#pragma unroll
    for (int j = 0; j < kChunk; ++j) v[j] = 0.f;
    if (c < a.nchunks) {
      cnt += kChunk;
      const int col = c * kChunk;
      if (load_x0) {
        const int64_t e0 = (row_x0 - 1) * int64_t(a.cols) + col;
        Keep8 keep = {{true, true, true, true, true, true, true, true}};
        if (dropout) {
          keep = keep8(e0, 0, a.drop);
          if (row_ok) store_mask8(a.dmask + e0, keep);
        }
#pragma unroll
        for (int k = 0; k < NI; ++k) VecIO<IT>::unpack(raw0[i][k], v + k * VecIO<IT>::N);
#pragma unroll
        for (int j = 0; j < kChunk; ++j) {
          float xv = v[j] * rowscale_val;
          if (dropout) xv = keep.k[j] ? xv * a.scale : 0.f;
          v[j] = xv;
        }
        if (a.colscale) {
          float cs[kChunk];
          load8_keep<WT>(static_cast<const WT*>(a.colscale) + col, cs);
#pragma unroll
          for (int j = 0; j < kChunk; ++j) v[j] *= cs[j];
        }
      }
      const int64_t e = row * int64_t(a.cols) + col;
      if (a.x1) {
        float w[kChunk];
        Keep8 keep = {{true, true, true, true, true, true, true, true}};
        if (dropout) {
          keep = keep8(e, 1, a.drop);
          if (row_ok) store_mask8(a.dmask1 + e, keep);
        }
#pragma unroll
        for (int k = 0; k < NI; ++k) VecIO<IT>::unpack(raw1[i][k], w + k * VecIO<IT>::N);
#pragma unroll
        for (int j = 0; j < kChunk; ++j) {
          float xv = w[j];
          if (dropout) xv = keep.k[j] ? xv * a.scale : 0.f;
          v[j] += xv;
        }
      }
      if (a.residual) {
        float w[kChunk];
#pragma unroll
        for (int k = 0; k < NR; ++k) VecIO<RT>::unpack(rawr[i][k], w + k * VecIO<RT>::N);
#pragma unroll
        for (int j = 0; j < kChunk; ++j) v[j] += w[j];
      }
      if (a.x && row_ok) store8<RT, false>(static_cast<RT*>(a.x) + e, v);
    }
  }

  const int first_wave = group * wpg;
  float mu, rs;
  if (a.is_rms) {
    SumTuple<2> s;
    s.v[0] = 0.f; s.v[1] = 0.f;
#pragma unroll
    for (int e = 0; e < NC * kChunk; ++e) { s.v[0] += xf[e]; s.v[1] = fmaf(xf[e], xf[e], s.v[1]); }
    s = group_allreduce_tuple(s, red, first_wave, wpg);
    mu = s.v[0] * a.inv_cols;
    rs = 1.0f / sqrtf(s.v[1] * a.inv_cols + a.eps);   // mean(x^2) = var + mu^2
  } else {
    // per-thread (count, mean, M2) of the chunks held; slots past the row's end were left out of cnt
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < NC * kChunk; ++e) s += xf[e];
    const float mean_t = cnt > 0 ? s / float(cnt) : 0.f;
    float m2 = 0.f;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      if (i * tpr + t < a.nchunks) {
#pragma unroll
        for (int j = 0; j < kChunk; ++j) { const float d = xf[i * kChunk + j] - mean_t; m2 = fmaf(d, d, m2); }
      }
    }
    MomentTuple m;
    m.v[0] = float(cnt); m.v[1] = mean_t; m.v[2] = m2;
    m = group_allreduce_tuple(m, red, first_wave, wpg);
    mu = m.v[1];
    rs = 1.0f / sqrtf(m.v[2] * a.inv_cols + a.eps);
  }
  if (t == 0 && row_ok) {
    a.mu[row] = mu;
    a.rs[row] = rs;
  }

  if (!row_ok || row_z <= 0) return;   // after the only barrier
  const float shift = a.is_rms ? 0.f : mu;
  const int64_t zbase = (row_z - 1) * int64_t(a.cols);
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = i * tpr + t;
    if (c < a.nchunks) {
      const int col = c * kChunk;
      float y[kChunk], g[kChunk], b[kChunk], o[kChunk];
#pragma unroll
      for (int j = 0; j < kChunk; ++j) { y[j] = rs * (xf[i * kChunk + j] - shift); b[j] = 0.f; }
      load8_keep<WT>(static_cast<const WT*>(a.gamma) + col, g);
      if (a.beta) load8_keep<WT>(static_cast<const WT*>(a.beta) + col, b);
#pragma unroll
      for (int j = 0; j < kChunk; ++j) o[j] = fmaf(g[j], y[j], b[j]);
      store8<IT, true>(static_cast<IT*>(a.z) + zbase + col, o);
      if (a.gamma1) {
#pragma unroll
        for (int j = 0; j < kChunk; ++j) b[j] = 0.f;
        load8_keep<WT>(static_cast<const WT*>(a.gamma1) + col, g);
        if (a.beta1) load8_keep<WT>(static_cast<const WT*>(a.beta1) + col, b);
#pragma unroll
        for (int j = 0; j < kChunk; ++j) o[j] = fmaf(g[j], y[j], b[j]);
        store8<IT, true>(static_cast<IT*>(a.z1) + zbase + col, o);
      }
    }
  }
}

// ===========================================================================
// backward
// ===========================================================================
constexpr int kMaxParts = 5;   // dgamma, dbeta, dgamma1, dbeta1, dcolscale

struct DalBwdArgs {
  const void* dz;
  const void* dz1;
  const void* dx;
  const void* x;
  const void* x0;
  const uint8_t* dmask;
  const uint8_t* dmask1;
  const float* mu;
  const float* rs;
  const void* gamma;
  const void* gamma1;
  const void* rowscale;
  const void* colscale;
  const int32_t* x0_subset;
  const int32_t* z_subset;
  void* dx0;
  void* dx1;
  void* dresidual;
  float* part[kMaxParts];   // [blocks of the grid, cols] each; nullptr: not wanted
  int64_t rows, x0_numrows, z_numrows;
  int cols, nchunks, tpr;
  float inv_cols, scale, rowscale_const;
  int is_rms, dropout;
};

// What dal_bwd_stream_kernel takes of it (see kCheapArgs)
struct DalStreamArgs {
  const void* dz;
  const void* dx;
  const void* x;
  const uint8_t* dmask;
  const float* mu;
  const float* rs;
  const void* gamma;
  void* dx0;
  void* dresidual;
  float* part[2];
  uint32_t rows_rms, cols;   // the highest bit of the rows: is_rms
  float inv_cols, scale;
  uint16_t tpr, threads;
  uint32_t blocks;
};
static_assert(sizeof(DalStreamArgs) <= kCheapArgs, "");

// A thread's column sums acc -> the partial row of its block.  The block's row groups are folded through LDS first: one
// partial row per group took the fold kernel longer than the backward itself (16384 x 768 bf16 73 us, 30 us now,
// with the rows that do not fill their threads on the streaming kernel; 8192 x 4104 110 -> 70 us).
// Every thread of the block calls (barriers); stage: [rows per block, cols] floats when a block holds several groups.
__device__ __forceinline__ void put_column_sums(float* part, float* acc, float* stage, int group, int rpb, bool in, int cols,
                                                int col) {
  if (part == nullptr) return;   // uniform
  if (rpb > 1) {
    __syncthreads();
    if (in && group > 0) {
      float* mine = stage + group * cols + col;
#pragma unroll
      for (int j = 0; j < kChunk; ++j) mine[j] = acc[j];
    }
    __syncthreads();
    if (in && group == 0) {
      for (int g = 1; g < rpb; ++g) {
#pragma unroll
        for (int j = 0; j < kChunk; ++j) acc[j] += stage[g * cols + col + j];
      }
    }
  }
  if (in && group == 0) {
    float* out = part + int64_t(blockIdx.x) * cols + col;
    st16(out, VecIO<float>::pack(acc));
    st16(out + 4, VecIO<float>::pack(acc + 4));
  }
}

// One chunk of 8 columns per thread.  COLSCALE: per-column scaling (and its gradient); G1: a second
// affine output (dz1 / gamma1 and their gradients).
template <typename IT, typename RT, typename WT, bool COLSCALE, bool G1>
__global__ __launch_bounds__(1024)
void dal_bwd_kernel(DalBwdArgs a) {
  __shared__ float red[2][kMaxWaves * 2];   // double-buffered by step parity
  extern __shared__ __align__(16) float stage[];
  const int tpr = a.tpr;
  const int group = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / tpr);
  const int t = int(threadIdx.x) - group * tpr;
  const int rpb = int(blockDim.x) / tpr;
  const int wpg = tpr >> 6;
  const int first_wave = group * wpg;
  const bool in = t < a.nchunks;
  const int col = (in ? t : a.nchunks - 1) * kChunk;   // an idle thread shadows the last chunk, stores nothing
  const bool subset = a.x0_subset != nullptr;
  const bool dropout = a.dropout != 0;

  float g0[kChunk];
  [[maybe_unused]] float g1[G1 ? kChunk : 1];
  [[maybe_unused]] float cs[COLSCALE ? kChunk : 1];
  load8_keep<WT>(static_cast<const WT*>(a.gamma) + col, g0);
  if constexpr (G1) load8_keep<WT>(static_cast<const WT*>(a.gamma1) + col, g1);
  if constexpr (COLSCALE) load8_keep<WT>(static_cast<const WT*>(a.colscale) + col, cs);

  float dg0[kChunk], db0[kChunk];
  [[maybe_unused]] float dg1[G1 ? kChunk : 1], db1[G1 ? kChunk : 1], dcs[COLSCALE ? kChunk : 1];
#pragma unroll
  for (int j = 0; j < kChunk; ++j) {
    dg0[j] = 0.f; db0[j] = 0.f;
    if constexpr (G1) { dg1[j] = 0.f; db1[j] = 0.f; }
    if constexpr (COLSCALE) dcs[j] = 0.f;
  }

  const int64_t stride = int64_t(gridDim.x) * rpb;
  int parity = 0;
  // both loop bounds are block-uniform: every thread of the block reaches the barrier of every step
  for (int64_t base = int64_t(blockIdx.x) * rpb; base < a.rows; base += stride) {
    const int64_t row_raw = base + group;
    const bool row_ok = row_raw < a.rows;
    const int64_t row = row_ok ? row_raw : a.rows - 1;
    const float mu = a.is_rms ? 0.f : a.mu[row];
    const float rs = a.rs[row];
    float rowscale_val = 1.f;
    int64_t row_x0 = row + 1, row_z = row + 1;
    if (subset) {
      rowscale_val = a.rowscale_const;
      row_x0 = subset_row(a.x0_subset, row, a.x0_numrows);
      row_z = subset_row(a.z_subset, row, a.z_numrows);
    } else if (a.rowscale) {
      rowscale_val = Cvt<IT>::load(static_cast<const IT*>(a.rowscale) + row);
    }
    const bool load_dz = row_z > 0;
    const bool save_dx0 = row_x0 > 0;
    const bool live = row_ok && in;
    const int64_t e = row * int64_t(a.cols) + col;

    float dz[kChunk], y[kChunk], dy[kChunk];
    [[maybe_unused]] float dz1[G1 ? kChunk : 1];
#pragma unroll
    for (int j = 0; j < kChunk; ++j) { dz[j] = 0.f; y[j] = 0.f; }
    if (load_dz) {
      load8<IT>(static_cast<const IT*>(a.dz) + (row_z - 1) * int64_t(a.cols) + col, dz);
      float xv[kChunk];
      load8<RT>(static_cast<const RT*>(a.x) + e, xv);
#pragma unroll
      for (int j = 0; j < kChunk; ++j) y[j] = rs * (xv[j] - mu);
    }
    if constexpr (G1) load8<IT>(static_cast<const IT*>(a.dz1) + e, dz1);
    SumTuple<2> s;
    s.v[0] = 0.f; s.v[1] = 0.f;
#pragma unroll
    for (int j = 0; j < kChunk; ++j) {
      const float d0 = live ? dz[j] : 0.f;
      float d = g0[j] * d0;
      dg0[j] = fmaf(d0, y[j], dg0[j]);
      db0[j] += d0;
      if constexpr (G1) {
        const float d1 = live ? dz1[j] : 0.f;
        d = fmaf(g1[j], d1, d);
        dg1[j] = fmaf(d1, y[j], dg1[j]);
        db1[j] += d1;
      }
      dy[j] = d;
      s.v[0] += d;
      s.v[1] = fmaf(d, y[j], s.v[1]);
    }
    s = group_allreduce_tuple(s, red[parity], first_wave, wpg);
    parity ^= 1;
    if (!live) continue;   // no barrier below this point

    const float mdy = a.is_rms ? 0.f : s.v[0] * a.inv_cols;
    const float mdyy = s.v[1] * a.inv_cols;
    float dxr[kChunk];
#pragma unroll
    for (int j = 0; j < kChunk; ++j) dxr[j] = rs * (dy[j] - fmaf(mdyy, y[j], mdy));
    if (a.dx) {
      float u[kChunk];
      load8<RT>(static_cast<const RT*>(a.dx) + e, u);
#pragma unroll
      for (int j = 0; j < kChunk; ++j) dxr[j] += u[j];
    }
    if (a.dresidual) store8<RT, false>(static_cast<RT*>(a.dresidual) + e, dxr);
    if (save_dx0) {
      const int64_t e0 = (row_x0 - 1) * int64_t(a.cols) + col;
      uint32_t keep = 0xffu;
      float o[kChunk];
#pragma unroll
      for (int j = 0; j < kChunk; ++j) o[j] = dxr[j] * rowscale_val;
      if (dropout) {
        keep = load_mask8(a.dmask + e0);
#pragma unroll
        for (int j = 0; j < kChunk; ++j) o[j] *= a.scale;
      }
      if constexpr (COLSCALE) {
        float xv0[kChunk];
        load8<IT>(static_cast<const IT*>(a.x0) + e0, xv0);
#pragma unroll
        for (int j = 0; j < kChunk; ++j) {
          const bool k = (keep >> j) & 1u;
          dcs[j] += k ? o[j] * xv0[j] : 0.f;
          o[j] *= cs[j];
        }
      }
#pragma unroll
      for (int j = 0; j < kChunk; ++j) o[j] = ((keep >> j) & 1u) ? o[j] : 0.f;
      store8<IT, true>(static_cast<IT*>(a.dx0) + e0, o);
    }
    if (a.dx1) {
      float o[kChunk];
      uint32_t keep = 0xffu;
      if (dropout) keep = load_mask8(a.dmask1 + e);
#pragma unroll
      for (int j = 0; j < kChunk; ++j) {
        const float v = dropout ? dxr[j] * a.scale : dxr[j];
        o[j] = ((keep >> j) & 1u) ? v : 0.f;
      }
      store8<IT, true>(static_cast<IT*>(a.dx1) + e, o);
    }
  }

  auto put = [&](float* part, float* acc) { put_column_sums(part, acc, stage, group, rpb, in, a.cols, col); };
  put(a.part[0], dg0);
  put(a.part[1], db0);
  if constexpr (G1) { put(a.part[2], dg1); put(a.part[3], db1); }
  if constexpr (COLSCALE) put(a.part[4], dcs);
}

// The pre-norm residual block's backward, the shape a transformer layer calls: dropout on, the gradient of
// the residual stream coming in (dx) and going out (dresidual), no scaling, no subsets, one affine pair.  With nothing
// optional left, the row loop holds no branch
// around a memory instruction, so the compiler counts outstanding loads exactly and PF rows stay in flight
// per thread group (a ring of register slots refilled as soon as a slot has been unpacked); rows past the
// end are clamped to the last row and their results dropped.  A thread past the row's last chunk works on that chunk with
// a zero gradient and stores nothing.
// TPR: the group width when the one group of a block is the whole block and its size is known at compile time
// (512 threads = 4096 columns), else 0: the launch bound and the cross-wavefront step of the row sums follow it.
template <typename IT, typename RT, typename WT, int PF, int TPR>
__global__ __launch_bounds__(TPR ? TPR : 1024)
void dal_bwd_stream_kernel(DalStreamArgs a) {
  const int64_t rows = a.rows_rms & 0x7fffffffu;
  const bool is_rms = a.rows_rms >> 31 != 0;
  const int cols = int(a.cols), nchunks = int(a.cols / uint32_t(kChunk));
  constexpr int NI = kChunk / VecIO<IT>::N;   // 16-byte vectors per chunk of the input type
  constexpr int NR = kChunk / VecIO<RT>::N;   //                       ... of the residual type
  __shared__ __align__(16) float red[2][kMaxWaves * 2];
  const int tpr = TPR ? TPR : a.tpr;
  const int group = TPR ? 0 : __builtin_amdgcn_readfirstlane(int(threadIdx.x) / tpr);
  const int t = int(threadIdx.x) - group * tpr;
  const int rpb = TPR ? 1 : a.threads / tpr;
  const int wpg = tpr >> 6;
  const int first_wave = group * wpg;
  const bool in = TPR || t < nchunks;
  const int col = (in ? t : nchunks - 1) * kChunk;
  extern __shared__ __align__(16) float stage[];

  float g0[kChunk];
  load8_keep<WT>(static_cast<const WT*>(a.gamma) + col, g0);
  float dg0[kChunk], db0[kChunk];
#pragma unroll
  for (int j = 0; j < kChunk; ++j) { dg0[j] = 0.f; db0[j] = 0.f; }

  const int64_t stride = int64_t(a.blocks) * rpb;
  const int64_t last_row = rows - 1;
  u32x4 ndz[PF][NI], nx[PF][NR], ndx[PF][NR];
  u32x2 nm[PF];
  float nmu[PF], nrs[PF];
  auto issue = [&](auto slot, int64_t r) {
    constexpr int d = decltype(slot)::value;
    const int64_t rc = r < last_row ? r : last_row;
    const int64_t e = rc * int64_t(cols) + col;
    nmu[d] = a.mu[rc];
    nrs[d] = a.rs[rc];
#pragma unroll
    for (int i = 0; i < NI; ++i) ndz[d][i] = ld16(static_cast<const IT*>(a.dz) + e + i * VecIO<IT>::N);
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      nx[d][i] = ld16(static_cast<const RT*>(a.x) + e + i * VecIO<RT>::N);
      ndx[d][i] = ld16(static_cast<const RT*>(a.dx) + e + i * VecIO<RT>::N);
    }
    nm[d] = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(a.dmask + e));
  };
  int64_t row0 = int64_t(blockIdx.x) * rpb + group;
  static_for<PF>([&](auto slot) { issue(slot, row0 + decltype(slot)::value * stride); });

  int parity = 0;
  auto step = [&](auto slot, auto guarded) {
    constexpr int d = decltype(slot)::value;
    constexpr bool GUARD = decltype(guarded)::value;
    const int64_t row = row0 + d * stride;
    const bool valid = !GUARD || row < rows;
    float dz[kChunk], y[kChunk], u[kChunk];
#pragma unroll
    for (int i = 0; i < NI; ++i) VecIO<IT>::unpack(ndz[d][i], &dz[i * VecIO<IT>::N]);
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      VecIO<RT>::unpack(nx[d][i], &y[i * VecIO<RT>::N]);
      VecIO<RT>::unpack(ndx[d][i], &u[i * VecIO<RT>::N]);
    }
    const u32x2 mw = nm[d];
    const float mu = is_rms ? 0.f : nmu[d];
    const float rs = nrs[d];
    issue(slot, row + int64_t(PF) * stride);   // the slot is free again

    SumTuple<2> s;
    s.v[0] = 0.f; s.v[1] = 0.f;
    float dy[kChunk];
#pragma unroll
    for (int j = 0; j < kChunk; ++j) {
      const float d0 = ((GUARD && !valid) || !in) ? 0.f : dz[j];
      y[j] = rs * (y[j] - mu);
      dy[j] = g0[j] * d0;
      dg0[j] = fmaf(d0, y[j], dg0[j]);
      db0[j] += d0;
      s.v[0] += dy[j];
      s.v[1] = fmaf(dy[j], y[j], s.v[1]);
    }
    if constexpr (TPR != 0) s = group_allreduce_tuple_fixed<SumTuple<2>, TPR / 64>(s, red[parity]);
    else s = group_allreduce_tuple(s, red[parity], first_wave, wpg);
    parity ^= 1;
    if (valid && in) {
      const float mdy = is_rms ? 0.f : s.v[0] * a.inv_cols;
      const float mdyy = s.v[1] * a.inv_cols;
      float o[kChunk];
#pragma unroll
      for (int j = 0; j < kChunk; ++j) {
        u[j] += rs * (dy[j] - fmaf(mdyy, y[j], mdy));
        const uint32_t byte = ((j < 4 ? mw.x : mw.y) >> (8 * (j & 3))) & 0xffu;
        o[j] = byte ? u[j] * a.scale : 0.f;
      }
      const int64_t e = row * int64_t(cols) + col;
      store8<RT, false>(static_cast<RT*>(a.dresidual) + e, u);
      store8<IT, true>(static_cast<IT*>(a.dx0) + e, o);
    }
  };
  int64_t base = int64_t(blockIdx.x) * rpb;
  const int64_t round = int64_t(PF) * stride;
  // rounds in which every slot of every group of this block holds an existing row, then the guarded tail;
  // both bounds are block-uniform, so every thread reaches the barrier of every step
#pragma nounroll
  for (; base + int64_t(PF - 1) * stride + rpb <= rows; base += round) {
    static_for<PF>([&](auto slot) { step(slot, std::false_type{}); });
    row0 += round;
  }
#pragma nounroll
  for (; base < rows; base += round) {
    static_for<PF>([&](auto slot) { step(slot, std::true_type{}); });
    row0 += round;
  }

  put_column_sums(a.part[0], dg0, stage, group, rpb, in, cols, col);
  put_column_sums(a.part[1], db0, stage, group, rpb, in, cols, col);
}

// The same for few rows, in one launch: three trips to memory otherwise (rows, partial rows, their fold).  The first a.blocks
// workgroups form the column sums from the operands themselves (column_sums_of_few_rows), the others dx0 and dresidual, to the same
// bits; part: dgamma and dbeta.  Nothing that is written may lie over what is read, but
// dresidual may be dx.
template <typename IT, typename RT, typename WT>
__global__ __launch_bounds__(kSmallThreads)
void dal_bwd_small_kernel(DalStreamArgs a) {
  constexpr int NI = kChunk / VecIO<IT>::N, NR = kChunk / VecIO<RT>::N, LANES = NR == 1 ? 8 : 4;
  __shared__ __align__(16) float red[kMaxWaves * 2];
  const int rows = int(a.rows_rms & 0x7fffffffu), cols = int(a.cols), nchunks = int(a.cols / uint32_t(kChunk));
  const bool is_rms = a.rows_rms >> 31 != 0;
  struct Fetched {
    u32x4 dz[NI], x[NR];
    float mu, rs;
  };
  const auto fetch = [&](int64_t r, int col) {
    Fetched f;
    const int64_t e = r * int64_t(cols) + col;
#pragma unroll
    for (int i = 0; i < NI; ++i) f.dz[i] = ld16_keep(static_cast<const IT*>(a.dz) + e + i * VecIO<IT>::N);
#pragma unroll
    for (int i = 0; i < NR; ++i) f.x[i] = ld16_keep(static_cast<const RT*>(a.x) + e + i * VecIO<RT>::N);
    f.mu = is_rms ? 0.f : a.mu[r];
    f.rs = a.rs[r];
    return f;
  };
  const auto unpack = [&](const Fetched& f, float* dz, float* y) {
#pragma unroll
    for (int i = 0; i < NI; ++i) VecIO<IT>::unpack(f.dz[i], dz + i * VecIO<IT>::N);
#pragma unroll
    for (int i = 0; i < NR; ++i) VecIO<RT>::unpack(f.x[i], y + i * VecIO<RT>::N);
#pragma unroll
    for (int j = 0; j < kChunk; ++j) y[j] = f.rs * (y[j] - f.mu);
  };
  if (blockIdx.x < a.blocks) {
    const int first = int(blockIdx.x) * LANES, col = min(first + (int(threadIdx.x) & (LANES - 1)), nchunks - 1) * kChunk;
    column_sums_of_few_rows<2, kChunk, LANES>(
        rows, [&](int64_t r) { return fetch(r, col); },
        [&](const Fetched& f, bool in, float (&acc)[2][kChunk]) {
          float dz[kChunk], y[kChunk];
          unpack(f, dz, y);
#pragma unroll
          for (int j = 0; j < kChunk; ++j) {
            acc[0][j] = in ? fmaf(dz[j], y[j], acc[0][j]) : acc[0][j];
            acc[1][j] += in ? dz[j] : 0.f;
          }
        },
        [&](int k, int c, float sum) {
          WT* out = reinterpret_cast<WT*>(a.part[k]);
          if (out != nullptr && first * kChunk + c < cols) Cvt<WT>::store(out + first * kChunk + c, sum);
        });
    return;
  }
  const int tpr = a.tpr, rpb = kSmallThreads / tpr;
  const int group = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / tpr), t = int(threadIdx.x) - group * tpr;
  // (the wavefronts that no row is left for work on the last one too and store nothing)
  const bool idle = group >= rpb, in = t < nchunks;
  const int64_t wanted = idle ? rows : int64_t(blockIdx.x - a.blocks) * rpb + group, row = wanted < rows ? wanted : rows - 1;
  const int col = (in ? t : nchunks - 1) * kChunk;
  const int64_t e = row * int64_t(cols) + col;
  const Fetched f = fetch(row, col);
  u32x4 ndx[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) ndx[i] = ld16(static_cast<const RT*>(a.dx) + e + i * VecIO<RT>::N);
  const u32x2 mw = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(a.dmask + e));
  float g0[kChunk], dz[kChunk], y[kChunk], u[kChunk];
  load8_keep<WT>(static_cast<const WT*>(a.gamma) + col, g0);
  unpack(f, dz, y);
#pragma unroll
  for (int i = 0; i < NR; ++i) VecIO<RT>::unpack(ndx[i], &u[i * VecIO<RT>::N]);
  SumTuple<2> s;
  s.v[0] = 0.f; s.v[1] = 0.f;
  float dy[kChunk];
#pragma unroll
  for (int j = 0; j < kChunk; ++j) {
    dy[j] = g0[j] * (in ? dz[j] : 0.f);
    s.v[0] += dy[j];
    s.v[1] = fmaf(dy[j], y[j], s.v[1]);
  }
  s = group_allreduce_tuple(s, red, idle ? 0 : group * (tpr >> 6), tpr >> 6);
  if (wanted >= rows || !in) return;
  const float mdy = is_rms ? 0.f : s.v[0] * a.inv_cols;
  const float mdyy = s.v[1] * a.inv_cols;
  float o[kChunk];
#pragma unroll
  for (int j = 0; j < kChunk; ++j) {
    u[j] += f.rs * (dy[j] - fmaf(mdyy, y[j], mdy));
    const uint32_t byte = ((j < 4 ? mw.x : mw.y) >> (8 * (j & 3))) & 0xffu;
    o[j] = byte ? u[j] * a.scale : 0.f;
  }
  store8<RT, false>(static_cast<RT*>(a.dresidual) + e, u);
  store8<IT, true>(static_cast<IT*>(a.dx0) + e, o);
}

// Folds [nparts, cols] fp32 partial rows into a [cols] vector of WT (fold_partial_rows); blockIdx.y picks which of the (up to
// five) sums that are wanted.
struct DalFoldArgs {
  const float* part[kMaxParts];
  void* out[kMaxParts];
  int nparts, cols;
};

template <typename WT, int LANES>
__global__ __launch_bounds__(fold_threads(LANES))
void dal_fold_kernel(DalFoldArgs a) {
  const float s = fold_partial_rows<LANES>(a.part[blockIdx.y], a.nparts, a.cols, int(blockIdx.x));
  const int oc = int(blockIdx.x) * (4 * LANES) + int(threadIdx.x);
  if (threadIdx.x < 4 * LANES && oc < a.cols) Cvt<WT>::store(static_cast<WT*>(a.out[blockIdx.y]) + oc, s);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
template <typename T> struct TypeTag { using type = T; };

// the (weight, input, residual) combinations the reference registers kernels for
template <typename F>
static int dispatch_types(int wtype, int itype, int rtype, const char* who, F&& f) {
#define HK_DAL_CASE(W, I, R, WT, IT, RT) \
  if (wtype == W && itype == I && rtype == R) return f(TypeTag<IT>{}, TypeTag<RT>{}, TypeTag<WT>{})
  HK_DAL_CASE(HK_FLOAT32, HK_FLOAT32, HK_FLOAT32, float, float, float);
  HK_DAL_CASE(HK_FLOAT16, HK_FLOAT16, HK_FLOAT16, fp16, fp16, fp16);
  HK_DAL_CASE(HK_BFLOAT16, HK_BFLOAT16, HK_BFLOAT16, bf16, bf16, bf16);
  HK_DAL_CASE(HK_FLOAT32, HK_FLOAT16, HK_FLOAT32, float, fp16, float);
  HK_DAL_CASE(HK_FLOAT32, HK_BFLOAT16, HK_FLOAT32, float, bf16, float);
  HK_DAL_CASE(HK_FLOAT16, HK_FLOAT16, HK_FLOAT32, fp16, fp16, float);
  HK_DAL_CASE(HK_BFLOAT16, HK_BFLOAT16, HK_FLOAT32, bf16, bf16, float);
  HK_DAL_CASE(HK_FLOAT32, HK_FLOAT16, HK_FLOAT16, float, fp16, fp16);
  HK_DAL_CASE(HK_FLOAT32, HK_BFLOAT16, HK_BFLOAT16, float, bf16, bf16);
  HK_DAL_CASE(HK_FLOAT16, HK_FLOAT32, HK_FLOAT32, fp16, float, float);
#undef HK_DAL_CASE
  set_last_error("%s: no kernel for weight dtype %d, input dtype %d, residual dtype %d", who, wtype, itype,
                 rtype);
  return HK_ERR_UNSUPPORTED;
}

static bool aligned8(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7u) == 0; }

struct BwdShape {
  int tpr, rpb, block, grid;
  int64_t nparts;
};

static BwdShape plan_dal_bwd(int64_t rows, int cols) {
  BwdShape p{};
  const int nchunks = cols / kChunk;
  p.tpr = (nchunks + 63) / 64 * 64;
  p.rpb = p.tpr > 512 ? 1 : 512 / p.tpr;
  const int forced_rpb = tune_get(TUNE_NORM_BWD_ROWS_PER_BLOCK);
  if (forced_rpb > 0) p.rpb = std::max(1, std::min(forced_rpb, 1024 / p.tpr));
  p.block = p.tpr * p.rpb;
  // two 512-thread workgroups (one of 1024) per compute unit
  int64_t grid = int64_t(device_cu_count()) * (p.block > 512 ? 1 : 2);
  if (tune_get(TUNE_NORM_BWD_BLOCKS) > 0) grid = tune_get(TUNE_NORM_BWD_BLOCKS);
  const int64_t useful = (rows + p.rpb - 1) / p.rpb;
  if (grid > useful) grid = useful;
  if (grid < 1) grid = 1;
  p.grid = int(grid);
  p.nparts = grid;
  return p;
}

static int count_parts(const hkDropoutAddLnBwdParams& p) {
  // slots are fixed (dgamma, dbeta, dgamma1, dbeta1, dcolscale); the workspace holds the highest one in use
  int n = 0;
  if (p.dgamma) n = 1;
  if (p.dbeta) n = 2;
  if (p.dgamma1) n = 3;
  if (p.dbeta1) n = 4;
  if (p.dcolscale) n = 5;
  return n;
}

static int check_common(const char* who, int64_t rows, int64_t cols, float dropout_p) {
  HK_REQUIRE(rows >= 0 && cols >= 0, HK_ERR_INVALID, "%s: negative shape", who);
  HK_REQUIRE(rows <= 0x7fffffffLL, HK_ERR_INVALID, "%s: too many rows (%lld)", who, (long long) rows);
  HK_REQUIRE(cols % 8 == 0 && cols <= 8192, HK_ERR_INVALID,
             "%s: hidden size must be a multiple of 8 and at most 8192, got %lld", who, (long long) cols);
  HK_REQUIRE(dropout_p >= 0.f && dropout_p < 1.f, HK_ERR_INVALID, "%s: dropout_p %g outside [0, 1)", who,
             double(dropout_p));
  return HK_OK;
}

} // namespace hk

using namespace hk;

extern "C" {

int hk_dropout_add_ln_fwd_ex(const hkDropoutAddLnFwdParams* pp, hkStream_t stream) {
  const char* who = "hk_dropout_add_ln_fwd_ex";
  HK_REQUIRE(pp != nullptr, HK_ERR_INVALID, "%s: null parameter block", who);
  const hkDropoutAddLnFwdParams& p = *pp;
  int rc = check_common(who, p.rows, p.cols, p.dropout_p);
  if (rc != HK_OK) return rc;
  HK_REQUIRE(p.epsilon >= 0.f, HK_ERR_INVALID, "%s: epsilon must be >= 0", who);
  const bool subset = p.x0_subset != nullptr || p.z_subset != nullptr;
  const bool parallel = p.x1 != nullptr || p.gamma1 != nullptr || p.z1 != nullptr || p.beta1 != nullptr ||
                        p.dmask1 != nullptr;
  HK_REQUIRE(!subset || (p.x0_subset && p.z_subset), HK_ERR_INVALID,
             "%s: x0_subset and z_subset come together", who);
  HK_REQUIRE(!subset || (p.x0_numrows >= 0 && p.z_numrows >= 0), HK_ERR_INVALID,
             "%s: negative x0_numrows / z_numrows", who);
  HK_REQUIRE(!(parallel && (subset || p.rowscale || p.colscale)), HK_ERR_UNSUPPORTED,
             "%s: the parallel-residual form takes no rowscale, colscale or row subsets", who);
  HK_REQUIRE(!p.gamma1 || p.z1, HK_ERR_INVALID, "%s: gamma1 given without z1", who);
  HK_REQUIRE(!(p.z1 || p.beta1) || p.gamma1, HK_ERR_INVALID, "%s: z1 / beta1 given without gamma1", who);
  if (p.rows == 0 || p.cols == 0) return HK_OK;
  HK_REQUIRE(p.x0 && p.gamma && p.z && p.mu && p.rs, HK_ERR_INVALID, "%s: null input/output", who);
  const bool dropout = p.dropout_p > 0.f;
  HK_REQUIRE(!dropout || p.dmask, HK_ERR_INVALID, "%s: dmask is required when dropout_p > 0", who);
  HK_REQUIRE(!dropout || !p.x1 || p.dmask1, HK_ERR_INVALID,
             "%s: dmask1 is required when dropout_p > 0 and x1 is given", who);
  HK_REQUIRE(aligned16(p.x0) && aligned16(p.x1) && aligned16(p.residual) && aligned16(p.gamma) &&
                 aligned16(p.beta) && aligned16(p.gamma1) && aligned16(p.beta1) && aligned16(p.colscale) &&
                 aligned16(p.z) && aligned16(p.z1) && aligned16(p.x) && aligned8(p.dmask) && aligned8(p.dmask1),
             HK_ERR_INVALID, "%s: data pointers must be 16-byte aligned (masks 8-byte)", who);

  // nothing beyond the plain interface: the tuned row kernels take it
  const bool plain = !dropout && !subset && !parallel && !p.rowscale && !p.colscale &&
                     p.itype == p.rtype && p.itype == p.wtype;
  if (plain) {
    return hk_dropout_add_ln_fwd(p.itype, p.rtype, p.wtype, p.x0, p.residual, p.gamma, p.beta, p.z, p.x, p.mu,
                                 p.rs, p.rows, p.cols, p.epsilon, p.is_rms_norm, stream);
  }

  DalFwdArgs a{};
  a.x0 = p.x0; a.x1 = p.x1; a.residual = p.residual; a.gamma = p.gamma; a.beta = p.beta;
  a.gamma1 = p.gamma1; a.beta1 = p.beta1; a.rowscale = subset ? nullptr : p.rowscale; a.colscale = p.colscale;
  a.x0_subset = p.x0_subset; a.z_subset = p.z_subset;
  a.z = p.z; a.z1 = p.z1; a.x = p.x; a.dmask = p.dmask; a.dmask1 = p.dmask1; a.mu = p.mu; a.rs = p.rs;
  a.rows = p.rows; a.x0_numrows = subset ? p.x0_numrows : p.rows; a.z_numrows = subset ? p.z_numrows : p.rows;
  a.cols = int(p.cols); a.nchunks = int(p.cols) / kChunk;
  a.eps = p.epsilon; a.inv_cols = 1.0f / float(p.cols);
  a.scale = 1.0f / (1.0f - p.dropout_p); a.rowscale_const = p.rowscale_const;
  a.is_rms = p.is_rms_norm ? 1 : 0; a.dropout = dropout ? 1 : 0;
  a.drop.seed_lo = uint32_t(p.seed); a.drop.seed_hi = uint32_t(p.seed >> 32);
  a.drop.off_lo = uint32_t(p.offset); a.drop.off_hi = uint32_t(p.offset >> 32);
  a.drop.keep_max = keep_max(1.0f - p.dropout_p);

  // chunks per thread: the fewest that keep a row within 256 threads
  const int nc = a.nchunks <= 256 ? 1 : (a.nchunks <= 512 ? 2 : 4);
  a.tpr = dal_fwd_threads(a.nchunks, nc);
  const int rpb = std::max(1, 256 / a.tpr);
  const dim3 block{unsigned(a.tpr * rpb)}, grid{unsigned((p.rows + rpb - 1) / rpb)};
  hipStream_t s = as_hip(stream);
  return dispatch_types(p.wtype, p.itype, p.rtype, who, [&](auto it, auto rt, auto wt) {
    using IT = typename decltype(it)::type;
    using RT = typename decltype(rt)::type;
    using WT = typename decltype(wt)::type;
    auto launch = [&](const auto& given) {
      using A = typename std::decay<decltype(given)>::type;
      // Rows of four chunks a thread, 16 bits: 20 wavefronts a compute unit of the 32 that the flat arguments' 60 registers let in
      // (us, 32 / 20; the others' 72 registers, 28: bf16 3743 x 5000 32.9 / 31.6, 32.2, x 5648 38.1 / 36.0, 36.8, x 6144 38.7 / 36.6, 37.9, 7600 x
      // 5648 69.3 / 65.4, 66.6, x 7512 92.2 / 89.4, 90.3, 12000 x 5376 101.7 / 99.1, 101.9, x 6144 112.1 / 115.0, 111.3).
      const auto resident = [&] {
        size_t lds = 0;
        if (sizeof(A) <= kCheapArgs && sizeof(IT) == 2 && sizeof(RT) == 2)
          lds_bytes_for_residency(std::max(1, 20 / int(block.x / kWave)), sizeof(float) * kMaxWaves * 3, &lds);
        return lds;
      };
      switch (nc) {
        case 1:
          if (dropout) HK_LAUNCH((dal_fwd_kernel<IT, RT, WT, 1, true, A>), grid, block, 0, s, given);
          else HK_LAUNCH((dal_fwd_kernel<IT, RT, WT, 1, false, A>), grid, block, 0, s, given);
          break;
        case 2: HK_LAUNCH((dal_fwd_kernel<IT, RT, WT, 2, true, A>), grid, block, 0, s, given); break;
        default: HK_LAUNCH((dal_fwd_kernel<IT, RT, WT, 4, true, A>), grid, block, resident(), s, given); break;
      }
    };
    profile_before(s);
    if (DalFwdFlat::holds(a)) launch(DalFwdFlat(a));
    else launch(a);
    profile_after(s);
    return launch_check("dal_fwd_kernel");
  });
}

int hk_dropout_add_ln_bwd_ex_workspace_bytes(const hkDropoutAddLnBwdParams* pp, size_t* bytes) {
  const char* who = "hk_dropout_add_ln_bwd_ex_workspace_bytes";
  HK_REQUIRE(pp != nullptr && bytes != nullptr, HK_ERR_INVALID, "%s: null argument", who);
  const hkDropoutAddLnBwdParams& p = *pp;
  *bytes = 0;
  int rc = check_common(who, p.rows, p.cols, p.dropout_p);
  if (rc != HK_OK) return rc;
  if (p.rows == 0 || p.cols == 0) return HK_OK;
  const BwdShape sh = plan_dal_bwd(p.rows, int(p.cols));
  size_t general = size_t(count_parts(p)) * size_t(sh.nparts) * size_t(p.cols) * sizeof(float);
  // a call without extra features is handed to the plain backward, which sizes its own scratch
  size_t plain = 0;
  if (p.itype == p.rtype && p.itype == p.wtype) {
    rc = hk_norm_bwd_workspace_bytes(p.itype, p.rows, p.cols, &plain);
    if (rc != HK_OK) return rc;
  }
  *bytes = std::max(general, plain);
  return HK_OK;
}

int hk_dropout_add_ln_bwd_ex(const hkDropoutAddLnBwdParams* pp, hkStream_t stream) {
  const char* who = "hk_dropout_add_ln_bwd_ex";
  HK_REQUIRE(pp != nullptr, HK_ERR_INVALID, "%s: null parameter block", who);
  const hkDropoutAddLnBwdParams& p = *pp;
  int rc = check_common(who, p.rows, p.cols, p.dropout_p);
  if (rc != HK_OK) return rc;
  const bool subset = p.x0_subset != nullptr || p.z_subset != nullptr;
  const bool g1 = p.gamma1 != nullptr;
  const bool parallel = g1 || p.dz1 != nullptr || p.dx1 != nullptr || p.dmask1 != nullptr ||
                        p.dgamma1 != nullptr || p.dbeta1 != nullptr;
  const bool colscale = p.colscale != nullptr;
  HK_REQUIRE(!subset || (p.x0_subset && p.z_subset), HK_ERR_INVALID,
             "%s: x0_subset and z_subset come together", who);
  HK_REQUIRE(!subset || (p.x0_numrows >= 0 && p.z_numrows >= 0), HK_ERR_INVALID,
             "%s: negative x0_numrows / z_numrows", who);
  HK_REQUIRE(!(parallel && (subset || p.rowscale || colscale)), HK_ERR_UNSUPPORTED,
             "%s: the parallel-residual form takes no rowscale, colscale or row subsets", who);
  HK_REQUIRE(!g1 || p.dz1, HK_ERR_INVALID, "%s: gamma1 given without dz1", who);
  HK_REQUIRE(!(p.dz1 || p.dgamma1 || p.dbeta1) || g1, HK_ERR_INVALID,
             "%s: dz1 / dgamma1 / dbeta1 given without gamma1", who);
  HK_REQUIRE(colscale || !p.dcolscale, HK_ERR_INVALID, "%s: dcolscale given without colscale", who);
  hipStream_t s = as_hip(stream);
  if (p.cols == 0) return HK_OK;
  if (p.rows == 0) {
    // no rows: the column sums are empty sums
    const size_t wbytes = size_t(p.cols) * ((p.wtype == HK_FLOAT32) ? 4 : 2);
    void* outs[kMaxParts] = {p.dgamma, p.dbeta, p.dgamma1, p.dbeta1, p.dcolscale};
    for (void* o : outs) {
      if (o) {
        rc = hk_memset(o, 0, wbytes, stream);
        if (rc != HK_OK) return rc;
      }
    }
    return HK_OK;
  }
  HK_REQUIRE(p.dz && p.x && p.mu && p.rs && p.gamma && p.dx0, HK_ERR_INVALID, "%s: null input/output", who);
  const bool dropout = p.dropout_p > 0.f;
  HK_REQUIRE(!dropout || p.dmask, HK_ERR_INVALID, "%s: dmask is required when dropout_p > 0", who);
  HK_REQUIRE(!dropout || !p.dx1 || p.dmask1, HK_ERR_INVALID,
             "%s: dmask1 is required when dropout_p > 0 and dx1 is wanted", who);
  HK_REQUIRE(!colscale || p.x0, HK_ERR_INVALID, "%s: x0 is required with colscale", who);
  HK_REQUIRE(aligned16(p.dz) && aligned16(p.dz1) && aligned16(p.dx) && aligned16(p.x) && aligned16(p.x0) &&
                 aligned16(p.gamma) && aligned16(p.gamma1) && aligned16(p.colscale) && aligned16(p.dx0) &&
                 aligned16(p.dx1) && aligned16(p.dresidual) && aligned8(p.dmask) && aligned8(p.dmask1),
             HK_ERR_INVALID, "%s: data pointers must be 16-byte aligned (masks 8-byte)", who);

  const bool plain = !dropout && !subset && !parallel && !p.rowscale && !colscale &&
                     p.itype == p.rtype && p.itype == p.wtype;
  if (plain) {
    return hk_dropout_add_ln_bwd(p.itype, p.rtype, p.wtype, p.dz, p.dx, p.x, p.mu, p.rs, p.gamma, p.dx0,
                                 p.dresidual, p.dgamma, p.dbeta, p.rows, p.cols, p.is_rms_norm, p.workspace,
                                 p.workspace_bytes, stream);
  }

  BwdShape sh = plan_dal_bwd(p.rows, int(p.cols));
  // the pre-norm residual block has a kernel of its own; it keeps two rows in flight per
  // thread group and runs best with one workgroup per compute unit (measured: 264 us against 283 us with
  // two at [32768 x 4096] bf16, 29.6 against 32.3 us at
  // [16384 x 768]).  The workspace was sized for the larger grid.
  const bool stream_form = dropout && p.dx && p.dresidual && !subset && !p.rowscale && !colscale && !parallel &&
                           tune_get(TUNE_NORM_BWD_PREFETCH) != 1;
  if (stream_form && tune_get(TUNE_NORM_BWD_BLOCKS) <= 0 && sh.grid > device_cu_count()) {
    sh.grid = device_cu_count();
    sh.nparts = sh.grid;
  }
  const int nslots = count_parts(p);
  const size_t slot_floats = size_t(sh.nparts) * size_t(p.cols);
  const size_t need = size_t(nslots) * slot_floats * sizeof(float);
  if (nslots > 0) {
    HK_REQUIRE(p.workspace != nullptr && p.workspace_bytes >= need, HK_ERR_WORKSPACE,
               "%s: workspace of %zu bytes needed, %zu given", who, need, p.workspace_bytes);
    HK_REQUIRE(aligned16(p.workspace), HK_ERR_INVALID, "%s: workspace must be 16-byte aligned", who);
  }

  DalBwdArgs a{};
  a.dz = p.dz; a.dz1 = p.dz1; a.dx = p.dx; a.x = p.x; a.x0 = p.x0; a.dmask = p.dmask; a.dmask1 = p.dmask1;
  a.mu = p.mu; a.rs = p.rs; a.gamma = p.gamma; a.gamma1 = p.gamma1;
  a.rowscale = subset ? nullptr : p.rowscale; a.colscale = p.colscale;
  a.x0_subset = p.x0_subset; a.z_subset = p.z_subset;
  a.dx0 = p.dx0; a.dx1 = p.dx1; a.dresidual = p.dresidual;
  void* outs[kMaxParts] = {p.dgamma, p.dbeta, p.dgamma1, p.dbeta1, p.dcolscale};
  for (int k = 0; k < kMaxParts; ++k)
    a.part[k] = outs[k] ? static_cast<float*>(p.workspace) + size_t(k) * slot_floats : nullptr;
  a.rows = p.rows; a.x0_numrows = subset ? p.x0_numrows : p.rows; a.z_numrows = subset ? p.z_numrows : p.rows;
  a.cols = int(p.cols); a.nchunks = int(p.cols) / kChunk; a.tpr = sh.tpr;
  a.inv_cols = 1.0f / float(p.cols); a.scale = 1.0f / (1.0f - p.dropout_p); a.rowscale_const = p.rowscale_const;
  a.is_rms = p.is_rms_norm ? 1 : 0; a.dropout = dropout ? 1 : 0;

  DalFoldArgs fold{};
  int wanted = 0;
  for (int k = 0; k < kMaxParts; ++k)
    if (outs[k]) { fold.part[wanted] = a.part[k]; fold.out[wanted++] = outs[k]; }
  fold.nparts = int(sh.nparts); fold.cols = int(p.cols);

  const dim3 grid{unsigned(sh.grid)}, block{unsigned(sh.block)};
  return dispatch_types(p.wtype, p.itype, p.rtype, who, [&](auto it, auto rt, auto wt) {
    using IT = typename decltype(it)::type;
    using RT = typename decltype(rt)::type;
    using WT = typename decltype(wt)::type;
    profile_before(s);
    // two rows in flight where the ring fits the registers (a 16-bit residual stream), else one
    constexpr int PF = sizeof(RT) == 2 ? 2 : 1;
    const bool full = int(p.cols) / kChunk == sh.tpr;
    const size_t lds = sh.rpb > 1 ? size_t(sh.rpb) * size_t(p.cols) * sizeof(float) : 0;
    const DalStreamArgs f{a.dz, a.dx, a.x, a.dmask, a.mu, a.rs, a.gamma, a.dx0, a.dresidual, {a.part[0], a.part[1]},
                          uint32_t(a.rows) | (a.is_rms ? 0x80000000u : 0u), uint32_t(a.cols), a.inv_cols, a.scale,
                          uint16_t(a.tpr), uint16_t(sh.block), uint32_t(sh.grid)};
    // dal_bwd_small_kernel where it measured faster, forward and backward, us, two launches of the backward / one: bf16 64 x 512 12.5 /
    // 9.7, 256 x 4096 15.8 / 10.4, 768 x 2048 15.5 / 12.3, x 8192 36.6 / 29.6, 1024 x 512 12.5 / 10.8, x 8192 40.8 / 37.6, 1500 x 1024
    // 15.1 / 15.5, x 8192 53.6 / 51.6; fp32 256 x 8192 28.8 / 24.1, 768 x 1024 15.8 / 12.4, x 4096 31.2 / 28.9, x 6144 45.6 / 47.8, 1024 x
    // 2048 23.2 / 22.7, x 4096 38.7 / 39.0.
    const int64_t n = p.rows * p.cols, ni = n * int64_t(sizeof(IT)), nr = n * int64_t(sizeof(RT)), nw = p.cols * int64_t(sizeof(WT)),
                  ns = p.rows * int64_t(sizeof(float));
    const Span dz{p.dz, ni}, dx{p.dx, nr}, x{p.x, nr}, mask{p.dmask, n}, mu{p.mu, ns}, rs{p.rs, ns}, gamma{p.gamma, nw};
    const Span dx0{p.dx0, ni}, dresidual{p.dresidual, nr}, dgamma{p.dgamma, nw}, dbeta{p.dbeta, nw};
    // (dresidual may be dx: an element of it is read by the thread that stores it.  What two launches write over each other, the
    // column sums win.)
    const bool one_launch = apart({dx0, dgamma, dbeta}, {dz, dx, x, mask, mu, rs, gamma}) && apart({dresidual}, {dz, x, mask, mu, rs, gamma}) &&
                            apart({dgamma, dbeta}, {dx0, dresidual});
    if (stream_form && one_launch && p.rows <= (sizeof(RT) == 2 ? 1024 : 768) && nr <= (int64_t(16) << 20) &&
        tune_get(TUNE_NORM_BWD_BLOCKS) <= 0 && tune_get(TUNE_NORM_BWD_ROWS_PER_BLOCK) <= 0) {
      const int lanes = sizeof(RT) == 2 ? 8 : 4, rpb = kSmallThreads / sh.tpr;
      DalStreamArgs few = f;
      few.part[0] = static_cast<float*>(p.dgamma);
      few.part[1] = static_cast<float*>(p.dbeta);
      few.blocks = wanted ? uint32_t((a.nchunks + lanes - 1) / lanes) : 0;   // (the rest to the same bits without them)
      HK_LAUNCH((dal_bwd_small_kernel<IT, RT, WT>), dim3(few.blocks + unsigned((p.rows + rpb - 1) / rpb)), dim3(kSmallThreads), 0, s, few);
      profile_after(s);
      return launch_check("dal_bwd_small_kernel");
    }
    if (stream_form && full && sh.tpr == 512 && sh.block == 512) HK_LAUNCH((dal_bwd_stream_kernel<IT, RT, WT, PF, 512>), grid, block, lds, s, f);
    else if (stream_form) HK_LAUNCH((dal_bwd_stream_kernel<IT, RT, WT, PF, 0>), grid, block, lds, s, f);
    else if (g1) HK_LAUNCH((dal_bwd_kernel<IT, RT, WT, false, true>), grid, block, lds, s, a);
    else if (colscale) HK_LAUNCH((dal_bwd_kernel<IT, RT, WT, true, false>), grid, block, lds, s, a);
    else HK_LAUNCH((dal_bwd_kernel<IT, RT, WT, false, false>), grid, block, lds, s, a);
    profile_after(s);
    int r = launch_check("dal_bwd_kernel");
    if (r != HK_OK || wanted == 0) return r;
    auto launch_fold = [&](auto kernel, int lanes) {
      HK_LAUNCH(kernel, dim3(unsigned((p.cols + 4 * lanes - 1) / (4 * lanes)), unsigned(wanted)), dim3(unsigned(fold_threads(lanes))), 0, s,
                fold);
    };
    if (fold_lanes(int(p.cols), wanted) == 8) launch_fold(dal_fold_kernel<WT, 8>, 8);
    else launch_fold(dal_fold_kernel<WT, 32>, 32);
    return launch_check("dal_fold_kernel");
  });
}

} // extern "C"
