// Shared declarations of the LayerNorm / RMSNorm kernels: argument blocks, launch plans and the per-dtype entry
// points that the dispatch in hk_norm.hip calls.  The kernels themselves live in hk_norm_fwd_impl.h and
// hk_norm_bwd_impl.h and are instantiated once per storage type in hk_norm_{fwd,bwd}_{f32,bf16,f16}.hip, so
// that the types compile in parallel.
#pragma once

#include "hk_common.h"

#include <algorithm>
#include <type_traits>

namespace hk {

// Rows are `cols` elements long and lie `*_pitch` elements apart (pitch == cols for a dense array; a wider
// pitch is a column slice of a wider buffer).  Pitches are in elements of the array's type.
struct NormFwdArgs {
  const void* x;
  const void* residual;
  const void* gamma;
  const void* beta;
  void* y;
  void* x_out;
  void* mean;
  void* stat;
  int64_t rows;
  int64_t x_pitch, res_pitch, y_pitch, xout_pitch;
  // rows on several levels (see LevelSteps), in walk order: n0 * n1 * n2 = rows; one level is n0 = rows
  int64_t n0, n1, n2;
  RowNumbering rn;
  LevelSteps x_lv, res_lv, y_lv, xout_lv;
  int cols;
  int nvec;
  int spare;             // see RaggedRow
  uint16_t threads;      // of a workgroup
  float eps;
  float inv_cols;
  int is_rms;
  int stat_kind;
  int stats_f32;
  __device__ __forceinline__ const NormFwdArgs& args() const { return *this; }
};

// The same of rows on one level, all but the forward of two rows per workgroup, which only large arrays take (see kCheapArgs):
// 16 rows of 4096 bf16 columns with a residual 4.7 -> 4.4 us a call, LayerNorm of 145 x 320, forward and backward, 12.7 -> 12.0.
struct NormFwdFlat {
  const void* x;
  const void* residual;
  const void* gamma;
  const void* beta;
  void* y;
  void* x_out;
  void* mean;
  void* stat;
  uint32_t rows, cols, nvec;
  uint32_t x_pitch, res_pitch, y_pitch, xout_pitch;
  float eps, inv_cols;
  uint16_t threads;
  uint8_t spare, flags;   // flags: bit 0 is_rms, 1 stats_f32, from 2 on stat_kind
  // whether rows below 2^31 elements apart, on one level, are all that a holds
  static bool holds(const NormFwdArgs& a) {
    const int64_t far = std::max(std::max(a.x_pitch, a.y_pitch), std::max(a.residual ? a.res_pitch : 0, a.x_out ? a.xout_pitch : 0));
    return a.n0 == a.rows && a.rows <= 0x7fffffff && far <= 0x7fffffff;
  }
  explicit NormFwdFlat(const NormFwdArgs& a)
      : x(a.x), residual(a.residual), gamma(a.gamma), beta(a.beta), y(a.y), x_out(a.x_out), mean(a.mean), stat(a.stat),
        rows(uint32_t(a.rows)), cols(uint32_t(a.cols)), nvec(uint32_t(a.nvec)), x_pitch(uint32_t(a.x_pitch)),
        res_pitch(a.residual ? uint32_t(a.res_pitch) : 0), y_pitch(uint32_t(a.y_pitch)), xout_pitch(a.x_out ? uint32_t(a.xout_pitch) : 0), eps(a.eps), inv_cols(a.inv_cols),
        threads(uint16_t(a.threads)), spare(uint8_t(a.spare)),
        flags(uint8_t((a.is_rms ? 1 : 0) | (a.stats_f32 ? 2 : 0) | a.stat_kind << 2)) {}
  __device__ __forceinline__ NormFwdArgs args() const {
    NormFwdArgs a{};
    a.x = x; a.residual = residual; a.gamma = gamma; a.beta = beta; a.y = y; a.x_out = x_out; a.mean = mean; a.stat = stat;
    a.rows = a.n0 = rows; a.n1 = a.n2 = 1;
    a.rn = RowNumbering{1, 0, 0};
    a.x_pitch = x_pitch; a.res_pitch = res_pitch; a.y_pitch = y_pitch; a.xout_pitch = xout_pitch;
    a.cols = int(cols); a.nvec = int(nvec); a.spare = spare; a.eps = eps; a.inv_cols = inv_cols; a.threads = threads;
    a.is_rms = flags & 1; a.stats_f32 = flags >> 1 & 1; a.stat_kind = flags >> 2;
    return a;
  }
};
static_assert(sizeof(NormFwdFlat) <= kCheapArgs, "");

enum NormBwdMode { BWD_LN = 0, BWD_RMS = 1, BWD_LN_MEMEFF = 2 };

struct NormBwdArgs {
  const void* dy;
  const void* x;        // forward input, or forward output in BWD_LN_MEMEFF
  const void* gamma;
  const void* beta;     // BWD_LN_MEMEFF only
  const void* mean;
  const void* stat;
  const void* dx_in;    // optional upstream gradient added to dx
  void* dx;
  void* dres;           // optional second copy of dx (dresidual)
  float* part_dgamma;   // [grid, cols]
  float* part_dbeta;    // [grid, cols]
  int64_t rows;
  int64_t dy_pitch, x_pitch, dx_pitch, dxin_pitch, dres_pitch;
  // rows on several levels (see LevelSteps), in walk order; the walking kernel splits its walk index itself
  int64_t n0, n1, n2;
  RowNumbering rn;
  uint32_t ws0, ws1, ws2;   // the walking kernel's row stride (its grid size) split over the walk levels
  LevelSteps dy_lv, x_lv, dx_lv, dxin_lv, dres_lv;
  int cols;
  int nvec;
  int part_pitch;       // elements between partial rows: cols rounded up to whole vectors
  int tpr;              // threads per row
  float eps;
  float inv_cols;
  int stat_kind;
  int stats_f32;
  int clamp_gamma;
  uint16_t threads;     // of a workgroup
  int blocks;           // of the launch
  template <typename T, int MODE> __device__ __forceinline__ const NormBwdArgs& args() const { return *this; }
};

// What the lean instances take of it: rows on one level, no optional operands (see kCheapArgs)
struct NormBwdFlat {
  const void* dy;
  const void* x;
  const void* gamma;
  const void* mean;     // BWD_LN_MEMEFF, which has none: beta
  const void* stat;
  void* dx;
  float* part_dgamma;
  float* part_dbeta;
  uint32_t rows, cols, dy_pitch, x_pitch, dx_pitch, blocks;
  float eps, inv_cols;
  uint16_t tpr, threads;
  uint8_t stat_kind, clamp_gamma;
  // whether rows below 2^31 elements apart, on one level, are all that a holds beside optional operands
  static bool holds(const NormBwdArgs& a) {
    return a.n0 == a.rows && a.rows <= 0x7fffffff && std::max(std::max(a.dy_pitch, a.x_pitch), a.dx_pitch) <= 0x7fffffff;
  }
  NormBwdFlat(const NormBwdArgs& a, int mode)
      : dy(a.dy), x(a.x), gamma(a.gamma), mean(mode == BWD_LN_MEMEFF ? a.beta : a.mean), stat(a.stat), dx(a.dx),
        part_dgamma(a.part_dgamma), part_dbeta(a.part_dbeta), rows(uint32_t(a.rows)), cols(uint32_t(a.cols)), dy_pitch(uint32_t(a.dy_pitch)),
        x_pitch(uint32_t(a.x_pitch)), dx_pitch(uint32_t(a.dx_pitch)), blocks(uint32_t(a.blocks)), eps(a.eps), inv_cols(a.inv_cols),
        tpr(uint16_t(a.tpr)), threads(uint16_t(a.threads)), stat_kind(uint8_t(a.stat_kind)), clamp_gamma(uint8_t(a.clamp_gamma)) {}
  template <typename T, int MODE>
  __device__ __forceinline__ NormBwdArgs args() const {
    NormBwdArgs a{};
    a.dy = dy; a.x = x; a.gamma = gamma; a.stat = stat; a.dx = dx; a.part_dgamma = part_dgamma; a.part_dbeta = part_dbeta;
    if constexpr (MODE == BWD_LN_MEMEFF) a.beta = mean;
    else a.mean = mean;
    a.rows = a.n0 = rows; a.n1 = a.n2 = 1;
    a.dy_pitch = dy_pitch; a.x_pitch = x_pitch; a.dx_pitch = dx_pitch;
    a.cols = int(cols);
    a.nvec = (a.cols + VecIO<T>::N - 1) / VecIO<T>::N;
    a.part_pitch = a.nvec * VecIO<T>::N;
    a.tpr = tpr; a.threads = threads; a.blocks = int(blocks); a.eps = eps; a.inv_cols = inv_cols;
    a.stat_kind = stat_kind; a.clamp_gamma = clamp_gamma;
    return a;
  }
};
static_assert(sizeof(NormBwdFlat) <= kCheapArgs, "");

struct BwdPlan {
  bool reg_path;
  bool any;             // the instance for rows of any length and alignment
  int lpr;              // lanes of a wavefront that hold a row; 0: whole wavefronts, with a barrier per row
  int tpr, nv, rpb, grid;
  int block;
  size_t lds_bytes;
  size_t ws_bytes;
};

static inline int pow2_ceil(int v) {
  int p = 1;
  while (p < v) p <<= 1;
  return p;
}

template <typename T>
__device__ __forceinline__ void store_stat(void* base, int64_t row, float v, int stats_f32) {
  if (base == nullptr) return;
  if (stats_f32) static_cast<float*>(base)[row] = v;
  else Cvt<T>::store(static_cast<T*>(base) + row, v);
}

template <typename CT>
__device__ __forceinline__ CT block_sum_generic(CT v, CT* lds) {
  const int tid = threadIdx.x;
  lds[tid] = v;
  __syncthreads();
  for (int s = 256 >> 1; s > 0; s >>= 1) {
    if (tid < s) lds[tid] += lds[tid + s];
    __syncthreads();
  }
  CT r = lds[0];
  __syncthreads();
  return r;
}

template <typename T, typename CT>
struct GenericIO {
  static __device__ __forceinline__ CT ld(const T* p) { return CT(Cvt<T>::load(p)); }
  static __device__ __forceinline__ void st(T* p, CT v) { Cvt<T>::store(p, v); }
};

// Per-type entry points (T = float, bf16, fp16), defined by the explicit instantiations.
template <typename T> int norm_fwd_typed(NormFwdArgs a, hipStream_t s);
template <typename T> BwdPlan plan_norm_bwd(int64_t rows, int cols, bool aligned);
template <typename T> BwdPlan plan_norm_bwd_lanes(int64_t rows, int cols);
template <typename T> int norm_bwd_typed(NormBwdArgs a, int mode, void* dgamma, void* dbeta, void* ws,
                                          size_t ws_bytes, hipStream_t s);
// double precision: one workgroup per row, arithmetic in double (with the fp32 instantiations)
int norm_fwd_f64(const NormFwdArgs& a, hipStream_t s);
int norm_bwd_f64(const NormBwdArgs& a, int mode, void* dgamma, void* dbeta, hipStream_t s);

} // namespace hk
