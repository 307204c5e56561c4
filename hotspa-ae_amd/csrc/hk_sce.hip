// Fused softmax cross-entropy forward / backward for gfx950 (sparse int64
// labels with an ignored index, and dense labels).
//
// A logits row is read from HBM once and kept in registers; each thread folds
// its elements into a (max, sum-of-exp) pair, pairs are merged online across
// lanes (DPP) and waves (LDS).  Forward writes one loss per row; backward
// rescales the stored exponentials into (softmax - onehot) * grad_loss and
// writes the row once.  Rows whose label equals the ignored index are not read
// at all: loss 0 / a zero gradient row is written.
//
// Sparse labels take rows of any length and alignment this way (see RowSpan); 16-bit rows of 32768 to 97792 columns keep
// a part in LDS (RowTail, sce_packed_kernel), longer ones are streamed (sce_long_kernel).
#include "hk_common.h"

#include <algorithm>

namespace hk {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr float kNegInf = -__builtin_huge_valf();

struct SceArgs {
  const void* logits;
  const int64_t* labels;   // sparse
  const void* dlabels;     // dense labels (same shape as logits)
  const void* grad_loss;   // backward
  void* out;               // forward: loss [rows]; backward: dlogits
  int64_t rows;
  // elements between the starts of consecutive rows of logits / dense labels / dlogits (0 = dense: cols)
  int64_t x_pitch, lab_pitch, out_pitch;
  // rows on several levels (see LevelSteps); one level: n0 = rows.  labels, losses, per-row gradients and
  // statistics are dense [rows] arrays and take the row's number
  int64_t n0, n1, n2;
  RowNumbering rn;
  LevelSteps x_lv, lab_lv, out_lv;
  int cols;
  int nvec;
  int64_t ignored_index;
  // sparse forward on a column shard [vocab_start, vocab_start + cols) of a wider row: instead of a loss,
  // stats[0..rows) = the shard's row maximum, stats[rows..2 rows) = sum of exp(x - that maximum),
  // stats[2 rows..3 rows) = the logit at the label when the label falls into the shard, else 0
  float* stats;
  int64_t vocab_start;
  // backward of a reduced loss: grad_loss holds ONE value (the gradient of the mean / sum) and every row uses
  // round_T(that value * grad_scale), which is what broadcasting it times 1/rows into a [rows] array of the
  // storage type first would have handed to this kernel
  int grad_scalar;
  double grad_scale;
  uint16_t threads;   // of a workgroup
};
// What the kernels take of it (see kCheapArgs); steps below 2^31 elements, what lies further apart goes out in several launches.
// Loss per token and gradient of 678 x 2432 fp16 8.5 -> 7.85 us a pass.
struct SceFlat {
  const void* logits;
  const void* labels;        // sparse or dense
  const void* grad_loss;     // forward: stats
  void* out;
  int64_t ignored_index;
  union {
    double grad_scale;
    int64_t vocab_start;     // forward
  };
  uint32_t rows, n0, x_pitch, lab_pitch, out_pitch, rn0, rn1, rn2;
  ShortLevelSteps x_lv, out_lv;
  int cols;
  uint16_t threads;
  uint8_t grad_scalar;
  // MODE as in sce_generic_kernel
  template <int MODE>
  static SceFlat of(const SceArgs& a) {
    SceFlat f{};
    f.logits = a.logits; f.out = a.out; f.ignored_index = a.ignored_index;
    f.labels = MODE < 2 ? static_cast<const void*>(a.labels) : a.dlabels;
    if (MODE & 1) { f.grad_loss = a.grad_loss; f.grad_scale = a.grad_scale; f.grad_scalar = uint8_t(a.grad_scalar != 0); }
    else { f.grad_loss = a.stats; f.vocab_start = a.vocab_start; }
    f.rows = uint32_t(a.rows); f.n0 = uint32_t(a.n0); f.cols = a.cols; f.threads = a.threads;
    f.rn0 = uint32_t(a.rn.rn0); f.rn1 = uint32_t(a.rn.rn1); f.rn2 = uint32_t(a.rn.rn2);
    // (a step of a level of one row is not taken; one of an operand that the mode has not neither)
    if (a.n0 > 1) { f.x_pitch = uint32_t(a.x_pitch); f.lab_pitch = uint32_t(MODE < 2 ? 0 : a.lab_pitch); f.out_pitch = uint32_t(MODE & 1 ? a.out_pitch : 0); }
    if (a.n1 > 1) { f.x_lv.p1 = int(a.x_lv.p1); f.out_lv.p1 = int(MODE & 1 ? a.out_lv.p1 : 0); }
    if (a.n2 > 1) { f.x_lv.p2 = int(a.x_lv.p2); f.out_lv.p2 = int(MODE & 1 ? a.out_lv.p2 : 0); }
    return f;
  }
  template <typename T, int MODE>
  __device__ __forceinline__ SceArgs args() const {
    SceArgs a{};
    a.logits = logits; a.out = out; a.ignored_index = ignored_index;
    if constexpr (MODE < 2) a.labels = static_cast<const int64_t*>(labels);
    else a.dlabels = labels;
    if constexpr (MODE & 1) { a.grad_loss = grad_loss; a.grad_scale = grad_scale; a.grad_scalar = grad_scalar; }
    else if constexpr (MODE == 0) { a.stats = static_cast<float*>(const_cast<void*>(grad_loss)); a.vocab_start = vocab_start; }
    a.rows = rows; a.n0 = n0; a.cols = cols; a.threads = threads;
    a.nvec = int((uint32_t(cols) + VecIO<T>::N - 1) / VecIO<T>::N);
    a.x_pitch = x_pitch; a.lab_pitch = lab_pitch; a.out_pitch = out_pitch;
    a.rn = RowNumbering{rn0, rn1, rn2};
    a.x_lv = LevelSteps{x_lv.p1, x_lv.p2}; a.out_lv = LevelSteps{out_lv.p1, out_lv.p2};
    return a;
  }
};
static_assert(sizeof(SceFlat) <= kCheapArgs, "");

template <typename T, typename CT>
__device__ __forceinline__ CT sce_row_grad(const SceArgs& a, int64_t row) {
  const T* gp = static_cast<const T*>(a.grad_loss);
  if (!a.grad_scalar) return CT(Cvt<T>::load(gp + row));
  T rounded;
  Cvt<T>::store(&rounded, CT(Cvt<T>::load(gp)) * CT(a.grad_scale));
  return CT(Cvt<T>::load(&rounded));
}

// i0: the row's place within the innermost level (blockIdx.y / z are the outer levels); row: its number
template <bool WAVE_ROW>
__device__ __forceinline__ void row_coords(const SceArgs& a, int& tpr, int& t, int64_t& i0, int64_t& row, int& nwaves) {
  tpr = WAVE_ROW ? kWave : a.threads;
  t = WAVE_ROW ? int(threadIdx.x & 63) : int(threadIdx.x);
  i0 = WAVE_ROW ? int64_t(blockIdx.x) * (256 / kWave) + wave_index() : int64_t(blockIdx.x);
  row = dense_row_index(i0, a.rn);
  nwaves = WAVE_ROW ? 1 : a.threads >> 6;
}

// Rows whose maximum lies at the type's lowest or highest values (past_log2_range(p.v[0]) after the reduction): the sum
// and the gradient from the row itself.
template <typename T, bool WAVE_ROW>
__device__ __forceinline__ float sce_extreme_count(const T* xr, int cols, int t, int tpr, int nwaves, float* red, float& M) {
  return row_max_count<T>(xr, cols, t, tpr, [&](auto v) {
    if constexpr (WAVE_ROW) return wave_allreduce_tuple(v);
    else { __syncthreads(); return group_allreduce_tuple(v, red, 0, nwaves); }   // red may still be read
  }, M);
}
template <typename T, bool WAVE_ROW>
__device__ __forceinline__ void sce_extreme_bwd(const T* xr, T* dxr, int cols, int lab, float g, int t, int tpr, int nwaves,
                                                float* red) {
  float M;
  const float n = sce_extreme_count<T, WAVE_ROW>(xr, cols, t, tpr, nwaves, red, M);
  const float scale = g / (M == kNegInf ? __builtin_nanf("") : n);   // a row of nothing but -inf has no softmax
  for (int64_t c = t; c < cols; c += tpr)
    Cvt<T>::store(dxr + c, (Cvt<T>::load(xr + c) == M ? 1.f : 0.f) * scale - (c == lab ? g : 0.f));
}

// ------------------------------- sparse forward ----------------------------
// A row as the 16-byte vectors that lie on 16-byte boundaries of the logits, and up to 2 (N - 1) elements before and
// after them, one of which each of the first 2 N threads takes.  The order of a row's elements does not matter to its
// sum, and accesses that straddle cache lines cost more than the few single ones: 4096 x 50257 bf16, vectors counted
// from the row's start (odd 2-byte boundaries) against this: forward 100 / 83 us, backward 216 / 160 us.
// RAGGED == false: whole vectors on the grid, nothing else.
template <typename T, bool RAGGED>
struct RowSpan {
  static constexpr int N = VecIO<T>::N;
  int head, nvec, edge;   // elements before the vectors; vectors; column of this thread's single element, or -1
  __device__ __forceinline__ RowSpan(const T* row, int cols, int t) : head(0), nvec(uint32_t(cols) / N), edge(-1) {
    if constexpr (RAGGED) {
      const int past = int(reinterpret_cast<uintptr_t>(row) & 15u) / int(sizeof(T));
      head = min((N - past) & (N - 1), cols);
      nvec = (cols - head) / N;
      const int rest = head + nvec * N, k = t - N;
      if (t < head) edge = t;
      else if (k >= 0 && k < cols - rest) edge = rest + k;
    }
  }
  // vector v, -inf past the last one (inside: it is known to be there, uniform).  KEEP: the row is read again
  template <bool KEEP>
  __device__ __forceinline__ u32x4 load(const T* row, int v, bool inside) const {
    u32x4 raw = neg_inf_vec<T>();
    if (inside || v < nvec) {
      if constexpr (RAGGED) raw = KEEP ? ld16_any_keep<T>(row + head + v * N) : ld16_any<T>(row + head + v * N);
      else raw = KEEP ? ld16_keep(row + v * N) : ld16(row + v * N);
    }
    return raw;
  }
  // (the output may lie on another phase of the 16-byte grid than the logits)
  __device__ __forceinline__ void store(T* row, int v, const float* f) const {
    if constexpr (RAGGED) st16_any(row + head + v * N, VecIO<T>::pack(f));
    else st16_stream(row + v * N, VecIO<T>::pack(f));
  }
  // the vector that holds column c and its place in it; no thread's vector when a single element or none does.  In scalar
  // registers, as c is: compared per lane, the gradient's one-hot term cost 5 to 7 % of a short row (30000 x 512 bf16 15.5
  // against 14.8 us)
  struct Place { int vec, element; };
  __device__ __forceinline__ Place place_of(int c) const {
    const int at = c - head;
    return {at < 0 ? -1 : int(uint32_t(at) / N), at & (N - 1)};
  }
  __device__ __forceinline__ float load_edge(const T* row) const {
    return RAGGED && edge >= 0 ? Cvt<T>::load(row + edge) : kNegInf;
  }
  __device__ __forceinline__ void store_edge(T* row, float v) const {
    if (RAGGED && edge >= 0) Cvt<T>::store(row + edge, v);
  }
};

// what the forward writes for an ignored row, and for one whose (ML, sum, maximum) is p (one thread per row)
template <typename T>
__device__ __forceinline__ void sce_store_ignored(const SceArgs& a, int64_t row) {
  if (a.stats) {
    a.stats[row] = kNegInf;
    a.stats[a.rows + row] = 0.f;
    a.stats[2 * a.rows + row] = 0.f;
  } else {
    Cvt<T>::store(static_cast<T*>(a.out) + row, 0.f);
  }
}
template <typename T>
__device__ __forceinline__ void sce_store_loss(const SceArgs& a, int64_t row, int64_t label, const T* xr,
                                               const MaxSumMaxTuple& p) {
  const float M = p.v[2];
  if (a.stats) {
    // sum exp(x - M) = S * 2^(ML - M * log2e); 0 where nothing but -inf is, NaN where a NaN is among it
    a.stats[row] = M;
    a.stats[a.rows + row] = (M == kNegInf) ? p.v[1] * 0.f
        : past_log2_range(p.v[0]) ? p.v[1] : p.v[1] * __builtin_amdgcn_exp2f(-fmaf(M, kLog2e, -p.v[0]));
    const int64_t local = label - a.vocab_start;
    a.stats[2 * a.rows + row] = (local >= 0 && local < a.cols) ? Cvt<T>::load(xr + local) : 0.f;
    return;
  }
  float r;
  if (label >= 0 && label < a.cols) {
    const float xl = Cvt<T>::load(xr + label);
    // sum exp(x - M) = S * 2^(ML - M * log2e); the fma recovers the rounding of ML exactly
    // (a row of extreme values has its sum relative to M itself)
    const float log2s = __builtin_amdgcn_logf(p.v[1]) - (past_log2_range(p.v[0]) ? 0.f : fmaf(M, kLog2e, -p.v[0]));
    // M - xl first: the difference of two logits is (nearly) exact however large their common offset is, and
    // the sum then rounds at the size of the loss, not of the logits
    r = log2s * kLn2 + (M - xl);
  } else {
    r = __builtin_nanf("");  // label outside [0, cols): no logit to gather
  }
  Cvt<T>::store(static_cast<T*>(a.out) + row, r);
}

template <typename T, int NV, bool WAVE_ROW, bool RAGGED>
__global__ __launch_bounds__(WAVE_ROW ? 256 : 1024)
void sce_sparse_fwd_kernel(SceFlat given) {
  const SceArgs a = given.args<T, 0>();
  constexpr int VEC = VecIO<T>::N;
  __shared__ float red[kMaxWaves * 3];
  int tpr, t, nwaves;
  int64_t i0, row;
  row_coords<WAVE_ROW>(a, tpr, t, i0, row, nwaves);
  if (WAVE_ROW && i0 >= a.n0) return;

  const int64_t label = a.labels[row];
  if (label == a.ignored_index) {          // uniform over the row's threads
    if (t == 0) sce_store_ignored<T>(a, row);
    return;
  }
  const T* xr = static_cast<const T*>(a.logits) + i0 * a.x_pitch + outer_level_offset(a.x_lv);
  // slots past the row's end hold -inf: they change neither the maximum nor the sum
  const RowSpan<T, RAGGED> span(xr, a.cols, t);
  float f[NV * VEC];
  float edge;
  {
    u32x4 raw[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i)
      raw[i] = span.template load<false>(xr, i * tpr + t, (i + 1) * tpr <= span.nvec);
    edge = span.load_edge(xr);
#pragma unroll
    for (int i = 0; i < NV; ++i) VecIO<T>::unpack(raw[i], &f[i * VEC]);
  }
  static_assert((NV * VEC) % 2 == 0, "pairs of elements per max3");
  float m = RAGGED ? max3(edge, f[0], f[1]) : fmaxf(f[0], f[1]);
#pragma unroll
  for (int e = 2; e < NV * VEC; e += 2) m = max3(m, f[e], f[e + 1]);
  // ml: this thread's maximum in the log2 domain, rounded once (see OnlineSoftmaxTuple)
  const float ml = log2_of_max(m);
  // four independent chains: the exponential unit's latency is not serialised behind one accumulator
  float s4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int e = 0; e < NV * VEC; ++e) s4[e & 3] += __builtin_amdgcn_exp2f(fmaf(f[e], kLog2e, -ml));
  if constexpr (RAGGED) s4[0] += __builtin_amdgcn_exp2f(fmaf(edge, kLog2e, -ml));
  const float s = (s4[0] + s4[1]) + (s4[2] + s4[3]);
  MaxSumMaxTuple p;
  p.v[0] = ml; p.v[1] = s; p.v[2] = m;
  p = WAVE_ROW ? wave_allreduce_tuple(p) : group_allreduce_tuple(p, red, 0, nwaves);
  if (past_log2_range(p.v[0])) p.v[1] = sce_extreme_count<T, WAVE_ROW>(xr, a.cols, t, tpr, nwaves, red, p.v[2]);   // uniform
  if (t == 0) sce_store_loss<T>(a, row, label, xr, p);
}

// ------------------------------- sparse backward ---------------------------
// A 1024-thread workgroup is four wavefronts on every SIMD: two such workgroups fit a compute unit only at the
// full eight wavefronts per SIMD, i.e. at 64 registers or fewer.  The second launch bound asks the compiler for
// that; without it the kernel came out at 68 registers and ran with one workgroup per compute unit (448 us
// instead of 345 us at 16384 x 32000 bf16).  Eight fp32 vectors per thread do not fit 64 registers and keep the
// looser bound.
template <typename T, int NV>
constexpr int sce_min_waves(bool wave_row) { return wave_row ? 1 : (sizeof(T) == 4 && NV == 8 ? 4 : 8); }

// the label's column if the row has it, else one that no vector holds
__device__ __forceinline__ int sce_label_column(int64_t label, int cols) {
  return label >= 0 && label < cols ? int(label) : -1;
}

// a zero gradient row for an ignored label
template <typename T, bool RAGGED>
__device__ __forceinline__ void sce_store_zero_row(T* dxr, int cols, int t, int tpr) {
  const RowSpan<T, RAGGED> span(dxr, cols, t);
  const float zero[VecIO<T>::N] = {};
  for (int v = t; v < span.nvec; v += tpr) span.store(dxr, v, zero);
  span.store_edge(dxr, 0.f);
}

// The vectors of a row past NV per thread, kept in LDS as they were loaded: [rounds][threads].  A wavefront reads back what
// it loaded itself (directly, through no register), so there is no barrier; `arrived` waits for it.
template <typename T, int NV>
struct RowTail {
  const RowSpan<T, true>& span;
  u32x4* lds;
  int t, tpr;
  __device__ __forceinline__ void load(const T* row) const {
    for (int v = NV * tpr, k = 0; v < span.nvec; v += tpr, k += tpr) {
      if (v + t < span.nvec) {   // lane i's 16 bytes go to the wavefront's address + 16 i
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(row + span.head + (v + t) * span.N),
                                         (__attribute__((address_space(3))) void*)(lds + k + wave_index() * kWave), 16, 0,
                                         kBufStream);
      }
    }
  }
  static __device__ __forceinline__ void arrived() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
  // f(unpacked elements, index of the vector) for this thread's share
  template <typename F>
  __device__ __forceinline__ void each(F&& f) const {
    for (int v = NV * tpr + t, k = t; v < span.nvec; v += tpr, k += tpr) {
      float e[RowSpan<T, true>::N];
      VecIO<T>::unpack(lds[k], e);
      f(e, v);
    }
  }
};

template <typename T, int NV, bool WAVE_ROW, bool RAGGED, bool TAIL = false>
__global__ __launch_bounds__(WAVE_ROW ? 256 : 1024, (sce_min_waves<T, NV>(WAVE_ROW)))
void sce_sparse_bwd_kernel(SceFlat given) {
  const SceArgs a = given.args<T, 1>();
  constexpr int VEC = VecIO<T>::N;
  extern __shared__ __align__(16) u32x4 tail_lds[];   // TAIL: the row's vectors past NV per thread
  __shared__ float red[kMaxWaves * 2];
  int tpr, t, nwaves;
  int64_t i0, row;
  row_coords<WAVE_ROW>(a, tpr, t, i0, row, nwaves);
  if (WAVE_ROW && i0 >= a.n0) return;

  T* dxr = static_cast<T*>(a.out) + i0 * a.out_pitch + outer_level_offset(a.out_lv);
  const int64_t label = a.labels[row];
  if (label == a.ignored_index) {
    sce_store_zero_row<T, RAGGED>(dxr, a.cols, t, tpr);
    return;
  }
  const T* xr = static_cast<const T*>(a.logits) + i0 * a.x_pitch + outer_level_offset(a.x_lv);
  // slots past the row's end hold -inf: they change neither the maximum nor the sum
  const RowSpan<T, RAGGED> span(xr, a.cols, t);
  u32x4 raw[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i)
    raw[i] = span.template load<false>(xr, i * tpr + t, (i + 1) * tpr <= span.nvec);
  [[maybe_unused]] float edge = span.load_edge(xr);
  const auto tail = [&] { if constexpr (TAIL) return RowTail<T, NV>{span, tail_lds, t, tpr}; else return 0; }();
  if constexpr (TAIL) tail.load(xr);
  const float g = sce_row_grad<T, float>(a, row);
  float e[NV * VEC];
#pragma unroll
  for (int i = 0; i < NV; ++i) VecIO<T>::unpack(raw[i], &e[i * VEC]);
  static_assert((NV * VEC) % 2 == 0, "pairs of elements per max3");
  float m = RAGGED ? max3(edge, e[0], e[1]) : fmaxf(e[0], e[1]);
#pragma unroll
  for (int k = 2; k < NV * VEC; k += 2) m = max3(m, e[k], e[k + 1]);
  if constexpr (TAIL) {
    tail.arrived();
    tail.each([&](const float* f, int) {
#pragma unroll
      for (int j = 0; j < VEC; j += 2) m = max3(m, f[j], f[j + 1]);
    });
  }
  const float ml = log2_of_max(m);
  // four independent chains, as in the forward kernel
  float s4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < NV * VEC; ++k) {
    e[k] = __builtin_amdgcn_exp2f(fmaf(e[k], kLog2e, -ml));
    s4[k & 3] += e[k];
  }
  if constexpr (RAGGED) {
    edge = __builtin_amdgcn_exp2f(fmaf(edge, kLog2e, -ml));
    s4[0] += edge;
  }
  if constexpr (TAIL) {
    tail.each([&](const float* f, int) {
#pragma unroll
      for (int j = 0; j < VEC; ++j) s4[j & 3] += __builtin_amdgcn_exp2f(fmaf(f[j], kLog2e, -ml));
    });
  }
  const float s = (s4[0] + s4[1]) + (s4[2] + s4[3]);
  MaxSumTuple p;
  p.v[0] = ml; p.v[1] = s;
  p = WAVE_ROW ? wave_allreduce_tuple(p) : group_allreduce_tuple(p, red, 0, nwaves);
  const int lab = sce_label_column(label, a.cols);
  if (past_log2_range(p.v[0])) {   // uniform
    sce_extreme_bwd<T, WAVE_ROW>(xr, dxr, a.cols, lab, g, t, tpr, nwaves, red);
    return;
  }
  const auto place = span.place_of(lab);
  const float scale = __builtin_amdgcn_exp2f(ml - p.v[0]) / p.v[1] * g;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int v = i * tpr + t;
    if (v < span.nvec) {
#pragma unroll
      for (int j = 0; j < VEC; ++j) e[i * VEC + j] *= scale;
      if (v == place.vec) {
#pragma unroll
        for (int j = 0; j < VEC; ++j)
          if (j == place.element) e[i * VEC + j] -= g;
      }
      span.store(dxr, v, &e[i * VEC]);
    }
  }
  if constexpr (TAIL) {
    const float inv = g / p.v[1];
    tail.each([&](float* f, int v) {
#pragma unroll
      for (int j = 0; j < VEC; ++j) f[j] = __builtin_amdgcn_exp2f(fmaf(f[j], kLog2e, -p.v[0])) * inv;
      if (v == place.vec) {
#pragma unroll
        for (int j = 0; j < VEC; ++j)
          if (j == place.element) f[j] -= g;
      }
      span.store(dxr, v, f);
    });
  }
  if constexpr (RAGGED) {
    float d = edge * scale - (span.edge == lab ? g : 0.f);
    // a row of one class (uniform; such a row has no vectors): the element over itself is exactly one and its gradient
    // exactly zero, where the line above, contracted, leaves the rounding error of 1 / edge
    if (a.cols == 1) d = edge / p.v[1] * g - (lab == 0 ? g : 0.f);
    span.store_edge(dxr, d);
  }
}

// ------------------------------- long rows ---------------------------------
// Sparse labels, rows that do not fit a workgroup's registers (32768 fp32 elements) and LDS (97792 16-bit ones): the workgroup
// streams the row, kLongVecs vectors per thread and step, and every thread keeps a running (maximum, sum of exponentials) that it re-bases once per step.
// The backward reads the row a second time, from its end, so that what was read last is found in the nearest cache
// (1024 x 128256 bf16 116 -> 111 us), and is bound by what that second read costs: 1024 x 128256 bf16 679 us by
// elements -> 111 us (4.7 TB/s of row and gradient), forward 307 -> 48 us (5.5 TB/s).  Every step has as many threads
// as its share of the row needs (4096 x 50257 bf16, which has kernels of its own now: 160 and 83 us, with 1024
// throughout 167 and 86 us).
constexpr int kLongThreads = 1024;
constexpr int kLongVecs = 4;

template <typename T, bool BWD>
__global__ __launch_bounds__(kLongThreads, 8)
void sce_long_kernel(SceFlat given) {
  const SceArgs a = given.args<T, (BWD ? 1 : 0)>();
  constexpr int VEC = VecIO<T>::N;
  constexpr int U = kLongVecs, NE = U * VEC;
  __shared__ float red[kMaxWaves * 3];
  const int t = int(threadIdx.x), tpr = a.threads, nwaves = tpr >> 6;
  const int64_t i0 = blockIdx.x, row = dense_row_index(i0, a.rn);
  const int64_t label = a.labels[row];
  T* dxr = BWD ? static_cast<T*>(a.out) + i0 * a.out_pitch + outer_level_offset(a.out_lv) : nullptr;
  if (label == a.ignored_index) {
    if constexpr (BWD) sce_store_zero_row<T, true>(dxr, a.cols, t, tpr);
    else if (t == 0) sce_store_ignored<T>(a, row);
    return;
  }
  const T* xr = static_cast<const T*>(a.logits) + i0 * a.x_pitch + outer_level_offset(a.x_lv);
  const RowSpan<T, true> span(xr, a.cols, t);
  const float edge = span.load_edge(xr);
  float m = edge, ml = log2_of_max(m);
  float s = edge == kNegInf ? 0.f : __builtin_amdgcn_exp2f(fmaf(edge, kLog2e, -ml));
#pragma nounroll
  for (int base = 0; base < span.nvec; base += U * tpr) {
    u32x4 raw[U];
    if (base + U * tpr <= span.nvec) {   // uniform
#pragma unroll
      for (int i = 0; i < U; ++i) raw[i] = span.template load<BWD>(xr, base + i * tpr + t, true);
    } else {
#pragma unroll
      for (int i = 0; i < U; ++i) raw[i] = span.template load<BWD>(xr, base + i * tpr + t, false);
    }
    float f[NE];
#pragma unroll
    for (int i = 0; i < U; ++i) VecIO<T>::unpack(raw[i], &f[i * VEC]);
    const float before = ml;
#pragma unroll
    for (int e = 0; e < NE; e += 2) m = max3(m, f[e], f[e + 1]);
    ml = log2_of_max(m);
    float s4[4] = {s * __builtin_amdgcn_exp2f(before - ml), 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < NE; ++e) s4[e & 3] += __builtin_amdgcn_exp2f(fmaf(f[e], kLog2e, -ml));
    s = (s4[0] + s4[1]) + (s4[2] + s4[3]);
  }
  if constexpr (!BWD) {
    MaxSumMaxTuple p;
    p.v[0] = ml; p.v[1] = s; p.v[2] = m;
    p = group_allreduce_tuple(p, red, 0, nwaves);
    if (past_log2_range(p.v[0])) p.v[1] = sce_extreme_count<T, false>(xr, a.cols, t, tpr, nwaves, red, p.v[2]);   // uniform
    if (t == 0) sce_store_loss<T>(a, row, label, xr, p);
  } else {
    const float g = sce_row_grad<T, float>(a, row);
    MaxSumTuple p;
    p.v[0] = ml; p.v[1] = s;
    p = group_allreduce_tuple(p, red, 0, nwaves);
    const int lab = sce_label_column(label, a.cols);
    if (past_log2_range(p.v[0])) {   // uniform
      sce_extreme_bwd<T, false>(xr, dxr, a.cols, lab, g, t, tpr, nwaves, red);
      return;
    }
    const auto place = span.place_of(lab);
    const float ML = p.v[0];
    const float scale = g / p.v[1];
    auto grad = [&](float x, bool at_label) {
      const float o = __builtin_amdgcn_exp2f(fmaf(x, kLog2e, -ML)) * scale;
      return at_label ? o - g : o;
    };
#pragma nounroll
    for (int base = (span.nvec - 1) / (U * tpr) * (U * tpr); base >= 0; base -= U * tpr) {
      u32x4 raw[U];
#pragma unroll
      for (int i = 0; i < U; ++i) raw[i] = span.template load<false>(xr, base + i * tpr + t, false);
#pragma unroll
      for (int i = 0; i < U; ++i) {
        const int v = base + i * tpr + t;
        if (v < span.nvec) {
          float o[VEC];
          VecIO<T>::unpack(raw[i], o);
#pragma unroll
          for (int j = 0; j < VEC; ++j) o[j] = grad(o[j], false);
          if (v == place.vec) {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
              if (j == place.element) o[j] -= g;
          }
          span.store(dxr, v, o);
        }
      }
    }
    span.store_edge(dxr, grad(edge, span.edge == lab));
  }
}

// --------------------------- rows kept as loaded ---------------------------
// Sparse labels, 16-bit rows longer than 32768 columns: kPackedVecs vectors per thread stay in registers as they were loaded
// and are unpacked once per pass (maximum, sum, gradient), the rest of the row is kept in LDS (RowTail), so that the row is
// read once and four, three or two rows share a compute unit (pick_sce_long_shape; 64 registers or fewer: 46 forward, 58
// backward).  Bound by HBM in the forward, and by how far the loads, the arithmetic (two exponentials an element) and the
// stores of two rows overlap in the backward.  us, forward / backward, streamed by sce_long_kernel and so: 4096 x 50257 bf16
// 95 / 168 and 65 / 145 (up to 65024 columns the backward is sce_sparse_bwd_kernel's), 2500 x 80000 74 / 164 and 68 / 145, 4096 x
// 65536 102 / 200 and 86 / 183.
constexpr int kPackedVecs = 8;

// The compiler would keep the unpacked elements from one pass to the next otherwise: twice the registers.
template <int NV>
__device__ __forceinline__ void unpack_again(u32x4 (&raw)[NV]) {
#pragma unroll
  for (int i = 0; i < NV; ++i) asm volatile("" : "+v"(raw[i]));
}

template <typename T, bool BWD>
__global__ __launch_bounds__(1024, 8)
void sce_packed_kernel(SceFlat given) {
  const SceArgs a = given.args<T, (BWD ? 1 : 0)>();
  constexpr int VEC = VecIO<T>::N, NV = kPackedVecs;
  extern __shared__ __align__(16) u32x4 tail_lds[];   // the vectors past NV per thread
  __shared__ float red[kMaxWaves * 3];
  const int t = int(threadIdx.x), tpr = a.threads, nwaves = tpr >> 6;
  const int64_t i0 = blockIdx.x, row = dense_row_index(i0, a.rn);
  const int64_t label = a.labels[row];
  T* dxr = BWD ? static_cast<T*>(a.out) + i0 * a.out_pitch + outer_level_offset(a.out_lv) : nullptr;
  if (label == a.ignored_index) {
    if constexpr (BWD) sce_store_zero_row<T, true>(dxr, a.cols, t, tpr);
    else if (t == 0) sce_store_ignored<T>(a, row);
    return;
  }
  const T* xr = static_cast<const T*>(a.logits) + i0 * a.x_pitch + outer_level_offset(a.x_lv);
  const RowSpan<T, true> span(xr, a.cols, t);
  u32x4 raw[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i)
    raw[i] = span.template load<false>(xr, i * tpr + t, (i + 1) * tpr <= span.nvec);
  const float edge = span.load_edge(xr);
  const RowTail<T, NV> tail{span, tail_lds, t, tpr};
  tail.load(xr);
  float m = edge;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    float f[VEC];
    VecIO<T>::unpack(raw[i], f);
#pragma unroll
    for (int j = 0; j < VEC; j += 2) m = max3(m, f[j], f[j + 1]);
  }
  tail.arrived();
  tail.each([&](const float* f, int) {
#pragma unroll
    for (int j = 0; j < VEC; j += 2) m = max3(m, f[j], f[j + 1]);
  });
  const float ml = log2_of_max(m);
  unpack_again(raw);
  float s4[4] = {__builtin_amdgcn_exp2f(fmaf(edge, kLog2e, -ml)), 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    float f[VEC];
    VecIO<T>::unpack(raw[i], f);
#pragma unroll
    for (int j = 0; j < VEC; ++j) s4[j & 3] += __builtin_amdgcn_exp2f(fmaf(f[j], kLog2e, -ml));
  }
  tail.each([&](const float* f, int) {
#pragma unroll
    for (int j = 0; j < VEC; ++j) s4[j & 3] += __builtin_amdgcn_exp2f(fmaf(f[j], kLog2e, -ml));
  });
  const float s = (s4[0] + s4[1]) + (s4[2] + s4[3]);
  if constexpr (!BWD) {
    MaxSumMaxTuple p;
    p.v[0] = ml; p.v[1] = s; p.v[2] = m;
    p = group_allreduce_tuple(p, red, 0, nwaves);
    if (past_log2_range(p.v[0])) p.v[1] = sce_extreme_count<T, false>(xr, a.cols, t, tpr, nwaves, red, p.v[2]);   // uniform
    if (t == 0) sce_store_loss<T>(a, row, label, xr, p);
  } else {
    const float g = sce_row_grad<T, float>(a, row);
    MaxSumTuple p;
    p.v[0] = ml; p.v[1] = s;
    p = group_allreduce_tuple(p, red, 0, nwaves);
    const int lab = sce_label_column(label, a.cols);
    if (past_log2_range(p.v[0])) {   // uniform
      sce_extreme_bwd<T, false>(xr, dxr, a.cols, lab, g, t, tpr, nwaves, red);
      return;
    }
    const auto place = span.place_of(lab);
    const float ML = p.v[0], scale = g / p.v[1];
    const auto put = [&](float* o, int v) {
#pragma unroll
      for (int j = 0; j < VEC; ++j) o[j] = __builtin_amdgcn_exp2f(fmaf(o[j], kLog2e, -ML)) * scale;
      if (v == place.vec) {
#pragma unroll
        for (int j = 0; j < VEC; ++j)
          if (j == place.element) o[j] -= g;
      }
      span.store(dxr, v, o);
    };
    unpack_again(raw);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int v = i * tpr + t;
      if (v < span.nvec) {
        float o[VEC];
        VecIO<T>::unpack(raw[i], o);
        put(o, v);
      }
    }
    tail.each(put);
    span.store_edge(dxr, __builtin_amdgcn_exp2f(fmaf(edge, kLog2e, -ML)) * scale - (span.edge == lab ? g : 0.f));
  }
}

// ------------------------------- dense labels ------------------------------
// loss = (M + log S) * sum(l) - sum(l * x);  dx = (softmax - l) * g
template <typename T, int NV, bool WAVE_ROW, bool BWD>
__global__ __launch_bounds__(WAVE_ROW ? 256 : 1024, (sce_min_waves<T, NV>(WAVE_ROW)))
void sce_dense_kernel(SceFlat given) {
  const SceArgs a = given.args<T, (BWD ? 3 : 2)>();
  constexpr int VEC = VecIO<T>::N;
  __shared__ float red[kMaxWaves * 3];
  __shared__ float red2[kMaxWaves * 2];
  int tpr, t, nwaves;
  int64_t i0, row;
  row_coords<WAVE_ROW>(a, tpr, t, i0, row, nwaves);
  if (WAVE_ROW && i0 >= a.n0) return;

  const T* xr = static_cast<const T*>(a.logits) + i0 * a.x_pitch + outer_level_offset(a.x_lv);
  const T* lr = static_cast<const T*>(a.dlabels) + i0 * a.lab_pitch + outer_level_offset(a.lab_lv);
  u32x4 rx[NV], rl[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int v = i * tpr + t;
    rx[i] = u32x4{0, 0, 0, 0};
    rl[i] = u32x4{0, 0, 0, 0};
    if (v < a.nvec) { rx[i] = ld16(xr + v * VEC); rl[i] = ld16(lr + v * VEC); }
  }
  float m = kNegInf;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (i * tpr + t < a.nvec) {
      float f[VEC];
      VecIO<T>::unpack(rx[i], f);
#pragma unroll
      for (int j = 0; j < VEC; ++j) m = fmaxf(m, f[j]);
    }
  }
  const float ml = (m == kNegInf) ? 0.f : m * kLog2e;
  float s = 0.f;
  SumTuple<2> ls;
  ls.v[0] = 0.f; ls.v[1] = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (i * tpr + t < a.nvec) {
      float f[VEC], l[VEC];
      VecIO<T>::unpack(rx[i], f);
      VecIO<T>::unpack(rl[i], l);
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        s += __builtin_amdgcn_exp2f(fmaf(f[j], kLog2e, -ml));
        if constexpr (!BWD) { ls.v[0] += l[j]; ls.v[1] = fmaf(l[j], f[j], ls.v[1]); }
      }
    }
  }
  MaxSumMaxTuple p;
  p.v[0] = (m == kNegInf) ? kNegInf : ml; p.v[1] = s; p.v[2] = m;
  p = WAVE_ROW ? wave_allreduce_tuple(p) : group_allreduce_tuple(p, red, 0, nwaves);
  if constexpr (!BWD) {
    ls = WAVE_ROW ? wave_allreduce_tuple(ls) : group_allreduce_tuple(ls, red2, 0, nwaves);
    if (t == 0) {
      const float M = p.v[2];
      const float log2s = __builtin_amdgcn_logf(p.v[1]) - fmaf(M, kLog2e, -p.v[0]);
      const float lse = log2s * kLn2 + M;
      Cvt<T>::store(static_cast<T*>(a.out) + row, lse * ls.v[0] - ls.v[1]);
    }
  } else {
    const float g = sce_row_grad<T, float>(a, row);
    const float ML = (p.v[0] == kNegInf) ? 0.f : p.v[0];
    const float inv = 1.0f / p.v[1];
    T* dxr = static_cast<T*>(a.out) + i0 * a.out_pitch + outer_level_offset(a.out_lv);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int v = i * tpr + t;
      if (v < a.nvec) {
        float f[VEC], l[VEC];
        VecIO<T>::unpack(rx[i], f);
        VecIO<T>::unpack(rl[i], l);
#pragma unroll
        for (int j = 0; j < VEC; ++j)
          f[j] = (__builtin_amdgcn_exp2f(fmaf(f[j], kLog2e, -ML)) * inv - l[j]) * g;
        const u32x4 o = VecIO<T>::pack(f);
        st16_stream(dxr + v * VEC, o);
      }
    }
  }
}

// ------------------------------- fallback ----------------------------------
// Dense labels of any cols / alignment, and fp64: one workgroup per row, strided passes.
template <typename T, typename CT>
struct SceIO {
  static __device__ __forceinline__ CT ld(const T* p) { return CT(Cvt<T>::load(p)); }
  static __device__ __forceinline__ void st(T* p, CT v) { Cvt<T>::store(p, v); }
};
template <typename CT> __device__ __forceinline__ CT sce_exp(CT v);
template <> __device__ __forceinline__ float sce_exp<float>(float v) { return __builtin_amdgcn_exp2f(v * kLog2e); }
template <> __device__ __forceinline__ double sce_exp<double>(double v) { return exp(v); }
template <typename CT> __device__ __forceinline__ CT sce_log(CT v);
template <> __device__ __forceinline__ float sce_log<float>(float v) { return __builtin_amdgcn_logf(v) * kLn2; }
template <> __device__ __forceinline__ double sce_log<double>(double v) { return log(v); }

template <typename CT>
__device__ __forceinline__ CT sce_block_reduce(CT v, CT* lds, bool is_max) {
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

// MODE 0: sparse fwd, 1: sparse bwd, 2: dense fwd, 3: dense bwd
template <typename T, typename CT, int MODE>
__global__ __launch_bounds__(256)
void sce_generic_kernel(SceArgs a) {
  __shared__ CT lds[256];
  const int64_t i0 = blockIdx.x;
  const int64_t row = dense_row_index(i0, a.rn);
  const int64_t cols = a.cols;
  const T* xr = static_cast<const T*>(a.logits) + i0 * a.x_pitch + outer_level_offset(a.x_lv);
  int64_t label = 0;
  if (MODE < 2) {
    label = a.labels[row];
    if (label == a.ignored_index) {
      if (MODE == 0) {
        if (threadIdx.x == 0) {
          if (a.stats) {
            a.stats[row] = kNegInf;
            a.stats[a.rows + row] = 0.f;
            a.stats[2 * a.rows + row] = 0.f;
          } else {
            SceIO<T, CT>::st(static_cast<T*>(a.out) + row, CT(0));
          }
        }
      } else {
        T* dxr = static_cast<T*>(a.out) + i0 * a.out_pitch + outer_level_offset(a.out_lv);
        for (int64_t c = threadIdx.x; c < cols; c += 256) SceIO<T, CT>::st(dxr + c, CT(0));
      }
      return;
    }
  }
  CT m = -__builtin_huge_val();
  for (int64_t c = threadIdx.x; c < cols; c += 256) {
    const CT v = SceIO<T, CT>::ld(xr + c);
    m = v > m ? v : m;
  }
  m = sce_block_reduce<CT>(m, lds, true);
  CT s = 0;
  for (int64_t c = threadIdx.x; c < cols; c += 256) s += sce_exp<CT>(SceIO<T, CT>::ld(xr + c) - m);
  s = sce_block_reduce<CT>(s, lds, false);
  if (MODE == 0 && a.stats) {
    if (threadIdx.x == 0) {
      const int64_t local = label - a.vocab_start;
      a.stats[row] = float(m);
      a.stats[a.rows + row] = float(s);
      a.stats[2 * a.rows + row] = (local >= 0 && local < cols) ? float(SceIO<T, CT>::ld(xr + local)) : 0.f;
    }
  } else if (MODE == 0) {
    if (threadIdx.x == 0) {
      CT r;
      if (label >= 0 && label < cols) r = sce_log<CT>(s) + (m - SceIO<T, CT>::ld(xr + label));
      else r = CT(__builtin_nanf(""));
      SceIO<T, CT>::st(static_cast<T*>(a.out) + row, r);
    }
  } else if (MODE == 2) {
    const T* lr = static_cast<const T*>(a.dlabels) + i0 * a.lab_pitch + outer_level_offset(a.lab_lv);
    CT sl = 0, slx = 0;
    for (int64_t c = threadIdx.x; c < cols; c += 256) {
      const CT l = SceIO<T, CT>::ld(lr + c);
      sl += l;
      slx += l * SceIO<T, CT>::ld(xr + c);
    }
    sl = sce_block_reduce<CT>(sl, lds, false);
    slx = sce_block_reduce<CT>(slx, lds, false);
    if (threadIdx.x == 0)
      SceIO<T, CT>::st(static_cast<T*>(a.out) + row, (sce_log<CT>(s) + m) * sl - slx);
  } else {
    const CT g = sce_row_grad<T, CT>(a, row);
    const CT inv = CT(1) / s;
    T* dxr = static_cast<T*>(a.out) + i0 * a.out_pitch + outer_level_offset(a.out_lv);
    const T* lr = MODE == 3 ? static_cast<const T*>(a.dlabels) + i0 * a.lab_pitch + outer_level_offset(a.lab_lv) : nullptr;
    for (int64_t c = threadIdx.x; c < cols; c += 256) {
      CT pr = sce_exp<CT>(SceIO<T, CT>::ld(xr + c) - m) * inv;
      if (MODE == 1) pr = (c == label) ? (pr * g - g) : pr * g;
      else pr = (pr - SceIO<T, CT>::ld(lr + c)) * g;
      SceIO<T, CT>::st(dxr + c, pr);
    }
  }
}

static inline int pow2_ceil_sce(int v) {
  int p = 1;
  while (p < v) p <<= 1;
  return p;
}

// least4: the fewest threads that take 4 vectors each
static bool pick_sce_shape(int nvec, int max_nv_wave, int max_nv, int least4, int* threads, int* nv) {
  const int forced = tune_get(TUNE_SCE_THREADS);
  if (forced > 0) {
    int t = std::min(1024, std::max(64, (forced + 63) / 64 * 64));
    int n = pow2_ceil_sce((nvec + t - 1) / t);
    if (n > max_nv) return false;
    *threads = t; *nv = n;
    return true;
  }
  if (nvec <= 64 * max_nv_wave) {
    *threads = 64;
    *nv = pow2_ceil_sce((nvec + 63) / 64);
    return true;
  }
  // long rows, measured at 32000 bf16 columns: the widest vector count the
  // kernel is built for wins (512 threads x 8 vectors beat 1024 x 4 forward).  Fewer than 256 threads, three wavefronts
  // that is, are still better than half the vectors in more of them, most of all where those leave a wavefront idle: us at
  // 8000 x 4100 bf16 forward 192 x 4 15.6, 320 x 2 20.7 (128 x 8 15.8), 6000 x 6144 14.0 and 19.5, 8000 x 2464 fp32 13.8
  // and 18.6; backward, 10326 x 2112 bf16, 192 x 2 16.9, 320 x 1 26.8, 8000 x 4100 192 x 4 24.6, 320 x 2 27.4.
  for (int n = max_nv; n >= 1; n >>= 1) {
    int t = ((nvec + n - 1) / n + 63) / 64 * 64;
    if (t <= 1024 && (t >= (n > 4 ? 256 : n == 4 ? least4 : 192) || n == 1)) { *threads = t; *nv = n; return true; }
  }
  for (int n = 1; n <= max_nv; n <<= 1) {
    int t = ((nvec + n - 1) / n + 63) / 64 * 64;
    if (t <= 1024) { *threads = t; *nv = n; return true; }
  }
  return false;
}

// 16-bit rows with a tail in LDS (threads 0: none).  The forward keeps four rows under way per compute unit where that
// fits (512 threads and up to 39 KiB of LDS each), then three where rows are many and two would leave wavefronts idle (rows x
// 58000, three / two: 750 22.2 / 19.3, 1300 31.7 / 31.6, 4096 80 / 87 us; 4096 x 61000, 960 threads for two, 84 / 89, x 62000, 1024
// threads, 85.0 / 83.4; x 66688 88.5 / 86.6), then two; past 8 vectors in 1024 threads one or two rows per compute unit are
// streamed (packed / streamed: 300 x 66688 14.6 / 13.6, 500 x 97000 21.5 / 20.7, 1024 x 75000 30.5 / 35.2 us); the backward, whose reads and
// writes do not like company, two (4096 x 50257 bf16, rows per compute unit 2 / 3 / 4: forward 78.3 / 69.0 / 65, backward 152 / 154 / 163 us),
// with the exponentials of 4 vectors per thread in registers as far as two tails of less than 64 KiB reach, 65024 columns
// (against packed rows x 33000 102 -> 94, x 50257 152 -> 145; x 65024 181, x 65025 packed 193, x 65536, without a tail, 183
// us).  Longer than 97792 columns, 8 vectors and such a tail: streamed (x 80000, 2500 rows, streamed 74 / 164, so 68 / 145;
// x 97792 79 / 175, x 97793 streamed 80 / 208 us).  fp32 rows, 4096 x 32000 and x 20001, gain nothing: 175 / 178 and 116 / 113 us.
struct SceLongShape {
  int threads;
  bool packed;        // sce_packed_kernel, else sce_sparse_bwd_kernel
  size_t lds_bytes;
};
template <bool BWD>
static SceLongShape pick_sce_long_shape(int nvec, int64_t rows) {
  SceLongShape l{0, false, 0};
  const int64_t cus = device_cu_count();
  if (nvec <= 4 * 1024 || (!BWD && nvec > kPackedVecs * 1024 && rows <= 2 * cus)) return l;
  size_t per_cu = 0, per_block = 0;
  device_lds_bytes(&per_cu, &per_block);
  per_block = std::min<size_t>(per_block, 65536);
  const size_t red = 512;   // the reduction's own array
  const auto fits = [&](int vectors, int rows_per_cu) {
    l.lds_bytes = size_t(std::max(0, vectors) + 63) / 64 * 64 * 16;   // a wavefront's share is whole
    return l.lds_bytes <= per_block - red && l.lds_bytes + red <= per_cu / size_t(rows_per_cu);
  };
  if (BWD && fits(nvec - 4 * 1024, 2)) { l.threads = 1024; return l; }
  l.packed = true;
  for (int per = BWD ? 2 : 4; per >= 2; --per) {
    if (per == 3 && (nvec > kPackedVecs * 960 || rows <= 4 * cus)) continue;
    const int most = per == 4 ? 512 : per == 3 ? 640 : 1024;   // 32 wavefronts in all
    const int threads = std::min(most, ((nvec + kPackedVecs - 1) / kPackedVecs + 63) / 64 * 64);
    if (fits(nvec - kPackedVecs * threads, per)) { l.threads = threads; return l; }
  }
  return l;
}

// MODE as in sce_generic_kernel
template <typename T, int MODE, bool WAVE_ROW, bool RAGGED>
static int launch_sce_nv(SceArgs given, int nv, dim3 grid, dim3 block, hipStream_t s) {
  given.threads = uint16_t(block.x);
  const SceFlat a = SceFlat::of<MODE>(given);
  // fp32 rows of 8 vectors a thread, backward: 20 wavefronts a compute unit where rows are of any boundary or 9 or 10 wavefronts, up to
  // which they fit twice.  56 registers would let 32 in, which the lines that rows share suffer from (us, 32 / 20; with 73 registers
  // 24 were in): 5307 x 11001 81.2 / 78.3, 79.4, x 14001 107.4 / 100.4, 102.3, 9000 x 13001 169 / 158, 161, 1500 x 9001 20.3 / 19.8, 20.8, x
  // 10001 22.7 / 23.4, 22.7, 620 x 18113 18.9 / 17.7, 17.3, x 18112 18.0 / 16.2, 16.2, 4000 x 20480 112.9 / 108.2, 110.5.  Whole vectors, 9000 x 9600 109.8 /
  // 112.9 and x 15104 186.6 / 172.9, are left as they are, and so are longer rows, 620 x 21954 21.3 / 23.6, x 29229 27.9 / 30.8.
  const auto resident = [&](int n) {
    size_t lds = 0;
    const int waves = int(block.x / kWave);
    if (MODE == 1 && !WAVE_ROW && VecIO<T>::N == 4 && n == 8 && waves <= 10 && (RAGGED || waves >= 9))
      lds_bytes_for_residency(20 / waves, sizeof(float) * kMaxWaves * 2, &lds);
    return lds;
  };
#define HK_SCE_LAUNCH(N)                                                                         \
  do {                                                                                           \
    if constexpr (MODE == 0) HK_LAUNCH((sce_sparse_fwd_kernel<T, N, WAVE_ROW, RAGGED>), grid, block, 0, s, a); \
    else if constexpr (MODE == 1) HK_LAUNCH((sce_sparse_bwd_kernel<T, N, WAVE_ROW, RAGGED>), grid, block, resident(N), s, a); \
    else if constexpr (MODE == 2) HK_LAUNCH((sce_dense_kernel<T, N, WAVE_ROW, false>), grid, block, 0, s, a); \
    else HK_LAUNCH((sce_dense_kernel<T, N, WAVE_ROW, true>), grid, block, 0, s, a);       \
  } while (0)
  profile_before(s);
  switch (nv) {
    case 1: HK_SCE_LAUNCH(1); break;
    case 2: HK_SCE_LAUNCH(2); break;
    case 4: HK_SCE_LAUNCH(4); break;
    case 8:
      if constexpr (MODE == 0 || VecIO<T>::N == 4) { HK_SCE_LAUNCH(8); break; }
      [[fallthrough]];
    default:
      set_last_error("softmax cross-entropy: no kernel for %d vectors per thread", nv);
      return HK_ERR_UNSUPPORTED;
  }
#undef HK_SCE_LAUNCH
  profile_after(s);
  return launch_check("sce kernel");
}

template <typename T, int MODE>
static int sce_typed(SceArgs a, hipStream_t s) {
  constexpr int VEC = VecIO<T>::N;
  constexpr bool BWD = (MODE & 1) != 0;
  if constexpr (MODE < 2) {   // (dense labels, a reduced loss and the statistics of a shard come with rows side by side)
    const bool far0 = far_level(a.n0, {a.x_pitch, BWD ? a.out_pitch : 0}), far1 = far_level(a.n1, {a.x_lv.p1, BWD ? a.out_lv.p1 : 0}),
               far2 = far_level(a.n2, {a.x_lv.p2, BWD ? a.out_lv.p2 : 0});
    if (far0 || far1 || far2) {
      return each_near_part(a, far0, far1, far2, [&](SceArgs part, int64_t i, int64_t j, int64_t k) {
        const auto at = [&](int64_t pitch, const LevelSteps& l) { return i * pitch + j * l.p1 + k * l.p2; };
        const int64_t number = i * a.rn.rn0 + j * a.rn.rn1 + k * a.rn.rn2;
        part.logits = static_cast<const T*>(a.logits) + at(a.x_pitch, a.x_lv);
        part.labels = a.labels + number;
        if (BWD) part.grad_loss = static_cast<const T*>(a.grad_loss) + number;
        part.out = static_cast<T*>(a.out) + (BWD ? at(a.out_pitch, a.out_lv) : number);
        return sce_typed<T, MODE>(part, s);
      });
    }
  }
  auto steps_ok = [](int64_t pitch, const LevelSteps& l) { return pitch % VEC == 0 && l.p1 % VEC == 0 && l.p2 % VEC == 0; };
  const bool vec_ok = a.cols % VEC == 0 && aligned16(a.logits) && aligned16(a.dlabels) &&
                      (MODE == 0 || MODE == 2 || (aligned16(a.out) && steps_ok(a.out_pitch, a.out_lv))) &&
                      steps_ok(a.x_pitch, a.x_lv) && (MODE < 2 || steps_ok(a.lab_pitch, a.lab_lv));
  a.nvec = (a.cols + VEC - 1) / VEC;
  // sparse forward only keeps the packed row; the others keep 32 floats or two rows, in a wavefront 16 floats of fp32
  // (10000 x 1634 backward 64 x 8 25.5, 256 x 2 23.4; x 1100 17.5, 192 x 2 16.2 us)
  const int max_nv = (MODE == 0) ? 8 : 32 / VEC;
  // (dense labels, fp32, 64 x 8 / as now, forward and backward: 10000 x 1100 64 / 16 and 64 / 24, x 2048 86 / 26 and 89 / 40)
  const int max_nv_wave = (MODE == 0) ? 8 : 4;
  // Three wavefronts of 4 vectors, 513 to 768 in all, against five or six of 2, us at 16000 rows of 514, 576 and 700 vectors: bf16
  // sparse backward 46.2 / 47.5, 47.6 / 50.4 and 62.3 / 60.6, dense forward 42.3 / 46.4, 45.0 / 46.5 and 55.6 / 60.6, dense backward
  // 69.8 / 65.9, 70.0 / 69.6 and 93.2 / 87.1; fp32 sparse backward 46.6 / 44.9, 47.3 / 47.5 and 61.7 / 58.0, dense forward 42.3 /
  // 39.5, 44.2 / 42.4 and 56.0 / 52.1, dense backward 68.4 / 65.0, 71.0 / 68.3 and 93.8 / 88.1.
  const int least4 = MODE == 0 || (VEC == 8 && MODE != 3) ? 192 : 256;
  int threads = 0, nv = 0;
  const bool shaped = pick_sce_shape(a.nvec, max_nv_wave, max_nv, least4, &threads, &nv);
  const dim3 levels{unsigned(a.n0), unsigned(a.n1), unsigned(a.n2)};
  auto launch = [&](auto ragged) {
    constexpr bool RAGGED = decltype(ragged)::value;
    if (threads == 64) {
      dim3 grid(unsigned((a.n0 + 3) / 4), unsigned(a.n1), unsigned(a.n2)), block(256);
      return launch_sce_nv<T, MODE, true, RAGGED>(a, nv, grid, block, s);
    }
    return launch_sce_nv<T, MODE, false, RAGGED>(a, nv, levels, dim3{unsigned(threads)}, s);
  };
  if constexpr (MODE < 2 && VEC == 8) {
    const SceLongShape l = pick_sce_long_shape<MODE == 1>(a.nvec, a.rows);
    if (l.threads > 0 && tune_get(TUNE_SCE_THREADS) <= 0) {
      const dim3 block{unsigned(l.threads)};
      a.threads = uint16_t(l.threads);
      const SceFlat f = SceFlat::of<MODE>(a);
      profile_before(s);
      if constexpr (MODE == 1) {
        if (l.packed) HK_LAUNCH((sce_packed_kernel<T, true>), levels, block, l.lds_bytes, s, f);
        else HK_LAUNCH((sce_sparse_bwd_kernel<T, 4, false, true, true>), levels, block, l.lds_bytes, s, f);
      } else {
        HK_LAUNCH((sce_packed_kernel<T, false>), levels, block, l.lds_bytes, s, f);
      }
      profile_after(s);
      return launch_check("sce kernel");
    }
  }
  if (vec_ok && shaped) return launch(std::false_type{});
  if constexpr (MODE < 2) {
    if (shaped) return launch(std::true_type{});
    // equal steps: as many threads as the vectors of one step need
    const int steps = (a.nvec + kLongVecs * kLongThreads - 1) / (kLongVecs * kLongThreads);
    const int per_step = (a.nvec + steps * kLongVecs - 1) / (steps * kLongVecs);
    threads = (per_step + 63) / 64 * 64;
    a.threads = uint16_t(threads);
    profile_before(s);
    HK_LAUNCH((sce_long_kernel<T, MODE == 1>), levels, dim3(unsigned(threads)), 0, s, SceFlat::of<MODE>(a));
    profile_after(s);
    return launch_check("sce_long_kernel");
  } else {
    HK_LAUNCH((sce_generic_kernel<T, float, MODE>), levels, dim3(256), 0, s, a);
    return launch_check("sce_generic_kernel");
  }
}

template <int MODE>
static int sce_dispatch(int dtype, SceArgs& a, hipStream_t s, const char* who) {
  HK_REQUIRE(a.rows >= 0 && a.cols >= 0, HK_ERR_INVALID, "%s: negative shape", who);
  if (a.rows == 0) return HK_OK;
  HK_REQUIRE(a.cols > 0, HK_ERR_INVALID, "%s: rows without classes", who);
  HK_REQUIRE(a.rows <= 0x7fffffffLL, HK_ERR_INVALID, "%s: too many rows", who);
  HK_REQUIRE(a.logits && a.out, HK_ERR_INVALID, "%s: null input/output", who);
  HK_REQUIRE(MODE >= 2 || a.labels, HK_ERR_INVALID, "%s: null labels", who);
  HK_REQUIRE(MODE < 2 || a.dlabels, HK_ERR_INVALID, "%s: null labels", who);
  HK_REQUIRE((MODE & 1) == 0 || a.grad_loss, HK_ERR_INVALID, "%s: null grad_loss", who);
  if (a.x_pitch == 0) a.x_pitch = a.cols;
  if (a.lab_pitch == 0) a.lab_pitch = a.cols;
  if (a.out_pitch == 0) a.out_pitch = a.cols;
  if (a.n0 == 0) { a.n0 = a.rows; a.n1 = a.n2 = 1; a.rn = RowNumbering{1, 0, 0}; }   // one level
  HK_REQUIRE(a.n0 == 1 || (a.x_pitch >= a.cols && a.lab_pitch >= a.cols && a.out_pitch >= a.cols), HK_ERR_INVALID,
             "%s: a row pitch is smaller than the %d columns of a row", who, a.cols);
  switch (dtype) {
    case HK_FLOAT32: return sce_typed<float, MODE>(a, s);
    case HK_BFLOAT16: return sce_typed<bf16, MODE>(a, s);
    case HK_FLOAT16: return sce_typed<fp16, MODE>(a, s);
    case HK_FLOAT64:
      HK_LAUNCH((sce_generic_kernel<double, double, MODE>), dim3(unsigned(a.n0), unsigned(a.n1), unsigned(a.n2)),
                dim3(256), 0, s, a);
      return launch_check("sce_generic_kernel<double>");
    default:
      set_last_error("%s: not implemented for dtype %d", who, dtype);
      return HK_ERR_UNSUPPORTED;
  }
}

} // namespace hk

using namespace hk;

extern "C" {

int hk_sce_sparse_fwd(int dtype, const void* logits, const int64_t* labels, void* loss, int64_t rows,
                      int64_t cols, int64_t ignored_index, hkStream_t stream) {
  HK_REQUIRE(cols <= 0x3fffffff, HK_ERR_INVALID, "hk_sce_sparse_fwd: cols too large");
  SceArgs a{};
  a.logits = logits; a.labels = labels; a.out = loss; a.rows = rows; a.cols = int(cols);
  a.ignored_index = ignored_index;
  return sce_dispatch<0>(dtype, a, as_hip(stream), "hk_sce_sparse_fwd");
}

// logits_steps / out_steps (out_steps may be null): the operands' steps in the rows' own order
static int sce_levels(SceArgs& a, const int64_t level_rows[3], const int64_t* logits_steps, const int64_t* out_steps,
                      const char* who) {
  HK_REQUIRE(level_rows, HK_ERR_INVALID, "%s: null level_rows", who);
  const int64_t n0 = level_rows[0], n1 = level_rows[1], n2 = level_rows[2];
  HK_REQUIRE(n0 >= 0 && n1 >= 0 && n2 >= 0, HK_ERR_INVALID, "%s: negative level count", who);
  a.rows = 0;
  if (n0 == 0 || n1 == 0 || n2 == 0) return HK_OK;
  HK_REQUIRE(n0 <= 0x7fffffffLL && n0 * n1 <= 0x7fffffffLL && n0 * n1 * n2 <= 0x7fffffffLL, HK_ERR_INVALID,
             "%s: too many rows", who);
  a.rows = n0 * n1 * n2;
  int64_t key[3] = {0, 0, 0};
  for (int k = 0; k < 3; ++k) key[k] = logits_steps[k] + (out_steps ? out_steps[k] : 0);
  const RowWalk w = plan_row_walk(level_rows, key, /*on_grid=*/true);
  HK_REQUIRE(walk_fits_grid(w), HK_ERR_UNSUPPORTED,
             "%s: two of the three levels must hold at most 65535 rows each (got %lld, %lld, %lld)", who,
             (long long)n0, (long long)n1, (long long)n2);
  a.n0 = w.n[0]; a.n1 = w.n[1]; a.n2 = w.n[2]; a.rn = w.rn;
  walk_steps(w, logits_steps, &a.x_pitch, &a.x_lv);
  if (out_steps) walk_steps(w, out_steps, &a.out_pitch, &a.out_lv);
  return HK_OK;
}

int hk_sce_sparse_fwd_strided_rows(int dtype, const void* logits, const int64_t logits_steps[3],
                                   const int64_t* labels, void* loss, const int64_t level_rows[3], int64_t cols,
                                   int64_t ignored_index, hkStream_t stream) {
  const char* who = "hk_sce_sparse_fwd_strided_rows";
  HK_REQUIRE(logits_steps, HK_ERR_INVALID, "%s: null steps", who);
  HK_REQUIRE(cols >= 0 && cols <= 0x3fffffff, HK_ERR_INVALID, "%s: bad cols", who);
  SceArgs a{};
  int rc = sce_levels(a, level_rows, logits_steps, nullptr, who);
  if (rc != HK_OK) return rc;
  a.logits = logits; a.labels = labels; a.out = loss; a.cols = int(cols);
  a.ignored_index = ignored_index;
  return sce_dispatch<0>(dtype, a, as_hip(stream), who);
}

int hk_sce_sparse_bwd_strided_rows(int dtype, const void* logits, const int64_t logits_steps[3],
                                   const int64_t* labels, const void* grad_loss, void* dlogits,
                                   const int64_t dlogits_steps[3], const int64_t level_rows[3], int64_t cols,
                                   int64_t ignored_index, hkStream_t stream) {
  const char* who = "hk_sce_sparse_bwd_strided_rows";
  HK_REQUIRE(logits_steps && dlogits_steps, HK_ERR_INVALID, "%s: null steps", who);
  HK_REQUIRE(cols >= 0 && cols <= 0x3fffffff, HK_ERR_INVALID, "%s: bad cols", who);
  SceArgs a{};
  int rc = sce_levels(a, level_rows, logits_steps, dlogits_steps, who);
  if (rc != HK_OK) return rc;
  a.logits = logits; a.labels = labels; a.grad_loss = grad_loss; a.out = dlogits; a.cols = int(cols);
  a.ignored_index = ignored_index;
  return sce_dispatch<1>(dtype, a, as_hip(stream), who);
}

int hk_sce_sparse_fwd_pitched(int dtype, const void* logits, int64_t logits_pitch, const int64_t* labels,
                              void* loss, int64_t rows, int64_t cols, int64_t ignored_index, hkStream_t stream) {
  HK_REQUIRE(cols <= 0x3fffffff, HK_ERR_INVALID, "hk_sce_sparse_fwd_pitched: cols too large");
  HK_REQUIRE(logits_pitch > 0, HK_ERR_INVALID, "hk_sce_sparse_fwd_pitched: a row pitch must be positive");
  SceArgs a{};
  a.logits = logits; a.labels = labels; a.out = loss; a.rows = rows; a.cols = int(cols);
  a.x_pitch = logits_pitch; a.ignored_index = ignored_index;
  return sce_dispatch<0>(dtype, a, as_hip(stream), "hk_sce_sparse_fwd_pitched");
}

int hk_sce_sparse_bwd_pitched(int dtype, const void* logits, int64_t logits_pitch, const int64_t* labels,
                              const void* grad_loss, void* dlogits, int64_t dlogits_pitch, int64_t rows,
                              int64_t cols, int64_t ignored_index, hkStream_t stream) {
  HK_REQUIRE(cols <= 0x3fffffff, HK_ERR_INVALID, "hk_sce_sparse_bwd_pitched: cols too large");
  HK_REQUIRE(logits_pitch > 0 && dlogits_pitch > 0, HK_ERR_INVALID,
             "hk_sce_sparse_bwd_pitched: a row pitch must be positive");
  SceArgs a{};
  a.logits = logits; a.labels = labels; a.grad_loss = grad_loss; a.out = dlogits; a.rows = rows;
  a.cols = int(cols); a.x_pitch = logits_pitch; a.out_pitch = dlogits_pitch; a.ignored_index = ignored_index;
  return sce_dispatch<1>(dtype, a, as_hip(stream), "hk_sce_sparse_bwd_pitched");
}

int hk_vocab_parallel_ce_stats(int dtype, const void* logits, const int64_t* labels, float* stats, int64_t rows,
                               int64_t cols, int64_t vocab_start, int64_t ignored_index, hkStream_t stream) {
  HK_REQUIRE(cols <= 0x3fffffff, HK_ERR_INVALID, "hk_vocab_parallel_ce_stats: cols too large");
  HK_REQUIRE(rows == 0 || stats != nullptr, HK_ERR_INVALID, "hk_vocab_parallel_ce_stats: null output");
  SceArgs a{};
  a.logits = logits; a.labels = labels; a.out = stats; a.rows = rows; a.cols = int(cols);
  a.ignored_index = ignored_index; a.stats = stats; a.vocab_start = vocab_start;
  return sce_dispatch<0>(dtype, a, as_hip(stream), "hk_vocab_parallel_ce_stats");
}

int hk_sce_sparse_bwd(int dtype, const void* logits, const int64_t* labels, const void* grad_loss,
                      void* dlogits, int64_t rows, int64_t cols, int64_t ignored_index,
                      hkStream_t stream) {
  HK_REQUIRE(cols <= 0x3fffffff, HK_ERR_INVALID, "hk_sce_sparse_bwd: cols too large");
  SceArgs a{};
  a.logits = logits; a.labels = labels; a.grad_loss = grad_loss; a.out = dlogits; a.rows = rows;
  a.cols = int(cols); a.ignored_index = ignored_index;
  return sce_dispatch<1>(dtype, a, as_hip(stream), "hk_sce_sparse_bwd");
}

int hk_sce_sparse_bwd_reduced(int dtype, const void* logits, const int64_t* labels, const void* grad_output,
                              double scale, void* dlogits, int64_t rows, int64_t cols, int64_t ignored_index,
                              hkStream_t stream) {
  HK_REQUIRE(cols <= 0x3fffffff, HK_ERR_INVALID, "hk_sce_sparse_bwd_reduced: cols too large");
  SceArgs a{};
  a.logits = logits; a.labels = labels; a.grad_loss = grad_output; a.out = dlogits; a.rows = rows;
  a.cols = int(cols); a.ignored_index = ignored_index;
  a.grad_scalar = 1;
  a.grad_scale = round_to_dtype(dtype, scale);
  return sce_dispatch<1>(dtype, a, as_hip(stream), "hk_sce_sparse_bwd_reduced");
}

int hk_sce_dense_bwd_reduced(int dtype, const void* logits, const void* labels, const void* grad_output,
                             double scale, void* dlogits, int64_t rows, int64_t cols, hkStream_t stream) {
  HK_REQUIRE(cols <= 0x3fffffff, HK_ERR_INVALID, "hk_sce_dense_bwd_reduced: cols too large");
  SceArgs a{};
  a.logits = logits; a.dlabels = labels; a.grad_loss = grad_output; a.out = dlogits; a.rows = rows;
  a.cols = int(cols);
  a.grad_scalar = 1;
  a.grad_scale = round_to_dtype(dtype, scale);
  return sce_dispatch<3>(dtype, a, as_hip(stream), "hk_sce_dense_bwd_reduced");
}

int hk_sce_dense_fwd(int dtype, const void* logits, const void* labels, void* loss, int64_t rows,
                     int64_t cols, hkStream_t stream) {
  HK_REQUIRE(cols <= 0x3fffffff, HK_ERR_INVALID, "hk_sce_dense_fwd: cols too large");
  SceArgs a{};
  a.logits = logits; a.dlabels = labels; a.out = loss; a.rows = rows; a.cols = int(cols);
  return sce_dispatch<2>(dtype, a, as_hip(stream), "hk_sce_dense_fwd");
}

int hk_sce_dense_bwd(int dtype, const void* logits, const void* labels, const void* grad_loss,
                     void* dlogits, int64_t rows, int64_t cols, hkStream_t stream) {
  HK_REQUIRE(cols <= 0x3fffffff, HK_ERR_INVALID, "hk_sce_dense_bwd: cols too large");
  SceArgs a{};
  a.logits = logits; a.dlabels = labels; a.grad_loss = grad_loss; a.out = dlogits; a.rows = rows;
  a.cols = int(cols);
  return sce_dispatch<3>(dtype, a, as_hip(stream), "hk_sce_dense_bwd");
}

} // extern "C"
