// Spatial batch normalisation of an NCHW array in training mode, forward and
// backward, with the semantics of cuDNN's cudnnBatchNormalizationForwardTraining /
// cudnnBatchNormalizationBackward in CUDNN_BATCHNORM_SPATIAL mode (what the
// reference calls): per channel over N, H, W.
//
// A channel's data is N runs of H*W contiguous elements, C*H*W apart.  Three forms:
//  - a channel that fits a workgroup's registers (65536 16-bit or 32768 32-bit elements, half of that in the backward): one launch, one workgroup per
//    channel reads it once, agrees on its statistics and writes the result;
//  - longer ones: partial statistics from several workgroups per channel, then a pass whose workgroups merge their
//    channel's partials themselves (the input is read twice, the second time from the memory-side cache where it fits);
//  - fp64 and planes shorter than a 16-byte vector: element by element, three launches.
// The first two take planes of any length and alignment: the partial last vector of a run is read as the run's last whole
// one, the elements it shares with the vector before it are left out of the sums.
#include "hk_common.h"

#include <algorithm>
#include <type_traits>

namespace hk {

template <typename T> struct BnCT { using type = float; };
template <> struct BnCT<double> { using type = double; };

struct BnShape {
  int64_t N, C, HW;
  int64_t per_channel;    // N * HW
  int splits;
};

// A thread's walk over the elements v0, v0 + stride, v0 + 2 stride, ... (< per_channel) of channel c: the offset of the
// current one, kept up by additions (one division per thread at the start, none per element).
struct BnWalk {
  int64_t off;        // offset of the current element
  int64_t in_plane;   // its index inside its H*W plane
  int64_t left;       // elements still to do, the current one included
  int64_t step_off, step_in_plane, wrap_off, hw;
  __device__ __forceinline__ BnWalk(const BnShape& s, int64_t c, int64_t v0, int64_t stride) {
    const int64_t n = v0 / s.HW;
    in_plane = v0 - n * s.HW;
    off = (n * s.C + c) * s.HW + in_plane;
    left = v0 < s.per_channel ? (s.per_channel - v0 + stride - 1) / stride : 0;
    const int64_t q = stride / s.HW;                     // whole planes per step
    step_in_plane = stride - q * s.HW;
    step_off = q * s.C * s.HW + step_in_plane;
    wrap_off = (s.C - 1) * s.HW;                         // from the end of a plane to the same channel of the next image
    hw = s.HW;
  }
  __device__ __forceinline__ void next() {
    in_plane += step_in_plane;
    off += step_off;
    const bool wrap = in_plane >= hw;
    in_plane -= wrap ? hw : 0;
    off += wrap ? wrap_off : 0;
    --left;
  }
};

template <typename CT>
__device__ __forceinline__ CT block_sum(CT v, CT* lds) {
  const int tid = threadIdx.x;
  lds[tid] = v;
  __syncthreads();
  for (int s = 256 >> 1; s > 0; s >>= 1) {
    if (tid < s) lds[tid] += lds[tid + s];
    __syncthreads();
  }
  const CT r = lds[0];
  __syncthreads();
  return r;
}

// (count, mean, M2) of a slice of one channel -> part[(c * splits + split) * 3 ..]
template <typename T, typename CT>
__global__ __launch_bounds__(256)
void bn_stats_kernel(const T* __restrict__ x, BnShape s, CT* __restrict__ part) {
  __shared__ CT lds[256];
  const int64_t c = blockIdx.x;
  const int split = blockIdx.y;
  // per thread: sums of (x - K) and (x - K)^2 about a pivot K, the thread's first element, so that a large common
  // offset of the channel never enters a sum; no division inside the loop
  BnWalk w(s, c, int64_t(split) * 256 + threadIdx.x, int64_t(s.splits) * 256);
  CT cnt = 0, mean = 0, m2 = 0;
  if (w.left > 0) {
    const CT K = CT(Cvt<T>::load(x + w.off));
    CT s1 = 0, s2 = 0;
    cnt = 1;
    for (w.next(); w.left > 0; w.next()) {
      const CT d = CT(Cvt<T>::load(x + w.off)) - K;
      s1 += d;
      s2 += d * d;
      cnt += 1;
    }
    mean = K + s1 / cnt;
    m2 = s2 - s1 * (s1 / cnt);
    m2 = m2 > 0 ? m2 : CT(0);
  }
  // block merge: total count and mean first, then M2 about the block mean
  const CT bcnt = block_sum<CT>(cnt, lds);
  const CT bsum = block_sum<CT>(mean * cnt, lds);
  const CT bmean = bcnt > 0 ? bsum / bcnt : CT(0);
  const CT d = mean - bmean;
  const CT bm2 = block_sum<CT>(m2 + d * d * cnt, lds);
  if (threadIdx.x == 0) {
    CT* o = part + (c * s.splits + split) * 3;
    o[0] = bcnt; o[1] = bmean; o[2] = bm2;
  }
}

// What the statistics of a channel leave behind; returns the inverse standard deviation.  (The running variance takes
// the unbiased estimate, as cuDNN does.)
template <typename PT, typename CT>
__device__ __forceinline__ CT bn_invstd(CT var, double eps) {
  if constexpr (std::is_same<CT, double>::value) return 1.0 / sqrt(var + eps);
  else return 1.0f / sqrtf(var + float(eps));
}
template <typename PT>
struct BnRunning {
  PT mean, var;   // as they were
  __device__ __forceinline__ BnRunning(const PT* running_mean, const PT* running_var, int64_t c)
      : mean(running_mean ? running_mean[c] : PT(0)), var(running_var ? running_var[c] : PT(0)) {}
};
template <typename PT, typename CT>
__device__ __forceinline__ void bn_store_stats(int64_t c, CT cnt, CT mean, CT m2, CT invstd, double momentum,
                                               const BnRunning<PT>& was, PT* running_mean, PT* running_var, PT* save_mean,
                                               PT* save_invstd) {
  if (save_mean) save_mean[c] = PT(mean);
  if (save_invstd) save_invstd[c] = PT(invstd);
  if (running_mean) running_mean[c] = PT((1.0 - momentum) * double(was.mean) + momentum * double(mean));
  if (running_var) {
    const double unbiased = cnt > 1 ? double(m2) / (double(cnt) - 1.0) : double(cnt > 0 ? m2 / cnt : CT(0));
    running_var[c] = PT((1.0 - momentum) * double(was.var) + momentum * unbiased);
  }
}

// One thread per channel: merge the slices; write the saved mean / inverse standard deviation, update the
// running statistics (the running variance takes the unbiased estimate, as cuDNN does), and leave
// coef[c] = scale * invstd, coef[C + c] = mean, coef[2 C + c] = bias for the element-wise pass.
template <typename PT, typename CT>
__global__ __launch_bounds__(256)
void bn_finalize_kernel(const CT* __restrict__ part, int64_t C, int splits, const PT* __restrict__ scale,
                        const PT* __restrict__ bias, double momentum, double eps, PT* running_mean,
                        PT* running_var, PT* save_mean, PT* save_invstd, CT* __restrict__ coef) {
  const int64_t c = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (c >= C) return;
  CT cnt = 0, mean = 0, m2 = 0;
  for (int k = 0; k < splits; ++k) {
    const CT* p = part + (c * splits + k) * 3;
    const CT nb = p[0];
    if (nb <= 0) continue;
    const CT n = cnt + nb;
    const CT delta = p[1] - mean;
    mean += delta * (nb / n);
    m2 += p[2] + delta * delta * (cnt * nb / n);
    cnt = n;
  }
  const CT invstd = bn_invstd<PT, CT>(cnt > 0 ? m2 / cnt : CT(0), eps);
  bn_store_stats<PT, CT>(c, cnt, mean, m2, invstd, momentum, BnRunning<PT>(running_mean, running_var, c), running_mean, running_var,
                         save_mean, save_invstd);
  coef[c] = CT(scale[c]) * invstd;
  coef[C + c] = mean;
  coef[2 * C + c] = CT(bias[c]);
}

// Channel of element v of a dense [N, C, H*W] array, and whether the whole wavefront shares it (it does unless the
// wavefront crosses from one plane into the next): then the channel's coefficients are fetched once per
// wavefront through the scalar unit instead of once per lane.
template <typename IT>
__device__ __forceinline__ IT bn_channel(IT v, IT hw, IT C, bool& uniform) {
  const IT plane = v / hw;
  const IT plane0 = IT(__builtin_amdgcn_readfirstlane(uint32_t(plane)));
  uniform = __builtin_amdgcn_ballot_w64(plane != plane0) == 0;
  return uniform ? plane0 % C : plane % C;
}

// y = (x - mean) * (scale * invstd) + bias; the mean is subtracted first: folding it into the constant term
// would cancel badly for a channel whose mean is large against its spread.  IT: index type (32-bit when the
// array allows it: the per-lane division is then a few instructions).
template <typename T, typename CT, typename IT>
__global__ __launch_bounds__(256)
void bn_apply_kernel(const T* x, T* y, const CT* __restrict__ coef, IT total, IT hw, IT C) {
  const IT v = IT(blockIdx.x) * kStreamThreads + threadIdx.x;
  if (v >= total) return;
  const CT f = CT(Cvt<T>::load(x + size_t(v)));
  bool uniform;
  const IT c = bn_channel<IT>(v, hw, C, uniform);
  CT a, mean, b;
  if (uniform) {
    const IT c0 = IT(__builtin_amdgcn_readfirstlane(uint32_t(c)));
    a = coef[c0]; mean = coef[size_t(C) + c0]; b = coef[2 * size_t(C) + c0];
  } else {
    a = coef[c]; mean = coef[size_t(C) + c]; b = coef[2 * size_t(C) + c];
  }
  Cvt<T>::store(y + size_t(v), (f - mean) * a + b);
}

// per-channel partial sums of dy and dy * (x - mean) * invstd -> part[(c * splits + split) * 2 ..]
template <typename T, typename PT, typename CT>
__global__ __launch_bounds__(256)
void bn_bwd_stats_kernel(const T* __restrict__ dy, const T* __restrict__ x, BnShape s,
                         const PT* __restrict__ save_mean, const PT* __restrict__ save_invstd,
                         CT* __restrict__ part) {
  __shared__ CT lds[256];
  const int64_t c = blockIdx.x;
  const int split = blockIdx.y;
  const CT mean = CT(save_mean[c]), invstd = CT(save_invstd[c]);
  CT sdy = 0, sdyx = 0;
  for (BnWalk w(s, c, int64_t(split) * 256 + threadIdx.x, int64_t(s.splits) * 256); w.left > 0; w.next()) {
    const CT g = CT(Cvt<T>::load(dy + w.off));
    sdy += g;
    sdyx += g * ((CT(Cvt<T>::load(x + w.off)) - mean) * invstd);
  }
  sdy = block_sum<CT>(sdy, lds);
  sdyx = block_sum<CT>(sdyx, lds);
  if (threadIdx.x == 0) {
    CT* o = part + (c * s.splits + split) * 2;
    o[0] = sdy; o[1] = sdyx;
  }
}

// dscale = sum dy * xhat, dbias = sum dy; coefficients of dx = k0 * dy + k1 * (x - mean) + k2 with
//   dx = scale * invstd * (dy - dbias / m - xhat * dscale / m),  xhat = (x - mean) * invstd
template <typename PT, typename CT>
__global__ __launch_bounds__(256)
void bn_bwd_finalize_kernel(const CT* __restrict__ part, int64_t C, int splits, CT count,
                            const PT* __restrict__ scale, const PT* __restrict__ save_mean,
                            const PT* __restrict__ save_invstd, PT* dscale, PT* dbias, CT* __restrict__ coef) {
  const int64_t c = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (c >= C) return;
  CT sdy = 0, sdyx = 0;
  for (int k = 0; k < splits; ++k) {
    sdy += part[(c * splits + k) * 2];
    sdyx += part[(c * splits + k) * 2 + 1];
  }
  if (dscale) dscale[c] = PT(sdyx);
  if (dbias) dbias[c] = PT(sdy);
  const CT mean = CT(save_mean[c]), invstd = CT(save_invstd[c]);
  const CT a = CT(scale[c]) * invstd;
  coef[c] = a;
  coef[C + c] = -a * invstd * sdyx / count;
  coef[2 * C + c] = -a * sdy / count;
  coef[3 * C + c] = mean;
}

template <typename T, typename CT, typename IT>
__global__ __launch_bounds__(256)
void bn_bwd_apply_kernel(const T* dy, const T* x, T* dx, const CT* __restrict__ coef, IT total, IT hw, IT C) {
  const IT v = IT(blockIdx.x) * kStreamThreads + threadIdx.x;
  if (v >= total) return;
  const CT g = CT(Cvt<T>::load(dy + size_t(v))), f = CT(Cvt<T>::load(x + size_t(v)));
  bool uniform;
  const IT c = bn_channel<IT>(v, hw, C, uniform);
  CT k0, k1, k2, mean;
  if (uniform) {
    const IT c0 = IT(__builtin_amdgcn_readfirstlane(uint32_t(c)));
    k0 = coef[c0]; k1 = coef[size_t(C) + c0]; k2 = coef[2 * size_t(C) + c0]; mean = coef[3 * size_t(C) + c0];
  } else {
    k0 = coef[c]; k1 = coef[size_t(C) + c]; k2 = coef[2 * size_t(C) + c]; mean = coef[3 * size_t(C) + c];
  }
  Cvt<T>::store(dx + size_t(v), k0 * g + (k1 * (f - mean) + k2));
}

// ---------------------------------------------------------------------------
// planes as 16-byte vectors
// ---------------------------------------------------------------------------
// IT: what counts a channel's vectors and a plane's elements, 32 bits unless the array is past 2^31 elements
template <typename IT>
struct BnRuns {
  int C;
  IT HW;
  IT run_vecs;         // vectors per run, the partial one included
  IT total;            // vectors per channel
  int64_t image;       // C * HW
};
// (One for each direction, the launch's threads in it, see kCheapArgs: 4 x 130 x 484 bf16, both ways, 9.4 -> 9.1 us.)
struct BnFwdParams {
  const float *scale, *bias;
  float *running_mean, *running_var, *save_mean, *save_invstd;   // outputs (each may be null)
  double momentum, eps;
  float count;
  int threads;         // bn_fwd_channel_kernel: of a workgroup
};
struct BnBwdParams {
  const float *scale, *mean, *invstd;
  float *dscale, *dbias;
  float count;
  int threads;         // bn_bwd_channel_kernel: of a workgroup
};
static_assert(2 * 8 + sizeof(BnRuns<int>) + sizeof(BnFwdParams) <= kCheapArgs && 3 * 8 + sizeof(BnRuns<int>) + sizeof(BnBwdParams) <= kCheapArgs, "");

// A thread's walk over the vectors v0, v0 + stride, ... of a channel
template <typename T, typename IT>
struct BnVecWalk {
  static constexpr int VEC = VecIO<T>::N;
  using UT = typename std::make_unsigned<IT>::type;
  const BnRuns<IT>& r;
  IT index, v;           // vector in the channel, and in its run
  int64_t plane;         // offset of the run from the channel's first
  IT stride, step_v;
  int64_t step_plane;
  __device__ __forceinline__ BnVecWalk(const BnRuns<IT>& runs, IT v0, int by) : r(runs), index(v0), stride(by) {
    const UT n = UT(v0) / UT(r.run_vecs), q = UT(by) / UT(r.run_vecs);
    v = v0 - IT(n) * r.run_vecs;
    plane = int64_t(n) * r.image;
    step_v = by - IT(q) * r.run_vecs;
    step_plane = int64_t(q) * r.image;
  }
  __device__ __forceinline__ bool live() const { return index < r.total; }
  // offset of the loaded vector (the channel's first one past the end), and how many of its elements belong to others
  __device__ __forceinline__ int64_t off() const { return live() ? plane + vec_column<T, true>(v, r.HW) : 0; }
  __device__ __forceinline__ int skip() const {
    const IT left = r.HW - v * VEC;
    return !live() ? VEC : left >= VEC ? 0 : VEC - int(left);
  }
  __device__ __forceinline__ void next() {
    index += stride;
    v += step_v;
    plane += step_plane;
    const bool wrap = v >= r.run_vecs;
    v -= wrap ? r.run_vecs : 0;
    plane += wrap ? r.image : 0;
  }
};
// One workgroup per channel, NV vectors per thread in registers.  The mean first, as sums about the channel's first
// element K (a large common offset never enters a sum), then the squares about it.  What the rounding of the mean
// left out is kept as a second term, so that elements near the mean keep their digits.  (Parameters and running statistics fetched
// beside the elements: 64 x 256 x 196 bf16, forward and backward, 11.2 / 11.3 us.)
// Three launches and two reads of the input before (bf16, forward / backward): 64 x 256 x 196 24.4 / 23.6 us -> 11.2 /
// 10.3, of which 10 are the call's own; 2 x 512 x 3969 27.9 / 27.0 -> 10.5 / 10.1.  Short odd planes are bound by cache
// lines that neighbouring channels share: 16 of them stay on one XCD (channels handed out in turn / in runs of 4 / 16 / 32, GPU
// us: 256 x 1024 x 49 34.4, 43.7 / 29.8, 38.1 / 27.5, 35.7 / 27.0, 35.1, 1.8 TB/s; 64 x 1000 x 49 fp32 9.6, 12.0 / 8.1, 10.4 /
// 7.9, 10.3 / 8.0, 10.2; 64 x 256 x 196 6.7, 6.3 / 6.5, 6.3 / 6.2, 6.0 / 6.2, 6.0; planes of whole lines do not care).
template <typename T, int NV, typename IT>
__global__ __launch_bounds__(1024)
void bn_fwd_channel_kernel(const T* x, T* y, BnRuns<IT> r, BnFwdParams p) {
  constexpr int VEC = VecIO<T>::N;
  __shared__ float red[2][kMaxWaves * 2];
  const int c = int(xcd_run_block<16>(blockIdx.x, uint32_t(r.C))), nwaves = p.threads >> 6;
  const int64_t base = int64_t(c) * r.HW;
  u32x4 raw[NV];
  IT off[NV];
  int skip[NV];
  BnVecWalk<T, IT> w(r, IT(threadIdx.x), p.threads);
#pragma unroll
  for (int i = 0; i < NV; ++i, w.next()) {
    off[i] = IT(w.off());
    skip[i] = w.skip();
    raw[i] = ld16_any<T>(x + base + off[i]);
  }
  const float K = Cvt<T>::load(x + base);
  SumTuple<1> s = SumTuple<1>::identity();
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    float f[VEC];
    VecIO<T>::unpack(raw[i], f);
#pragma unroll
    for (int j = 0; j < VEC; ++j) s.v[0] += j < skip[i] ? 0.f : f[j] - K;
  }
  const float near = K + group_allreduce_tuple(s, red[0], 0, nwaves).v[0] / p.count;
  SumTuple<2> q = SumTuple<2>::identity();
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    float f[VEC];
    VecIO<T>::unpack(raw[i], f);
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const float d = j < skip[i] ? 0.f : f[j] - near;
      q.v[0] += d;
      q.v[1] = fmaf(d, d, q.v[1]);
    }
  }
  q = group_allreduce_tuple(q, red[1], 0, nwaves);
  const float rest = q.v[0] / p.count;   // mean = near + rest
  const float about = q.v[1] - q.v[0] * rest, m2 = about < 0.f ? 0.f : about;   // (a NaN stays one)
  const float invstd = bn_invstd<float, float>(m2 / p.count, p.eps);
  const float a = p.scale[c] * invstd, b = p.bias[c];
  if (threadIdx.x == 0)
    bn_store_stats<float, float>(c, p.count, near + rest, m2, invstd, p.momentum,
                                 BnRunning<float>(p.running_mean, p.running_var, c), p.running_mean, p.running_var, p.save_mean,
                                 p.save_invstd);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (skip[i] < VEC) {
      float f[VEC];
      VecIO<T>::unpack(raw[i], f);
#pragma unroll
      for (int j = 0; j < VEC; ++j) f[j] = ((f[j] - near) - rest) * a + b;
      st16_any(y + base + off[i], VecIO<T>::pack(f));   // shared elements: the same bits twice
    }
  }
}

// dx = scale * invstd * (dy - sum dy / m - xhat * sum(dy xhat) / m),  xhat = (x - mean) * invstd
struct BnBwdCoef {
  float k0, k1, k2, mean;
  __device__ __forceinline__ BnBwdCoef(const BnBwdParams& p, float scale, float sdy, float sdyx, float mean_, float invstd) : mean(mean_) {
    const float a = scale * invstd;
    k0 = a;
    k1 = -a * invstd * sdyx / p.count;
    k2 = -a * sdy / p.count;
  }
  __device__ __forceinline__ float operator()(float g, float x) const { return k0 * g + (k1 * (x - mean) + k2); }
};

template <typename T, int NV, typename IT>
__global__ __launch_bounds__(1024)
void bn_bwd_channel_kernel(const T* dy, const T* x, T* dx, BnRuns<IT> r, BnBwdParams p) {
  constexpr int VEC = VecIO<T>::N;
  __shared__ float red[kMaxWaves * 2];
  const int c = int(xcd_run_block<16>(blockIdx.x, uint32_t(r.C))), nwaves = p.threads >> 6;
  const int64_t base = int64_t(c) * r.HW;
  u32x4 rg[NV], rx[NV];
  IT off[NV];
  int skip[NV];
  BnVecWalk<T, IT> w(r, IT(threadIdx.x), p.threads);
#pragma unroll
  for (int i = 0; i < NV; ++i, w.next()) {
    off[i] = IT(w.off());
    skip[i] = w.skip();
    rg[i] = ld16_any<T>(dy + base + off[i]);
    rx[i] = ld16_any<T>(x + base + off[i]);
  }
  const float mean = p.mean[c], invstd = p.invstd[c];
  SumTuple<2> s = SumTuple<2>::identity();
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    float g[VEC], f[VEC];
    VecIO<T>::unpack(rg[i], g);
    VecIO<T>::unpack(rx[i], f);
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const float gj = j < skip[i] ? 0.f : g[j], xj = j < skip[i] ? mean : f[j];
      s.v[0] += gj;
      s.v[1] = fmaf(gj, (xj - mean) * invstd, s.v[1]);
    }
  }
  s = group_allreduce_tuple(s, red, 0, nwaves);
  if (threadIdx.x == 0) {
    if (p.dscale) p.dscale[c] = s.v[1];
    if (p.dbias) p.dbias[c] = s.v[0];
  }
  const BnBwdCoef k(p, p.scale[c], s.v[0], s.v[1], mean, invstd);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (skip[i] < VEC) {
      float g[VEC], f[VEC];
      VecIO<T>::unpack(rg[i], g);
      VecIO<T>::unpack(rx[i], f);
#pragma unroll
      for (int j = 0; j < VEC; ++j) g[j] = k(g[j], f[j]);
      st16_any(dx + base + off[i], VecIO<T>::pack(g));
    }
  }
}

// Longer channels: kBnVecs vectors per thread in flight.  Bound by three (forward) and five (backward) streams at 6.3 to
// 6.5 TB/s: 64 x 256 x 3136 bf16 55.7 / 83.2 -> 49.2 / 79.4 us, odd planes (32 x 100 x 3025 fp16, element by element
// before) 63.9 / 57.2 -> 18.1 / 24.0 us.
constexpr int kBnVecs = 4;

// (count, mean, M2) of the slice blockIdx.y of channel blockIdx.x -> part[(c * splits + split) * 3 ..]
template <typename T, typename IT>
__global__ __launch_bounds__(256)
void bn_fwd_partial_kernel(const T* __restrict__ x, BnRuns<IT> r, int splits, float* __restrict__ part) {
  constexpr int VEC = VecIO<T>::N, U = kBnVecs;
  __shared__ float red[2][kMaxWaves * 2];
  const int64_t c = blockIdx.x;
  const T* base = x + c * r.HW;
  BnVecWalk<T, IT> w(r, IT(blockIdx.y) * 256 + IT(threadIdx.x), splits * 256);
  // sums about a pivot K, the mean of the thread's first vector: a large common offset never enters a sum
  float K = 0.f, s1 = 0.f, s2 = 0.f, cnt = 0.f;
  while (w.live()) {
    u32x4 raw[U];
    int skip[U];
#pragma unroll
    for (int i = 0; i < U; ++i, w.next()) {
      skip[i] = w.skip();
      raw[i] = ld16_any_keep<T>(base + w.off());
    }
#pragma unroll
    for (int i = 0; i < U; ++i) {
      float f[VEC];
      VecIO<T>::unpack(raw[i], f);
      if (i == 0 && cnt == 0.f) {
        float k = 0.f;
#pragma unroll
        for (int j = 0; j < VEC; ++j) k += j < skip[0] ? 0.f : f[j];
        K = k / float(VEC - max(skip[0], 0));
      }
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        const float d = j < skip[i] ? 0.f : f[j] - K;
        s1 += d;
        s2 = fmaf(d, d, s2);
      }
      cnt += float(VEC - max(skip[i], 0));
    }
  }
  const float mean = cnt > 0.f ? K + s1 / cnt : 0.f;
  const float about = cnt > 0.f ? s2 - s1 * (s1 / cnt) : 0.f, m2 = about < 0.f ? 0.f : about;   // (a NaN stays one)
  // total count and mean first, then M2 about that mean
  const SumTuple<2> t = group_allreduce_tuple(SumTuple<2>{{cnt, mean * cnt}}, red[0], 0, 4);
  const float bmean = t.v[0] > 0.f ? t.v[1] / t.v[0] : 0.f, d = mean - bmean;
  const SumTuple<1> q = group_allreduce_tuple(SumTuple<1>{{fmaf(d * d, cnt, m2)}}, red[1], 0, 4);
  if (threadIdx.x == 0) {
    float* o = part + (c * splits + blockIdx.y) * 3;
    o[0] = t.v[0]; o[1] = bmean; o[2] = q.v[0];
  }
}

// Workgroup (chunk, channel) = divmod(blockIdx.x, C): kBnVecs vectors per thread, loaded before the channel's partials
// are merged; every wavefront merges them for itself.  The first chunk's workgroup writes the statistics.
template <typename T, typename IT>
__global__ __launch_bounds__(256)
void bn_fwd_merge_apply_kernel(const T* x, T* y, BnRuns<IT> r, BnFwdParams p, int splits, const float* __restrict__ part) {
  constexpr int VEC = VecIO<T>::N, U = kBnVecs;
  const int chunk = int(blockIdx.x / uint32_t(r.C)), c = int(blockIdx.x - uint32_t(chunk) * uint32_t(r.C));
  const int64_t base = int64_t(c) * r.HW;
  u32x4 raw[U];
  IT v[U];
  int64_t plane[U];
  BnVecWalk<T, IT> w(r, IT(chunk) * (256 * U) + IT(threadIdx.x), 256);
#pragma unroll
  for (int i = 0; i < U; ++i, w.next()) {
    raw[i] = ld16_any<T>(x + base + w.off());
    v[i] = w.live() ? w.v : r.run_vecs;      // a vector past the run's end stores nothing
    plane[i] = w.plane;
  }
  const float scale = p.scale[c], b = p.bias[c];
  const BnRunning<float> was(p.running_mean, p.running_var, c);   // (with the parameters, before the partials are merged)
  const float* mine = part + int64_t(c) * splits * 3;
  const float near = mine[1];              // about the first slice's mean: mean = near + rest, as in bn_fwd_channel_kernel
  float d1 = 0.f;
  for (int k = int(threadIdx.x & 63); k < splits; k += kWave) d1 = fmaf(mine[k * 3], mine[k * 3 + 1] - near, d1);
  const float rest = wave_allreduce_tuple(SumTuple<1>{{d1}}).v[0] / p.count;
  SumTuple<1> q = SumTuple<1>::identity();
  for (int k = int(threadIdx.x & 63); k < splits; k += kWave) {
    const float d = (mine[k * 3 + 1] - near) - rest;
    q.v[0] += fmaf(d * d, mine[k * 3], mine[k * 3 + 2]);
  }
  const float m2 = wave_allreduce_tuple(q).v[0];
  const float invstd = bn_invstd<float, float>(m2 / p.count, p.eps);
  const float a = scale * invstd;
#pragma unroll
  for (int i = 0; i < U; ++i) {
    float f[VEC];
    VecIO<T>::unpack(raw[i], f);
#pragma unroll
    for (int j = 0; j < VEC; ++j) f[j] = ((f[j] - near) - rest) * a + b;
    // in place, a shared element may have been replaced before it was read here: only own ones go out
    if (v[i] < r.run_vecs) store_row_vec<T, true, false>(y + base + plane[i], v[i], f, r.HW);
  }
  if (chunk == 0 && threadIdx.x == 0)
    bn_store_stats<float, float>(c, p.count, near + rest, m2, invstd, p.momentum, was, p.running_mean, p.running_var,
                                 p.save_mean, p.save_invstd);
}

// sums of dy and dy * xhat of a slice -> part[(c * splits + split) * 2 ..]
template <typename T, typename IT>
__global__ __launch_bounds__(256)
void bn_bwd_partial_kernel(const T* __restrict__ dy, const T* __restrict__ x, BnRuns<IT> r, BnBwdParams p, int splits,
                           float* __restrict__ part) {
  constexpr int VEC = VecIO<T>::N, U = kBnVecs / 2;
  __shared__ float red[kMaxWaves * 2];
  const int64_t c = blockIdx.x;
  const int64_t base = c * r.HW;
  const float mean = p.mean[c], invstd = p.invstd[c];
  SumTuple<2> s = SumTuple<2>::identity();
  BnVecWalk<T, IT> w(r, IT(blockIdx.y) * 256 + IT(threadIdx.x), splits * 256);
  while (w.live()) {
    u32x4 rg[U], rx[U];
    int skip[U];
#pragma unroll
    for (int i = 0; i < U; ++i, w.next()) {
      const int64_t off = base + w.off();
      skip[i] = w.skip();
      rg[i] = ld16_any_keep<T>(dy + off);
      rx[i] = ld16_any_keep<T>(x + off);
    }
#pragma unroll
    for (int i = 0; i < U; ++i) {
      float g[VEC], f[VEC];
      VecIO<T>::unpack(rg[i], g);
      VecIO<T>::unpack(rx[i], f);
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        const float gj = j < skip[i] ? 0.f : g[j], xj = j < skip[i] ? mean : f[j];
        s.v[0] += gj;
        s.v[1] = fmaf(gj, (xj - mean) * invstd, s.v[1]);
      }
    }
  }
  s = group_allreduce_tuple(s, red, 0, 4);
  if (threadIdx.x == 0) {
    float* o = part + (c * splits + blockIdx.y) * 2;
    o[0] = s.v[0]; o[1] = s.v[1];
  }
}

template <typename T, typename IT>
__global__ __launch_bounds__(256)
void bn_bwd_merge_apply_kernel(const T* dy, const T* x, T* dx, BnRuns<IT> r, BnBwdParams p, int splits,
                               const float* __restrict__ part) {
  constexpr int VEC = VecIO<T>::N, U = kBnVecs / 2;
  const int chunk = int(blockIdx.x / uint32_t(r.C)), c = int(blockIdx.x - uint32_t(chunk) * uint32_t(r.C));
  const int64_t base = int64_t(c) * r.HW;
  u32x4 rg[U], rx[U];
  IT v[U];
  int64_t plane[U];
  BnVecWalk<T, IT> w(r, IT(chunk) * (256 * U) + IT(threadIdx.x), 256);
#pragma unroll
  for (int i = 0; i < U; ++i, w.next()) {
    const int64_t off = base + w.off();
    rg[i] = ld16_any<T>(dy + off);
    rx[i] = ld16_any<T>(x + off);
    v[i] = w.live() ? w.v : r.run_vecs;
    plane[i] = w.plane;
  }
  const float mean = p.mean[c], invstd = p.invstd[c], scale = p.scale[c];
  const float* mine = part + int64_t(c) * splits * 2;
  SumTuple<2> s = SumTuple<2>::identity();
  for (int k = int(threadIdx.x & 63); k < splits; k += kWave) { s.v[0] += mine[k * 2]; s.v[1] += mine[k * 2 + 1]; }
  s = wave_allreduce_tuple(s);
  if (chunk == 0 && threadIdx.x == 0) {
    if (p.dscale) p.dscale[c] = s.v[1];
    if (p.dbias) p.dbias[c] = s.v[0];
  }
  const BnBwdCoef k(p, scale, s.v[0], s.v[1], mean, invstd);
#pragma unroll
  for (int i = 0; i < U; ++i) {
    float g[VEC], f[VEC];
    VecIO<T>::unpack(rg[i], g);
    VecIO<T>::unpack(rx[i], f);
#pragma unroll
    for (int j = 0; j < VEC; ++j) g[j] = k(g[j], f[j]);
    if (v[i] < r.run_vecs) store_row_vec<T, true, false>(dx + base + plane[i], v[i], g, r.HW);
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static int bn_splits(int64_t C, int64_t per_channel) {
  // enough workgroups to fill the chip (about 8 per compute unit), each with at least 8 loads per thread
  if (C <= 0) return 1;   // an empty array: callers return before launching anything
  const int64_t want = (int64_t(device_cu_count()) * 8 + C - 1) / C;
  const int64_t most = std::max<int64_t>(1, per_channel / (256 * 8));
  return int(std::max<int64_t>(1, std::min<int64_t>(std::min(want, most), 1024)));
}

static BnShape bn_shape(int64_t N, int64_t C, int64_t HW) {
  BnShape s{};
  s.N = N; s.C = C; s.HW = HW;
  s.per_channel = N * HW;
  s.splits = bn_splits(C, s.per_channel);
  return s;
}

static size_t bn_ws_bytes(int64_t N, int64_t C, int64_t HW, size_t ct_size) {
  // partials for the element-wise decomposition (the largest one) + four coefficient rows
  const BnShape s = bn_shape(N, C, HW);
  return (size_t(C) * size_t(s.splits) * 3 + size_t(C) * 4) * ct_size;
}

// How the vector kernels take an [N, C, HW] array; form 0: they don't
template <typename IT>
struct BnPlan {
  int form;            // 1: a workgroup per channel; 2: partials and merge
  BnRuns<IT> runs;
  int threads, nv;     // form 1
  int splits;          // form 2
};
template <typename T, typename IT>
static BnPlan<IT> bn_plan(int64_t N, int64_t C, int64_t HW, int max_splits, int max_nv) {
  constexpr int VEC = VecIO<T>::N;
  BnPlan<IT> b{};
  const int64_t run_vecs = (HW + VEC - 1) / VEC, total = N * run_vecs;
  // the walk's count of vectors and its steps stay below IT's most, the workgroups of either form below the grid's
  if (HW < VEC || (sizeof(IT) == 4 && (N * C * HW > 0x7fffffffLL || total > 0x3fffffff))) return b;
  if (C > 0x7fffffffLL || (total / (128 * kBnVecs) + 1) * C > 0x7fffffffLL) return b;
  b.runs.C = int(C); b.runs.HW = IT(HW); b.runs.image = C * HW;
  b.runs.run_vecs = IT(run_vecs);
  b.runs.total = IT(total);
  // workgroups of nv vectors a thread that a compute unit runs at once: 32 wavefronts, fewer past 64 registers a thread
  const auto at_once = [&](int nv) {
    const int waves = nv == 8 ? (VEC == 8 ? 16 : 24) : max_nv == 4 && nv == 4 && VEC == 8 ? 20 : 32;
    return waves / int(((total + nv - 1) / nv + 63) / 64);
  };
  const int64_t cus = device_cu_count();
  for (int nv = 1; nv <= max_nv; nv <<= 1) {
    // one vector a thread while there are fewer channels than two workgroups per compute unit, else two at least
    if (total > int64_t(nv) * 1024 || (nv == 1 && total > 64 && C > 2 * device_cu_count())) continue;
    // and twice the fewest where not all channels run at once so and more of them do then, backward as many (forward and backward, us,
    // fewest / twice: 64 x 600 x 196 bf16 25.4 / 22.2, 10 x 900 x 1024 24.7 / 20.4, 30 x 999 x 441 39.8 / 33.8, backward as it was 35.4, 40 x
    // 1000 x 144 fp32 27.3 / 22.6; where all run at once or no more do, 2 x 600 x 3000 fp16 12.2 / 12.65, 100 x 1024 x 49 20.1 / 20.6, 38 x
    // 587 x 576, forward, of 33.7 both ways, 2.5 more)
    const bool more = max_nv == 4 ? at_once(2 * nv) >= at_once(nv) : at_once(2 * nv) > at_once(nv);
    // the 16-bit backward of two vectors: not in every width.  Fewest / twice, by wavefronts of the fewest, 800 channels of planes off
    // the vectors' boundaries and on them: 9 20 x 413 13.0 / 13.8 and 4 x 2064 10.1 / 10.5, 10 20 x 477 14.7 / 14.5 and 4 x 2400 11.5 / 11.05, 11
    // 20 x 533 15.8 / 17.3 and 4 x 2680 12.4 / 13.3, 12 20 x 573 17.0 / 18.0 and 4 x 2896 13.3 / 14.2, 15 20 x 717 20.4 / 21.3 and 4 x 3600 15.9 /
    // 16.1, 16 20 x 757 21.35 / 22.4; 13 20 x 621 18.15 / 18.95, of 1000 channels 22.7 / 21.0; 64 x 196 of 768, 860 and 1024 14.2 / 14.75, 19.5 / 17.8
    // and 20.3 / 19.5, 14 30 x 441 17.4 / 17.5, 21.0 / 20.5 and 25.0 / 22.7
    const int waves = int(((total + nv - 1) / nv + 63) / 64);
    const bool pays = max_nv != 4 || VEC != 8 || nv != 2 || waves <= 8 || waves == 10 ||
                      ((waves == 13 || waves == 14) && 4 * C > 13 * cus);
    if (2 * nv <= max_nv && C > cus * at_once(nv) && more && pays) nv *= 2;
    b.form = 1;
    b.nv = nv;
    b.threads = int(((total + nv - 1) / nv + 63) / 64 * 64);
    return b;
  }
  b.form = 2;
  const int64_t want = (int64_t(device_cu_count()) * 8 + C - 1) / C, round = 256 * kBnVecs;
  const int64_t most = std::max<int64_t>(1, std::min<int64_t>(std::min(want, (total + round - 1) / round), std::min(max_splits, 256)));
  // as few slices as take one or two rounds of loads: a last one that is nearly empty costs a trip to memory like any other (us: 31 x 404
  // x 2304 fp16 32.8 / 48.4 -> 30.1 / 45.9, 107 x 26 x 2601 bf16 forward 15.0 -> 14.0, 200 x 100 x 1000 both ways 65.0 -> 60.8).  Where they
  // take more, the compute units' room counts (140 x 65 x 4761 bf16, 32 slices / 28 119.4 / 124.0, 128 x 27 x 6084 fp32 112.4 / 111.2).
  const int64_t rounds = (total + round * most - 1) / (round * most);
  b.splits = int(rounds > 2 ? most : (total + round * rounds - 1) / (round * rounds));
  return b;
}
template <typename IT>
static inline unsigned bn_chunks(const BnRuns<IT>& r, int per_thread) {
  return unsigned((int64_t(r.total) + 256 * per_thread - 1) / (256 * per_thread)) * unsigned(r.C);
}

// the vector kernels' launches; *handled: they take the array
template <typename T, typename IT>
static int bn_fwd_vec(const T* x, T* y, BnFwdParams p, int64_t N, int64_t C, int64_t HW, int max_splits, float* part,
                      hipStream_t st, bool* handled) {
  const BnPlan<IT> b = bn_plan<T, IT>(N, C, HW, max_splits, 8);
  *handled = b.form != 0;
  if (b.form == 1) {
    const dim3 grid{unsigned(C)}, block{unsigned(b.threads)};
    p.threads = b.threads;
    profile_before(st);
    switch (b.nv) {
      case 1: HK_LAUNCH((bn_fwd_channel_kernel<T, 1, IT>), grid, block, 0, st, x, y, b.runs, p); break;
      case 2: HK_LAUNCH((bn_fwd_channel_kernel<T, 2, IT>), grid, block, 0, st, x, y, b.runs, p); break;
      case 4: HK_LAUNCH((bn_fwd_channel_kernel<T, 4, IT>), grid, block, 0, st, x, y, b.runs, p); break;
      default: HK_LAUNCH((bn_fwd_channel_kernel<T, 8, IT>), grid, block, 0, st, x, y, b.runs, p);
    }
    profile_after(st);
    return launch_check("bn_fwd_channel_kernel");
  }
  if (b.form == 2) {
    HK_LAUNCH((bn_fwd_partial_kernel<T, IT>), dim3(unsigned(C), unsigned(b.splits)), dim3(256), 0, st, x, b.runs, b.splits, part);
    const int rc = launch_check("bn_fwd_partial_kernel");
    if (rc != HK_OK) return rc;
    profile_before(st);
    HK_LAUNCH((bn_fwd_merge_apply_kernel<T, IT>), dim3(bn_chunks(b.runs, kBnVecs)), dim3(256), 0, st, x, y, b.runs, p, b.splits, part);
    profile_after(st);
    return launch_check("bn_fwd_merge_apply_kernel");
  }
  return HK_OK;
}

template <typename T, typename IT>
static int bn_bwd_vec(const T* dy, const T* x, T* dx, BnBwdParams p, int64_t N, int64_t C, int64_t HW, int max_splits,
                      float* part, hipStream_t st, bool* handled) {
  const BnPlan<IT> b = bn_plan<T, IT>(N, C, HW, max_splits, 4);
  *handled = b.form != 0;
  if (b.form == 1) {
    const dim3 grid{unsigned(C)}, block{unsigned(b.threads)};
    p.threads = b.threads;
    profile_before(st);
    switch (b.nv) {
      case 1: HK_LAUNCH((bn_bwd_channel_kernel<T, 1, IT>), grid, block, 0, st, dy, x, dx, b.runs, p); break;
      case 2: HK_LAUNCH((bn_bwd_channel_kernel<T, 2, IT>), grid, block, 0, st, dy, x, dx, b.runs, p); break;
      default: HK_LAUNCH((bn_bwd_channel_kernel<T, 4, IT>), grid, block, 0, st, dy, x, dx, b.runs, p);
    }
    profile_after(st);
    return launch_check("bn_bwd_channel_kernel");
  }
  if (b.form == 2) {
    HK_LAUNCH((bn_bwd_partial_kernel<T, IT>), dim3(unsigned(C), unsigned(b.splits)), dim3(256), 0, st, dy, x, b.runs, p, b.splits, part);
    const int rc = launch_check("bn_bwd_partial_kernel");
    if (rc != HK_OK) return rc;
    profile_before(st);
    HK_LAUNCH((bn_bwd_merge_apply_kernel<T, IT>), dim3(bn_chunks(b.runs, kBnVecs / 2)), dim3(256), 0, st, dy, x, dx, b.runs, p, b.splits, part);
    profile_after(st);
    return launch_check("bn_bwd_merge_apply_kernel");
  }
  return HK_OK;
}

template <typename T, typename PT>
static int bn_fwd_typed(const void* x, const void* scale, const void* bias, void* y, double momentum, double eps,
                        void* running_mean, void* running_var, void* save_mean, void* save_invstd, int64_t N,
                        int64_t C, int64_t HW, void* ws, hipStream_t st) {
  using CT = typename BnCT<T>::type;
  CT* part = static_cast<CT*>(ws);
  const T* xp = static_cast<const T*>(x);
  T* yp = static_cast<T*>(y);
  const BnShape s = bn_shape(N, C, HW);
  if constexpr (!std::is_same<T, double>::value) {
    BnFwdParams p{};
    p.scale = static_cast<const float*>(scale); p.bias = static_cast<const float*>(bias);
    p.running_mean = static_cast<float*>(running_mean); p.running_var = static_cast<float*>(running_var);
    p.save_mean = static_cast<float*>(save_mean); p.save_invstd = static_cast<float*>(save_invstd);
    p.momentum = momentum; p.eps = eps; p.count = float(N * HW);
    bool handled = false;
    int rc = bn_fwd_vec<T, int>(xp, yp, p, N, C, HW, s.splits, part, st, &handled);
    if (!handled) rc = bn_fwd_vec<T, int64_t>(xp, yp, p, N, C, HW, s.splits, part, st, &handled);
    if (handled) return rc;
  }
  CT* coef = part + size_t(C) * size_t(s.splits) * 3;
  const int64_t total = N * C * HW;
  HK_REQUIRE(C <= 0x7fffffffLL && (total + kStreamThreads - 1) / kStreamThreads <= 0x7fffffffLL, HK_ERR_INVALID,
             "hk_batch_norm_fwd: array too large");
  HK_LAUNCH((bn_stats_kernel<T, CT>), dim3(unsigned(C), unsigned(s.splits)), dim3(256), 0, st, xp, s, part);
  int rc = launch_check("bn_stats_kernel");
  if (rc != HK_OK) return rc;
  HK_LAUNCH((bn_finalize_kernel<PT, CT>), dim3(unsigned((C + 255) / 256)), dim3(256), 0, st, part, C, s.splits,
            static_cast<const PT*>(scale), static_cast<const PT*>(bias), momentum, eps, static_cast<PT*>(running_mean),
            static_cast<PT*>(running_var), static_cast<PT*>(save_mean), static_cast<PT*>(save_invstd), coef);
  rc = launch_check("bn_finalize_kernel");
  if (rc != HK_OK) return rc;
  const dim3 grid{unsigned((total + kStreamThreads - 1) / kStreamThreads)}, block{kStreamThreads};
  profile_before(st);
  if (total < 0x7fffffffLL)
    HK_LAUNCH((bn_apply_kernel<T, CT, uint32_t>), grid, block, 0, st, xp, yp, coef, uint32_t(total), uint32_t(HW), uint32_t(C));
  else
    HK_LAUNCH((bn_apply_kernel<T, CT, int64_t>), grid, block, 0, st, xp, yp, coef, total, HW, C);
  profile_after(st);
  return launch_check("bn_apply_kernel");
}

template <typename T, typename PT>
static int bn_bwd_typed(const void* dy, const void* x, const void* scale, void* dx, void* dscale, void* dbias,
                        const void* save_mean, const void* save_invstd, int64_t N, int64_t C, int64_t HW, void* ws,
                        hipStream_t st) {
  using CT = typename BnCT<T>::type;
  CT* part = static_cast<CT*>(ws);
  const T *gp = static_cast<const T*>(dy), *xp = static_cast<const T*>(x);
  T* op = static_cast<T*>(dx);
  const BnShape s = bn_shape(N, C, HW);
  if constexpr (!std::is_same<T, double>::value) {
    BnBwdParams p{};
    p.scale = static_cast<const float*>(scale);
    p.mean = static_cast<const float*>(save_mean); p.invstd = static_cast<const float*>(save_invstd);
    p.dscale = static_cast<float*>(dscale); p.dbias = static_cast<float*>(dbias);
    p.count = float(N * HW);
    bool handled = false;
    int rc = bn_bwd_vec<T, int>(gp, xp, op, p, N, C, HW, s.splits, part, st, &handled);
    if (!handled) rc = bn_bwd_vec<T, int64_t>(gp, xp, op, p, N, C, HW, s.splits, part, st, &handled);
    if (handled) return rc;
  }
  CT* coef = part + size_t(C) * size_t(s.splits) * 3;
  const int64_t total = N * C * HW;
  HK_REQUIRE(C <= 0x7fffffffLL && (total + kStreamThreads - 1) / kStreamThreads <= 0x7fffffffLL, HK_ERR_INVALID,
             "hk_batch_norm_bwd: array too large");
  HK_LAUNCH((bn_bwd_stats_kernel<T, PT, CT>), dim3(unsigned(C), unsigned(s.splits)), dim3(256), 0, st, gp, xp, s,
            static_cast<const PT*>(save_mean), static_cast<const PT*>(save_invstd), part);
  int rc = launch_check("bn_bwd_stats_kernel");
  if (rc != HK_OK) return rc;
  HK_LAUNCH((bn_bwd_finalize_kernel<PT, CT>), dim3(unsigned((C + 255) / 256)), dim3(256), 0, st, part, C, s.splits,
            CT(N * HW), static_cast<const PT*>(scale), static_cast<const PT*>(save_mean),
            static_cast<const PT*>(save_invstd), static_cast<PT*>(dscale), static_cast<PT*>(dbias), coef);
  rc = launch_check("bn_bwd_finalize_kernel");
  if (rc != HK_OK) return rc;
  const dim3 grid{unsigned((total + kStreamThreads - 1) / kStreamThreads)}, block{kStreamThreads};
  profile_before(st);
  if (total < 0x7fffffffLL)
    HK_LAUNCH((bn_bwd_apply_kernel<T, CT, uint32_t>), grid, block, 0, st, gp, xp, op, coef, uint32_t(total), uint32_t(HW), uint32_t(C));
  else
    HK_LAUNCH((bn_bwd_apply_kernel<T, CT, int64_t>), grid, block, 0, st, gp, xp, op, coef, total, HW, C);
  profile_after(st);
  return launch_check("bn_bwd_apply_kernel");
}

static int bn_check(const char* who, int dtype, int64_t N, int64_t C, int64_t HW, const void* ws, size_t ws_bytes,
                    size_t* need) {
  HK_REQUIRE(N >= 0 && C >= 0 && HW >= 0, HK_ERR_INVALID, "%s: negative shape", who);
  HK_REQUIRE(dtype == HK_FLOAT32 || dtype == HK_BFLOAT16 || dtype == HK_FLOAT16 || dtype == HK_FLOAT64,
             HK_ERR_UNSUPPORTED, "%s: not implemented for dtype %d", who, dtype);
  *need = 0;
  if (N * C * HW == 0) return HK_OK;   // before the split plan, which divides by C
  *need = bn_ws_bytes(N, C, HW, dtype == HK_FLOAT64 ? 8 : 4);
  HK_REQUIRE(ws != nullptr && ws_bytes >= *need, HK_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given",
             who, *need, ws_bytes);
  HK_REQUIRE(aligned16(ws), HK_ERR_INVALID, "%s: workspace must be 16-byte aligned", who);
  return HK_OK;
}

} // namespace hk

using namespace hk;

extern "C" {

int hk_batch_norm_workspace_bytes(int dtype, int64_t N, int64_t C, int64_t HW, size_t* bytes) {
  HK_REQUIRE(bytes, HK_ERR_INVALID, "hk_batch_norm_workspace_bytes: null output");
  HK_REQUIRE(N >= 0 && C >= 0 && HW >= 0, HK_ERR_INVALID, "hk_batch_norm_workspace_bytes: negative shape");
  *bytes = (N * C * HW == 0) ? 0 : bn_ws_bytes(N, C, HW, dtype == HK_FLOAT64 ? 8 : 4);
  return HK_OK;
}

int hk_batch_norm_fwd(int dtype, const void* x, const void* scale, const void* bias, void* y, double momentum,
                      double eps, void* running_mean, void* running_var, void* save_mean, void* save_invstd,
                      int64_t N, int64_t C, int64_t HW, void* workspace, size_t workspace_bytes,
                      hkStream_t stream) {
  size_t need = 0;
  int rc = bn_check("hk_batch_norm_fwd", dtype, N, C, HW, workspace, workspace_bytes, &need);
  if (rc != HK_OK) return rc;
  if (N * C * HW == 0) return HK_OK;
  HK_REQUIRE(x && scale && bias && y, HK_ERR_INVALID, "hk_batch_norm_fwd: null input/output");
  hipStream_t st = as_hip(stream);
  switch (dtype) {
    case HK_FLOAT32:
      return bn_fwd_typed<float, float>(x, scale, bias, y, momentum, eps, running_mean, running_var, save_mean,
                                        save_invstd, N, C, HW, workspace, st);
    case HK_BFLOAT16:
      return bn_fwd_typed<bf16, float>(x, scale, bias, y, momentum, eps, running_mean, running_var, save_mean,
                                       save_invstd, N, C, HW, workspace, st);
    case HK_FLOAT16:
      return bn_fwd_typed<fp16, float>(x, scale, bias, y, momentum, eps, running_mean, running_var, save_mean,
                                       save_invstd, N, C, HW, workspace, st);
    default:
      return bn_fwd_typed<double, double>(x, scale, bias, y, momentum, eps, running_mean, running_var, save_mean,
                                          save_invstd, N, C, HW, workspace, st);
  }
}

int hk_batch_norm_bwd(int dtype, const void* dy, const void* x, const void* scale, void* dx, void* dscale,
                      void* dbias, const void* save_mean, const void* save_invstd, int64_t N, int64_t C,
                      int64_t HW, void* workspace, size_t workspace_bytes, hkStream_t stream) {
  size_t need = 0;
  int rc = bn_check("hk_batch_norm_bwd", dtype, N, C, HW, workspace, workspace_bytes, &need);
  if (rc != HK_OK) return rc;
  if (N * C * HW == 0) return HK_OK;
  HK_REQUIRE(dy && x && scale && dx && save_mean && save_invstd, HK_ERR_INVALID,
             "hk_batch_norm_bwd: null input/output");
  hipStream_t st = as_hip(stream);
  switch (dtype) {
    case HK_FLOAT32:
      return bn_bwd_typed<float, float>(dy, x, scale, dx, dscale, dbias, save_mean, save_invstd, N, C, HW, workspace, st);
    case HK_BFLOAT16:
      return bn_bwd_typed<bf16, float>(dy, x, scale, dx, dscale, dbias, save_mean, save_invstd, N, C, HW, workspace, st);
    case HK_FLOAT16:
      return bn_bwd_typed<fp16, float>(dy, x, scale, dx, dscale, dbias, save_mean, save_invstd, N, C, HW, workspace, st);
    default:
      return bn_bwd_typed<double, double>(dy, x, scale, dx, dscale, dbias, save_mean, save_invstd, N, C, HW, workspace, st);
  }
}

} // extern "C"
