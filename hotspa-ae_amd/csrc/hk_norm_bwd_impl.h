// LayerNorm / RMSNorm backward kernels and their launch logic, included by the per-type instantiation files.
//
// A persistent grid walks the rows; every thread owns a fixed set of columns, keeps the dgamma / dbeta column
// sums of its rows in registers, and the workgroup writes ONE fp32 partial row per block which a small second
// kernel folds into dgamma / dbeta.
#pragma once

#include "hk_norm.h"

namespace hk {

__device__ __forceinline__ float clamp_by_magnitude(float g, float eps) {
  // |g| < eps is pushed out to +-eps keeping the sign (zero counts as positive)
  if (g >= 0.f) return g < eps ? eps : g;
  return g > -eps ? -eps : g;
}

// Column-owner backward kernel.  A group of `tpr` threads walks rows; thread t
// owns the same columns in every row, so its dgamma / dbeta sums stay in
// registers.  With xc = x - mu (x for RMSNorm), t = dy * gamma and
// m2 = mean(t * xc):   dx = rs * t - rs * mean(t) - xc * rs^3 * m2,
// two fused multiply-adds per element once the row sums are known.
//
// PF rows per thread group are in flight at any time (a ring of register slots,
// refilled as soon as a slot has been unpacked).  The steady-state loop is
// written without a single branch around a memory instruction: out-of-range
// rows are clamped instead of skipped, EXACT says that no thread has a column
// past the row's end, STATS_F32 fixes the statistics' type, EXTRA says whether the
// optional operands (an upstream gradient added to dx, a second copy of dx) exist
// at all.  Only then does the compiler count outstanding loads exactly; any branch
// around a load in the loop makes it wait for all of them at every step, which
// flattens the ring to depth one.  Rows that do not fill a whole round of PF steps
// go through the same step with its guards switched on.
//
// MAXT is the launch bound: the register budget follows the block size the plan
// really uses (a 640-thread block of the 5120-column LayerNorm may hold 170
// registers per lane where a 1024-thread block may hold 128), which is what lets
// the LayerNorm modes, with the mean in their ring as well, keep two rows in flight.
//
// FIXED says that one group of exactly MAXT threads is the whole block: the group's
// width, and with it the number of wavefront partials every thread adds up after the
// barrier, is then a constant and the cross-wavefront step is straight-line code.
// Whatever the hot case never has is decided at compile time there: EXTRA also stands
// for "gamma clamped in dx on request" (a uniform branch between two copies of the
// arithmetic otherwise, whose merge costs one register move per live value per row);
// without EXTRA, CLAMP says at compile time whether gamma enters dx clamped (the fused
// LayerNorm's backward does that in both of its modes, the plain one never).
//
// The lean RMSNorm instances (MODE == BWD_RMS without EXTRA) form no column sums of dy: an RMSNorm has no bias, and
// eight additions and eight registers per row and thread are a tenth of the loop.  A caller that asks for dbeta
// under RMSNorm all the same (the dropout-add-norm interface allows it) is served by the general instance.
//
// LEVELS (FIXED instances without optional operands only): the rows lie on several levels (see LevelSteps).  The
// loads are issued in strictly increasing row order, one grid size apart, so the walk index of the next row to
// issue is kept as a running (j0, j1, j2) in scalar registers and advanced by the split grid size with two
// carries: no division in the loop, nothing on the vector unit.  The general instance takes levels too, with
// optional operands, by splitting each row number with two divisions.
//
// RAGGED: rows of any length and alignment, see AnyBoundary.  The row's partial last vector is
// read as its last whole one; the elements that it shares with the vector before it are left out of the row sums, their
// dx comes out of both to the same bits and is stored twice, in whole vectors (element by element, up to seven stores
// per row: 14549 x 3579 bf16 68.5 us instead of 57.2).  The partial rows of the column sums keep whole vectors
// (part_pitch), of which the fold takes every column once.  LayerNorm backward of 8191 x 1021 bf16: 1114 us element by
// element, 13.8 us so (8192 x 1024 on the 16-byte grid: 12.9); of 8192 x 8191 fp32 1328 -> 150 us (5.4 TB/s).
//
// LPR: that many lanes of a wavefront hold a row (plan_norm_bwd_lanes); 0 for whole wavefronts.
template <typename T, int NV, int MODE, int PF, bool EXACT, bool STATS_F32, bool EXTRA, int MAXT, bool FIXED,
          bool CLAMP, bool LEVELS = false, bool RAGGED = false, int LPR = 0>
__global__ __launch_bounds__(MAXT)
void norm_bwd_kernel(typename std::conditional<LEVELS || EXTRA, NormBwdArgs, NormBwdFlat>::type given) {
  const NormBwdArgs a = given.template args<T, MODE>();
  static_assert(LPR == 0 || (RAGGED && LPR < kWave && NV == 1), "several rows to a wavefront: any boundary, a vector per lane");
  static_assert(!LEVELS || (FIXED && !EXTRA && EXACT), "the running walk index is built for the lean instances");
  static_assert(!RAGGED || (!FIXED && !EXACT), "rows of any boundary: any group width, a partial last vector");
  constexpr int VEC = VecIO<T>::N;
  constexpr int NE = NV * VEC;
  constexpr int KS = (MODE == BWD_RMS) ? 1 : 2;   // row sums to reduce: RMSNorm has no mean term
  constexpr bool WITH_DB = EXTRA || MODE != BWD_RMS;   // column sums of dy (dbeta)
  using StatT = typename std::conditional<STATS_F32, float, T>::type;
  using RowSums = SumTuple<KS>;
  extern __shared__ __align__(16) float lds[];   // [2][rows_per_block, part_pitch] staging of both column sums (staging_bytes)
  __shared__ __align__(16) float red[2][kMaxWaves * KS];  // double-buffered by step parity

  const int tpr = FIXED ? MAXT : LPR ? LPR : a.tpr;   // without LPR a multiple of 64: a wavefront never straddles two rows
  const int rpb = FIXED ? 1 : a.threads / tpr;
  const int group = FIXED ? 0 : LPR ? int(threadIdx.x) / tpr : __builtin_amdgcn_readfirstlane(int(threadIdx.x) / tpr);
  const int t = int(threadIdx.x) - group * tpr;
  const int waves_per_group = tpr >> 6;
  const int first_wave = group * waves_per_group;

  // column vectors of this thread; a thread past the row's end (only when !EXACT) reads the last vector
  // again and has its dy forced to zero, so it adds nothing and stores nothing
  int vidx[NV];
  bool vin[NV];
  int col[NV];                            // first column that vector i loads
  [[maybe_unused]] uint32_t own[VEC];     // RAGGED: which elements of the last loaded vector count in the row sums
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int v = i * tpr + t;
    vin[i] = EXACT || v < a.nvec;
    vidx[i] = vin[i] ? v : a.nvec - 1;
    col[i] = vec_column<T, RAGGED>(vidx[i], a.cols);
    if constexpr (RAGGED) {
      const int skip = (v + 1) * VEC - a.cols;   // VEC or more past the row's end
      if (i == NV - 1) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) own[j] = skip > j ? 0u : 0xffffffffu;
      }
    }
  }
  auto ld_row = [](const T* p) { if constexpr (RAGGED) return ld16_any<T>(p); else return ld16(p); };
  auto ld_par = [](const T* p) { if constexpr (RAGGED) return ld16_any_keep<T>(p); else return ld16_keep(p); };

  [[maybe_unused]] const bool clamp = MODE == BWD_LN_MEMEFF || CLAMP || (EXTRA && a.clamp_gamma != 0);

  float dg[NE], db[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) { dg[e] = 0.f; db[e] = 0.f; }

  const int64_t stride = int64_t(a.blocks) * rpb;
  const int64_t last_row = a.rows - 1;
  u32x4 nx[PF][NV], ndy[PF][NV];
  StatT nmu[PF], nsv[PF];
  const StatT* meanp = static_cast<const StatT*>(a.mean);
  const StatT* statp = static_cast<const StatT*>(a.stat);
  // LEVELS: walk index of the next row to issue, and where each slot's dx row goes
  [[maybe_unused]] uint32_t wj0 = 0, wj1 = 0, wj2 = 0;
  [[maybe_unused]] int64_t dxo[PF];
  if constexpr (LEVELS) {
    const RowSplit first = split_row(int64_t(blockIdx.x), a.n0, a.n1);
    wj0 = __builtin_amdgcn_readfirstlane(first.j0);
    wj1 = __builtin_amdgcn_readfirstlane(first.j1);
    wj2 = __builtin_amdgcn_readfirstlane(first.j2);
  }
  // loads of row r into slot d; r past the end re-reads the last row (its results are never used)
  auto issue = [&](auto slot, int64_t r) {
    constexpr int d = decltype(slot)::value;
    const int64_t rc = r < last_row ? r : last_row;
    int64_t xo = rc * a.x_pitch, dyo = rc * a.dy_pitch, number = rc;
    if constexpr (LEVELS) {
      // a row past the end reads row 0 instead (any row will do)
      const bool ok = r <= last_row;
      const RowSplit sp{ok ? wj0 : 0u, ok ? wj1 : 0u, ok ? wj2 : 0u};
      xo = split_offset(sp, a.x_pitch, a.x_lv);
      dyo = split_offset(sp, a.dy_pitch, a.dy_lv);
      number = split_number(sp, a.rn);
      dxo[d] = split_offset(sp, a.dx_pitch, a.dx_lv);
      // the next row to issue lies one grid size further on
      wj0 += a.ws0;
      uint32_t carry = wj0 >= uint32_t(a.n0) ? 1u : 0u;
      wj0 -= carry ? uint32_t(a.n0) : 0u;
      wj1 += a.ws1 + carry;
      carry = wj1 >= uint32_t(a.n1) ? 1u : 0u;
      wj1 -= carry ? uint32_t(a.n1) : 0u;
      wj2 += a.ws2 + carry;
    }
    if constexpr (EXTRA) {
      if (a.n0 != a.rows) {   // rows on several levels: uniform
        const RowSplit sp = split_row(rc, a.n0, a.n1);
        xo = split_offset(sp, a.x_pitch, a.x_lv);
        dyo = split_offset(sp, a.dy_pitch, a.dy_lv);
        number = split_number(sp, a.rn);
      }
    }
    if constexpr (MODE == BWD_LN) nmu[d] = meanp[number];
    nsv[d] = statp[number];
    const T* xr = static_cast<const T*>(a.x) + xo;
    const T* dyr = static_cast<const T*>(a.dy) + dyo;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      nx[d][i] = ld_row(xr + col[i]);
      ndy[d][i] = ld_row(dyr + col[i]);
    }
  };
  int64_t row0 = int64_t(blockIdx.x) * rpb + group;
  // gamma (and beta) of this thread's columns as fp32; a missing gamma is all ones
  float gm[NE];
  [[maybe_unused]] float bt[MODE == BWD_LN_MEMEFF ? NE : 1];
  auto load_parameters = [&] {
    const T* gp = static_cast<const T*>(a.gamma);
    const T* bp = static_cast<const T*>(a.beta);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
#pragma unroll
      for (int j = 0; j < VEC; ++j) gm[i * VEC + j] = 1.f;
      if (gp) VecIO<T>::unpack(ld_par(gp + col[i]), &gm[i * VEC]);
      if constexpr (MODE == BWD_LN_MEMEFF) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) bt[i * VEC + j] = 0.f;
        if (bp) VecIO<T>::unpack(ld_par(bp + col[i]), &bt[i * VEC]);
      }
    }
  };
  // behind the first rows' loads, so that one latency covers both; the longest walks (one group of a whole workgroup) are
  // the better for it the other way round (32768 x 4096, forward and backward: 0.2 % of 216 us)
  if constexpr (FIXED) load_parameters();
  static_for<PF>([&](auto slot) { issue(slot, row0 + decltype(slot)::value * stride); });
  if constexpr (!FIXED) load_parameters();

  int parity = 0;
  // guarded: check that the slot's row exists (the tail); otherwise it is known to
  auto step = [&](auto slot, auto guarded) {
    constexpr int d = decltype(slot)::value;
    constexpr bool GUARD = decltype(guarded)::value;
    const int64_t row = row0 + d * stride;
    const bool valid = !GUARD || row < a.rows;
    float xs[NE], ts[NE];                 // xc (x_hat in the memory-efficient mode) and dy * gamma
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      VecIO<T>::unpack(nx[d][i], &xs[i * VEC]);
      VecIO<T>::unpack(ndy[d][i], &ts[i * VEC]);
      if (!EXACT && !RAGGED) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) ts[i * VEC + j] = vin[i] ? ts[i * VEC + j] : 0.f;
      }
    }
    [[maybe_unused]] float mu = 0.f;
    if constexpr (MODE == BWD_LN) mu = Cvt<StatT>::to_float(nmu[d]);
    const float sv = Cvt<StatT>::to_float(nsv[d]);
    // RMSNorm keeps the inverse root mean square, never a variance
    const float rs = (MODE != BWD_RMS && a.stat_kind == HK_STAT_VAR) ? 1.0f / sqrtf(sv + a.eps) : sv;
    [[maybe_unused]] int64_t dx_offset = 0;
    if constexpr (LEVELS) dx_offset = dxo[d];   // the refill below reuses the slot
    // the slot is free again: refill it with the row PF steps ahead
    issue(slot, row + int64_t(PF) * stride);

    // an element that the row's last vector shares with the one before it counts once in the row sums; its column
    // sums stay with the fold, which takes each column from one of them
    auto in_sums = [&](float v, int e) {
      if constexpr (RAGGED) return e >= NE - VEC ? u2f(f2u(v) & own[e - (NE - VEC)]) : v;
      else return v;
    };
    RowSums s = RowSums::identity();
    float& s_prod = s.v[KS - 1];            // sum(dy g xc) (sum(dy (y - beta)) in the memory-efficient mode)
    // new column sums go to copies first: a guarded step of a missing row must leave dg / db alone
    // without a branch around the arithmetic
    auto accumulate = [&](auto clamped) {
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const float dz = (GUARD && !valid) ? 0.f : ts[e];
        if constexpr (MODE == BWD_LN_MEMEFF) {
          const float yb = xs[e] - bt[e];
          const float kg = clamp_by_magnitude(gm[e], a.eps);
          const float xhat = yb / kg;
          s.v[0] = fmaf(in_sums(dz, e), gm[e], s.v[0]);
          s_prod = fmaf(in_sums(dz, e), in_sums(yb, e), s_prod);
          dg[e] = fmaf(dz, xhat, dg[e]);
          if constexpr (WITH_DB) db[e] += dz;
          xs[e] = xhat;
          ts[e] = dz * kg;
        } else {
          const float xc = (MODE == BWD_RMS) ? xs[e] : xs[e] - mu;
          const float dzr = dz * rs;
          const float q = dzr * gm[e];
          s_prod = fmaf(in_sums(q, e), in_sums(xc, e), s_prod);
          if constexpr (MODE != BWD_RMS) s.v[0] += in_sums(q, e);
          dg[e] = fmaf(dzr, xc, dg[e]);
          if constexpr (WITH_DB) db[e] += dz;
          xs[e] = xc;
          // the per-element term of dx uses the clamped gamma when asked to
          if constexpr (decltype(clamped)::value) ts[e] = dzr * clamp_by_magnitude(gm[e], a.eps);
          else ts[e] = q;
        }
      }
    };
    if constexpr (!EXTRA) accumulate(std::integral_constant<bool, MODE == BWD_LN_MEMEFF || CLAMP>{});
    else if (clamp) accumulate(std::true_type{});   // uniform
    else accumulate(std::false_type{});

    if constexpr (LPR != 0) {
      // No barrier separates the steps of a lane group: without this the column sums of every step of a round are
      // formed at the round's end, and each step's row stays in registers until then (LayerNorm, bf16: 123 registers
      // instead of 94).
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        asm volatile("" : "+v"(dg[e]));
        if constexpr (WITH_DB) asm volatile("" : "+v"(db[e]));
      }
    }
    if constexpr (LPR != 0) s = lanes_allreduce_tuple<LPR>(s);
    else if constexpr (FIXED) s = group_allreduce_tuple_fixed<RowSums, MAXT / 64>(s, red[parity]);
    else s = group_allreduce_tuple(s, red[parity], first_wave, waves_per_group);
    parity ^= 1;
    if (valid) {
      // plain modes: s0 = rs * sum(dy g), s1 = rs * sum(dy g xc);  dx = q - s0/n - xc * rs^2 * s1/n
      // memory-efficient: s0 = sum(dy g), s1 = sum(dy (y - beta));   dx = rs * (dy kg - s0/n - xhat * s1/n)
      float rc1, k3;
      if constexpr (MODE == BWD_LN_MEMEFF) {
        rc1 = rs * s.v[0] * a.inv_cols;
        k3 = rs * s_prod * a.inv_cols;
      } else {
        rc1 = (MODE == BWD_RMS) ? 0.f : s.v[0] * a.inv_cols;
        k3 = rs * rs * s_prod * a.inv_cols;
      }
      T* dxr = static_cast<T*>(a.dx) + (LEVELS ? dx_offset : row * a.dx_pitch);
      [[maybe_unused]] T* drr = nullptr;
      [[maybe_unused]] const T* dir = nullptr;
      if constexpr (EXTRA) {
        const bool levels = a.n0 != a.rows;   // uniform
        RowSplit sp{};
        if (levels) {
          sp = split_row(row, a.n0, a.n1);
          dxr = static_cast<T*>(a.dx) + split_offset(sp, a.dx_pitch, a.dx_lv);
        }
        if (a.dres) drr = static_cast<T*>(a.dres) + (levels ? split_offset(sp, a.dres_pitch, a.dres_lv) : row * a.dres_pitch);
        if (a.dx_in) {
          dir = static_cast<const T*>(a.dx_in) + (levels ? split_offset(sp, a.dxin_pitch, a.dxin_lv) : row * a.dxin_pitch);
        }
      }
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        if (EXACT || vin[i]) {
          const int v = vidx[i];
          float o[VEC];
#pragma unroll
          for (int j = 0; j < VEC; ++j) {
            const float base = (MODE == BWD_LN_MEMEFF) ? fmaf(ts[i * VEC + j], rs, -rc1)
                                                       : ts[i * VEC + j] - rc1;
            o[j] = fmaf(-xs[i * VEC + j], k3, base);
          }
          if constexpr (EXTRA) {
            if (dir) {
              float u[VEC];
              VecIO<T>::unpack(ld_row(dir + col[i]), u);
#pragma unroll
              for (int j = 0; j < VEC; ++j) o[j] += u[j];
            }
          }
          if constexpr (RAGGED) {
            // (an upstream gradient that is added in place must not be read after a neighbour has stored over it)
            store_row_vec<T, true, !EXTRA>(dxr, v, o, a.cols);
            if (drr) store_row_vec<T, true, false>(drr, v, o, a.cols);
          } else {
            const u32x4 pk = VecIO<T>::pack(o);
            st16_stream(dxr + v * VEC, pk);
            if constexpr (EXTRA) {
              if (drr) st16(drr + v * VEC, pk);
            }
          }
        }
      }
    }
  };
  // Every thread of the block takes the same number of steps (both loop bounds are block-uniform), so
  // the barrier inside the group reduction is reached by all of them.
  int64_t base = int64_t(blockIdx.x) * rpb;
  const int64_t round = int64_t(PF) * stride;
  // rounds in which every slot of every group of this block holds an existing row
#pragma nounroll
  for (; base + int64_t(PF - 1) * stride + rpb <= a.rows; base += round) {
    static_for<PF>([&](auto slot) { step(slot, std::false_type{}); });
    row0 += round;
  }
#pragma nounroll
  for (; base < a.rows; base += round) {
    static_for<PF>([&](auto slot) { step(slot, std::true_type{}); });
    row0 += round;
  }

  // fold the row groups of this block, then write one partial row per block, as 16-byte streaming stores (the partial
  // rows are read by the fold kernel, never again by this one; left in the cache they would only wait for the
  // write-back at the kernel's end)
  static_assert(VEC % 4 == 0, "whole float4 vectors per 16-byte vector of the data type");
  float* outs[2] = {a.part_dgamma, WITH_DB ? a.part_dbeta : nullptr};
  auto put = [&](float* dst, const float* acc, bool stream) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      if (!EXACT && !vin[i]) continue;
#pragma unroll
      for (int j = 0; j < VEC; j += 4) {
        const u32x4 pk = {f2u(acc[i * VEC + j]), f2u(acc[i * VEC + j + 1]), f2u(acc[i * VEC + j + 2]),
                          f2u(acc[i * VEC + j + 3])};
        if (stream) st16_stream(dst + vidx[i] * VEC + j, pk);
        else st16(dst + vidx[i] * VEC + j, pk);
      }
    }
  };
  if (FIXED || rpb == 1) {   // every thread writes its own sums
    if (outs[0]) put(outs[0] + int64_t(blockIdx.x) * a.part_pitch, dg, true);
    if (WITH_DB && outs[1]) put(outs[1] + int64_t(blockIdx.x) * a.part_pitch, db, true);
    return;
  }
  // Several groups: every group stages its sums, then neighbouring threads fold neighbouring columns, 16 bytes each.
  // (Folded by the first group alone, element by element, either sum took 4 us of a kernel that has 2 us of rows:
  // LayerNorm of 1218 x 92 fp16 11.3 us.)
  const int pitch = a.part_pitch, region = rpb * pitch;
  auto fold = [&](const float* src, float* dst) {
    if (dst == nullptr) return;
    for (int c = int(threadIdx.x) * 4; c < pitch; c += a.threads * 4) {
      float r[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
      for (int g = 0; g < rpb; ++g) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(src + g * pitch + c);
        r[0] += u2f(v.x); r[1] += u2f(v.y); r[2] += u2f(v.z); r[3] += u2f(v.w);
      }
      st16(dst + int64_t(blockIdx.x) * pitch + c, u32x4{f2u(r[0]), f2u(r[1]), f2u(r[2]), f2u(r[3])});
    }
  };
  put(lds + group * pitch, dg, false);
  if constexpr (WITH_DB) put(lds + region + group * pitch, db, false);
  __syncthreads();
  fold(lds, outs[0]);
  if constexpr (WITH_DB) fold(lds + region, outs[1]);
}

// Folds the [nparts, pitch] fp32 partial rows into dgamma / dbeta of type T (fold_partial_rows); blockIdx.y picks which.  Rows
// of whole 16-byte vectors of T: pitch == cols; otherwise the last vector of a partial row holds the row's last columns, the
// first pitch - cols of its elements being another vector's.
template <typename T, int LANES>
__global__ __launch_bounds__(fold_threads(LANES))
void norm_bwd_finalize_kernel(const float* part0, const float* part1, T* out0, T* out1, int nparts, int cols, int pitch) {
  T* out = blockIdx.y == 0 ? out0 : out1;
  const float s = fold_partial_rows<LANES>(blockIdx.y == 0 ? part0 : part1, nparts, pitch, int(blockIdx.x));
  const int oc = int(blockIdx.x) * (4 * LANES) + int(threadIdx.x);
  if (int(threadIdx.x) >= 4 * LANES || oc >= pitch) return;
  const int shift = pitch - cols, tail = pitch - VecIO<T>::N;   // shift > 0: the partial last vector
  if (shift == 0 || oc < tail) Cvt<T>::store(out + oc, s);
  else if (oc >= tail + shift) Cvt<T>::store(out + oc - shift, s);
}

constexpr int small_lanes(bool ragged) { return ragged ? 4 : 8; }
// The whole backward of a small array in one launch.  Its time is that of launches and trips to memory, of which the kernels above
// take three (rows, partial rows, their fold), so here the first a.blocks workgroups form the column sums from the operands
// themselves, LANES vectors of every row each, and the others dx: what is read twice comes from a cache.  Nothing that
// is written may lie over what is read (see column_sums_of_few_rows).  dx comes out to the same bits as from norm_bwd_kernel: the
// plan's threads and vectors, its order of operations.
template <typename T, int NV, int MODE, bool RAGGED>
__global__ __launch_bounds__(kSmallThreads)
void norm_bwd_small_kernel(NormBwdFlat given) {
  constexpr int LANES = small_lanes(RAGGED);
  const NormBwdArgs a = given.template args<T, MODE>();
  constexpr int VEC = VecIO<T>::N, SUMS = MODE == BWD_RMS ? 1 : 2;
  __shared__ __align__(16) float red[kMaxWaves * SUMS];
  auto ld_row = [](const T* p) { if constexpr (RAGGED) return ld16_any_keep<T>(p); else return ld16_keep(p); };
  auto rs_of = [&](float sv) { return (MODE != BWD_RMS && a.stat_kind == HK_STAT_VAR) ? 1.0f / sqrtf(sv + a.eps) : sv; };
  const float* meanp = static_cast<const float*>(a.mean);
  const float* statp = static_cast<const float*>(a.stat);
  const T* xp = static_cast<const T*>(a.x);
  const T* dyp = static_cast<const T*>(a.dy);
  const int rows = int(a.rows);
  if (int(blockIdx.x) < a.blocks) {
    struct Fetched {
      u32x4 x, dy;
      float mu, sv;
    };
    const int first = int(blockIdx.x) * LANES;
    const int col = vec_column<T, RAGGED>(min(first + (int(threadIdx.x) & (LANES - 1)), a.nvec - 1), a.cols);
    column_sums_of_few_rows<SUMS, VEC, LANES>(
        rows,
        [&](int64_t r) {
          return Fetched{ld_row(xp + r * a.x_pitch + col), ld_row(dyp + r * a.dy_pitch + col), MODE == BWD_LN ? meanp[r] : 0.f, statp[r]};
        },
        [&](const Fetched& f, bool in, float (&acc)[SUMS][VEC]) {
          const float rs = rs_of(f.sv);
          float x[VEC], d[VEC];
          VecIO<T>::unpack(f.x, x);
          VecIO<T>::unpack(f.dy, d);
#pragma unroll
          for (int j = 0; j < VEC; ++j) {
            const float more = fmaf(d[j] * rs, MODE == BWD_LN ? x[j] - f.mu : x[j], acc[0][j]);
            acc[0][j] = in ? more : acc[0][j];
            if constexpr (SUMS == 2) acc[1][j] += in ? d[j] : 0.f;
          }
        },
        [&](int k, int c, float sum) {
          T* out = reinterpret_cast<T*>(k == 0 ? a.part_dgamma : a.part_dbeta);
          const int v = first + c / VEC;
          const int at = vec_column<T, RAGGED>(v, a.cols) + c % VEC;   // a column that two vectors hold: from the first
          if (v < a.nvec && out != nullptr && at >= v * VEC) Cvt<T>::store(out + at, sum);
        });
    return;
  }

  const int tpr = a.tpr, rpb = kSmallThreads / tpr;
  const int group = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / tpr), t = int(threadIdx.x) - group * tpr;
  // (the wavefronts that no row is left for work on the last one too and store nothing)
  const bool idle = group >= rpb;
  const int64_t wanted = idle ? rows : int64_t(int(blockIdx.x) - a.blocks) * rpb + group, row = wanted < rows ? wanted : rows - 1;
  const T* xr = xp + row * a.x_pitch;
  const T* dyr = dyp + row * a.dy_pitch;
  const T* gp = static_cast<const T*>(a.gamma);
  u32x4 rx[NV], rdy[NV], rg[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = vec_column<T, RAGGED>(min(i * tpr + t, a.nvec - 1), a.cols);
    rx[i] = ld_row(xr + c);
    rdy[i] = ld_row(dyr + c);
    if (gp) rg[i] = ld_row(gp + c);   // uniform
  }
  const float mu = MODE == BWD_LN ? meanp[row] : 0.f, rs = rs_of(statp[row]);
  float xs[NV][VEC], ts[NV][VEC];
  SumTuple<SUMS> s = SumTuple<SUMS>::identity();
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    float g[VEC];
    VecIO<T>::unpack(rx[i], xs[i]);
    VecIO<T>::unpack(rdy[i], ts[i]);
#pragma unroll
    for (int j = 0; j < VEC; ++j) g[j] = 1.f;
    if (gp) VecIO<T>::unpack(rg[i], g);
    const int v = i * tpr + t;
    if constexpr (!RAGGED) {
#pragma unroll
      for (int j = 0; j < VEC; ++j) ts[i][j] = v < a.nvec ? ts[i][j] : 0.f;
    }
    auto in_sums = [&](float f, int j) {   // as in norm_bwd_kernel
      if (RAGGED && i == NV - 1) return u2f(f2u(f) & ((v + 1) * VEC - a.cols > j ? 0u : 0xffffffffu));
      return f;
    };
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const float xc = MODE == BWD_RMS ? xs[i][j] : xs[i][j] - mu;
      const float dzr = ts[i][j] * rs;
      const float q = dzr * g[j];
      s.v[SUMS - 1] = fmaf(in_sums(q, j), in_sums(xc, j), s.v[SUMS - 1]);
      if constexpr (MODE != BWD_RMS) s.v[0] += in_sums(q, j);
      xs[i][j] = xc;
      ts[i][j] = MODE == BWD_LN && a.clamp_gamma ? dzr * clamp_by_magnitude(g[j], a.eps) : q;
    }
  }
  s = group_allreduce_tuple(s, red, idle ? 0 : group * (tpr >> 6), tpr >> 6);
  if (wanted >= rows) return;
  const float rc1 = MODE == BWD_RMS ? 0.f : s.v[0] * a.inv_cols, k3 = rs * rs * s.v[SUMS - 1] * a.inv_cols;
  T* dxr = static_cast<T*>(a.dx) + row * a.dx_pitch;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int v = i * tpr + t;
    if (v < a.nvec) {
      float o[VEC];
#pragma unroll
      for (int j = 0; j < VEC; ++j) o[j] = fmaf(-xs[i][j], k3, ts[i][j] - rc1);
      store_row_vec<T, RAGGED, true>(dxr, v, o, a.cols);
    }
  }
}

// Fallback backward for rows the register kernel cannot take (shorter than a 16-byte vector, more than 8192 columns,
// no scratch given for rows off the 16-byte grid): one workgroup
// per row for dx, then a column kernel for dgamma / dbeta (re-reads dy and x).
template <typename T, typename CT>
__global__ __launch_bounds__(256)
void norm_bwd_generic_dx_kernel(NormBwdArgs a, int mode) {
  __shared__ CT lds[256];
  const int64_t i0 = blockIdx.x;                       // row within the innermost level
  const int64_t row = dense_row_index(i0, a.rn);
  const T* xr = static_cast<const T*>(a.x) + i0 * a.x_pitch + outer_level_offset(a.x_lv);
  const T* dyr = static_cast<const T*>(a.dy) + i0 * a.dy_pitch + outer_level_offset(a.dy_lv);
  const T* gp = static_cast<const T*>(a.gamma);
  const T* bp = static_cast<const T*>(a.beta);
  CT mu = 0;
  if (mode == BWD_LN) {
    mu = a.stats_f32 ? CT(static_cast<const float*>(a.mean)[row])
                     : GenericIO<T, CT>::ld(static_cast<const T*>(a.mean) + row);
  }
  const CT sv = a.stats_f32 ? CT(static_cast<const float*>(a.stat)[row])
                            : GenericIO<T, CT>::ld(static_cast<const T*>(a.stat) + row);
  const CT rs = a.stat_kind == HK_STAT_VAR ? CT(1) / sqrt(sv + CT(a.eps)) : sv;
  const bool clamp = a.clamp_gamma != 0 || mode == BWD_LN_MEMEFF;
  auto kgamma = [&](CT g) -> CT {
    if (!clamp) return g;
    const CT e = CT(a.eps);
    if (g >= CT(0)) return g < e ? e : g;
    return g > -e ? -e : g;
  };
  auto xhat_of = [&](int c, CT g) -> CT {
    const CT xv = GenericIO<T, CT>::ld(xr + c);
    if (mode == BWD_LN_MEMEFF) return (xv - (bp ? GenericIO<T, CT>::ld(bp + c) : CT(0))) / kgamma(g);
    if (mode == BWD_RMS) return rs * xv;
    return rs * (xv - mu);
  };
  CT s1 = 0, s2 = 0;
  for (int c = threadIdx.x; c < a.cols; c += 256) {
    const CT g = gp ? GenericIO<T, CT>::ld(gp + c) : CT(1);
    const CT d = GenericIO<T, CT>::ld(dyr + c);
    if (mode == BWD_LN_MEMEFF) {
      const CT yb = GenericIO<T, CT>::ld(xr + c) - (bp ? GenericIO<T, CT>::ld(bp + c) : CT(0));
      s2 += d * yb;
    } else {
      s2 += d * g * xhat_of(c, g);
    }
    if (mode != BWD_RMS) s1 += d * g;
  }
  s1 = block_sum_generic<CT>(s1, lds);
  s2 = block_sum_generic<CT>(s2, lds);
  const CT inv = CT(1) / CT(a.cols);
  const CT c1 = s1 * inv, c2 = s2 * inv;
  T* dxr = static_cast<T*>(a.dx) + i0 * a.dx_pitch + outer_level_offset(a.dx_lv);
  T* drr = a.dres ? static_cast<T*>(a.dres) + i0 * a.dres_pitch + outer_level_offset(a.dres_lv) : nullptr;
  const T* dir = a.dx_in ? static_cast<const T*>(a.dx_in) + i0 * a.dxin_pitch + outer_level_offset(a.dxin_lv) : nullptr;
  for (int c = threadIdx.x; c < a.cols; c += 256) {
    const CT g = gp ? GenericIO<T, CT>::ld(gp + c) : CT(1);
    const CT d = GenericIO<T, CT>::ld(dyr + c);
    CT o = rs * (d * kgamma(g) - c1 - xhat_of(c, g) * c2);
    if (dir) o += GenericIO<T, CT>::ld(dir + c);
    GenericIO<T, CT>::st(dxr + c, o);
    if (drr) GenericIO<T, CT>::st(drr + c, o);
  }
}

// dgamma[c] = sum_r dy*xhat, dbeta[c] = sum_r dy : 64 columns per block, the
// 4 waves take interleaved rows, fold through LDS.
template <typename T, typename CT>
__global__ __launch_bounds__(256)
void norm_bwd_generic_cols_kernel(NormBwdArgs a, int mode, T* dgamma, T* dbeta) {
  __shared__ CT lds[2][4][kWave];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int c = blockIdx.x * kWave + lane;
  const T* gp = static_cast<const T*>(a.gamma);
  const T* bp = static_cast<const T*>(a.beta);
  CT sg = 0, sb = 0;
  if (c < a.cols) {
    const CT g = gp ? GenericIO<T, CT>::ld(gp + c) : CT(1);
    CT kg = g;
    {
      const CT e = CT(a.eps);
      if (g >= CT(0)) kg = g < e ? e : g; else kg = g > -e ? -e : g;
    }
    const CT b = (bp && mode == BWD_LN_MEMEFF) ? GenericIO<T, CT>::ld(bp + c) : CT(0);
    const bool levels = a.n0 != a.rows;
    for (int64_t r = w; r < a.rows; r += 4) {
      int64_t dyo = r * a.dy_pitch, xo = r * a.x_pitch, number = r;
      if (levels) {
        const RowSplit sp = split_row(r, a.n0, a.n1);
        dyo = split_offset(sp, a.dy_pitch, a.dy_lv);
        xo = split_offset(sp, a.x_pitch, a.x_lv);
        number = split_number(sp, a.rn);
      }
      const CT d = GenericIO<T, CT>::ld(static_cast<const T*>(a.dy) + dyo + c);
      const CT xv = GenericIO<T, CT>::ld(static_cast<const T*>(a.x) + xo + c);
      CT xhat;
      if (mode == BWD_LN_MEMEFF) {
        xhat = (xv - b) / kg;
      } else {
        const CT sv = a.stats_f32 ? CT(static_cast<const float*>(a.stat)[number])
                                  : GenericIO<T, CT>::ld(static_cast<const T*>(a.stat) + number);
        const CT rs = a.stat_kind == HK_STAT_VAR ? CT(1) / sqrt(sv + CT(a.eps)) : sv;
        CT mu = 0;
        if (mode == BWD_LN)
          mu = a.stats_f32 ? CT(static_cast<const float*>(a.mean)[number])
                           : GenericIO<T, CT>::ld(static_cast<const T*>(a.mean) + number);
        xhat = rs * (xv - mu);
      }
      sg += d * xhat;
      sb += d;
    }
  }
  lds[0][w][lane] = sg;
  lds[1][w][lane] = sb;
  __syncthreads();
  if (w == 0 && c < a.cols) {
    CT tg = 0, tb = 0;
    for (int i = 0; i < 4; ++i) { tg += lds[0][i][lane]; tb += lds[1][i][lane]; }
    if (dgamma) GenericIO<T, CT>::st(dgamma + c, tg);
    if (dbeta) GenericIO<T, CT>::st(dbeta + c, tb);
  }
}

// LDS in which the row groups of a workgroup stage both column sums.  A thread has 8 columns in workgroups of up to 1024
// threads, or 16 in up to 512, so that this is at most 64 KiB (8 groups of 1021 to 1024 columns, say); with the 256 bytes of
// the reductions' own array it is within the 160 KiB that a workgroup may have, one workgroup being all that a compute
// unit is given.
static inline size_t staging_bytes(int groups, int pitch) {
  return groups > 1 ? size_t(2) * size_t(groups) * size_t(pitch) * sizeof(float) : 0;
}

// Many rows of up to 32 vectors, dense or pitched, on any boundary, without optional operands: 16 or 32 lanes to a row,
// a vector per lane, two rows in flight per group.  A wavefront to a row leaves half of its lanes and more idle; that
// shows once its workgroups, 16 rows each on every compute unit, have to walk (LayerNorm bf16, 32768 x 64 12.9 -> 8.1 us,
// 32768 x 256 14.3 -> 12.9, 10490 x 80 7.1 -> 6.2), and not before (2530 x 71 5.8 against 6.1, 1218 x 92 5.1 against 5.8).
// Longer rows do not gain from a wavefront of their own either, although it needs no barrier: 31451 x 1792 58.2 -> 63.7,
// 8191 x 1021 13.3 -> 14.7, 4002 x 904 8.4 -> 9.0.
template <typename T>
BwdPlan plan_norm_bwd_lanes(int64_t rows, int cols) {
  constexpr int VEC = VecIO<T>::N;
  BwdPlan p{};
  const int nvec = (cols + VEC - 1) / VEC, pitch = nvec * VEC;
  if (cols < VEC || nvec > 32 || rows <= int64_t(device_cu_count()) * 16) return p;
  p.lpr = nvec <= 16 ? 16 : 32;
  p.nv = 1;
  p.tpr = p.lpr;
  p.block = 512;
  p.rpb = p.block / p.lpr;
  int64_t grid = tune_get(TUNE_NORM_BWD_BLOCKS);
  if (grid <= 0) grid = device_cu_count();
  p.grid = int(std::max<int64_t>(1, std::min<int64_t>(grid, (rows + p.rpb - 1) / p.rpb)));
  p.reg_path = true;
  p.lds_bytes = staging_bytes(p.rpb, pitch);
  p.ws_bytes = size_t(2) * size_t(p.grid) * pitch * sizeof(float);
  return p;
}

// Rows that the aligned plan does not take: the general instance at 8 columns per thread (bf16, fp16; 4 for short fp32
// rows), one 1024-thread workgroup per compute unit, as many rows per step as fit it.  The partial rows stay within
// 16 MiB (what the library's own scratch holds) by using fewer workgroups for the longest rows.
template <typename T>
BwdPlan plan_norm_bwd_any(int64_t rows, int cols) {
  constexpr int VEC = VecIO<T>::N;
  BwdPlan p{};
  if (cols < VEC) return p;
  const int nvec = (cols + VEC - 1) / VEC, pitch = nvec * VEC;
  const int nv = VEC == 4 && nvec > 1024 ? 2 : 1;
  const int tpr = ((nvec + nv - 1) / nv + 63) / 64 * 64;
  if (tpr > 1024) return p;
  const int rpb = std::max(1, 1024 / tpr);
  int64_t grid = tune_get(TUNE_NORM_BWD_BLOCKS);
  if (grid <= 0) grid = device_cu_count();
  grid = std::min<int64_t>(grid, (rows + rpb - 1) / rpb);
  grid = std::min<int64_t>(grid, (int64_t(16) << 20) / (int64_t(2) * pitch * int64_t(sizeof(float))));
  if (grid < 1) grid = 1;
  p.reg_path = p.any = true;
  p.tpr = tpr; p.nv = nv; p.rpb = rpb; p.grid = int(grid); p.block = tpr * rpb;
  p.lds_bytes = staging_bytes(rpb, pitch);
  p.ws_bytes = size_t(2) * size_t(grid) * pitch * sizeof(float);
  return p;
}

template <typename T>
BwdPlan plan_norm_bwd(int64_t rows, int cols, bool aligned) {
  constexpr int VEC = VecIO<T>::N;
  BwdPlan p{};
  p.reg_path = false;
  if (!aligned || cols % VEC != 0) return plan_norm_bwd_any<T>(rows, cols);
  const int nvec = cols / VEC;
  // column-owner kernel: the dgamma / dbeta accumulators of a thread must stay
  // in registers: 8 columns per thread by default, 16 when a thread count is forced
  const int max_nv = (tune_get(TUNE_NORM_BWD_THREADS) > 0 ? 16 : 8) / VEC;
  int tpr = tune_get(TUNE_NORM_BWD_THREADS);
  int nv;
  if (tpr > 0) {
    tpr = std::min(1024, std::max(64, (tpr + 63) / 64 * 64));
    nv = pow2_ceil((nvec + tpr - 1) / tpr);
    if (nv > max_nv) return plan_norm_bwd_any<T>(rows, cols);
  } else {
    nv = max_nv;
    // short rows: fewer vectors per thread rather than a partly idle wavefront
    while (nv > 1 && (nvec + nv - 1) / nv < 64) nv >>= 1;
    tpr = ((nvec + nv - 1) / nv + 63) / 64 * 64;
    if (tpr > 1024) return plan_norm_bwd_any<T>(rows, cols);
  }
  // kernels with more than one vector per thread are built for 512-thread blocks
  const int max_block = nv == 1 ? 1024 : 512;
  if (tpr > max_block) return plan_norm_bwd_any<T>(rows, cols);
  int rpb = tune_get(TUNE_NORM_BWD_ROWS_PER_BLOCK);
  if (rpb <= 0) {
    rpb = std::max(1, max_block / tpr);
    // 512 threads already stream a whole 4096-column row per step; pairing two such groups in one
    // workgroup only adds waves to every barrier (measured 2-3 % slower than one group per workgroup)
    if (tpr >= 512) rpb = 1;
  }
  rpb = std::max(1, std::min(rpb, max_block / tpr));
  int grid = tune_get(TUNE_NORM_BWD_BLOCKS);
  if (grid <= 0) grid = device_cu_count();   // one 1024-thread workgroup per CU measured fastest
  const int64_t max_useful = (rows + rpb - 1) / rpb;
  if (grid > max_useful) grid = int(max_useful);
  if (grid < 1) grid = 1;
  p.reg_path = true;
  p.tpr = tpr; p.nv = nv; p.rpb = rpb; p.grid = grid; p.block = tpr * rpb;
  p.lds_bytes = staging_bytes(rpb, cols);
  p.ws_bytes = size_t(2) * grid * cols * sizeof(float);
  return p;
}

// launch bound of the kernel instance that runs a block of `block` threads
static inline int bound_for(int block) {
  return block <= 512 ? 512 : (block <= 640 ? 640 : (block <= 768 ? 768 : 1024));
}

template <typename T, int MODE, int NV, int MAXT>
static int launch_norm_bwd_inst(const NormBwdArgs& a, const BwdPlan& p, int pf, hipStream_t s) {
  dim3 grid{unsigned(p.grid)}, block{unsigned(p.block)};
  const bool exact = int64_t(p.nv) * p.tpr == a.nvec;
  const bool f32 = a.stats_f32 != 0;
  // the kernel's "extra" instance takes the optional operands behind uniform branches, and the clamp request in
  // the modes that have no instance of their own for it
  const bool want_clamp = a.clamp_gamma != 0 && MODE != BWD_LN_MEMEFF;   // the memory-efficient mode always clamps
  // one group that is the whole block, of exactly the bound's size: the instance with a constant group width
  const bool fixed = p.rpb == 1 && p.block == MAXT;
  // rows on several levels: the lean fixed instances keep a running walk index; every other case splits each row
  // number in the general instance
  const bool levels = a.n0 != a.rows;
  // (dbeta under RMSNorm counts as optional: the lean RMSNorm instances do not form it)
  const bool optional = a.dx_in != nullptr || a.dres != nullptr || (want_clamp && MODE != BWD_LN) ||
                        (MODE == BWD_RMS && a.part_dbeta != nullptr);
  const bool extra = optional || (levels ? !(fixed && exact) : !NormBwdFlat::holds(a));
  // the deep ring exists for the plain case only: full rows, no optional operands
  if (!exact || extra) pf = 1;
#define HK_BWD_LAUNCH_L(P, E, F, X, FX, C, L)                                                                            \
  do {                                                                                                                  \
    if constexpr (X || L) HK_LAUNCH((norm_bwd_kernel<T, NV, MODE, P, E, F, X, MAXT, FX, C, L>), grid, block, p.lds_bytes, s, a); \
    else HK_LAUNCH((norm_bwd_kernel<T, NV, MODE, P, E, F, X, MAXT, FX, C, L>), grid, block, p.lds_bytes, s, NormBwdFlat(a, MODE)); \
  } while (0)
#define HK_BWD_LAUNCH(P, E, F, X, FX, C) HK_BWD_LAUNCH_L(P, E, F, X, FX, C, false)
#define HK_BWD_LEAN_L(P, F, FX, L)                                          \
  do {                                                                      \
    if constexpr (MODE == BWD_LN) {                                         \
      if (want_clamp) HK_BWD_LAUNCH_L(P, true, F, false, FX, true, L); else HK_BWD_LAUNCH_L(P, true, F, false, FX, false, L); \
    } else {                                                                \
      HK_BWD_LAUNCH_L(P, true, F, false, FX, false, L);                     \
    }                                                                       \
  } while (0)
#define HK_BWD_LEAN(P, F, FX) HK_BWD_LEAN_L(P, F, FX, false)
#define HK_BWD_F(F)                                                         \
  do {                                                                      \
    if (exact && !extra && fixed && levels) { if (pf >= 2) HK_BWD_LEAN_L(2, F, true, true); else HK_BWD_LEAN_L(1, F, true, true); } \
    else if (exact && !extra && fixed) { if (pf >= 2) HK_BWD_LEAN(2, F, true); else HK_BWD_LEAN(1, F, true); } \
    else if (exact && !extra) { if (pf >= 2) HK_BWD_LEAN(2, F, false); else HK_BWD_LEAN(1, F, false); } \
    else if (exact) HK_BWD_LAUNCH(1, true, F, true, false, false);          \
    else if (!extra && !want_clamp) HK_BWD_LAUNCH(1, false, F, false, false, false); \
    else HK_BWD_LAUNCH(1, false, F, true, false, false);                    \
  } while (0)
  if constexpr (MODE == BWD_LN && !std::is_same<T, float>::value) {
    if (f32) HK_BWD_F(true); else HK_BWD_F(false);
  } else {
    HK_BWD_F(true);   // for float data "statistics in the data type" and "in float" are the same kernel
  }
#undef HK_BWD_F
#undef HK_BWD_LEAN
#undef HK_BWD_LEAN_L
#undef HK_BWD_LAUNCH
#undef HK_BWD_LAUNCH_L
  return HK_OK;
}

template <typename T, int MODE, bool CLAMP, int MAXT>
static void launch_norm_bwd_lanes(const NormBwdArgs& a, const BwdPlan& p, hipStream_t s) {
  const dim3 grid{unsigned(p.grid)}, block{unsigned(p.block)};
#define HK_BWD_LANES(NV, LPR) \
  HK_LAUNCH((norm_bwd_kernel<T, NV, MODE, 2, false, true, false, MAXT, false, CLAMP, false, true, LPR>), grid, block, \
            p.lds_bytes, s, NormBwdFlat(a, MODE))
  if (p.lpr == 16) HK_BWD_LANES(1, 16); else HK_BWD_LANES(1, 32);
#undef HK_BWD_LANES
}

template <typename T, int MODE>
static int launch_norm_bwd_any(const NormBwdArgs& a, const BwdPlan& p, hipStream_t s) {
  const dim3 grid{unsigned(p.grid)}, block{unsigned(p.block)};
#define HK_BWD_ANY_P(P, NV, F, X)                                                                                            \
  do {                                                                                                                    \
    if constexpr (X) HK_LAUNCH((norm_bwd_kernel<T, NV, MODE, P, false, F, X, 1024, false, false, false, true>), grid, block, p.lds_bytes, s, a); \
    else HK_LAUNCH((norm_bwd_kernel<T, NV, MODE, P, false, F, X, 1024, false, false, false, true>), grid, block, p.lds_bytes, s, NormBwdFlat(a, MODE)); \
  } while (0)
#define HK_BWD_ANY(NV, F) HK_BWD_ANY_P(1, NV, F, true)
  const bool extra = a.dx_in != nullptr || a.dres != nullptr || a.clamp_gamma != 0 || !NormBwdFlat::holds(a) ||
                     (MODE == BWD_RMS && a.part_dbeta != nullptr) || !a.stats_f32;
  profile_before(s);
  if constexpr (MODE != BWD_LN_MEMEFF) {
    if (!extra) {
      // two rows in flight where a workgroup holds few groups and is not full (16384 x 5001 bf16 LayerNorm 122 -> 109 us,
      // x 3001 66 -> 61); one otherwise (x 2047 46 against 50 us, 10000 x 8191 142 against 148, 8192 x 8191 fp32 150
      // against 190)
      if constexpr (VecIO<T>::N == 4) {
        if (p.nv == 2) HK_BWD_ANY_P(1, 2, true, false); else HK_BWD_ANY_P(1, 1, true, false);
      } else {
        if (p.tpr > 256 && p.tpr < 1024) HK_BWD_ANY_P(2, 1, true, false); else HK_BWD_ANY_P(1, 1, true, false);
      }
      profile_after(s);
      return launch_check("norm_bwd_kernel");
    }
  }
  if constexpr (VecIO<T>::N == 4) {
    if (p.nv == 2) HK_BWD_ANY(2, true); else HK_BWD_ANY(1, true);   // statistics "in the data type" are the same
  } else if constexpr (MODE == BWD_LN) {
    if (a.stats_f32) HK_BWD_ANY(1, true); else HK_BWD_ANY(1, false);
  } else {
    HK_BWD_ANY(1, true);
  }
#undef HK_BWD_ANY
#undef HK_BWD_ANY_P
  profile_after(s);
  return launch_check("norm_bwd_kernel");
}

template <typename T, int MODE>
static int launch_norm_bwd_nv(const NormBwdArgs& a, const BwdPlan& p, hipStream_t s) {
  int pf = tune_get(TUNE_NORM_BWD_PREFETCH);
  // Rows in flight per thread group, measured on the lean instances: at 512 threads per row (4096 bf16 columns,
  // RMSNorm, main kernel) depth 1 / 2 / 3 / 4 / 6 run 134.8 / 130.4 / 133.0 / 134.0 / 136.5 us; at 640 threads
  // (5120 columns, LayerNorm) depth 1 / 2 / 3 run 85.2 / 85.7 / 87.6 us and depths 4 and 6 collapse (252 / 371 us).
  // More bytes in flight than two rows of a 512-thread group (32 KB per compute unit) only lose, as they do for a
  // plain copy kernel; deeper instances than 2 are therefore not built.
  if (pf <= 0) pf = p.block <= 512 ? 2 : 1;
  // statistics in the data dtype only ever come with the plain LayerNorm backward
  if (!a.stats_f32 && MODE != BWD_LN) {
    set_last_error("norm_bwd: this mode keeps its statistics in float32");
    return HK_ERR_INVALID;
  }
  if constexpr (MODE != BWD_LN_MEMEFF) {
    if (p.lpr) {
      profile_before(s);
      if constexpr (MODE == BWD_LN) {
        if (a.clamp_gamma) launch_norm_bwd_lanes<T, MODE, true, 512>(a, p, s);
        else launch_norm_bwd_lanes<T, MODE, false, 512>(a, p, s);
      } else {
        launch_norm_bwd_lanes<T, MODE, false, 512>(a, p, s);
      }
      profile_after(s);
      return launch_check("norm_bwd_kernel");
    }
  }
  if (p.any) return launch_norm_bwd_any<T, MODE>(a, p, s);
  const int bound = bound_for(p.block);
  const bool have_kernel = p.nv == 1 || p.nv == 2 || (p.nv == 4 && VecIO<T>::N == 4);
  if (!have_kernel) {
    set_last_error("norm_bwd: no kernel for %d vectors per thread", p.nv);
    return HK_ERR_UNSUPPORTED;
  }
  // every argument check has passed: only now are the timing events of a measurement handed to the launch, so an
  // early return never leaves them for an unrelated launch to claim
  profile_before(s);
  int rc = HK_ERR_UNSUPPORTED;
  if (p.nv == 1) {
    if (bound == 512) rc = launch_norm_bwd_inst<T, MODE, 1, 512>(a, p, pf, s);
    else if (bound == 640) rc = launch_norm_bwd_inst<T, MODE, 1, 640>(a, p, pf, s);
    else if (bound == 768) rc = launch_norm_bwd_inst<T, MODE, 1, 768>(a, p, pf, s);
    else rc = launch_norm_bwd_inst<T, MODE, 1, 1024>(a, p, pf, s);
  } else if (p.nv == 2) {
    rc = launch_norm_bwd_inst<T, MODE, 2, 512>(a, p, pf, s);       // plans with nv > 1 stay within 512 threads
  } else if (p.nv == 4) {
    if constexpr (VecIO<T>::N == 4) rc = launch_norm_bwd_inst<T, MODE, 4, 512>(a, p, pf, s);
  }
  profile_after(s);
  if (rc != HK_OK) return rc;
  return launch_check("norm_bwd_kernel");
}

// norm_bwd_small_kernel where it measured faster: while its column sums take about one trip to memory.  Forward and backward, us,
// three launches / so, rows of whole vectors: 16 x 640 bf16 12.0 / 8.8, 512 x 4096 12.6 / 10.3 (LayerNorm 14.3 / 10.9), 768 x 2048 11.8
// / 11.1, x 4096 14.7 / 12.3, x 8192 20.6 / 16.5, fp32 30.1 / 27.9; 1024 x 512 bf16 11.9 / 9.4, x 2048 11.8 / 12.9, fp32 x 8192
// 36.2 / 37.7, 1536 x 640 bf16 11.9 / 13.0.  Of any boundary, whose columns are split into narrower tiles (4 / 8 vectors, 512 x 1021
// 10.3 / 10.6, 768 x 1021 12.2 / 14.0): 512 x 1021 bf16 12.4 / 10.3, x 8191 19.8 / 19.0, 256 x 8191 fp32 19.0 / 17.7, 640 x 1021
// bf16 12.5 / 12.2, 512 x 8191 fp32 25.2 / 28.6.
template <typename T, int MODE>
static bool launch_norm_bwd_small(NormBwdArgs a, const BwdPlan& p, void* dgamma, void* dbeta, hipStream_t s) {
  constexpr int VEC = VecIO<T>::N;
  const int64_t row_bytes = int64_t(a.cols) * int64_t(sizeof(T));
  const bool small = p.any ? a.rows <= 512 && a.rows * row_bytes <= (int64_t(8) << 20) : a.rows <= (row_bytes <= 1024 ? 1024 : 768);
  if (!small || p.lpr || p.nv > (VEC == 4 ? 2 : 1) || tune_get(TUNE_NORM_BWD_ROWS_PER_BLOCK) > 0 || tune_get(TUNE_NORM_BWD_BLOCKS) > 0 ||
      tune_get(TUNE_NORM_BWD_PREFETCH) > 0) return false;
  const auto rows_of = [&](const void* at, int64_t pitch) { return Span{at, ((a.rows - 1) * pitch + a.cols) * int64_t(sizeof(T))}; };
  const Span dy = rows_of(a.dy, a.dy_pitch), x = rows_of(a.x, a.x_pitch), dx = rows_of(a.dx, a.dx_pitch), gamma{a.gamma, row_bytes};
  const Span mean{a.mean, a.rows * int64_t(sizeof(float))}, stat{a.stat, mean.bytes}, dg{dgamma, row_bytes}, db{dbeta, row_bytes};
  // (what two launches write over each other, the column sums win)
  if (!apart({dx, dg, db}, {dy, x, gamma, mean, stat}) || !apart({dg, db}, {dx})) return false;
  const int nvec = (a.cols + VEC - 1) / VEC, lanes = small_lanes(p.any), rpb = kSmallThreads / p.tpr;
  a.tpr = p.tpr;
  a.threads = kSmallThreads;
  a.blocks = dgamma || dbeta ? (nvec + lanes - 1) / lanes : 0;
  a.part_dgamma = static_cast<float*>(dgamma);
  a.part_dbeta = static_cast<float*>(dbeta);
  const NormBwdFlat f(a, MODE);
  const dim3 grid{unsigned(a.blocks) + unsigned((a.rows + rpb - 1) / rpb)}, block{kSmallThreads};
  profile_before(s);
#define HK_BWD_SMALL(NV)                                                                              \
  do {                                                                                                \
    if (p.any) HK_LAUNCH((norm_bwd_small_kernel<T, NV, MODE, true>), grid, block, 0, s, f);           \
    else HK_LAUNCH((norm_bwd_small_kernel<T, NV, MODE, false>), grid, block, 0, s, f);                \
  } while (0)
  if (p.nv == 1) HK_BWD_SMALL(1);
  else if constexpr (VEC == 4) HK_BWD_SMALL(2);
#undef HK_BWD_SMALL
  profile_after(s);
  return true;
}

template <typename T>
int norm_bwd_typed(NormBwdArgs a, int mode, void* dgamma, void* dbeta, void* ws, size_t ws_bytes,
                   hipStream_t s) {
  constexpr int VEC = VecIO<T>::N;
  auto steps_ok = [](int64_t pitch, const LevelSteps& l) { return pitch % VEC == 0 && l.p1 % VEC == 0 && l.p2 % VEC == 0; };
  const bool aligned = aligned16(a.dy) && aligned16(a.x) && aligned16(a.dx) && aligned16(a.gamma) &&
                       aligned16(a.beta) && aligned16(a.dx_in) && aligned16(a.dres) &&
                       steps_ok(a.dy_pitch, a.dy_lv) && steps_ok(a.x_pitch, a.x_lv) && steps_ok(a.dx_pitch, a.dx_lv) &&
                       (!a.dx_in || steps_ok(a.dxin_pitch, a.dxin_lv)) && (!a.dres || steps_ok(a.dres_pitch, a.dres_lv));
  BwdPlan p = plan_norm_bwd<T>(a.rows, a.cols, aligned);
  const bool want_cols = dgamma != nullptr || dbeta != nullptr;
  // rows that once took no scratch do without it still
  if (p.any && want_cols && (ws == nullptr || ws_bytes < p.ws_bytes || !aligned16(ws))) p.reg_path = false;
  if (p.any && !a.stats_f32 && mode != BWD_LN) p.reg_path = false;
  const bool lean = p.reg_path && tune_get(TUNE_NORM_BWD_THREADS) <= 0 && mode != BWD_LN_MEMEFF && a.stats_f32 && !a.dx_in &&
                    !a.dres && NormBwdFlat::holds(a) && !(mode == BWD_RMS && (dbeta != nullptr || a.clamp_gamma));
  if (p.reg_path && tune_get(TUNE_NORM_BWD_THREADS) <= 0) {
    const BwdPlan q = lean ? plan_norm_bwd_lanes<T>(a.rows, a.cols) : BwdPlan{};
    // (a scratch that was sized for the other plans alone still serves them)
    if (q.reg_path && (!want_cols || (ws != nullptr && ws_bytes >= q.ws_bytes && aligned16(ws)))) p = q;
  }
  if (!p.reg_path) {
    HK_LAUNCH((norm_bwd_generic_dx_kernel<T, float>), dim3(unsigned(a.n0), unsigned(a.n1), unsigned(a.n2)), dim3(256),
              0, s, a, mode);
    int rc = launch_check("norm_bwd_generic_dx_kernel");
    if (rc != HK_OK) return rc;
    if (dgamma || dbeta) {
      HK_LAUNCH((norm_bwd_generic_cols_kernel<T, float>), dim3(unsigned((a.cols + 63) / 64)),
                         dim3(256), 0, s, a, mode, static_cast<T*>(dgamma), static_cast<T*>(dbeta));
      rc = launch_check("norm_bwd_generic_cols_kernel");
    }
    return rc;
  }
  a.nvec = (a.cols + VEC - 1) / VEC;
  a.part_pitch = a.nvec * VEC;
  if (want_cols) {
    HK_REQUIRE(ws != nullptr && ws_bytes >= p.ws_bytes, HK_ERR_WORKSPACE,
               "norm_bwd: workspace of %zu bytes needed, %zu given", p.ws_bytes, ws_bytes);
    HK_REQUIRE(aligned16(ws), HK_ERR_INVALID, "norm_bwd: workspace must be 16-byte aligned");
    a.part_dgamma = dgamma ? static_cast<float*>(ws) : nullptr;
    a.part_dbeta = dbeta ? static_cast<float*>(ws) + size_t(p.grid) * a.part_pitch : nullptr;
  } else {
    a.part_dgamma = nullptr;
    a.part_dbeta = nullptr;
  }
  if (lean && (mode == BWD_LN ? launch_norm_bwd_small<T, BWD_LN>(a, p, dgamma, dbeta, s)
                              : launch_norm_bwd_small<T, BWD_RMS>(a, p, dgamma, dbeta, s)))
    return launch_check("norm_bwd_small_kernel");
  a.tpr = p.tpr;
  a.threads = uint16_t(p.block);
  a.blocks = p.grid;
  {
    // the walking kernel's row stride, split over the walk levels (used by the instances with a running walk index)
    const uint64_t stride = uint64_t(p.grid) * uint64_t(p.rpb);
    const uint64_t q = stride / uint64_t(a.n0);
    a.ws0 = uint32_t(stride - q * uint64_t(a.n0));
    a.ws1 = uint32_t(q % uint64_t(a.n1));
    a.ws2 = uint32_t(q / uint64_t(a.n1));
  }
  int rc;
  switch (mode) {
    case BWD_LN: rc = launch_norm_bwd_nv<T, BWD_LN>(a, p, s); break;
    case BWD_RMS: rc = launch_norm_bwd_nv<T, BWD_RMS>(a, p, s); break;
    default: rc = launch_norm_bwd_nv<T, BWD_LN_MEMEFF>(a, p, s); break;
  }
  if (rc != HK_OK || !want_cols) return rc;
  const bool both = dgamma != nullptr && dbeta != nullptr;
  auto fold = [&](auto kernel, int lanes) {
    HK_LAUNCH(kernel, dim3(unsigned((a.part_pitch + 4 * lanes - 1) / (4 * lanes)), both ? 2 : 1), dim3(unsigned(fold_threads(lanes))), 0, s,
              dgamma ? a.part_dgamma : a.part_dbeta, a.part_dbeta, static_cast<T*>(dgamma ? dgamma : dbeta), static_cast<T*>(dbeta),
              p.grid, a.cols, a.part_pitch);
  };
  if (fold_lanes(a.part_pitch, both ? 2 : 1) == 8) fold(norm_bwd_finalize_kernel<T, 8>, 8);
  else fold(norm_bwd_finalize_kernel<T, 32>, 32);
  return launch_check("norm_bwd_finalize_kernel");
}

} // namespace hk
