// Varlen RMSNorm / LayerNorm, forward and backward, for gfx950.
//
// Norms act per token row, so the packed (rows, dim) buffer is processed
// with no reference to the offsets (the reference's kernels ignore them too,
// src/scree/kernels/triton/varlen_rmsnorm.py:7-8).
//
// Fast path: one wavefront per row.  Each lane keeps CHUNKS 16-byte vectors
// of the row in registers (dim = CHUNKS * 64 lanes * 16 bytes at most), so x
// is read from HBM exactly once; the reductions are wave-wide shuffles.  Rows
// of at most 128 vectors take 4 to 64 lanes each (short rows, below).
// Rows that are not whole vectors, and unaligned buffers, run the same kernels
// with element-aligned vectors (odd widths, below).  Generic path (rows shorter
// than one vector or longer than the fast path holds): one wavefront per row
// looping over the columns.
//
// Backward (norm_bwd_cols): each thread of a block (or, at up to 256 vectors
// per row, of a team of waves in it) owns fixed 16-byte column vectors across
// the block's rows, so the parameter gradients accumulate in
// its fp32 registers; the row statistics are reduced across the block through
// LDS, dx is written per row, and each block writes one partial row of
// parameter gradients, which a column-sum kernel adds in a fixed order.  No
// atomics: results are bit-identical from run to run.
#include <algorithm>
#include <initializer_list>
#include <type_traits>

#include "common.h"

namespace scree {
namespace {

constexpr int kWave = 64;
constexpr int kFwdWaves = 4;       // rows (waves) per forward block
constexpr int kMaxParts = 512;     // partial rows of a backward, at most
constexpr int kMaxChunks = 16;     // 16-byte vectors per lane on the fast path

// --------------------------------------------------------------- odd widths
// ODD kernels take rows that are not whole 16-byte vectors, or buffers that are
// not 16-byte aligned: vectors are read and written at element alignment (the
// hardware takes any, and a row's unaligned vectors still cover whole cache
// lines between them), and the last vector of a row is moved back to end with
// it.  Its first `dup` elements are then also the previous vector's: both lanes
// compute and store the same values, and only the sums leave them out.
// Scalar loops over the columns, which these replace, were bound by the issue
// of 2-byte loads.  RMSNorm / LayerNorm / add+RMSNorm, us, before -> now:
// 12,160 x 1,001 bf16 forward 27/39/36 -> 11/13/20, backward 90/91/100 ->
// 22/26/26; 12,160 x 4,095 bf16 forward 137/195/184 -> 37/45/70, backward
// 269/271/351 -> 61/71/83; 1,000 x 130 fp16 backward 15/16/15 -> 7/8/7.
typedef unsigned int u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef unsigned int u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
template <typename T, bool ODD>
struct RowVec {
  static constexpr int VEC = 16 / sizeof(T);
  typedef typename std::conditional<sizeof(T) == 2, u32x4_a2, u32x4_a4>::type u32x4e;
  int nvec, dim;
  __device__ __forceinline__ explicit RowVec(int d) : nvec(ODD ? (d + VEC - 1) / VEC : d / VEC), dim(d) {}
  // column of vector v's first element, and how many of its elements repeat
  __device__ __forceinline__ int col(int v) const { return ODD ? min(v * VEC, dim - VEC) : v * VEC; }
  __device__ __forceinline__ int dup(int v) const { return ODD && v == nvec - 1 ? nvec * VEC - dim : 0; }
  static __device__ __forceinline__ bool counts(int e, int dup) { return !ODD || e >= dup; }
  static __device__ __forceinline__ uint4 ld(const T* p) {
    if constexpr (!ODD) return ld16(p);
    const u32x4e v = *reinterpret_cast<const u32x4e*>(p);
    return make_uint4(v.x, v.y, v.z, v.w);
  }
  static __device__ __forceinline__ uint4 ld_nt(const T* p) {
    if constexpr (!ODD) return ld16_nt(p);
    const u32x4e v = __builtin_nontemporal_load(reinterpret_cast<const u32x4e*>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
  }
  static __device__ __forceinline__ void st_nt(T* p, const uint4& v) {
    if constexpr (!ODD) {
      st16_nt(p, v);
    } else {
      const u32x4e u = {v.x, v.y, v.z, v.w};
      __builtin_nontemporal_store(u, reinterpret_cast<u32x4e*>(p));
    }
  }
  // For rows past 128 vectors: a wide odd row's vectors straddle cache lines
  // that the next instruction completes, which plain stores leave in L2 until
  // then (add+RMSNorm, 12,160 x 4,095 bf16: 70 us against 85 nontemporal; on
  // rows of 770 nontemporal is the faster, 10.3 against 12.0 for LayerNorm).
  static __device__ __forceinline__ void st_wide(T* p, const uint4& v) {
    if constexpr (!ODD) {
      st16_nt(p, v);
    } else {
      const u32x4e u = {v.x, v.y, v.z, v.w};
      *reinterpret_cast<u32x4e*>(p) = u;
    }
  }
};

// ------------------------------------------------------------------ forward
// RES (RMSNorm only): the normalised row is h = x + res, rounded to T as a
// separate addition would round it; h is written out and normalised.
template <int WAVES>
constexpr int fwd_threads() { return WAVES * kWave; }
// LayerNorm's workgroups are kLnWaves rows (waves) that stage the weight and
// bias rows in LDS once; RMSNorm's are kFwdWaves rows with the weights in
// registers.
constexpr int kLnWaves = 8;
template <bool LAYER>
constexpr int fwd_waves() { return LAYER ? kLnWaves : kFwdWaves; }

template <typename T, int CHUNKS, bool LAYER, bool RES, bool ODD>
__global__ __launch_bounds__(fwd_threads<fwd_waves<LAYER>()>()) void norm_fwd_vec(
    const T* __restrict__ x, const T* __restrict__ res, const T* __restrict__ w,
    const T* __restrict__ b, T* __restrict__ hout, T* __restrict__ y,
    float* __restrict__ mean_out, float* __restrict__ rstd_out, int64_t rows, int dim, float eps) {
  constexpr int VEC = 16 / sizeof(T);
  constexpr int WAVES = fwd_waves<LAYER>();
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t row = (int64_t)blockIdx.x * WAVES + (threadIdx.x / kWave);
  const bool live = row < rows;
  typedef RowVec<T, ODD> RV;
  const RV rv(dim);
  const int nvec = rv.nvec;
  const T* xr = x + row * (int64_t)dim;
  uint4 v[CHUNKS];
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int vi = c * kWave + lane;
    v[c] = live && vi < nvec ? RV::ld_nt(xr + rv.col(vi)) : make_uint4(0, 0, 0, 0);
  }
  // LayerNorm: the block copies the weight and bias rows into LDS while its
  // rows load (one L2 read per block instead of per row, and off the
  // registers); the output reads them from there.
  constexpr int NMAX = LAYER ? CHUNKS * kWave * VEC : 1;
  __shared__ __align__(16) T wb[2 * NMAX];
  if constexpr (LAYER) {
    for (int vi = threadIdx.x; vi < nvec; vi += WAVES * kWave) {
      *reinterpret_cast<uint4*>(wb + vi * VEC) = w ? RV::ld(w + rv.col(vi)) : make_uint4(0, 0, 0, 0);
      *reinterpret_cast<uint4*>(wb + NMAX + vi * VEC) = b ? RV::ld(b + rv.col(vi)) : make_uint4(0, 0, 0, 0);
    }
    __syncthreads();
  }
  if (!live) return;
  // RMSNorm loads its weight vectors with the row, so their (L2) latency
  // overlaps the row's instead of following the reduction.
  constexpr bool kEarlyW = !LAYER;
  uint4 wvs[kEarlyW ? CHUNKS : 1];
  if constexpr (kEarlyW) {
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const int vi = c * kWave + lane;
      wvs[c] = (w && vi < nvec) ? RV::ld(w + rv.col(vi)) : make_uint4(0, 0, 0, 0);
    }
  }
  if (RES) {
    const T* rr = res + row * (int64_t)dim;
    T* hr = hout + row * (int64_t)dim;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const int vi = c * kWave + lane;
      if (vi < nvec) {
        const uint4 av = RV::ld_nt(rr + rv.col(vi));
        float f[VEC];
#pragma unroll
        for (int e = 0; e < VEC; ++e) f[e] = elem<T>(v[c], e) + elem<T>(av, e);
        v[c] = pack16<T>(f);
        RV::st_wide(hr + rv.col(vi), v[c]);
      }
    }
  }
  const float fdim = (float)dim;
  float mu = 0.f, rstd;
  if (LAYER) {
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const int dup = rv.dup(c * kWave + lane);
#pragma unroll
      for (int e = 0; e < VEC; ++e) s += RV::counts(e, dup) ? elem<T>(v[c], e) : 0.f;
    }
    mu = wave_sum(s) / fdim;
    float s2 = 0.f;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      if (c * kWave + lane < nvec) {
        const int dup = rv.dup(c * kWave + lane);
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          const float d = RV::counts(e, dup) ? elem<T>(v[c], e) - mu : 0.f;
          s2 = __builtin_fmaf(d, d, s2);
        }
      }
    }
    rstd = 1.0f / sqrtf(wave_sum(s2) / fdim + eps);
  } else {
    // Explicit fused multiply-adds fix the rounding of every step, so the
    // add + RMSNorm and the plain RMSNorm instantiations (where the compiler
    // could contract a*a + b*b either way) give identical statistics.
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const int dup = rv.dup(c * kWave + lane);
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        const float t = RV::counts(e, dup) ? elem<T>(v[c], e) : 0.f;
        s = __builtin_fmaf(t, t, s);
      }
    }
    rstd = 1.0f / sqrtf(wave_sum(s) / fdim + eps);
  }
  T* yr = y + row * (int64_t)dim;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int vi = c * kWave + lane;
    if (vi < nvec) {
      uint4 wv = make_uint4(0, 0, 0, 0), bv = make_uint4(0, 0, 0, 0);
      if constexpr (kEarlyW) {
        wv = wvs[c];
      } else {
        wv = *reinterpret_cast<const uint4*>(wb + vi * VEC);
        bv = *reinterpret_cast<const uint4*>(wb + NMAX + vi * VEC);
      }
      float f[VEC];
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        float t = LAYER ? (elem<T>(v[c], e) - mu) * rstd : elem<T>(v[c], e) * rstd;
        if (w) t *= elem<T>(wv, e);
        if (LAYER && b) t += elem<T>(bv, e);
        f[e] = t;
      }
      RV::st_wide(yr + rv.col(vi), pack16<T>(f));
    }
  }
  if (lane == 0) {
    if (rstd_out) rstd_out[row] = rstd;
    if (LAYER && mean_out) mean_out[row] = mu;
  }
}

// ------------------------------------------------------------- short rows
// Rows of at most 128 16-byte vectors (1,024 columns in 16 bits, 512 in fp32).
// A wave-per-row or block-per-row kernel leaves most of its lanes
// without a column there: at 128 bf16 columns 16 of a wave's 64, and 16 of the
// 512 threads of norm_bwd_cols.  Here LPR lanes (a power of two) hold a row,
// CH vectors each, so a wave holds 64 / LPR rows; the host picks the pair that
// covers the row with the fewest idle lanes (short_shape).  Row sums are DPP
// and permlane steps within the LPR lanes: no LDS, no barrier.  Bound by HBM
// on large inputs.  Measured (us, forward RMS / LN / add, backward RMS / LN /
// add; the wave-per-row and norm_bwd_cols kernels before):
//   194,560 x 128 bf16  44/61/72, 246/301/462 -> 19/21/36, 32/33/38
//   100,000 x 32 fp32   20/27/28,  88/108/206 ->  6/7/11,  12/13/14
//   12,160 x 768 fp16    9/12/15,   25/32/40  ->  8/8/14,  18/20/20
//   12,160 x 1,024 bf16 11/13/19,   27/31/42  -> 11/12/18, 20/22/23
// From 129 to 256 vectors a row the backward's norm_bwd_cols takes several
// rows per block instead (teams of waves): 12,160 x 1,536 bf16 30/35/46 ->
// 26/29/34, x 2,048 34/39/50 -> 31/34/40.
//
// Sum over the two 32-lane halves, and over the two 16-lane rows of each half,
// in every lane: the permlane swaps exchange halves (rows) of two copies, so
// one holds the lower and the other the upper value.  (Written out: the
// builtin folds two equal inputs into one result.)
__device__ __forceinline__ float halves_sum(float x) {
  float lo = x, hi = x;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(lo), "+v"(hi));
  return lo + hi;
}
__device__ __forceinline__ float rows_sum(float x) {
  float lo = x, hi = x;
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(lo), "+v"(hi));
  return lo + hi;
}
template <int LPR>
__device__ __forceinline__ float group_sum(float v) {
  static_assert(LPR >= 4 && LPR <= 64 && (LPR & (LPR - 1)) == 0, "LPR: a power of two, 4 to 64");
  auto dpp = [](float x, auto ctrl) {
    return x + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                   0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, false));
  };
  v = dpp(v, std::integral_constant<int, 0xB1>{});                             // lane ^ 1
  v = dpp(v, std::integral_constant<int, 0x4E>{});                             // lane ^ 2
  if constexpr (LPR >= 8) v = dpp(v, std::integral_constant<int, 0x141>{});   // across 4 (half mirror)
  if constexpr (LPR >= 16) v = dpp(v, std::integral_constant<int, 0x140>{});  // across 8 (mirror)
  if constexpr (LPR >= 32) v = rows_sum(v);
  if constexpr (LPR >= 64) v = halves_sum(v);
  return v;
}
// The converse: the sum of lane l of every LPR-lane group of the wave.
template <int LPR>
__device__ __forceinline__ float subgroups_sum(float v) {
  auto dpp = [](float x, auto ctrl) {
    return x + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                   0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, false));
  };
  if constexpr (LPR <= 4) v = dpp(v, std::integral_constant<int, 0x124>{});  // rotate by 4 in the row
  if constexpr (LPR <= 8) v = dpp(v, std::integral_constant<int, 0x128>{});  // by 8
  if constexpr (LPR <= 16) v = rows_sum(v);
  if constexpr (LPR <= 32) v = halves_sum(v);
  return v;
}
// Row groups a wave of the forward loads before it reduces any, in launches
// that still give every CU two workgroups; below that one group per wave (613
// x 192 bf16: 4.2 us with four groups, 3.4 with one; 12,160 x 768 fp16: 7.5 us
// with two, 8.0 with one).
template <int CH>
constexpr int short_groups() {
  return CH == 1 ? 4 : 2;
}

template <typename T, int LPR, int CH, int G, bool LAYER, bool RES, bool ODD>
__global__ __launch_bounds__(kFwdWaves* kWave) void norm_fwd_short(
    const T* __restrict__ x, const T* __restrict__ res, const T* __restrict__ w,
    const T* __restrict__ b, T* __restrict__ hout, T* __restrict__ y,
    float* __restrict__ mean_out, float* __restrict__ rstd_out, int64_t rows, int dim, float eps) {
  constexpr int VEC = 16 / sizeof(T), RPW = kWave / LPR;
  const int lane = threadIdx.x & (kWave - 1), l = lane % LPR;
  typedef RowVec<T, ODD> RV;
  const RV rv(dim);
  // consecutive waves take consecutive row groups, a workgroup G strips of them
  const int64_t first = ((int64_t)blockIdx.x * G * kFwdWaves + threadIdx.x / kWave) * RPW + lane / LPR;
  uint4 v[G][CH], av[RES ? G : 1][CH], wv[CH], bv[LAYER ? CH : 1];
  bool own[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) own[c] = c * LPR + l < rv.nvec;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int64_t row = first + g * kFwdWaves * RPW;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int64_t off = row * dim + rv.col(c * LPR + l);
      const bool ok = own[c] && row < rows;
      v[g][c] = ok ? RV::ld_nt(x + off) : make_uint4(0, 0, 0, 0);
      if (RES) av[g][c] = ok ? RV::ld_nt(res + off) : make_uint4(0, 0, 0, 0);
    }
  }
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int off = rv.col(c * LPR + l);
    wv[c] = (w && own[c]) ? RV::ld(w + off) : make_uint4(0, 0, 0, 0);
    if (LAYER) bv[c] = (b && own[c]) ? RV::ld(b + off) : make_uint4(0, 0, 0, 0);
  }
  const float fdim = (float)dim;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int64_t row = first + g * kFwdWaves * RPW;
    const bool live = row < rows;
    if (RES) {
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        float f[VEC];
#pragma unroll
        for (int e = 0; e < VEC; ++e) f[e] = elem<T>(v[g][c], e) + elem<T>(av[g][c], e);
        v[g][c] = pack16<T>(f);
        if (live && own[c]) RV::st_nt(hout + row * dim + rv.col(c * LPR + l), v[g][c]);
      }
    }
    float mu = 0.f, s = 0.f;
    if (LAYER) {
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const int dup = rv.dup(c * LPR + l);
#pragma unroll
        for (int e = 0; e < VEC; ++e) s += RV::counts(e, dup) ? elem<T>(v[g][c], e) : 0.f;
      }
      mu = group_sum<LPR>(s) / fdim;
      s = 0.f;
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      if (LAYER && !own[c]) continue;
      const int dup = rv.dup(c * LPR + l);
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        float d = LAYER ? elem<T>(v[g][c], e) - mu : elem<T>(v[g][c], e);
        if (!RV::counts(e, dup)) d = 0.f;
        s = __builtin_fmaf(d, d, s);
      }
    }
    const float rstd = 1.0f / sqrtf(group_sum<LPR>(s) / fdim + eps);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      float f[VEC];
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        float t = LAYER ? (elem<T>(v[g][c], e) - mu) * rstd : elem<T>(v[g][c], e) * rstd;
        if (w) t *= elem<T>(wv[c], e);
        if (LAYER && b) t += elem<T>(bv[c], e);
        f[e] = t;
      }
      if (live && own[c]) RV::st_nt(y + row * dim + rv.col(c * LPR + l), pack16<T>(f));
    }
    if (live && l == 0) {
      if (rstd_out) rstd_out[row] = rstd;
      if (LAYER && mean_out) mean_out[row] = mu;
    }
  }
}

template <typename T, bool LAYER, bool RES>
__global__ __launch_bounds__(kFwdWaves* kWave) void norm_fwd_generic(
    const T* __restrict__ x, const T* __restrict__ res, const T* __restrict__ w,
    const T* __restrict__ b, T* __restrict__ hout, T* __restrict__ y,
    float* __restrict__ mean_out, float* __restrict__ rstd_out, int64_t rows, int dim, float eps) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t row = (int64_t)blockIdx.x * kFwdWaves + (threadIdx.x / kWave);
  if (row >= rows) return;
  const T* xr = x + row * (int64_t)dim;
  const T* rr = RES ? res + row * (int64_t)dim : nullptr;
  // Element j of the normalised row: x, or h = x + res rounded to T (each
  // pass recomputes it rather than reading back the h it stores).
  auto at = [&](int j) -> float {
    return RES ? to_f32(from_f32<T>(to_f32(xr[j]) + to_f32(rr[j]))) : to_f32(xr[j]);
  };
  const float fdim = (float)dim;
  float mu = 0.f, rstd;
  if (LAYER) {
    float s = 0.f;
    for (int j = lane; j < dim; j += kWave) s += at(j);
    mu = wave_sum(s) / fdim;
    float s2 = 0.f;
    for (int j = lane; j < dim; j += kWave) {
      const float d = at(j) - mu;
      s2 = __builtin_fmaf(d, d, s2);
    }
    rstd = 1.0f / sqrtf(wave_sum(s2) / fdim + eps);
  } else {
    float s = 0.f;
    for (int j = lane; j < dim; j += kWave) {
      const float t = at(j);
      s = __builtin_fmaf(t, t, s);
    }
    rstd = 1.0f / sqrtf(wave_sum(s) / fdim + eps);
  }
  T* yr = y + row * (int64_t)dim;
  T* hr = RES ? hout + row * (int64_t)dim : nullptr;
  for (int j = lane; j < dim; j += kWave) {
    const float hj = at(j);
    if (RES) hr[j] = from_f32<T>(hj);
    float t = LAYER ? (hj - mu) * rstd : hj * rstd;
    if (w) t *= to_f32(w[j]);
    if (LAYER && b) t += to_f32(b[j]);
    yr[j] = from_f32<T>(t);
  }
  if (lane == 0) {
    if (rstd_out) rstd_out[row] = rstd;
    if (LAYER && mean_out) mean_out[row] = mu;
  }
}

// ----------------------------------------------------------------- backward
// Column-ownership layout.  A block of kBwdThreads threads takes every
// G-th step of R rows (G = grid size: block b takes rows b*R .. b*R+R-1,
// then those G*R rows further on, ...), so at any moment the grid works on
// one contiguous stretch of G*R rows and its reads and writes spread over
// all HBM channels; a contiguous range of rows per block put the blocks'
// concurrent streams ~40 rows apart at config 2 and ran ~10 % slower.  Thread
// t owns the 16-byte column vectors t + k*kBwdThreads (k < CPT) of every row
// the block takes.  Per step of R rows the thread loads its
// vectors of x and dy, the row statistics (sum x*g for RMS; sum g and
// sum g*xhat for LN) are reduced across the wave by shuffles and across the
// block through a double-buffered LDS array (one barrier per step), then the
// thread writes dx for its vectors and adds its parameter gradients into
// fp32 registers.  At the end each thread writes its own columns of the
// block's partial row: no intra-block reduction, and the partial rows are
// summed by norm_param_colsum in a fixed order.
// partial layout: [part][param][dim] fp32, param 0 = dweight, 1 = dbias.
constexpr int kBwdThreads = 512;
constexpr int kBwdWarps = kBwdThreads / kWave;

// LayerNorm's x-hat = (x - mean) * rstd of one row as one FMA.  The rounding of
// mean * rstd is then in every x-hat of the row, and with row means of 10 and
// more standard deviations it is the largest error of dx and dweight (1.2 times
// that of a subtraction and a product, which the column loops used).  ODD rows
// add it back; whole vectors keep the single FMA (12,160 x 768 fp16, backward:
// 19.3 us, 20.3 with the second operation).
template <bool ODD>
struct XHat {
  float rstd, off, lo;
  __device__ __forceinline__ XHat(float mean, float rs) : rstd(rs), off(-mean * rs), lo(ODD ? fmaf(-mean, rs, mean * rs) : 0.f) {}
  __device__ __forceinline__ float operator()(float x) const {
    const float h = fmaf(x, rstd, off);
    return ODD ? h + lo : h;
  }
};

// One step's rows: this thread's 16-byte vectors of x, dy (and dres) for R
// rows, with the rows' statistics.  The kernel keeps two of these and loads
// the next step's rows while it reduces and writes the current one.
template <typename T, int CPT, int R, int TEAM, bool LAYER, bool RES, bool ODD>
struct BwdRows {
  uint4 xv[R][CPT], gv[R][CPT], hv[RES ? R : 1][CPT];
  float rs[R], mu[R];

  __device__ __forceinline__ void load(const T* __restrict__ x, const T* __restrict__ dy,
                                       const T* __restrict__ dres,
                                       const float* __restrict__ mean_in,
                                       const float* __restrict__ rstd_in, const bool* own,
                                       int64_t rb, int64_t r1, int dim, const int (&cols)[CPT]) {
    typedef RowVec<T, ODD> RV;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int64_t row = rb + r;
      const bool ok = row < r1;
      rs[r] = ok ? rstd_in[row] : 0.f;
      mu[r] = (LAYER && ok) ? mean_in[row] : 0.f;
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        const int64_t off = row * (int64_t)dim + cols[k];
        xv[r][k] = (ok && own[k]) ? RV::ld_nt(x + off) : make_uint4(0, 0, 0, 0);
        gv[r][k] = (ok && own[k]) ? RV::ld_nt(dy + off) : make_uint4(0, 0, 0, 0);
        if (RES) hv[r][k] = (ok && own[k]) ? RV::ld_nt(dres + off) : make_uint4(0, 0, 0, 0);
      }
    }
  }
};

// The rows of one step: row sums reduced across the wave by shuffles and
// across the block through red[buf] (one barrier), then dx written and the
// parameter gradients accumulated in aw / ab.  `wf` holds this thread's
// weights as fp32 (ones without a weight).  Per row, x-hat = x * rstd - mean
// * rstd is one FMA and the output folds its row constants into two more:
//   LayerNorm  dx = rstd * g - rstd*b * x-hat - rstd*a,  a = mean(g), b = mean(g * x-hat)
//   RMSNorm    dx = rstd * g - k * x,                    k = rstd^3 * mean(g * x)
// with g = dy * w (reference varlen_layernorm.py:64-74, varlen_rmsnorm.py:58-65).
template <typename T, int CPT, int R, int TEAM, bool LAYER, bool RES, bool ODD>
__device__ __forceinline__ void norm_bwd_step(BwdRows<T, CPT, R, TEAM, LAYER, RES, ODD>& st,
                                              float (&red)[2][R][2][TEAM / kWave], int buf,
                                              const float (&wf)[CPT][16 / sizeof(T)],
                                              const bool* own, const int (&cols)[CPT],
                                              const int (&dups)[CPT],
                                              float (&aw)[CPT][16 / sizeof(T)],
                                              float (&ab)[LAYER ? CPT : 1][16 / sizeof(T)],
                                              T* __restrict__ dx, int64_t rb, int64_t r1, int dim,
                                              float inv_dim, int tid) {
  constexpr int VEC = 16 / sizeof(T);
  const int lane = tid & (kWave - 1), wave = tid / kWave;
  float s1[R], s2[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    s1[r] = 0.f;
    s2[r] = 0.f;
    const XHat<ODD> xhat(st.mu[r], st.rs[r]);
#pragma unroll
    for (int k = 0; k < CPT; ++k)
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        const float xx = elem<T>(st.xv[r][k], e);
        float g = elem<T>(st.gv[r][k], e) * wf[k][e];
        if (!RowVec<T, ODD>::counts(e, dups[k])) g = 0.f;
        if (LAYER) {
          s1[r] += g;
          s2[r] = fmaf(g, xhat(xx), s2[r]);
        } else {
          s1[r] = fmaf(xx, g, s1[r]);
        }
      }
    s1[r] = wave_sum_last(s1[r]);
    if (LAYER) s2[r] = wave_sum_last(s2[r]);
  }
  if (lane == kWave - 1) {  // the wave's sums are complete in its last lane
#pragma unroll
    for (int r = 0; r < R; ++r) {
      red[buf][r][0][wave] = s1[r];
      red[buf][r][1][wave] = s2[r];
    }
  }
  __syncthreads();
  // Keep the rows packed across the barrier: re-derive the fp32 values
  // below instead of holding the converted floats live.
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      asm volatile("" : "+v"(st.xv[r][k].x), "+v"(st.xv[r][k].y), "+v"(st.xv[r][k].z), "+v"(st.xv[r][k].w));
      asm volatile("" : "+v"(st.gv[r][k].x), "+v"(st.gv[r][k].y), "+v"(st.gv[r][k].z), "+v"(st.gv[r][k].w));
      if (RES)
        asm volatile("" : "+v"(st.hv[RES ? r : 0][k].x), "+v"(st.hv[RES ? r : 0][k].y),
                     "+v"(st.hv[RES ? r : 0][k].z), "+v"(st.hv[RES ? r : 0][k].w));
    }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    float t1 = 0.f, t2 = 0.f;
#pragma unroll
    for (int q = 0; q < TEAM / kWave; ++q) {
      t1 += red[buf][r][0][q];
      if (LAYER) t2 += red[buf][r][1][q];
    }
    const int64_t row = rb + r;
    if (row >= r1) continue;
    const float rr = st.rs[r];
    // LayerNorm: c1 = -rstd * mean(g), c2 = -rstd * mean(g * x-hat);
    // RMSNorm: c2 = -rstd^3 * mean(g * x).
    const XHat<ODD> xhat(st.mu[r], rr);
    const float c1 = -rr * (t1 * inv_dim);
    const float c2 = LAYER ? -rr * (t2 * inv_dim) : -(rr * rr * rr) * (t1 * inv_dim);
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      if (!own[k]) continue;
      float f[VEC];
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        const float xx = elem<T>(st.xv[r][k], e);
        const float d = elem<T>(st.gv[r][k], e);
        const float g = d * wf[k][e];
        if (LAYER) {
          const float xh = xhat(xx);
          f[e] = fmaf(rr, g, fmaf(c2, xh, c1));
          aw[k][e] = fmaf(d, xh, aw[k][e]);
          ab[LAYER ? k : 0][e] += d;
        } else {
          f[e] = fmaf(rr, g, c2 * xx);
          aw[k][e] = fmaf(d * rr, xx, aw[k][e]);
        }
        if (RES) f[e] += elem<T>(st.hv[RES ? r : 0][k], e);
      }
      RowVec<T, ODD>::st_wide(dx + row * (int64_t)dim + cols[k], pack16<T>(f));
    }
  }
}

// RES: dx also receives dres (the gradient reaching the normalised input by
// another path, e.g. the residual stream of an add + RMSNorm).
template <typename T, int CPT, int R, int TW, int TEAMS, bool LAYER, bool RES, bool ODD>
__global__ __launch_bounds__(TW* TEAMS* kWave) void norm_bwd_cols(
    const T* __restrict__ dy, const T* __restrict__ x, const T* __restrict__ w,
    const float* __restrict__ mean_in, const float* __restrict__ rstd_in,
    const T* __restrict__ dres, T* __restrict__ dx, float* __restrict__ partial, int64_t rows,
    int dim, int nparam) {
  constexpr int VEC = 16 / sizeof(T);
  constexpr int TEAM = TW * kWave;
  __shared__ float red[TEAMS][2][R][2][TW];
  // (a team is whole waves: its index, and with it every row's address, is scalar)
  const int team = TEAMS > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / TEAM) : 0;
  const int tid = (int)threadIdx.x - team * TEAM;
  typedef RowVec<T, ODD> RV;
  const RV rv(dim);

  float wf[CPT][VEC];  // this thread's weights as fp32, ones without a weight
  bool own[CPT];
  int cols[CPT], dups[CPT];  // first column of each vector, and its repeated elements (ODD)
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int v = tid + k * TEAM;
    own[k] = v < rv.nvec;
    cols[k] = rv.col(v);
    dups[k] = rv.dup(v);
    const uint4 wv = (w && own[k]) ? RV::ld(w + cols[k]) : make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < VEC; ++e) wf[k][e] = w ? elem<T>(wv, e) : 1.0f;
  }
  float aw[CPT][VEC], ab[LAYER ? CPT : 1][VEC];
#pragma unroll
  for (int k = 0; k < CPT; ++k)
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      aw[k][e] = 0.f;
      ab[LAYER ? k : 0][e] = 0.f;
    }

  // Two row sets: while one step reduces and writes, the next step's rows
  // load.  Steps are S rows apart; rows past the end load as zeros and are
  // not written.
  BwdRows<T, CPT, R, TEAM, LAYER, RES, ODD> A, B;
  const float inv_dim = 1.0f / (float)dim;
  // (with several teams every one runs the block's count of steps: they share
  // the steps' barriers; rows past the end load as zeros)
  const int64_t S = (int64_t)gridDim.x * TEAMS * R;
  const int64_t lead = (int64_t)blockIdx.x * TEAMS * R;  // the block's first row
  const int64_t first = lead + team * R, lag = first - lead;
  if (lead < rows) A.load(x, dy, dres, mean_in, rstd_in, own, first, rows, dim, cols);
  for (int64_t rb = first; rb - lag < rows; rb += 2 * S) {
    if (rb - lag + S < rows) B.load(x, dy, dres, mean_in, rstd_in, own, rb + S, rows, dim, cols);
    norm_bwd_step<T, CPT, R, TEAM, LAYER, RES, ODD>(A, red[team], 0, wf, own, cols, dups, aw, ab, dx, rb, rows, dim, inv_dim, tid);
    if (rb - lag + S >= rows) break;
    if (rb - lag + 2 * S < rows) A.load(x, dy, dres, mean_in, rstd_in, own, rb + 2 * S, rows, dim, cols);
    norm_bwd_step<T, CPT, R, TEAM, LAYER, RES, ODD>(B, red[team], 1, wf, own, cols, dups, aw, ab, dx, rb + S, rows, dim, inv_dim, tid);
  }
  __shared__ __align__(16) float tsum[TEAMS > 1 ? TEAMS - 1 : 1][TEAMS > 1 ? CPT * TEAM * VEC : 1];
  auto write = [&](int p, auto& acc) {
    float* out = partial + ((int64_t)blockIdx.x * nparam + p) * dim;
    if constexpr (TEAMS > 1) {  // the other teams' sums, added in team order
      __syncthreads();
      if (team > 0) {
#pragma unroll
        for (int k = 0; k < CPT; ++k)
#pragma unroll
          for (int e = 0; e < VEC; ++e) tsum[team - 1][(tid + k * TEAM) * VEC + e] = acc[k][e];
      }
      __syncthreads();
      if (team > 0) return;
#pragma unroll
      for (int t = 0; t < TEAMS - 1; ++t)
#pragma unroll
        for (int k = 0; k < CPT; ++k)
#pragma unroll
          for (int e = 0; e < VEC; ++e) acc[k][e] += tsum[t][(tid + k * TEAM) * VEC + e];
    }
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      if (!own[k]) continue;
      float* o = out + cols[k];
      if constexpr (ODD) {
#pragma unroll
        for (int e = 0; e < VEC; ++e)
          if (RV::counts(e, dups[k])) o[e] = acc[k][e];
        continue;
      }
#pragma unroll
      for (int e = 0; e < VEC; e += 4)
        *reinterpret_cast<float4*>(o + e) = make_float4(acc[k][e], acc[k][e + 1], acc[k][e + 2], acc[k][e + 3]);
    }
  };
  if (nparam > 0) write(0, aw);
  if constexpr (LAYER) {
    if (nparam > 1) write(1, ab);
  }
}

// Short rows (see norm_fwd_short).  A lane keeps its columns' parameter sums in
// registers over every row it takes; at the end the wave's row groups are
// summed by lane exchanges and the block's waves through LDS, in a fixed
// order, into the block's partial row.  Blocks take interleaved row groups as
// in norm_bwd_cols; the next group loads during the current one where both fit
// 128 registers (CH == 1), else four waves per SIMD cover the loads.
template <typename T, int LPR, int CH, bool LAYER, bool RES, bool ODD>
struct ShortRows {
  uint4 xv[CH], gv[CH], hv[CH];
  float rs, mu;
  __device__ __forceinline__ void load(const T* __restrict__ x, const T* __restrict__ dy,
                                       const T* __restrict__ dres,
                                       const float* __restrict__ mean_in,
                                       const float* __restrict__ rstd_in, const bool (&own)[CH],
                                       int64_t row, int64_t rows, const RowVec<T, ODD>& rv, int l) {
    typedef RowVec<T, ODD> RV;
    const bool ok = row < rows;
    rs = ok ? rstd_in[row] : 0.f;
    mu = (LAYER && ok) ? mean_in[row] : 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int64_t off = row * rv.dim + rv.col(c * LPR + l);
      xv[c] = (ok && own[c]) ? RV::ld_nt(x + off) : make_uint4(0, 0, 0, 0);
      gv[c] = (ok && own[c]) ? RV::ld_nt(dy + off) : make_uint4(0, 0, 0, 0);
      if (RES) hv[c] = (ok && own[c]) ? RV::ld_nt(dres + off) : make_uint4(0, 0, 0, 0);
    }
  }
};
// An empty asm over a packed vector: the compiler unpacks it again after it
// instead of holding the converted floats.
__device__ __forceinline__ void repack(uint4& v) {
  asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w));
}
// One step's rows; arithmetic per row as in norm_bwd_step.
template <typename T, int LPR, int CH, bool LAYER, bool RES, bool ODD>
__device__ __forceinline__ void norm_bwd_short_step(
    ShortRows<T, LPR, CH, LAYER, RES, ODD>& st, uint4 (&wv)[CH], bool has_w, const bool (&own)[CH],
    float (&aw)[CH][16 / sizeof(T)], float (&ab)[LAYER ? CH : 1][16 / sizeof(T)],
    T* __restrict__ dx, int64_t row, int64_t rows, const RowVec<T, ODD>& rv, float inv_dim, int l) {
  constexpr int VEC = 16 / sizeof(T);
  const float rr = st.rs;
  const XHat<ODD> xhat(st.mu, rr);
  float s1 = 0.f, s2 = 0.f;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    repack(wv[c]);
    const int dup = rv.dup(c * LPR + l);
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const float xx = elem<T>(st.xv[c], e);
      const float d = elem<T>(st.gv[c], e);
      float g = has_w ? d * elem<T>(wv[c], e) : d;
      if (!RowVec<T, ODD>::counts(e, dup)) g = 0.f;
      if (LAYER) {
        s1 += g;
        s2 = fmaf(g, xhat(xx), s2);
      } else {
        s1 = fmaf(xx, g, s1);
      }
    }
  }
  s1 = group_sum<LPR>(s1);
  if (LAYER) s2 = group_sum<LPR>(s2);
  const float c1 = -rr * (s1 * inv_dim);
  const float c2 = LAYER ? -rr * (s2 * inv_dim) : -(rr * rr * rr) * (s1 * inv_dim);
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    repack(st.xv[c]);
    repack(st.gv[c]);
    repack(wv[c]);
    float f[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const float xx = elem<T>(st.xv[c], e);
      const float d = elem<T>(st.gv[c], e);
      const float g = has_w ? d * elem<T>(wv[c], e) : d;
      if (LAYER) {
        const float xh = xhat(xx);
        f[e] = fmaf(rr, g, fmaf(c2, xh, c1));
        aw[c][e] = fmaf(d, xh, aw[c][e]);
        ab[LAYER ? c : 0][e] += d;
      } else {
        f[e] = fmaf(rr, g, c2 * xx);
        aw[c][e] = fmaf(d * rr, xx, aw[c][e]);
      }
      if (RES) f[e] += elem<T>(st.hv[c], e);
    }
    if (row < rows && own[c]) RowVec<T, ODD>::st_nt(dx + row * rv.dim + rv.col(c * LPR + l), pack16<T>(f));
  }
}
template <typename T, int LPR, int CH, bool LAYER, bool RES, bool ODD>
__global__ __launch_bounds__(kBwdThreads, 4) void norm_bwd_short(
    const T* __restrict__ dy, const T* __restrict__ x, const T* __restrict__ w,
    const float* __restrict__ mean_in, const float* __restrict__ rstd_in,
    const T* __restrict__ dres, T* __restrict__ dx, float* __restrict__ partial, int64_t rows,
    int dim, int nparam) {
  constexpr int VEC = 16 / sizeof(T), RPW = kWave / LPR;
  constexpr int RPB = kBwdWarps * RPW;  // rows of the block per step
  __shared__ __align__(16) float sums[kBwdWarps][LPR * CH * VEC];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, l = lane % LPR;
  typedef RowVec<T, ODD> RV;
  const RV rv(dim);
  bool own[CH];
  uint4 wv[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    own[c] = c * LPR + l < rv.nvec;
    wv[c] = (w && own[c]) ? RV::ld(w + rv.col(c * LPR + l)) : make_uint4(0, 0, 0, 0);
  }
  float aw[CH][VEC], ab[LAYER ? CH : 1][VEC];
#pragma unroll
  for (int c = 0; c < CH; ++c)
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      aw[c][e] = 0.f;
      ab[LAYER ? c : 0][e] = 0.f;
    }
  const float inv_dim = 1.0f / (float)dim;
  const int64_t S = (int64_t)gridDim.x * RPB;
  int64_t row = (int64_t)blockIdx.x * RPB + wave * RPW + lane / LPR;
  ShortRows<T, LPR, CH, LAYER, RES, ODD> A;
  auto load = [&](ShortRows<T, LPR, CH, LAYER, RES, ODD>& st, int64_t r) {
    st.load(x, dy, dres, mean_in, rstd_in, own, r, rows, rv, l);
  };
  auto step = [&](ShortRows<T, LPR, CH, LAYER, RES, ODD>& st, int64_t r) {
    norm_bwd_short_step<T, LPR, CH, LAYER, RES, ODD>(st, wv, w != nullptr, own, aw, ab, dx, r, rows, rv,
                                                inv_dim, l);
  };
  // (the loops' condition is uniform over the wave: its first row)
  if constexpr (CH == 1) {
    ShortRows<T, LPR, CH, LAYER, RES, ODD> B;
    load(A, row);
    for (; row - lane / LPR < rows; row += 2 * S) {
      load(B, row + S);
      step(A, row);
      load(A, row + 2 * S);
      step(B, row + S);
    }
  } else {
#pragma unroll 1
    for (; row - lane / LPR < rows; row += S) {
      load(A, row);
      step(A, row);
    }
  }
  // (one call per array: a choice between them by p would keep both in memory)
  auto write = [&](int p, const auto& acc) {
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        const float t = subgroups_sum<LPR>(acc[c][e]);
        const int v = c * LPR + l;
        if (lane < LPR && v < rv.nvec && RV::counts(e, rv.dup(v))) sums[wave][rv.col(v) + e] = t;
      }
    __syncthreads();
    float* out = partial + ((int64_t)blockIdx.x * nparam + p) * dim;
    for (int i = threadIdx.x; i < dim; i += kBwdThreads) {
      float t = sums[0][i];
#pragma unroll
      for (int q = 1; q < kBwdWarps; ++q) t += sums[q][i];
      out[i] = t;
    }
  };
  if (nparam > 0) write(0, aw);
  if constexpr (LAYER) {
    if (nparam > 1) {
      __syncthreads();
      write(1, ab);
    }
  }
}

template <typename T, bool LAYER, bool RES>
__global__ __launch_bounds__(kFwdWaves* kWave) void norm_bwd_dx_generic(
    const T* __restrict__ dy, const T* __restrict__ x, const T* __restrict__ w,
    const float* __restrict__ mean_in, const float* __restrict__ rstd_in,
    const T* __restrict__ dres, T* __restrict__ dx, int64_t rows, int dim) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t row = (int64_t)blockIdx.x * kFwdWaves + (threadIdx.x / kWave);
  if (row >= rows) return;
  const T* xr = x + row * (int64_t)dim;
  const T* gr = dy + row * (int64_t)dim;
  const float r = rstd_in[row];
  const float mu = LAYER ? mean_in[row] : 0.f;
  const float fdim = (float)dim;
  float s1 = 0.f, s2 = 0.f;
  for (int j = lane; j < dim; j += kWave) {
    const float xx = to_f32(xr[j]);
    const float d = to_f32(gr[j]);
    const float g = w ? d * to_f32(w[j]) : d;
    if (LAYER) {
      s1 += g;
      s2 += g * ((xx - mu) * r);
    } else {
      s1 += xx * g;
    }
  }
  s1 = wave_sum(s1);
  if (LAYER) s2 = wave_sum(s2);
  const float k_rms = r * r * r * s1 / fdim;
  const float a_ln = s1 / fdim;
  const float b_ln = s2 / fdim;
  T* dxr = dx + row * (int64_t)dim;
  for (int j = lane; j < dim; j += kWave) {
    const float xx = to_f32(xr[j]);
    const float d = to_f32(gr[j]);
    const float g = w ? d * to_f32(w[j]) : d;
    float v = LAYER ? r * (g - a_ln - ((xx - mu) * r) * b_ln) : r * g - k_rms * xx;
    if (RES) v += to_f32(dres[row * (int64_t)dim + j]);
    dxr[j] = from_f32<T>(v);
  }
}

// grid (ceil(dim/256), nparts): thread owns one column, sums rows part, part+nparts, ...
template <typename T, bool LAYER>
__global__ __launch_bounds__(256) void norm_bwd_param_generic(
    const T* __restrict__ dy, const T* __restrict__ x, const float* __restrict__ mean_in,
    const float* __restrict__ rstd_in, float* __restrict__ partial, int64_t rows, int dim,
    int nparam) {
  const int col = blockIdx.x * 256 + threadIdx.x;
  const int part = blockIdx.y;
  const int nparts = gridDim.y;
  if (col >= dim) return;
  float aw = 0.f, ab = 0.f;
  for (int64_t row = part; row < rows; row += nparts) {
    const float xx = to_f32(x[row * (int64_t)dim + col]);
    const float d = to_f32(dy[row * (int64_t)dim + col]);
    const float r = rstd_in[row];
    if (LAYER) {
      aw += d * ((xx - mean_in[row]) * r);
      ab += d;
    } else {
      aw += d * xx * r;
    }
  }
  float* out = partial + (int64_t)part * nparam * dim;
  out[col] = aw;
  if (nparam > 1) out[dim + col] = ab;
}

// Column sums of the partial rows; output cast to out_dtype.
__device__ __forceinline__ void store_param(void* out, int col, float t, int out_dtype) {
  if (out_dtype == SCREE_DTYPE_F32) static_cast<float*>(out)[col] = t;
  else if (out_dtype == SCREE_DTYPE_F16) static_cast<f16*>(out)[col] = (f16)t;
  else static_cast<bf16*>(out)[col] = (bf16)t;
}

// Any dim: 16 columns x 16 row groups per block, every load in flight at once,
// then a fixed-order tree over the row groups in LDS.
__global__ __launch_bounds__(256) void norm_param_colsum(const float* __restrict__ partial,
                                                         int nparts, int nparam, int dim,
                                                         void* out0, void* out1, int out_dtype) {
  __shared__ float red[16][16];
  const int cq = threadIdx.x & 15, rg = threadIdx.x >> 4;
  const int col = blockIdx.x * 16 + cq;
  const int p = blockIdx.y;
  constexpr int kIt = kMaxParts / 16;
  float v[kIt];
#pragma unroll
  for (int j = 0; j < kIt; ++j) {
    const int i = rg + 16 * j;
    v[j] = (col < dim && i < nparts) ? partial[((int64_t)i * nparam + p) * dim + col] : 0.f;
  }
  float s = v[0];
#pragma unroll
  for (int j = 1; j < kIt; ++j) s += v[j];
  red[rg][cq] = s;
  __syncthreads();
  for (int st = 8; st >= 1; st >>= 1) {
    if (rg < st) red[rg][cq] += red[rg + st][cq];
    __syncthreads();
  }
  void* out = p == 0 ? out0 : out1;
  if (rg == 0 && col < dim && out) store_param(out, col, red[0][cq], out_dtype);
}

// Vector form (dim % 4 == 0): 16 columns x 64 row groups per block, 16-byte
// loads, then a fixed-order tree over the row groups in LDS (deterministic).
__global__ __launch_bounds__(256) void norm_param_colsum4(const float* __restrict__ partial,
                                                          int nparts, int nparam, int dim,
                                                          void* out0, void* out1, int out_dtype) {
  __shared__ float4 red[64][4];
  const int cq = threadIdx.x & 3, rg = threadIdx.x >> 2;
  // A block reads a 64-byte strip of each partial row; block b runs on XCD
  // b mod 8, so neighbouring strips (one 128-byte line) go to blocks of the
  // same XCD, whose L2 then fetches the line once instead of once per XCD.
  int slab = blockIdx.x;
  if ((gridDim.x & 7) == 0) slab = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int col = slab * 16 + cq * 4;
  const int p = blockIdx.y;
  // Every load in flight at once (at most kMaxParts / 64 per thread), then
  // the sum in row order.
  constexpr int kIt = kMaxParts / 64;
  float4 v[kIt];
#pragma unroll
  for (int j = 0; j < kIt; ++j) {
    const int i = rg + 64 * j;
    v[j] = (col < dim && i < nparts)
               ? *reinterpret_cast<const float4*>(partial + ((int64_t)i * nparam + p) * dim + col)
               : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  float4 s = v[0];
#pragma unroll
  for (int j = 1; j < kIt; ++j) {
    s.x += v[j].x; s.y += v[j].y; s.z += v[j].z; s.w += v[j].w;
  }
  red[rg][cq] = s;
  __syncthreads();
  for (int st = 32; st >= 1; st >>= 1) {
    if (rg < st) {
      const float4 o = red[rg + st][cq];
      float4 m = red[rg][cq];
      m.x += o.x; m.y += o.y; m.z += o.z; m.w += o.w;
      red[rg][cq] = m;
    }
    __syncthreads();
  }
  void* out = p == 0 ? out0 : out1;
  if (rg == 0 && col < dim && out) {
    const float4 t = red[0][cq];
    store_param(out, col + 0, t.x, out_dtype);
    store_param(out, col + 1, t.y, out_dtype);
    store_param(out, col + 2, t.z, out_dtype);
    store_param(out, col + 3, t.w, out_dtype);
  }
}

// --------------------------------------------------------------------- host
inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

inline int chunks_for(int nvec) {
  int need = (nvec + kWave - 1) / kWave;
  int c = 1;
  while (c < need) c <<= 1;
  return c;
}

inline int nparts_for(int64_t rows) {
  int64_t p = (rows + 7) / 8;
  if (p < 1) p = 1;
  if (p > kMaxParts) p = kMaxParts;
  return (int)p;
}

// How the vector kernels take rows of `dim` columns in these buffers: not at
// all (rows shorter than a vector, or of more than max_vecs), as whole aligned
// vectors, or as ODD ones.
enum class RowForm { kNone, kAligned, kOdd };
template <typename T>
RowForm row_form(int64_t dim, int64_t max_vecs, std::initializer_list<const void*> ptrs) {
  constexpr int VEC = 16 / sizeof(T);
  if (dim < VEC || (dim + VEC - 1) / VEC > max_vecs) return RowForm::kNone;
  if (dim % VEC) return RowForm::kOdd;
  for (const void* p : ptrs)
    if (p && !aligned16(p)) return RowForm::kOdd;
  return RowForm::kAligned;
}
constexpr int64_t kMaxFwdVecs = (int64_t)kMaxChunks * kWave;
constexpr int64_t kMaxBwdVecs = 2 * (int64_t)kBwdThreads;  // two per thread of a 512-thread block

// Lanes per row and vectors per lane of the short-row kernels: the pair that
// covers nvec vectors with the fewest idle lanes, {0, 0} past their range.
struct ShortShape {
  int lpr, ch;
};
inline ShortShape short_shape(int64_t nvec, bool thirds) {
  static const ShortShape kShapes[] = {{4, 1},  {8, 1},  {16, 1}, {32, 1},
                                       {16, 3}, {64, 1}, {32, 3}, {64, 2}};  // by size
  for (const ShortShape& s : kShapes)
    if (nvec <= s.lpr * s.ch && (thirds || s.ch != 3)) return s;
  return ShortShape{0, 0};
}
#define SCREE_SHORT_CASES(CASE) \
  CASE(4, 1)                    \
  CASE(8, 1)                    \
  CASE(16, 1)                   \
  CASE(32, 1)                   \
  CASE(16, 3)                   \
  CASE(64, 1)                   \
  CASE(32, 3)                   \
  CASE(64, 2)

// The vector kernels (rows of whole 16-byte vectors, or ODD).
template <typename T, bool LAYER, bool RES, bool ODD>
void launch_fwd_vec(const T* xp, const T* rp, const T* wp, const T* bp, T* hp, T* yp, float* mean,
                    float* rstd, int64_t rows, int64_t dim, float eps, hipStream_t stream) {
  const dim3 block(kFwdWaves * kWave);
  const int d = (int)dim;
  constexpr int64_t VEC = 16 / sizeof(T);
  const int64_t nvec = (dim + VEC - 1) / VEC;
  const ShortShape sh = short_shape(nvec, true);
  if (sh.ch) {
#define SCREE_FWD_SHORT_G(L, C, G)                                                                 \
  hipLaunchKernelGGL((norm_fwd_short<T, L, C, G, LAYER, RES, ODD>),                                     \
                   dim3((unsigned)((rows + per * G - 1) / (per * G))), block, 0, stream, xp, rp, \
                   wp, bp, hp, yp, mean, rstd, rows, d, eps)
#define SCREE_FWD_SHORT(L, C)                                                                      \
  if (sh.lpr == L && sh.ch == C) {                                                                 \
    constexpr int64_t per = (int64_t)kFwdWaves * (kWave / L);                                      \
    if (rows >= per * short_groups<C>() * 512)                                                     \
      SCREE_FWD_SHORT_G(L, C, short_groups<C>());                                                  \
    else                                                                                           \
      SCREE_FWD_SHORT_G(L, C, 1);                                                                  \
    return;                                                                                        \
  }
    SCREE_SHORT_CASES(SCREE_FWD_SHORT)
#undef SCREE_FWD_SHORT
#undef SCREE_FWD_SHORT_G
  }
  constexpr int W = fwd_waves<LAYER>();
  const dim3 vgrid((unsigned)((rows + W - 1) / W)), vblock(W * kWave);
  const int chunks = chunks_for((int)nvec);
#define SCREE_FWD_CASE(C)                                                                      \
  case C:                                                                                      \
  hipLaunchKernelGGL((norm_fwd_vec<T, C, LAYER, RES, ODD>), vgrid, vblock, 0, stream, xp, rp, wp, bp, \
                     hp, yp, mean, rstd, rows, d, eps);                                      \
  break;
  switch (chunks) {
    SCREE_FWD_CASE(4)
    SCREE_FWD_CASE(8)
    SCREE_FWD_CASE(16)
    default: break;  // chunks_for never exceeds kMaxChunks on the fast path
  }
#undef SCREE_FWD_CASE
}

// res / h non-null (RMSNorm only): normalise h = x + res and write h too.
template <typename T, bool LAYER, bool RES>
void launch_fwd_k(const T* xp, const T* rp, const T* wp, const T* bp, T* hp, T* yp, float* mean,
                  float* rstd, int64_t rows, int64_t dim, float eps, hipStream_t stream) {
  switch (row_form<T>(dim, kMaxFwdVecs, {xp, rp, wp, bp, hp, yp})) {
    case RowForm::kAligned:
      return launch_fwd_vec<T, LAYER, RES, false>(xp, rp, wp, bp, hp, yp, mean, rstd, rows, dim, eps, stream);
    case RowForm::kOdd:
      return launch_fwd_vec<T, LAYER, RES, true>(xp, rp, wp, bp, hp, yp, mean, rstd, rows, dim, eps, stream);
    case RowForm::kNone: break;
  }
  const dim3 grid((unsigned)((rows + kFwdWaves - 1) / kFwdWaves)), block(kFwdWaves * kWave);
  hipLaunchKernelGGL((norm_fwd_generic<T, LAYER, RES>), grid, block, 0, stream, xp, rp, wp, bp, hp, yp,
                     mean, rstd, rows, (int)dim, eps);
}

template <typename T, bool LAYER>
int launch_fwd(const void* x, const void* res, const void* w, const void* b, void* h, void* y,
               float* mean, float* rstd, int64_t rows, int64_t dim, float eps,
               hipStream_t stream) {
  const T* xp = static_cast<const T*>(x);
  const T* rp = static_cast<const T*>(res);
  const T* wp = static_cast<const T*>(w);
  const T* bp = static_cast<const T*>(b);
  T* hp = static_cast<T*>(h);
  T* yp = static_cast<T*>(y);
  if constexpr (!LAYER) {
    if (res) {
      launch_fwd_k<T, false, true>(xp, rp, wp, bp, hp, yp, mean, rstd, rows, dim, eps, stream);
      return check_launch("scree_add_rmsnorm_fwd");
    }
  }
  launch_fwd_k<T, LAYER, false>(xp, nullptr, wp, bp, nullptr, yp, mean, rstd, rows, dim, eps,
                                stream);
  return check_launch(LAYER ? "scree_layernorm_fwd" : "scree_rmsnorm_fwd");
}

// The vector kernels (rows of whole 16-byte vectors, or ODD); returns the
// number of partial rows written, at most `nparts`.
template <typename T, bool LAYER, bool RES, bool ODD>
int launch_bwd_vec(const T* dyp, const T* xp, const T* wp, const float* mean, const float* rstd,
                   const T* dresp, T* dxp, float* partial, bool want_params, int nparts,
                   int64_t rows, int64_t dim, hipStream_t stream) {
  const int d = (int)dim;
  const int nparam = LAYER ? 2 : 1;
  constexpr int VEC = 16 / sizeof(T);
  const int nvec = (int)((dim + VEC - 1) / VEC);
  const int cpt = (nvec + kBwdThreads - 1) / kBwdThreads;  // 1 or 2
  const dim3 grid((unsigned)nparts), block(kBwdThreads);
  const int np = want_params ? nparam : 0;
  // (three vectors per lane would spill with two sums each, or as ODD ones with a residual)
  constexpr bool kThirds = !LAYER && !(RES && ODD);
  const ShortShape sh = short_shape(nvec, kThirds);
  if (sh.ch) {
#define SCREE_BWD_SHORT(L, C)                                                                       \
  if constexpr (C != 3 || kThirds) {                                                                \
    if (sh.lpr == L && sh.ch == C) {                                                                \
      constexpr int64_t per = (int64_t)kBwdWarps * (kWave / L);                                     \
      nparts = (int)std::min<int64_t>(nparts, std::max<int64_t>(1, (rows + per - 1) / per));        \
      hipLaunchKernelGGL((norm_bwd_short<T, L, C, LAYER, RES, ODD>), dim3((unsigned)nparts), block, \
                         0, stream, dyp, xp, wp, mean, rstd, dresp, dxp, partial, rows, d, np);     \
      return nparts;                                                                                \
    }                                                                                               \
  }
    SCREE_SHORT_CASES(SCREE_BWD_SHORT)
#undef SCREE_BWD_SHORT
  }
  // rows per step: two steps' rows (double-buffered) fit 4 waves per SIMD
  // (LN keeps two sums per row; the residual gradient is one more vector).
  // At one vector per thread 2 rows per step measured best for all three
  // (RMSNorm at config 2: R = 1, 2, 3, 4 -> 90.8, 87.3, 89.1, 90.5 us).
  constexpr int R1 = 2;
  constexpr int R2 = (LAYER || RES) ? 1 : 2;
#define SCREE_BWD_COLS(CPT, R, TW, TEAMS)                                                          \
  hipLaunchKernelGGL((norm_bwd_cols<T, CPT, R, TW, TEAMS, LAYER, RES, ODD>), grid,                      \
                   dim3(TW * TEAMS * kWave), 0, stream, dyp, xp, wp, mean, rstd, dresp, dxp,     \
                   partial, rows, d, np)
  if (nvec <= 3 * kWave)
    SCREE_BWD_COLS(1, R1, 3, 2);
  else if (nvec <= 4 * kWave)
    SCREE_BWD_COLS(1, R1, 4, 2);
  else if (cpt == 1)
    SCREE_BWD_COLS(1, R1, kBwdWarps, 1);
  else
    SCREE_BWD_COLS(2, R2, kBwdWarps, 1);
#undef SCREE_BWD_COLS
  return nparts;
}

// dres non-null (RMSNorm only): dx also receives dres.  Returns the number of
// partial rows written, at most `nparts`.
template <typename T, bool LAYER, bool RES>
int launch_bwd_k(const T* dyp, const T* xp, const T* wp, const float* mean, const float* rstd,
                 const T* dresp, T* dxp, float* partial, bool want_params, int nparts,
                 int64_t rows, int64_t dim, hipStream_t stream) {
  switch (row_form<T>(dim, kMaxBwdVecs, {dyp, xp, wp, dresp, dxp})) {
    case RowForm::kAligned: return launch_bwd_vec<T, LAYER, RES, false>(dyp, xp, wp, mean, rstd, dresp, dxp, partial, want_params, nparts, rows, dim, stream);
    case RowForm::kOdd: return launch_bwd_vec<T, LAYER, RES, true>(dyp, xp, wp, mean, rstd, dresp, dxp, partial, want_params, nparts, rows, dim, stream);
    case RowForm::kNone: break;
  }
  const int d = (int)dim;
  const int nparam = LAYER ? 2 : 1;
  const dim3 grid((unsigned)((rows + kFwdWaves - 1) / kFwdWaves)), block(kFwdWaves * kWave);
  if (rows > 0)
    hipLaunchKernelGGL((norm_bwd_dx_generic<T, LAYER, RES>), grid, block, 0, stream, dyp, xp, wp,
                       mean, rstd, dresp, dxp, rows, d);
  if (want_params) {
    const dim3 pgrid((unsigned)((dim + 255) / 256), (unsigned)nparts);
    hipLaunchKernelGGL((norm_bwd_param_generic<T, LAYER>), pgrid, dim3(256), 0, stream, dyp, xp,
                       mean, rstd, partial, rows, d, nparam);
  }
  return nparts;
}

template <typename T, bool LAYER>
int launch_bwd(const void* dy, const void* x, const void* w, const float* mean, const float* rstd,
               const void* dres, void* dx, void* dw, void* db, int dparam_dtype, int64_t rows,
               int64_t dim, void* workspace, hipStream_t stream) {
  const T* dyp = static_cast<const T*>(dy);
  const T* xp = static_cast<const T*>(x);
  const T* wp = static_cast<const T*>(w);
  const T* dresp = static_cast<const T*>(dres);
  T* dxp = static_cast<T*>(dx);
  const int d = (int)dim;
  const int nparam = LAYER ? 2 : 1;
  const bool want_params = (dw != nullptr) || (db != nullptr);
  int nparts = nparts_for(rows);
  float* partial = static_cast<float*>(workspace);
  const char* fn = LAYER ? "scree_layernorm_bwd" : (dres ? "scree_add_rmsnorm_bwd" : "scree_rmsnorm_bwd");
  bool done = false;
  if constexpr (!LAYER) {
    if (dres) {
      nparts = launch_bwd_k<T, false, true>(dyp, xp, wp, mean, rstd, dresp, dxp, partial,
                                            want_params, nparts, rows, dim, stream);
      done = true;
    }
  }
  if (!done)
    nparts = launch_bwd_k<T, LAYER, false>(dyp, xp, wp, mean, rstd, nullptr, dxp, partial,
                                           want_params, nparts, rows, dim, stream);
  int rc = check_launch(fn);
  if (rc != SCREE_OK || !want_params) return rc;
  if (dim % 4 == 0) {
    const dim3 cgrid((unsigned)((dim + 15) / 16), (unsigned)nparam);
    hipLaunchKernelGGL(norm_param_colsum4, cgrid, dim3(256), 0, stream, partial, nparts, nparam, d,
                       dw, db, dparam_dtype);
  } else {
    const dim3 cgrid((unsigned)((dim + 15) / 16), (unsigned)nparam);
    hipLaunchKernelGGL(norm_param_colsum, cgrid, dim3(256), 0, stream, partial, nparts, nparam, d,
                       dw, db, dparam_dtype);
  }
  return check_launch(fn);
}

int validate_common(const char* fn, int64_t rows, int64_t dim, int dtype) {
  if (rows < 0 || rows >= ((int64_t)1 << 31))
    return set_error(SCREE_ERR_INVALID, "%s: rows must be in [0, 2^31), got %lld", fn, (long long)rows);
  if (dim < 1 || dim > (1 << 24))
    return set_error(SCREE_ERR_INVALID, "%s: dim must be in [1, 2^24], got %lld", fn, (long long)dim);
  if (dtype != SCREE_DTYPE_F32 && dtype != SCREE_DTYPE_F16 && dtype != SCREE_DTYPE_BF16)
    return set_error(SCREE_ERR_UNSUPPORTED, "%s: unknown dtype code %d", fn, dtype);
  if (rows * dim >= ((int64_t)1 << 40))
    return set_error(SCREE_ERR_INVALID, "%s: tensor too large", fn);
  return SCREE_OK;
}

}  // namespace
}  // namespace scree

using namespace scree;

extern "C" size_t scree_norm_bwd_workspace_bytes(int64_t rows, int64_t dim) {
  if (rows < 0 || dim < 1) return 0;
  return (size_t)nparts_for(rows) * 2u * (size_t)dim * sizeof(float);
}

extern "C" int scree_rmsnorm_fwd(const void* x, const void* weight, void* y, float* rstd,
                                 int64_t rows, int64_t dim, float eps, int dtype, void* stream) {
  const char* fn = "scree_rmsnorm_fwd";
  int rc = validate_common(fn, rows, dim, dtype);
  if (rc) return rc;
  if (rows == 0) return SCREE_OK;
  if (!x || !y) return set_error(SCREE_ERR_INVALID, "%s: x and y must be non-null", fn);
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case SCREE_DTYPE_F32: return launch_fwd<float, false>(x, nullptr, weight, nullptr, nullptr, y, nullptr, rstd, rows, dim, eps, s);
    case SCREE_DTYPE_F16: return launch_fwd<f16, false>(x, nullptr, weight, nullptr, nullptr, y, nullptr, rstd, rows, dim, eps, s);
    default: return launch_fwd<bf16, false>(x, nullptr, weight, nullptr, nullptr, y, nullptr, rstd, rows, dim, eps, s);
  }
}

extern "C" int scree_layernorm_fwd(const void* x, const void* weight, const void* bias, void* y,
                                   float* mean, float* rstd, int64_t rows, int64_t dim, float eps,
                                   int dtype, void* stream) {
  const char* fn = "scree_layernorm_fwd";
  int rc = validate_common(fn, rows, dim, dtype);
  if (rc) return rc;
  if (rows == 0) return SCREE_OK;
  if (!x || !y) return set_error(SCREE_ERR_INVALID, "%s: x and y must be non-null", fn);
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case SCREE_DTYPE_F32: return launch_fwd<float, true>(x, nullptr, weight, bias, nullptr, y, mean, rstd, rows, dim, eps, s);
    case SCREE_DTYPE_F16: return launch_fwd<f16, true>(x, nullptr, weight, bias, nullptr, y, mean, rstd, rows, dim, eps, s);
    default: return launch_fwd<bf16, true>(x, nullptr, weight, bias, nullptr, y, mean, rstd, rows, dim, eps, s);
  }
}

static int validate_bwd(const char* fn, const void* dy, const void* x, const float* rstd, void* dx,
                        bool want_params, int dparam_dtype, int64_t rows, int64_t dim,
                        void* workspace, size_t workspace_bytes) {
  // with no rows, empty row tensors may have no storage: only the parameter
  // gradients (sums over no rows: zeros) are written
  if (rows > 0 && (!dy || !x || !rstd || !dx))
    return set_error(SCREE_ERR_INVALID, "%s: dy, x, rstd and dx must be non-null", fn);
  if (want_params) {
    if (dparam_dtype != SCREE_DTYPE_F32 && dparam_dtype != SCREE_DTYPE_F16 &&
        dparam_dtype != SCREE_DTYPE_BF16)
      return set_error(SCREE_ERR_UNSUPPORTED, "%s: unknown parameter dtype code %d", fn, dparam_dtype);
    const size_t need = scree_norm_bwd_workspace_bytes(rows, dim);
    if (!workspace || workspace_bytes < need)
      return set_error(SCREE_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, got %zu", fn, need,
                       workspace ? workspace_bytes : (size_t)0);
  }
  return SCREE_OK;
}

extern "C" int scree_rmsnorm_bwd(const void* dy, const void* x, const void* weight,
                                 const float* rstd, void* dx, void* dweight, int dparam_dtype,
                                 int64_t rows, int64_t dim, int dtype, void* workspace,
                                 size_t workspace_bytes, void* stream) {
  const char* fn = "scree_rmsnorm_bwd";
  int rc = validate_common(fn, rows, dim, dtype);
  if (rc) return rc;
  if (dweight && !weight) return set_error(SCREE_ERR_INVALID, "%s: dweight requires weight", fn);
  if (rows == 0 && !dweight) return SCREE_OK;  // nothing to write; empty dweight is summed to 0 below
  rc = validate_bwd(fn, dy, x, rstd, dx, dweight != nullptr, dparam_dtype, rows, dim, workspace,
                    workspace_bytes);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case SCREE_DTYPE_F32: return launch_bwd<float, false>(dy, x, weight, nullptr, rstd, nullptr, dx, dweight, nullptr, dparam_dtype, rows, dim, workspace, s);
    case SCREE_DTYPE_F16: return launch_bwd<f16, false>(dy, x, weight, nullptr, rstd, nullptr, dx, dweight, nullptr, dparam_dtype, rows, dim, workspace, s);
    default: return launch_bwd<bf16, false>(dy, x, weight, nullptr, rstd, nullptr, dx, dweight, nullptr, dparam_dtype, rows, dim, workspace, s);
  }
}

extern "C" int scree_layernorm_bwd(const void* dy, const void* x, const void* weight,
                                   const float* mean, const float* rstd, void* dx, void* dweight,
                                   void* dbias, int dparam_dtype, int64_t rows, int64_t dim,
                                   int dtype, void* workspace, size_t workspace_bytes,
                                   void* stream) {
  const char* fn = "scree_layernorm_bwd";
  int rc = validate_common(fn, rows, dim, dtype);
  if (rc) return rc;
  if (dweight && !weight) return set_error(SCREE_ERR_INVALID, "%s: dweight requires weight", fn);
  if (rows == 0 && !dweight && !dbias) return SCREE_OK;
  if (rows > 0 && !mean) return set_error(SCREE_ERR_INVALID, "%s: mean must be non-null", fn);
  rc = validate_bwd(fn, dy, x, rstd, dx, dweight != nullptr || dbias != nullptr, dparam_dtype, rows,
                    dim, workspace, workspace_bytes);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case SCREE_DTYPE_F32: return launch_bwd<float, true>(dy, x, weight, mean, rstd, nullptr, dx, dweight, dbias, dparam_dtype, rows, dim, workspace, s);
    case SCREE_DTYPE_F16: return launch_bwd<f16, true>(dy, x, weight, mean, rstd, nullptr, dx, dweight, dbias, dparam_dtype, rows, dim, workspace, s);
    default: return launch_bwd<bf16, true>(dy, x, weight, mean, rstd, nullptr, dx, dweight, dbias, dparam_dtype, rows, dim, workspace, s);
  }
}

extern "C" int scree_add_rmsnorm_fwd(const void* x, const void* residual, const void* weight,
                                     void* h, void* y, float* rstd, int64_t rows, int64_t dim,
                                     float eps, int dtype, void* stream) {
  const char* fn = "scree_add_rmsnorm_fwd";
  int rc = validate_common(fn, rows, dim, dtype);
  if (rc) return rc;
  if (rows == 0) return SCREE_OK;
  if (!x || !residual || !h || !y)
    return set_error(SCREE_ERR_INVALID, "%s: x, residual, h and y must be non-null", fn);
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case SCREE_DTYPE_F32: return launch_fwd<float, false>(x, residual, weight, nullptr, h, y, nullptr, rstd, rows, dim, eps, s);
    case SCREE_DTYPE_F16: return launch_fwd<f16, false>(x, residual, weight, nullptr, h, y, nullptr, rstd, rows, dim, eps, s);
    default: return launch_fwd<bf16, false>(x, residual, weight, nullptr, h, y, nullptr, rstd, rows, dim, eps, s);
  }
}

extern "C" int scree_add_rmsnorm_bwd(const void* dy, const void* dh, const void* h,
                                     const void* weight, const float* rstd, void* dx,
                                     void* dweight, int dparam_dtype, int64_t rows, int64_t dim,
                                     int dtype, void* workspace, size_t workspace_bytes,
                                     void* stream) {
  const char* fn = "scree_add_rmsnorm_bwd";
  int rc = validate_common(fn, rows, dim, dtype);
  if (rc) return rc;
  if (dweight && !weight) return set_error(SCREE_ERR_INVALID, "%s: dweight requires weight", fn);
  if (rows == 0 && !dweight) return SCREE_OK;
  rc = validate_bwd(fn, dy, h, rstd, dx, dweight != nullptr, dparam_dtype, rows, dim, workspace,
                    workspace_bytes);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case SCREE_DTYPE_F32: return launch_bwd<float, false>(dy, h, weight, nullptr, rstd, dh, dx, dweight, nullptr, dparam_dtype, rows, dim, workspace, s);
    case SCREE_DTYPE_F16: return launch_bwd<f16, false>(dy, h, weight, nullptr, rstd, dh, dx, dweight, nullptr, dparam_dtype, rows, dim, workspace, s);
    default: return launch_bwd<bf16, false>(dy, h, weight, nullptr, rstd, dh, dx, dweight, nullptr, dparam_dtype, rows, dim, workspace, s);
  }
}
