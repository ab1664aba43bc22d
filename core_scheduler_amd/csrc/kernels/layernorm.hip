// LayerNorm forward / backward over the last dimension for gfx950.
//
// Replaces at::native_layer_norm (src/compute/layer_norm.cpp:163-169,
// :198-204) and the two at::native_layer_norm_backward calls (:263-266 for
// dx, :321-334 / :375-383 for dgamma and dbeta).  Statistics and all
// arithmetic are fp32 for f32/f16/bf16 storage (fp64 for f64):
//   mean = sum(x)/C, var = sum((x-mean)^2)/C (biased), rstd = 1/sqrt(var+eps)
//   y    = (x-mean)*rstd*gamma + beta
//   dx   = rstd * (g - mean_C(g) - xhat*mean_C(g*xhat)),  g = dy*gamma
//   dgamma = sum_rows(dy*xhat), dbeta = sum_rows(dy)
//
// Fast path: one wavefront owns whole rows.  A row lives in registers as
// 16-byte vectors (lane l holds vectors l, l+64, ...), the two row sums are
// wave64 butterflies, and nothing is read twice: forward moves x once in and
// y once out, backward reads dy and x once and produces dx and the
// per-column partial sums in the same pass.  Each lane keeps the partial
// dgamma/dbeta of its own columns in registers across all rows its wave
// visits; a workgroup folds its waves through LDS and writes one partial row
// per workgroup, and a second small kernel adds the partial rows in a fixed
// order, so the result does not depend on scheduling and uses no atomics.
//
// Rows wider than one wave's registers, rows that are not whole vectors and unaligned pointers go
// through the same scheme with several waves per row (ln_fwd_block_kernel, ln_bwd_block_kernel);
// fp64, rows beyond 16384 columns and a few ragged rows' backward through a plain one-workgroup-per-row path.
#include "common.hpp"

#include <math.h>

#include <atomic>
#include <type_traits>

// Every product and sum below is rounded as written: no multiply-add contraction, so that the
// template variants of one kernel (with and without the fused residual adds, every output
// mask) produce the same bits for the same row.
#pragma clang fp contract(off)

namespace cs_hip {
namespace {

// ------------------------------------------------------------ n-wide access
// N consecutive elements of T (N * sizeof(T) is 16 or 32 bytes) <-> fp32.
template <typename T, int N>
__device__ __forceinline__ void load_n(const T *p, float (&out)[N]) {
  constexpr int VN = Vec16<T>::n;
  static_assert(N % VN == 0, "whole 16-byte pieces");
#pragma unroll
  for (int q = 0; q < N / VN; ++q) {
    const Vec16<T> v = load16(p + q * VN);
#pragma unroll
    for (int k = 0; k < VN; ++k) out[q * VN + k] = to_acc(v.e[k]);
  }
}
template <typename T, int N>
__device__ __forceinline__ void store_n(T *p, const float (&in)[N]) {
  constexpr int VN = Vec16<T>::n;
  static_assert(N % VN == 0, "whole 16-byte pieces");
#pragma unroll
  for (int q = 0; q < N / VN; ++q) {
    Vec16<T> v;
#pragma unroll
    for (int k = 0; k < VN; ++k) v.e[k] = from_acc<T>(in[q * VN + k]);
    store16_stream(p + q * VN, v);
  }
}
// raw (still packed) row pieces, so a row costs 4 VGPRs per 16 bytes
template <typename T, int N>
struct Raw {
  Vec16<T> v[N / Vec16<T>::n];
};
template <typename T, int N>
__device__ __forceinline__ Raw<T, N> load_raw(const T *p) {
  Raw<T, N> r;
#pragma unroll
  for (int q = 0; q < N / Vec16<T>::n; ++q) r.v[q] = load16_stream(p + q * Vec16<T>::n);
  return r;
}
// Makes the compiler forget what it derived from the packed values, so code after
// this point unpacks them again instead of keeping the unpacked floats in registers.
template <typename T, int N>
__device__ __forceinline__ void forget_unpacked(Raw<T, N> &r) {
#pragma unroll
  for (int q = 0; q < N / Vec16<T>::n; ++q) {
    u32x4 w = __builtin_bit_cast(u32x4, r.v[q]);
    asm volatile("" : "+v"(w));
    r.v[q] = __builtin_bit_cast(Vec16<T>, w);
  }
}
template <typename T, int N>
__device__ __forceinline__ Raw<T, N> zero_raw() {
  Raw<T, N> r;
#pragma unroll
  for (int q = 0; q < N / Vec16<T>::n; ++q)
#pragma unroll
    for (int k = 0; k < Vec16<T>::n; ++k) r.v[q].e[k] = T{};
  return r;
}
template <typename T, int N>
__device__ __forceinline__ float raw_get(const Raw<T, N> &r, int i) {
  return to_acc(r.v[i / Vec16<T>::n].e[i % Vec16<T>::n]);
}

constexpr int kHalf = kWave / 2;

// Sum over the LPR lanes that share a row (all 64, or each half of the wave on its own).
template <int LPR>
__device__ __forceinline__ float row_lanes_sum(float v, bool upper) {
  v += dpp_f32<kDppQuadXor1>(v);
  v += dpp_f32<kDppQuadXor2>(v);
  v += dpp_f32<kDppHalfMirror>(v);
  v += dpp_f32<kDppRowMirror>(v);
  const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 0));
  const float r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 16));
  const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 32));
  const float r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 48));
  if constexpr (LPR == kWave) return (r0 + r1) + (r2 + r3);
  return upper ? r2 + r3 : r0 + r1;
}

// forward launch shape (rows a wave normalises per step, next step's rows prefetched or not)
#ifndef CS_LN_FWD_ROWS_VPL1
#define CS_LN_FWD_ROWS_VPL1 4
#endif
#ifndef CS_LN_FWD_ROWS_VPL2
#define CS_LN_FWD_ROWS_VPL2 4
#endif
#ifndef CS_LN_FWD_ROWS_VPL4
#define CS_LN_FWD_ROWS_VPL4 2
#endif
#ifndef CS_LN_FWD_PF
#define CS_LN_FWD_PF true
#endif
#ifndef CS_LN_ADD_ROWS_VPL1
#define CS_LN_ADD_ROWS_VPL1 4
#endif
#ifndef CS_LN_ADD_ROWS_VPL4
#define CS_LN_ADD_ROWS_VPL4 1
#endif
// two rows per wave (rows of up to 32, and of 65-96, vectors): row pairs a wave normalises per step
#ifndef CS_LN_FWD_HALF
#define CS_LN_FWD_HALF 1
#endif
#ifndef CS_LN_FWD_ROWS_H1
#define CS_LN_FWD_ROWS_H1 4
#endif
#ifndef CS_LN_FWD_ROWS_H3
#define CS_LN_FWD_ROWS_H3 2
#endif
#ifndef CS_LN_ADD_ROWS_H1
#define CS_LN_ADD_ROWS_H1 4
#endif
#ifndef CS_LN_ADD_ROWS_H3
#define CS_LN_ADD_ROWS_H3 2
#endif
#ifndef CS_LN_THREADS
#define CS_LN_THREADS 256
#endif
constexpr int kLnThreads = CS_LN_THREADS;  // 4 waves
// backward launch shape; the defaults are the measured best, the macros exist for tuning runs
#ifndef CS_LN_BWD_THREADS
#define CS_LN_BWD_THREADS 512
#endif
// grid cap of the backward row kernels (the partial rows the launch leaves behind are one per workgroup): 256 workgroups
// of 8 waves, two waves per SIMD, one workgroup per CU
#ifndef CS_LN_BWD_MAX_BLOCKS
#define CS_LN_BWD_MAX_BLOCKS 256
#endif
constexpr int kLnBwdThreads = CS_LN_BWD_THREADS;

// s / c as the general kernel divides: the product with 1/c alone would bring its rounding into the mean (rows of
// one value 316 times, at rstd = 1/sqrt(eps)).  The remainder of the product corrects it (Markstein); a sum that is
// not finite has none.
__device__ __forceinline__ float over_columns(float s, float c, float inv_c) {
  const float q = s * inv_c;
  const float corrected = __builtin_fmaf(__builtin_fmaf(-q, c, s), inv_c, q);
  return fabsf(s) < INFINITY ? corrected : q;
}

// ------------------------------------------------------------ fast forward
// VPL: 16-byte x vectors per lane; R: rows a wave handles per step.  A wave
// keeps gamma and beta for its columns in registers and walks rows
// gw*R, (gw + n_waves)*R, ...; the next step's rows are loaded before the
// current ones are normalised, so loads overlap the arithmetic and the
// parameters are read once per wave, not once per row.
// VN is the column count per vector position (set by x's type); T may be wider.
template <typename T, int VN, int VPL, int R>
struct RowSet {
  Raw<T, VN> v[R][VPL];
};

template <typename T, int VN, int VPL, int R, int LPR = kWave>
__device__ __forceinline__ void load_rows(RowSet<T, VN, VPL, R> &dst, const T *__restrict__ src,
                                          int64_t row0, int64_t rows, int C, int nvec, int lane) {
  // LPR lanes per row: with 32, the wave's halves hold rows row0 + 2r and row0 + 2r + 1
  constexpr int RPW = kWave / LPR;
  const int sub = lane / LPR, hl = lane % LPR;
#pragma unroll
  for (int r = 0; r < R; ++r) {
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      const int idx = hl + LPR * j;
      const int64_t row = row0 + r * RPW + sub;
      if (idx < nvec && row < rows) {
        dst.v[r][j] = load_raw<T, VN>(src + row * C + (int64_t)idx * VN);
      } else {
        dst.v[r][j] = zero_raw<T, VN>();
      }
    }
  }
}

// One row, every lane loading: lanes past the end of the row read its last vector again.  A load
// under a lane-dependent condition can make the compiler wait for it before it issues the next
// one (it did for the third input of the backward kernel: two extra round trips per row), an
// unconditional one cannot.  What the extra lanes hold is masked where it matters (zero_past_row).
template <typename T, int VN, int VPL>
__device__ __forceinline__ void load_row_all_lanes(RowSet<T, VN, VPL, 1> &dst, const T *__restrict__ src,
                                                   int64_t row, int C, int nvec, int lane) {
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int idx = lane + kWave * j;
    dst.v[0][j] = load_raw<T, VN>(src + row * C + (int64_t)(idx < nvec ? idx : nvec - 1) * VN);
  }
}
template <typename T, int VN, int VPL>
__device__ __forceinline__ void zero_past_row(RowSet<T, VN, VPL, 1> &r, int nvec, int lane) {
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const bool past = lane + kWave * j >= nvec;
#pragma unroll
    for (int q = 0; q < VN / Vec16<T>::n; ++q) {
      u32x4 w = __builtin_bit_cast(u32x4, r.v[0][j].v[q]);
      w.x = past ? 0u : w.x;
      w.y = past ? 0u : w.y;
      w.z = past ? 0u : w.z;
      w.w = past ? 0u : w.w;
      r.v[0][j].v[q] = __builtin_bit_cast(Vec16<T>, w);
    }
  }
}

// HAS_RES: the rows that are normalised are x + residual, rounded to x's type (the sum is also
// written to sum_out, which may be x or residual itself): the residual add in front of the
// LayerNorm of a transformer block without a [rows, C] round trip between two launches.
template <typename TX, typename TY, typename TP, int VPL, int R, bool PF, bool HAS_RES, int LPR = kWave>
__global__ __launch_bounds__(kLnThreads) void ln_fwd_rows_kernel(
    const TX *x /* sum_out may be x: not restrict */, const TP *__restrict__ gamma, const TP *__restrict__ beta,
    TY *__restrict__ y, float *__restrict__ mean, float *__restrict__ rstd, int64_t rows, int C,
    float eps, const TX *res, TX *sum_out) {
  constexpr int VN = Vec16<TX>::n;
  constexpr int RPW = kWave / LPR;  // rows side by side in a wave: R * RPW rows per wave and step
  constexpr bool BY_VECTOR = VPL > 4;  // sums formed as ln_fwd_block_kernel forms them, which takes these widths too
  const int lane = threadIdx.x & (kWave - 1);
  const int sub = lane / LPR, hl = lane % LPR;
  const bool upper = sub != 0;
  const int64_t gw = (int64_t)blockIdx.x * (kLnThreads / kWave) + (threadIdx.x >> 6);
  const int64_t step = (int64_t)gridDim.x * (kLnThreads / kWave) * R * RPW;
  const int nvec = C / VN;
  int64_t row0 = gw * R * RPW;
  if (row0 >= rows) return;  // wave-uniform

  RowSet<TX, VN, VPL, R> cur, rcur;
  if constexpr (PF) {
    load_rows<TX, VN, VPL, R, LPR>(cur, x, row0, rows, C, nvec, lane);
    if constexpr (HAS_RES) load_rows<TX, VN, VPL, R, LPR>(rcur, res, row0, rows, C, nvec, lane);
  }
  float g[VPL][VN], b[VPL][VN];
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int idx = hl + LPR * j;
#pragma unroll
    for (int k = 0; k < VN; ++k) {
      g[j][k] = 0.f;
      b[j][k] = 0.f;
    }
    if (idx < nvec) {
      load_n<TP, VN>(gamma + idx * VN, g[j]);
      if (beta) load_n<TP, VN>(beta + idx * VN, b[j]);
    }
  }
  const float inv_c = 1.0f / (float)C;
  for (; row0 < rows; row0 += step) {
    RowSet<TX, VN, VPL, R> nxt, rnxt;
    if constexpr (PF) {
      if (row0 + step < rows) {
        load_rows<TX, VN, VPL, R, LPR>(nxt, x, row0 + step, rows, C, nvec, lane);
        if constexpr (HAS_RES) load_rows<TX, VN, VPL, R, LPR>(rnxt, res, row0 + step, rows, C, nvec, lane);
      }
    } else {
      load_rows<TX, VN, VPL, R, LPR>(cur, x, row0, rows, C, nvec, lane);
      if constexpr (HAS_RES) load_rows<TX, VN, VPL, R, LPR>(rcur, res, row0, rows, C, nvec, lane);
    }
    if constexpr (HAS_RES) {
      // cur = x + residual, one fp32 add and one rounding per element, as an add launch would give
#pragma unroll
      for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
          Vec16<TX> sum;
#pragma unroll
          for (int k = 0; k < VN; ++k)
            sum.e[k] = from_acc<TX>(raw_get<TX, VN>(cur.v[r][j], k) + raw_get<TX, VN>(rcur.v[r][j], k));
          cur.v[r][j].v[0] = sum;
          const int idx = hl + LPR * j;
          const int64_t row = row0 + r * RPW + sub;
          if (idx < nvec && row < rows) store16_stream(sum_out + row * C + (int64_t)idx * VN, sum);
        }
      }
    }
    // the R rows are independent: their reductions interleave
    float mu[R], rs[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < VPL; ++j) {
        float t = BY_VECTOR ? 0.f : s;
#pragma unroll
        for (int k = 0; k < VN; ++k) t += raw_get<TX, VN>(cur.v[r][j], k);
        s = BY_VECTOR ? s + t : t;
      }
      mu[r] = s;
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      mu[r] = row_lanes_sum<LPR>(mu[r], upper);
      mu[r] = BY_VECTOR ? over_columns(mu[r], (float)C, inv_c) : mu[r] * inv_c;
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float q = 0.f;
#pragma unroll
      for (int j = 0; j < VPL; ++j) {
        if (hl + LPR * j < nvec) {
          float t = BY_VECTOR ? 0.f : q;
#pragma unroll
          for (int k = 0; k < VN; ++k) {
            const float d = raw_get<TX, VN>(cur.v[r][j], k) - mu[r];
            t += d * d;
          }
          q = BY_VECTOR ? q + t : t;
        }
      }
      rs[r] = q;
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      rs[r] = row_lanes_sum<LPR>(rs[r], upper);
      rs[r] = 1.0f / sqrtf((BY_VECTOR ? over_columns(rs[r], (float)C, inv_c) : rs[r] * inv_c) + eps);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (row0 + r * RPW >= rows) break;  // wave-uniform
      const int64_t row = row0 + r * RPW + sub;
      const bool row_ok = row < rows;
      if (hl == 0 && row_ok) {
        mean[row] = mu[r];
        rstd[row] = rs[r];
      }
#pragma unroll
      for (int j = 0; j < VPL; ++j) {
        const int idx = hl + LPR * j;
        if (idx < nvec && row_ok) {
          float o[VN];
#pragma unroll
          for (int k = 0; k < VN; ++k)
            o[k] = (raw_get<TX, VN>(cur.v[r][j], k) - mu[r]) * rs[r] * g[j][k] + b[j][k];
          store_n<TY, VN>(y + row * C + (int64_t)idx * VN, o);
        }
      }
    }
    if constexpr (PF) {
      cur = nxt;
      if constexpr (HAS_RES) rcur = rnxt;
    }
  }
}

// Vector `idx` of a parameter row, zeros where the row has no such one: the last vector's again would do for anything that
// is masked later, but a lane's zero of dy times an infinite gamma is NaN.
template <typename T, int N>
__device__ __forceinline__ void load_n_or_zeros(RowBuffer row, bool there, int idx, float (&out)[N]) {
  constexpr int kBytes = N * (int)sizeof(T);
  const int at = there ? idx * kBytes : kOutside;
  if constexpr (kBytes == 8) {
    struct alignas(8) Half {
      T e[N];
    } v = __builtin_bit_cast(Half, __builtin_amdgcn_raw_buffer_load_b64(row, at, 0, 0));
#pragma unroll
    for (int k = 0; k < N; ++k) out[k] = to_acc(v.e[k]);
  } else {
    constexpr int VN = Vec16<T>::n;
#pragma unroll
    for (int q = 0; q < N / VN; ++q) {
      const auto v = __builtin_bit_cast(Vec16<T>, __builtin_amdgcn_raw_buffer_load_b128(row, at + q * 16, 0, 0));
#pragma unroll
      for (int k = 0; k < VN; ++k) out[q * VN + k] = to_acc(v.e[k]);
    }
  }
}
template <typename T, int VN, int VPL>
struct Strip {
  Raw<T, VN> v[VPL];
};
// every lane loads (from the last vector of the row again where it has none of its own)
template <typename T, int VN, int VPL, int LPR>
__device__ __forceinline__ void load_strip(Strip<T, VN, VPL> &dst, const T *src, int64_t row, int C, int nvec,
                                           int hl) {
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int idx = hl + LPR * j;
    dst.v[j] = load_raw<T, VN>(src + row * C + (int64_t)(idx < nvec ? idx : nvec - 1) * VN);
  }
}
template <typename T, int VN, int VPL, int LPR>
__device__ __forceinline__ void zero_strip_unless(Strip<T, VN, VPL> &r, bool row_ok, int nvec, int hl) {
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const bool keep = row_ok && hl + LPR * j < nvec;
#pragma unroll
    for (int q = 0; q < VN / Vec16<T>::n; ++q) {
      u32x4 w = __builtin_bit_cast(u32x4, r.v[j].v[q]);
      w.x = keep ? w.x : 0u;
      w.y = keep ? w.y : 0u;
      w.z = keep ? w.z : 0u;
      w.w = keep ? w.w : 0u;
      r.v[j].v[q] = __builtin_bit_cast(Vec16<T>, w);
    }
  }
}

// One step of ln_fwd_rows_kernel per wave, one wave to a workgroup: few rows are spread over the chip, and every load
// goes out at once (there the loads stand under the lane's condition, which makes each wait for the one before: hidden
// where a CU has waves enough, a chain of trips to memory where it has one).  The same sums in the same order.
template <typename TX, typename TY, typename TP, int VPL, bool HAS_RES, int LPR>
__global__ __launch_bounds__(kWave) void ln_fwd_few_kernel(
    const TX *x /* sum_out may be x: not restrict */, const TP *__restrict__ gamma, const TP *__restrict__ beta,
    TY *__restrict__ y, float *__restrict__ mean, float *__restrict__ rstd, int64_t rows, int C,
    float eps, const TX *res, TX *sum_out) {
  constexpr int VN = Vec16<TX>::n;
  static_assert(VPL <= 4, "the sums of longer rows are formed by vector");
  const int lane = threadIdx.x;
  const int sub = lane / LPR, hl = lane % LPR;
  const bool upper = sub != 0;
  const int64_t row = (int64_t)blockIdx.x * (kWave / LPR) + sub;
  const bool row_ok = row < rows;
  const int64_t rowc = row_ok ? row : rows - 1;
  const int nvec = C / VN;
  Strip<TX, VN, VPL> cur, rcur;
  load_strip<TX, VN, VPL, LPR>(cur, x, rowc, C, nvec, hl);
  if constexpr (HAS_RES) load_strip<TX, VN, VPL, LPR>(rcur, res, rowc, C, nvec, hl);
  float g[VPL][VN], b[VPL][VN];
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int idx = hl + LPR * j < nvec ? hl + LPR * j : nvec - 1;
    load_n<TP, VN>(gamma + idx * VN, g[j]);
  }
  const TP *bsrc = beta ? beta : gamma;
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int idx = hl + LPR * j < nvec ? hl + LPR * j : nvec - 1;
    load_n<TP, VN>(bsrc + idx * VN, b[j]);
  }
  if constexpr (HAS_RES) {
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      Vec16<TX> sum;
#pragma unroll
      for (int k = 0; k < VN; ++k) sum.e[k] = from_acc<TX>(raw_get<TX, VN>(cur.v[j], k) + raw_get<TX, VN>(rcur.v[j], k));
      cur.v[j].v[0] = sum;
      const int idx = hl + LPR * j;
      if (idx < nvec && row_ok) store16_stream(sum_out + row * C + (int64_t)idx * VN, sum);
    }
  }
  zero_strip_unless<TX, VN, VPL, LPR>(cur, true, nvec, hl);
  const float inv_c = 1.0f / (float)C;
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < VPL; ++j)
#pragma unroll
    for (int k = 0; k < VN; ++k) s += raw_get<TX, VN>(cur.v[j], k);
  const float mu = row_lanes_sum<LPR>(s, upper) * inv_c;
  float q = 0.f;
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    if (hl + LPR * j < nvec) {
#pragma unroll
      for (int k = 0; k < VN; ++k) {
        const float d = raw_get<TX, VN>(cur.v[j], k) - mu;
        q += d * d;
      }
    }
  }
  const float rs = 1.0f / sqrtf(row_lanes_sum<LPR>(q, upper) * inv_c + eps);
  if (!row_ok) return;
  if (hl == 0) {
    mean[row] = mu;
    rstd[row] = rs;
  }
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int idx = hl + LPR * j;
    if (idx < nvec) {
      float o[VN];
#pragma unroll
      for (int k = 0; k < VN; ++k) o[k] = (raw_get<TX, VN>(cur.v[j], k) - mu) * rs * g[j][k] + (beta ? b[j][k] : 0.f);
      store_n<TY, VN>(y + row * C + (int64_t)idx * VN, o);
    }
  }
}

// ------------------------------------------------- column sums of partial rows
// What a launch of the row kernel may do on the side: the column sums of an EARLIER call's partial
// rows (written by a launch that is complete when this one starts).  The first `blocks`
// workgroups of the grid do that and leave; the row work starts at workgroup `blocks`.
struct LnPending {
  const void *partial;   // nullptr: nothing pending
  void *dgamma, *dbeta;  // of the earlier call; either may be nullptr
  int nparts, accumulate, blocks;
};

// Adds `nparts` partial rows of P in a fixed order.  Partial rows are permuted: position
// p = k*nvec + idx holds column idx*vn + k (nvec = C/vn); columns past the last whole vector stay in
// place.  One tile = 32 positions of dgamma or
// dbeta: thread (cx, ry) of 32 x 16 sums partial rows ry, ry+16, ... for one position, sixteen
// loads in flight and none of them under a condition (this work waits for a row kernel and is all
// latency), then row 0 adds the 16 sub-sums in order.  `sub` is 16 x 32 floats of LDS.
constexpr int kLnFinCols = 32, kLnFinRows = 16, kLnFinInFlight = 16;

template <typename TP, int THREADS = kLnFinCols * kLnFinRows, typename A = float, typename P = float>
__device__ __forceinline__ void ln_finalize_tile(const P *__restrict__ partial, int nparts, TP *__restrict__ out,
                                                 int which, int tile, int C, int vn, int accumulate, A *sub,
                                                 int tid) {
  static_assert(THREADS >= kLnFinCols * kLnFinRows, "a tile takes 512 threads; further ones only join the barrier");
  const int cx = tid % kLnFinCols, ry = tid / kLnFinCols;
  const int col = tile * kLnFinCols + cx;  // a position in the permuted row
  A s = 0;
  if (col < C && ry < kLnFinRows) {
    const P *src = partial + (int64_t)which * C + col;
    const int64_t stride = 2 * (int64_t)C;
    for (int p0 = ry; p0 < nparts; p0 += kLnFinRows * kLnFinInFlight) {
      P v[kLnFinInFlight];
#pragma unroll
      for (int u = 0; u < kLnFinInFlight; ++u) {
        const int p = p0 + u * kLnFinRows;
        v[u] = src[(int64_t)(p < nparts ? p : nparts - 1) * stride];
      }
#pragma unroll
      for (int u = 0; u < kLnFinInFlight; ++u) s += (A)(p0 + u * kLnFinRows < nparts ? v[u] : (P)0);
    }
  }
  if (ry < kLnFinRows) sub[ry * kLnFinCols + cx] = s;
  __syncthreads();
  if (ry == 0 && col < C) {
    A t = 0;
#pragma unroll
    for (int r = 0; r < kLnFinRows; ++r) t += sub[r * kLnFinCols + cx];
    const int nvec = C / vn;
    // the column this position stands for
    const int real = col < nvec * vn ? (col % nvec) * vn + col / nvec : col;
    if (accumulate) t += (A)to_acc(out[real]);
    out[real] = from_acc<TP>((float)t);
  }
}
// workgroup b of the 2 * ceil(C/32) that cover a pending call: even b dgamma, odd b dbeta
template <typename TP, int THREADS = kLnFinCols * kLnFinRows, typename A = float, typename P = float>
__device__ __forceinline__ void ln_finalize_pending(const LnPending &pend, int b, int C, int vn, A *sub, int tid) {
  const int which = b & 1;
  TP *out = (TP *)(which == 0 ? pend.dgamma : pend.dbeta);
  if (out == nullptr) return;  // block-uniform
  ln_finalize_tile<TP, THREADS, A, P>((const P *)pend.partial, pend.nparts, out, which, b >> 1, C, vn, pend.accumulate,
                                      sub, tid);
}

// The column sums of few rows, straight from dy and x: they need the saved statistics but not the row sums of
// the backward pass, so workgroups of the row kernel's own launch take them, and neither partial rows nor a
// second launch (4 us behind the first, and 2.8 us of host time) are needed.  One tile = 32 columns of dgamma
// and dbeta: thread (cx, ry) of 32 x 16 stands in for partial rows ry, ry+16, ... of RPP rows each, as the row
// kernel and the finalize step would have left and added them, bit for bit where x-hat is finite.  All loads of a
// partial row are requested before the first use.  sub: 2 x 16 x 32 floats of LDS.
template <typename TDY, typename TX, typename TP, int RPP>
__device__ __forceinline__ void ln_columns_direct(const TDY *__restrict__ dy, const TX *__restrict__ x,
                                                  const float *__restrict__ mean, const float *__restrict__ rstd,
                                                  const LnPending &side, int64_t rows, int tile, int C, float *sub,
                                                  int tid) {
  const int cx = tid % kLnFinCols, ry = tid / kLnFinCols;
  const int col = tile * kLnFinCols + cx;
  const int64_t at = col < C ? col : C - 1;
  float sg = 0.f, sb = 0.f;
  static_assert(kWave == 2 * kLnFinCols, "a wave has the columns of two partial rows");
  auto add = [&](int p, auto all_rows) {
    constexpr bool full = decltype(all_rows)::value;
    TDY d[RPP];
    TX v[RPP];
    float mu[RPP], rs[RPP];
#pragma unroll
    for (int w = 0; w < RPP; ++w) {
      const int64_t row = (int64_t)p * RPP + w;
      const int64_t rowc = full || row < rows ? row : rows - 1;
      d[w] = dy[rowc * C + at];
      v[w] = x[rowc * C + at];
      mu[w] = mean[rowc];
      rs[w] = rstd[rowc];
    }
    float pg = 0.f, pb = 0.f;
#pragma unroll
    for (int w = 0; w < RPP; ++w) {
      float xh = (to_acc(v[w]) - mu[w]) * rs[w], dv = to_acc(d[w]);
      if constexpr (!full) {
        // both masked, as in ln_columns_wide, and only now: under the condition the loads would wait for one another
        asm volatile("" : "+v"(xh), "+v"(dv));
        const bool live = (int64_t)p * RPP + w < rows;
        xh = live ? xh : 0.f;
        dv = live ? dv : 0.f;
      }
      pg += __builtin_fmaf(dv, xh, 0.f);
      pb += dv;
    }
    sg += pg;
    sb += pb;
  };
  // The last partial row may lack rows.  A wave stands in for two neighbouring ones and takes both the same way: apart
  // they were two trips to memory ([123,768] bf16 4.5 us against 3.8).
  const int whole = (int)(rows / RPP);
  for (int p = ry; p < side.nparts; p += kLnFinRows) {
    if ((p | 1) < whole) {
      add(p, std::true_type{});
    } else {
      add(p, std::false_type{});
    }
  }
  sub[ry * kLnFinCols + cx] = sg;
  sub[(kLnFinRows + ry) * kLnFinCols + cx] = sb;
  __syncthreads();
  TP *out = (TP *)(ry == 0 ? side.dgamma : side.dbeta);
  if (ry < 2 && col < C && out != nullptr) {
    float t = 0.f;
#pragma unroll
    for (int r = 0; r < kLnFinRows; ++r) t += sub[(ry * kLnFinRows + r) * kLnFinCols + cx];
    if (side.accumulate) t += to_acc(out[col]);
    out[col] = from_acc<TP>(t);
  }
}

// The same for rows on several waves (ln_bwd_block_kernel), any width and alignment: sums in double, terms as that
// kernel forms them, so the two differ by roundings of a double.  A tile is 32 columns for 2 x `waves` row lanes, each
// with 16 rows under way.  sub: 2 x 2 x waves x 32 doubles of LDS.
constexpr int kLnWideTile = kHalf;
template <typename TDY, typename TX, typename TP>
__device__ __forceinline__ void ln_columns_wide(const TDY *__restrict__ dy, const TX *__restrict__ x,
                                                const float *__restrict__ mean, const float *__restrict__ rstd,
                                                const LnPending &side, int64_t rows, int tile, int C, double *sub) {
  constexpr int kInFlight = 16;
  const int cx = threadIdx.x % kLnWideTile, ry = threadIdx.x / kLnWideTile, lanes = blockDim.x / kLnWideTile;
  const int col = tile * kLnWideTile + cx;
  const int64_t at = col < C ? col : C - 1;
  double sg = 0., sb = 0.;
  for (int64_t r0 = ry; r0 < rows; r0 += (int64_t)lanes * kInFlight) {
    TDY d[kInFlight];
    TX v[kInFlight];
    float mu[kInFlight], rs[kInFlight];
#pragma unroll
    for (int u = 0; u < kInFlight; ++u) {
      const int64_t r = r0 + (int64_t)u * lanes, rr = r < rows ? r : rows - 1;
      d[u] = dy[rr * C + at];
      v[u] = x[rr * C + at];
      mu[u] = mean[rr];
      rs[u] = rstd[rr];
    }
#pragma unroll
    for (int u = 0; u < kInFlight; ++u) {
      const bool live = r0 + (int64_t)u * lanes < rows;
      // both masked: 0 * inf would leave a NaN in the sums
      const float xh = live ? (to_acc(v[u]) - mu[u]) * rs[u] : 0.f;
      const float dv = live ? to_acc(d[u]) : 0.f;
      sg += (double)(dv * xh);
      sb += (double)dv;
    }
  }
  sub[ry * kLnWideTile + cx] = sg;
  sub[(lanes + ry) * kLnWideTile + cx] = sb;
  __syncthreads();
  TP *out = (TP *)(ry == 0 ? side.dgamma : side.dbeta);
  if (ry < 2 && col < C && out != nullptr) {
    double t = 0.;
    for (int r = 0; r < lanes; ++r) t += sub[(ry * lanes + r) * kLnWideTile + cx];
    if (side.accumulate) t += (double)to_acc(out[col]);
    out[col] = from_acc<TP>((float)t);
  }
}

// ----------------------------------------------------------- fast backward
// Rows of 4 vectors per lane.  One wave per row, the row (dy and x) in registers, gamma and the per-column partial sums in
// registers for all rows a wave visits (rows gw, gw + n_waves, ...).  No software prefetch:
// two waves per SIMD are resident (the launch bound asks the compiler for that), so while one
// wave waits for its row the others compute; measured on MI355X this beats two rows per wave
// with the next step's rows prefetched ([16384,1600] bf16: 32.8 -> 30.3 us) because twice as many
// waves are in flight with half the registers each.
// The arithmetic uses explicit fused multiply-adds (contraction is off in this file, so every
// variant of the kernel rounds alike): 17 VALU operations per element instead of 27, which
// matters because at 16-bit storage this kernel is as close to its VALU limit as to HBM's.
// HAS_DRES: dx_out = dx + dresidual, the gradient add that follows LayerNorm::backward on the
// residual stream; dx is rounded to its type first, then the sum, as two kernels would.
// DIRECT: the launch's first workgroups take the column sums of this very call from its rows (ln_columns_direct).
template <typename TDY, typename TX, typename TDX, typename TP, bool HAS_DX, bool HAS_DP, bool HAS_DRES, bool DIRECT = false>
__global__ __launch_bounds__(kLnBwdThreads, 2) void ln_bwd_rows_kernel(
    const TDY *__restrict__ dy, const TX *__restrict__ x, const float *__restrict__ mean,
    const float *__restrict__ rstd, const TP *__restrict__ gamma, TDX *dx,
    float *__restrict__ partial, int64_t rows, int C, const TDX *dres /* dx may be dres */,
    const LnPending pend) {
  constexpr int VN = Vec16<TX>::n, VPL = 4;
  extern __shared__ float lds[];  // [waves per block][C], at least 16 x 32 floats with pending sums
  if ((int)blockIdx.x < pend.blocks) {
    if constexpr (DIRECT) {
      ln_columns_direct<TDY, TX, TP, kLnBwdThreads / kWave>(dy, x, mean, rstd, pend, rows, blockIdx.x, C, lds, threadIdx.x);
    } else {
      ln_finalize_pending<TP>(pend, blockIdx.x, C, VN, lds, threadIdx.x);
    }
    return;
  }
  const int bid = blockIdx.x - pend.blocks;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x >> 6;
  constexpr int kWaves = kLnBwdThreads / kWave;
  const int64_t step = (int64_t)(gridDim.x - pend.blocks) * kWaves;
  const int nvec = C / VN;
  const float inv_c = 1.0f / (float)C;

  float acc_g[VPL][VN], acc_b[VPL][VN], g[VPL][VN];
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
#pragma unroll
    for (int k = 0; k < VN; ++k) {
      acc_g[j][k] = 0.f;
      acc_b[j][k] = 0.f;
      g[j][k] = 0.f;
    }
    if (HAS_DX && lane + kWave * j < nvec) load_n<TP, VN>(gamma + (lane + kWave * j) * VN, g[j]);
  }

  for (int64_t row = (int64_t)bid * kWaves + wave; row < rows; row += step) {
    RowSet<TDY, VN, VPL, 1> dcur;
    RowSet<TX, VN, VPL, 1> xcur;
    RowSet<TDX, VN, VPL, 1> rcur;  // this row of dresidual, in flight during the reductions
    if constexpr (HAS_DRES) {
      // three inputs: with loads under the lane's own condition the compiler waits for each
      // piece of the third before it issues the next (two extra round trips per row at
      // [16384,1600]: 53.1 -> 46.4 us); every lane loads instead
      load_row_all_lanes<TDY, VN, VPL>(dcur, dy, row, C, nvec, lane);
      load_row_all_lanes<TX, VN, VPL>(xcur, x, row, C, nvec, lane);
      load_row_all_lanes<TDX, VN, VPL>(rcur, dres, row, C, nvec, lane);
      zero_past_row<TDY, VN, VPL>(dcur, nvec, lane);  // so that lanes past the row add nothing below
    } else {
      // two inputs: the conditional form has no such waits and needs half the registers
      // (34.0 against 36.4 us)
      load_rows<TDY, VN, VPL, 1>(dcur, dy, row, rows, C, nvec, lane);
      load_rows<TX, VN, VPL, 1>(xcur, x, row, rows, C, nvec, lane);
    }
    const float mu = mean[row], rs = rstd[row];
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
#pragma unroll
      for (int k = 0; k < VN; ++k) {
        // lanes past the row hold zeros in dy, so they add nothing
        const float xh = (raw_get<TX, VN>(xcur.v[0][j], k) - mu) * rs;
        const float dv = raw_get<TDY, VN>(dcur.v[0][j], k);
        if constexpr (HAS_DP) {
          acc_g[j][k] = __builtin_fmaf(dv, xh, acc_g[j][k]);
          acc_b[j][k] += dv;
        }
        if constexpr (HAS_DX) {
          const float gd = dv * g[j][k];
          s1 += gd;
          s2 = __builtin_fmaf(gd, xh, s2);
        }
      }
    }
    if constexpr (HAS_DX) {
      s1 = wave_reduce(s1, SumOp{}) * inv_c;
      s2 = wave_reduce(s2, SumOp{}) * inv_c;
      // x-hat and dy are unpacked again from the packed row rather than kept as floats across
      // the reduction: half the registers, a few more VALU ops
#pragma unroll
      for (int j = 0; j < VPL; ++j) {
        forget_unpacked(xcur.v[0][j]);
        forget_unpacked(dcur.v[0][j]);
        // also keeps the load of this piece up where it was issued: without a use outside the
        // branch below the compiler moves it into the branch, behind the reductions
        if constexpr (HAS_DRES) forget_unpacked(rcur.v[0][j]);
        const int idx = lane + kWave * j;
        if (idx < nvec) {
          float o[VN];
#pragma unroll
          for (int k = 0; k < VN; ++k) {
            const float xh = (raw_get<TX, VN>(xcur.v[0][j], k) - mu) * rs;
            const float dv = raw_get<TDY, VN>(dcur.v[0][j], k);
            // rstd * (dy gamma - mean(dy gamma) - xhat mean(dy gamma xhat))
            o[k] = rs * __builtin_fmaf(-xh, s2, __builtin_fmaf(dv, g[j][k], -s1));
            if constexpr (HAS_DRES)
              o[k] = round_through<TDX>(o[k]) + raw_get<TDX, VN>(rcur.v[0][j], k);
          }
          store_n<TDX, VN>(dx + row * C + (int64_t)idx * VN, o);
        }
      }
    }
  }

  if constexpr (HAS_DP) {
    // fold the block's waves, dgamma first, then dbeta through the same LDS.  Column
    // idx*VN + k is kept at position k*nvec + idx, in the LDS and in the partial rows: lanes
    // then write consecutive words (no bank conflicts); the last kernel undoes the permutation.
#pragma unroll
    for (int which = 0; which < 2; ++which) {
#pragma unroll
      for (int j = 0; j < VPL; ++j) {
        const int idx = lane + kWave * j;
        if (idx < nvec) {
#pragma unroll
          for (int k = 0; k < VN; ++k)
            lds[wave * C + k * nvec + idx] = which == 0 ? acc_g[j][k] : acc_b[j][k];
        }
      }
      __syncthreads();
      for (int c = threadIdx.x; c < C; c += kLnBwdThreads) {
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) s += lds[w * C + c];
        partial[((int64_t)bid * 2 + which) * C + c] = s;
      }
      __syncthreads();
    }
  }
}

// --------------------------------- rows on whole waves or on halves of a wave
// LPR lanes per row: 64 (a wave per row) or 32: two rows per wave, side by side, lanes 0-31 on row
// 2p, lanes 32-63 on row 2p + 1, for rows of at most 32 * VPL vectors.  A 768-column row of 16-bit
// data is 96 vectors = 32 lanes x 3, so every lane slot is used (on whole waves it takes two
// vectors per lane and leaves a quarter of them empty), a wave finishes two rows per round trip to
// memory, and the same number of waves leaves half as many rows behind them.  The two row sums
// are reduced per half; the column sums of the halves meet in the LDS fold at the end.
#ifndef CS_LN_PAIR_FOLD
#define CS_LN_PAIR_FOLD 1
#endif

// PF: the next step's rows are requested before the current ones are worked on.
// KEEP: x-hat and dy*gamma stay unpacked across the two row sums instead of being unpacked and
// normalised again for the second pass (at 16-bit storage the kernel is as close to the VALU
// limit as to the memory's); takes VPL * 2 * VN more registers.
// A wave per row forms fp32 results from dy and gamma again, so that their product is not rounded ahead of the subtraction
// and rstd not multiplied into each term: at a correlation of 0, 0.5, 0.9 and 0.999 between dy and x-hat their rms error
// against 64 bits is 4.4, 5.6, 11 and 29 e-8 at 512 columns, and was 4.4, 6.0, 13 and 34 (which 16-bit results round away).
template <typename TDY, typename TX, typename TDX, typename TP, int THREADS, int LPR, int VPL, int WPE, bool PF,
          bool KEEP,
          bool HAS_DX, bool HAS_DP, bool HAS_DRES, bool DIRECT>
__global__ __launch_bounds__(THREADS, WPE) void ln_bwd_kernel(
    const TDY *__restrict__ dy, const TX *__restrict__ x, const float *__restrict__ mean,
    const float *__restrict__ rstd, const TP *__restrict__ gamma, TDX *dx /* may be dres */,
    float *__restrict__ partial, int64_t rows, int C, const TDX *dres, const LnPending pend) {
  constexpr int VN = Vec16<TX>::n;
  constexpr int RPW = kWave / LPR;  // rows a wave works on side by side
  constexpr bool kUnrounded = LPR == kWave && std::is_same_v<TDX, float>;
  // One vector per lane: both rows' registers are requested again as soon as they are free, a row and a half under way
  // instead of one.  us per call, one row ahead / this: fp32 [40000,256] the sums alone 21.5 / 16.6, plain 26.2 / 25.7, bf16
  // [60000,512] the sums alone 28.9 / 23.5, with dresidual 45.6 / 44.8, [10000,512] 12.0 / 11.2.
  constexpr bool TWO_AHEAD = PF && LPR == kWave && VPL == 1;
  extern __shared__ float lds[];    // [RPW * waves per block][C], at least 16 x 32 floats
  if ((int)blockIdx.x < pend.blocks) {
    if constexpr (DIRECT) {
      ln_columns_direct<TDY, TX, TP, RPW * THREADS / kWave>(dy, x, mean, rstd, pend, rows, blockIdx.x, C, lds, threadIdx.x);
    } else {
      ln_finalize_pending<TP, THREADS>(pend, blockIdx.x, C, VN, lds, threadIdx.x);
    }
    return;
  }
  const int bid = blockIdx.x - pend.blocks, nblocks = gridDim.x - pend.blocks;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x >> 6;
  const bool upper = LPR == kHalf && lane >= kHalf;
  const int hl = lane & (LPR - 1);
  constexpr int kWaves = THREADS / kWave;
  const int64_t step = (int64_t)nblocks * kWaves;
  const int64_t nsteps = (rows + RPW - 1) / RPW;  // row groups: one per wave and step
  const int nvec = C / VN;
  const float inv_c = 1.0f / (float)C;

  const RowBuffer gamma_row = row_buffer(gamma, C * (int)sizeof(TP));
  float acc_g[VPL][VN], acc_b[VPL][VN], g[VPL][VN];
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int idx = hl + LPR * j;
#pragma unroll
    for (int k = 0; k < VN; ++k) {
      acc_g[j][k] = 0.f;
      acc_b[j][k] = 0.f;
    }
    if constexpr (HAS_DX) load_n_or_zeros<TP, VN>(gamma_row, idx < nvec, idx, g[j]);
  }

  struct Row {
    Strip<TDY, VN, VPL> dy;
    Strip<TX, VN, VPL> x;
    Strip<TDX, VN, VPL> res;  // this row of dresidual, in flight during the reductions
    float mu, rs;
  };
  auto issue = [&](Row &in, int64_t p_) {
    const int64_t row = RPW * p_ + (upper ? 1 : 0);
    const int64_t rowc = row < rows ? row : rows - 1;
    load_strip<TDY, VN, VPL, LPR>(in.dy, dy, rowc, C, nvec, hl);
    load_strip<TX, VN, VPL, LPR>(in.x, x, rowc, C, nvec, hl);
    if constexpr (HAS_DRES) load_strip<TDX, VN, VPL, LPR>(in.res, dres, rowc, C, nvec, hl);
    in.mu = mean[rowc];
    in.rs = rstd[rowc];
  };
  int64_t p = (int64_t)bid * kWaves + wave;
  Row cur, nxt;
  auto work = [&](Row &in, int64_t p) {
    Strip<TDY, VN, VPL> &dcur = in.dy;
    Strip<TX, VN, VPL> &xcur = in.x;
    Strip<TDX, VN, VPL> &rcur = in.res;
    const float mu = in.mu, rs = in.rs;
    const int64_t row = RPW * p + (upper ? 1 : 0);
    const bool row_ok = row < rows;
    zero_strip_unless<TDY, VN, VPL, LPR>(dcur, row_ok, nvec, hl);  // lanes without data add nothing below
    float s1 = 0.f, s2 = 0.f;
    float xh[KEEP ? VPL : 1][VN], gd[KEEP ? VPL : 1][VN];
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      const int jj = KEEP ? j : 0;
#pragma unroll
      for (int k = 0; k < VN; ++k) {
        xh[jj][k] = (raw_get<TX, VN>(xcur.v[j], k) - mu) * rs;
        const float dv = raw_get<TDY, VN>(dcur.v[j], k);
        if constexpr (HAS_DP) {
          acc_g[j][k] = __builtin_fmaf(dv, xh[jj][k], acc_g[j][k]);
          acc_b[j][k] += dv;
        }
        if constexpr (HAS_DX) {
          const float t = dv * g[j][k];
          s1 += t;
          s2 = __builtin_fmaf(t, xh[jj][k], s2);
          gd[jj][k] = kUnrounded ? dv : t;
        }
      }
    }
    if constexpr (HAS_DX) {
      // rstd * (dy gamma - mean(dy gamma) - xhat mean(dy gamma xhat)), folded with the row's three
      // factors first: two operations per element
      s1 = row_lanes_sum<LPR>(s1, upper) * inv_c;
      s2 = row_lanes_sum<LPR>(s2, upper) * inv_c;
      const float cb = -s1 * rs, cc = -s2 * rs;
#pragma unroll
      for (int j = 0; j < VPL; ++j) {
        const int jj = KEEP ? j : 0;
        if constexpr (!KEEP) {
          // unpacked again from the packed row rather than kept as floats across the reduction
          forget_unpacked(xcur.v[j]);
          forget_unpacked(dcur.v[j]);
        }
        if constexpr (HAS_DRES) forget_unpacked(rcur.v[j]);  // keeps its load where it was issued
        const int idx = hl + LPR * j;
        float o[VN];
#pragma unroll
        for (int k = 0; k < VN; ++k) {
          if constexpr (!KEEP) {
            xh[jj][k] = (raw_get<TX, VN>(xcur.v[j], k) - mu) * rs;
            gd[jj][k] = raw_get<TDY, VN>(dcur.v[j], k) * (kUnrounded ? 1.f : g[j][k]);
          }
          if constexpr (kUnrounded) {
            o[k] = rs * __builtin_fmaf(-xh[jj][k], s2, __builtin_fmaf(gd[jj][k], g[j][k], -s1));
          } else {
            o[k] = __builtin_fmaf(xh[jj][k], cc, __builtin_fmaf(gd[jj][k], rs, cb));
          }
          if constexpr (HAS_DRES) o[k] = round_through<TDX>(o[k]) + raw_get<TDX, VN>(rcur.v[j], k);
        }
        if (row_ok && idx < nvec) store_n<TDX, VN>(dx + row * C + (int64_t)idx * VN, o);
      }
    }
  };
  if constexpr (TWO_AHEAD) {
    if (p < nsteps) {
      issue(cur, p);
      issue(nxt, p + step);
      for (; p + step < nsteps; p += 2 * step) {
        work(cur, p);
        issue(cur, p + 2 * step);
        work(nxt, p + step);
        issue(nxt, p + 3 * step);
      }
      if (p < nsteps) work(cur, p);
    }
  } else {
    if constexpr (PF) {
      if (p < nsteps) issue(cur, p);
    }
    for (; p < nsteps; p += step) {
      if constexpr (PF) {
        if (p + step < nsteps) issue(nxt, p + step);
      } else {
        issue(cur, p);
      }
      work(cur, p);
      if constexpr (PF) cur = nxt;
    }
  }

#if CS_LN_PAIR_FOLD <= 0
  if constexpr (HAS_DP) {
    float t = 0.f;
#pragma unroll
    for (int j = 0; j < VPL; ++j)
#pragma unroll
      for (int k = 0; k < VN; ++k) t += acc_g[j][k] * acc_b[j][k];
    if (t == 12345.678f) partial[threadIdx.x] = t;
  }
#endif
  if constexpr (HAS_DP && CS_LN_PAIR_FOLD > 0) {
    // Fold the block's waves (half-waves), dgamma first, then dbeta through the same LDS.  Column
    // idx*VN + k is kept at position k*nvec + idx, in the LDS and in the partial rows: lanes
    // then write consecutive words (no bank conflicts); the finalize step undoes the permutation.
    // (Measured against 16-byte LDS writes in a layout that suits them, with 16-byte or 4-byte
    // reads: 0.3-0.9 us slower per launch at [8192,768] than these 4-byte accesses.)
    const int hw = wave * RPW + (upper ? 1 : 0);
#pragma unroll
    for (int which = 0; which < 2; ++which) {
#pragma unroll
      for (int j = 0; j < VPL; ++j) {
        const int idx = hl + LPR * j;
        if (idx < nvec) {
#pragma unroll
          for (int k = 0; k < VN; ++k) lds[hw * C + k * nvec + idx] = which == 0 ? acc_g[j][k] : acc_b[j][k];
        }
      }
      lds_barrier();
      for (int c = threadIdx.x; c < C; c += THREADS) {
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < RPW * kWaves; ++w) s += lds[w * C + c];
        partial[((int64_t)bid * 2 + which) * C + c] = s;
      }
      if (which == 0) lds_barrier();
    }
  }
}

// --------------------------------------------------- rows on several waves
// Rows wider than the register plans above, and rows of any width that are not whole aligned
// vectors.  A row belongs to a group of `gw` waves (1 to 16), lane i of the group's 64*gw lanes
// owning vectors i, i + 64*gw, ... (VPT of them); a workgroup holds as many groups as fit and walks
// rows.  UA: rows may start anywhere: vectors are accessed at element alignment, and the columns past
// the last whole vector (fewer than one vector of them) are single elements of the group's first
// lanes, which load them unconditionally (a load under a lane's condition would hold up the others).
//
// Bound by HBM; what it took to get near was the number of loads in flight.  A wave-sized row slice
// per wave and 8 elements per lane leave registers for two rows (the next one requested as soon as
// the one before the current is done), gamma, beta or the column sums.  Whole vectors are accessed through a RowBuffer,
// so that nothing in a step depends on a lane or on whether there is such a row: as long as it did, the compiler could not
// tell how many accesses were under way and waited, at the head of every row, for the row just requested as well.
// [4096,5120] bf16 with the residual, before / now: forward 32.4 / 29.9 us (5.6 TB/s; one workgroup per row behind a
// separate add 64 us), backward 42.5 / 35.4 and 4.6 for the sums (4.7 TB/s without the partial rows' 42 MB; 382 with the
// plain kernels, whose column sums ran on 80 workgroups).  [5824,7040] fp16 forward 66.9 / 56.2, [544,7616] fp32 21.6 / 15.6.
// The backward is as close to its arithmetic as to the memory: 200 operations a row and lane, two of them fp64 adds, ten
// waves on four SIMDs.  [12000,1003] fp32 37.6 + 41 us against 58.5 + 1121.
template <typename T, int N, bool UA>
__device__ __forceinline__ Raw<T, N> load_piece(const T *p) {
  Raw<T, N> r;
#pragma unroll
  for (int q = 0; q < N / Vec16<T>::n; ++q) {
    if constexpr (UA) {
      r.v[q] = load16_unaligned_stream(p + q * Vec16<T>::n);
    } else {
      r.v[q] = load16_stream(p + q * Vec16<T>::n);
    }
  }
  return r;
}
template <typename T, int N, bool UA>
__device__ __forceinline__ void store_piece(T *p, const float (&in)[N]) {
  constexpr int VN = Vec16<T>::n;
#pragma unroll
  for (int q = 0; q < N / VN; ++q) {
    Vec16<T> v;
#pragma unroll
    for (int k = 0; k < VN; ++k) v.e[k] = from_acc<T>(in[q * VN + k]);
    if constexpr (UA) {
      store16_unaligned_stream(p + q * VN, v);
    } else {
      store16_stream(p + q * VN, v);
    }
  }
}
template <typename T, int N>
__device__ __forceinline__ void store_piece(RowBuffer row, int offset, const float (&in)[N]) {
  constexpr int VN = Vec16<T>::n;
#pragma unroll
  for (int q = 0; q < N / VN; ++q) {
    Vec16<T> v;
#pragma unroll
    for (int k = 0; k < VN; ++k) v.e[k] = from_acc<T>(in[q * VN + k]);
    store16_stream(row, offset + q * 16, v);
  }
}
// One lane's share of a row: VPT vectors and, with UA, one single element.
template <typename T, int VN, int VPT, bool UA>
struct Share {
  Raw<T, VN> v[VPT];
  T e;
};
// Which columns a lane owns.
template <int VN, int VPT, bool UA>
struct Lanes {
  int at[VPT];   // first column of each vector (a lane without a vector re-reads the row's last one)
  bool has[VPT];
  template <typename T>
  __device__ __forceinline__ int offset(int j) const {  // in a RowBuffer
    return has[j] ? at[j] * (int)sizeof(T) : kOutside;
  }
  int ecol;      // the single element's column
  bool ehas;
  __device__ __forceinline__ Lanes(int C, int gw, int lane_in_group) {
    const int nvec = C / VN;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      const int idx = lane_in_group + kWave * gw * j;
      has[j] = idx < nvec;
      at[j] = (has[j] ? idx : nvec - 1) * VN;
      if (UA && nvec == 0) at[j] = 0;
    }
    const int tail = C - nvec * VN;
    ehas = UA && lane_in_group < tail;
    ecol = nvec * VN + (lane_in_group < tail ? lane_in_group : 0);
    if (ecol >= C) ecol = C - 1;
  }
};
template <typename T, int VN, int VPT, bool UA>
__device__ __forceinline__ void load_share(Share<T, VN, VPT, UA> &s, const T *row, const Lanes<VN, VPT, UA> &l,
                                           bool any_vec) {
  if (!UA || any_vec) {  // grid-uniform: with fewer than VN columns there is no vector to read
#pragma unroll
    for (int j = 0; j < VPT; ++j) s.v[j] = load_piece<T, VN, UA>(row + l.at[j]);
  }
  if constexpr (UA) s.e = row[l.ecol];
}

// the same of row `r` of whole aligned vectors: zeros where the lane has no vector, and past the last row
template <typename T, int VN, int VPT>
__device__ __forceinline__ void load_share(Share<T, VN, VPT, false> &s, const T *base, int64_t r, int64_t rows, int C,
                                           const Lanes<VN, VPT, false> &l) {
  const RowBuffer row = row_buffer(base + (r < rows ? r : 0) * C, r < rows ? C * (int)sizeof(T) : 0);
#pragma unroll
  for (int j = 0; j < VPT; ++j)
#pragma unroll
    for (int q = 0; q < VN / Vec16<T>::n; ++q) s.v[j].v[q] = load16_stream<T>(row, l.template offset<T>(j) + q * 16);
}

constexpr int kLnBlockMaxWaves = 16;

// Sum over a group's row; v[j] belongs to the lane's vector j.  Rows of 257 to 512 vectors (BY_LANE) have three
// plans, which all add in one order, so that they give the same bits: lane l's vectors l, l + 64, ... first, one after
// the other, then the lanes.  Other widths have one plan each: a wave's lanes first, then the waves.  Every wave
// of the workgroup must call it.  The caller alternates between two arrays, so one barrier is enough.
template <bool BY_LANE, int VPT>
__device__ __forceinline__ float row_sum(const float (&v)[VPT], int gw, int wave, int group, int lane, float *red) {
  if constexpr (BY_LANE) {
    const int n = gw * VPT;  // at most 8
    float *mine = red + group * n * kWave + lane;
#pragma unroll
    for (int j = 0; j < VPT; ++j) mine[(wave - group * gw + gw * j) * kWave] = v[j];
    lds_barrier();
    float part[8], t = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) part[i] = mine[(i < n ? i : 0) * kWave];
#pragma unroll
    for (int i = 0; i < 8; ++i) t += i < n ? part[i] : 0.f;
    return wave_reduce(t, SumOp{});
  }
  float t = v[0];
#pragma unroll
  for (int j = 1; j < VPT; ++j) t += v[j];
  if (gw == 1) return wave_reduce(t, SumOp{});  // workgroup-uniform
  t = wave_sum_in_last_lane(t);
  if (lane == kWave - 1) red[wave] = t;
  lds_barrier();
  const int w = lane % kLnBlockMaxWaves;
  const float r = red[group * gw + (w < gw ? w : 0)];
  return row16_sum(w < gw ? r : 0.f);
}

// A wave's number, where UNIFORM known to be the same for all of its lanes: rows then have scalar addresses and descriptors,
// and the statistics come by scalar loads.  Ragged rows of one fp32 vector a lane, and dx alone of one vector a lane, are the quicker
// without (fp32 [40000,65] with dresidual 22.6 us uniform, 18.9 by lane, forward [10000,300] 6.6 / 6.1, dx alone [6144,3] 4.35 /
// 3.8); the others not, as it takes a dozen registers (bf16 forward [4096,7001] 28.7 / 35.1, with the residual [4096,5001]
// 39.1 / 45.7).
template <bool UNIFORM>
__device__ __forceinline__ int block_wave() {
  const int wave = threadIdx.x >> 6;
  return UNIFORM ? __builtin_amdgcn_readfirstlane(wave) : wave;
}

template <typename TX, typename TY, typename TP, int VPT, bool HAS_RES, bool UA, bool BY_LANE>
__global__ __launch_bounds__(kLnBlockMaxWaves *kWave) void ln_fwd_block_kernel(
    const TX *x /* sum_out may be x: not restrict */, const TP *__restrict__ gamma, const TP *__restrict__ beta,
    TY *__restrict__ y, float *__restrict__ mean, float *__restrict__ rstd, int64_t rows, int C, float eps,
    const TX *res, TX *sum_out, int gw, int groups) {
  constexpr int VN = Vec16<TX>::n;
  __shared__ float red[2][kLnBlockMaxWaves * (BY_LANE ? VPT * kWave : 1)];
  const int lane = threadIdx.x & (kWave - 1), wave = block_wave<(!UA || VPT > 1 || sizeof(TX) == 2)>();
  const int group = wave / gw, lig = threadIdx.x - group * gw * kWave;
  const bool any_vec = C >= VN;
  const Lanes<VN, VPT, UA> own(C, gw, lig);
  const float fc = (float)C, inv_c = 1.0f / fc;
  const int64_t stride = (int64_t)gridDim.x * groups;
  const int64_t steps = (rows + stride - 1) / stride;  // the same for every group: they share barriers
  int64_t row = (int64_t)blockIdx.x * groups + group;

  // Two rows' registers: a row is requested as soon as the registers of the one two steps before it
  // are free, so that one row is on its way while another is worked on.
  struct Row {
    Share<TX, VN, VPT, UA> x, res;
  };
  auto fetch = [&](Row &d, int64_t r) {
    if constexpr (UA) {
      const int64_t at = (r < rows ? r : rows - 1) * C;
      load_share(d.x, x + at, own, any_vec);
      if constexpr (HAS_RES) load_share(d.res, res + at, own, any_vec);
    } else {
      load_share(d.x, x, r, rows, C, own);
      if constexpr (HAS_RES) load_share(d.res, res, r, rows, C, own);
    }
  };
  float g[VPT][VN], b[VPT][VN], ge = 0.f, be = 0.f;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
#pragma unroll
    for (int k = 0; k < VN; ++k) g[j][k] = b[j][k] = 0.f;
    if (own.has[j]) {
      if constexpr (UA) {
#pragma unroll
        for (int k = 0; k < VN; ++k) g[j][k] = to_acc(gamma[own.at[j] + k]);
        if (beta)
#pragma unroll
          for (int k = 0; k < VN; ++k) b[j][k] = to_acc(beta[own.at[j] + k]);
      } else {
        load_n<TP, VN>(gamma + own.at[j], g[j]);
        if (beta) load_n<TP, VN>(beta + own.at[j], b[j]);
      }
    }
  }
  if constexpr (UA) {
    ge = to_acc(gamma[own.ecol]);
    if (beta) be = to_acc(beta[own.ecol]);
  }
  Row even, odd;
  fetch(even, row);
  if (!UA || steps > 1) fetch(odd, row + stride);
  auto work = [&](Row &in, int64_t row) {
    Share<TX, VN, VPT, UA> &cur = in.x, &rcur = in.res;
    const bool row_ok = row < rows;
    const int64_t at = (row_ok ? row : 0) * C;
    const int y_bytes = row_ok ? C * (int)sizeof(TY) : 0;
    if constexpr (HAS_RES) {
      // cur = x + residual, one fp32 add and one rounding per element, as an add launch would give
#pragma unroll
      for (int j = 0; j < VPT; ++j) {
        Vec16<TX> sum;
#pragma unroll
        for (int k = 0; k < VN; ++k)
          sum.e[k] = from_acc<TX>(raw_get<TX, VN>(cur.v[j], k) + raw_get<TX, VN>(rcur.v[j], k));
        cur.v[j].v[0] = sum;
        if constexpr (UA) {
          if (own.has[j] && row_ok) store16_unaligned_stream(sum_out + at + own.at[j], sum);
        } else {
          store16_stream(row_buffer(sum_out + at, row_ok ? C * (int)sizeof(TX) : 0), own.template offset<TX>(j), sum);
        }
      }
      if constexpr (UA) {
        cur.e = from_acc<TX>(to_acc(cur.e) + to_acc(rcur.e));
        if (own.ehas && row_ok) sum_out[at + own.ecol] = cur.e;
      }
    }
    float s[VPT], q[VPT];
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      float t = 0.f;
#pragma unroll
      for (int k = 0; k < VN; ++k) t += raw_get<TX, VN>(cur.v[j], k);
      s[j] = own.has[j] ? t : 0.f;
    }
    if constexpr (UA) s[0] += own.ehas ? to_acc(cur.e) : 0.f;
    const float mu = over_columns(row_sum<BY_LANE>(s, gw, wave, group, lane, red[0]), fc, inv_c);
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      float t = 0.f;
#pragma unroll
      for (int k = 0; k < VN; ++k) {
        const float d = raw_get<TX, VN>(cur.v[j], k) - mu;
        t += d * d;
      }
      q[j] = own.has[j] ? t : 0.f;
    }
    if constexpr (UA) {
      const float d = to_acc(cur.e) - mu;
      q[0] += own.ehas ? d * d : 0.f;
    }
    const float rs = 1.0f / sqrtf(over_columns(row_sum<BY_LANE>(q, gw, wave, group, lane, red[1]), fc, inv_c) + eps);
    if constexpr (!UA) {
      const int64_t r = row_ok ? row : 0;
      const int first = lig == 0 ? 0 : kOutside, bytes = row_ok ? (int)sizeof(float) : 0;
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(mu), row_buffer(mean + r, bytes), first, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(rs), row_buffer(rstd + r, bytes), first, 0, 0);
#pragma unroll
      for (int j = 0; j < VPT; ++j) {
        float o[VN];
#pragma unroll
        for (int k = 0; k < VN; ++k) o[k] = (raw_get<TX, VN>(cur.v[j], k) - mu) * rs * g[j][k] + b[j][k];
        store_piece<TY, VN>(row_buffer(y + at, y_bytes), own.template offset<TY>(j), o);
      }
    } else if (row_ok) {
      if (lig == 0) {
        mean[row] = mu;
        rstd[row] = rs;
      }
#pragma unroll
      for (int j = 0; j < VPT; ++j) {
        if (own.has[j]) {
          float o[VN];
#pragma unroll
          for (int k = 0; k < VN; ++k) o[k] = (raw_get<TX, VN>(cur.v[j], k) - mu) * rs * g[j][k] + b[j][k];
          store_piece<TY, VN, UA>(y + at + own.at[j], o);
        }
      }
      if constexpr (UA) {
        if (own.ehas) y[at + own.ecol] = from_acc<TY>((to_acc(cur.e) - mu) * rs * ge + be);
      }
    }
  };
  if constexpr (UA) {
    for (int64_t it = 0; it < steps; it += 2, row += 2 * stride) {
      work(even, row);
      if (it + 2 < steps) fetch(even, row + 2 * stride);
      if (it + 1 < steps) {
        work(odd, row + stride);
        if (it + 3 < steps) fetch(odd, row + 3 * stride);
      }
    }
    return;
  }
  // Every step requests two rows, there or not, and the first step stands before the loop: what is under way at the
  // loop's head is then the same whichever way it was reached, and the compiler waits for exactly the row it needs.
  const auto step = [&] {
    work(even, row);
    __builtin_amdgcn_sched_barrier(0);  // neither row's work moves into the other's
    fetch(even, row + 2 * stride);
    __builtin_amdgcn_sched_barrier(0);
    work(odd, row + stride);
    __builtin_amdgcn_sched_barrier(0);
    fetch(odd, row + 3 * stride);
    __builtin_amdgcn_sched_barrier(0);
    row += 2 * stride;
  };
  if (steps > 1) {
    step();
    for (int64_t it = 3; it < steps; it += 2) step();
  }
  if (steps & 1) work(even, row);
}

// Backward of the same rows.  The column sums of a lane's own columns stay in registers over all the
// rows it visits, in double: they may span thousands of rows, and at full-rate fp64 the two adds per
// element cost no time next to the row's traffic.  The groups of a workgroup meet in the LDS, and one
// partial row leaves per workgroup, in the column order of ln_finalize_tile, in which a wave's LDS and global
// accesses are contiguous.  It is in double too, so that a sum is rounded once (`wide`); in fp32 only where the
// caller may keep partial rows for a later call (see block_two_calls).
// Whether a lane's next row fits the registers (128 at 16 waves a workgroup) next to its column sums,
// gamma and the current row: requested a row ahead where it does.
template <typename TDY, typename TX, typename TDX, int E, bool HAS_DP, bool HAS_DRES, bool UA>
constexpr bool bwd_block_prefetches() {
  const int row = E * (int)(sizeof(TDY) + sizeof(TX) + (HAS_DRES ? sizeof(TDX) : 0)) / 4;
  return (HAS_DP ? 4 * E : 0) + E + 2 * row <= (UA ? 60 : 70);
}
struct LnNoSide {};
template <typename TDY, typename TX, typename TDX, typename TP, int VPT, bool HAS_DX, bool HAS_DP, bool HAS_DRES,
          bool UA, bool DIRECT = false>
__global__ __launch_bounds__(kLnBlockMaxWaves *kWave) void ln_bwd_block_kernel(
    const TDY *__restrict__ dy, const TX *__restrict__ x, const float *__restrict__ mean,
    const float *__restrict__ rstd, const TP *__restrict__ gamma, TDX *dx /* may be dres */,
    void *__restrict__ partial, int wide, int64_t rows, int C, const TDX *dres, int gw, int groups,
    const std::conditional_t<DIRECT, LnPending, LnNoSide> side) {
  constexpr int VN = Vec16<TX>::n;
  static_assert(!DIRECT || !HAS_DP, "the launch's first workgroups take the column sums");
  constexpr bool PF = bwd_block_prefetches<TDY, TX, TDX, VPT * VN, HAS_DP, HAS_DRES, UA>();
  extern __shared__ double group_sums[];  // [groups][C] for the fold
  __shared__ float red[2][2][kLnBlockMaxWaves];
  if constexpr (DIRECT) {
    if ((int)blockIdx.x < side.blocks) {
      ln_columns_wide<TDY, TX, TP>(dy, x, mean, rstd, side, rows, blockIdx.x, C, group_sums);
      return;
    }
  }
  unsigned bid = blockIdx.x, nblocks = gridDim.x;
  if constexpr (DIRECT) {
    bid -= side.blocks;
    nblocks -= side.blocks;
  }
  const int lane = threadIdx.x & (kWave - 1), wave = block_wave<(!UA || VPT > 1 || (HAS_DP && sizeof(TX) == 2))>();
  const int group = wave / gw, lig = threadIdx.x - group * gw * kWave;
  const bool any_vec = C >= VN;
  const Lanes<VN, VPT, UA> own(C, gw, lig);
  const float inv_c = 1.0f / (float)C;
  const int64_t stride = (int64_t)nblocks * groups;
  const int64_t steps = (rows + stride - 1) / stride;
  int64_t row = (int64_t)bid * groups + group;

  struct Row {
    Share<TDY, VN, VPT, UA> dy;
    Share<TX, VN, VPT, UA> x;
    Share<TDX, VN, VPT, UA> res;
    float mu, rs;
  };
  auto fetch = [&](Row &d, int64_t r) {
    const int64_t rr = r < rows ? r : rows - 1;
    if constexpr (UA) {
      load_share(d.dy, dy + rr * C, own, any_vec);
      load_share(d.x, x + rr * C, own, any_vec);
      if constexpr (HAS_DRES) load_share(d.res, dres + rr * C, own, any_vec);
    } else {
      load_share(d.dy, dy, r, rows, C, own);
      load_share(d.x, x, r, rows, C, own);
      if constexpr (HAS_DRES) load_share(d.res, dres, r, rows, C, own);
    }
    d.mu = mean[rr];
    d.rs = rstd[rr];
  };
  double acc_g[VPT][VN], acc_b[VPT][VN], eacc_g = 0., eacc_b = 0.;
  float g[VPT][VN], ge = 0.f;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
#pragma unroll
    for (int k = 0; k < VN; ++k) {
      acc_g[j][k] = 0.;
      acc_b[j][k] = 0.;
      g[j][k] = 0.f;
    }
    if (HAS_DX && own.has[j]) {
      if constexpr (UA) {
#pragma unroll
        for (int k = 0; k < VN; ++k) g[j][k] = to_acc(gamma[own.at[j] + k]);
      } else {
        load_n<TP, VN>(gamma + own.at[j], g[j]);
      }
    }
  }
  if constexpr (UA && HAS_DX) {
    ge = to_acc(gamma[own.ecol]);
    ge = own.ehas ? ge : 0.f;
  }
  Row even, odd;  // as in the forward kernel, where both fit
  fetch(even, row);
  if (PF && (!UA || steps > 1)) fetch(odd, row + stride);

  int parity = 0;
  auto work = [&](Row &in, int64_t row) {
    Share<TDY, VN, VPT, UA> &dcur = in.dy;
    Share<TX, VN, VPT, UA> &xcur = in.x;
    Share<TDX, VN, VPT, UA> &rcur = in.res;
    const float mu = in.mu, rs = in.rs;
    const bool row_ok = row < rows;
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      const bool live = own.has[j] && row_ok;
      const float live_mu = live ? mu : 0.f, live_rs = live ? rs : 0.f;
#pragma unroll
      for (int k = 0; k < VN; ++k) {
        // zero both where there is no row or vector: 0 * inf would leave a NaN in the sums.  (A RowBuffer reads zeros there.)
        float xh, dv;
        if constexpr (UA) {
          xh = live ? (raw_get<TX, VN>(xcur.v[j], k) - mu) * rs : 0.f;
          dv = live ? raw_get<TDY, VN>(dcur.v[j], k) : 0.f;
        } else {
          xh = (raw_get<TX, VN>(xcur.v[j], k) - live_mu) * live_rs;
          dv = raw_get<TDY, VN>(dcur.v[j], k);
        }
        if constexpr (HAS_DP) {
          acc_g[j][k] += (double)(dv * xh);
          acc_b[j][k] += (double)dv;
        }
        if constexpr (HAS_DX) {
          const float gd = dv * g[j][k];
          s1 += gd;
          s2 = __builtin_fmaf(gd, xh, s2);
        }
      }
    }
    float exh = 0.f, edv = 0.f;
    if constexpr (UA) {
      const bool live = own.ehas && row_ok;
      exh = live ? (to_acc(xcur.e) - mu) * rs : 0.f;
      edv = live ? to_acc(dcur.e) : 0.f;
      if constexpr (HAS_DP) {
        eacc_g += (double)(edv * exh);
        eacc_b += (double)edv;
      }
      if constexpr (HAS_DX) {
        const float gd = edv * ge;
        s1 += gd;
        s2 = __builtin_fmaf(gd, exh, s2);
      }
    }
    if constexpr (HAS_DX) {
      if (gw > 1) {  // workgroup-uniform
        s1 = wave_sum_in_last_lane(s1);
        s2 = wave_sum_in_last_lane(s2);
        if (lane == kWave - 1) {
          red[parity][0][wave] = s1;
          red[parity][1][wave] = s2;
        }
        lds_barrier();
        const int w = lane % kLnBlockMaxWaves, from = group * gw + (w < gw ? w : 0);
        const float a = red[parity][0][from], c = red[parity][1][from];
        s1 = row16_sum(w < gw ? a : 0.f);
        s2 = row16_sum(w < gw ? c : 0.f);
        parity ^= 1;  // the other pair next time: one barrier per row is enough
      } else {
        s1 = wave_reduce(s1, SumOp{});
        s2 = wave_reduce(s2, SumOp{});
      }
      s1 *= inv_c;
      s2 *= inv_c;
      if (!UA || row_ok) {
        const RowBuffer out = row_buffer(dx + (row_ok ? row : 0) * C, row_ok ? C * (int)sizeof(TDX) : 0);
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
          if (!UA || own.has[j]) {
            float o[VN];
#pragma unroll
            for (int k = 0; k < VN; ++k) {
              const float xh = (raw_get<TX, VN>(xcur.v[j], k) - mu) * rs;
              const float dv = raw_get<TDY, VN>(dcur.v[j], k);
              o[k] = rs * __builtin_fmaf(-xh, s2, __builtin_fmaf(dv, g[j][k], -s1));
              if constexpr (HAS_DRES) o[k] = round_through<TDX>(o[k]) + raw_get<TDX, VN>(rcur.v[j], k);
            }
            if constexpr (UA) {
              store_piece<TDX, VN, UA>(dx + row * C + own.at[j], o);
            } else {
              store_piece<TDX, VN>(out, own.template offset<TDX>(j), o);
            }
          }
        }
        if constexpr (UA) {
          if (own.ehas) {
            float o = rs * __builtin_fmaf(-exh, s2, __builtin_fmaf(edv, ge, -s1));
            if constexpr (HAS_DRES) o = round_through<TDX>(o) + to_acc(rcur.e);
            dx[row * C + own.ecol] = from_acc<TDX>(o);
          }
        }
      }
    }
  };
  if constexpr (UA && PF) {
    for (int64_t it = 0; it < steps; it += 2, row += 2 * stride) {
      work(even, row);
      if (it + 2 < steps) fetch(even, row + 2 * stride);
      if (it + 1 < steps) {
        work(odd, row + stride);
        if (it + 3 < steps) fetch(odd, row + 3 * stride);
      }
    }
  } else if constexpr (PF) {
    const auto step = [&] {  // as in the forward kernel
      work(even, row);
      __builtin_amdgcn_sched_barrier(0);  // neither row's work moves into the other's
      fetch(even, row + 2 * stride);
      __builtin_amdgcn_sched_barrier(0);
      work(odd, row + stride);
      __builtin_amdgcn_sched_barrier(0);
      fetch(odd, row + 3 * stride);
      __builtin_amdgcn_sched_barrier(0);
      row += 2 * stride;
    };
    if (steps > 1) {
      step();
      for (int64_t it = 3; it < steps; it += 2) step();
    }
    if (steps & 1) work(even, row);
  } else {
    for (int64_t it = 0; it < steps; ++it, row += stride) {
      work(even, row);
      if (it + 1 < steps) fetch(even, row + stride);
    }
  }

  if constexpr (HAS_DP) {
    const int nvec = C / VN;
    // one group: its registers are the partial row ([4096,5120] bf16 42.4 us against 44.1 through the LDS; where
    // four vectors a lane spill anyway, [300,16384] fp32, 71 against 60)
    if (VPT <= 2 && groups == 1 && wide) {
      double *out = (double *)partial + (int64_t)blockIdx.x * 2 * C;
#pragma unroll
      for (int j = 0; j < VPT; ++j) {
        if (own.has[j]) {
#pragma unroll
          for (int k = 0; k < VN; ++k) {
            out[k * nvec + lig + kWave * gw * j] = acc_g[j][k];
            out[C + k * nvec + lig + kWave * gw * j] = acc_b[j][k];
          }
        }
      }
      if (UA && own.ehas) {
        out[own.ecol] = eacc_g;
        out[C + own.ecol] = eacc_b;
      }
      return;
    }
#pragma unroll
    for (int which = 0; which < 2; ++which) {
      double *mine = group_sums + (size_t)group * C;
#pragma unroll
      for (int j = 0; j < VPT; ++j) {
        if (own.has[j]) {
#pragma unroll
          for (int k = 0; k < VN; ++k) mine[k * nvec + lig + kWave * gw * j] = which == 0 ? acc_g[j][k] : acc_b[j][k];
        }
      }
      if (UA && own.ehas) mine[own.ecol] = which == 0 ? eacc_g : eacc_b;
      lds_barrier();
      const int64_t at = ((int64_t)blockIdx.x * 2 + which) * C;
      for (int c = threadIdx.x; c < C; c += blockDim.x) {
        double t = 0.;
        for (int w = 0; w < groups; ++w) t += group_sums[(size_t)w * C + c];
        if (wide) {
          ((double *)partial)[at + c] = t;
        } else {
          ((float *)partial)[at + c] = (float)t;
        }
      }
      if (which == 0) lds_barrier();
    }
  }
}

// The column sums as a launch of their own: grid 2 * ceil(C/32) workgroups of 32 x 16 threads, even
// ones dgamma, odd ones dbeta (the same tiles, in the same order of additions, as the pending
// form inside the row kernel's launch).
template <typename TP, typename A, typename P>
__global__ __launch_bounds__(kLnFinCols *kLnFinRows) void ln_bwd_finalize_kernel(
    const P *__restrict__ partial, int nparts, TP *__restrict__ dgamma, TP *__restrict__ dbeta,
    int C, int vn, int accumulate) {
  __shared__ A sub[kLnFinRows * kLnFinCols];
  const LnPending pend{partial, dgamma, dbeta, nparts, accumulate, (int)gridDim.x};
  ln_finalize_pending<TP, kLnFinCols * kLnFinRows, A, P>(pend, blockIdx.x, C, vn, sub, threadIdx.x);
}

// ------------------------------------------------------ elementwise add
// out = a + b, one fp32 (fp64) add and one rounding per element; out may be a or b.
constexpr int kAddUnroll = 2;  // 16-byte vectors per lane, all requested before the first use

template <typename T>
__global__ __launch_bounds__(kLnThreads) void ew_add_kernel(const T *a, const T *b, T *out, int64_t n,
                                                            bool vec_ok) {
  constexpr int VN = Vec16<T>::n;
  using U = typename Acc<T>::type;
  constexpr int64_t kChunk = (int64_t)kLnThreads * kAddUnroll * VN;
  const int64_t begin = (int64_t)blockIdx.x * kChunk;
  const int64_t end = begin + kChunk < n ? begin + kChunk : n;
  if (vec_ok && end - begin == kChunk) {
    Vec16<T> va[kAddUnroll], vb[kAddUnroll];
#pragma unroll
    for (int u = 0; u < kAddUnroll; ++u) {
      const int64_t off = begin + ((int64_t)u * kLnThreads + threadIdx.x) * VN;
      va[u] = load16_stream(a + off);
      vb[u] = load16_stream(b + off);
    }
#pragma unroll
    for (int u = 0; u < kAddUnroll; ++u) {
      const int64_t off = begin + ((int64_t)u * kLnThreads + threadIdx.x) * VN;
      Vec16<T> vo;
#pragma unroll
      for (int k = 0; k < VN; ++k) vo.e[k] = from_acc<T>((U)(to_acc(va[u].e[k]) + to_acc(vb[u].e[k])));
      store16(out + off, vo);  // read again by the kernel that follows: keep it cached
    }
    return;
  }
  for (int64_t i = begin + threadIdx.x; i < end; i += kLnThreads)
    out[i] = from_acc<T>((U)(to_acc(a[i]) + to_acc(b[i])));
}

template <typename T>
int launch_add(const void *a, const void *b, void *out, int64_t n, hipStream_t s) {
  if (n <= 0) return CS_OK;
  const bool vec_ok = is_aligned16(a) && is_aligned16(b) && is_aligned16(out);
  const int64_t blocks = ceil_div(n, (int64_t)kLnThreads * kAddUnroll * Vec16<T>::n);
  if (blocks > 0x7fffffffLL) return CS_ERR_TOO_LARGE;
  ew_add_kernel<T><<<dim3((unsigned)blocks), dim3(kLnThreads), 0, s>>>((const T *)a, (const T *)b, (T *)out, n,
                                                                      vec_ok);
  return launch_status();
}

int launch_add_dtype(int dtype, const void *a, const void *b, void *out, int64_t n, hipStream_t s) {
  switch (dtype) {
    case CS_F32: return launch_add<float>(a, b, out, n, s);
    case CS_F64: return launch_add<double>(a, b, out, n, s);
    case CS_F16: return launch_add<f16_t>(a, b, out, n, s);
    case CS_BF16: return launch_add<bf16_t>(a, b, out, n, s);
  }
  return CS_ERR_UNSUPPORTED;
}

// ------------------------------------------------------------ general path
// One workgroup per row, any C, any alignment, fp64 included.
template <typename TX, typename TY, typename TP>
__global__ __launch_bounds__(kLnThreads) void ln_fwd_general_kernel(
    const TX *__restrict__ x, const TP *__restrict__ gamma, const TP *__restrict__ beta,
    TY *__restrict__ y, typename Acc<TX>::type *__restrict__ mean,
    typename Acc<TX>::type *__restrict__ rstd, int64_t rows, int64_t C, typename Acc<TX>::type eps) {
  using U = typename Acc<TX>::type;
  __shared__ U scratch[kLnThreads / kWave];
  const int64_t row = row_of_grid();
  if (row >= rows) return;
  const TX *xr = x + row * C;
  U s = 0;
  for (int64_t c = threadIdx.x; c < C; c += kLnThreads) s += to_acc(xr[c]);
  const U mu = block_reduce(s, SumOp{}, (U)0, scratch) / (U)C;
  U q = 0;
  for (int64_t c = threadIdx.x; c < C; c += kLnThreads) {
    const U d = to_acc(xr[c]) - mu;
    q += d * d;
  }
  const U var = block_reduce(q, SumOp{}, (U)0, scratch) / (U)C;
  const U rs = (U)1 / sqrt(var + eps);
  if (threadIdx.x == 0) {
    mean[row] = mu;
    rstd[row] = rs;
  }
  for (int64_t c = threadIdx.x; c < C; c += kLnThreads) {
    const U bb = beta ? (U)to_acc(beta[c]) : (U)0;
    y[row * C + c] = from_acc<TY>((U)((to_acc(xr[c]) - mu) * rs * (U)to_acc(gamma[c]) + bb));
  }
}

template <typename TDY, typename TX, typename TDX, typename TP>
__global__ __launch_bounds__(kLnThreads) void ln_bwd_dx_general_kernel(
    const TDY *__restrict__ dy, const TX *__restrict__ x,
    const typename Acc<TX>::type *__restrict__ mean,
    const typename Acc<TX>::type *__restrict__ rstd, const TP *__restrict__ gamma,
    TDX *__restrict__ dx, int64_t rows, int64_t C, const TDX *__restrict__ dres) {
  using U = typename Acc<TX>::type;
  __shared__ U scratch[kLnThreads / kWave];
  const int64_t row = row_of_grid();
  if (row >= rows) return;
  const U mu = mean[row], rs = rstd[row];
  U s1 = 0, s2 = 0;
  for (int64_t c = threadIdx.x; c < C; c += kLnThreads) {
    const U gd = (U)to_acc(dy[row * C + c]) * (U)to_acc(gamma[c]);
    const U xh = ((U)to_acc(x[row * C + c]) - mu) * rs;
    s1 += gd;
    s2 += gd * xh;
  }
  s1 = block_reduce(s1, SumOp{}, (U)0, scratch) / (U)C;
  s2 = block_reduce(s2, SumOp{}, (U)0, scratch) / (U)C;
  for (int64_t c = threadIdx.x; c < C; c += kLnThreads) {
    const U gd = (U)to_acc(dy[row * C + c]) * (U)to_acc(gamma[c]);
    const U xh = ((U)to_acc(x[row * C + c]) - mu) * rs;
    TDX o = from_acc<TDX>((U)(rs * (gd - s1 - xh * s2)));
    if (dres) o = from_acc<TDX>((U)(round_through<TDX>((U)to_acc(o)) + (U)to_acc(dres[row * C + c])));
    dx[row * C + c] = o;
  }
}

// grid ceil(C/64) blocks of (64, 4): thread (cx, ry) walks rows ry, ry+4, ...  A thread adds
// rows/4 terms one after the other, so the running sums are kept in double: in float the
// rounding of a sum of thousands of O(1) terms reaches several 1e-5.
template <typename TDY, typename TX, typename TP>
__global__ __launch_bounds__(256) void ln_bwd_param_general_kernel(
    const TDY *__restrict__ dy, const TX *__restrict__ x,
    const typename Acc<TX>::type *__restrict__ mean,
    const typename Acc<TX>::type *__restrict__ rstd, TP *__restrict__ dgamma,
    TP *__restrict__ dbeta, int64_t rows, int64_t C, int accumulate) {
  using U = typename Acc<TX>::type;
  __shared__ double sg[4][64], sb[4][64];
  const int64_t col = (int64_t)blockIdx.x * 64 + threadIdx.x;
  double ag = 0, ab = 0;
  if (col < C) {
    for (int64_t r = threadIdx.y; r < rows; r += 4) {
      const U d = to_acc(dy[r * C + col]);
      ag += (double)(d * (((U)to_acc(x[r * C + col]) - mean[r]) * rstd[r]));
      ab += (double)d;
    }
  }
  sg[threadIdx.y][threadIdx.x] = ag;
  sb[threadIdx.y][threadIdx.x] = ab;
  __syncthreads();
  if (threadIdx.y == 0 && col < C) {
    double tg = 0, tb = 0;
    for (int r = 0; r < 4; ++r) {
      tg += sg[r][threadIdx.x];
      tb += sb[r][threadIdx.x];
    }
    if (dgamma) {
      if (accumulate) tg += (double)to_acc(dgamma[col]);
      dgamma[col] = from_acc<TP>((typename Acc<TP>::type)tg);
    }
    if (dbeta) {
      if (accumulate) tb += (double)to_acc(dbeta[col]);
      dbeta[col] = from_acc<TP>((typename Acc<TP>::type)tb);
    }
  }
}

// ---------------------------------------------------------------- dispatch
struct FastPlan {
  int vpl = 0;       // 0: not eligible
  int fwd_rows = 1;  // rows a wave normalises per step, forward
};
// x vectors per lane needed for C columns of x_dtype when a wave owns whole rows; those kernels are
// instantiated for 1, 2 and 4.  A fifth to eighth vector per lane: the forward has both kinds of plan (see
// wave_per_row8); in the backward several waves per row are faster ([4096,3072] bf16 with the residual 27.0 us
// against 37.0, [8192,2048] fp32 50.2 / 73.9, without it [4096,4096] bf16 27.3 / 28.3).
FastPlan fast_plan(int64_t C, int x_dtype) {
  FastPlan p;
  const int vn = 16 / (int)dtype_size(x_dtype);
  if (x_dtype == CS_F64 || C <= 0 || C % vn != 0) return p;
  const int64_t nvec = C / vn;
  const int64_t per_lane = ceil_div(nvec, (int64_t)kWave);
  if (per_lane <= 1) {
    p.vpl = 1;
    p.fwd_rows = CS_LN_FWD_ROWS_VPL1;
  } else if (per_lane <= 2) {
    p.vpl = 2;
    p.fwd_rows = CS_LN_FWD_ROWS_VPL2;
  } else if (per_lane <= 4) {
    p.vpl = 4;
    p.fwd_rows = CS_LN_FWD_ROWS_VPL4;
  }
  return p;
}

// Grid caps: beyond these the waves loop over rows (with prefetch) instead of
// the grid growing, which keeps the parameters in registers for many rows
// and bounds the number of partial rows the backward pass leaves behind.
#ifndef CS_LN_FWD_MAX_BLOCKS
#define CS_LN_FWD_MAX_BLOCKS 512
#endif
constexpr int kLnFwdMaxBlocks = CS_LN_FWD_MAX_BLOCKS;
constexpr int kLnBwdMaxBlocks = CS_LN_BWD_MAX_BLOCKS;

int ln_blocks(int64_t rows, int rows_per_wave, int cap, int threads = kLnThreads) {
  const int64_t rows_per_block = (int64_t)(threads / kWave) * rows_per_wave;
  const int64_t b = ceil_div(rows, rows_per_block);
  return (int)(b < cap ? b : cap);
}

// Forward: 512 workgroups of 4 waves, the two waves per SIMD that most of these kernels' registers allow: of twice as
// many the second half starts when the first has ended, asks for its parameters again and ends with a part-filled
// step.  us per call, 1024 / 512 workgroups: bf16 [16384,768] with the residual 18.9 / 17.5, [16384,512] 14.1 / 12.3,
// fp16 [16384,640] 21.5 / 17.1; without it [8192,1600] 13.6 / 11.4, [16384,1024] 15.4 / 13.8, [5000,3072] 14.5 / 13.0.
// 1024 still, us with them / with 512,
// * without the residual: up to 64 vectors, whose registers let more waves in (bf16 [40000,320] 13.5 / 16.3, fp32 [20000,160]
//   6.9 / 7.7, [50000,256] 11.3 / 12.9), fp32 up to 96 ([20000,320] 8.4 / 10.4, [20000,384] 9.4 / 11.2), and where 512 would make a second
//   step less than half full of fp32 rows ([5000,1024] 7.6 / 8.2, [9000,448] 6.9 / 7.5, [2100,1280] 5.5 / 5.9) or of 65 to 96
//   vectors (bf16 [9000,768] 7.0 / 7.5; from a step and a half on 512 are 10% the quicker);
// * with it: up to 64 vectors of fp32 ([20000,160] 9.3 / 10.5) and of 16 bits up to 14336 rows ([9000,512] bf16 8.9 / 9.8, fp16
//   10.8 / 11.8; but [16384,512] 13.6 / 11.9, 15.1 / 13.2), up to 128 (fp16 64) from 20481 to 32768 rows, where three or four steps
//   of 512 are more than two of 1024 (by 2-13%), and fp32 rows of more than 384 from 10241 rows on ([14600,2048] 77 / 85).
int fwd_blocks(int64_t rows, int rows_per_wave, int64_t nvec, bool residual, int x_dtype) {
  const int64_t step = (int64_t)kLnFwdMaxBlocks * (kLnThreads / kWave) * rows_per_wave;
  const bool fp32 = x_dtype == CS_F32;
  bool twice = nvec <= kHalf;
  if (!residual) {
    const bool halves = nvec > kWave && nvec <= 3 * kHalf;
    twice |= nvec <= kWave || (fp32 && halves) || ((fp32 || halves) && rows * 2 <= step * 3);
  } else {
    twice |= nvec <= kWave && (fp32 || rows <= 14336);
    twice |= nvec <= (x_dtype == CS_F16 ? 1 : 2) * kWave && rows > 20480 && rows <= 32768;
    twice |= fp32 && nvec > 6 * kWave && rows > 10240;
  }
  return ln_blocks(rows, rows_per_wave, twice ? 2 * kLnFwdMaxBlocks : kLnFwdMaxBlocks);
}

// Two vectors per lane and the residual: rows a wave normalises per step.  Two, so that the last step of the 512
// workgroups is seldom nearly empty ([5000,1024] bf16 10.9 us with four, 9.4 with two; [10000,1024] 16.1 / 15.4);
// four where one workgroup per CU then holds them all ([2500,512] fp32 6.0 us with two, 5.4 with four) or where their
// steps are more than three quarters full ([8192,1024] bf16 11.9 / 11.5, [16384,1024] 24.5 / 22.9).  fp16 takes its sums
// through more registers: with four rows 262 of them, one wave per SIMD ([8192,1024] 13.4 us with two, 22.5 with four).
// Four vectors per lane: one row (bf16 [3000,1600] 10.2 us with two, 8.7 with one, [16384,2048] 48.0 / 46.3, fp16
// [8192,1536] 34.6 / 19.8).
int add_rows_vpl2(int64_t rows, bool fp16) {
  const int64_t one_each = 256 * (kLnThreads / kWave) * 4, step = 2 * one_each;
  if (fp16) return 2;
  return rows <= one_each || rows * 4 > ceil_div(rows, step) * step * 3 ? 4 : 2;
}

// Rows on several waves (ln_fwd_block_kernel, ln_bwd_block_kernel): everything the row-per-wave plans
// do not take, up to 16 elements per lane of 1024 lanes, at any width and alignment.
struct BlockPlan {
  int vpt = 0;                      // 16-byte vectors per lane; 0: not eligible
  int gw = 0, groups = 0, blocks = 0;  // waves per row, rows side by side in a workgroup, workgroups
};
// the fold of the widest row: 16 elements per lane and a tail of fewer than 8
constexpr size_t kLnBlockFoldLds = ((size_t)16 * kLnBlockMaxWaves * kWave + 7) * sizeof(double);
BlockPlan block_plan(int64_t rows, int64_t C, int x_dtype, bool backward, bool residual, bool whole_vectors = false) {
  BlockPlan p;
  if (x_dtype == CS_F64 || C <= 0) return p;
  const int vn = 16 / (int)dtype_size(x_dtype);
  const int64_t nvec = C >= vn ? C / vn : 1;
  // One vector per lane: [4096,5120] bf16 backward 41.6 us against 58.2 with two (registers), forward
  // with the residual 31.9 against 38.1.  A forward without residual has half the loads in flight
  // per row, and two pay where the row then still has two waves or more: [4096,4099] 13.9 against 15.6, but
  // [4096,5120] 23.1 against 20.5.
  int vpt = !backward && !residual && nvec > 4 * kWave && nvec <= 8 * kWave ? 2 : 1;
  while (ceil_div(nvec, (int64_t)kWave * vpt) > kLnBlockMaxWaves) vpt *= 2;
  if (vpt * vn > 16) return p;
  p.vpt = vpt;
  p.gw = (int)ceil_div(nvec, (int64_t)kWave * vpt);
  // Forward with the residual, whole vectors: one workgroup of up to 12 waves per CU, whose loads are never waited for
  // ahead of time (see ln_fwd_block_kernel); 512 workgroups of 8 waves put more under way than the memory likes
  // ([4096,5120] bf16 30.9 us against 29.9, [16384,2304] 57.0 / 52.5, [16384,3584] 85.5 / 78.3).  Not where those make one
  // step: [300,2304] 4.2 against 4.8.  Nor fp16 of up to 8 waves, whose conversions want more of them: [4096,3584] 22.5 us
  // on 512, 27.7 on 256, [8192,4096] 49.1 / 54.1.
  const bool even_flow = !backward && residual && whole_vectors &&
                         (p.gw > kLnBlockMaxWaves / 2 || (rows > 512 && x_dtype != CS_F16));
  // Backward: as many rows side by side as 16 waves hold, so that one workgroup per CU, hence 256
  // partial rows, keeps the CU busy ([12000,1003] fp32 40.3 us against 43.3 with 8 waves; 512
  // workgroups 41.2, and [4096,5120] bf16 49.9 against 41.9).  Forward: 8 waves and two workgroups
  // per CU ([4096,1001] bf16 9.7 us against 11.4 with 16 waves, [4096,5120] 32.3 against 37.5 with 1024
  // workgroups).
  int groups = (backward ? kLnBlockMaxWaves : even_flow ? 12 : kLnBlockMaxWaves / 2) / p.gw;
  // Fewer side by side where there are not rows enough for every CU: [300,1003] bf16 backward 8.3 us against 8.5,
  // [64,1003] 6.8 against 8.7; up to three stay ([300,4099] 16.2 against 17.6, [300,2056] 9.9 / 11.8).  Rounded down in
  // the backward, so that the number of partial rows grows with the rows: a buffer for a long batch holds a short one's.
  if (!backward) {
    const int64_t per_cu = even_flow ? rows / 256 : ceil_div(rows, (int64_t)256);
    if (groups > per_cu) groups = (int)per_cu;
  } else if (groups > 3 && groups > rows / 256) {
    groups = (int)(rows / 256);
  }
  if (groups < 1) groups = 1;
  while (backward && groups > 1 && (size_t)groups * C * sizeof(double) > kLnBlockFoldLds) --groups;
  p.groups = groups;
  const int cap = backward || even_flow ? 256 : 512;
  const int64_t b = ceil_div(rows, (int64_t)p.groups);
  p.blocks = (int)(b < cap ? b : cap);
  return p;
}

// Forward rows that ln_fwd_few_kernel takes: until its waves, one step each, are more than the chip holds at once,
// which comes the earlier the more vectors a lane loads.  us per call, ln_fwd_rows_kernel / this one: bf16 [77,768] 3.6
// / 2.9, with the residual 4.2 / 3.1, [1536,768] 5.2 / 4.2, [2048,768] 5.3 / 4.6, [3072,768] 5.6 / 6.3; [512,1024] 5.8 /
// 3.4, [2048,1024] 6.2 / 4.7, [3072,1024] 6.7 / 6.7; [1024,1600] 5.8 / 4.9, [1536,1600] 6.2 / 6.9; [4096,64] 4.3 / 3.4,
// without it [4096,512] 4.3 / 4.0, [8192,320] 5.0 / 5.2, [3072,768] 4.5 / 4.3, [4096,768] 4.7 / 4.8.
bool few_forward_rows(int64_t rows, int vpl, bool halves, bool residual) {
  const int64_t loads = rows * vpl * (residual ? 2 : 1);
  return halves ? loads <= 9216 : loads <= 8192 && rows <= 4096;
}

// Forward of 257 to 512 whole vectors: a wave per row with eight vectors a lane, or several waves per row (the
// same bits).  The several waves have more loads in flight where there are few rows, and where the residual
// doubles a row's loads; in between their last step of 512 workgroups is nearly empty.  Wave per row / several
// waves, us per call: bf16 [300,3072] 4.4 / 4.0, [600,3072] 4.6 / 5.1, [12000,2304] 24.7 / 28.4; with the residual
// [300,3072] 5.4 / 4.7, [1024,3072] 6.4 / 7.8, [1500,3072] 10.8 / 10.5, [12000,2304] 51.5 / 44.5.  fp32, rows half as
// long: [300,1280] 3.5 / 3.7, [3000,1280] 6.4 / 9.4; with the residual [300,1280] 4.2 / 3.9, [600,1280] 4.4 / 5.9,
// [12000,1280] 45.5 / 46.4.
bool wave_per_row8(int64_t rows, int64_t C, int x_dtype, bool residual) {
  if (x_dtype == CS_F64 || C <= 0) return false;
  const int vn = 16 / (int)dtype_size(x_dtype);
  if (C % vn != 0 || C / vn <= 4 * kWave || C / vn > 8 * kWave) return false;
  if (x_dtype == CS_F32) return !residual || rows > 512;
  return rows > 512 && (!residual || rows <= 1024);
}

template <typename TX, typename TY, typename TP>
int fwd_typed(const void *x, const void *gamma, const void *beta, void *y, void *mean, void *rstd,
              int64_t rows, int64_t C, double eps, bool aligned, int x_dtype, const void *res,
              void *sum_out, hipStream_t s) {
  const FastPlan p = aligned ? fast_plan(C, x_dtype) : FastPlan{};
  if constexpr (!std::is_same_v<TX, double>) {
    if (p.vpl != 0) {
      // rows of up to 32 vectors, and of 65 to 96 (C = 768 at 16 bit), go two to a wave: no lane
      // slot stays empty
      const int64_t nvec = C / Vec16<TX>::n;
      const int half_vpl = !CS_LN_FWD_HALF ? 0 : nvec <= kHalf ? 1 : (nvec > kWave && nvec <= 3 * kHalf) ? 3 : 0;
      if (few_forward_rows(rows, half_vpl != 0 ? half_vpl : p.vpl, half_vpl != 0, res != nullptr)) {
#define CS_LN_FWD_FEW(VPL, HAS_RES, LPR)                                                                              \
  ln_fwd_few_kernel<TX, TY, TP, VPL, HAS_RES, LPR>                                                                    \
      <<<dim3((unsigned)ceil_div(rows, (int64_t)(kWave / LPR))), dim3(kWave), 0, s>>>(                                \
          (const TX *)x, (const TP *)gamma, (const TP *)beta, (TY *)y, (float *)mean, (float *)rstd, rows, (int)C,    \
          (float)eps, (const TX *)res, (TX *)sum_out)
#define CS_LN_FWD_FEW2(VPL, LPR)      \
  if (res) {                          \
    CS_LN_FWD_FEW(VPL, true, LPR);    \
  } else {                            \
    CS_LN_FWD_FEW(VPL, false, LPR);   \
  }
        if (half_vpl == 1) {
          CS_LN_FWD_FEW2(1, kHalf)
        } else if (half_vpl == 3) {
          CS_LN_FWD_FEW2(3, kHalf)
        } else if (p.vpl == 1) {
          CS_LN_FWD_FEW2(1, kWave)
        } else if (p.vpl == 2) {
          CS_LN_FWD_FEW2(2, kWave)
        } else {
          CS_LN_FWD_FEW2(4, kWave)
        }
#undef CS_LN_FWD_FEW2
#undef CS_LN_FWD_FEW
        return launch_status();
      }
      if (half_vpl != 0) {
        const int groups = res ? (half_vpl == 1 ? CS_LN_ADD_ROWS_H1 : CS_LN_ADD_ROWS_H3)
                               : (half_vpl == 1 ? CS_LN_FWD_ROWS_H1 : CS_LN_FWD_ROWS_H3);
        const dim3 grid((unsigned)fwd_blocks(rows, 2 * groups, nvec, res != nullptr, x_dtype)),
            block(kLnThreads);
#define CS_LN_FWD_H(VPL, R, HAS_RES)                                                                 \
  ln_fwd_rows_kernel<TX, TY, TP, VPL, R, CS_LN_FWD_PF, HAS_RES, kHalf><<<grid, block, 0, s>>>(       \
      (const TX *)x, (const TP *)gamma, (const TP *)beta, (TY *)y, (float *)mean, (float *)rstd, rows, \
      (int)C, (float)eps, (const TX *)res, (TX *)sum_out)
        if (res && half_vpl == 1) {
          CS_LN_FWD_H(1, CS_LN_ADD_ROWS_H1, true);
        } else if (res) {
          CS_LN_FWD_H(3, CS_LN_ADD_ROWS_H3, true);
        } else if (half_vpl == 1) {
          CS_LN_FWD_H(1, CS_LN_FWD_ROWS_H1, false);
        } else {
          CS_LN_FWD_H(3, CS_LN_FWD_ROWS_H3, false);
        }
#undef CS_LN_FWD_H
        return launch_status();
      }
      // with the residual stream a wave holds two inputs per row: fewer rows per step
      constexpr bool kFp16 = std::is_same_v<TX, f16_t>;
      const int r_rows = res ? (p.vpl == 1   ? CS_LN_ADD_ROWS_VPL1
                                : p.vpl == 2 ? add_rows_vpl2(rows, kFp16)
                                             : CS_LN_ADD_ROWS_VPL4)
                             : p.fwd_rows;
      const dim3 grid((unsigned)fwd_blocks(rows, r_rows, nvec, res != nullptr, x_dtype)), block(kLnThreads);
#define CS_LN_FWD(VPL, R, HAS_RES)                                                          \
  ln_fwd_rows_kernel<TX, TY, TP, VPL, R, CS_LN_FWD_PF, HAS_RES><<<grid, block, 0, s>>>(     \
      (const TX *)x, (const TP *)gamma, (const TP *)beta, (TY *)y, (float *)mean,           \
      (float *)rstd, rows, (int)C, (float)eps, (const TX *)res, (TX *)sum_out)
      if (res) {
        if (p.vpl == 1) {
          CS_LN_FWD(1, CS_LN_ADD_ROWS_VPL1, true);
        } else if (p.vpl == 2 && r_rows == 2) {
          CS_LN_FWD(2, 2, true);
        } else if (p.vpl == 2) {
          if constexpr (!kFp16) CS_LN_FWD(2, 4, true);
        } else {
          CS_LN_FWD(4, CS_LN_ADD_ROWS_VPL4, true);
        }
      } else if (p.vpl == 1) {
        CS_LN_FWD(1, CS_LN_FWD_ROWS_VPL1, false);
      } else if (p.vpl == 2) {
        CS_LN_FWD(2, CS_LN_FWD_ROWS_VPL2, false);
      } else {
        CS_LN_FWD(4, CS_LN_FWD_ROWS_VPL4, false);
      }
#undef CS_LN_FWD
      return launch_status();
    }
  }
  if constexpr (!std::is_same_v<TX, double>) {
    if (aligned && wave_per_row8(rows, C, x_dtype, res != nullptr)) {
      const dim3 grid((unsigned)fwd_blocks(rows, 1, C / Vec16<TX>::n, res != nullptr, x_dtype)), block(kLnThreads);
      if (res) {
        ln_fwd_rows_kernel<TX, TY, TP, 8, 1, CS_LN_FWD_PF, true><<<grid, block, 0, s>>>(
            (const TX *)x, (const TP *)gamma, (const TP *)beta, (TY *)y, (float *)mean, (float *)rstd, rows, (int)C,
            (float)eps, (const TX *)res, (TX *)sum_out);
      } else {
        ln_fwd_rows_kernel<TX, TY, TP, 8, 1, CS_LN_FWD_PF, false><<<grid, block, 0, s>>>(
            (const TX *)x, (const TP *)gamma, (const TP *)beta, (TY *)y, (float *)mean, (float *)rstd, rows, (int)C,
            (float)eps, nullptr, nullptr);
      }
      return launch_status();
    }
    const bool ua = !aligned || C % Vec16<TX>::n != 0;
    const BlockPlan b = block_plan(rows, C, x_dtype, false, res != nullptr, !ua);
    if (b.vpt != 0) {
      const dim3 grid((unsigned)b.blocks), block((unsigned)(b.gw * b.groups * kWave));
      // rows of 257 to 512 vectors: see row_sum
      const bool by_lane = C / Vec16<TX>::n > 4 * kWave && C / Vec16<TX>::n <= 8 * kWave;
#define CS_LN_FWD_B(VPT, HAS_RES, UA, BY_LANE)                                                         \
  ln_fwd_block_kernel<TX, TY, TP, VPT, HAS_RES, UA, BY_LANE><<<grid, block, 0, s>>>(                    \
      (const TX *)x, (const TP *)gamma, (const TP *)beta, (TY *)y, (float *)mean, (float *)rstd, rows, \
      (int)C, (float)eps, (const TX *)res, (TX *)sum_out, b.gw, b.groups)
#define CS_LN_FWD_B2(VPT, BY_LANE)                    \
  if (res && ua) {                                    \
    CS_LN_FWD_B(VPT, true, true, BY_LANE);            \
  } else if (res) {                                   \
    CS_LN_FWD_B(VPT, true, false, BY_LANE);           \
  } else if (ua) {                                    \
    CS_LN_FWD_B(VPT, false, true, BY_LANE);           \
  } else {                                            \
    CS_LN_FWD_B(VPT, false, false, BY_LANE);          \
  }
      if (b.vpt == 1 && by_lane) {
        CS_LN_FWD_B2(1, true)
      } else if (b.vpt == 1) {
        CS_LN_FWD_B2(1, false)
      } else if (b.vpt == 2 && by_lane) {  // without the residual only
        if (ua) {
          CS_LN_FWD_B(2, false, true, true);
        } else {
          CS_LN_FWD_B(2, false, false, true);
        }
      } else if (b.vpt == 2) {
        CS_LN_FWD_B2(2, false)
      } else {
        if constexpr (Vec16<TX>::n == 4) {
          CS_LN_FWD_B2(4, false)
        }
      }
#undef CS_LN_FWD_B2
#undef CS_LN_FWD_B
      return launch_status();
    }
  }
  using U = typename Acc<TX>::type;
  if (rows > 0x7fffffffLL) return CS_ERR_TOO_LARGE;
  if (res) {
    // no fast plan: the sum as its own launch, then the general kernel on it
    const int st = launch_add<TX>(x, res, sum_out, rows * C, s);
    if (st != CS_OK) return st;
    x = sum_out;
  }
  ln_fwd_general_kernel<TX, TY, TP><<<row_grid(rows), dim3(kLnThreads), 0, s>>>(
      (const TX *)x, (const TP *)gamma, (const TP *)beta, (TY *)y, (U *)mean, (U *)rstd, rows, C,
      (U)eps);
  return launch_status();
}

// ---- backward plans.  Which row kernel takes a shape, with what launch: one function, used by
// the launches, the workspace sizes and the partial-row counts alike.
#ifndef CS_LN_PAIRS
#define CS_LN_PAIRS 1
#endif
#ifndef CS_LN_H3_ALONE_PF
#define CS_LN_H3_ALONE_PF 1
#endif
#ifndef CS_LN_H3_WPE
#define CS_LN_H3_WPE 2
#endif
#ifndef CS_LN_PAIR_PF
#define CS_LN_PAIR_PF false
#endif
#ifndef CS_LN_PAIR_KEEP
#define CS_LN_PAIR_KEEP true
#endif
#ifndef CS_LN_PAIR_MAX_BLOCKS
#define CS_LN_PAIR_MAX_BLOCKS 256
#endif
// Rows of 4 vectors per lane (the 1600-column row at 16 bit) on ln_bwd_kernel, a wave per row:
// 0 never, 1 when only dgamma/dbeta are asked for, 2 always.  Measured at [16384,1600] bf16 with
// 512 threads, against ln_bwd_rows_kernel: dgamma/dbeta alone 22.4 against 45.8 us (every lane
// loads: nothing serialises the loads), dx alone 29.0 against 28.4 us, all three 33.3 against
// 33.7 us; with the next row prefetched, or 1024 threads, the kernel spills.  The two kernels give
// the same partial rows bit for bit (same rows per wave, same order of additions).
#ifndef CS_LN_W4_NEW
#define CS_LN_W4_NEW 1
#endif
#ifndef CS_LN_W4_THREADS
#define CS_LN_W4_THREADS 512
#endif
#ifndef CS_LN_W4_WPE
#define CS_LN_W4_WPE 2
#endif
#ifndef CS_LN_W4_PF
#define CS_LN_W4_PF false
#endif
#ifndef CS_LN_W4_KEEP
#define CS_LN_W4_KEEP false
#endif
enum BwdKind {
  kBwdNone = 0,  // no row-in-registers plan: the general kernels
  kBwdHalf1,     // ln_bwd_kernel, two rows per wave, 1 vector per lane (rows of up to 32 vectors)
  kBwdHalf3,     // ln_bwd_kernel, two rows per wave, 3 vectors per lane (65 to 96 vectors: C = 768 at 16 bit)
  kBwdWave4,     // ln_bwd_kernel, a wave per row, 4 vectors per lane
  kBwdWave,      // ln_bwd_kernel, a wave per row, 1 or 2 vectors per lane
  kBwdRows,      // ln_bwd_rows_kernel, 4 vectors per lane
  kBwdBlock,     // ln_bwd_block_kernel, several waves per row
};
struct BwdPlan {
  BwdKind kind = kBwdNone;
  int vpl = 0;
  int threads = kLnBwdThreads;
  int blocks = 0;         // workgroups of row work = partial rows left behind when dgamma/dbeta are wanted
  size_t fold_lds = 0;    // LDS of the column-sum fold
  size_t partial_elem = sizeof(float);  // bytes of a partial row's element
  bool two_calls = true;  // the partial rows may be added up by a later call (kBwdBlock: see block_two_calls)
  bool direct = false;    // kBwdBlock: the launch of dx takes the column sums (direct_wide_rows)
  bool four_waves = false;  // kBwdWave: four waves per SIMD that load a row at a time (see there)
  BlockPlan block;
};
constexpr int kLnMaxPartialRows = 512;
static_assert(2 * kLnBwdMaxBlocks <= kLnMaxPartialRows && CS_LN_PAIR_MAX_BLOCKS <= kLnMaxPartialRows,
              "every plan's grid cap fits the finalize step's row limit");

// Widths of the several-waves kernel whose backward pass can be split into a row pass and a later
// sum: whole vectors, up to 512 of them.  (Wider rows leave more partial rows than a caller that
// holds on to them should have to keep, and ragged ones have no aligned form.)
bool block_two_calls(int64_t C, int x_dtype) {
  if (x_dtype == CS_F64 || C <= 0) return false;
  const int vn = 16 / (int)dtype_size(x_dtype);
  return C % vn == 0 && C / vn > 4 * kWave && C / vn <= 8 * kWave;
}

// Rows on several waves, few enough that the column sums are taken straight from them in the launch of dx
// (ln_columns_wide); the split form's partial rows are fp32, so its widths keep the two launches.  Saved are a launch,
// and 16 bytes a column of partial row written and read again per workgroup, which was more than the rows themselves.
// As long as a row lane of ln_columns_wide has fewer than four rounds of 16 rows, up to 512 rows, 1024 of 1536 columns
// and more.  us per call with dresidual, two launches / one: bf16 [16,1003] 6.1 / 3.8, [64,4099] 16.7 / 6.2,
// [128,1909] 9.4 / 4.4, [300,5120] 21.0 / 10.4, [416,7424] 25 / 15, [1024,5120] 25.3 / 23.1, [1536,5120] 29.0 / 31.1;
// [300,257] 7.9 / 13.8, [300,1003] 10.3 / 10.3; fp32 [512,1909] 14.9 / 9.8, [768,1003] 11.7 / 12.1, [512,8192] 29.5 /
// 20.5, [1024,7424] 37.1 / 35.3.  The sums alone take that form as well: [300,9001] fp32 25.0 / 12.8.
bool direct_wide_rows(const BlockPlan &b, int64_t rows, int64_t C) {
  return rows <= (C < 1536 ? 512 : 1024) && rows < 64 * 2 * (int64_t)(b.gw * b.groups);
}

// What a backward call asks for, as far as its plan depends on it.
struct BwdWants {
  bool dx = true, sums = true;
  // no output lies over an input, and the sums are to be complete when the call is: they may be taken in the launch of dx
  bool apart = false;
};

// Ragged, unaligned and wide rows that the general kernels are the shorter way for.  us, several waves per row /
// general:
// The sums alone are one launch there, a chain of rows / 4 steps at any width; better as long as a row lane of
// ln_columns_wide has not 16 rows to load at once: bf16 [16,257] 3.6 / 3.0, [64,257] 4.5 / 4.5, [64,1003] 3.7 / 4.5,
// [64,4099] 5.9 / 4.6, fp32 [64,1909] 5.6 / 4.4, [64,9001] 7.4 / 4.5, rows shorter than a vector [64,3] 4.3 / 4.1 (but
// [65,257] 5.8 / 6.6 in two launches).
// dx alone never: it has the bits it has with the sums (up to 256 columns are 0.2-0.5 us slower for that, [64,65] bf16 3.5
// / 3.1; wider rows [64,4099] 4.6 / 7.8, [16,8200] fp32 4.5 / 12.6).
// All three where an output lies over an input: up to 64 rows of up to 512 vectors, which then need no workspace whatever
// the call (bf16 [8,65] 6.5 / 5.1, [16,257] 7.3 / 6.2; [64,65] 7.3 / 8.6, [64,1003] 7.6 / 10.3).  With four fp32 vectors
// per lane the kernel of several waves spills up to 60 registers: whole [16,8200] 19.2 / 15.7, [16,12288] 21.5 / 20.2,
// [32,12288] 22.9 / 29.5, ragged [64,9001] 28.5 / 20.7, [300,9001] 51.4 / 46.4, [512,9001] 51.1 / 67.5, [300,16383] 83.5 /
// 71.5, [512,16383] 81.3 / 90.6.
bool general_rows(const BwdWants &w, const BlockPlan &b, int64_t rows, int64_t C, int x_dtype, bool aligned) {
  const int64_t vn = 16 / (int64_t)dtype_size(x_dtype);
  if (!w.dx) return rows <= 64 && (C < vn || rows < 16 * 2 * (int64_t)(b.gw * b.groups));
  if (!w.sums) return false;
  if (b.vpt == 4) return rows <= (aligned && C % vn == 0 ? 16 : 384);
  return rows <= 64 && C / vn <= 8 * kWave;
}

// A wave per row: four waves per SIMD on 512 workgroups, a row at a time, instead of two that have the next rows under way.
// us per call, two waves / four.
// One vector per lane, dx alone: there are no column sums in the registers.  bf16 [3000,512] 3.95 / 3.76, [8192,512] 6.5 /
// 5.8, [30000,512] 18.8 / 16.8, fp32 [8192,256] 6.1 / 5.4.  With the sums, many rows of up to 56 vectors, which leave lanes
// idle; plain / with dresidual / the sums alone: bf16 [14000,264] 11.8 / 11.1, 12.3 / 12.2, 9.0 / 9.0, [60000,264] 30.8 / 25.7, 33.7 /
// 30.8, 20.5 / 19.4, fp32 [14000,160] 11.3 / 10.1, 11.7 / 10.6, 8.0 / 8.4, [60000,160] 30.3 / 24.1, 31.9 / 29.4, 18.4 / 18.2 (but fp32
// [14000,132] 11.6 / 11.6, 11.7 / 11.9, 8.6 / 10.2).  Of 57 to 64 vectors rows with dresidual fill the memory with the two: bf16
// [60000,512] 37.8 / 36.1, 45.2 / 46.9, 23.6 / 23.9.  All forms of a call have to leave the same partial rows (the split form,
// which is asked for them without knowing of a dx or dresidual, gives the bits of the single call), and dresidual is what
// training has.
// Two vectors per lane, dx alone: fp16 [8192,896] 9.7 / 8.8, [12289,896] 13.3 / 12.6, bf16 [5000,1024] 7.4 / 7.0, [16384,1024]
// 17.8 / 17.7; not where those rows make two steps or fewer of the two waves (bf16 [4096,1024] 5.3 / 5.9, fp32 [4096,400]
// 4.5 / 4.9), or so many that their rows in flight are the better use of the memory ([30000,1024] 31.5 / 32.7, fp16
// [30000,896] 27.6 / 28.5).
bool four_waves(int64_t rows, int64_t nvec, bool sums) {
  const int64_t step = (int64_t)kLnBwdMaxBlocks * (kLnBwdThreads / kWave);
  if (nvec > kWave) return !sums && rows > 2 * step && rows <= 10 * step;
  return !sums || (rows > 5 * step && nvec <= 56);
}

// A wave per row: more rows than these have 512 workgroups, so that a wave's fp32 chain of column sums is no longer than
// with four waves per SIMD.  Error of dgamma and dbeta on 256, of that on 512: 1.08 at 131072 rows, 1.2 at 262144, 1.34 at a million.
// (No slower: fp32 [262144,256] 142 / 142 us with ln_bwd_rows_kernel / now, bf16 [80000,1024] 90.5 / 89.1.)
constexpr int64_t kOneWorkgroupRows = 65536;

BwdPlan bwd_plan(int64_t rows, int64_t C, int x_dtype, bool aligned, const BwdWants &w = BwdWants{}) {
  BwdPlan b;
  const FastPlan p = aligned ? fast_plan(C, x_dtype) : FastPlan{};
  if (p.vpl == 0) {
    const bool two_calls = aligned && block_two_calls(C, x_dtype);
    b.block = block_plan(rows, C, x_dtype, true, false);
    if (b.block.vpt == 0) return b;
    const bool direct = w.sums && w.apart && !two_calls && direct_wide_rows(b.block, rows, C);
    if (!two_calls && !(direct && w.dx) && general_rows(w, b.block, rows, C, x_dtype, aligned)) return b;
    b.kind = kBwdBlock;
    b.vpl = b.block.vpt;
    b.threads = b.block.gw * b.block.groups * kWave;
    b.blocks = b.block.blocks;
    b.fold_lds = (size_t)b.block.groups * C * sizeof(double);
    b.two_calls = two_calls;
    b.partial_elem = b.two_calls ? sizeof(float) : sizeof(double);
    b.direct = direct;
    return b;
  }
  const int vn = 16 / (int)dtype_size(x_dtype);
  const int64_t nvec = C / vn;
  b.vpl = p.vpl;
  if (CS_LN_PAIRS && (nvec <= kHalf || (nvec > kWave && nvec <= 3 * kHalf))) {
    b.kind = nvec <= kHalf ? kBwdHalf1 : kBwdHalf3;
    b.vpl = nvec <= kHalf ? 1 : 3;
    const int64_t n = ceil_div((rows + 1) / 2, (int64_t)(kLnBwdThreads / kWave));
    b.blocks = (int)(n < CS_LN_PAIR_MAX_BLOCKS ? n : CS_LN_PAIR_MAX_BLOCKS);
    b.fold_lds = (size_t)(kLnBwdThreads / kWave) * 2 * C * sizeof(float);
  } else if (p.vpl == 4 && (CS_LN_W4_NEW == 2 || (CS_LN_W4_NEW == 1 && !w.dx))) {
    b.kind = kBwdWave4;
    b.threads = CS_LN_W4_THREADS;
    b.blocks = ln_blocks(rows, 1, kLnBwdMaxBlocks, b.threads);
    b.fold_lds = (size_t)(b.threads / kWave) * C * sizeof(float);
  } else {
    // Up to two vectors per lane, the next row requested while this one is worked on and x-hat kept across the row sums
    // fit two waves per SIMD.  ln_bwd_rows_kernel with three or four took 512 workgroups for them, of which with
    // dresidual a CU held one at a time, and left twice the partial rows.  us per call with dresidual, those / these: bf16
    // [1500,1024] 8.5 / 8.2, [4096,1024] 15.9 / 11.6, [8192,1024] 21.8 / 18.0, [16384,1024] 33.2 / 27.7, [4096,512] 9.2 /
    // 8.2, fp16 [8192,896] 20.8 / 16.5, fp32 [8192,512] 16.8 / 15.9; without it bf16 [4096,1024] 11.9 / 10.0; an earlier
    // call's sums in the launch [8192,1024] 20.1 / 16.6, [1500,512] 4.5 / 4.3.  Level at plain [16384,512] (14.9).
    b.kind = p.vpl <= 2 ? kBwdWave : kBwdRows;
    b.four_waves = b.kind == kBwdWave && four_waves(rows, nvec, w.sums);
    const bool many_rows = b.kind == kBwdWave && rows > kOneWorkgroupRows;
    b.blocks = ln_blocks(rows, 1, b.four_waves || many_rows ? 2 * kLnBwdMaxBlocks : kLnBwdMaxBlocks, kLnBwdThreads);
    b.fold_lds = (size_t)(kLnBwdThreads / kWave) * C * sizeof(float);
  }
  return b;
}

// Rows few enough that the column sums are taken straight from them (ln_columns_direct): up to 16 partial rows'
// worth a thread makes one trip to memory, and up to 512 rows the one launch is the shorter way.  Kernels of a
// backward call, us, two launches / one, with dresidual: bf16 [77,768] 9.0 / 4.2, [256,768] 9.5 / 4.6, [512,768]
// 9.7 / 6.6, [1024,768] 10.0 / 10.3; [512,64] 7.0 / 5.7, [512,512] 7.3 / 7.0, [512,1024] 8.7 / 7.2, [512,1600]
// 11.3 / 7.3, [1024,1024] 9.1 / 12.0; fp32 [512,384] 8.8 / 6.2, [1024,384] 9.0 / 9.8.
constexpr int64_t kDirectRows = 512;
bool direct_sums(const BwdPlan &p, int64_t rows) {
  return (p.kind == kBwdHalf1 || p.kind == kBwdHalf3 || p.kind == kBwdWave || p.kind == kBwdRows) && rows <= kDirectRows;
}

bool overlap(const void *a, size_t a_bytes, const void *b, size_t b_bytes) {
  const char *p = (const char *)a, *q = (const char *)b;
  return p < q + b_bytes && q < p + a_bytes;
}

// Column order inside a partial row, as the `vn` of ln_finalize_tile: every row kernel leaves column
// idx*vn + k at position k*(C/vn) + idx.
int partial_vn(int x_dtype) { return 16 / (int)dtype_size(x_dtype); }

// How partial rows are stored and added up.
enum PartialRows {
  kFloatRows,            // fp32, added in fp32: the row-per-wave kernels
  kFloatRowsDoubleSums,  // fp32, added in double: the several-waves kernel where the sum may be a later call
  kDoubleRows,           // double throughout: the several-waves kernel elsewhere
};
// partial rows that a caller holds on to
PartialRows kept_rows(int64_t C, int x_dtype) {
  return fast_plan(C, x_dtype).vpl == 0 ? kFloatRowsDoubleSums : kFloatRows;
}

enum BwdPhase { kBwdWhole = 0, kBwdRowsOnly = 1 };

// An earlier call's partial rows whose column sums ride in this call's launch (host side of
// LnPending); partial == nullptr: none.
struct PendingSums {
  const void *partial = nullptr;
  int64_t nparts = 0;
  void *dgamma = nullptr, *dbeta = nullptr;
  int accumulate = 0;
};

template <typename TP, typename A, typename P>
int launch_finalize_in(const void *partial, int64_t nparts, void *dgamma, void *dbeta, int64_t C, int vn,
                       int accumulate, hipStream_t s) {
  ln_bwd_finalize_kernel<TP, A, P><<<dim3(2 * (unsigned)ceil_div(C, (int64_t)kLnFinCols)), dim3(kLnFinCols * kLnFinRows), 0, s>>>(
      (const P *)partial, (int)nparts, (TP *)dgamma, (TP *)dbeta, (int)C, vn, accumulate);
  return launch_status();
}

template <typename TP>
int launch_finalize(PartialRows kind, const void *partial, int64_t nparts, void *dgamma, void *dbeta, int64_t C, int vn,
                    int accumulate, hipStream_t s) {
  switch (kind) {
    case kFloatRows: return launch_finalize_in<TP, float, float>(partial, nparts, dgamma, dbeta, C, vn, accumulate, s);
    case kFloatRowsDoubleSums:
      return launch_finalize_in<TP, double, float>(partial, nparts, dgamma, dbeta, C, vn, accumulate, s);
    case kDoubleRows: return launch_finalize_in<TP, double, double>(partial, nparts, dgamma, dbeta, C, vn, accumulate, s);
  }
  return CS_ERR_UNSUPPORTED;
}

// A launch may ask for more dynamic LDS than the 64 KB it gets by default once the kernel's limit
// has been raised; once per kernel and device.
template <typename K>
int allow_lds(K kernel, size_t bytes, size_t most, std::atomic<bool> *done) {
  if (bytes <= 64 * 1024) return CS_OK;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return (int)hipErrorInvalidDevice;
  if (!done[dev].load(std::memory_order_acquire)) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)most);
    if (e != hipSuccess) return (int)e;
    done[dev].store(true, std::memory_order_release);
  }
  return CS_OK;
}

template <typename TDY, typename TX, typename TDX, typename TP, int THREADS, int LPR, int VPL, int WPE, bool PF,
          bool KEEP, bool HAS_DX, bool HAS_DP, bool HAS_DRES, bool DIRECT = false>
int launch_bwd_kernel(const void *dy, const void *x, const void *mean, const void *rstd, const void *gamma,
                      void *dx, void *workspace, int64_t rows, int64_t C, const void *dres, const LnPending &pend,
                      int blocks, size_t lds, hipStream_t s) {
  static std::atomic<bool> lds_allowed[64];
  auto kernel = ln_bwd_kernel<TDY, TX, TDX, TP, THREADS, LPR, VPL, WPE, PF, KEEP, HAS_DX, HAS_DP, HAS_DRES, DIRECT>;
  // the fold of the widest row this instantiation takes: [rows side by side x waves][C] floats
  constexpr size_t kMostLds = (size_t)THREADS * VPL * Vec16<TX>::n * sizeof(float);
  const int st = allow_lds(kernel, lds, kMostLds, lds_allowed);
  if (st != CS_OK) return st;
  kernel<<<dim3((unsigned)(blocks + pend.blocks)), dim3(THREADS), lds, s>>>(
      (const TDY *)dy, (const TX *)x, (const float *)mean, (const float *)rstd, (const TP *)gamma, (TDX *)dx,
      (float *)workspace, rows, (int)C, (const TDX *)dres, pend);
  return launch_status();
}

// dx and, by further workgroups of the launch, the column sums straight from the rows
template <typename TDY, typename TX, typename TDX, typename TP, int VPT>
int launch_bwd_block_direct(const void *dy, const void *x, const void *mean, const void *rstd, const void *gamma,
                            void *dx, int64_t rows, int64_t C, const void *dres, const BlockPlan &b, bool ua,
                            const LnPending &side, hipStream_t s) {
  const dim3 grid((unsigned)(b.blocks + side.blocks)), block((unsigned)(b.gw * b.groups * kWave));
  const size_t lds = (size_t)2 * block.x * sizeof(double);
#define CS_LN_BLOCK_DIRECT(HAS_DRES, UA)                                                                            \
  ln_bwd_block_kernel<TDY, TX, TDX, TP, VPT, true, false, HAS_DRES, UA, true><<<grid, block, lds, s>>>(              \
      (const TDY *)dy, (const TX *)x, (const float *)mean, (const float *)rstd, (const TP *)gamma, (TDX *)dx,       \
      nullptr, 0, rows, (int)C, (const TDX *)dres, b.gw, b.groups, side)
  if (dres && ua) {
    CS_LN_BLOCK_DIRECT(true, true);
  } else if (dres) {
    CS_LN_BLOCK_DIRECT(true, false);
  } else if (ua) {
    CS_LN_BLOCK_DIRECT(false, true);
  } else {
    CS_LN_BLOCK_DIRECT(false, false);
  }
#undef CS_LN_BLOCK_DIRECT
  return launch_status();
}

template <typename TDY, typename TX, typename TDX, typename TP, int VPT, bool HAS_DX, bool HAS_DP, bool HAS_DRES>
int launch_bwd_block(const void *dy, const void *x, const void *mean, const void *rstd, const void *gamma, void *dx,
                     void *workspace, int64_t rows, int64_t C, const void *dres, const BwdPlan &plan, bool ua,
                     size_t lds, hipStream_t s) {
  const auto kernel = ua ? ln_bwd_block_kernel<TDY, TX, TDX, TP, VPT, HAS_DX, HAS_DP, HAS_DRES, true>
                         : ln_bwd_block_kernel<TDY, TX, TDX, TP, VPT, HAS_DX, HAS_DP, HAS_DRES, false>;
  if (!HAS_DP) lds = 0;
  // the widest row alone takes 128 KB next to the kernel's own half kilobyte
  static std::atomic<bool> lds_allowed[2][64];
  const int st = allow_lds(kernel, lds + 512, kLnBlockFoldLds + 512, lds_allowed[ua]);
  if (st != CS_OK) return st;
  kernel<<<dim3((unsigned)plan.blocks), dim3((unsigned)plan.threads), lds, s>>>(
      (const TDY *)dy, (const TX *)x, (const float *)mean, (const float *)rstd, (const TP *)gamma, (TDX *)dx,
      workspace, plan.partial_elem == sizeof(double), rows, (int)C, (const TDX *)dres, plan.block.gw, plan.block.groups,
      LnNoSide{});
  return launch_status();
}

template <typename TDY, typename TX, typename TDX, typename TP>
int bwd_typed(const void *dy, const void *x, const void *mean, const void *rstd,
              const void *gamma, void *dx, void *dgamma, void *dbeta, void *workspace,
              size_t workspace_bytes, int64_t rows, int64_t C, bool aligned, int x_dtype,
              int accumulate, const void *dres, hipStream_t s, BwdPhase phase = kBwdWhole,
              PendingSums pending = PendingSums{}) {
  // rows only: the partial rows are the product, the parameter gradients come from a later
  // cs_layernorm_backward_finalize (or ride in a later call's launch)
  const bool want_dp = phase == kBwdRowsOnly || dgamma != nullptr || dbeta != nullptr;
  // One launch reads the inputs for the sums, and for dx, while other workgroups of it write: a caller that has an
  // output written over an input gets the two launches
  const size_t n = (size_t)rows * C, stat = (size_t)rows * sizeof(float), params = (size_t)C * sizeof(TP);
  const auto clear_of = [&](const void *out, size_t bytes, const void *in, size_t in_bytes) {
    return out == nullptr || in == nullptr || !overlap(out, bytes, in, in_bytes);
  };
  const size_t out = n * sizeof(TDX);
  const bool dx_apart = clear_of(dx, out, dy, n * sizeof(TDY)) && clear_of(dx, out, x, n * sizeof(TX));
  bool apart = dx_apart;
  for (const void *sum : {(const void *)dgamma, (const void *)dbeta})
    apart = apart && clear_of(sum, params, dy, n * sizeof(TDY)) && clear_of(sum, params, x, n * sizeof(TX)) &&
            clear_of(sum, params, mean, stat) && clear_of(sum, params, rstd, stat) &&
            clear_of(sum, params, gamma, params) && clear_of(sum, params, dres, out);
  BwdPlan plan = bwd_plan(rows, C, x_dtype, aligned, {dx != nullptr, want_dp, apart && phase == kBwdWhole});
  if (phase == kBwdRowsOnly && (plan.kind == kBwdNone || !plan.two_calls || std::is_same_v<TX, double>))
    return aligned ? CS_ERR_UNSUPPORTED : CS_ERR_MISALIGNED;
  if constexpr (!std::is_same_v<TX, double>) {
    // Few rows on several waves: the sums straight from the rows, in the launch of dx
    if (plan.direct) {
      BlockPlan b = plan.block;
      if (!dx) b.blocks = 0;  // the sums alone
      const bool ua = !aligned || C % Vec16<TX>::n != 0;
      const LnPending side{nullptr, dgamma, dbeta, 0, accumulate, (int)ceil_div(C, (int64_t)kLnWideTile)};
#define CS_LN_WIDE(VPT) \
  return launch_bwd_block_direct<TDY, TX, TDX, TP, VPT>(dy, x, mean, rstd, gamma, dx, rows, C, dres, b, ua, side, s)
      if (b.vpt == 1) CS_LN_WIDE(1);
      if (b.vpt == 2) CS_LN_WIDE(2);
      if constexpr (Vec16<TX>::n == 4) CS_LN_WIDE(4);
#undef CS_LN_WIDE
    }
  }
  const size_t need = want_dp ? (size_t)plan.blocks * 2 * C * plan.partial_elem : 0;
  const bool ws_ok = need == 0 || (workspace != nullptr && workspace_bytes >= need && aligned_to(workspace, plan.partial_elem));
  // a caller may bring no workspace where no sum in two steps was promised: the general kernels
  if (plan.kind == kBwdBlock && !plan.two_calls && !ws_ok) plan = BwdPlan{};
  if constexpr (!std::is_same_v<TX, double>) {
    if (plan.kind != kBwdNone) {
      const int blocks = plan.blocks;
      if (!ws_ok) return CS_ERR_WORKSPACE;
      // the several-waves kernel carries no pending sums: those get their own launch first
      LnPending pend{nullptr, nullptr, nullptr, 0, 0, 0};
      if (pending.partial != nullptr && (pending.dgamma != nullptr || pending.dbeta != nullptr)) {
        if (plan.kind == kBwdBlock) {
          const int st = launch_finalize<TP>(kept_rows(C, x_dtype), pending.partial, pending.nparts, pending.dgamma,
                                             pending.dbeta, C, partial_vn(x_dtype), pending.accumulate, s);
          if (st != CS_OK) return st;
        } else {
          pend = LnPending{pending.partial, pending.dgamma, pending.dbeta, (int)pending.nparts,
                           pending.accumulate, 2 * (int)ceil_div(C, (int64_t)kLnFinCols)};
        }
      }
      // Few rows: the sums straight from the rows, in this launch
      if (direct_sums(plan, rows) && phase == kBwdWhole && want_dp && dx && apart && pend.blocks == 0) {
        const LnPending side{nullptr, dgamma, dbeta, blocks, accumulate, (int)ceil_div(C, (int64_t)kLnFinCols)};
        const size_t lds = (size_t)2 * kLnFinRows * kLnFinCols * sizeof(float);
        const dim3 grid((unsigned)(blocks + side.blocks)), block((unsigned)plan.threads);
        int st = CS_OK;
#define CS_LN_DIRECT(LPR, VPL, HAS_DRES)                                                                               \
  if (LPR != 0) {                                                                                                      \
    st = launch_bwd_kernel<TDY, TX, TDX, TP, kLnBwdThreads, LPR ? LPR : 64, LPR ? VPL : 1, 2, false, CS_LN_PAIR_KEEP,  \
                           true, false, HAS_DRES, true>(dy, x, mean, rstd, gamma, dx, workspace, rows, C, dres, side,  \
                                                        blocks, lds, s);                                               \
  } else {                                                                                                             \
    ln_bwd_rows_kernel<TDY, TX, TDX, TP, true, false, HAS_DRES, true><<<grid, block, lds, s>>>(                        \
        (const TDY *)dy, (const TX *)x, (const float *)mean, (const float *)rstd, (const TP *)gamma, (TDX *)dx,        \
        (float *)workspace, rows, (int)C, (const TDX *)dres, side);                                                    \
    st = launch_status();                                                                                              \
  }
#define CS_LN_DIRECT2(LPR, VPL)           \
  if (dres) {                             \
    CS_LN_DIRECT(LPR, VPL, true)          \
  } else {                                \
    CS_LN_DIRECT(LPR, VPL, false)         \
  }
        if (plan.kind == kBwdHalf1) {
          CS_LN_DIRECT2(32, 1)
        } else if (plan.kind == kBwdHalf3) {
          CS_LN_DIRECT2(32, 3)
        } else if (plan.kind == kBwdWave && plan.vpl == 1) {
          CS_LN_DIRECT2(64, 1)
        } else if (plan.kind == kBwdWave) {
          CS_LN_DIRECT2(64, 2)
        } else {
          CS_LN_DIRECT2(0, 4)
        }
#undef CS_LN_DIRECT2
#undef CS_LN_DIRECT
        return st;
      }
      size_t lds = want_dp ? plan.fold_lds : 0;
      const size_t pend_lds = (size_t)kLnFinRows * kLnFinCols * sizeof(float);
      if (pend.blocks != 0 && lds < pend_lds) lds = pend_lds;
      const dim3 grid((unsigned)(blocks + pend.blocks)), block((unsigned)plan.threads);
      int st = CS_OK;
// (the first two arguments are CS_LN_BWD_MASK's and have no use here)
#define CS_LN_BWD(UNUSED, UNUSED_TOO, HAS_DX, HAS_DP, HAS_DRES)                             \
  ln_bwd_rows_kernel<TDY, TX, TDX, TP, HAS_DX, HAS_DP, HAS_DRES>                            \
      <<<grid, block, lds, s>>>((const TDY *)dy, (const TX *)x, (const float *)mean,        \
                                (const float *)rstd, (const TP *)gamma, (TDX *)dx,          \
                                (float *)workspace, rows, (int)C, (const TDX *)dres, pend)
#define CS_LN_K32(VPL, WPE, HAS_DX, HAS_DP, HAS_DRES)                                                          \
  st = launch_bwd_kernel<TDY, TX, TDX, TP, kLnBwdThreads, 32, VPL, WPE, CS_LN_PAIR_PF, CS_LN_PAIR_KEEP, HAS_DX, \
                         HAS_DP, HAS_DRES>(dy, x, mean, rstd, gamma, dx, workspace, rows, C, dres, pend, blocks, \
                                           lds, s)
#define CS_LN_K32PF(VPL, WPE, HAS_DX, HAS_DP, HAS_DRES)                                                        \
  st = launch_bwd_kernel<TDY, TX, TDX, TP, kLnBwdThreads, 32, VPL, WPE, true, CS_LN_PAIR_KEEP, HAS_DX, HAS_DP,   \
                         HAS_DRES>(dy, x, mean, rstd, gamma, dx, workspace, rows, C, dres, pend, blocks, lds, s)
#define CS_LN_K64(VPL, WPE, HAS_DX, HAS_DP, HAS_DRES)                                                          \
  st = launch_bwd_kernel<TDY, TX, TDX, TP, CS_LN_W4_THREADS, 64, VPL, WPE, CS_LN_W4_PF, CS_LN_W4_KEEP, HAS_DX,  \
                         HAS_DP, HAS_DRES>(dy, x, mean, rstd, gamma, dx, workspace, rows, C, dres, pend, blocks, \
                                           lds, s)
#define CS_LN_K64PF(VPL, WPE, HAS_DX, HAS_DP, HAS_DRES)                                                        \
  st = launch_bwd_kernel<TDY, TX, TDX, TP, kLnBwdThreads, 64, VPL, WPE, WPE == 2, true, HAS_DX, HAS_DP, HAS_DRES>( \
      dy, x, mean, rstd, gamma, dx, workspace, rows, C, dres, pend, blocks, lds, s)
#define CS_LN_K64PF1(VPL, WPE, HAS_DX, HAS_DP, HAS_DRES) CS_LN_K64PF(VPL, (HAS_DP ? WPE : 4), HAS_DX, HAS_DP, HAS_DRES)
#define CS_LN_BWD_MASK(K, VPL, WPE)             \
  if (dx && want_dp && dres) {                  \
    K(VPL, WPE, true, true, true);              \
  } else if (dx && dres) {                      \
    K(VPL, WPE, true, false, true);             \
  } else if (dx && want_dp) {                   \
    K(VPL, WPE, true, true, false);             \
  } else if (dx) {                              \
    K(VPL, WPE, true, false, false);            \
  } else {                                      \
    K(VPL, WPE, false, true, false);            \
  }
      if (plan.kind == kBwdHalf1) {
        CS_LN_BWD_MASK(CS_LN_K32, 1, 4)
      } else if (plan.kind == kBwdHalf3) {
        // On its own a launch is one workgroup per CU, so a wave may take twice the registers and
        // load its next two rows while it works on the current ones ([8192,768]: 13.7 -> 13.1 us, with
        // dresidual 16.1 -> 15.7).  With an earlier call's sums in the launch their workgroups must
        // fit next to a row workgroup on the same CU, which the larger register budget rules out
        // (11.3 -> 12.1 us), so that form keeps two workgroups per CU and no prefetch.
        if (pend.blocks == 0 && dx != nullptr && CS_LN_H3_ALONE_PF) {  // sums alone: 10.9 us without, 11.3 with
          CS_LN_BWD_MASK(CS_LN_K32PF, 3, 1)
        } else {
          CS_LN_BWD_MASK(CS_LN_K32, 3, CS_LN_H3_WPE)
        }
      } else if (plan.kind == kBwdWave4) {
#if CS_LN_W4_NEW == 2
        CS_LN_BWD_MASK(CS_LN_K64, 4, CS_LN_W4_WPE)
#else
        CS_LN_K64(4, CS_LN_W4_WPE, false, true, false);
#endif
      } else if (plan.kind == kBwdBlock) {
        const bool ua = !aligned || C % Vec16<TX>::n != 0;
#define CS_LN_BWD_B(VPT, HAS_DX, HAS_DP, HAS_DRES)                                                                \
  st = launch_bwd_block<TDY, TX, TDX, TP, VPT, HAS_DX, HAS_DP, HAS_DRES>(dy, x, mean, rstd, gamma, dx, workspace, \
                                                                         rows, C, dres, plan, ua, lds, s)
// (the second argument is CS_LN_BWD_MASK's and has no use here)
#define CS_LN_BWD_BLOCK(VPT, UNUSED, HAS_DX, HAS_DP, HAS_DRES)                   \
  if constexpr (VPT * Vec16<TX>::n > 8 && HAS_DX && HAS_DP) {                    \
    CS_LN_BWD_B(VPT, false, true, false);                                        \
    if (st == CS_OK) CS_LN_BWD_B(VPT, true, false, HAS_DRES);                    \
  } else {                                                                       \
    CS_LN_BWD_B(VPT, HAS_DX, HAS_DP, HAS_DRES);                                  \
  }
        // with 16 elements per lane the column sums and dx do not fit the registers together: two
        // passes over the rows ([1024,16000] bf16 with dresidual: 54 us against 136)
        if (plan.vpl == 1) {
          CS_LN_BWD_MASK(CS_LN_BWD_BLOCK, 1, 0)
        } else if (plan.vpl == 2) {
          CS_LN_BWD_MASK(CS_LN_BWD_BLOCK, 2, 0)
        } else {
          if constexpr (Vec16<TX>::n == 4) {
            CS_LN_BWD_MASK(CS_LN_BWD_BLOCK, 4, 0)
          }
        }
#undef CS_LN_BWD_BLOCK
#undef CS_LN_BWD_B
      } else if (plan.kind == kBwdWave && plan.vpl == 1) {
        if (plan.four_waves) {
          CS_LN_BWD_MASK(CS_LN_K64PF1, 1, 4)
        } else {
          CS_LN_BWD_MASK(CS_LN_K64PF1, 1, 2)
        }
      } else if (plan.kind == kBwdWave && plan.four_waves) {
        if (dres) {
          CS_LN_K64PF(2, 4, true, false, true);
        } else {
          CS_LN_K64PF(2, 4, true, false, false);
        }
      } else if (plan.kind == kBwdWave) {
        CS_LN_BWD_MASK(CS_LN_K64PF, 2, 2)
      } else {
        CS_LN_BWD_MASK(CS_LN_BWD, 4, 2)
      }
#undef CS_LN_BWD_MASK
#undef CS_LN_K32
#undef CS_LN_K32PF
#undef CS_LN_K64
#undef CS_LN_K64PF
#undef CS_LN_K64PF1
#undef CS_LN_BWD
      if (st == CS_OK) st = launch_status();
      if (st == CS_OK && want_dp && phase == kBwdWhole)
        st = launch_finalize<TP>(plan.kind != kBwdBlock ? kFloatRows : plan.two_calls ? kFloatRowsDoubleSums : kDoubleRows,
                                 workspace, blocks, dgamma, dbeta, C, partial_vn(x_dtype), accumulate, s);
      return st;
    }
  }
  using U = typename Acc<TX>::type;
  if (rows > 0x7fffffffLL) return CS_ERR_TOO_LARGE;
  const auto sums = [&] {
    ln_bwd_param_general_kernel<TDY, TX, TP>
        <<<dim3((unsigned)ceil_div(C, (int64_t)64)), dim3(64, 4), 0, s>>>(
            (const TDY *)dy, (const TX *)x, (const U *)mean, (const U *)rstd, (TP *)dgamma,
            (TP *)dbeta, rows, C, accumulate);
    return launch_status();
  };
  // ahead of a dx that is written over what they read; otherwise behind it, as they may be written over gamma
  const bool sums_first = want_dp && dx && !dx_apart;
  if (sums_first) {
    const int st = sums();
    if (st != CS_OK) return st;
  }
  if (dx) {
    ln_bwd_dx_general_kernel<TDY, TX, TDX, TP><<<row_grid(rows), dim3(kLnThreads), 0, s>>>(
        (const TDY *)dy, (const TX *)x, (const U *)mean, (const U *)rstd, (const TP *)gamma,
        (TDX *)dx, rows, C, (const TDX *)dres);
    const int st = launch_status();
    if (st != CS_OK) return st;
  }
  return want_dp && !sums_first ? sums() : CS_OK;
}

bool wide_ok(int narrow, int other) { return other == narrow || other == CS_F32; }

}  // namespace
}  // namespace cs_hip

using namespace cs_hip;

namespace {
int ln_forward(const void *x, const void *residual, void *sum_out, const void *gamma,
               const void *beta, void *y, void *mean, void *rstd, int64_t rows, int64_t C,
               double eps, int x_dtype, int y_dtype, int param_dtype, void *stream) {
  if (rows < 0 || C <= 0) return CS_ERR_INVALID_ARGUMENT;
  if (dtype_size(x_dtype) == 0 || dtype_size(y_dtype) == 0 || dtype_size(param_dtype) == 0)
    return CS_ERR_UNSUPPORTED;
  if (!wide_ok(x_dtype, y_dtype) || !wide_ok(x_dtype, param_dtype)) return CS_ERR_UNSUPPORTED;
  if (x_dtype == CS_F64 && (y_dtype != CS_F64 || param_dtype != CS_F64)) return CS_ERR_UNSUPPORTED;
  if (rows == 0) return CS_OK;
  if (!x || !gamma || !y || !mean || !rstd) return CS_ERR_INVALID_ARGUMENT;
  if ((residual == nullptr) != (sum_out == nullptr)) return CS_ERR_INVALID_ARGUMENT;
  if (residual && (!aligned_to(residual, dtype_size(x_dtype)) || !aligned_to(sum_out, dtype_size(x_dtype))))
    return CS_ERR_MISALIGNED;
  if (!aligned_to(x, dtype_size(x_dtype)) || !aligned_to(y, dtype_size(y_dtype)) ||
      !aligned_to(gamma, dtype_size(param_dtype)) ||
      (beta && !aligned_to(beta, dtype_size(param_dtype))) || !aligned_to(mean, 4) ||
      !aligned_to(rstd, 4))
    return CS_ERR_MISALIGNED;
  const bool aligned = is_aligned16(x) && (!residual || (is_aligned16(residual) && is_aligned16(sum_out))) &&
                       is_aligned16(y) && is_aligned16(gamma) && (!beta || is_aligned16(beta));
  hipStream_t s = as_stream(stream);
#define CS_CALL(TX, TY, TP)                                                                       \
  return fwd_typed<TX, TY, TP>(x, gamma, beta, y, mean, rstd, rows, C, eps, aligned, x_dtype, residual, \
                               sum_out, s)
  const bool y_wide = y_dtype != x_dtype, p_wide = param_dtype != x_dtype;
  switch (x_dtype) {
    case CS_F32: CS_CALL(float, float, float);
    case CS_F64: CS_CALL(double, double, double);
    case CS_F16:
      if (y_wide && p_wide) CS_CALL(f16_t, float, float);
      if (y_wide) CS_CALL(f16_t, float, f16_t);
      if (p_wide) CS_CALL(f16_t, f16_t, float);
      CS_CALL(f16_t, f16_t, f16_t);
    case CS_BF16:
      if (y_wide && p_wide) CS_CALL(bf16_t, float, float);
      if (y_wide) CS_CALL(bf16_t, float, bf16_t);
      if (p_wide) CS_CALL(bf16_t, bf16_t, float);
      CS_CALL(bf16_t, bf16_t, bf16_t);
  }
#undef CS_CALL
  return CS_ERR_UNSUPPORTED;
}
}  // namespace

extern "C" int cs_layernorm_forward(const void *x, const void *gamma, const void *beta, void *y,
                                    void *mean, void *rstd, int64_t rows, int64_t C, double eps,
                                    int x_dtype, int y_dtype, int param_dtype, void *stream) {
  return ln_forward(x, nullptr, nullptr, gamma, beta, y, mean, rstd, rows, C, eps, x_dtype, y_dtype,
                    param_dtype, stream);
}

extern "C" int cs_add_layernorm_forward(const void *x, const void *residual, void *sum_out,
                                        const void *gamma, const void *beta, void *y, void *mean,
                                        void *rstd, int64_t rows, int64_t C, double eps,
                                        int x_dtype, int y_dtype, int param_dtype, void *stream) {
  if (rows > 0 && (!residual || !sum_out)) return CS_ERR_INVALID_ARGUMENT;
  return ln_forward(x, residual, sum_out, gamma, beta, y, mean, rstd, rows, C, eps, x_dtype, y_dtype,
                    param_dtype, stream);
}

extern "C" size_t cs_layernorm_backward_workspace_bytes(int64_t rows, int64_t C) {
  if (rows <= 0 || C <= 0) return 0;
  // the most partial rows any plan leaves for this many rows, whatever the storage type
  size_t most = 0;
  for (int dt : {CS_F32, CS_F16}) {
    for (bool aligned : {true, false}) {
      const BwdPlan b = bwd_plan(rows, C, dt, aligned);
      if (b.blocks * b.partial_elem > most) most = b.blocks * b.partial_elem;
    }
  }
  return most * 2 * (size_t)C;
}

namespace {
int ln_backward(const void *dy, const void *x, const void *mean, const void *rstd,
                const void *gamma, const void *dres, void *dx, void *dgamma, void *dbeta,
                void *workspace, size_t workspace_bytes, int64_t rows, int64_t C, int dy_dtype,
                int x_dtype, int dx_dtype, int param_dtype, int accumulate, void *stream,
                BwdPhase phase = kBwdWhole, PendingSums pending = PendingSums{}) {
  if (rows < 0 || C <= 0) return CS_ERR_INVALID_ARGUMENT;
  if (dtype_size(x_dtype) == 0 || dtype_size(dy_dtype) == 0 || dtype_size(dx_dtype) == 0 ||
      dtype_size(param_dtype) == 0)
    return CS_ERR_UNSUPPORTED;
  if (!wide_ok(x_dtype, dy_dtype) || !wide_ok(x_dtype, dx_dtype) || !wide_ok(x_dtype, param_dtype))
    return CS_ERR_UNSUPPORTED;
  if (x_dtype == CS_F64 && (dy_dtype != CS_F64 || dx_dtype != CS_F64 || param_dtype != CS_F64))
    return CS_ERR_UNSUPPORTED;
  if (phase == kBwdWhole && !dx && !dgamma && !dbeta) return CS_OK;
  if (rows == 0) {
    // an empty batch still defines dgamma/dbeta: zero unless accumulating;
    // nothing to launch for that without rows, so leave it to the caller
    return CS_OK;
  }
  if (!dy || !x || !mean || !rstd || (dx && !gamma)) return CS_ERR_INVALID_ARGUMENT;
  if (dres && !dx) return CS_ERR_INVALID_ARGUMENT;
  if (dres && !aligned_to(dres, dtype_size(dx_dtype))) return CS_ERR_MISALIGNED;
  if (!aligned_to(dy, dtype_size(dy_dtype)) || !aligned_to(x, dtype_size(x_dtype)) ||
      (dx && !aligned_to(dx, dtype_size(dx_dtype))) ||
      (gamma && !aligned_to(gamma, dtype_size(param_dtype))) ||
      (dgamma && !aligned_to(dgamma, dtype_size(param_dtype))) ||
      (dbeta && !aligned_to(dbeta, dtype_size(param_dtype))) || !aligned_to(mean, 4) ||
      !aligned_to(rstd, 4))
    return CS_ERR_MISALIGNED;
  const bool aligned = is_aligned16(dy) && is_aligned16(x) && (!dx || is_aligned16(dx)) &&
                       (!dx || is_aligned16(gamma)) && (!workspace || is_aligned16(workspace)) &&
                       (!dres || is_aligned16(dres));
  hipStream_t s = as_stream(stream);
#define CS_CALL(TDY, TX, TDX, TP)                                                              \
  return bwd_typed<TDY, TX, TDX, TP>(dy, x, mean, rstd, gamma, dx, dgamma, dbeta, workspace,   \
                                     workspace_bytes, rows, C, aligned, x_dtype, accumulate, dres, s, phase, \
                                     pending)
  const bool dy_wide = dy_dtype != x_dtype, dx_wide = dx_dtype != x_dtype,
             p_wide = param_dtype != x_dtype;
  switch (x_dtype) {
    case CS_F32: CS_CALL(float, float, float, float);
    case CS_F64: CS_CALL(double, double, double, double);
    case CS_F16:
      // autocast runs: fp32 dy and dx with fp32 parameters; plain runs: all f16
      if (dy_wide && dx_wide && p_wide) CS_CALL(float, f16_t, float, float);
      if (!dy_wide && !dx_wide && p_wide) CS_CALL(f16_t, f16_t, f16_t, float);
      if (!dy_wide && !dx_wide && !p_wide) CS_CALL(f16_t, f16_t, f16_t, f16_t);
      return CS_ERR_UNSUPPORTED;
    case CS_BF16:
      if (dy_wide && dx_wide && p_wide) CS_CALL(float, bf16_t, float, float);
      if (!dy_wide && !dx_wide && p_wide) CS_CALL(bf16_t, bf16_t, bf16_t, float);
      if (!dy_wide && !dx_wide && !p_wide) CS_CALL(bf16_t, bf16_t, bf16_t, bf16_t);
      return CS_ERR_UNSUPPORTED;
  }
#undef CS_CALL
  return CS_ERR_UNSUPPORTED;
}
}  // namespace

extern "C" int cs_layernorm_backward(const void *dy, const void *x, const void *mean,
                                     const void *rstd, const void *gamma, void *dx, void *dgamma,
                                     void *dbeta, void *workspace, size_t workspace_bytes,
                                     int64_t rows, int64_t C, int dy_dtype, int x_dtype,
                                     int dx_dtype, int param_dtype, int accumulate, void *stream) {
  return ln_backward(dy, x, mean, rstd, gamma, nullptr, dx, dgamma, dbeta, workspace, workspace_bytes,
                     rows, C, dy_dtype, x_dtype, dx_dtype, param_dtype, accumulate, stream);
}

extern "C" int cs_layernorm_backward_add(const void *dy, const void *x, const void *mean,
                                         const void *rstd, const void *gamma,
                                         const void *dresidual, void *dx, void *dgamma,
                                         void *dbeta, void *workspace, size_t workspace_bytes,
                                         int64_t rows, int64_t C, int dy_dtype, int x_dtype,
                                         int dx_dtype, int param_dtype, int accumulate,
                                         void *stream) {
  if (rows > 0 && (!dresidual || !dx)) return CS_ERR_INVALID_ARGUMENT;
  return ln_backward(dy, x, mean, rstd, gamma, dresidual, dx, dgamma, dbeta, workspace,
                     workspace_bytes, rows, C, dy_dtype, x_dtype, dx_dtype, param_dtype, accumulate,
                     stream);
}

extern "C" int64_t cs_layernorm_backward_partial_rows(int64_t rows, int64_t C, int x_dtype) {
  if (rows <= 0 || C <= 0 || dtype_size(x_dtype) == 0) return 0;
  const BwdPlan b = bwd_plan(rows, C, x_dtype, true);
  return b.two_calls ? b.blocks : 0;
}

extern "C" int cs_layernorm_backward_one_launch(int64_t rows, int64_t C, int x_dtype) {
  if (rows <= 0 || C <= 0 || dtype_size(x_dtype) == 0) return 0;
  return direct_sums(bwd_plan(rows, C, x_dtype, true), rows) ? 1 : 0;
}

extern "C" int cs_layernorm_backward_rows(const void *dy, const void *x, const void *mean,
                                          const void *rstd, const void *gamma,
                                          const void *dresidual, void *dx, void *partials,
                                          size_t partials_bytes, int64_t rows, int64_t C,
                                          int dy_dtype, int x_dtype, int dx_dtype,
                                          int param_dtype, void *stream) {
  if (rows <= 0 || C <= 0 || !partials || !gamma) return CS_ERR_INVALID_ARGUMENT;
  if (dresidual && !dx) return CS_ERR_INVALID_ARGUMENT;
  return ln_backward(dy, x, mean, rstd, gamma, dresidual, dx, nullptr, nullptr, partials,
                     partials_bytes, rows, C, dy_dtype, x_dtype, dx_dtype, param_dtype, 0, stream,
                     kBwdRowsOnly);
}

extern "C" int cs_layernorm_backward_finalize(const void *partials, int64_t partial_rows,
                                              void *dgamma, void *dbeta, int64_t C, int x_dtype,
                                              int param_dtype, int accumulate, void *stream) {
  if (C <= 0 || partial_rows <= 0 || !partials) return CS_ERR_INVALID_ARGUMENT;
  if (dtype_size(x_dtype) == 0 || dtype_size(param_dtype) == 0 || x_dtype == CS_F64 ||
      !wide_ok(x_dtype, param_dtype))
    return CS_ERR_UNSUPPORTED;
  if (C % (16 / (int)dtype_size(x_dtype)) != 0 || partial_rows > kLnMaxPartialRows) return CS_ERR_INVALID_ARGUMENT;
  const int vn = partial_vn(x_dtype);
  const PartialRows kind = kept_rows(C, x_dtype);
  if (!dgamma && !dbeta) return CS_OK;
  if (!is_aligned16(partials) || (dgamma && !aligned_to(dgamma, dtype_size(param_dtype))) ||
      (dbeta && !aligned_to(dbeta, dtype_size(param_dtype))))
    return CS_ERR_MISALIGNED;
  hipStream_t s = as_stream(stream);
  switch (param_dtype) {
    case CS_F32: return launch_finalize<float>(kind, partials, partial_rows, dgamma, dbeta, C, vn, accumulate, s);
    case CS_F16: return launch_finalize<f16_t>(kind, partials, partial_rows, dgamma, dbeta, C, vn, accumulate, s);
    case CS_BF16: return launch_finalize<bf16_t>(kind, partials, partial_rows, dgamma, dbeta, C, vn, accumulate, s);
  }
  return CS_ERR_UNSUPPORTED;
}

extern "C" int cs_layernorm_backward_rows_pending(const void *dy, const void *x, const void *mean,
                                                  const void *rstd, const void *gamma,
                                                  const void *dresidual, void *dx, void *partials,
                                                  size_t partials_bytes, const void *pending_partials,
                                                  int64_t pending_partial_rows, void *pending_dgamma,
                                                  void *pending_dbeta, int pending_accumulate,
                                                  int64_t rows, int64_t C, int dy_dtype, int x_dtype,
                                                  int dx_dtype, int param_dtype, void *stream) {
  if (rows <= 0 || C <= 0 || !partials || !gamma) return CS_ERR_INVALID_ARGUMENT;
  if (dresidual && !dx) return CS_ERR_INVALID_ARGUMENT;
  PendingSums pending;
  if (pending_partials != nullptr) {
    if (pending_partial_rows <= 0 || pending_partial_rows > kLnMaxPartialRows) return CS_ERR_INVALID_ARGUMENT;
    // the sums are read while this call's partial rows are written: they cannot share memory
    const char *a = (const char *)pending_partials, *b = (const char *)partials;
    const size_t pend_bytes = (size_t)pending_partial_rows * 2 * (size_t)C * sizeof(float);
    if (a < b + partials_bytes && b < a + pend_bytes) return CS_ERR_INVALID_ARGUMENT;
    if (!is_aligned16(pending_partials) || (pending_dgamma && !aligned_to(pending_dgamma, dtype_size(param_dtype))) ||
        (pending_dbeta && !aligned_to(pending_dbeta, dtype_size(param_dtype))))
      return CS_ERR_MISALIGNED;
    pending.partial = pending_partials;
    pending.nparts = pending_partial_rows;
    pending.dgamma = pending_dgamma;
    pending.dbeta = pending_dbeta;
    pending.accumulate = pending_accumulate;
  }
  return ln_backward(dy, x, mean, rstd, gamma, dresidual, dx, nullptr, nullptr, partials,
                     partials_bytes, rows, C, dy_dtype, x_dtype, dx_dtype, param_dtype, 0, stream,
                     kBwdRowsOnly, pending);
}
