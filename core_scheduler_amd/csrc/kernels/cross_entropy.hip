// Fused classifier for gfx950: row softmax + cross-entropy loss + dlogits in
// one pass over the logits.
//
// Replaces at::log_softmax + at::nll_loss_forward
// (src/compute/cross_entropy.cpp:57-63) and at::nll_loss_backward +
// at::_log_softmax_backward_data (:103-109), which between them make about
// five passes over [N, V] and keep three [N, V] temporaries:
//   loss_i    = logsumexp(x_i) - x_i[t_i]            (0 for ignored rows)
//   loss      = sum_i loss_i / #{not ignored}        (MEAN)  |  sum_i loss_i (SUM)
//   dlogits_i = (softmax(x_i) - onehot(t_i)) * s,    s = dloss / #{not ignored} (MEAN) | dloss
//
// A row is read from HBM once and its gradient written once: 2 accesses per
// element.  Which kernel does that depends on the row's width:
//   up to 2048 vectors of 16 bytes   ce_rows_kernel: one workgroup per row, the row in
//   (4096 of many rows)              registers, exact two-step max and sum (wave64
//                                    butterfly, then LDS across the waves)
//   up to 7168 (8192 at fp32)        ce_rows_stream_kernel: one persistent workgroup per
//                                    CU that loads the next row while it works on the
//                                    current one (50257 bf16 = 6283 vectors = 7 per lane)
//   up to 20480 with a gradient      ce_rows_hold_kernel: one persistent workgroup per CU keeps
//                                    one row and loads the next into the registers it frees
//   the loss alone of many rows      ce_loss_rows_kernel: one workgroup per row, nothing kept
//   up to 16384 fp32 vectors of the  ce_rows_kernel with 1024 lanes (the loss alone, and the gradient
//   few rows the last two leave      of a few rows more than there are CUs)
//   wider, or the loss alone of a    ce_rows_wide_kernel: two sweeps over the row, the
//   few rows                         second one served by the cache
//   fp64, unaligned base pointers    ce_rows_general_kernel
// Probabilities are 2^(x*log2e - max*log2e) / sum with one fma and one hardware exp2 per
// element; the row loss is ln(sum) - (x_t - max).
#include "common.hpp"

#include <math.h>

#include <atomic>
#include <type_traits>

namespace cs_hip {
namespace {

constexpr float kLog2e = 1.44269504088896340736f;
constexpr float kLn2 = 0.69314718055994530942f;

// workspace: [0] int32 count of rows not ignored, [1] float the same number,
// then (from byte 256) N floats of row loss when the caller keeps none.
constexpr size_t kWsHeader = 256;

__device__ __forceinline__ bool target_counts(int64_t t, int64_t V, int64_t ignore_index) {
  return t != ignore_index && t >= 0 && t < V;
}

// Both one-workgroup kernels below keep kSmallInFlight loads per lane in flight: with one load
// at a time a quarter of a million rows took 75 us each.
constexpr int kSmallInFlight = 8;

// What one lane, and then the workgroup, knows of the rows: a loss, how many count, and the sum of their class weights.
struct RowSums {
  float loss;
  int count;
  float weight;
};
// Lane t's rows t, t + 1024, ...: `load` a step's, each its own before the first is used (a row past the end re-reads the
// last one), then `use` them.  One row a lane where there are no more: eight loads for one cost 0.3 us.
template <int ROWS, typename Load, typename Use>
__device__ __forceinline__ void rows_of_lane_by(int64_t N, Load &&load, Use &&use) {
  for (int64_t i0 = threadIdx.x; i0 < N; i0 += (int64_t)1024 * ROWS) {
#pragma unroll
    for (int u = 0; u < ROWS; ++u) {
      const int64_t i = i0 + (int64_t)u * 1024;
      load(u, i < N ? i : N - 1);
    }
#pragma unroll
    for (int u = 0; u < ROWS; ++u) use(u, i0 + (int64_t)u * 1024 < N);
  }
}
template <typename Load, typename Use>
__device__ __forceinline__ void rows_of_lane(int64_t N, Load &&load, Use &&use) {
  if (N <= 1024) {  // kernel-uniform
    rows_of_lane_by<1>(N, load, use);
  } else {
    rows_of_lane_by<kSmallInFlight>(N, load, use);
  }
}
// Lane t's share of the count and the weights, these in kSmallInFlight interleaved sums.
__device__ __forceinline__ void count_rows(RowSums &sums, const int64_t *__restrict__ targets, int64_t N, int64_t V,
                                           int64_t ignore_index, const float *__restrict__ class_weight) {
  int64_t t[kSmallInFlight];
  if (class_weight == nullptr) {  // kernel-uniform
    rows_of_lane(
        N, [&](int u, int64_t i) { t[u] = targets[i]; },
        [&](int u, bool there) { sums.count += there && target_counts(t[u], V, ignore_index); });
    return;
  }
  float w[kSmallInFlight], wsum[kSmallInFlight];
#pragma unroll
  for (int u = 0; u < kSmallInFlight; ++u) wsum[u] = 0.f;
  rows_of_lane(
      N,
      [&](int u, int64_t i) {
        t[u] = targets[i];
        w[u] = class_weight[target_counts(t[u], V, ignore_index) ? t[u] : 0];
      },
      [&](int u, bool there) {
        const bool counts = there && target_counts(t[u], V, ignore_index);
        sums.count += counts;
        wsum[u] += counts ? w[u] : 0.f;
      });
#pragma unroll
  for (int u = 0; u < kSmallInFlight; ++u) sums.weight += wsum[u];
}
// The workgroup's sums, for its first wave, with one exchange: each in the order of block_reduce.  (The weights only where
// there are any.)
template <bool LOSS>
__device__ __forceinline__ RowSums block_sums(RowSums s, bool weighted) {
  __shared__ float loss_of[16], weight_of[16];
  __shared__ int count_of[16];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
  if constexpr (LOSS) s.loss = wave_reduce(s.loss, SumOp{});
  s.count = wave_reduce(s.count, SumOp{});
  if (weighted) s.weight = wave_reduce(s.weight, SumOp{});  // workgroup-uniform
  if (lane == 0) {
    if constexpr (LOSS) loss_of[wave] = s.loss;
    count_of[wave] = s.count;
    if (weighted) weight_of[wave] = s.weight;
  }
  __syncthreads();
  if (wave != 0) return s;
  const bool mine = lane < 16;
  if constexpr (LOSS) s.loss = wave_reduce(mine ? loss_of[lane & 15] : 0.f, SumOp{});
  s.count = wave_reduce(mine ? count_of[lane & 15] : 0, SumOp{});
  if (weighted) s.weight = wave_reduce(mine ? weight_of[lane & 15] : 0.f, SumOp{});
  return s;
}

// The same number for a row kernel of few rows, by every wave for itself: eight targets a lane, all requested at once,
// and no launch ahead of the rows.  Only the gradient of a mean without class weights asks (see ce_run).
constexpr int64_t kCountInRows = 8 * kWave;
__device__ __forceinline__ int rows_that_count(const int *__restrict__ ws_count, const int64_t *__restrict__ targets,
                                               int64_t N, int64_t V, int64_t ignore_index) {
  if (ws_count != nullptr) return *ws_count;  // kernel-uniform: a launch ahead has counted
  const int lane = threadIdx.x & (kWave - 1), n = (int)N;
  int64_t t[kCountInRows / kWave];
#pragma unroll
  for (int u = 0; u < kCountInRows / kWave; ++u) {
    const int i = u * kWave + lane;
    t[u] = targets[i < n ? i : n - 1];
  }
  int c = 0;
#pragma unroll
  for (int u = 0; u < kCountInRows / kWave; ++u)
    c += __popcll(__ballot(u * kWave + lane < n && target_counts(t[u], V, ignore_index)));
  return c;
}

__global__ __launch_bounds__(1024) void ce_count_kernel(const int64_t *__restrict__ targets,
                                                        int64_t N, int64_t V,
                                                        int64_t ignore_index,
                                                        int *__restrict__ ws_count,
                                                        float *__restrict__ ws_weight,
                                                        const float *__restrict__ class_weight) {
  RowSums sums{0.f, 0, 0.f};
  count_rows(sums, targets, N, V, ignore_index, class_weight);
  sums = block_sums<false>(sums, class_weight != nullptr);
  if (threadIdx.x == 0) {
    *ws_count = sums.count;
    // without class weights every row that counts weighs 1
    *ws_weight = class_weight != nullptr ? sums.weight : (float)sums.count;
  }
}

// Fixed-order sum of the row losses: thread t adds rows t, t+1024, ... into kSmallInFlight
// interleaved sums, which are then added in order; the 1024 sub-sums are folded by the
// butterfly.  Independent of scheduling.
//
// COUNT: the rows are counted here and not by a launch ahead of the row pass, whose gradient needs the
// count for a mean and for nothing else.  The loss alone of [509,50257] bf16: 19.4 -> 16.1 us per call,
// [4096,50304] 86.7 -> 84.4, [16,1000] fp32 17.3 (24.3 with the launch and a slower way to it).
template <bool COUNT>
__global__ __launch_bounds__(1024) void ce_reduce_kernel(const float *__restrict__ row_loss,
                                                         int64_t N, int *__restrict__ ws_count,
                                                         int reduction, float *__restrict__ loss,
                                                         float *__restrict__ total_weight,
                                                         const int64_t *__restrict__ targets, int64_t V,
                                                         int64_t ignore_index,
                                                         const float *__restrict__ class_weight) {
  const int tid = threadIdx.x;
  float v[kSmallInFlight], part[kSmallInFlight];
#pragma unroll
  for (int u = 0; u < kSmallInFlight; ++u) part[u] = 0.f;
  rows_of_lane(
      N, [&](int u, int64_t i) { v[u] = row_loss[i]; }, [&](int u, bool there) { part[u] += there ? v[u] : 0.f; });
  RowSums sums{0.f, 0, 0.f};
#pragma unroll
  for (int u = 0; u < kSmallInFlight; ++u) sums.loss += part[u];
  if constexpr (COUNT) count_rows(sums, targets, N, V, ignore_index, class_weight);
  sums = block_sums<true>(sums, COUNT && class_weight != nullptr);
  if (tid == 0) {
    // the float next to the count: the number of rows that count, or the sum of their class weights
    float total;
    if constexpr (COUNT) {
      total = class_weight != nullptr ? sums.weight : (float)sums.count;
      *ws_count = sums.count;
      reinterpret_cast<float *>(ws_count)[1] = total;
    } else {
      total = reinterpret_cast<const float *>(ws_count)[1];
    }
    if (loss) *loss = reduction == CS_REDUCTION_MEAN ? sums.loss / total : sums.loss;
    if (total_weight) *total_weight = total;
  }
}

constexpr int kNarrowMostThreads = 1024;
template <typename T>
__device__ __forceinline__ float vec_get(const Vec16<T> &v, int k) {
  return to_acc(v.e[k]);
}

// TD is the dlogits storage: T, or float when the caller wants fp32 gradients
// for 16-bit logits.
template <typename T, typename TD, int N_ELEMS>
__device__ __forceinline__ void store_out(TD *p, const float (&o)[N_ELEMS]) {
  constexpr int DN = Vec16<TD>::n;
#pragma unroll
  for (int q = 0; q < N_ELEMS / DN; ++q) {
    Vec16<TD> v;
#pragma unroll
    for (int k = 0; k < DN; ++k) v.e[k] = from_acc<TD>(o[q * DN + k]);
    store16_stream(p + q * DN, v);
  }
}

// The same for a vector that starts at column c0 of a row that does not own all of it.
template <typename TD, int N_ELEMS>
__device__ __forceinline__ void store_own(TD *p, const float (&o)[N_ELEMS], int c0, int stride) {
#pragma unroll
  for (int k = 0; k < N_ELEMS; ++k)
    if (c0 + k >= 0 && c0 + k < stride) p[k] = from_acc<TD>(o[k]);
}

// elements of T in a 128-byte line
template <typename T>
constexpr int kLineElems = 128 / (int)sizeof(T);

// EPV elements of T in one 8- or 16-byte access.  The streaming kernel reads 16-bit logits 8
// bytes per lane when it writes fp32 gradients, so that every store is a full 16 bytes per lane
// and a wave's store covers one contiguous kilobyte (with 16-byte loads each lane would own 32
// output bytes and every store instruction would touch only half of each 64-byte line).
template <typename T, int EPV>
struct alignas(EPV * sizeof(T)) VecE {
  T e[EPV];
};
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
template <typename T, int EPV>
__device__ __forceinline__ VecE<T, EPV> load_e_stream(const T *p) {
  static_assert(EPV * sizeof(T) == 16 || EPV * sizeof(T) == 8, "8- or 16-byte accesses");
  if constexpr (EPV * sizeof(T) == 16) {
    const u32x4 raw = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p));
    return __builtin_bit_cast(VecE<T, EPV>, raw);
  } else {
    const u32x2 raw = __builtin_nontemporal_load(reinterpret_cast<const u32x2 *>(p));
    return __builtin_bit_cast(VecE<T, EPV>, raw);
  }
}

// Waves per SIMD that a narrow row's registers have to allow: workgroups are short, and rows that make a little more than
// one round of the resident ones take two (fp16 [3000,3001] with fp32 gradients, 82 registers: 20.1 us, 16.3 with 80).
constexpr int narrow_waves(int bytes, int access) { return bytes > 64 ? 4 : access == 16 ? 8 : 6; }
// Narrow rows: a workgroup per row, the whole row in registers, VPT accesses of EPV elements a lane, all under way before
// the first is used; as many waves as the row has such shares.  RAGGED: lanes own aligned vectors of the whole array, as in
// the streaming kernel below.  What is no class column is overwritten with -inf in the packed registers, so that no pass
// masks element by element; a lane past the row's end loads its last vector again.
template <typename T, typename TD, int VPT, int EPV, bool RAGGED, int MOST_THREADS = kNarrowMostThreads>
__global__ __launch_bounds__(MOST_THREADS, narrow_waves(VPT *EPV * (int)sizeof(T), EPV * (int)sizeof(T))) void ce_rows_kernel(
    const T *logits, TD *dlogits, const int64_t *__restrict__ targets, float *__restrict__ row_loss,
    const int *__restrict__ ws_count, int64_t N, int64_t V, int64_t row_stride, int64_t ignore_index, int reduction,
    float dloss, const float *__restrict__ class_weight) {
  constexpr int VN = EPV;
  __shared__ float scratch[MOST_THREADS / kWave];
  const int64_t row = row_of_grid();
  if (row >= N) return;
  const int tid = threadIdx.x, block = blockDim.x;
  const int iV = (int)V, stride = (int)row_stride;
  const int off = RAGGED ? (int)((row * row_stride) & (kLineElems<T> - 1)) : 0;
  const int nvec = RAGGED ? (off + stride + VN - 1) / VN : stride / VN;
  const T *x = logits + row * row_stride - off;
  TD *d = dlogits + row * row_stride - off;
  const int64_t target = targets[row];
  const bool counts = target_counts(target, V, ignore_index);  // block-uniform
  // a vector the row does not own all of
  auto shared_vector = [&](int c0) { return RAGGED && (c0 < 0 || c0 + VN > stride); };

  if (!counts) {
    if (tid == 0 && row_loss) row_loss[row] = 0.f;
    if (dlogits) {
      float z[VN];
#pragma unroll
      for (int k = 0; k < VN; ++k) z[k] = 0.f;
      for (int idx = tid; idx < nvec; idx += block) {
        const int c0 = idx * VN - off;
        if (shared_vector(c0)) {
          store_own<TD, VN>(d + (int64_t)idx * VN, z, c0, stride);
        } else {
          store_out<T, TD, VN>(d + (int64_t)idx * VN, z);
        }
      }
    }
    return;
  }

  float scale = dloss;
  if (reduction == CS_REDUCTION_MEAN)
    scale = dloss / (class_weight ? reinterpret_cast<const float *>(ws_count)[1]
                                  : (float)rows_that_count(ws_count, targets, N, V, ignore_index));
  const float wt = class_weight ? class_weight[target] : 1.f;
  scale *= wt;
  // The array's last vector may not lie whole inside it: that of the last row, and of rows shorter than a vector ahead of
  // it.  Where such a row has no other, nothing is loaded in one piece.
  const int whole = nvec - (RAGGED && row * row_stride - off + (int64_t)nvec * VN > N * row_stride ? 1 : 0);
  VecE<T, EPV> xr[VPT] = {};
  if (!RAGGED || whole > 0) {  // block-uniform
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      const int idx = tid + block * j;
      xr[j] = load_e_stream<T, EPV>(x + (int64_t)(idx < whole ? idx : whole - 1) * VN);
    }
  }
  const float x_t = tid == 0 ? to_acc(x[off + target]) : 0.f;
  if (RAGGED && whole < nvec) {  // block-uniform
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      if (tid + block * j == nvec - 1) {
#pragma unroll
        for (int k = 0; k < VN; ++k) {
          const int c = (nvec - 1) * VN - off + k;
          xr[j].e[k] = x[off + (c < stride ? c : 0)];
        }
      }
    }
  }

  // ---- row maximum
  float m = -INFINITY;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    const int c0 = (tid + block * j) * VN - off;
    if (c0 + VN > iV || (RAGGED && j == 0 && c0 < 0)) {
#pragma unroll
      for (int k = 0; k < VN; ++k)
        if (c0 + k >= iV || (RAGGED && j == 0 && c0 + k < 0)) xr[j].e[k] = from_acc<T>(-INFINITY);
    }
#pragma unroll
    for (int k = 0; k < VN; ++k) m = fmaxf(m, to_acc(xr[j].e[k]));
  }
  m = block_reduce(m, MaxOp{}, -INFINITY, scratch);
  const float m2 = m * kLog2e;

  // ---- sum of exponentials: a tree over the lane's elements, then the lanes
  float part[VPT];
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    float e[VN];
#pragma unroll
    for (int k = 0; k < VN; ++k) e[k] = __builtin_amdgcn_exp2f(__builtin_fmaf(to_acc(xr[j].e[k]), kLog2e, -m2));
#pragma unroll
    for (int w = VN / 2; w > 0; w /= 2)
#pragma unroll
      for (int k = 0; k < w; ++k) e[k] += e[k + w];
    part[j] = e[0];
  }
#pragma unroll
  for (int w = VPT; w > 1; w = (w + 1) / 2)
#pragma unroll
    for (int j = 0; j < w / 2; ++j) part[j] += part[j + (w + 1) / 2];
  const float s = block_reduce(part[0], SumOp{}, 0.f, scratch);

  const float log2_s = __builtin_amdgcn_logf(s);  // v_log_f32 is log2
  // loss = ln(sum exp(x - max)) - (x_t - max): the difference to the maximum is formed with one
  // fused multiply-add against the same rounded m2 the sum used, so a loss near 0 keeps its digits
  if (tid == 0 && row_loss) {
    const float l = (log2_s - __builtin_fmaf(x_t, kLog2e, -m2)) * kLn2;
    row_loss[row] = class_weight ? l * wt : l;
  }
  if (dlogits == nullptr) return;

  // ---- dlogits = (p - onehot) * scale with p = 2^(x*log2e - m2) / s.  The exponent is taken
  // relative to the row maximum with one fused multiply-add, the same expression the sum above
  // used, so the rounding of m2 cancels between numerator and denominator and p keeps fp32
  // accuracy; folding log2(s) and log2(scale) into the exponent instead costs ~1e-6 relative,
  // which the subtraction at the target column amplifies when p is close to 1.
  const float factor = scale / s;  // s >= 1: the maximum contributes 2^0
  const int t_at = (int)target + off, t_vec = t_at / VN, t_sub = t_at % VN;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    const int idx = tid + block * j;
    if (idx < nvec) {
      const int c0 = idx * VN - off;
      float o[VN];
#pragma unroll
      for (int k = 0; k < VN; ++k)
        o[k] = __builtin_amdgcn_exp2f(__builtin_fmaf(to_acc(xr[j].e[k]), kLog2e, -m2)) * factor;
      if (c0 + VN > iV) {  // last class vector and the padding: 0 also where the sum is not finite
#pragma unroll
        for (int k = 0; k < VN; ++k)
          if (c0 + k >= iV) o[k] = 0.f;
      }
      if (idx == t_vec) {
#pragma unroll
        for (int k = 0; k < VN; ++k)
          if (k == t_sub) o[k] -= scale;
      }
      if (shared_vector(c0)) {
        store_own<TD, VN>(d + (int64_t)idx * VN, o, c0, stride);
      } else {
        store_out<T, TD, VN>(d + (int64_t)idx * VN, o);
      }
    }
  }
}

// Element k of v as fp32.  fp16 is converted straight out of its half of the 32-bit register
// (the sub-dword select of the conversion instruction): shifting the upper half down first
// costs a temporary register per element, which the 13 x 4 plan does not have (the plans with
// 16-byte loads have, and keep the compiler's own sequence).
template <typename T, int EPV>
__device__ __forceinline__ float widen(const VecE<T, EPV> &v, int k) {
  if constexpr (std::is_same_v<T, f16_t> && EPV == 4) {
    typedef uint32_t words_t __attribute__((ext_vector_type(EPV / 2)));
    const words_t w = __builtin_bit_cast(words_t, v);
    const uint32_t word = w[k >> 1];
    float f;
    if (k & 1) {
      asm("v_cvt_f32_f16_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:WORD_1" : "=v"(f) : "v"(word));
    } else {
      asm("v_cvt_f32_f16_e32 %0, %1" : "=v"(f) : "v"(word));
    }
    return f;
  } else {
    return to_acc(v.e[k]);
  }
}

// Streaming variant for wide rows (the GPT-2 vocabulary): one 1024-lane
// workgroup per CU walks rows blockIdx.x, blockIdx.x + gridDim.x, ... and
// loads the next row into a second register set before it starts on the
// current one, so the CU's memory pipe stays busy while its VALUs work; the
// stores of a finished row drain under the next row's arithmetic.  Without
// this, all workgroups load, compute and store in lockstep and HBM idles for
// the whole compute phase.
//
// Each element costs one hardware exp2: lane-local max first, then
// e = 2^((x - m_lane) log2e) is kept in registers, one exchange of (max, sum)
// pairs across the 16 waves gives the row's max and sum, and the output is
// e * f with one per-lane factor f = 2^(m_lane*log2e - max*log2e) * scale / sum.
//
// HAS_W: per-class weights (nll_loss's `weight`): a row's gradient and loss carry w[target], and
// the mean divides by the sum of those weights, which the count launch left next to the count.
//
// RAGGED: the row stride is not a multiple of the access width (a vocabulary used unpadded), so rows
// start anywhere.  The lanes still own whole aligned vectors of the [N, stride] array, counted from the
// 128-byte line the row starts in; elements of the neighbouring rows count as padding, and a vector that
// a row owns only part of is written element by element.  [8192,50257] unpadded bf16: 289 us against 366
// in two sweeps (padded rows 287), with fp32 gradients [6000,50257] 341 against 442.  Counted from the
// nearest 16-byte vector instead of the line, so that every access of a wave straddles lines: 312 and 373.
template <typename T, typename TD, int VPT, int EPV, bool HAS_W, bool RAGGED>
__global__ __launch_bounds__(1024) void ce_rows_stream_kernel(
    const T *logits, TD *dlogits, const int64_t *__restrict__ targets, float *__restrict__ row_loss,
    const int *__restrict__ ws_count, int64_t N, int64_t V, int64_t row_stride,
    int64_t ignore_index, int reduction, float dloss, const float *__restrict__ class_weight) {
  constexpr int BLOCK = 1024;
  constexpr int VN = EPV;  // elements per lane per access
  constexpr int kWaves = BLOCK / kWave;
  __shared__ float red_m[2][kWaves], red_s[2][kWaves];
  int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid >> 6;
  const int iV = (int)V;
  const int nvec_even = (int)(row_stride / VN);
  // A ragged row: elements between the 128-byte line it starts in and its start, vectors from that line
  // to its end, and how many of these lie whole inside the array (all but perhaps the last row's last
  // one).  From the line, not only from the nearest vector, so that the waves' accesses cover whole lines.
  auto off_of = [&](int64_t r) { return RAGGED ? (int)((r * row_stride) & (kLineElems<T> - 1)) : 0; };
  auto vecs_of = [&](int off) { return RAGGED ? (int)((off + row_stride + VN - 1) / VN) : nvec_even; };
  auto whole_of = [&](int64_t r, int off) {
    return vecs_of(off) - (RAGGED && r == N - 1 && (off + (int)row_stride) % VN != 0 ? 1 : 0);
  };

  float scale0 = dloss;
  if (reduction == CS_REDUCTION_MEAN)
    scale0 = dloss / (HAS_W ? reinterpret_cast<const float *>(ws_count)[1]
                            : (float)rows_that_count(ws_count, targets, N, V, ignore_index));
  [[maybe_unused]] const float log2_scale0 = __builtin_amdgcn_logf(fabsf(scale0));  // -inf for 0: every output 0

  // Workgroups go round the eight XCDs in launch order.  The workgroups of one XCD take
  // neighbouring rows of each round of gridDim rows (XCD 0 the first eighth, and so on) rather
  // than every eighth row: [8192,50257] bf16 282.7 us per call against 285.2, with fp32 gradients
  // 444.5 against 450.8.
  int64_t row = (gridDim.x % 8 == 0) ? (int64_t)(blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8 : blockIdx.x;
  VecE<T, EPV> cur[VPT];
  int64_t tgt = 0;
  bool live = false;
  float x_t = 0.f, wt = 1.f;
  if (row < N) {
    tgt = targets[row];
    live = target_counts(tgt, V, ignore_index);
    if (live) {
      if constexpr (HAS_W) wt = class_weight[tgt];
      const int off = off_of(row), nload = whole_of(row, off);
      const T *x = logits + row * row_stride - off;
#pragma unroll
      for (int j = 0; j < VPT; ++j) {
        const int idx = tid + BLOCK * j;
        if (idx < nload) cur[j] = load_e_stream<T, EPV>(x + (int64_t)idx * VN);
      }
      if (tid == 0) x_t = to_acc(x[off + tgt]);
    }
  }
  int parity = 0;
  while (row < N) {
    if constexpr (RAGGED) asm volatile("" : "+v"(tid));  // a lane's column offsets, kept from row to row, would spill
    // ---- issue the next row's loads
    const int64_t nrow = row + gridDim.x;
    VecE<T, EPV> nxt[VPT];
    int64_t ntgt = 0;
    bool nlive = false;
    float nx_t = 0.f, nwt = 1.f;
    if (nrow < N) {
      ntgt = targets[nrow];
      nlive = target_counts(ntgt, V, ignore_index);
      if (nlive) {
        if constexpr (HAS_W) nwt = class_weight[ntgt];
        const int off = off_of(nrow), nload = whole_of(nrow, off);
        const T *x = logits + nrow * row_stride - off;
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
          const int idx = tid + BLOCK * j;
          // (kept under the lane's condition here: the compiler issues these back to back as they
          // are, and the unconditional form spills 56 bytes per lane: 283 -> 305 us)
          if (idx < nload) nxt[j] = load_e_stream<T, EPV>(x + (int64_t)idx * VN);
        }
        if (tid == 0) nx_t = to_acc(x[off + ntgt]);
      }
    }

    const int off = off_of(row), nvec = vecs_of(off);
    if (!live) {
      if (tid == 0 && row_loss) row_loss[row] = 0.f;
      if (dlogits) {
        float z[VN];
#pragma unroll
        for (int k = 0; k < VN; ++k) z[k] = 0.f;
        for (int idx = tid; idx < nvec; idx += BLOCK) {
          const int c0 = idx * VN - off;
          if (RAGGED && (c0 < 0 || c0 + VN > (int)row_stride)) {
            store_own<TD, VN>(dlogits + row * row_stride + c0, z, c0, (int)row_stride);
          } else {
            store_out<T, TD, VN>(dlogits + row * row_stride - off + (int64_t)idx * VN, z);
          }
        }
      }
    } else {
      if (RAGGED && row == N - 1 && whole_of(row, off) < nvec) {  // the array's last vector is not whole
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
          const int idx = tid + BLOCK * j;
          if (idx == nvec - 1) {
#pragma unroll
            for (int k = 0; k < VN; ++k) {
              const int c = idx * VN - off + k;
              cur[j].e[k] = logits[row * row_stride + (c < (int)row_stride ? c : 0)];
            }
          }
        }
      }
      // ---- widen, mask what is not a class column to -inf, lane-local max
      float e[VPT][VN];
      float m = -INFINITY;
#pragma unroll
      for (int j = 0; j < VPT; ++j) {
        const int c0 = (tid + BLOCK * j) * VN - off;
        const bool starts_before = RAGGED && j == 0 && c0 < 0;
        if (c0 + VN <= iV && !starts_before) {
#pragma unroll
          for (int k = 0; k < VN; ++k) {
            e[j][k] = widen(cur[j], k);
            m = fmaxf(m, e[j][k]);
          }
        } else {
#pragma unroll
          for (int k = 0; k < VN; ++k) {
            const bool mine = c0 + k < iV && !(RAGGED && j == 0 && c0 + k < 0);
            e[j][k] = mine ? widen(cur[j], k) : -INFINITY;
            m = fmaxf(m, e[j][k]);
          }
        }
      }
      // a lane without any class column: any finite stand-in keeps 2^(-inf - m) = 0
      const float ml2 = (m == -INFINITY ? 0.f : m) * kLog2e;
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < VPT; ++j)
#pragma unroll
        for (int k = 0; k < VN; ++k) {
          e[j][k] = __builtin_amdgcn_exp2f(e[j][k] * kLog2e - ml2);
          if constexpr (!RAGGED) s += e[j][k];
        }
      // Once a dominant term sits in s, every further add rounds at its size: unpadded rows, which the two-sweep
      // kernel took before, are added pairwise within 16 elements and once onto the running sum, as there
      // (1.3e-7 rms in the loss of confident rows; 2.5e-7 one element after the other)
      if constexpr (RAGGED) {
        constexpr int CH = 16 / VN;
        float part[CH];
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
          float c[VN];
#pragma unroll
          for (int k = 0; k < VN; ++k) c[k] = e[j][k];
#pragma unroll
          for (int w = VN / 2; w > 0; w /= 2)
#pragma unroll
            for (int k = 0; k < w; ++k) c[k] += c[k + w];
          part[j % CH] = c[0];
          if (j % CH == CH - 1 || j == VPT - 1) {
#pragma unroll
            for (int u = j % CH + 1; u < CH; ++u) part[u] = 0.f;
#pragma unroll
            for (int w = CH / 2; w > 0; w /= 2)
#pragma unroll
              for (int u = 0; u < w; ++u) part[u] += part[u + w];
            s += part[0];
          }
        }
      }
      // ---- (max, sum) across the wave, then across the 16 waves.  A lane without a finite
      // value brings its sum as it is, 0 or the NaN it met: its stand-in maximum must not pass for a
      // real one (the real ones may all lie far below it), and its sum must not meet an overflowed 2^(0 - max)
      const bool empty = m == -INFINITY;
      const float mw2 = wave_reduce(empty ? -INFINITY : ml2, MaxOp{});
      const float sw = wave_reduce(empty ? s : s * __builtin_amdgcn_exp2f(ml2 - mw2), SumOp{});
      if (lane == 0) {
        red_m[parity][wave] = mw2;
        red_s[parity][wave] = sw;
      }
      __syncthreads();
      const float pm = lane < kWaves ? red_m[parity][lane] : -INFINITY;
      const float ps = lane < kWaves ? red_s[parity][lane] : 0.f;
      const float M2 = wave_reduce(pm, MaxOp{});
      const float S = wave_reduce(pm == -INFINITY ? ps : ps * __builtin_amdgcn_exp2f(pm - M2), SumOp{});
      parity ^= 1;  // the other pair of arrays next time: one barrier per row is enough
      const float log2_S = __builtin_amdgcn_logf(S);
      // loss = ln(sum exp(x - max)) - (x_t - max), the difference to the maximum formed with one
      // fused multiply-add against the rounded M2 the sum was taken with
      {
        const float l = (log2_S - __builtin_fmaf(x_t, kLog2e, -M2)) * kLn2;
        if (tid == 0 && row_loss) row_loss[row] = HAS_W ? l * wt : l;
      }
      // the row's scale: the call's, times the weight of the row's class
      const float scale = HAS_W ? scale0 * wt : scale0;

      if (RAGGED && dlogits && !(S > 0.f)) {
        // no finite logit, or a NaN or +inf among them: NaN for every class, 0 in the padding.  (Rows of whole
        // vectors give 0 for all but the target where no logit is finite, and a NaN row's padding is NaN; the
        // branch, in any form tried, costs them 1%: [8192,50257] bf16 285 -> 288 us.)
        for (int c = tid; c < (int)row_stride; c += BLOCK)
          dlogits[row * row_stride + c] = from_acc<TD>(c < iV ? __builtin_nanf("") : 0.f);
      } else if (dlogits) {
        // e was taken relative to the lane's maximum.  A lane that holds no class column has e = 0 everywhere;
        // give it f = 0 so that 0 * f cannot meet an overflowed factor
        float f;
        if constexpr (RAGGED) {
          f = empty ? 0.f : __builtin_amdgcn_exp2f(ml2 - M2) * (scale / S);
        } else {
          // The logarithms of sum and scale folded into the exponent: one instruction a row, at 4.8e-7 rms
          // of every element against 2.4e-7.  Rows of whole vectors have always been formed so, and have
          // no registers for more (the product spills 4 a lane at 7 vectors of bf16).
          const float log2_scale = HAS_W ? log2_scale0 + __builtin_amdgcn_logf(fabsf(wt)) : log2_scale0;
          f = empty ? 0.f : __builtin_amdgcn_exp2f(ml2 - M2 - log2_S + log2_scale);
          f = scale < 0.f ? -f : f;
        }
        const int t_at = (int)tgt + off;
        const int t_vec = t_at / VN, t_sub = t_at % VN;
        TD *d = dlogits + row * row_stride - off;
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
          const int idx = tid + BLOCK * j;
          if (idx < nvec) {
            float o[VN];
#pragma unroll
            for (int k = 0; k < VN; ++k) o[k] = e[j][k] * f;
            if (idx == t_vec) {
              // the folded factor's error would be amplified by subtracting `scale` when p is close to 1: the
              // target element is formed as a product
              const float exact = RAGGED ? f : __builtin_amdgcn_exp2f(ml2 - M2) * (scale * __builtin_amdgcn_rcpf(S));
#pragma unroll
              for (int k = 0; k < VN; ++k)
                if (k == t_sub) o[k] = e[j][k] * exact - scale;
            }
            // (written out here: as a lambda the store cost 56 bytes of scratch per lane)
            if (RAGGED && (idx * VN - off < 0 || idx * VN - off + VN > (int)row_stride)) {
              store_own<TD, VN>(d + (int64_t)idx * VN, o, idx * VN - off, (int)row_stride);
            } else {
              store_out<T, TD, VN>(d + (int64_t)idx * VN, o);
            }
          }
        }
      }
    }
#pragma unroll
    for (int j = 0; j < VPT; ++j) cur[j] = nxt[j];
    live = nlive;
    tgt = ntgt;
    x_t = nx_t;
    wt = nwt;
    row = nrow;
  }
}

// A packed access as 32-bit words: element k as fp32, and element k replaced.
template <typename T, int EPV>
struct Words {
  static constexpr int n = EPV * (int)sizeof(T) / 4;
  typedef uint32_t type __attribute__((ext_vector_type(EPV * sizeof(T) / 4)));
};
template <typename T, int EPV>
__device__ __forceinline__ float word_elem(const typename Words<T, EPV>::type &w, int k) {
  if constexpr (std::is_same_v<T, float>) {
    return __uint_as_float(w[k]);
  } else if constexpr (std::is_same_v<T, bf16_t>) {
    return __uint_as_float((k & 1) ? w[k >> 1] & 0xffff0000u : w[k >> 1] << 16);
  } else {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)((k & 1) ? w[k >> 1] >> 16 : w[k >> 1]));
  }
}
template <typename T, int EPV>
__device__ __forceinline__ void set_word_elem(typename Words<T, EPV>::type &w, int k, T v) {
  if constexpr (sizeof(T) == 4) {
    w[k] = __builtin_bit_cast(uint32_t, v);
  } else {
    const uint32_t b = __builtin_bit_cast(uint16_t, v);
    w[k >> 1] = (k & 1) ? (w[k >> 1] & 0xffffu) | b << 16 : (w[k >> 1] & 0xffff0000u) | b;
  }
}

// Rows too wide for two register sets (vocabularies of 57K to 160K at 16 bit, 32K to 80K at fp32): one
// persistent 1024-lane workgroup per CU keeps ONE row, packed, in its registers.  The first pass takes the
// running (max, sum) of the vectors as they arrive; the second forms each vector's gradient, stores it and
// loads the same vector of the next row into the registers just freed, so loads and stores go out
// side by side and the row is read from HBM once.  The two-sweep kernel below reads it again
// out of the caches.  Two exponentials per element (13 us of VALU time a row, by count) stay under the row's 20 us
// of memory time because both passes run while memory does.
//
// Per call, against two sweeps: [4096,128256] bf16 457 -> 401 us (5.2 TB/s), [4096,152064] 536 -> 478,
// [4096,100003] unpadded 374 -> 316, [2048,128256] with fp32 gradients 390 -> 308, [4096,60032] fp16
// 210 -> 189, [2048,80000] fp32 288 -> 257.  Having a quarter of the next row under way before the
// current one is finished (the registers allow it) did not matter, 400 us at [4096,128256] and 480 at 152064:
// the exchange between the passes is not what keeps the kernel from the streaming kernel's 5.8 TB/s.
//
// The registers hold the row and little else (20 vectors of 16 bytes are 80 of 128), so the row is kept as
// 32-bit words, and the empty asm statements keep the compiler from carrying widened elements
// from the first pass into the second or a lane's VPT offsets from row to row (both spill).
//
// VPT accesses of EPV elements per lane; RAGGED as in the streaming kernel.  Lanes past the row's
// end load its last vector again (one address per wave) instead of branching round the load.  Elements
// that are no class column are overwritten with -inf in the packed registers, so that neither pass masks
// element by element.
template <typename T, typename TD, int VPT, int EPV, bool RAGGED>
__global__ __launch_bounds__(1024) void ce_rows_hold_kernel(
    const T *logits, TD *dlogits, const int64_t *__restrict__ targets, float *__restrict__ row_loss,
    const int *__restrict__ ws_count, int64_t N, int64_t V, int64_t row_stride, int64_t ignore_index,
    int reduction, float dloss, const float *__restrict__ class_weight) {
  constexpr int BLOCK = 1024;
  constexpr int VN = EPV;
  constexpr int CH = 16 / VN;  // vectors per step of the first pass: 16 elements
  static_assert(VPT % CH == 0, "whole steps");
  constexpr int kWaves = BLOCK / kWave;
  __shared__ float red_m[2][kWaves], red_s[2][kWaves];
  using W = typename Words<T, EPV>::type;
  int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid >> 6;
  const int iV = (int)V, stride = (int)row_stride;
  auto off_of = [&](int64_t r) { return RAGGED ? (int)((r * row_stride) & (kLineElems<T> - 1)) : 0; };
  auto vecs_of = [&](int off) { return RAGGED ? (off + stride + VN - 1) / VN : stride / VN; };
  auto whole_of = [&](int64_t r, int off) {
    return vecs_of(off) - (RAGGED && r == N - 1 && (off + stride) % VN != 0 ? 1 : 0);
  };
  // vector j of this lane, of the row that starts at x; `last`: the last one to be loaded
  auto load = [&](const T *x, int j, int last) {
    const int idx = tid + BLOCK * j;
    const uint32_t bytes = (uint32_t)(idx < last ? idx : last) * (uint32_t)(VN * sizeof(T));
    return __builtin_nontemporal_load(reinterpret_cast<const W *>(reinterpret_cast<const char *>(x) + bytes));
  };

  float scale0 = dloss;
  if (reduction == CS_REDUCTION_MEAN)
    scale0 = dloss / (class_weight ? reinterpret_cast<const float *>(ws_count)[1]
                                   : (float)rows_that_count(ws_count, targets, N, V, ignore_index));

  // neighbouring rows on one XCD, as in the streaming kernel
  int64_t row = (gridDim.x % 8 == 0) ? (int64_t)(blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8 : blockIdx.x;
  if (row >= N) return;
  W cur[VPT];
  int64_t tgt = targets[row];
  bool live = target_counts(tgt, V, ignore_index);
  T x_t;
  {
    const int off = off_of(row), last = live ? whole_of(row, off) - 1 : 0;
    const T *x = logits + row * row_stride - off;
    x_t = x[off + (live ? tgt : 0)];
#pragma unroll
    for (int j = 0; j < VPT; ++j) cur[j] = load(x, j, last);
  }
  int parity = 0;
  for (;;) {
    asm volatile("" : "+v"(tid));
    // the next row; where there is none, or it is ignored, every load below is of one vector
    const int64_t nrow = row + gridDim.x;
    const bool more = nrow < N;
    const int64_t ntgt = targets[more ? nrow : row];
    const bool nlive = more && target_counts(ntgt, V, ignore_index);
    const int noff = more ? off_of(nrow) : 0;
    const T *nx = logits + (more ? nrow * row_stride - noff : 0);
    const int nlast = nlive ? whole_of(nrow, noff) - 1 : 0;
    const int off = off_of(row), nvec = vecs_of(off);
    TD *d = dlogits + row * row_stride - off;
    // An ignored row goes the same way as a row without class columns: no first pass, and zeros out.
    // (A branch of its own, with the next row's loads in it, makes the compiler spill the row.)
    const int vcols = live ? iV : 0, nsum = live ? nvec : 0;
    const float wt = class_weight && live ? class_weight[tgt] : 1.f;
    if (RAGGED && row == N - 1 && whole_of(row, off) < nvec) {  // the array's last vector is not whole
#pragma unroll
      for (int j = 0; j < VPT; ++j) {
        const int idx = tid + BLOCK * j;
        if (idx == nvec - 1) {
#pragma unroll
          for (int k = 0; k < VN; ++k) {
            const int c = idx * VN - off + k;
            set_word_elem<T, EPV>(cur[j], k, logits[row * row_stride + (c < stride ? c : 0)]);
          }
        }
      }
    }
    // ---- running maximum (times log2 e) and the sum relative to it
    float m2 = -INFINITY, s = 0.f;
#pragma unroll
    for (int q = 0; q < VPT / CH; ++q) {
      if (q * CH * BLOCK < nsum) {  // block-uniform
        float cm = -INFINITY;
        float xs[CH][VN];
#pragma unroll
        for (int u = 0; u < CH; ++u) {
          const int j = q * CH + u;
          const int c0 = (tid + BLOCK * j) * VN - off;
          if (c0 + VN > vcols || (RAGGED && j == 0 && c0 < 0)) {
#pragma unroll
            for (int k = 0; k < VN; ++k)
              if (c0 + k >= vcols || (RAGGED && j == 0 && c0 + k < 0)) set_word_elem<T, EPV>(cur[j], k, from_acc<T>(-INFINITY));
          }
#pragma unroll
          for (int k = 0; k < VN; ++k) {
            xs[u][k] = word_elem<T, EPV>(cur[j], k);
            cm = fmaxf(cm, xs[u][k]);
          }
        }
        const float cm2 = cm * kLog2e;
        if (cm2 > m2) {
          s *= __builtin_amdgcn_exp2f(m2 - cm2);  // 0 the first time (m2 = -inf, s = 0)
          m2 = cm2;
        }
        // nothing finite so far: every term is 2^-inf (or NaN) against any finite stand-in
        const float ref = m2 == -INFINITY ? 0.f : m2;
        // pairwise within the step and one add onto the running sum, as in the two-sweep kernel
        float part[CH];
#pragma unroll
        for (int u = 0; u < CH; ++u) {
          float e[VN];
#pragma unroll
          for (int k = 0; k < VN; ++k) e[k] = __builtin_amdgcn_exp2f(__builtin_fmaf(xs[u][k], kLog2e, -ref));
#pragma unroll
          for (int w = VN / 2; w > 0; w /= 2)
#pragma unroll
            for (int k = 0; k < w; ++k) e[k] += e[k + w];
          part[u] = e[0];
        }
#pragma unroll
        for (int w = CH / 2; w > 0; w /= 2)
#pragma unroll
          for (int u = 0; u < w; ++u) part[u] += part[u + w];
        s += part[0];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- (max, sum) across the wave, then across the waves.  A lane without a finite value
    // brings its sum as it is: 0, or the NaN it met.
    const float mw2 = wave_reduce(m2, MaxOp{});
    const float sw = wave_reduce(m2 == -INFINITY ? s : s * __builtin_amdgcn_exp2f(m2 - mw2), SumOp{});
    if (lane == 0) {
      red_m[parity][wave] = mw2;
      red_s[parity][wave] = sw;
    }
    lds_barrier();
    const float pm = lane < kWaves ? red_m[parity][lane] : -INFINITY;
    const float ps = lane < kWaves ? red_s[parity][lane] : 0.f;
    const float M2 = wave_reduce(pm, MaxOp{});
    const float S = wave_reduce(pm == -INFINITY ? ps : ps * __builtin_amdgcn_exp2f(pm - M2), SumOp{});
    parity ^= 1;  // the other pair of arrays next time: one barrier per row is enough
    const float scale = scale0 * wt;
    if (tid == 0 && row_loss) {
      const float l = (__builtin_amdgcn_logf(S) - __builtin_fmaf(to_acc(x_t), kLog2e, -M2)) * kLn2;
      row_loss[row] = live ? l * wt : 0.f;
    }
    const T nx_t = nx[noff + (nlive ? ntgt : 0)];
#pragma unroll
    for (int j = 0; j < VPT; ++j) asm volatile("" : "+v"(cur[j]));
    asm volatile("" : "+v"(tid));
    // ---- gradient (p - onehot) * scale with p = 2^(x log2e - M2) / S, and the next row's loads
    const float factor = scale / S;
    const int t_at = (int)tgt + off;
    const int t_vec = live ? t_at / VN : -1, t_sub = t_at % VN;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      const int idx = tid + BLOCK * j, c0 = idx * VN - off;
      if (j * BLOCK < nvec) {  // block-uniform
        float o[VN];
#pragma unroll
        for (int k = 0; k < VN; ++k)
          o[k] = __builtin_amdgcn_exp2f(__builtin_fmaf(word_elem<T, EPV>(cur[j], k), kLog2e, -M2)) * factor;
        if (idx == t_vec) {
#pragma unroll
          for (int k = 0; k < VN; ++k)
            if (k == t_sub) o[k] -= scale;
        }
        if (c0 + VN > vcols) {  // 0 also where the row's maximum or sum is not finite
#pragma unroll
          for (int k = 0; k < VN; ++k)
            if (c0 + k >= vcols) o[k] = 0.f;
        }
        if (idx < nvec) {
          if (RAGGED && (c0 < 0 || c0 + VN > stride)) {
            store_own<TD, VN>(d + (int64_t)idx * VN, o, c0, stride);
          } else {
            store_out<T, TD, VN>(d + (int64_t)idx * VN, o);
          }
        }
      }
      cur[j] = load(nx, j, nlast);
      __builtin_amdgcn_sched_barrier(0);  // a load hoisted above its vector's use would need registers of its own
    }
    if (!more) break;
    row = nrow;
    tgt = ntgt;
    live = nlive;
    x_t = nx_t;
  }
}

// The loss alone (validation) of rows beyond the small register plans: one workgroup per row, the row read
// once in chunks of four 16-byte vectors per lane, two chunks in registers (one on its way while the other
// joins the lane's running (max, sum)).  No row is kept and no workgroup lives longer than its row, so eight
// workgroups of 256 share a CU and cover each other's waits and exchanges, where the streaming kernel
// has one workgroup of 1024 per CU and one barrier per row between loads.  Bound by HBM reads.
//
// Per call, against the kernels for fewer rows: [8192,50257] bf16 152 -> 128 us (6.4 TB/s), [4096,50257] 81 -> 68,
// [8192,17000] 92 -> 52, [8192,128256] 357 -> 312, [4096,50257] fp16 89 -> 69, fp32 [4096,10000] 42 -> 28,
// [4096,50257] 141 -> 123, [4096,100000] 271 -> 240.
//
// Rows may start anywhere: vectors count from the 128-byte line a row starts in, as in the streaming
// kernel, and what is no class column counts as -inf.  Lanes past the row's end load its last vector again.
template <typename T, int BLOCK>
__global__ __launch_bounds__(BLOCK, 6) void ce_loss_rows_kernel(
    const T *__restrict__ logits, const int64_t *__restrict__ targets, float *__restrict__ row_loss, int64_t N,
    int64_t V, int64_t row_stride, int64_t ignore_index, const float *__restrict__ class_weight) {
  constexpr int VN = Vec16<T>::n;
  constexpr int U = 4, CH = 8 / VN;  // vectors per chunk, and of these per step of 8 elements
  constexpr int kWaves = BLOCK / kWave;
  __shared__ float red_m[kWaves], red_s[kWaves];
  using W = typename Words<T, VN>::type;
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int64_t row = blockIdx.x;
  const int64_t tgt = targets[row];
  if (!target_counts(tgt, V, ignore_index)) {
    if (tid == 0) row_loss[row] = 0.f;
    return;
  }
  const int stride = (int)row_stride;
  const int off = (int)((row * row_stride) & (kLineElems<T> - 1));
  const T *x = logits + row * row_stride - off;
  // Vectors that hold class columns.  The array's last one may not lie whole inside it: its columns
  // [iV, V) are then added one to a lane.
  int nvec = (int)((off + V + VN - 1) / VN), iV = (int)V;
  if (row == N - 1 && nvec * VN > off + stride) iV = --nvec * VN - off;
  const int last = nvec - 1;
  const int steps = (nvec + U * BLOCK - 1) / (U * BLOCK);

  // (the empty asm statements keep the compiler from widening a vector before it is used and from carrying
  // every vector's column from chunk to chunk: both spill)
  auto load = [&](W (&c)[U], int q) {
    int t = tid;
    asm volatile("" : "+v"(t));
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int idx = t + BLOCK * (q * U + u);
      const uint32_t bytes = (uint32_t)(idx < last ? idx : last) * 16u;
      c[u] = __builtin_nontemporal_load(reinterpret_cast<const W *>(reinterpret_cast<const char *>(x) + bytes));
    }
  };
  // Maximum times log2 e, the sum relative to it, the sum of the two chunks at hand, and what rounding took from
  // the sum: once a dominant term sits in it, every further add rounds at its size
  float m2 = -INFINITY, s = 0.f, pair = 0.f, lost = 0.f;
  auto step = [&](W (&c)[U], int q) {
    int t = tid * VN - off;
    asm volatile("" : "+v"(t));
    // where a chunk may reach past the row's class columns (block-uniform)
    const bool edge = q == 0 || (q + 1) * (U * BLOCK * VN) - off > iV;
#pragma unroll
    for (int h = 0; h < U; h += CH) {
      float cm = -INFINITY;
      float xs[CH][VN];
#pragma unroll
      for (int u = 0; u < CH; ++u) {
        asm volatile("" : "+v"(c[h + u]));
        const int c0 = t + VN * BLOCK * (q * U + h + u);
#pragma unroll
        for (int k = 0; k < VN; ++k) xs[u][k] = word_elem<T, VN>(c[h + u], k);
        if (edge) {
#pragma unroll
          for (int k = 0; k < VN; ++k) xs[u][k] = (uint32_t)(c0 + k) < (uint32_t)iV ? xs[u][k] : -INFINITY;
        }
#pragma unroll
        for (int k = 0; k < VN; ++k) cm = fmaxf(cm, xs[u][k]);
      }
      const float cm2 = cm * kLog2e;
      if (cm2 > m2) {
        const float f = __builtin_amdgcn_exp2f(m2 - cm2);  // 0 the first time (m2 = -inf, s = 0)
        s *= f;
        pair *= f;
        lost *= f;
        m2 = cm2;
      }
      // nothing finite so far: every term is 2^-inf (or NaN) against any finite stand-in
      const float ref = m2 == -INFINITY ? 0.f : m2;
      float part[CH];
#pragma unroll
      for (int u = 0; u < CH; ++u) {
        float e[VN];
#pragma unroll
        for (int k = 0; k < VN; ++k)
          e[k] = __builtin_amdgcn_exp2f(__builtin_fmaf(xs[u][k], kLog2e, -ref));
#pragma unroll
        for (int w = VN / 2; w > 0; w /= 2)
#pragma unroll
          for (int k = 0; k < w; ++k) e[k] += e[k + w];
        part[u] = e[0];
      }
#pragma unroll
      for (int w = CH / 2; w > 0; w /= 2)
#pragma unroll
        for (int u = 0; u < w; ++u) part[u] += part[u + w];
      pair += part[0];
      __builtin_amdgcn_sched_barrier(0);  // 8 elements widened at a time
    }
  };

  const T x_t = x[off + tgt];
  W even[U], odd[U];
  load(even, 0);
  if (steps > 1) load(odd, 1);
  for (int q = 0; q < steps; q += 2) {
    step(even, q);
    if (q + 2 < steps) load(even, q + 2);
    if (q + 1 < steps) {
      step(odd, q + 1);
      if (q + 3 < steps) load(odd, q + 3);
    }
    const float sum = s + pair, added = sum - s;
    lost += (s - (sum - added)) + (pair - added);
    s = sum;
    pair = 0.f;
  }
  s += lost;
  if (tid < (int)V - iV) {
    const float v = to_acc(x[off + iV + tid]), v2 = v * kLog2e;
    if (v2 > m2) {
      s *= __builtin_amdgcn_exp2f(m2 - v2);
      m2 = v2;
    }
    s += __builtin_amdgcn_exp2f(__builtin_fmaf(v, kLog2e, m2 == -INFINITY ? 0.f : -m2));
  }
  // (max, sum) across the wave, then across the waves.  A lane without a finite value brings its
  // sum as it is: 0, or the NaN it met.
  const float mw2 = wave_reduce(m2, MaxOp{});
  const float sw = wave_reduce(m2 == -INFINITY ? s : s * __builtin_amdgcn_exp2f(m2 - mw2), SumOp{});
  if (lane == 0) {
    red_m[tid >> 6] = mw2;
    red_s[tid >> 6] = sw;
  }
  lds_barrier();
  if (tid < kWave) {
    const float pm = lane < kWaves ? red_m[lane] : -INFINITY;
    const float ps = lane < kWaves ? red_s[lane] : 0.f;
    const float M2 = wave_reduce(pm, MaxOp{});
    const float S = wave_reduce(pm == -INFINITY ? ps : ps * __builtin_amdgcn_exp2f(pm - M2), SumOp{});
    if (tid == 0) {
      const float l = (__builtin_amdgcn_logf(S) - __builtin_fmaf(to_acc(x_t), kLog2e, -M2)) * kLn2;
      row_loss[row] = class_weight ? l * class_weight[tgt] : l;
    }
  }
}

// Rows too wide for registers, rows too wide for the streaming kernel where only the loss is wanted or the
// row-holding kernel would run a second round of few rows, and few unpadded rows with fp32 gradients that would leave
// the streaming kernel's lanes half empty.  Persistent workgroups walk rows.  A row is split into a head of
// single elements up to the first 16-byte boundary, a body of whole vectors and a tail; the
// base pointers are 16-byte aligned, so gradient rows split at the same columns.  The body is
// read twice in chunks of kWideU vectors per lane: the first sweep keeps a running (max, sum)
// per lane (rescaling the sum when the maximum moves: one exp2 per element plus one per
// chunk), the second sweep re-reads the row, which the first one left in the L2 / last-level
// cache, and writes the gradient.  Only a handful of scalars is carried between the sweeps,
// so two workgroups share a CU and cover each other's waits.
constexpr int kWideU = 2;  // 16-byte vectors per lane and chunk
static_assert(kWideU == 2, "the chunk sum below adds two vector sums");

template <typename T, typename TD>
__global__ __launch_bounds__(1024, 8) void ce_rows_wide_kernel(
    const T *logits, TD *dlogits, const int64_t *__restrict__ targets, float *__restrict__ row_loss,
    const int *__restrict__ ws_count, int64_t N, int64_t V, int64_t row_stride,
    int64_t ignore_index, int reduction, float dloss, const float *__restrict__ class_weight) {
  constexpr int VN = Vec16<T>::n;
  constexpr int BLOCK = 1024;
  constexpr int kWaves = BLOCK / kWave;
  constexpr int kTailLane = 32;  // lanes [0, VN) own head elements, [32, 32 + VN) tail elements
  static_assert(VN <= kTailLane, "head and tail lanes overlap");
  __shared__ float red_m[kWaves], red_s[kWaves];
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid >> 6;
  const int stride = (int)row_stride;  // the host checks that it fits
  const int vcols = (int)V;
  // per-class weights (at::nll_loss's `weight`): a row's loss and gradient are scaled by the
  // weight of its target, and the mean is over the sum of those weights
  float scale0 = dloss;
  if (reduction == CS_REDUCTION_MEAN)
    scale0 = dloss / (class_weight ? reinterpret_cast<const float *>(ws_count)[1]
                                   : (float)rows_that_count(ws_count, targets, N, V, ignore_index));

  for (int64_t row = blockIdx.x; row < N; row += gridDim.x) {
    const int64_t tgt = targets[row];
    const T *x = logits + row * row_stride;
    TD *d = dlogits ? dlogits + row * row_stride : nullptr;
    // columns [0, head) before the first aligned vector, nvec vectors, then the rest
    int head = (int)((VN - (row * row_stride) % VN) % VN);
    head = head < stride ? head : stride;
    const int nvec = (stride - head) / VN;
    const int tail0 = head + nvec * VN;
    int ecol = -1;  // the single element this lane owns, if any
    if (tid < head) ecol = tid;
    if (tid >= kTailLane && tail0 + (tid - kTailLane) < stride) ecol = tail0 + (tid - kTailLane);
    const T *xb = x + head;
    TD *db = d ? d + head : nullptr;

    if (!target_counts(tgt, V, ignore_index)) {  // block-uniform
      if (tid == 0 && row_loss) row_loss[row] = 0.f;
      if (d) {
        float z[VN];
#pragma unroll
        for (int k = 0; k < VN; ++k) z[k] = 0.f;
        for (int idx = tid; idx < nvec; idx += BLOCK) store_out<T, TD, VN>(db + (int64_t)idx * VN, z);
        if (ecol >= 0) d[ecol] = from_acc<TD>(0.f);
      }
      continue;
    }
    // ---- sweep 1: running maximum (times log2 e) and the sum relative to it
    float xe = -INFINITY;
    if (ecol >= 0 && ecol < vcols) xe = to_acc(x[ecol]);
    float m2 = xe * kLog2e;
    // the same expression as in the second sweep (the fma sees the product unrounded, so this is not exactly 1)
    float s = xe == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(__builtin_fmaf(xe, kLog2e, -m2));
    for (int base = tid; base < nvec + tid; base += BLOCK * kWideU) {
      Vec16<T> v[kWideU];
#pragma unroll
      for (int u = 0; u < kWideU; ++u) {
        const int idx = base + BLOCK * u;
        // cached: read again below.  Every lane loads, see ce_rows_kernel.
        v[u] = load16(xb + (int64_t)(idx < nvec ? idx : nvec - 1) * VN);
      }
      float xs[kWideU][VN];
      float cm = -INFINITY;
#pragma unroll
      for (int u = 0; u < kWideU; ++u) {
        const int idx = base + BLOCK * u;
        const int c0 = head + idx * VN;
#pragma unroll
        for (int k = 0; k < VN; ++k) {
          xs[u][k] = (idx < nvec && c0 + k < vcols) ? vec_get(v[u], k) : -INFINITY;  // padding, lanes past the row
          cm = fmaxf(cm, xs[u][k]);
        }
      }
      const float cm2 = cm * kLog2e;
      if (cm2 > m2) {
        s *= __builtin_amdgcn_exp2f(m2 - cm2);  // 0 the first time (m2 = -inf, s = 0)
        m2 = cm2;
      }
      if (m2 != -INFINITY) {
        // pairwise within the chunk, one add onto the running sum: once a dominant term sits
        // in s, every further add rounds at its size, so there should be few of them
        float part[kWideU];
#pragma unroll
        for (int u = 0; u < kWideU; ++u) {
          float e[VN];
#pragma unroll
          for (int k = 0; k < VN; ++k) e[k] = __builtin_amdgcn_exp2f(__builtin_fmaf(xs[u][k], kLog2e, -m2));
#pragma unroll
          for (int w = VN / 2; w > 0; w /= 2)
#pragma unroll
            for (int k = 0; k < w; ++k) e[k] += e[k + w];
          part[u] = e[0];
        }
        s += part[0] + part[1];
      }
    }
    // ---- (max, sum) across the wave, then across the waves
    const float mw2 = wave_reduce(m2, MaxOp{});
    const float sw = wave_reduce(m2 == -INFINITY ? 0.f : s * __builtin_amdgcn_exp2f(m2 - mw2), SumOp{});
    __syncthreads();  // the previous row's readers are done with red_m / red_s
    if (lane == 0) {
      red_m[wave] = mw2;
      red_s[wave] = sw;
    }
    __syncthreads();
    const float pm = lane < kWaves ? red_m[lane] : -INFINITY;
    const float ps = lane < kWaves ? red_s[lane] : 0.f;
    const float M2 = wave_reduce(pm, MaxOp{});
    const float S = wave_reduce(pm == -INFINITY ? 0.f : ps * __builtin_amdgcn_exp2f(pm - M2), SumOp{});
    const float wt = class_weight ? class_weight[tgt] : 1.0f;
    const float scale = class_weight ? scale0 * wt : scale0;
    if (tid == 0 && row_loss) {
      const float x_t = to_acc(x[tgt]);
      const float l = (__builtin_amdgcn_logf(S) - __builtin_fmaf(x_t, kLog2e, -M2)) * kLn2;
      row_loss[row] = class_weight ? l * wt : l;
    }
    if (!d) continue;
    // ---- sweep 2: p = 2^(x log2e - M2) / S, gradient (p - onehot) * scale
    const float factor = scale / S;
    const int t_vec = tgt >= head ? (int)((tgt - head) / VN) : -1;  // past the body if in the tail
    const int t_sub = (int)((tgt - head) % VN);
    if (ecol >= 0) {
      float o = 0.f;
      if (ecol < vcols) {
        o = __builtin_amdgcn_exp2f(__builtin_fmaf(xe, kLog2e, -M2)) * factor;
        if (ecol == tgt) o -= scale;
      }
      d[ecol] = from_acc<TD>(o);
    }
    for (int base = tid; base < nvec + tid; base += BLOCK * kWideU) {
      Vec16<T> v[kWideU];
#pragma unroll
      for (int u = 0; u < kWideU; ++u) {
        const int idx = base + BLOCK * u;
        v[u] = load16_stream(xb + (int64_t)(idx < nvec ? idx : nvec - 1) * VN);
      }
#pragma unroll
      for (int u = 0; u < kWideU; ++u) {
        const int idx = base + BLOCK * u;
        if (idx < nvec) {
          const int c0 = head + idx * VN;
          float o[VN];
#pragma unroll
          for (int k = 0; k < VN; ++k)
            o[k] = c0 + k < vcols ? __builtin_amdgcn_exp2f(__builtin_fmaf(vec_get(v[u], k), kLog2e, -M2)) * factor : 0.f;
          if (idx == t_vec) {
#pragma unroll
            for (int k = 0; k < VN; ++k)
              if (k == t_sub) o[k] -= scale;
          }
          store_out<T, TD, VN>(db + (int64_t)idx * VN, o);
        }
      }
    }
  }
}

// Any V, stride and alignment; fp64 too.  Three sweeps over the row, the
// later ones served by the cache.
template <typename T, typename TD>
__global__ __launch_bounds__(256) void ce_rows_general_kernel(
    const T *__restrict__ logits, TD *__restrict__ dlogits, const int64_t *__restrict__ targets,
    float *__restrict__ row_loss, const int *__restrict__ ws_count, int64_t N, int64_t V, int64_t row_stride,
    int64_t ignore_index, int reduction, float dloss, const float *__restrict__ class_weight) {
  using U = typename Acc<T>::type;
  __shared__ U scratch[4];
  const int64_t row = row_of_grid();
  if (row >= N) return;
  const T *x = logits + row * row_stride;
  const int64_t target = targets[row];
  const bool counts = target_counts(target, V, ignore_index);
  if (!counts) {
    if (threadIdx.x == 0 && row_loss) row_loss[row] = 0.f;
    if (dlogits)
      for (int64_t c = threadIdx.x; c < row_stride; c += 256)
        dlogits[row * row_stride + c] = from_acc<TD>((typename Acc<TD>::type)0);
    return;
  }
  U m = -INFINITY;
  for (int64_t c = threadIdx.x; c < V; c += 256) {
    const U v = to_acc(x[c]);
    m = v > m ? v : m;
  }
  m = block_reduce(m, MaxOp{}, (U)-INFINITY, scratch);
  U s = 0;
  for (int64_t c = threadIdx.x; c < V; c += 256) s += exp((U)to_acc(x[c]) - m);
  s = block_reduce(s, SumOp{}, (U)0, scratch);
  const U lse = m + log(s);
  const U wt = class_weight ? (U)class_weight[target] : (U)1;
  if (threadIdx.x == 0 && row_loss) row_loss[row] = (float)((lse - (U)to_acc(x[target])) * wt);
  if (!dlogits) return;
  U scale = (U)dloss;
  if (reduction == CS_REDUCTION_MEAN)
    scale = (U)dloss / (class_weight ? (U) reinterpret_cast<const float *>(ws_count)[1]
                                     : (U)rows_that_count(ws_count, targets, N, V, ignore_index));
  scale *= wt;
  for (int64_t c = threadIdx.x; c < row_stride; c += 256) {
    U o = 0;
    if (c < V) {
      o = exp((U)to_acc(x[c]) - lse);
      if (c == target) o -= (U)1;
      o *= scale;
    }
    dlogits[row * row_stride + c] = from_acc<TD>((typename Acc<TD>::type)o);
  }
}

// The loss alone of few long rows: whole rows leave CUs idle (fewer rows than there are) or half of them to a second
// round, so a row is split over several workgroups of 256 lanes, which leave a maximum and a sum each for the last
// launch.  A workgroup's columns are in registers before the first is used, and its sum is a tree.  Rows may start
// anywhere: vectors count from the 128-byte line a row starts in (counted from the row itself, at element alignment,
// [1024,50257] bf16 took 30.0 us, [509,50257] 15.7).  Bound by HBM reads where the rows are many, by the two launches
// otherwise.
//
// Per call, us, whole rows / split, bf16: [300,50257] 15.5 / 11.8, [509,50257] 17.3 / 14.6, [1024,50257] 28.1 / 23.0,
// [600,16399] 15.3 / 11.8, [8,128256] 14.4 / 9.6, [128,128256] 18.1 / 12.3, [1024,128256] 52.5 / 46.4; fp32
// [300,50257] 20.6 / 15.2, [1024,50257] 42.2 / 36.3.
constexpr int kSplitThreads = 256;
constexpr int kMostSplits = 32;
constexpr int64_t kSplitRows = 1024;  // one row per lane of the last launch at most

template <typename T, int VPT>
__global__ __launch_bounds__(kSplitThreads) void ce_loss_split_kernel(
    const T *__restrict__ logits, const int64_t *__restrict__ targets, float2 *__restrict__ parts,
    float *__restrict__ target_logits, int64_t N, int64_t V, int64_t row_stride, int64_t ignore_index, int span,
    unsigned splits) {
  constexpr int VN = Vec16<T>::n;
  constexpr int kWaves = kSplitThreads / kWave;
  __shared__ float2 red[kWaves];
  const int tid = threadIdx.x;
  const int64_t row = blockIdx.x / splits;
  const int sp = (int)(blockIdx.x % splits);
  const int64_t tgt = targets[row];
  if (!target_counts(tgt, V, ignore_index)) return;  // the last launch reads nothing of this row
  const T *x = logits + row * row_stride;
  // Columns [lo, hi), in vectors that count from the line the row starts in.  A lane's vectors past them are the last one
  // again; the array's last one, which may not lie whole inside it, is moved back to end with the array.
  const int iV = (int)V, off = (int)((row * row_stride) & (kLineElems<T> - 1));
  const int lo = sp * span - off, hi = lo + span < iV ? lo + span : iV;
  int last = hi > lo ? lo + (hi - lo - 1) / VN * VN : 0;
  if (row == N - 1 && last > (int)row_stride - VN) last = (int)row_stride - VN;
  Vec16<T> v[VPT];
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    const int c = lo + (tid + kSplitThreads * j) * VN;
    v[j] = load16_unaligned_stream(x + (c < last ? c : last));
  }
  if (sp == 0 && tid == 0) target_logits[row] = to_acc(x[tgt]);
  float m = -INFINITY;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    const int c = lo + (tid + kSplitThreads * j) * VN;
    if (c < 0 || c + VN > hi) {
      const int at = c < last ? c : last, from = c > 0 ? c : 0;
#pragma unroll
      for (int k = 0; k < VN; ++k)
        if (at + k < from || at + k >= hi) v[j].e[k] = from_acc<T>(-INFINITY);
    }
#pragma unroll
    for (int k = 0; k < VN; ++k) m = fmaxf(m, to_acc(v[j].e[k]));
  }
  const float m2 = wave_reduce(m, MaxOp{}) * kLog2e;
  const float ref = m2 == -INFINITY ? 0.f : m2;  // nothing finite: every term is 0, or the NaN that was met
  float part[VPT];
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    float e[VN];
#pragma unroll
    for (int k = 0; k < VN; ++k) e[k] = __builtin_amdgcn_exp2f(__builtin_fmaf(to_acc(v[j].e[k]), kLog2e, -ref));
#pragma unroll
    for (int w = VN / 2; w > 0; w /= 2)
#pragma unroll
      for (int k = 0; k < w; ++k) e[k] += e[k + w];
    part[j] = e[0];
  }
#pragma unroll
  for (int w = 1; w < VPT; w *= 2)
#pragma unroll
    for (int j = 0; j + w < VPT; j += 2 * w) part[j] += part[j + w];
  const float sum = wave_reduce(part[0], SumOp{});
  if ((tid & (kWave - 1)) == 0) red[tid >> 6] = float2{m2, sum};
  lds_barrier();
  if (tid == 0) {
    float bm = red[0].x, bs = 0.f;
#pragma unroll
    for (int w = 1; w < kWaves; ++w) bm = fmaxf(bm, red[w].x);
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
      bs += red[w].x == -INFINITY ? red[w].y : red[w].y * __builtin_amdgcn_exp2f(red[w].x - bm);
    parts[(int64_t)row * splits + sp] = float2{bm, bs};
  }
}

// Row losses from the splits, their sum in a fixed order and the count: a row per lane.
__global__ __launch_bounds__(1024) void ce_loss_combine_kernel(
    const float2 *__restrict__ parts, const float *__restrict__ target_logits, int splits,
    float *__restrict__ row_loss, int64_t N, int *__restrict__ ws_count, int reduction, float *__restrict__ loss,
    float *__restrict__ total_weight, const int64_t *__restrict__ targets, int64_t V, int64_t ignore_index,
    const float *__restrict__ class_weight) {
  const int tid = threadIdx.x;
  const int row = tid < (int)N ? tid : (int)N - 1;
  const int64_t tgt = targets[row];
  const float x_t = target_logits[row];
  const bool counts = tid < (int)N && target_counts(tgt, V, ignore_index);
  float m2 = -INFINITY, s = 0.f;
  for (int q0 = 0; q0 < splits; q0 += 8) {
    float2 p[8];  // in flight together
#pragma unroll
    for (int u = 0; u < 8; ++u) p[u] = parts[(int64_t)row * splits + (q0 + u < splits ? q0 + u : splits - 1)];
    float pm = m2;
#pragma unroll
    for (int u = 0; u < 8; ++u) pm = fmaxf(pm, p[u].x);
    if (m2 != -INFINITY) s *= __builtin_amdgcn_exp2f(m2 - pm);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (q0 + u < splits) s += p[u].x == -INFINITY ? p[u].y : p[u].y * __builtin_amdgcn_exp2f(p[u].x - pm);
    m2 = pm;
  }
  const float wt = counts && class_weight != nullptr ? class_weight[tgt] : 1.f;
  const float l = counts ? (__builtin_amdgcn_logf(s) - __builtin_fmaf(x_t, kLog2e, -m2)) * kLn2 * wt : 0.f;
  if (tid < (int)N) row_loss[row] = l;
  const RowSums sums = block_sums<true>(RowSums{l, counts, counts ? wt : 0.f}, class_weight != nullptr);
  if (tid == 0) {
    const float total = class_weight != nullptr ? sums.weight : (float)sums.count;
    *ws_count = sums.count;
    reinterpret_cast<float *>(ws_count)[1] = total;
    if (loss) *loss = reduction == CS_REDUCTION_MEAN ? sums.loss / total : sums.loss;
    if (total_weight) *total_weight = total;
  }
}

// CUs of the current device, asked once per device (threads may race to fill a slot: they
// store the same value).
int64_t compute_units() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Two-sweep kernel: two workgroups of 1024 lanes per CU.
template <typename T, typename TD>
void launch_wide(const void *logits, void *dlogits, const int64_t *targets, float *row_loss,
                 const int *ws_count, int64_t N, int64_t V, int64_t row_stride, int64_t ignore_index,
                 int reduction, float dloss, const float *class_weight, hipStream_t s) {
  const int64_t cus = compute_units();
  const dim3 grid((unsigned)(N < 2 * cus ? N : 2 * cus));
  ce_rows_wide_kernel<T, TD><<<grid, dim3(1024), 0, s>>>(
      (const T *)logits, (TD *)dlogits, targets, row_loss, ws_count, N, V, row_stride, ignore_index,
      reduction, dloss, class_weight);
}

// Accesses (of 16 bytes; 8 where 16-bit logits give fp32 gradients) a row may take for the streaming
// kernel: 7 or 8 fp32, 7 16-bit or 13 half-width ones per lane.
template <typename T, typename TD>
struct StreamPlan {
  static constexpr int kEpv = sizeof(T) == 2 && sizeof(TD) == 4 ? 4 : Vec16<T>::n;
  static constexpr int kMostVecs = 1024 * (kEpv * sizeof(T) == 8 ? 13 : sizeof(T) == 4 ? 8 : 7);
};

// One persistent workgroup per CU, the row in registers.  The widest plans (8 vectors per lane at 16
// bit, 16 half vectors with fp32 gradients) measured slower than the two-sweep kernel and are not
// built.
template <typename T, typename TD, bool RAGGED>
void launch_stream(const void *logits, void *dlogits, const int64_t *targets, float *row_loss,
                   const int *ws_count, int64_t N, int64_t V, int64_t row_stride, int64_t ignore_index,
                   int reduction, float dloss, const float *class_weight, hipStream_t s) {
  constexpr int EPV = StreamPlan<T, TD>::kEpv;
  const int64_t cus = compute_units();
  const dim3 grid((unsigned)(N < cus ? N : cus)), block(1024);
  // a ragged row is counted from the line it starts in
  const int64_t nvec = (row_stride + (RAGGED ? kLineElems<T> - 1 : 0) + EPV - 1) / EPV;
#define CS_CE_STREAM(VPT)                                                                                \
  if (class_weight != nullptr) {                                                                         \
    ce_rows_stream_kernel<T, TD, VPT, EPV, true, RAGGED><<<grid, block, 0, s>>>(                          \
        (const T *)logits, (TD *)dlogits, targets, row_loss, ws_count, N, V, row_stride, ignore_index,   \
        reduction, dloss, class_weight);                                                                 \
  } else {                                                                                               \
    ce_rows_stream_kernel<T, TD, VPT, EPV, false, RAGGED><<<grid, block, 0, s>>>(                         \
        (const T *)logits, (TD *)dlogits, targets, row_loss, ws_count, N, V, row_stride, ignore_index,   \
        reduction, dloss, nullptr);                                                                      \
  }
  if constexpr (EPV * sizeof(T) == 8) {
    CS_CE_STREAM(13);
  } else if (nvec <= 1024 * 4) {
    CS_CE_STREAM(4);
  } else if (nvec <= 1024 * 7) {
    CS_CE_STREAM(7);
  } else {
    if constexpr (sizeof(T) == 4) {
      CS_CE_STREAM(8);
    }
  }
#undef CS_CE_STREAM
}

// Rows of up to 2048 vectors of 16 bytes, four accesses a lane (eight of 8 bytes for fp32 gradients of 16-bit logits; half
// or a quarter of that where one wave then has the row, three quarters where those take no more waves) and as many waves as
// that takes: false where the row is too wide.
// Twice as wide where there are more than two rows per CU; of unpadded rows, whose edges take more instructions, one and a
// half times.  (Before, one wave of eight accesses up to 512
// vectors and four waves beyond; unpadded and weighted rows in two sweeps; wider ones by the streaming kernel.)
// us per call, before / now, bf16 unless said: padded [8192,4096] 29.8 / 28.6, [7501,7808] 46.1 / 42.7, [8192,16384]
// 94.7 / 92.6; unpadded [16384,1001] 48.1 / 24.9, [13786,3378] 55.0 / 39.6, [6000,10001] 82.7 / 46.9, [2099,15215] 36.3 /
// 29.4, fp32 [4096,7999] 62.1 / 49.6; fp32 gradients [15248,4553] fp16 109.4 / 77.5, [11936,9472] 156 / 119, [4096,16000]
// 110 / 73; weighted [2000,12000] 32.6 / 24.8; few rows [16,4160] 7.8 / 6.6, [277,3448] 8.8 / 7.9.  The wider ones:
// [2099,20215] 50.0 / 39.4, [1000,20215] 25.5 / 23.6, [6000,20215] fp16 weighted 119 / 88, [4096,32000] 97 / 89,
// [4096,20000] with fp32 gradients 114 / 92; but unpadded [4096,32001] 106 / 113, [300,30000] 14.1 / 15.4, fp32
// [338,15424] 13.6 / 14.6.
// Three quarters, four accesses a lane (or eight) / three: unpadded fp16 [3000,4097] 19.4 / 18.2, [3000,2001] with fp32 gradients
// 15.9 / 14.9, the loss alone of padded bf16 [30000,2624] 39 / 34.8, fp16 [9000,3008] 17.1 / 15.7.
template <typename T, typename TD, bool RAGGED>
bool launch_narrow(const void *logits, void *dlogits, const int64_t *targets, float *row_loss, const int *ws_count,
                   int64_t N, int64_t V, int64_t row_stride, int64_t ignore_index, int reduction, float dloss,
                   const float *class_weight, hipStream_t s) {
  constexpr int EPV = StreamPlan<T, TD>::kEpv, U = EPV * sizeof(T) == 8 ? 8 : 4;
  const int64_t nvec = (row_stride + (RAGGED ? kLineElems<T> - 1 : 0) + EPV - 1) / EPV;
  const int threads = N <= 2 * compute_units() ? 512 : RAGGED ? 768 : kNarrowMostThreads;
  if (nvec > threads * U) return false;
#define CS_CE_NARROW(VPT)                                                                                          \
  ce_rows_kernel<T, TD, VPT, EPV, RAGGED>                                                                          \
      <<<row_grid(N), dim3((unsigned)(ceil_div(nvec, (int64_t)(kWave * VPT)) * kWave)), 0, s>>>(                   \
          (const T *)logits, (TD *)dlogits, targets, row_loss, ws_count, N, V, row_stride, ignore_index, reduction, \
          dloss, class_weight)
  if (nvec <= kWave * U / 4) {
    CS_CE_NARROW(U / 4);
  } else if (nvec <= kWave * U / 2) {
    CS_CE_NARROW(U / 2);
  } else if (ceil_div(nvec, (int64_t)(kWave * U * 3 / 4)) == ceil_div(nvec, (int64_t)(kWave * U))) {
    CS_CE_NARROW(U * 3 / 4);
  } else {
    CS_CE_NARROW(U);
  }
#undef CS_CE_NARROW
  return true;
}

// Vectors per lane of the row-holding kernel: three, four or five units.
template <typename T, typename TD>
struct HoldPlan {
  static constexpr int kEpv = StreamPlan<T, TD>::kEpv;
  static constexpr int kUnit = kEpv * sizeof(T) == 8 ? 8 : 4;
  static constexpr int kMostVecs = 1024 * 5 * kUnit;
};

template <typename T, typename TD, bool RAGGED>
void launch_hold(const void *logits, void *dlogits, const int64_t *targets, float *row_loss,
                 const int *ws_count, int64_t N, int64_t V, int64_t row_stride, int64_t ignore_index,
                 int reduction, float dloss, const float *class_weight, hipStream_t s) {
  constexpr int EPV = HoldPlan<T, TD>::kEpv, U = HoldPlan<T, TD>::kUnit;
  const int64_t cus = compute_units();
  const dim3 grid((unsigned)(N < cus ? N : cus)), block(1024);
  const int64_t nvec = (row_stride + (RAGGED ? kLineElems<T> - 1 : 0) + EPV - 1) / EPV;
#define CS_CE_HOLD(VPT)                                                                                  \
  ce_rows_hold_kernel<T, TD, VPT, EPV, RAGGED><<<grid, block, 0, s>>>(                                    \
      (const T *)logits, (TD *)dlogits, targets, row_loss, ws_count, N, V, row_stride, ignore_index,     \
      reduction, dloss, class_weight)
  if (nvec <= 1024 * 3 * U) {
    CS_CE_HOLD(3 * U);
  } else if (nvec <= 1024 * 4 * U) {
    CS_CE_HOLD(4 * U);
  } else {
    CS_CE_HOLD(5 * U);
  }
#undef CS_CE_HOLD
}

template <typename T, typename TD>
int launch_rows(const void *logits, void *dlogits, const int64_t *targets, float *row_loss,
                const int *ws_count, int64_t N, int64_t V, int64_t row_stride,
                int64_t ignore_index, int reduction, float dloss, const float *class_weight, hipStream_t s) {
  constexpr int VN = Vec16<T>::n;
  const bool base_ok = !std::is_same_v<T, double> && is_aligned16(logits) &&
                       (!dlogits || is_aligned16(dlogits)) && row_stride <= (int64_t(1) << 30);
  const bool vec_ok = base_ok && row_stride % VN == 0;
  const dim3 grid((unsigned)N);
  if constexpr (!std::is_same_v<T, double>) {
    // per-class weights: every kernel but the fp32 one of 1024 lanes and 16 vectors takes them
    const int64_t nvec_all = row_stride / VN;
    const bool streams = nvec_all > 256 * 8 &&
                         row_stride <= (int64_t)StreamPlan<T, TD>::kEpv * StreamPlan<T, TD>::kMostVecs;
    const int64_t cus = compute_units();
    // The loss alone, of more than four rows per CU: a workgroup per row.  Of fewer rows each has too few loads
    // under way, and what it saves is within the launches' time: [1024,50257] bf16 25.5 us against 27.3, but
    // fp32 38.5 against 34.9 and [1024,128256] bf16 48.8 against 44.4; at 2048 rows 38.4 against 46.5 and 84.1
    // against 97.8.  Rows of more than 8192 vectors: 512 lanes ([8192,128256] bf16 315 us; 318 with 256).
    if (dlogits == nullptr && base_ok && nvec_all > 256 * 8 && N > 4 * cus && row_stride < (int64_t(1) << 29)) {
      if (nvec_all <= 1024 * 8) {
        ce_loss_rows_kernel<T, 256><<<grid, dim3(256), 0, s>>>((const T *)logits, targets, row_loss, N, V, row_stride,
                                                               ignore_index, class_weight);
      } else {
        ce_loss_rows_kernel<T, 512><<<grid, dim3(512), 0, s>>>((const T *)logits, targets, row_loss, N, V,
                                                                 row_stride, ignore_index, class_weight);
      }
      return launch_status();
    }
    // The loss alone needs no second pass: nothing to hold a row for.  A few rows more than there are
    // CUs are a second round of whole rows for the row-holding kernel, while the others run two rows per CU or
    // (fp32 rows of whole vectors) start the next row as soon as one ends.  Where the line lies, held row / the
    // alternative in us: [340,57600] bf16 28.1 / 25.7, [384,57600] 28.3 / 26.4, [450,57600] 28.4 / 28.6; [340,100003]
    // 42.3 / 43.3, [300,128256] 49.1 / 48.1, [384,128256] 48.0 / 53.5; with fp32 gradients [300,57601] 40.8 / 41.1,
    // [384,57601] 39.7 / 42.8; fp32 [300,40000] 30.8 / 29.3, [340,40001] 32.4 / 30.8, [384,40001] 31.9 / 33.1.
    const bool past_one_round = sizeof(T) == 4                                    ? 5 * N > 7 * cus
                                : sizeof(TD) == sizeof(T) && row_stride < 80000 ? 2 * N > 3 * cus
                                                                                : 4 * N > 5 * cus;
    const bool holds = dlogits != nullptr && nvec_all > 256 * 8 && (N <= cus || past_one_round);
    if (base_ok && nvec_all <= kNarrowMostThreads * 4 &&
        (vec_ok ? launch_narrow<T, TD, false>(logits, dlogits, targets, row_loss, ws_count, N, V, row_stride, ignore_index,
                                              reduction, dloss, class_weight, s)
                : launch_narrow<T, TD, true>(logits, dlogits, targets, row_loss, ws_count, N, V, row_stride, ignore_index,
                                             reduction, dloss, class_weight, s)))
      return launch_status();
    if (vec_ok && (class_weight == nullptr || streams)) {
      if (row_stride <= (int64_t)StreamPlan<T, TD>::kEpv * StreamPlan<T, TD>::kMostVecs) {
        launch_stream<T, TD, false>(logits, dlogits, targets, row_loss, ws_count, N, V, row_stride, ignore_index,
                                    reduction, dloss, class_weight, s);
      } else if (holds && row_stride <= (int64_t)HoldPlan<T, TD>::kEpv * HoldPlan<T, TD>::kMostVecs) {
        launch_hold<T, TD, false>(logits, dlogits, targets, row_loss, ws_count, N, V, row_stride, ignore_index,
                                  reduction, dloss, class_weight, s);
      } else if (sizeof(T) == 4 && nvec_all <= 1024 * 16) {
        // fp32 rows up to 65536 columns still fit in registers (at 16 bit this plan spills)
        if constexpr (sizeof(T) == 4)
          ce_rows_kernel<T, TD, 16, VN, false, 1024><<<row_grid(N), dim3(1024), 0, s>>>(
              (const T *)logits, (TD *)dlogits, targets, row_loss, ws_count, N, V, row_stride, ignore_index, reduction,
              dloss, nullptr);
      } else {
        launch_wide<T, TD>(logits, dlogits, targets, row_loss, ws_count, N, V, row_stride, ignore_index,
                           reduction, dloss, class_weight, s);
      }
      return launch_status();
    }
    // Unpadded rows that fill little of the streaming plan take two sweeps: with fp32 gradients of 16-bit logits the few rows
    // of up to 24576 columns that launch_narrow leaves (two per CU; us streamed / in two sweeps, bf16 [64,18001] 10.7 / 10.5,
    // [257,18001] 16.8 / 15.6, [257,22001] 17.7 / 17.5, weighted rows and fp16 10-20% in favour of the two sweeps from 257 to 400
    // rows; but [512,22001] 19.8 / 21.3, [512,24001] 20.3 / 22.7; wider ones, [3100,26001] 108 / 116), and the loss alone of more than
    // two rows per CU of four to six of its seven accesses ([600,38001] 21.4 / 19.5, [860,46001] 27.8 / 27.0; but [600,50257]
    // 22.3 / 23.5).  So few rows come here for the loss alone only in separate phases, or with a workspace that has no room
    // for their splits (loss_splits).
    const bool sparse = sizeof(TD) > sizeof(T) ? row_stride <= 24 * 1024
                                               : sizeof(T) == 2 && dlogits == nullptr && N > 2 * cus &&
                                                     row_stride > 32 * 1024 && row_stride <= 48 * 1024;
    if (base_ok && nvec_all > 256 * 8 && !sparse &&
        row_stride + kLineElems<T> <= (int64_t)StreamPlan<T, TD>::kEpv * StreamPlan<T, TD>::kMostVecs) {
      launch_stream<T, TD, true>(logits, dlogits, targets, row_loss, ws_count, N, V, row_stride, ignore_index,
                                 reduction, dloss, class_weight, s);
      return launch_status();
    }
    if (base_ok && holds && !sparse &&
        row_stride + kLineElems<T> <= (int64_t)HoldPlan<T, TD>::kEpv * HoldPlan<T, TD>::kMostVecs) {
      launch_hold<T, TD, true>(logits, dlogits, targets, row_loss, ws_count, N, V, row_stride, ignore_index,
                               reduction, dloss, class_weight, s);
      return launch_status();
    }
    if (base_ok && sizeof(TD) >= sizeof(T)) {
      // rows that start off a 16-byte boundary: split per row into head, vectors and tail
      launch_wide<T, TD>(logits, dlogits, targets, row_loss, ws_count, N, V, row_stride, ignore_index,
                         reduction, dloss, class_weight, s);
      return launch_status();
    }
  }
  ce_rows_general_kernel<T, TD><<<row_grid(N), dim3(256), 0, s>>>((const T *)logits, (TD *)dlogits, targets, row_loss,
                                                                  ws_count, N, V, row_stride, ignore_index,
                                                                  reduction, dloss, class_weight);
  return launch_status();
}

}  // namespace
}  // namespace cs_hip

using namespace cs_hip;

namespace {
// what every call takes: the header and a row loss each
size_t ce_least_workspace(int64_t N) { return kWsHeader + ((size_t)N * sizeof(float) + 255) / 256 * 256; }
// and behind it the splits of few rows: a target logit and kMostSplits pairs each
size_t ce_split_workspace(int64_t N) { return (size_t)N * (sizeof(float) + kMostSplits * sizeof(float2)) + 256; }
}  // namespace

extern "C" size_t cs_fused_classifier_workspace_bytes(int64_t N) {
  if (N < 0) return 0;
  if (N <= kSplitRows) return ce_least_workspace(N) + ce_split_workspace(N);
  // what the most rows that are split take, at least: the size never falls as the rows grow
  const size_t most = ce_least_workspace(kSplitRows) + ce_split_workspace(kSplitRows), least = ce_least_workspace(N);
  return least > most ? least : most;
}

namespace {

struct CeArgs {
  const void *logits;
  void *dlogits;
  const int64_t *targets;
  float *row_loss;
  float *loss;
  float *total_weight;
  void *workspace;
  size_t workspace_bytes;
  int64_t N, V, row_stride, ignore_index;
  int reduction;
  float dloss;
  int dtype, dlogits_dtype;
  const float *class_weight = nullptr;  // [V] fp32, or NULL: every class weighs 1
};

int ce_validate(const CeArgs &a) {
  if (a.N < 0 || a.V <= 0 || a.row_stride < a.V) return CS_ERR_INVALID_ARGUMENT;
  if (a.reduction != CS_REDUCTION_NONE && a.reduction != CS_REDUCTION_MEAN &&
      a.reduction != CS_REDUCTION_SUM)
    return CS_ERR_INVALID_ARGUMENT;
  const size_t es = dtype_size(a.dtype), ds = dtype_size(a.dlogits_dtype);
  if (es == 0 || ds == 0) return CS_ERR_UNSUPPORTED;
  if (a.dlogits_dtype != a.dtype && !(a.dlogits_dtype == CS_F32 && es == 2))
    return CS_ERR_UNSUPPORTED;
  if (a.N > 0x7fffffffLL || a.V > 0x7fffffffLL || a.row_stride > 0x7fffffffLL)
    return CS_ERR_TOO_LARGE;
  if (!a.workspace || a.workspace_bytes < ce_least_workspace(a.N) ||
      !aligned_to(a.workspace, 256))
    return CS_ERR_WORKSPACE;
  if (a.reduction == CS_REDUCTION_NONE && !a.row_loss) return CS_ERR_INVALID_ARGUMENT;
  if (a.reduction != CS_REDUCTION_NONE && !a.loss) return CS_ERR_INVALID_ARGUMENT;
  if (a.N > 0 && (!a.logits || !a.targets)) return CS_ERR_INVALID_ARGUMENT;
  if ((a.logits && !aligned_to(a.logits, es)) || (a.dlogits && !aligned_to(a.dlogits, ds)) ||
      (a.targets && !aligned_to(a.targets, 8)) || (a.row_loss && !aligned_to(a.row_loss, 4)) ||
      (a.loss && !aligned_to(a.loss, 4)) || (a.total_weight && !aligned_to(a.total_weight, 4)) ||
      (a.class_weight && !aligned_to(a.class_weight, 4)))
    return CS_ERR_MISALIGNED;
  if (a.dlogits == a.logits && a.dlogits_dtype != a.dtype) return CS_ERR_INVALID_ARGUMENT;
  return CS_OK;
}

// vectors of a row, the longest way it may lie to its first line
int64_t split_vecs(const CeArgs &a) {
  const int64_t es = (int64_t)dtype_size(a.dtype), line = a.row_stride % (128 / es) != 0 ? 128 / es - 1 : 0;
  return ceil_div(a.V + line, 16 / es);
}

// Workgroups per row for the loss alone of few rows, each with at most eight vectors a lane: eight to a CU, four where
// there are fewer rows than CUs.  0 where whole rows are taken: rows of up to 8192 vectors of which every CU has one
// ([200,50257] bf16 10.6 us whole, 11.0 split) or more than four (ce_loss_rows_kernel).
int loss_splits(const CeArgs &a) {
  if (a.dlogits != nullptr || a.N <= 0 || a.N > kSplitRows || a.dtype == CS_F64) return 0;
  if (a.workspace_bytes < cs_fused_classifier_workspace_bytes(a.N)) return 0;  // a caller who reckons it without this
  const int64_t vn = 16 / (int64_t)dtype_size(a.dtype), cus = compute_units();
  if (a.row_stride / vn <= (a.N <= cus ? 1024 * 8 : 256 * 8) || a.row_stride > (int64_t(1) << 30)) return 0;
  const int64_t vecs = split_vecs(a), least = ceil_div(vecs, (int64_t)kSplitThreads * 8);
  if (least > kMostSplits) return 0;
  int64_t splits = ceil_div((a.N <= cus ? 4 : 8) * cus, a.N);
  const int64_t most = ceil_div(vecs, (int64_t)kSplitThreads);
  if (splits > most) splits = most;
  if (splits > kMostSplits) splits = kMostSplits;
  return (int)(splits > least ? splits : least);
}

template <typename T>
int launch_loss_split(const CeArgs &a, int splits, float *rows, int *ws_count, hipStream_t s) {
  constexpr int VN = Vec16<T>::n;
  char *ws = static_cast<char *>(a.workspace) + ce_least_workspace(a.N);
  float2 *parts = reinterpret_cast<float2 *>(ws);
  float *target_logits = reinterpret_cast<float *>(parts + a.N * kMostSplits);
  const int64_t span_vecs = ceil_div(split_vecs(a), (int64_t)splits);
  const dim3 grid((unsigned)(a.N * splits)), block(kSplitThreads);
#define CS_CE_SPLIT(VPT)                                                                                              \
  ce_loss_split_kernel<T, VPT><<<grid, block, 0, s>>>((const T *)a.logits, a.targets, parts, target_logits, a.N, a.V, \
                                                      a.row_stride, a.ignore_index, (int)(span_vecs * VN),          \
                                                      (unsigned)splits)
  switch (ceil_div(span_vecs, (int64_t)kSplitThreads)) {
    case 1: CS_CE_SPLIT(1); break;
    case 2: CS_CE_SPLIT(2); break;
    case 3: CS_CE_SPLIT(3); break;
    case 4: CS_CE_SPLIT(4); break;
    case 5: CS_CE_SPLIT(5); break;
    case 6: CS_CE_SPLIT(6); break;
    case 7: CS_CE_SPLIT(7); break;
    default: CS_CE_SPLIT(8); break;
  }
#undef CS_CE_SPLIT
  const int st = launch_status();
  if (st != CS_OK) return st;
  ce_loss_combine_kernel<<<dim3(1), dim3(1024), 0, s>>>(
      parts, target_logits, splits, rows, a.N, ws_count, a.reduction,
      a.reduction == CS_REDUCTION_NONE ? nullptr : a.loss, a.total_weight, a.targets, a.V, a.ignore_index, a.class_weight);
  return launch_status();
}

// phases: 1 = count the rows that are not ignored, 2 = the row pass,
// 4 = reduce the row losses
int ce_run(const CeArgs &a, int phases, void *stream) {
  int st = ce_validate(a);
  if (st != CS_OK) return st;
  hipStream_t s = as_stream(stream);
  char *ws = static_cast<char *>(a.workspace);
  int *ws_count = reinterpret_cast<int *>(ws);
  float *ws_weight = reinterpret_cast<float *>(ws) + 1;
  float *rows = a.row_loss ? a.row_loss : reinterpret_cast<float *>(ws + kWsHeader);
  if (phases == (1 | 2 | 4)) {
    const int splits = loss_splits(a);
    if (splits > 0) {
      switch (a.dtype) {
        case CS_F32: return launch_loss_split<float>(a, splits, rows, ws_count, s);
        case CS_F16: return launch_loss_split<f16_t>(a, splits, rows, ws_count, s);
        case CS_BF16: return launch_loss_split<bf16_t>(a, splits, rows, ws_count, s);
      }
    }
  }
  // Only the gradient of a mean needs the count before the rows; otherwise the last launch counts.
  const bool mean_gradient = a.dlogits != nullptr && a.reduction == CS_REDUCTION_MEAN;
  // Few rows are counted by the row kernel itself (rows_that_count).
  const bool count_in_rows = mean_gradient && a.class_weight == nullptr && a.N <= kCountInRows;
  const bool count_last = phases == (1 | 2 | 4) && (!mean_gradient || count_in_rows);
  if ((phases & 1) && !count_last) {
    ce_count_kernel<<<dim3(1), dim3(1024), 0, s>>>(a.targets, a.N, a.V, a.ignore_index, ws_count,
                                                   ws_weight, a.class_weight);
    st = launch_status();
    if (st != CS_OK) return st;
  }
  if ((phases & 2) && a.N > 0) {
#define CS_CALL(T, TD)                                                                      \
  st = launch_rows<T, TD>(a.logits, a.dlogits, a.targets, rows, count_last ? nullptr : ws_count, a.N, a.V, \
                          a.row_stride, a.ignore_index,                                     \
                          mean_gradient ? CS_REDUCTION_MEAN : CS_REDUCTION_SUM, a.dloss, a.class_weight, s)
    const bool wide = a.dlogits_dtype != a.dtype;
    switch (a.dtype) {
      case CS_F32: CS_CALL(float, float); break;
      case CS_F64: CS_CALL(double, double); break;
      case CS_F16:
        if (wide) {
          CS_CALL(f16_t, float);
        } else {
          CS_CALL(f16_t, f16_t);
        }
        break;
      case CS_BF16:
        if (wide) {
          CS_CALL(bf16_t, float);
        } else {
          CS_CALL(bf16_t, bf16_t);
        }
        break;
    }
#undef CS_CALL
    if (st != CS_OK) return st;
  }
  if (phases & 4) {
    float *loss = a.reduction == CS_REDUCTION_NONE ? nullptr : a.loss;
    if (count_last) {
      ce_reduce_kernel<true><<<dim3(1), dim3(1024), 0, s>>>(rows, a.N, ws_count, a.reduction, loss, a.total_weight,
                                                            a.targets, a.V, a.ignore_index, a.class_weight);
    } else {
      ce_reduce_kernel<false><<<dim3(1), dim3(1024), 0, s>>>(rows, a.N, ws_count, a.reduction, loss, a.total_weight,
                                                             nullptr, a.V, a.ignore_index, nullptr);
    }
    st = launch_status();
  }
  return st;
}

}  // namespace

extern "C" int cs_fused_classifier(const void *logits, void *dlogits, const int64_t *targets,
                                   float *row_loss, float *loss, float *total_weight,
                                   void *workspace, size_t workspace_bytes, int64_t N, int64_t V,
                                   int64_t row_stride, int64_t ignore_index, int reduction,
                                   float dloss, int dtype, int dlogits_dtype, void *stream) {
  const CeArgs a{logits, dlogits, targets,      row_loss,  loss,  total_weight, workspace,
                 workspace_bytes, N, V, row_stride, ignore_index, reduction, dloss, dtype,
                 dlogits_dtype};
  return ce_run(a, 1 | 2 | 4, stream);
}

extern "C" int cs_fused_classifier_weighted(const void *logits, void *dlogits, const int64_t *targets,
                                            const float *class_weight, float *row_loss, float *loss,
                                            float *total_weight, void *workspace, size_t workspace_bytes,
                                            int64_t N, int64_t V, int64_t row_stride, int64_t ignore_index,
                                            int reduction, float dloss, int dtype, int dlogits_dtype,
                                            void *stream) {
  CeArgs a{logits, dlogits, targets,      row_loss,  loss,  total_weight, workspace,
           workspace_bytes, N, V, row_stride, ignore_index, reduction, dloss, dtype,
           dlogits_dtype};
  a.class_weight = class_weight;
  return ce_run(a, 1 | 2 | 4, stream);
}

// ------------------------------------------------- the call that allocates nothing
// Device memory that belongs to the library, one copy per GPU, held until the process ends:
// the workspace of cs_fused_classifier_static.  In host code this name is only a handle for
// hipGetSymbolAddress; the address that kernels and the host use is the one that call returns.
static __device__ __align__(256) unsigned char scratch[CS_FUSED_CLASSIFIER_STATIC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
// the scratch array's address on each device, looked up once per device (threads may race to
// fill a slot: they store the same value)
std::atomic<void *> scratch_ptr[kMaxDevices];

int static_scratch(void **out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxDevices) return CS_ERR_UNSUPPORTED;
  void *p = scratch_ptr[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    // the current device's copy of the array
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (p == nullptr) return CS_ERR_WORKSPACE;
    scratch_ptr[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return CS_OK;
}
}  // namespace

extern "C" int64_t cs_fused_classifier_static_max_rows(void) {
  return ((int64_t)CS_FUSED_CLASSIFIER_STATIC_SCRATCH_BYTES - (int64_t)kWsHeader) / (int64_t)sizeof(float);
}

extern "C" int cs_fused_classifier_static(const void *logits, void *dlogits, const int64_t *targets,
                                          float *row_loss, float *loss, float *total_weight,
                                          int64_t N, int64_t V, int64_t row_stride,
                                          int64_t ignore_index, int reduction, float dloss,
                                          int dtype, int dlogits_dtype, void *stream) {
  if (N > cs_fused_classifier_static_max_rows()) return CS_ERR_STATIC_LIMIT;
  void *ws = nullptr;
  const int st = static_scratch(&ws);
  if (st != CS_OK) return st;
  // Nothing in the scratch has to start at zero: the launch that counts overwrites the header and
  // the row pass overwrites the N row losses that the reduction then reads.
  const CeArgs a{logits, dlogits, targets, row_loss, loss, total_weight, ws,
                 (size_t)CS_FUSED_CLASSIFIER_STATIC_SCRATCH_BYTES, N, V, row_stride, ignore_index,
                 reduction, dloss, dtype, dlogits_dtype};
  return ce_run(a, 1 | 2 | 4, stream);
}

extern "C" int cs_fused_classifier_phases(const void *logits, void *dlogits,
                                          const int64_t *targets, float *row_loss, float *loss,
                                          float *total_weight, void *workspace,
                                          size_t workspace_bytes, int64_t N, int64_t V,
                                          int64_t row_stride, int64_t ignore_index, int reduction,
                                          float dloss, int dtype, int dlogits_dtype, int phases,
                                          void *stream) {
  if (phases <= 0 || phases > 7) return CS_ERR_INVALID_ARGUMENT;
  const CeArgs a{logits, dlogits, targets,      row_loss,  loss,  total_weight, workspace,
                 workspace_bytes, N, V, row_stride, ignore_index, reduction, dloss, dtype,
                 dlogits_dtype};
  return ce_run(a, phases, stream);
}
