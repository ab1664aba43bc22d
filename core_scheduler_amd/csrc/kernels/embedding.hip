// Embedding gather(-add) forward and deterministic scatter-add backward for
// gfx950.
//
// forward  : out[i,:] = weight[ids[i],:]                (src/compute/embedding.cpp:117-121)
// fwd-add  : out[b,t,:] = wte[ids[b,t],:] + wpe[t,:]    (example/gpt2/gpt2_single_device.cpp:541-545)
// backward : dweight[k,:] (+)= sum_{i: ids[i]==k} dout[i,:], dense, rows that
//            were never indexed are zero            (src/compute/embedding.cpp:147-157)
// positions: dwpe[t,:] (+)= sum_b dout[b,t,:]           (gpt2_single_device.cpp:565-566)
//
// The backward uses no floating point atomics.  It sorts (id, position) keys,
// so equal ids become one contiguous segment in ascending position order, and
// adds each segment's rows in a fixed order in fp32, which makes the result
// independent of scheduling.  Four launches:
//   1. tile sort  - each workgroup bitonic-sorts 1024 keys, one per lane:
//                   exchanges below 64 lanes are wave shuffles, the rest go
//                   through LDS.
//   2. merge rank - every key finds its global rank by binary search in the
//                   other tiles (staged in LDS) and is scattered to its place.
//                   Launches 1 and 2 keep few CUs busy, so further workgroups
//                   of both zero the whole table meanwhile (`=` semantics).
//   3. reduce     - a segmented sum.  A workgroup owns 32 consecutive sorted
//                   entries, each of its 8 waves owns 4 of them and loads
//                   their rows at once.  Runs of equal ids inside a wave are
//                   added in registers; runs that cross waves are folded
//                   through LDS in wave order; a segment that crosses
//                   workgroups leaves one fp32 partial row per workgroup, so
//                   a hot row is read by as many CUs as it has windows.
//   4. finish     - the workgroups of a crossing segment's first window add
//                   that segment's partial rows in window order.  Further
//                   workgroups of the same launch sum the position-table
//                   gradient, which needs no order (of launch 3 where the list
//                   is short, of launch 1 where that has little to fill).
// A list of at most 8192 entries skips 1 and 2: one launch ranks every key by
// comparing it with all others (see emb_bwd_rank_kernel), and does the zero
// fill next to that.  A list of at most 1024 entries of whole aligned vectors
// needs no sort: see emb_bwd_list_kernel.
// The traffic that matters is the dense write of dweight (V*C elements), one
// read of dout and a second write of the indexed rows.
#include "common.hpp"

#include <atomic>
#include <type_traits>

namespace cs_hip {
namespace {

constexpr int kThreads = 256;

// ------------------------------------------------------------------ forward
// One 16-byte vector per thread step, kFwdUnroll steps per thread; `nvec` vectors per row.
// The row and the vector of a thread's first step come from one 32-bit division, the later
// steps advance them by the constant 256 = step_rows * nvec + step_vecs.  Every load of a full
// workgroup is issued without a lane-dependent condition (an index out of range reads row 0 and
// the result is replaced by zeros): the position rows and the indices go first, the table rows
// as soon as the indices are there, so a thread makes two round trips however many steps it has.
#ifndef CS_EMB_FWD_UNROLL
#define CS_EMB_FWD_UNROLL 2
#endif
constexpr int kFwdUnroll = CS_EMB_FWD_UNROLL;

//
// UA: a row of any C >= VN columns, anywhere in memory.  Accesses are at element alignment and the last vector of
// a row is moved back to end with it, so two lanes write its first elements, with the same values.
// One element per thread and a 64-bit division each before: forward and backward together, see
// emb_bwd_reduce_ragged_kernel.
template <typename T, typename IdxT, bool ADD, bool UA>
__global__ __launch_bounds__(kThreads) void emb_fwd_vec_kernel(
    const T *__restrict__ weight, const T *__restrict__ wpe, const IdxT *__restrict__ ids,
    T *__restrict__ out, int64_t n_rows, int64_t C, uint32_t nvec, int64_t num_weights, uint32_t T_len) {
  constexpr int VN = Vec16<T>::n;
  auto column = [&](uint32_t vec) {
    const int64_t c = (int64_t)vec * VN;
    return !UA || c + VN <= C ? c : C - VN;
  };
  auto load = [](const T *p) {
    if constexpr (UA) return load16_unaligned_stream(p);
    return load16(p);
  };
  auto store = [](T *p, const Vec16<T> &v) {
    if constexpr (UA) {
      store16_unaligned_stream(p, v);
    } else {
      store16_stream(p, v);
    }
  };
  constexpr uint32_t kChunk = kThreads * kFwdUnroll;
  const int64_t total = n_rows * nvec;
  // the workgroup's first row: 32-bit divisions where the whole output has fewer than 2^32
  // vectors (a 64-bit division by a variable is a hundred instructions)
  const int64_t chunk_base = (int64_t)blockIdx.x * kChunk;
  int64_t row_base;
  uint32_t rem_base, t_base = 0u;
  if (total <= 0xFFFFFFFFll) {
    const uint32_t cb = (uint32_t)chunk_base;
    const uint32_t rb = cb / nvec;
    rem_base = cb - rb * nvec;
    if constexpr (ADD) t_base = rb % T_len;
    row_base = rb;
  } else {
    row_base = chunk_base / nvec;
    rem_base = (uint32_t)(chunk_base - row_base * nvec);
    if constexpr (ADD) t_base = (uint32_t)(row_base % T_len);
  }
  const uint32_t step_rows = kThreads / nvec, step_vecs = kThreads % nvec;
  const uint32_t local = rem_base + threadIdx.x;
  uint32_t drow = local / nvec;
  uint32_t vec = local - drow * nvec;
  const bool full = chunk_base + kChunk <= total;  // workgroup-uniform

  uint32_t drows[kFwdUnroll], vecs[kFwdUnroll];
#pragma unroll
  for (int u = 0; u < kFwdUnroll; ++u) {
    drows[u] = drow;
    vecs[u] = vec;
    drow += step_rows;
    vec += step_vecs;
    if (vec >= nvec) {
      vec -= nvec;
      ++drow;
    }
  }
  const int64_t row_stride = UA ? C : (int64_t)nvec * VN;
  if (full) {
    IdxT raw_id[kFwdUnroll];
    Vec16<T> w[kFwdUnroll], p[kFwdUnroll];
#pragma unroll
    for (int u = 0; u < kFwdUnroll; ++u) raw_id[u] = ids[row_base + drows[u]];
    if constexpr (ADD) {
#pragma unroll
      for (int u = 0; u < kFwdUnroll; ++u) {
        uint32_t t = t_base + drows[u];  // below 2 T_len + 256: the workgroup spans few rows
        t = t % T_len;
        p[u] = load(wpe + (int64_t)t * row_stride + column(vecs[u]));
      }
    }
    bool ok[kFwdUnroll];
#pragma unroll
    for (int u = 0; u < kFwdUnroll; ++u) {
      const int64_t id = (int64_t)raw_id[u];
      ok[u] = id >= 0 && id < num_weights;
      w[u] = load(weight + (ok[u] ? id : 0) * row_stride + column(vecs[u]));
    }
#pragma unroll
    for (int u = 0; u < kFwdUnroll; ++u) {
      Vec16<T> r;
#pragma unroll
      for (int k = 0; k < VN; ++k) {
        if constexpr (ADD) {
          // fp32 add, one rounding: equals the storage-type add bit for bit
          r.e[k] = ok[u] ? from_acc<T>(to_acc(w[u].e[k]) + to_acc(p[u].e[k])) : T{};
        } else {
          r.e[k] = ok[u] ? w[u].e[k] : T{};
        }
      }
      store(out + (row_base + drows[u]) * row_stride + column(vecs[u]), r);
    }
    return;
  }
  // the last, ragged workgroup
  for (int u = 0; u < kFwdUnroll; ++u) {
    const int64_t row = row_base + drows[u];
    if (row >= n_rows) break;
    const int64_t id = (int64_t)ids[row];
    const bool ok = id >= 0 && id < num_weights;
    Vec16<T> r;
#pragma unroll
    for (int k = 0; k < VN; ++k) r.e[k] = T{};
    if (ok) {
      r = load(weight + id * row_stride + column(vecs[u]));
      if constexpr (ADD) {
        const Vec16<T> pv = load(wpe + (row % T_len) * row_stride + column(vecs[u]));
#pragma unroll
        for (int k = 0; k < VN; ++k) r.e[k] = from_acc<T>(to_acc(r.e[k]) + to_acc(pv.e[k]));
      }
    }
    store(out + row * row_stride + column(vecs[u]), r);
  }
}

// rows shorter than a vector, and few elements of ragged ones (kFewElements)
template <typename T, typename IdxT, bool ADD>
__global__ __launch_bounds__(kThreads) void emb_fwd_scalar_kernel(
    const T *__restrict__ weight, const T *__restrict__ wpe, const IdxT *__restrict__ ids,
    T *__restrict__ out, int64_t n_rows, int64_t C, int64_t num_weights, int64_t T_len) {
  const int64_t total = n_rows * C;
  for (int64_t f = (int64_t)blockIdx.x * kThreads + threadIdx.x; f < total;
       f += (int64_t)gridDim.x * kThreads) {
    const int64_t row = f / C, c = f - row * C;
    const int64_t id = (int64_t)ids[row];
    const bool ok = id >= 0 && id < num_weights;
    if constexpr (ADD) {
      out[f] = ok ? from_acc<T>(to_acc(weight[id * C + c]) + to_acc(wpe[(row % T_len) * C + c]))
                  : T{};
    } else {
      out[f] = ok ? weight[id * C + c] : T{};
    }
  }
}

// ----------------------------------------------------------- backward: keys
// A key orders first by id, then by position.  32-bit keys are used when
// (num_weights << shift) fits, with shift = log2 of the padded entry count.
template <typename KeyT>
struct KeyCodec;
template <>
struct KeyCodec<uint32_t> {
  static constexpr uint32_t kSentinel = 0xFFFFFFFFu;
  __device__ static uint32_t make(uint32_t id, uint32_t pos, int shift) {
    return (id << shift) | pos;
  }
  __device__ static uint32_t id(uint32_t key, int shift) { return key >> shift; }
  __device__ static uint32_t pos(uint32_t key, int shift) { return key & ((1u << shift) - 1u); }
};
template <>
struct KeyCodec<uint64_t> {
  static constexpr uint64_t kSentinel = ~0ull;
  __device__ static uint64_t make(uint32_t id, uint32_t pos, int) {
    return ((uint64_t)id << 32) | pos;
  }
  __device__ static uint32_t id(uint64_t key, int) { return (uint32_t)(key >> 32); }
  __device__ static uint32_t pos(uint64_t key, int) { return (uint32_t)key; }
};

constexpr int kTile = 1024;  // keys per sorted tile = lanes of the sorting workgroup
constexpr uint32_t kNoId = 0xFFFFFFFFu;
#ifndef CS_EMB_WINDOW
#define CS_EMB_WINDOW 32
#endif
constexpr int kWindow = CS_EMB_WINDOW;  // sorted entries per reducing workgroup (at most 64)

// Position-table gradient for one 16-byte vector: dwpe[t, :] (+)= sum_b dout[b, t, :].
template <typename T>
__device__ __forceinline__ void positions_vector(const T *__restrict__ dout, T *__restrict__ dwpe,
                                                 int64_t f, int64_t B, int64_t TC,
                                                 int accumulate) {
  constexpr int VN = Vec16<T>::n;
  float a[VN];
#pragma unroll
  for (int k = 0; k < VN; ++k) a[k] = 0.f;
  // eight loads in flight, none under a condition (a batch row past the end re-reads the last
  // one and is not added)
  for (int64_t b0 = 0; b0 < B; b0 += 8) {
    Vec16<T> v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int64_t b = b0 + u < B ? b0 + u : B - 1;
      v[u] = load16_stream(dout + b * TC + f * VN);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (b0 + u < B)
#pragma unroll
        for (int k = 0; k < VN; ++k) a[k] += to_acc(v[u].e[k]);
  }
  Vec16<T> o;
  if (accumulate) {
    const Vec16<T> old = load16(dwpe + f * VN);
#pragma unroll
    for (int k = 0; k < VN; ++k) o.e[k] = from_acc<T>(to_acc(old.e[k]) + a[k]);
  } else {
#pragma unroll
    for (int k = 0; k < VN; ++k) o.e[k] = from_acc<T>(a[k]);
  }
  store16_stream(dwpe + f * VN, o);
}

// The same for a workgroup of THREADS lanes, with the batch dimension split over S = 2^log2_s lanes
// per vector: a lane walks its rows with 8 loads in flight, so a long batch is a long chain of
// round trips unless it is cut up.  Lane (v, q) adds the rows of slice q for vector v of the
// workgroup's THREADS / S; slices 1.. are left in LDS and slice 0 adds them in order, so the sum
// is a fixed tree.  lds: (S - 1) * (THREADS / S) * VN floats.  With S = 1 this is positions_vector.
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kPosMaxLog2Slices = 4;
constexpr size_t kPosLdsBytesPerLane = 32;  // bound for every S and element type

template <typename T, int THREADS>
__device__ __forceinline__ void positions_block(const T *__restrict__ dout, T *__restrict__ dwpe,
                                                int64_t blk, int64_t B, int64_t TC, int accumulate,
                                                int log2_s, f32x4 *lds, int tid) {
  constexpr int VN = Vec16<T>::n;
  constexpr int kPieces = VN / 4;  // f32x4 pieces of one vector's sums
  if (log2_s == 0) {  // block-uniform
    const int64_t f = blk * THREADS + tid;
    if (f < TC / VN) positions_vector<T>(dout, dwpe, f, B, TC, accumulate);
    return;
  }
  constexpr int kInFlight = 4;  // loads per lane: with the batch cut up there are lanes enough
  const int S = 1 << log2_s;
  const int V = THREADS >> log2_s;
  constexpr int kLog2Threads = __builtin_ctz(THREADS);
  static_assert(1 << kLog2Threads == THREADS && THREADS >> kPosMaxLog2Slices > 0, "a power of two above S");
  const int v = tid & (V - 1);
  const int q = tid >> (kLog2Threads - log2_s);
  const int64_t f = blk * V + v;
  const bool ok = f < TC / VN;
  const int64_t per = (B + S - 1) / S;
  const int64_t b_lo = q * per;
  const int64_t b_hi = b_lo + per < B ? b_lo + per : B;
  float a[VN];
#pragma unroll
  for (int k = 0; k < VN; ++k) a[k] = 0.f;
  if (ok) {
    for (int64_t b0 = b_lo; b0 < b_hi; b0 += kInFlight) {
      Vec16<T> r[kInFlight];
#pragma unroll
      for (int u = 0; u < kInFlight; ++u) {
        const int64_t b = b0 + u < b_hi ? b0 + u : b_hi - 1;
        r[u] = load16_stream(dout + b * TC + f * VN);
      }
#pragma unroll
      for (int u = 0; u < kInFlight; ++u)
        if (b0 + u < b_hi)
#pragma unroll
          for (int k = 0; k < VN; ++k) a[k] += to_acc(r[u].e[k]);
    }
  }
  if (q > 0 && ok) {
#pragma unroll
    for (int h = 0; h < kPieces; ++h) {
      const f32x4 piece = {a[4 * h], a[4 * h + 1], a[4 * h + 2], a[4 * h + 3]};
      lds[((q - 1) * kPieces + h) * V + v] = piece;
    }
  }
  __syncthreads();
  if (q != 0 || !ok) return;
  for (int qq = 1; qq < S; ++qq) {
#pragma unroll
    for (int h = 0; h < kPieces; ++h) {
      const f32x4 piece = lds[((qq - 1) * kPieces + h) * V + v];
      a[4 * h] += piece.x;
      a[4 * h + 1] += piece.y;
      a[4 * h + 2] += piece.z;
      a[4 * h + 3] += piece.w;
    }
  }
  Vec16<T> o;
  if (accumulate) {
    const Vec16<T> old = load16(dwpe + f * VN);
#pragma unroll
    for (int k = 0; k < VN; ++k) o.e[k] = from_acc<T>(to_acc(old.e[k]) + a[k]);
  } else {
#pragma unroll
    for (int k = 0; k < VN; ++k) o.e[k] = from_acc<T>(a[k]);
  }
  store16_stream(dwpe + f * VN, o);
}

// Zero fill of the table, spread over the sort and merge launches, whose own work leaves
// most CUs idle.  Every row is zeroed before the reduce launch writes the indexed ones.
// One fill workgroup clears a fixed number of 16-byte vectors, chosen per launch.
#ifndef CS_EMB_FILL_VECS_RANK
#define CS_EMB_FILL_VECS_RANK 2048
#endif
#ifndef CS_EMB_FILL_VECS_SORT
#define CS_EMB_FILL_VECS_SORT 1024
#endif
#ifndef CS_EMB_FILL_VECS_MERGE
#define CS_EMB_FILL_VECS_MERGE 256
#endif
// Two vectors per lane next to the ranking workgroups (27.9 us per call against 28.6 with one), one
// per lane next to the sort and merge workgroups (16384 tokens x 1600: 60.7 us per call against 65.5
// with 2048 vectors per workgroup in both, 62.7 with 2048 / 256, 62.1 with 1024 / 1024).
constexpr int kFillVecsRank = CS_EMB_FILL_VECS_RANK;
constexpr int kFillVecsSort = CS_EMB_FILL_VECS_SORT;
constexpr int kFillVecsMerge = CS_EMB_FILL_VECS_MERGE;
#ifndef CS_EMB_FILL_SORT_PCT
#define CS_EMB_FILL_SORT_PCT 50  // share of the table cleared in the sort launch
#endif

template <int THREADS, int kFillVecs>
__device__ __forceinline__ void zero_fill_block(u32x4 *__restrict__ dst, int64_t vecs, int64_t blk,
                                                int tid) {
  const u32x4 z = {0u, 0u, 0u, 0u};
  const int64_t v0 = blk * kFillVecs;
  static_assert(kFillVecs % THREADS == 0, "whole vectors per lane");
#pragma unroll 8
  for (int u = 0; u < kFillVecs / THREADS; ++u) {
    const int64_t i = v0 + (int64_t)u * THREADS + tid;
    if (i < vecs) store_stream(dst + i, z);
  }
}

// The position sums that ride in another kernel's launch, on `blocks` workgroups of it.
template <typename T>
struct Positions {
  const T *dout;
  T *dwpe;
  int64_t B, TC;
  int accumulate, log2_slices;
  int64_t blocks;
};

// The table's bytes ahead of its first whole vector and behind its last one (fewer than 16 each).
struct FillEdges {
  uint16_t *head, *tail;
  int head_len, tail_len;  // in 2-byte units: every element type is a whole number of them
};
__device__ __forceinline__ void zero_edges(const FillEdges &e, int tid) {
  if (tid < e.head_len) e.head[tid] = 0;
  if (tid < e.tail_len) e.tail[tid] = 0;
}

// Launch layout, in block order:
//   [0, n_tiles)                sort one tile of 1024 keys
//   + 1                         preset sorted_id to "no id"
//   + positions.blocks          position-table gradient, where kPosFewFill says so
//   + the rest                  zero fill of fill_dst[0, fill_vecs)
template <typename KeyT, typename IdxT, typename T>
__global__ __launch_bounds__(kTile) void emb_bwd_tile_sort_kernel(
    const IdxT *__restrict__ ids, KeyT *__restrict__ tiles, uint32_t *__restrict__ sorted_id,
    int64_t n, int n_tiles, int shift, int64_t num_weights, int64_t padding_idx,
    u32x4 *__restrict__ fill_dst, int64_t fill_vecs, FillEdges edges, Positions<T> positions) {
  // the sorting workgroups keep two key arrays here, the position workgroups their slice sums
  __shared__ f32x4 shared_raw[kTile * kPosLdsBytesPerLane / sizeof(f32x4)];
  static_assert(2 * kTile * sizeof(KeyT) <= sizeof(shared_raw), "the key arrays fit the shared buffer");
  KeyT(*keys)[kTile] = reinterpret_cast<KeyT(*)[kTile]>(shared_raw);
  const int tid = threadIdx.x;
  const int64_t blk = blockIdx.x;
  if (blk > n_tiles + positions.blocks) {
    zero_fill_block<kTile, kFillVecsSort>(fill_dst, fill_vecs, blk - n_tiles - positions.blocks - 1, tid);
    return;
  }
  if (blk > n_tiles) {
    positions_block<T, kTile>(positions.dout, positions.dwpe, blk - n_tiles - 1, positions.B, positions.TC,
                              positions.accumulate, positions.log2_slices, shared_raw, tid);
    return;
  }
  if (blk == n_tiles) {
    zero_edges(edges, tid);
    for (int64_t i = tid; i < n; i += kTile) sorted_id[i] = kNoId;
    return;
  }
  const int64_t p = blk * kTile + tid;
  KeyT key = KeyCodec<KeyT>::kSentinel;
  if (p < n) {
    const int64_t id = (int64_t)ids[p];
    if (id >= 0 && id < num_weights && id != padding_idx)
      key = KeyCodec<KeyT>::make((uint32_t)id, (uint32_t)p, shift);
  }
  // bitonic network, ascending, one key per lane
  int buf = 0;
  for (int k = 2; k <= kTile; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      KeyT other;
      if (j >= kWave) {
        keys[buf][tid] = key;
        __syncthreads();
        other = keys[buf][tid ^ j];
        buf ^= 1;  // the next exchange writes the other array: one barrier per step
      } else {
        other = __shfl_xor(key, j, kWave);
      }
      const bool up = (tid & k) == 0;     // this 2k-block sorts ascending
      const bool lower = (tid & j) == 0;  // this lane is the lower index of its pair
      const KeyT lo = key < other ? key : other;
      const KeyT hi = key < other ? other : key;
      key = (lower == up) ? lo : hi;
    }
  }
  tiles[p] = key;
}

// One thread per key.  rank = own index in own tile + lower bounds in all
// other tiles.  The tiles are staged in LDS a chunk at a time and four of
// them are searched side by side, so the probes overlap.
constexpr int kMergeChunkBytes = 32768;

// Blocks past the keys zero fill_dst[0, fill_vecs).
template <typename KeyT>
__global__ __launch_bounds__(kThreads) void emb_bwd_merge_kernel(
    const KeyT *__restrict__ tiles, uint32_t *__restrict__ sorted_id,
    uint32_t *__restrict__ sorted_pos, int n_tiles, int shift, u32x4 *__restrict__ fill_dst,
    int64_t fill_vecs) {
  constexpr int kChunkTiles = kMergeChunkBytes / (kTile * (int)sizeof(KeyT));
  constexpr int kSide = 4;
  constexpr int kVecPerThread = kMergeChunkBytes / 16 / kThreads;  // 8
  __shared__ u32x4 staged_raw[kMergeChunkBytes / 16];
  const int64_t key_blocks = (int64_t)n_tiles * (kTile / kThreads);
  if ((int64_t)blockIdx.x >= key_blocks) {
    zero_fill_block<kThreads, kFillVecsMerge>(fill_dst, fill_vecs, (int64_t)blockIdx.x - key_blocks, threadIdx.x);
    return;
  }
  const KeyT *staged = reinterpret_cast<const KeyT *>(staged_raw);
  const int64_t g = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int own = (int)(g / kTile);  // block-uniform: 256 divides 1024
  const int local = (int)(g % kTile);
  const KeyT key = tiles[g];
  const bool real = key != KeyCodec<KeyT>::kSentinel;
  int64_t rank = local;
  for (int c0 = 0; c0 < n_tiles; c0 += kChunkTiles) {
    const int c_tiles = n_tiles - c0 < kChunkTiles ? n_tiles - c0 : kChunkTiles;
    const int c_vecs = c_tiles * kTile * (int)sizeof(KeyT) / 16;
    const u32x4 *src = reinterpret_cast<const u32x4 *>(tiles + (int64_t)c0 * kTile);
    u32x4 v[kVecPerThread];
#pragma unroll
    for (int u = 0; u < kVecPerThread; ++u) {
      const int i = u * kThreads + threadIdx.x;
      v[u] = src[i < c_vecs ? i : c_vecs - 1];  // all requested before the first is used
    }
    __syncthreads();  // the previous chunk is no longer being searched
#pragma unroll
    for (int u = 0; u < kVecPerThread; ++u) {
      const int i = u * kThreads + threadIdx.x;
      if (i < c_vecs) staged_raw[i] = v[u];
    }
    __syncthreads();
    for (int b0 = 0; b0 < c_tiles; b0 += kSide) {
      const KeyT *tile[kSide];
      int lb[kSide];
#pragma unroll
      for (int u = 0; u < kSide; ++u) {
        const int b = b0 + u < c_tiles ? b0 + u : c_tiles - 1;
        tile[u] = staged + b * kTile;
        lb[u] = 0;
      }
      // lower bound in a power-of-two tile: kTile/2, kTile/4, ... 1, then one last probe
      for (int step = kTile >> 1; step > 0; step >>= 1) {
        KeyT probe[kSide];
#pragma unroll
        for (int u = 0; u < kSide; ++u) probe[u] = tile[u][lb[u] + step - 1];
#pragma unroll
        for (int u = 0; u < kSide; ++u) lb[u] += probe[u] < key ? step : 0;
      }
#pragma unroll
      for (int u = 0; u < kSide; ++u) {
        const int b = c0 + b0 + u;
        if (b0 + u >= c_tiles || b == own) continue;
        // lb counts the keys < key so far; one last probe decides the element at the bound
        const KeyT at = tile[u][lb[u]];
        rank += lb[u] + (at < key ? 1 : 0);
      }
    }
  }
  if (!real) return;
  sorted_id[rank] = KeyCodec<KeyT>::id(key, shift);
  sorted_pos[rank] = KeyCodec<KeyT>::pos(key, shift);
}

// -------------------------------------------- backward: ranking a short list
// With few enough keys (they all fit in the LDS of one workgroup) sorting takes one launch
// instead of two: a key's place in the sorted order is the number of keys below it (keys are
// distinct: they contain the position), found by comparing it with every other key.  That is
// n^2 comparisons, 2 VALU operations each and nothing else, spread evenly over the chip, next
// to the zero fill that the same launch does.
//
// A workgroup of 1024 lanes ranks OWN = 32 or 16 keys.  It first builds every key of the list
// in its LDS.  Lane l then owns key (l mod OWN) of the workgroup's and belongs to one of
// 1024 / OWN groups; group g compares against the 16-byte key quads g, g + 1024 / OWN, ...: the
// groups of a wave read adjacent quads (no bank conflict, every lane of a group the same
// address).  The partial counts of a key are added through the LDS.
//
// 16 keys where that is at most one workgroup per CU (4096 entries) and the fill takes less time than the
// ranking (a table of up to 32 MB), 32 otherwise.  Launch, us, 32 / 16: 4000 entries and a table of 8 MB
// 6.9 / 6.0, 30 MB 8.1 / 7.0, 46 MB 8.6 / 9.5, 77 MB 13.7 / 15.0; 8192 entries and 77 MB (a second round of ranking
// workgroups) 14.8 / 20.4.  64 keys take 9.6 us at 4000 entries.
// Launch layout, in block order (the ranking workgroups run longest, so they start first):
//   [0, rank_blocks)            rank OWN keys each; also preset the unused tail of sorted_id
//   + the rest                  zero fill of fill_dst[0, fill_vecs)
constexpr int kRankThreads = 1024;
constexpr int64_t kRankFewKeys = 4096;          // 16 keys per workgroup up to here,
constexpr int64_t kRankFewFill = (int64_t)1 << 21;  // and up to this many 16-byte vectors of fill
#ifndef CS_EMB_RANK_MAX_KEY_BYTES
#define CS_EMB_RANK_MAX_KEY_BYTES 32768
#endif
constexpr size_t kRankMaxKeyBytes = CS_EMB_RANK_MAX_KEY_BYTES;  // longest key list that is ranked this way
constexpr size_t kRankPartBytes = (size_t)kRankThreads * sizeof(int);

template <typename KeyT, typename IdxT, int kRankOwn>
__global__ __launch_bounds__(kRankThreads) void emb_bwd_rank_kernel(
    const IdxT *__restrict__ ids, uint32_t *__restrict__ sorted_id,
    uint32_t *__restrict__ sorted_pos, int64_t n, int n_quads, int shift, int64_t num_weights,
    int64_t padding_idx, int rank_blocks, u32x4 *__restrict__ fill_dst, int64_t fill_vecs, FillEdges edges) {
  constexpr int kRankGroups = kRankThreads / kRankOwn;
  typedef KeyT Quad __attribute__((ext_vector_type(4)));
  extern __shared__ u32x4 rank_lds[];  // the key list and the partial counts
  __shared__ int valid_of_wave[kRankThreads / kWave];
  const int tid = threadIdx.x;
  const int64_t blk = blockIdx.x;
  if (blk == 0) zero_edges(edges, tid);
  if (blk >= rank_blocks) {
    zero_fill_block<kRankThreads, kFillVecsRank>(fill_dst, fill_vecs, blk - rank_blocks, tid);
    return;
  }
  KeyT *keys = reinterpret_cast<KeyT *>(rank_lds);  // [4 n_quads], padded with sentinels
  int *part = reinterpret_cast<int *>(keys + (size_t)n_quads * 4);  // [kRankGroups][kRankOwn]
  const int lane = tid & (kWave - 1);
  const int wave = tid >> 6;
  const int n_keys = n_quads * 4;

  // ---- every key of the list, and how many are real
  int mine = 0;
  constexpr int kIdsInFlight = 8;  // the whole list of 8192 in one round trip
  for (int i0 = tid; i0 < n_keys; i0 += kRankThreads * kIdsInFlight) {
    IdxT raw[kIdsInFlight];
#pragma unroll
    for (int u = 0; u < kIdsInFlight; ++u) {
      const int i = i0 + u * kRankThreads;
      raw[u] = ids[i < n ? i : n - 1];  // no load under a condition: they all go out at once
    }
#pragma unroll
    for (int u = 0; u < kIdsInFlight; ++u) {
      const int i = i0 + u * kRankThreads;
      if (i >= n_keys) break;
      KeyT key = KeyCodec<KeyT>::kSentinel;
      const int64_t id = (int64_t)raw[u];
      if (i < n && id >= 0 && id < num_weights && id != padding_idx)
        key = KeyCodec<KeyT>::make((uint32_t)id, (uint32_t)i, shift);
      keys[i] = key;
      mine += key != KeyCodec<KeyT>::kSentinel ? 1 : 0;
    }
  }
  const int in_wave = wave_reduce(mine, SumOp{});
  if (lane == 0) valid_of_wave[wave] = in_wave;
  __syncthreads();
  int n_valid = 0;
#pragma unroll
  for (int w = 0; w < kRankThreads / kWave; ++w) n_valid += valid_of_wave[w];

  // ---- entries past the real keys read "no id": each ranking workgroup presets a share
  {
    const int tail = (int)n - n_valid;
    const int share = (tail + rank_blocks - 1) / rank_blocks;
    for (int i = tid; i < share; i += kRankThreads) {
      const int64_t at = (int64_t)n_valid + blk * share + i;
      if (at < n) sorted_id[at] = kNoId;
    }
  }

  // ---- partial counts
  const int slot = lane & (kRankOwn - 1);
  const int group = wave * (kWave / kRankOwn) + lane / kRankOwn;
  const int own_at = (int)blk * kRankOwn + slot;
  const KeyT own = own_at < n_keys ? keys[own_at] : KeyCodec<KeyT>::kSentinel;
  const Quad *quads = reinterpret_cast<const Quad *>(keys);
  int below = 0;
#pragma unroll 4
  for (int q = group; q < n_quads; q += kRankGroups) {
    const Quad k = quads[q];
    below += (k.x < own ? 1 : 0) + (k.y < own ? 1 : 0) + (k.z < own ? 1 : 0) + (k.w < own ? 1 : 0);
  }
  part[group * kRankOwn + slot] = below;
  __syncthreads();
  if (tid < kRankOwn && own != KeyCodec<KeyT>::kSentinel) {
    int rank = 0;
#pragma unroll
    for (int g = 0; g < kRankGroups; ++g) rank += part[g * kRankOwn + tid];
    sorted_id[rank] = KeyCodec<KeyT>::id(own, shift);
    sorted_pos[rank] = KeyCodec<KeyT>::pos(own, shift);
  }
}

__device__ __forceinline__ uint32_t lane_value(uint32_t v, int lane) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
}

// ------------------------------------------------------ backward: reduction
constexpr int kOwn = 4;                         // sorted entries per wave
constexpr int kRedWaves = kWindow / kOwn;       // 8
constexpr int kRedThreads = kRedWaves * kWave;  // 512: two workgroups share a CU
constexpr int kFinThreads = 256;                // finish kernel: lanes of a workgroup
constexpr int64_t kFinWideRow = 1024;           // two columns to each beyond this row length,
constexpr int64_t kFinMostAtOnce = 2048;        // and where there are more workgroups than this
#ifndef CS_EMB_FIN_DIRECT_ROWS
#define CS_EMB_FIN_DIRECT_ROWS 8
#endif
#ifndef CS_EMB_FIN_MAX_GROUPS
#define CS_EMB_FIN_MAX_GROUPS 8
#endif
#ifndef CS_EMB_FIN_IN_FLIGHT
#define CS_EMB_FIN_IN_FLIGHT 8
#endif
constexpr int kFinInFlight = CS_EMB_FIN_IN_FLIGHT;      // rows a lane of a group loads before it adds (a multiple of 8)
constexpr int kFinDirectRows = CS_EMB_FIN_DIRECT_ROWS;  // segments of up to this many partial rows: one column per lane
constexpr int kFinMaxGroups = CS_EMB_FIN_MAX_GROUPS;    // lane groups that share the rows of a longer segment
#ifndef CS_EMB_VPL
#define CS_EMB_VPL 2
#endif
constexpr int kVpl = CS_EMB_VPL;                // 16-byte column vectors per lane per column chunk

// Lists of up to this many windows (8192 entries, one reducing workgroup per CU) have the position-table sums in
// the reduce launch, longer ones in the finish launch (see there): kernels of a call, us, reduce / finish /
// before both, next to the zero fill: [1,123] x 768 24.3 / 25.3 / 24.1, [4,512] x 768 27.2 / 27.5 / 28.8,
// [8,512] x 1600 49.7 / 50.1 / 53.2, [6,1024] x 768 30.3 / 30.7 / 31.8, [8,1024] x 1600 56.7 / 56.7 / 61.6.
// A longer list with little to fill (16-byte vectors; none where the gradient is added to) has them in the sort launch,
// which leaves most of the chip idle then: kernels of a call, us, finish / sort: 16384 x 1600 bf16 accumulating 56.8 /
// 51.9 (Zipf) and 63.1 / 58.4 (uniform), tables of 3 MB 45.1 / 41.5, 32 MB 49.1 / 47.2, 64 MB 51.2 / 51.4, 161 MB 55.7 /
// 57.4; 32768 x 768 46 MB 54.5 / 53.8, 77 MB 55.1 / 57.1; 16384 x 512 fp32 8 MB 34.7 / 30.9, 103 MB 37.0 / 39.6.
// Lists of up to this many windows have a slice of 64 vectors of the columns to a workgroup, so that more than half of the
// CUs have one: kernels of a call, us, whole rows / slices: 4000 x 512 fp32 14.2 / 13.5, added to the table 16.7 / 14.1,
// [3,400] x 1600 fp32 26.3 / 18.4, [4,1024] x 1600 into 1000 rows 20.4 / 19.1, [3,349] x 1024
// 14.9 / 14.0; but [8,1024] x 768 25.6 / 26.3, 16384 x 1600 56.2 / 58.9.  Rows of two slices only while every workgroup has
// a CU: 2048 x 640 bf16 13.2 / 12.7, but [14,309] x 640 15.7 / 16.3, into 1000 rows 14.7 / 15.7, [14,309] x 1024 20.9 /
// 21.2 (three slices, fp32 x 640: 18.5 / 17.6).
constexpr int64_t kSlicedWindows = 192;
constexpr int64_t kSlicedWindowsTwo = 128;
constexpr int64_t kPosFewFill = (int64_t)3 << 20;
constexpr int64_t kPosEarlyWindows = 256;

// Workgroup w reduces sorted entries [kWindow w, kWindow (w + 1)).  partial rows live at
// partial[(w*2 + slot) * C]: slot 0 for a run that came in over the window's
// left edge and ends inside, slot 1 for a run that leaves over its right edge.
template <typename T, int VPL>
__global__ __launch_bounds__(kRedThreads, 2048 / kRedThreads) void emb_bwd_reduce_kernel(
    const T *__restrict__ dout, const uint32_t *__restrict__ sorted_id,
    const uint32_t *__restrict__ sorted_pos, T *__restrict__ dweight, float *__restrict__ partial,
    int64_t n, int64_t C, int accumulate, int by_freq, int64_t windows, int slices, T *__restrict__ dwpe, int64_t B,
    int64_t TC, int pos_log2_slices) {
  constexpr int VN = Vec16<T>::n;
  constexpr int kChunkCols = kWave * VPL * VN;
  extern __shared__ float lds[];  // [kRedWaves][2 slots][kChunkCols]
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid >> 6;
  const int nvec = (int)(C / VN);
  if (blockIdx.x >= windows * slices) {
    positions_block<T, kRedThreads>(dout, dwpe, blockIdx.x - windows * slices, B, TC, accumulate, pos_log2_slices,
                                    reinterpret_cast<f32x4 *>(lds), tid);
    return;
  }
  const int64_t w = slices == 1 ? blockIdx.x : blockIdx.x / (unsigned)slices;
  const int slice = (int)(blockIdx.x - w * slices);
  const int64_t p0 = w * kWindow;

  // ---- ids of the window (lane l <-> entry p0 + l), the entry before and the entry after
  const int64_t p = p0 + lane;
  const bool in_window = lane < kWindow;
  // lanes 0..3: the positions of this wave's four entries, asked for together with the ids
  // (an entry past the real ones holds no position; it is never used)
  // The four index loads go out together: none sits under a lane-dependent condition (an entry
  // past the end re-reads the last one and is masked afterwards).
  const int64_t own_p = p0 + wave * kOwn + lane;
  const int64_t last = n - 1;
  const uint32_t raw_pos = sorted_pos[own_p < last ? own_p : last];
  const uint32_t raw_id = sorted_id[p < last ? p : last];
  const uint32_t raw_prev = sorted_id[p > 0 ? (p - 1 < last ? p - 1 : last) : 0];
  uint32_t raw_next = sorted_id[p0 + kWindow < last ? p0 + kWindow : last];  // uniform load
  // keeps the compiler from moving three of the loads below the early exit, where each would
  // wait for the one before it
  asm volatile("" : "+v"(raw_next) : "v"(raw_pos), "v"(raw_id), "v"(raw_prev));
  const uint32_t lane_pos = (lane < kOwn && own_p < n) ? raw_pos : 0u;
  const uint32_t my_id = (in_window && p < n) ? raw_id : kNoId;
  const uint32_t prev_id = (in_window && p > 0 && p <= n) ? raw_prev : kNoId;
  const uint64_t valid = __ballot(my_id != kNoId);
  if (valid == 0) return;  // nothing sorted into this window
  const int n_valid = __popcll(valid);  // valid entries are a prefix of the window
  // true segment heads, and run starts inside the window (a head, or entry 0)
  const uint64_t heads = __ballot(my_id != kNoId && (p == 0 || my_id != prev_id));
  const uint64_t starts = heads | 1ull;
  const uint32_t next_id = (p0 + kWindow < n) ? raw_next : kNoId;
  const uint32_t last_id = __shfl(my_id, n_valid - 1, kWave);
  const bool leaves = n_valid == kWindow && next_id == last_id;    // last run goes over the right edge

  // Of a run [a, b) inside the window: is it a whole segment?
  //   begins here  <=> a is a true head          ends here <=> b < n_valid, or b == n_valid and !leaves
  auto run_end = [&](int a) -> int {  // end of the run that starts at entry a
    const uint64_t later = a >= 63 ? 0ull : (starts >> (a + 1)) << (a + 1);
    const int b = later ? __ffsll((long long)later) - 1 : n_valid;
    return b < n_valid ? b : n_valid;
  };

  for (int cb = slice * kWave * VPL; cb < nvec; cb += slices * kWave * VPL) {
    // ---- level 1: this wave's four entries
    const int e0 = wave * kOwn;
    // all kOwn * VPL row loads are in flight before the first is used: an entry past the valid
    // ones reads row 0, a vector past the row re-reads the row's last one; neither is added
    Vec16<T> r[kOwn][VPL];
#pragma unroll
    for (int e = 0; e < kOwn; ++e) {
      const int64_t pos = e0 + e < n_valid ? (int64_t)__shfl(lane_pos, e, kWave) : 0;
#pragma unroll
      for (int j = 0; j < VPL; ++j) {
        const int idx = cb + lane + kWave * j;
        r[e][j] = load16_stream(dout + pos * C + (int64_t)(idx < nvec ? idx : nvec - 1) * VN);
      }
    }
    float acc[VPL][VN];
    int piece_start = e0;
#pragma unroll
    for (int e = 0; e < kOwn; ++e) {
      const int q = e0 + e;
      if (q >= n_valid) break;
      const bool starts_here = (starts >> q) & 1ull;
      if (e == 0 || starts_here) {
        piece_start = q;
#pragma unroll
        for (int j = 0; j < VPL; ++j)
#pragma unroll
          for (int k = 0; k < VN; ++k) acc[j][k] = 0.f;
      }
#pragma unroll
      for (int j = 0; j < VPL; ++j) {
        if (cb + lane + kWave * j < nvec) {
#pragma unroll
          for (int k = 0; k < VN; ++k) acc[j][k] += to_acc(r[e][j].e[k]);
        }
      }
      const bool piece_ends = e == kOwn - 1 || q + 1 >= n_valid || ((starts >> (q + 1)) & 1ull);
      if (!piece_ends) continue;
      // the run this piece belongs to
      const bool run_starts_in_piece = (starts >> piece_start) & 1ull;
      const bool run_ends_in_piece = q + 1 >= n_valid || ((starts >> (q + 1)) & 1ull);
      const uint32_t id = __shfl(my_id, q, kWave);
      if (run_starts_in_piece && run_ends_in_piece) {
        // a whole run of the window, inside one wave
        const bool seg_begins = (heads >> piece_start) & 1ull;
        const bool seg_ends = !(q + 1 >= n_valid && leaves);
        if (seg_begins && seg_ends) {
          T *dst = dweight + (int64_t)id * C;
          // scale_grad_by_freq: the sum over the id's entries divided by their number
          const float inv = by_freq ? 1.0f / (float)(q - piece_start + 1) : 1.0f;
#pragma unroll
          for (int j = 0; j < VPL; ++j) {
            const int idx = cb + lane + kWave * j;
            if (idx < nvec) {
              Vec16<T> o;
              if (accumulate) {
                const Vec16<T> old = load16(dst + (int64_t)idx * VN);
#pragma unroll
                for (int k = 0; k < VN; ++k) o.e[k] = from_acc<T>(to_acc(old.e[k]) + acc[j][k] * inv);
              } else {
#pragma unroll
                for (int k = 0; k < VN; ++k) o.e[k] = from_acc<T>(acc[j][k] * inv);
              }
              store16_stream(dst + (int64_t)idx * VN, o);
            }
          }
        } else {
          float *dst = partial + (w * 2 + (seg_ends ? 0 : 1)) * C;
#pragma unroll
          for (int j = 0; j < VPL; ++j) {
            const int idx = cb + lane + kWave * j;
            if (idx < nvec) {
#pragma unroll
              for (int k = 0; k < VN; ++k) dst[(int64_t)idx * VN + k] = acc[j][k];
            }
          }
        }
      } else {
        // part of a run that spans waves: slot 1 if it reaches this wave's last entry
        const int slot = e == kOwn - 1 ? 1 : 0;
        // four columns per 16-byte LDS word; word (j*H + h)*64 + lane holds columns
        // (lane + 64 j)*VN + 4h .. + 3, so the lanes of a wave write consecutive words
                constexpr int H = VN / 4;
        f32x4 *dst = reinterpret_cast<f32x4 *>(lds) + (wave * 2 + slot) * (kChunkCols / 4);
#pragma unroll
        for (int j = 0; j < VPL; ++j)
#pragma unroll
          for (int h = 0; h < H; ++h)
            dst[(j * H + h) * kWave + lane] =
                f32x4{acc[j][4 * h], acc[j][4 * h + 1], acc[j][4 * h + 2], acc[j][4 * h + 3]};
      }
    }
    __syncthreads();
    // ---- level 2: runs of the window that span waves, folded in wave order.  A run that
    // spans waves is folded by the wave it starts in (wave 0 for the run that came in over the
    // left edge): that is at most one run per wave, so all folds proceed side by side.
    {
      const int first = wave * kOwn;
      const uint64_t mine = (starts >> first) & ((1ull << kOwn) - 1ull);  // run starts among my entries
      const int boundary = first + kOwn;  // the next wave's first entry
      const bool crosses = boundary < kWindow && ((valid >> boundary) & 1ull) &&
                           !((starts >> boundary) & 1ull);
      if (mine != 0 && crosses) {  // wave-uniform
        const int a = first + (63 - __clzll((long long)mine));  // my last run start: the run that crosses
        const int b = run_end(a);
        const int wb = (b - 1) / kOwn;
        const bool last_reaches_end = (b % kOwn) == 0;  // the run's piece in wave wb ends at its last entry
        const uint32_t id = __shfl(my_id, a, kWave);
        const bool seg_begins = (heads >> a) & 1ull;
        const bool seg_ends = !(b >= n_valid && leaves);
        const bool whole = seg_begins && seg_ends;
        T *drow = dweight + (int64_t)id * C;
        float *prow = partial + (w * 2 + (seg_ends ? 0 : 1)) * C;
        typedef float f32x4 __attribute__((ext_vector_type(4)));
        const f32x4 *lds4 = reinterpret_cast<const f32x4 *>(lds);
        constexpr int kSlices = kChunkCols / 4 / kWave;  // groups of four columns per lane (VPL * VN / 4)
        f32x4 t[kSlices];
#pragma unroll
        for (int v = 0; v < kSlices; ++v) t[v] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int ww = wave; ww <= wb; ++ww) {
          // wave ww's piece of this run reaches its last entry unless the run ends inside it
          const int slot = (ww < wb || last_reaches_end) ? 1 : 0;
          const f32x4 *src = lds4 + (ww * 2 + slot) * (kChunkCols / 4) + lane;
          f32x4 x[kSlices];
#pragma unroll
          for (int v = 0; v < kSlices; ++v) x[v] = src[kWave * v];  // independent LDS reads
#pragma unroll
          for (int v = 0; v < kSlices; ++v) t[v] += x[v];
        }
#pragma unroll
        for (int v = 0; v < kSlices; ++v) {
          // slice v = j*H + h of the layout above
          constexpr int H = VN / 4;
          const int64_t col = ((int64_t)cb + lane + kWave * (v / H)) * VN + 4 * (v % H);
          if (col >= C) continue;  // C is a multiple of VN columns here
          if (whole) {
            const float inv = by_freq ? 1.0f / (float)(b - a) : 1.0f;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              float o = t[v][k] * inv;
              if (accumulate) o += to_acc(drow[col + k]);
              drow[col + k] = from_acc<T>(o);
            }
          } else {
            *reinterpret_cast<f32x4 *>(prow + col) = t[v];
          }
        }
      }
    }
    __syncthreads();
  }
}

// The last level of the segmented sum.  A workgroup looks at window w for kFinThreads * PER of the columns: if
// the run that leaves the window over its right edge began in it (a true segment head), this is that
// segment's first window, and the workgroup adds the segment's partial rows in window order: slot 1 of
// every window the segment leaves, slot 0 of the one it ends in.
//
// Bound by a chain of trips to memory (ids, partial rows) that leaves HBM idle, so the position-table sums of
// a long list, which read all of dout and wait for nothing, run next to it: the first workgroups of the grid,
// because the others are short.  Next to the tile sort they would wait for the bytes of its zero fill (but see
// kPosFewFill).  Kernels of a call, us: 16384 tokens x 1600 Zipf ids 73.3 -> 69.2, uniform 85.9 -> 84.6,
// 32768 x 768 fp32 93.5 -> 89.9; in the reduce launch of such a list they cost what they save.  256 columns per
// workgroup, so that a hot row's sum is shared by several: 14.2 us with the positions at 16384 x 1600; 512
// columns 14.4, 1024 15.2; positions last 17.3.  PER: columns a lane; two for many windows of more than 1024 columns,
// whose workgroups are more than the chip holds at once if most windows are left by a run (backward, one / two:
// 16384 x 1600 bf16 into 1000 rows 37.6 / 36.2, x 2048 fp32 59.5 / 54.4; Zipf ids of 50257 rows 48.5 / 48.5; but
// 32768 x 768 48.5 / 50.0, and one id in every entry 42.4 / 51.2).  dout is read past the caches in both launches:
// kept there it pushes out what a call right behind reads (this launch 14.2 -> 12.3 us, but a gather of the same
// tokens next 12.9 -> 20.1).  That weighs calls back to back; where other work lies between them, the next gather
// finds nothing in the caches either way.
template <typename T, int PER>
__global__ __launch_bounds__(kFinThreads, 5) void emb_bwd_finish_kernel(
    const uint32_t *__restrict__ sorted_id, const float *__restrict__ partial,
    T *__restrict__ dweight, int64_t n, int64_t C, int accumulate, int by_freq, int64_t fin_blocks, int slices,
    const T *__restrict__ dout, T *__restrict__ dwpe, int64_t B, int64_t TC, int pos_log2_slices) {
  constexpr int kFinWaves = kFinThreads / kWave;
  __shared__ int first_other[kFinWaves];
  __shared__ int first_tail[kFinWaves];
  __shared__ f32x4 lds[kFinThreads * kPosLdsBytesPerLane / sizeof(f32x4)];
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid >> 6;
  const int64_t blk = (int64_t)blockIdx.x - (gridDim.x - fin_blocks);
  if (blk < 0) {
    positions_block<T, kFinThreads>(dout, dwpe, blockIdx.x, B, TC, accumulate, pos_log2_slices, lds, tid);
    return;
  }
  const int64_t w = (unsigned)blk / (unsigned)slices;
  const int c0 = (int)(blk - w * slices) * kFinThreads * PER;  // the workgroup's first column
  const int cols = (int)C - c0 < kFinThreads * PER ? (int)C - c0 : kFinThreads * PER;
  const int64_t last = w * kWindow + kWindow - 1;
  if (last + 1 >= n) return;  // nothing after this window
  // Everything the decisions below read, and the two partial rows of the usual case (a segment
  // that ends in the next window), is loaded here at once: taken one after another, each behind
  // the test of the one before, these were five trips to memory behind the kernel boundary.
  // Lane t probes window w + 1 + t: its last entry (does the segment leave it?) and its first
  // (does the segment reach it?).
  const int64_t pw = w + 1 + tid;
  const int64_t pq = pw * kWindow + kWindow - 1;
  uint32_t raw_last = sorted_id[last];
  uint32_t raw_next = sorted_id[last + 1];
  uint32_t raw_first = sorted_id[w * kWindow];
  uint32_t raw_before = sorted_id[w > 0 ? w * kWindow - 1 : 0];
  uint32_t raw_q = sorted_id[pq < n ? pq : n - 1];
  uint32_t raw_f = sorted_id[pw * kWindow < n ? pw * kWindow : n - 1];
  float pre_leave[PER], pre_enter[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int64_t col = c0 + (tid + kFinThreads * j < cols ? tid + kFinThreads * j : 0);
    pre_leave[j] = partial[(w * 2 + 1) * C + col];        // window w, left over its right edge
    pre_enter[j] = partial[((w + 1) * 2 + 0) * C + col];  // window w + 1, entered over its left edge
  }
  asm volatile("" : "+v"(raw_last), "+v"(raw_next), "+v"(raw_first), "+v"(raw_before), "+v"(raw_q), "+v"(raw_f));
#pragma unroll
  for (int j = 0; j < PER; ++j) asm volatile("" : "+v"(pre_leave[j]), "+v"(pre_enter[j]));
  const uint32_t id = raw_last;
  if (id == kNoId || raw_next != id) return;  // no run leaves this window
  // its run began in this window unless the whole window (and the entry before it) has this id
  if (raw_first == id && w > 0 && raw_before == id) return;
  // windows after w whose last entry still has this id are left by the segment too; kFinThreads windows
  // per round.  w_hi: the first window whose last entry is not this id.  The segment ends inside
  // it when its first entry still has the id (`tail`), otherwise at the end of the window before.
  int64_t w_hi = -1;
  bool tail = false;
  for (int64_t base = w + 1; w_hi < 0; base += kFinThreads) {
    const int64_t ww = base + tid;
    const int64_t q = ww * kWindow + kWindow - 1;
    if (base != w + 1) {
      raw_q = sorted_id[q < n ? q : n - 1];
      raw_f = sorted_id[ww * kWindow < n ? ww * kWindow : n - 1];
    }
    const bool other = q >= n || raw_q != id;
    const uint64_t m = __ballot(other);
    const uint64_t reached = __ballot(ww * kWindow < n && raw_f == id);
    if (lane == 0) {
      const int at = m ? __ffsll((long long)m) - 1 : -1;
      first_other[wave] = at;
      first_tail[wave] = at >= 0 ? (int)((reached >> at) & 1) : 0;
    }
    __syncthreads();
    for (int k = 0; k < kFinWaves; ++k) {
      if (first_other[k] >= 0) {
        w_hi = base + k * kWave + first_other[k];
        tail = first_tail[k] != 0;
        break;
      }
    }
    __syncthreads();
  }
  const int64_t w_end = tail ? w_hi : w_hi - 1;  // the window the segment ends in (> w)
  // scale_grad_by_freq: the segment's length, from where it begins in window w to where it ends
  // in window w_end (it fills every window in between)
  float inv = 1.0f;
  if (by_freq) {
    const int64_t qa = w * kWindow + (lane < kWindow ? lane : kWindow - 1);
    const int64_t qb = w_end * kWindow + (lane < kWindow ? lane : kWindow - 1);
    const uint64_t in_first = __ballot(lane < kWindow && sorted_id[qa] == id);                        // a suffix of window w
    const uint64_t in_last = __ballot(lane < kWindow && qb < n && sorted_id[qb < n ? qb : n - 1] == id);  // a prefix of window w_end
    const int64_t count = __popcll(in_first) + (w_end - w - 1) * kWindow + __popcll(in_last);
    inv = 1.0f / (float)count;
  }
  T *dst = dweight + (int64_t)id * C;
  const bool usual = w_end == w + 1;
  // A hot id (many windows): the partial rows are dealt to groups of lanes, one 16-byte piece of a
  // row per lane, eight rows in flight per lane; the groups' sums meet in LDS and are added in
  // group order.  Taken one column per lane instead, the hottest row of a Zipf batch was a chain of
  // 9-18 trips to memory in a single workgroup while all others had finished.
  const int64_t rows_in = w_end - w + 1;  // partial rows of the segment
  const int vc = cols >> 2;               // 16-byte pieces of a row (C is a multiple of four columns here)
  if (rows_in > kFinDirectRows) {
    f32x4 *group_sum = lds;
    int groups = kFinThreads / vc;
    if (groups > kFinMaxGroups) groups = kFinMaxGroups;
    const int g = tid / vc, v = tid - g * vc;
    if (g < groups) {
      f32x4 acc[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) acc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int64_t r0 = g; r0 < rows_in; r0 += kFinInFlight * groups) {
        f32x4 x[kFinInFlight];
#pragma unroll
        for (int u = 0; u < kFinInFlight; ++u) {
          const int64_t r = r0 + (int64_t)u * groups;
          const int64_t rr = r < rows_in ? r : rows_in - 1;
          // rows before the last were left over the right edge (slot 1), the last was entered (slot 0)
          const int64_t slot = rr < rows_in - 1 ? (w + rr) * 2 + 1 : w_end * 2;
          x[u] = *reinterpret_cast<const f32x4 *>(partial + slot * C + c0 + 4 * v);
        }
#pragma unroll
        for (int u = 0; u < kFinInFlight; ++u) {
          const float keep = r0 + (int64_t)u * groups < rows_in ? 1.f : 0.f;
          acc[u & 7].x = fmaf(x[u].x, keep, acc[u & 7].x);
          acc[u & 7].y = fmaf(x[u].y, keep, acc[u & 7].y);
          acc[u & 7].z = fmaf(x[u].z, keep, acc[u & 7].z);
          acc[u & 7].w = fmaf(x[u].w, keep, acc[u & 7].w);
        }
      }
      f32x4 t;
      t.x = ((acc[0].x + acc[1].x) + (acc[2].x + acc[3].x)) + ((acc[4].x + acc[5].x) + (acc[6].x + acc[7].x));
      t.y = ((acc[0].y + acc[1].y) + (acc[2].y + acc[3].y)) + ((acc[4].y + acc[5].y) + (acc[6].y + acc[7].y));
      t.z = ((acc[0].z + acc[1].z) + (acc[2].z + acc[3].z)) + ((acc[4].z + acc[5].z) + (acc[6].z + acc[7].z));
      t.w = ((acc[0].w + acc[1].w) + (acc[2].w + acc[3].w)) + ((acc[4].w + acc[5].w) + (acc[6].w + acc[7].w));
      group_sum[tid] = t;
    }
    __syncthreads();
    if (g == 0) {
      f32x4 t = group_sum[v];
      for (int k = 1; k < groups; ++k) {
        const f32x4 o = group_sum[k * vc + v];
        t.x += o.x;
        t.y += o.y;
        t.z += o.z;
        t.w += o.w;
      }
      const float out[4] = {t.x * inv, t.y * inv, t.z * inv, t.w * inv};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        float o = out[k];
        if (accumulate) o += to_acc(dst[c0 + 4 * v + k]);
        dst[c0 + 4 * v + k] = from_acc<T>(o);
      }
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    if (tid + kFinThreads * j < cols) {
      const int64_t col = c0 + tid + kFinThreads * j;
      // eight interleaved sums keep eight loads in flight; the order is fixed all the same
      float t[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      int64_t ww = w;
      // every window before the last is left over its right edge (slot 1)
      for (; ww + 8 <= w_end; ww += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = partial[((ww + u) * 2 + 1) * C + col];
#pragma unroll
        for (int u = 0; u < 8; ++u) t[u] += v[u];
      }
      if (usual) {  // these came in with the loads above
        t[0] += pre_leave[j];
        t[7] += pre_enter[j];
      } else {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = ww + u < w_end ? partial[((ww + u) * 2 + 1) * C + col] : 0.f;
#pragma unroll
        for (int u = 0; u < 7; ++u) t[u] += v[u];  // at most seven windows are left
        t[7] += partial[(w_end * 2 + 0) * C + col];  // the run that ends there came in over the left edge
      }
      float total = (((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]))) * inv;
      if (accumulate) total += to_acc(dst[col]);
      dst[col] = from_acc<T>(total);
    }
  }
}

// -------------------------------------------- backward: a short list in one launch
// Up to kListMost entries of whole aligned vectors: no sort.  Four waves own an entry and compare the list, which the
// workgroup holds in its LDS, with the entry's id: they know how many ids are below it, so its place in the sorted
// list, and where the others of its segment are.  If its run of the segment starts there, they add the run's rows: up
// to kListWhole entries a run is the whole segment, in longer lists it is cut at the edges of the windows below and
// emb_bwd_finish_kernel adds the partial rows, as it does for the longer lists.  Further workgroups of the launch sum
// the position table, and others write zeros to the rows that no entry names.
//
// Bound by the launch and three trips to memory (the list, the rows, the stores), or by the zeros of a large table.
// us per call, rank + reduce + finish launches before / now, Zipf ids: [1,123] x 768 bf16 into 50257 rows 21.1 / 14.8 (its
// 77 MB of zeros alone 11.9), [9,19] x 128 into 5238 10.1 / 6.1, 16 x 64 into 1000 8.2 / 5.6, [16,41] x 640 into 32434
// 14.4 / 11.7, [1,500] x 512 fp32 added to 4000 rows 12.9 / 8.8, [1,1024] x 768 into 1000 rows 12.3 / 10.8 and into 50257
// 22.1 / 21.2.  Longer lists are left to the sort: the comparisons grow with the square, and a hot id's runs gather
// where its tokens are (all of 8192 x 768 this way: 26 / 49).  One id in every entry, the longest runs there are: x 768
// into 50257 rows 192 entries 21.5 / 19.1, 193 20.5 / 17.9, 1024 21.6 / 20.7.
constexpr int kListThreads = 512;
constexpr int kListGroup = 4;  // waves that share an entry
constexpr int kListEntries = kListThreads / kWave / kListGroup;
constexpr int kListMost = 1024;
constexpr int kListWhole = 192;
// Vectors a lane has of each row: a slice of the columns is 128 of them, and a run at most kWindow rows, one step of eight
// for each of the four waves.  Runs of a whole list are up to kListWhole rows: 16-bit rows then have 16 in flight, of one
// vector a lane, where the slices of 64 are not too many workgroups (one id in 192 entries x 768 into 1000 rows 11.8 / 7.5 us;
// fp32 needs too many registers for that: 99 instead of 80, and 64 columns 4.8 / 5.2).
constexpr int kListVecs = 2;
constexpr int kListInFlight = 16;
constexpr int64_t kListBlocks = 512;  // no more slices than make so many workgroups (1024 x 1600: 1024 41.7 us, 512 38.0)
constexpr int64_t kListFillBytes = 64 << 10;  // zeros a workgroup writes (n = 123 x 768, 77 MB: 32 KB 14.4 us, 64 14.6, 256 16.0)
constexpr int kListFillRows = 4096;  // most table rows a zero-filling workgroup looks after (a bit each in the LDS)

template <typename IdxT>
__device__ __forceinline__ uint32_t usable_id(IdxT raw, int64_t num_weights, int64_t padding_idx) {
  const int64_t id = (int64_t)raw;
  return id >= 0 && id < num_weights && id != padding_idx ? (uint32_t)id : kNoId;
}

// The pair of entries of the workgroup whose turn it is: of every window's the next comes first.  Runs of one id over the
// whole list start at the first entry of each window, and workgroups go to the eight XCDs in turn: in the list's own order
// all of them were on one (1024 entries x 768 into 50257 rows, not in any cache: 23.3 us, so 20.7).  Two slices use two XCDs,
// which will do (512 x 1600 into 1000 rows 11.7 / 10.4, but with different ids 9.8 / 10.9).
constexpr int kPairsAWindow = kWindow / kListEntries;
__device__ __forceinline__ int list_pair(int turn, int pairs) {
  const int window = turn / kPairsAWindow, first = window * kPairsAWindow;
  return first + kPairsAWindow <= pairs ? first + (turn + window) % kPairsAWindow : turn;
}

// Launch layout, in block order:
//   [0, entry_blocks)           kListEntries entries and a slice of the columns each
//   + positions.blocks          position-table gradient
//   + the rest                  zeros to the rows [blk * fill_rows, (blk + 1) * fill_rows) that no entry names
template <typename T, typename IdxT, int VECS>
__global__ __launch_bounds__(kListThreads, 4) void emb_bwd_list_kernel(
    const T *__restrict__ dout, const IdxT *__restrict__ ids, T *__restrict__ dweight, uint32_t *__restrict__ sorted_id,
    float *__restrict__ partial, int n, int C, int64_t num_weights, int64_t padding_idx, int accumulate, int by_freq,
    int entry_blocks, int slices, int fill_rows, Positions<T> positions) {
  constexpr int VN = Vec16<T>::n;
  constexpr int kWaves = kListThreads / kWave;
  constexpr int kPerLane = kListMost / kListThreads;
  constexpr int kChunks = kListMost / (4 * kWave);  // lane l looks at entries [4 l, 4 l + 4) of every chunk of 256
  // the waves' sums (an f32x4 a lane and slot), or the position sums' slices, or a bit per row
  constexpr int kPieces = VN / 4;
  __shared__ f32x4 lds[kListThreads * kPosLdsBytesPerLane / sizeof(f32x4)];
  static_assert(kPieces * kListThreads * sizeof(f32x4) <= sizeof(lds) && sizeof(lds) * 8 >= (size_t)kListFillRows, "they fit");
  __shared__ u32x4 listed[kListMost / 4];
  __shared__ uint16_t rows_of[kWaves][kListWhole];
  __shared__ int long_run[kListEntries];
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid >> 6;
  const int nvec = C / VN;
  const int64_t blk = blockIdx.x;
  if (blk >= entry_blocks && blk < entry_blocks + positions.blocks) {
    positions_block<T, kListThreads>(positions.dout, positions.dwpe, blk - entry_blocks, positions.B, positions.TC,
                                     positions.accumulate, positions.log2_slices, lds, tid);
    return;
  }

  uint32_t id[kPerLane];
  {
    IdxT raw[kPerLane] = {};
    if (n > 0) {
#pragma unroll
      for (int u = 0; u < kPerLane; ++u) {
        const int i = u * kListThreads + tid;
        raw[u] = ids[i < n ? i : n - 1];  // no load under a condition: they all go out at once
      }
    }
#pragma unroll
    for (int u = 0; u < kPerLane; ++u)
      id[u] = u * kListThreads + tid < n ? usable_id(raw[u], num_weights, padding_idx) : kNoId;
  }

  if (blk >= entry_blocks) {  // ---- zeros
    uint32_t *named = reinterpret_cast<uint32_t *>(lds);
    const int64_t row0 = (blk - entry_blocks - positions.blocks) * fill_rows;
    const int rows = num_weights - row0 < fill_rows ? (int)(num_weights - row0) : fill_rows;
    for (int i = tid; i < (rows + 31) / 32; i += kListThreads) named[i] = 0u;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPerLane; ++u) {
      const int64_t r = (int64_t)id[u] - row0;
      if (id[u] != kNoId && r >= 0 && r < rows) atomicOr(&named[r >> 5], 1u << (r & 31));
    }
    __syncthreads();
    T *base = dweight + row0 * C;
    const u32x4 z = {0u, 0u, 0u, 0u};
    const int total = rows * nvec;  // list_rows() bounds it
    const int step_rows = kListThreads / nvec, step_vecs = kListThreads % nvec;
    int row = tid / nvec, vec = tid - row * nvec;
#pragma unroll 4
    for (int f = tid; f < total; f += kListThreads) {
      if (!((named[row >> 5] >> (row & 31)) & 1u)) store_stream(reinterpret_cast<u32x4 *>(base) + f, z);
      row += step_rows;
      vec += step_vecs;
      if (vec >= nvec) {
        vec -= nvec;
        ++row;
      }
    }
    return;
  }

  uint32_t *list = reinterpret_cast<uint32_t *>(listed);
#pragma unroll
  for (int u = 0; u < kPerLane; ++u) list[u * kListThreads + tid] = id[u];
  __syncthreads();

  // ---- the group's entry: its place among the sorted, and its segment
  const int entry = wave / kListGroup, member = wave % kListGroup;
  const int turn = (int)blk / slices, slice = (int)blk - turn * slices;
  const int pair = slices == 1 ? list_pair(turn, (n + kListEntries - 1) / kListEntries) : turn;
  const int p = pair * kListEntries + entry;
  const uint32_t my_id = p < n ? list[p] : kNoId;
  uint32_t from[kChunks];  // the entries with this id, from this one on: a bit each
  int below = 0, before = 0, after = 0;
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const u32x4 v = listed[c * kWave + lane];
    uint32_t m = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      m |= v[k] == my_id ? 1u << k : 0u;
      below += v[k] < my_id ? 1 : 0;
    }
    const int at = p - (c * kWave + lane) * 4;  // this entry's bit, if it is one of the four
    const uint32_t earlier = at >= 4 ? m : at <= 0 ? 0u : m & ((1u << at) - 1u);
    from[c] = m & ~earlier;
    before += __popc(earlier);
    after += __popc(from[c]);
  }
  {  // a wave's counts are below 2^15: two to a register
    const int two = wave_reduce(below | before << 16, SumOp{});
    below = two & 0xFFFF;
    before = two >> 16;
    after = wave_reduce(after, SumOp{});
  }
  const int q = below + before;
  const int w = q / kWindow;
  const bool in_windows = n > kListWhole;
  if (in_windows && p < n && slice == 0 && member == 0 && lane == 0) sorted_id[q] = my_id;
  const bool leads = my_id != kNoId && (before == 0 || (in_windows && q % kWindow == 0));
  const int edge = in_windows ? (w + 1) * kWindow : q + after;
  const bool seg_ends = q + after <= edge;
  const bool whole = before == 0 && seg_ends;
  const int run = !leads ? 0 : seg_ends ? after : edge - q;
  if (member == 0 && lane == 0) long_run[entry] = run > 1;
  uint16_t *rows = rows_of[wave];  // every wave notes the run's rows for itself
  if (run == 1) {
    if (lane == 0) rows[0] = (uint16_t)p;
  } else if (run > 1) {
    int first = 0;
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      const uint64_t lanes_below = (1ull << lane) - 1ull;
      int at = first;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint64_t b = __ballot((from[c] >> k) & 1u);
        at += __popcll(b & lanes_below);
        first += __popcll(b);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if ((from[c] >> k) & 1u) {
          if (at < run) rows[at] = (uint16_t)((c * kWave + lane) * 4 + k);
          ++at;
        }
      }
    }
  }
  __syncthreads();

  // ---- the rows
  const float inv = by_freq ? 1.0f / (float)(before + after) : 1.0f;
  T *dst = dweight + (int64_t)my_id * C;
  float *dst_partial = partial + ((int64_t)w * 2 + (seg_ends ? 0 : 1)) * C;
  auto finish = [&](int at, const float(&sum)[VN]) {
    if (whole) {
      Vec16<T> o;
      if (accumulate) {
        const Vec16<T> old = load16(dst + (int64_t)at * VN);
#pragma unroll
        for (int k = 0; k < VN; ++k) o.e[k] = from_acc<T>(to_acc(old.e[k]) + sum[k] * inv);
      } else {
#pragma unroll
        for (int k = 0; k < VN; ++k) o.e[k] = from_acc<T>(sum[k] * inv);
      }
      store16_stream(dst + (int64_t)at * VN, o);
    } else {
#pragma unroll
      for (int h = 0; h < kPieces; ++h)
        *reinterpret_cast<f32x4 *>(dst_partial + (int64_t)at * VN + 4 * h) =
            f32x4{sum[4 * h], sum[4 * h + 1], sum[4 * h + 2], sum[4 * h + 3]};
    }
  };
  if (run == 1) {  // the waves share the columns
    const T *src = dout + (int64_t)p * C;
    for (int at = (slice * kListGroup + member) * kWave + lane; at < nvec; at += slices * kListGroup * kWave) {
      const Vec16<T> v = load16_stream(src + (int64_t)at * VN);
      float sum[VN];
#pragma unroll
      for (int k = 0; k < VN; ++k) sum[k] = 0.f + to_acc(v.e[k]);
      finish(at, sum);
    }
  }
  bool any_long = false;
#pragma unroll
  for (int e = 0; e < kListEntries; ++e) any_long |= long_run[e] != 0;
  if (!any_long) return;
  // the waves share the rows: kListInFlight vectors a lane in flight (a row past the run re-reads the last one, a vector
  // past the row the row's last one, and neither is added); a step's rows are added in pairs, the waves' sums in order
  constexpr int kRows = kListInFlight / VECS, kVecs = VECS;
  for (int cb = slice * kWave * kVecs; cb < nvec; cb += slices * kWave * kVecs) {
    float acc[kVecs][VN] = {};
    for (int e0 = member; run > 1 && e0 < run; e0 += kListGroup * kRows) {
      const int mine = e0 + (lane & (kRows - 1)) * kListGroup;
      const uint32_t pos = rows[mine < run ? mine : run - 1];
      Vec16<T> v[kRows][kVecs];
#pragma unroll
      for (int r = 0; r < kRows; ++r) {
        const T *src = dout + (int64_t)lane_value(pos, r) * C;
#pragma unroll
        for (int j = 0; j < kVecs; ++j) {
          const int at = cb + j * kWave + lane;
          v[r][j] = load16_stream(src + (int64_t)(at < nvec ? at : nvec - 1) * VN);
        }
      }
#pragma unroll
      for (int j = 0; j < kVecs; ++j)
#pragma unroll
        for (int k = 0; k < VN; ++k) {
          float x[kRows];
#pragma unroll
          for (int r = 0; r < kRows; ++r) x[r] = e0 + r * kListGroup < run ? to_acc(v[r][j].e[k]) : 0.f;
#pragma unroll
          for (int w = 1; w < kRows; w *= 2)
#pragma unroll
            for (int r = 0; r < kRows; r += 2 * w) x[r] += x[r + w];
          acc[j][k] += x[0];
        }
    }
#pragma unroll
    for (int j = 0; j < kVecs; ++j) {
      if (cb + j * kWave >= nvec) break;  // workgroup-uniform
#pragma unroll
      for (int h = 0; h < kPieces; ++h)
        lds[h * kListThreads + tid] = f32x4{acc[j][4 * h], acc[j][4 * h + 1], acc[j][4 * h + 2], acc[j][4 * h + 3]};
      __syncthreads();
      const int at = cb + j * kWave + lane;
      if (run > 1 && member == 0 && at < nvec) {
        float sum[VN];
#pragma unroll
        for (int h = 0; h < kPieces; ++h) {
          f32x4 t = lds[h * kListThreads + tid];
#pragma unroll
          for (int g = 1; g < kListGroup; ++g) t += lds[h * kListThreads + tid + g * kWave];
#pragma unroll
          for (int k = 0; k < 4; ++k) sum[4 * h + k] = t[k];
        }
        finish(at, sum);
      }
      __syncthreads();
    }
  }
}

// Standalone position-table gradient.  The vector form is positions_block on its own (the fused call runs it inside
// one of its launches: see kPosEarlyWindows and kPosFewFill); the scalar form takes any C and any alignment.
template <typename T>
__global__ __launch_bounds__(kTile) void emb_bwd_positions_vec_kernel(const T *__restrict__ dout,
                                                                      T *__restrict__ dwpe, int64_t B,
                                                                      int64_t TC, int accumulate,
                                                                      int log2_slices) {
  __shared__ f32x4 slices[kTile * kPosLdsBytesPerLane / sizeof(f32x4)];
  positions_block<T, kTile>(dout, dwpe, blockIdx.x, B, TC, accumulate, log2_slices, slices, threadIdx.x);
}

// Any C, any alignment: a column per lane, workgroup `blk` of `blocks`.
template <typename T>
__device__ __forceinline__ void positions_columns(const T *__restrict__ dout, T *__restrict__ dwpe, int64_t B,
                                                  int64_t TC, int accumulate, int64_t blk, int64_t blocks) {
  using U = typename Acc<T>::type;
  for (int64_t f = blk * kThreads + threadIdx.x; f < TC; f += blocks * kThreads) {
    double a = 0;  // sequential over the batch, so in double like the rows that are not whole vectors
    auto add = [&](auto count, int64_t b0) {  // so many rows in flight together
      T v[decltype(count)::value];
#pragma unroll
      for (int u = 0; u < decltype(count)::value; ++u) v[u] = dout[(b0 + u) * TC + f];
#pragma unroll
      for (int u = 0; u < decltype(count)::value; ++u) a += (double)to_acc(v[u]);
    };
    int64_t b0 = 0;
    for (; b0 + 8 <= B; b0 += 8) add(std::integral_constant<int, 8>{}, b0);
    // exactly the rest: filling up with the last row again cost a short batch twice what its rows do ([1,1000] x 1003
    // 6.0 us against 4.0)
    switch (B - b0) {
      case 1: add(std::integral_constant<int, 1>{}, b0); break;
      case 2: add(std::integral_constant<int, 2>{}, b0); break;
      case 3: add(std::integral_constant<int, 3>{}, b0); break;
      case 4: add(std::integral_constant<int, 4>{}, b0); break;
      case 5: add(std::integral_constant<int, 5>{}, b0); break;
      case 6: add(std::integral_constant<int, 6>{}, b0); break;
      case 7: add(std::integral_constant<int, 7>{}, b0); break;
    }
    if (accumulate) a += (double)to_acc(dwpe[f]);
    dwpe[f] = from_acc<T>((U)a);
  }
}
template <typename T>
__global__ __launch_bounds__(kThreads) void emb_bwd_positions_kernel(const T *__restrict__ dout,
                                                                     T *__restrict__ dwpe,
                                                                     int64_t B, int64_t TC,
                                                                     int accumulate) {
  positions_columns<T>(dout, dwpe, B, TC, accumulate, blockIdx.x, gridDim.x);
}

// ------------------------------------- backward: rows that are not whole vectors
// fp64, and rows that are not whole aligned 16-byte vectors: the same two levels in double, a column per lane.  (The
// wave-wide loads are contiguous, whatever the alignment; fp32 sums over vectors would round where these do not.)
// A workgroup adds one window's 64 sorted entries, a wave's worth of ids, for 256 columns; 16 rows are in flight.
// Further workgroups of the launch sum the position table.  One workgroup per table row, which walked that row's
// entries one load at a time, was the path before: a hot row was a chain of thousands of trips to memory.  us per
// gather + backward, before / now: bf16 8192 Zipf tokens x 301, 50257 rows 650 / 40, uniform 122 / 39; 16384 x 1599
// 3213 / 86, uniform 245 / 95; 32768 x 769, 100000 rows 6834 / 106, uniform 373 / 110; fp32 16384 x 1599 3489 / 124.
// (Short lists: see emb_bwd_runs_ragged_kernel.)
constexpr int kRagWindow = kWave;
constexpr int kRagThreads = 256;
constexpr int kRagInFlight = 16;

// Partial rows as emb_bwd_reduce_kernel leaves them: slot 0 entered over the window's left edge, slot 1 left over the
// right.  The first window has no slot 0 and the last no slot 1, so they start one row earlier.
__device__ __forceinline__ int64_t ragged_partial(int64_t w, int slot, int64_t C) { return (2 * w + slot - 1) * C; }

template <typename T>
__global__ __launch_bounds__(kRagThreads) void emb_bwd_reduce_ragged_kernel(
    const T *__restrict__ dout, const uint32_t *__restrict__ sorted_id, const uint32_t *__restrict__ sorted_pos,
    T *__restrict__ dweight, double *__restrict__ partial, int64_t n, int64_t C, int accumulate, int by_freq,
    unsigned slices, unsigned row_blocks, T *__restrict__ dwpe, int64_t B, int64_t TC) {
  using U = typename Acc<T>::type;
  static_assert(kRagThreads == kThreads, "the position sums' workgroups");
  if (blockIdx.x >= row_blocks) {
    positions_columns<T>(dout, dwpe, B, TC, accumulate, blockIdx.x - row_blocks, gridDim.x - row_blocks);
    return;
  }
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t w = blockIdx.x / slices;
  const int64_t c = (int64_t)(blockIdx.x % slices) * kRagThreads + threadIdx.x;
  const int64_t cc = c < C ? c : C - 1;
  const int64_t p0 = w * kRagWindow, p = p0 + lane, last = n - 1;
  const uint32_t raw_pos = sorted_pos[p < last ? p : last];
  const uint32_t raw_id = sorted_id[p < last ? p : last];
  const uint32_t raw_prev = sorted_id[p > 0 ? (p - 1 < last ? p - 1 : last) : 0];
  const uint32_t next_id = sorted_id[p0 + kRagWindow < last ? p0 + kRagWindow : last];
  const uint32_t my_id = p < n ? raw_id : kNoId;
  const uint64_t valid = __ballot(my_id != kNoId);
  if (valid == 0) return;
  const int n_valid = __popcll(valid);  // valid entries are a prefix
  const uint64_t heads = __ballot(my_id != kNoId && (p == 0 || my_id != raw_prev));
  const bool leaves = n_valid == kRagWindow && p0 + kRagWindow < n && next_id == lane_value(my_id, kWave - 1);
  const uint32_t my_pos = my_id != kNoId ? raw_pos : 0u;  // an unused entry reads row 0 and is not added
  double acc = 0;
  int start = 0;
  const uint32_t my_row = my_id != kNoId ? my_id : 0u;
  for (int e0 = 0; e0 < n_valid; e0 += kRagInFlight) {
    T v[kRagInFlight], old[kRagInFlight];
#pragma unroll
    for (int u = 0; u < kRagInFlight; ++u) v[u] = dout[(int64_t)lane_value(my_pos, e0 + u) * C + cc];
    if (accumulate) {  // requested with the rows, and not one by one where a segment ends
#pragma unroll
      for (int u = 0; u < kRagInFlight; ++u) old[u] = dweight[(int64_t)lane_value(my_row, e0 + u) * C + cc];
    }
#pragma unroll
    for (int u = 0; u < kRagInFlight; ++u) {
      const int e = e0 + u;
      if (e >= n_valid) break;  // wave-uniform, as every decision here
      acc += (double)to_acc(v[u]);
      const bool at_end = e + 1 == n_valid;
      if (!at_end && !((heads >> (e + 1)) & 1)) continue;
      const bool seg_ends = !(at_end && leaves);
      if (((heads >> start) & 1) && seg_ends) {
        if (by_freq) acc /= (double)(e + 1 - start);
        if (accumulate) acc += (double)to_acc(old[u]);
        if (c < C) dweight[(int64_t)lane_value(my_id, e) * C + c] = from_acc<T>((U)acc);
      } else if (c < C) {
        partial[ragged_partial(w, seg_ends ? 0 : 1, C) + c] = acc;
      }
      acc = 0;
      start = e + 1;
    }
  }
}

// The same of a short list: a workgroup per sorted entry and 256 columns, which adds the run of equal ids that starts
// there and returns at once where none does.  A wave that walks a window visits 64 entries one after the other while
// most of the chip is idle.  WINDOWS: a run is cut at the edges of the windows above and leaves their partial rows, so
// its chain is at most four rounds of loads; otherwise it is added whole, and neither partial rows nor the launch
// behind this one are needed.  The additions are in the order of the windows' either way.
//
// Whole up to 256 entries, where a list of one id is no slower than in windows (n = 256 x 301: 15.8 us against 15.4;
// n = 512 26 / 16); with windows up to 3072, as long as the workgroups are few enough to run at once.  us, windows'
// walk / this, bf16 x 301, table of 1000 rows, uniform: n = 100 21.0 / 6.2, 256 21.2 / 6.5, 500 21.7 / 9.8, 1000 22.2 /
// 11.6, 3000 20.9 / 15.8; of one id: n = 500 15.5 / 13.7, 1000 17.1 / 17.3, 3000 21.5 / 23.6; a table of 50257 rows,
// Zipf: n = 1000 26.2 / 15.5, 3000 27.3 / 18.5; x 1603, uniform: n = 1000 23.2 / 16.6, 2000 21.8 / 21.4, 4000 23.5 / 30.8.
constexpr int64_t kRagWholeEntries = 256;
constexpr int64_t kRagFewEntries = 3072;
constexpr int64_t kRagFewWorkgroups = 8192;

template <typename T, bool WINDOWS>
__global__ __launch_bounds__(kRagThreads) void emb_bwd_runs_ragged_kernel(
    const T *__restrict__ dout, const uint32_t *__restrict__ sorted_id, const uint32_t *__restrict__ sorted_pos,
    T *__restrict__ dweight, double *__restrict__ partial, int64_t n, int64_t C, int accumulate, int by_freq,
    unsigned slices, unsigned row_blocks, T *__restrict__ dwpe, int64_t B, int64_t TC) {
  using U = typename Acc<T>::type;
  if (blockIdx.x >= row_blocks) {
    positions_columns<T>(dout, dwpe, B, TC, accumulate, blockIdx.x - row_blocks, gridDim.x - row_blocks);
    return;
  }
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t p = blockIdx.x / slices, w = p / kRagWindow, last = n - 1;
  const int64_t c = (int64_t)(blockIdx.x % slices) * kRagThreads + threadIdx.x;
  const int64_t cc = c < C ? c : C - 1;
  const int64_t limit = WINDOWS && (w + 1) * kRagWindow < n ? (w + 1) * kRagWindow : n;
  const uint32_t id = sorted_id[p], prev = sorted_id[p > 0 ? p - 1 : 0];
  const uint32_t next = sorted_id[limit < last ? limit : last];
  uint32_t ids = sorted_id[p + lane < last ? p + lane : last], pos = sorted_pos[p + lane < last ? p + lane : last];
  const bool head = p == 0 || prev != id;
  if (id == kNoId || !(head || (WINDOWS && p % kRagWindow == 0))) return;
  T *dst = dweight + (int64_t)id * C + cc;
  const T old = accumulate ? *dst : T{};
  double acc = 0;
  auto add = [&](auto in_flight, int e0, int run) {
    constexpr int K = decltype(in_flight)::value;
    T v[K];
#pragma unroll
    for (int u = 0; u < K; ++u) v[u] = dout[(int64_t)lane_value(pos, e0 + u < run ? e0 + u : run - 1) * C + cc];
#pragma unroll
    for (int u = 0; u < K; ++u)
      if (e0 + u < run) acc += (double)to_acc(v[u]);  // workgroup-uniform, as every decision here
  };
  int64_t q = p;
  for (;;) {
    const uint64_t other = __ballot(q + lane >= limit || ids != id);
    const int run = other ? __ffsll((long long)other) - 1 : kWave;
    int e0 = 0;
    for (; run - e0 > 4; e0 += kRagInFlight) add(std::integral_constant<int, kRagInFlight>{}, e0, run);
    if (e0 < run) add(std::integral_constant<int, 4>{}, e0, run);
    q += run;
    if (run < kWave || q >= limit) break;
    ids = sorted_id[q + lane < last ? q + lane : last];
    pos = sorted_pos[q + lane < last ? q + lane : last];
  }
  if (c >= C) return;
  const bool leaves = WINDOWS && q == limit && limit < n && next == id;
  if (WINDOWS && (!head || leaves)) {
    partial[ragged_partial(w, leaves ? 1 : 0, C) + c] = acc;
    return;
  }
  if (by_freq) acc /= (double)(q - p);
  if (accumulate) acc += (double)to_acc(old);
  *dst = from_acc<T>((U)acc);
}

// The workgroup of a segment's first window adds its partial rows, as emb_bwd_finish_kernel does.
template <typename T>
__global__ __launch_bounds__(kRagThreads) void emb_bwd_finish_ragged_kernel(
    const uint32_t *__restrict__ sorted_id, const double *__restrict__ partial, T *__restrict__ dweight, int64_t n,
    int64_t C, int accumulate, int by_freq, unsigned slices) {
  using U = typename Acc<T>::type;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t w = blockIdx.x / slices;
  const int64_t c = (int64_t)(blockIdx.x % slices) * kRagThreads + threadIdx.x;
  const int64_t p0 = w * kRagWindow, next = p0 + kRagWindow;
  if (next >= n) return;  // nothing after this window
  const uint32_t id = sorted_id[next - 1], after = sorted_id[next], first = sorted_id[p0];
  const uint32_t before = sorted_id[p0 > 0 ? p0 - 1 : 0];
  if (id == kNoId || after != id || (first == id && p0 > 0 && before == id)) return;
  // lane l probes window base + l: does the segment leave it (its last entry), does it reach it (its first)?
  int64_t w_end = -1;
  for (int64_t base = w + 1; w_end < 0; base += kWave) {
    const int64_t a = (base + lane) * kRagWindow, q = a + kRagWindow - 1;
    const uint32_t id_a = sorted_id[a < n ? a : n - 1], id_q = sorted_id[q < n ? q : n - 1];
    const uint64_t stays = __ballot(q >= n || id_q != id), reached = __ballot(a < n && id_a == id);
    if (stays) {
      const int at = __ffsll((long long)stays) - 1;
      w_end = base + at - ((reached >> at) & 1 ? 0 : 1);
    }
  }
  double count = 1;
  if (by_freq) {
    const int64_t qa = p0 + lane, qb = w_end * kRagWindow + lane;
    const uint64_t in_first = __ballot(sorted_id[qa] == id);
    const uint64_t in_last = __ballot(qb < n && sorted_id[qb < n ? qb : n - 1] == id);
    count = (double)(__popcll(in_first) + (w_end - w - 1) * kRagWindow + __popcll(in_last));
  }
  if (c >= C) return;
  const int64_t rows = w_end - w + 1;
  double t[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int64_t r0 = 0; r0 < rows; r0 += 8) {
    double x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int64_t r = r0 + u < rows ? r0 + u : rows - 1;
      x[u] = partial[ragged_partial(w + r, r < rows - 1 ? 1 : 0, C) + c];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (r0 + u < rows) t[u] += x[u];
  }
  double total = ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
  if (by_freq) total /= count;
  T *dst = dweight + (int64_t)id * C + c;
  if (accumulate) total += (double)to_acc(*dst);
  *dst = from_acc<T>((U)total);
}

// ---------------------------------------------------------------- workspace
struct BwdLayout {
  int shift = 0;
  bool key64 = false;
  int64_t n_tiles = 0;
  int64_t n_windows = 0;
  size_t off_tiles = 0, off_sorted_id = 0, off_sorted_pos = 0, off_partial = 0;
  size_t bytes = 0;
};

size_t align256(size_t x) { return (x + 255) / 256 * 256; }

BwdLayout bwd_layout(int64_t n, int64_t C, int64_t num_weights) {
  BwdLayout L;
  L.n_tiles = ceil_div(n, (int64_t)kTile);
  const int64_t padded = L.n_tiles * kTile;
  while ((1ll << L.shift) < padded) ++L.shift;
  // ((V-1) << shift) | (2^shift - 1) must stay below the 32-bit sentinel
  L.key64 = L.shift >= 32 || ((uint64_t)num_weights << L.shift) > 0xFFFFFFFFull;
  L.n_windows = ceil_div(n, (int64_t)kWindow);
  size_t o = 0;
  L.off_tiles = o;
  o = align256(o + (size_t)padded * (L.key64 ? 8 : 4));
  L.off_sorted_id = o;
  o = align256(o + (size_t)n * 4);
  L.off_sorted_pos = o;
  o = align256(o + (size_t)n * 4);
  L.off_partial = o;
  // (the doubles of emb_bwd_reduce_ragged_kernel's windows, which are twice as long, fit as well)
  static_assert(kRagWindow == 2 * kWindow, "2 ceil(n / 64) - 2 rows of doubles are no more than 2 ceil(n / 32) of floats");
  o = align256(o + (size_t)L.n_windows * 2 * (size_t)C * sizeof(float));
  L.bytes = o;
  return L;
}

// Ragged or unaligned rows of up to so many elements in all are gathered element by element: every lane has one, where
// vectors leave most of the chip idle.  us, elements / vectors, bf16: 300 x 301 2.9 / 3.3, 1500 x 301 3.3 / 3.5, 2000 x
// 301 3.6 / 3.5, 4000 x 301 4.4 / 3.7; with positions 3.0 / 3.6, 3.6 / 3.8, 3.9 / 3.8; 8000 x 65 3.4 / 3.7, 16000 x 65
// 4.1 / 3.9; fp32 1500 x 301 3.4 / 3.5, 600 x 1003 3.7 / 3.6.
constexpr int64_t kFewElements = 1 << 19;

template <typename T, typename IdxT, bool ADD>
int fwd_launch(const void *weight, const void *wpe, const void *ids, void *out, int64_t n_rows,
               int64_t C, int64_t num_weights, int64_t T_len, hipStream_t s) {
  constexpr int VN = Vec16<T>::n;
  const int64_t nvec = ceil_div(C, (int64_t)VN);
  const int64_t vec_blocks = ceil_div(n_rows * nvec, (int64_t)kThreads * kFwdUnroll);
  const bool vec_ok = C % VN == 0 && is_aligned16(weight) && is_aligned16(out) &&
                      (!ADD || is_aligned16(wpe)) && nvec <= 0x7fffffff;
  if (vec_ok) {
    if (vec_blocks > 0x7fffffffLL) return CS_ERR_TOO_LARGE;
    emb_fwd_vec_kernel<T, IdxT, ADD, false><<<dim3((unsigned)vec_blocks), dim3(kThreads), 0, s>>>(
        (const T *)weight, (const T *)wpe, (const IdxT *)ids, (T *)out, n_rows, C, (uint32_t)nvec, num_weights,
        (uint32_t)T_len);
  } else if (n_rows * C > kFewElements && C >= VN && nvec <= 0x7fffffff && vec_blocks <= 0x7fffffffLL) {
    emb_fwd_vec_kernel<T, IdxT, ADD, true><<<dim3((unsigned)vec_blocks), dim3(kThreads), 0, s>>>(
        (const T *)weight, (const T *)wpe, (const IdxT *)ids, (T *)out, n_rows, C, (uint32_t)nvec, num_weights,
        (uint32_t)T_len);
  } else {
    int64_t blocks = ceil_div(n_rows * C, (int64_t)kThreads);
    if (blocks > 65536) blocks = 65536;
    emb_fwd_scalar_kernel<T, IdxT, ADD><<<dim3((unsigned)blocks), dim3(kThreads), 0, s>>>(
        (const T *)weight, (const T *)wpe, (const IdxT *)ids, (T *)out, n_rows, C, num_weights,
        T_len);
  }
  return launch_status();
}

template <typename T, bool ADD>
int fwd_idx(const void *weight, const void *wpe, const void *ids, void *out, int64_t n_rows,
            int64_t C, int64_t num_weights, int64_t T_len, int idx_dtype, hipStream_t s) {
  if (idx_dtype == CS_I32)
    return fwd_launch<T, int32_t, ADD>(weight, wpe, ids, out, n_rows, C, num_weights, T_len, s);
  if (idx_dtype == CS_I64)
    return fwd_launch<T, int64_t, ADD>(weight, wpe, ids, out, n_rows, C, num_weights, T_len, s);
  return CS_ERR_INVALID_ARGUMENT;
}

template <bool ADD>
int fwd_dispatch(const void *weight, const void *wpe, const void *ids, void *out, int64_t n_rows,
                 int64_t C, int64_t num_weights, int64_t T_len, int dtype, int idx_dtype,
                 void *stream) {
  if (n_rows < 0 || C <= 0 || num_weights < 0) return CS_ERR_INVALID_ARGUMENT;
  const size_t es = dtype_size(dtype);
  if (es == 0) return CS_ERR_UNSUPPORTED;
  if (idx_dtype != CS_I32 && idx_dtype != CS_I64) return CS_ERR_INVALID_ARGUMENT;
  if (n_rows == 0) return CS_OK;
  if (!weight || !ids || !out || (ADD && !wpe)) return CS_ERR_INVALID_ARGUMENT;
  // an empty table has no row 0 for the lanes that read it in place of an out-of-range id
  if (num_weights == 0) return CS_ERR_INVALID_ARGUMENT;
  // the vector kernel keeps the position-table length in 32 bits
  if (ADD && T_len > 0x7fffffffLL) return CS_ERR_TOO_LARGE;
  if (!aligned_to(weight, es) || !aligned_to(out, es) || (ADD && !aligned_to(wpe, es)) ||
      !aligned_to(ids, idx_dtype == CS_I64 ? 8 : 4))
    return CS_ERR_MISALIGNED;
  hipStream_t s = as_stream(stream);
  switch (dtype) {
    case CS_F32:
      return fwd_idx<float, ADD>(weight, wpe, ids, out, n_rows, C, num_weights, T_len, idx_dtype, s);
    case CS_F64:
      return fwd_idx<double, ADD>(weight, wpe, ids, out, n_rows, C, num_weights, T_len, idx_dtype, s);
    case CS_F16:
      return fwd_idx<f16_t, ADD>(weight, wpe, ids, out, n_rows, C, num_weights, T_len, idx_dtype, s);
    case CS_BF16:
      return fwd_idx<bf16_t, ADD>(weight, wpe, ids, out, n_rows, C, num_weights, T_len, idx_dtype, s);
  }
  return CS_ERR_UNSUPPORTED;
}

// Kernels whose dynamic LDS can exceed the 64 KB a launch gets by default ask for their maximum
// once per device.  `bytes` is one constant per kernel, so racing threads set the same value;
// `done` is that kernel's array of per-device flags.
int allow_dynamic_lds_once(const void *kernel, size_t bytes, std::atomic<bool> *done) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return (int)hipErrorInvalidDevice;
  if (!done[dev].load(std::memory_order_acquire)) {
    const hipError_t e =
        hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e != hipSuccess) return (int)e;
    done[dev].store(true, std::memory_order_release);
  }
  return CS_OK;
}
template <typename KeyT, typename IdxT, int OWN>
int rank_launch(const void *ids, uint32_t *sorted_id, uint32_t *sorted_pos, int64_t n, int64_t n_quads, int shift,
                int64_t num_weights, int64_t padding_idx, u32x4 *fill_dst, int64_t fill_vecs, const FillEdges &edges,
                hipStream_t s) {
  const int64_t rank_blocks = ceil_div(n_quads * 4, (int64_t)OWN);
  int64_t blocks = rank_blocks + ceil_div(fill_vecs, (int64_t)kFillVecsRank);
  if (blocks == 0) {
    if (edges.head_len + edges.tail_len == 0) return CS_OK;
    blocks = 1;
  }
  const size_t lds = (size_t)n_quads * 4 * sizeof(KeyT) + kRankPartBytes;
  static std::atomic<bool> done[64];
  const int st = allow_dynamic_lds_once(reinterpret_cast<const void *>(&emb_bwd_rank_kernel<KeyT, IdxT, OWN>),
                                        kRankMaxKeyBytes + kRankPartBytes, done);
  if (st != CS_OK) return st;
  emb_bwd_rank_kernel<KeyT, IdxT, OWN><<<dim3((unsigned)blocks), dim3(kRankThreads), lds, s>>>(
      (const IdxT *)ids, sorted_id, sorted_pos, n, (int)n_quads, shift, num_weights, padding_idx, (int)rank_blocks,
      fill_dst, fill_vecs, edges);
  return launch_status();
}

// lanes per vector of the position sum: enough that a lane walks at most ~16 rows of the batch
int position_slices(int64_t B) {
  int log2_slices = 0;
  while (log2_slices < kPosMaxLog2Slices && (B >> log2_slices) > 16) ++log2_slices;
  return log2_slices;
}

// a list short enough that its keys are ranked in one launch
template <typename KeyT>
bool ranked(int64_t n) {
  return (size_t)ceil_div(n, (int64_t)4) * 4 * sizeof(KeyT) <= kRankMaxKeyBytes;
}

// Sort + merge.  Both launches clear their share of fill_dst[0, fill_vecs), on the CUs the sorting leaves idle.
// `positions` ride in the sort launch (the caller plans none for a list that is ranked).
template <typename KeyT, typename IdxT, typename T>
int sort_launch(const void *ids, char *ws, const BwdLayout &L, int64_t n, int64_t num_weights,
                int64_t padding_idx, u32x4 *fill_dst, int64_t fill_vecs, const FillEdges &edges,
                const Positions<T> &positions, hipStream_t s) {
  KeyT *tiles = reinterpret_cast<KeyT *>(ws + L.off_tiles);
  uint32_t *sorted_id = reinterpret_cast<uint32_t *>(ws + L.off_sorted_id);
  uint32_t *sorted_pos = reinterpret_cast<uint32_t *>(ws + L.off_sorted_pos);
  const int64_t n_quads = ceil_div(n, (int64_t)4);
  if (ranked<KeyT>(n)) {
    // a short list: one launch ranks every key against all others
    return n_quads * 4 <= kRankFewKeys && fill_vecs <= kRankFewFill
               ? rank_launch<KeyT, IdxT, 16>(ids, sorted_id, sorted_pos, n, n_quads, L.shift, num_weights, padding_idx,
                                             fill_dst, fill_vecs, edges, s)
               : rank_launch<KeyT, IdxT, 32>(ids, sorted_id, sorted_pos, n, n_quads, L.shift, num_weights, padding_idx,
                                             fill_dst, fill_vecs, edges, s);
  }
  // whole fill workgroups to the sort launch, the remainder to the merge launch
  const int64_t sort_fill_blocks = ceil_div(fill_vecs, (int64_t)kFillVecsSort) * CS_EMB_FILL_SORT_PCT / 100;
  const int64_t sort_fill_vecs =
      sort_fill_blocks * kFillVecsSort < fill_vecs ? sort_fill_blocks * kFillVecsSort : fill_vecs;
  const int64_t merge_fill_blocks = ceil_div(fill_vecs - sort_fill_vecs, (int64_t)kFillVecsMerge);
  const int64_t blocks = L.n_tiles + 1 + positions.blocks + sort_fill_blocks;
  const int64_t mblocks = L.n_tiles * kTile / kThreads + merge_fill_blocks;
  if (blocks > 0x7fffffffLL || mblocks > 0x7fffffffLL) return CS_ERR_TOO_LARGE;
  emb_bwd_tile_sort_kernel<KeyT, IdxT, T><<<dim3((unsigned)blocks), dim3(kTile), 0, s>>>(
      (const IdxT *)ids, tiles, sorted_id, n, (int)L.n_tiles, L.shift, num_weights, padding_idx, fill_dst,
      sort_fill_vecs, edges, positions);
  int st = launch_status();
  if (st != CS_OK) return st;
  emb_bwd_merge_kernel<KeyT><<<dim3((unsigned)mblocks), dim3(kThreads), 0, s>>>(
      tiles, sorted_id, sorted_pos, (int)L.n_tiles, L.shift,
      fill_dst ? fill_dst + sort_fill_vecs : nullptr, fill_vecs - sort_fill_vecs);
  return launch_status();
}

template <typename T, int VPL>
int reduce_launch(const void *dout, const uint32_t *sorted_id, const uint32_t *sorted_pos, void *dweight, float *partial,
                  int64_t n, int64_t C, int accumulate, int by_freq, int64_t windows, int slices, int64_t pos_blocks,
                  void *dwpe, int64_t B, int64_t TC, int pos_log2_slices, hipStream_t s) {
  constexpr int VN = Vec16<T>::n;
  constexpr size_t kFold = (size_t)kRedWaves * 2 * kWave * VPL * VN * sizeof(float), kPos = kRedThreads * kPosLdsBytesPerLane;
  constexpr size_t lds = kFold > kPos ? kFold : kPos;
  const int64_t blocks = windows * slices + pos_blocks;
  if (blocks > 0x7fffffffLL) return CS_ERR_TOO_LARGE;
  static std::atomic<bool> done[64];
  const int st = allow_dynamic_lds_once(reinterpret_cast<const void *>(&emb_bwd_reduce_kernel<T, VPL>), lds, done);
  if (st != CS_OK) return st;
  emb_bwd_reduce_kernel<T, VPL><<<dim3((unsigned)blocks), dim3(kRedThreads), lds, s>>>(
      (const T *)dout, sorted_id, sorted_pos, (T *)dweight, partial, n, C, accumulate, by_freq, windows, slices, (T *)dwpe, B,
      TC, pos_log2_slices);
  return launch_status();
}

// `pos_blocks` workgroups of position sums ahead of those that finish `windows` windows.
template <typename T>
int finish_launch(const void *dout, const uint32_t *sorted_id, const float *partial, void *dweight, void *dwpe, int64_t n,
                  int64_t C, int accumulate, int by_freq, int64_t windows, int64_t pos_blocks, int64_t B, int64_t TC,
                  int pos_log2_slices, hipStream_t s) {
  const bool wide = C > kFinWideRow && windows * ceil_div(C, (int64_t)kFinThreads) > kFinMostAtOnce;
  const int64_t slices = ceil_div(C, (int64_t)kFinThreads * (wide ? 2 : 1));
  const int64_t fin_blocks = windows * slices, blocks = fin_blocks + pos_blocks;
  if (blocks > 0x7fffffffLL) return CS_ERR_TOO_LARGE;
  if (blocks == 0) return CS_OK;
  const auto finish = wide ? emb_bwd_finish_kernel<T, 2> : emb_bwd_finish_kernel<T, 1>;
  finish<<<dim3((unsigned)blocks), dim3(kFinThreads), 0, s>>>(sorted_id, partial, (T *)dweight, n, C, accumulate, by_freq,
                                                              fin_blocks, (int)slices, (const T *)dout, (T *)dwpe, B, TC,
                                                              pos_log2_slices);
  return launch_status();
}

// Lists that emb_bwd_list_kernel takes: short, and of rows whose zero-filling workgroups count their vectors in 32 bits.
bool list_rows(int64_t n, int64_t C) { return n <= kListMost && C <= 0x7fffffffLL / kListFillRows; }

template <typename T, typename IdxT>
int list_launch(const void *dout, const void *ids, void *dweight, char *ws, const BwdLayout &L, int64_t n, int64_t C,
                int64_t num_weights, int64_t padding_idx, int accumulate, int by_freq, const Positions<T> &positions,
                hipStream_t s) {
  uint32_t *sorted_id = reinterpret_cast<uint32_t *>(ws + L.off_sorted_id);
  float *partial = reinterpret_cast<float *>(ws + L.off_partial);
  const int64_t pairs = ceil_div(n, (int64_t)kListEntries);
  const bool in_windows = n > kListWhole;
  const int64_t nvec = C / Vec16<T>::n;
  const bool narrow = sizeof(T) == 2 && !in_windows && pairs * ceil_div(nvec, (int64_t)kWave) <= kListBlocks;
  int64_t slices = ceil_div(nvec, (int64_t)(narrow ? 1 : kListVecs) * kWave);
  if (pairs * slices > kListBlocks) slices = pairs < kListBlocks ? kListBlocks / pairs : 1;
  const int64_t entry_blocks = pairs * slices;
  int64_t fill_rows = ceil_div(kListFillBytes, C * (int64_t)sizeof(T));
  if (fill_rows > kListFillRows) fill_rows = kListFillRows;
  const int64_t fill_blocks = accumulate ? 0 : ceil_div(num_weights, fill_rows);
  const int64_t blocks = entry_blocks + positions.blocks + fill_blocks;
  if (blocks > 0x7fffffffLL) return CS_ERR_TOO_LARGE;
  if (blocks == 0) return CS_OK;
  auto kernel = emb_bwd_list_kernel<T, IdxT, kListVecs>;
  if constexpr (sizeof(T) == 2) {
    if (narrow) kernel = emb_bwd_list_kernel<T, IdxT, 1>;
  }
  kernel<<<dim3((unsigned)blocks), dim3(kListThreads), 0, s>>>(
      (const T *)dout, (const IdxT *)ids, (T *)dweight, sorted_id, partial, (int)n, (int)C, num_weights, padding_idx,
      accumulate, by_freq, (int)entry_blocks, (int)slices, (int)fill_rows, positions);
  const int st = launch_status();
  if (st != CS_OK || !in_windows) return st;
  return finish_launch<T>(dout, sorted_id, partial, dweight, nullptr, n, C, accumulate, by_freq, L.n_windows, 0, 0, 1, 0, s);
}

template <typename T>
int bwd_typed(const void *dout, const void *ids, void *dweight, void *dwpe, char *ws,
              const BwdLayout &L, int64_t n, int64_t C, int64_t num_weights, int64_t padding_idx,
              int64_t B, int64_t T_len, int idx_dtype, int accumulate, int by_freq, hipStream_t s) {
  constexpr int VN = Vec16<T>::n;
  const bool vec_ok = !std::is_same_v<T, double> && C % VN == 0 && is_aligned16(dout) &&
                      is_aligned16(dweight) && (!dwpe || is_aligned16(dwpe));
  const int64_t TC = T_len * C;
  // `=` semantics on the fast path: the whole table is zeroed, then indexed rows are written
  u32x4 *fill_dst = nullptr;
  int64_t fill_vecs = 0;
  FillEdges edges{nullptr, nullptr, 0, 0};
  if (!accumulate) {
    char *table = static_cast<char *>(dweight);
    const int64_t bytes = num_weights * C * (int64_t)sizeof(T);
    int64_t head = (int64_t)((16 - reinterpret_cast<uintptr_t>(table) % 16) % 16);
    if (head > bytes) head = bytes;
    fill_dst = reinterpret_cast<u32x4 *>(table + head);
    fill_vecs = (bytes - head) / 16;
    char *tail = table + head + fill_vecs * 16;
    edges = FillEdges{reinterpret_cast<uint16_t *>(table), reinterpret_cast<uint16_t *>(tail), (int)(head / 2),
                      (int)((table + bytes - tail) / 2)};
  }
  if (!vec_ok && num_weights > 0x7fffffffLL) return CS_ERR_TOO_LARGE;
  using P = std::conditional_t<std::is_same_v<T, double>, float, T>;  // (fp64 rows are summed by column)
  const int log2_s = position_slices(B);
  auto pos_blocks = [&](int threads) { return dwpe ? ceil_div(TC / VN, (int64_t)(threads >> log2_s)) : 0; };
  if constexpr (!std::is_same_v<T, double>) {
    if (vec_ok && list_rows(n, C)) {
      const Positions<T> positions{(const T *)dout, (T *)dwpe, B, TC, accumulate, log2_s, pos_blocks(kListThreads)};
      const auto launch = idx_dtype == CS_I64 ? list_launch<T, int64_t> : list_launch<T, int32_t>;
      return launch(dout, ids, dweight, ws, L, n, C, num_weights, padding_idx, accumulate, by_freq, positions, s);
    }
  }
  const bool pos_first = vec_ok && fill_vecs <= kPosFewFill && !(L.key64 ? ranked<uint64_t>(n) : ranked<uint32_t>(n));
  const Positions<P> positions{(const P *)dout, (P *)dwpe, B, TC, accumulate, log2_s, pos_first ? pos_blocks(kTile) : 0};
  int st;
#define CS_SORT(KeyT, IdxT) \
  sort_launch<KeyT, IdxT, P>(ids, ws, L, n, num_weights, padding_idx, fill_dst, fill_vecs, edges, positions, s)
  if (L.key64) {
    st = idx_dtype == CS_I64 ? CS_SORT(uint64_t, int64_t) : CS_SORT(uint64_t, int32_t);
  } else {
    st = idx_dtype == CS_I64 ? CS_SORT(uint32_t, int64_t) : CS_SORT(uint32_t, int32_t);
  }
#undef CS_SORT
  if (st != CS_OK) return st;
  const uint32_t *sorted_id = reinterpret_cast<const uint32_t *>(ws + L.off_sorted_id);
  const uint32_t *sorted_pos = reinterpret_cast<const uint32_t *>(ws + L.off_sorted_pos);
  if (!vec_ok) {
    double *partial = reinterpret_cast<double *>(ws + L.off_partial);
    const int64_t slices = ceil_div(C, (int64_t)kRagThreads);
    const bool whole = n <= kRagWholeEntries, runs = whole || (n <= kRagFewEntries && n * slices <= kRagFewWorkgroups);
    const int64_t window_blocks = ceil_div(n, (int64_t)kRagWindow) * slices;
    const int64_t row_blocks = runs ? n * slices : window_blocks;
    int64_t pos_blocks = dwpe ? ceil_div(TC, (int64_t)kThreads) : 0;
    if (pos_blocks > 65536) pos_blocks = 65536;
    if (row_blocks + pos_blocks > 0x7fffffffLL) return CS_ERR_TOO_LARGE;
    if (row_blocks + pos_blocks == 0) return CS_OK;
    const auto kernel = whole  ? emb_bwd_runs_ragged_kernel<T, false>
                        : runs ? emb_bwd_runs_ragged_kernel<T, true>
                               : emb_bwd_reduce_ragged_kernel<T>;
    kernel<<<dim3((unsigned)(row_blocks + pos_blocks)), dim3(kRagThreads), 0, s>>>(
        (const T *)dout, sorted_id, sorted_pos, (T *)dweight, partial, n, C, accumulate, by_freq, (unsigned)slices,
        (unsigned)row_blocks, (T *)dwpe, B, TC);
    st = launch_status();
    if (st != CS_OK || whole || n <= kRagWindow) return st;  // no segment leaves its workgroup
    emb_bwd_finish_ragged_kernel<T><<<dim3((unsigned)window_blocks), dim3(kRagThreads), 0, s>>>(
        sorted_id, partial, (T *)dweight, n, C, accumulate, by_freq, (unsigned)slices);
    return launch_status();
  }
  if constexpr (!std::is_same_v<T, double>) {
    float *partial = reinterpret_cast<float *>(ws + L.off_partial);
    const int64_t windows = n > 0 ? L.n_windows : 0;
    // The position sums go where the chip is idle: next to the finish workgroups, or next to the reducing ones of a
    // list too short to occupy the chip with those.
    const bool pos_early = windows > 0 && windows <= kPosEarlyWindows;
    if (windows > 0) {
      const int64_t pos = pos_early && !pos_first ? pos_blocks(kRedThreads) : 0;
      const int64_t nvec = C / VN;
      if (nvec > kWave && windows <= (nvec > 2 * kWave ? kSlicedWindows : kSlicedWindowsTwo)) {
        st = reduce_launch<T, 1>(dout, sorted_id, sorted_pos, dweight, partial, n, C, accumulate, by_freq, windows,
                                 (int)ceil_div(nvec, (int64_t)kWave), pos, dwpe, B, TC, log2_s, s);
      } else {
        st = reduce_launch<T, kVpl>(dout, sorted_id, sorted_pos, dweight, partial, n, C, accumulate, by_freq, windows, 1, pos,
                                    dwpe, B, TC, log2_s, s);
      }
      if (st != CS_OK) return st;
    }
    return finish_launch<T>(dout, sorted_id, partial, dweight, dwpe, n, C, accumulate, by_freq, windows,
                            pos_early || pos_first ? 0 : pos_blocks(kFinThreads), B, TC, log2_s, s);
  }
  return CS_ERR_UNSUPPORTED;
}

int bwd_dispatch(const void *dout, const void *ids, void *dweight, void *dwpe, void *workspace,
                 size_t workspace_bytes, int64_t n, int64_t C, int64_t num_weights,
                 int64_t padding_idx, int64_t B, int64_t T_len, int dtype, int idx_dtype,
                 int accumulate, void *stream, int by_freq = 0) {
  if (n < 0 || C <= 0 || num_weights <= 0) return CS_ERR_INVALID_ARGUMENT;
  const size_t es = dtype_size(dtype);
  if (es == 0) return CS_ERR_UNSUPPORTED;
  if (idx_dtype != CS_I32 && idx_dtype != CS_I64) return CS_ERR_INVALID_ARGUMENT;
  if (num_weights >= 0xFFFFFFFFll || n >= 0x7FFFFFFFll) return CS_ERR_TOO_LARGE;
  if (!dweight || (n > 0 && (!dout || !ids))) return CS_ERR_INVALID_ARGUMENT;
  if (!aligned_to(dweight, es) || (dout && !aligned_to(dout, es)) ||
      (dwpe && !aligned_to(dwpe, es)) || (ids && !aligned_to(ids, idx_dtype == CS_I64 ? 8 : 4)))
    return CS_ERR_MISALIGNED;
  const BwdLayout L = bwd_layout(n > 0 ? n : 1, C, num_weights);
  if (!workspace || workspace_bytes < L.bytes || !aligned_to(workspace, 256))
    return CS_ERR_WORKSPACE;
  char *ws = static_cast<char *>(workspace);
  hipStream_t s = as_stream(stream);
  switch (dtype) {
    case CS_F32:
      return bwd_typed<float>(dout, ids, dweight, dwpe, ws, L, n, C, num_weights, padding_idx, B,
                              T_len, idx_dtype, accumulate, by_freq, s);
    case CS_F64:
      return bwd_typed<double>(dout, ids, dweight, dwpe, ws, L, n, C, num_weights, padding_idx, B,
                               T_len, idx_dtype, accumulate, by_freq, s);
    case CS_F16:
      return bwd_typed<f16_t>(dout, ids, dweight, dwpe, ws, L, n, C, num_weights, padding_idx, B,
                              T_len, idx_dtype, accumulate, by_freq, s);
    case CS_BF16:
      return bwd_typed<bf16_t>(dout, ids, dweight, dwpe, ws, L, n, C, num_weights, padding_idx, B,
                               T_len, idx_dtype, accumulate, by_freq, s);
  }
  return CS_ERR_UNSUPPORTED;
}

}  // namespace
}  // namespace cs_hip

using namespace cs_hip;

extern "C" int cs_embedding_forward(const void *weight, const void *indices, void *out,
                                    int64_t n_indices, int64_t C, int64_t num_weights, int dtype,
                                    int idx_dtype, void *stream) {
  return fwd_dispatch<false>(weight, nullptr, indices, out, n_indices, C, num_weights, 1, dtype,
                             idx_dtype, stream);
}

extern "C" int cs_embedding_forward_add(const void *wte, const void *wpe, const void *indices,
                                        void *out, int64_t B, int64_t T, int64_t C,
                                        int64_t num_weights, int dtype, int idx_dtype,
                                        void *stream) {
  if (B < 0 || T <= 0) return CS_ERR_INVALID_ARGUMENT;
  return fwd_dispatch<true>(wte, wpe, indices, out, B * T, C, num_weights, T, dtype, idx_dtype,
                            stream);
}

extern "C" size_t cs_embedding_backward_workspace_bytes(int64_t n_indices, int64_t C,
                                                        int64_t num_weights) {
  if (n_indices < 0 || C <= 0 || num_weights <= 0) return 0;
  return bwd_layout(n_indices > 0 ? n_indices : 1, C, num_weights).bytes;
}

extern "C" int cs_embedding_backward(const void *dout, const void *indices, void *dweight,
                                     void *workspace, size_t workspace_bytes, int64_t n_indices,
                                     int64_t C, int64_t num_weights, int64_t padding_idx,
                                     int dtype, int idx_dtype, int accumulate, void *stream) {
  return bwd_dispatch(dout, indices, dweight, nullptr, workspace, workspace_bytes, n_indices, C,
                      num_weights, padding_idx, 0, 1, dtype, idx_dtype, accumulate, stream);
}

extern "C" int cs_embedding_backward_scaled(const void *dout, const void *indices, void *dweight,
                                            void *workspace, size_t workspace_bytes, int64_t n_indices,
                                            int64_t C, int64_t num_weights, int64_t padding_idx,
                                            int dtype, int idx_dtype, int accumulate, void *stream) {
  return bwd_dispatch(dout, indices, dweight, nullptr, workspace, workspace_bytes, n_indices, C,
                      num_weights, padding_idx, 0, 1, dtype, idx_dtype, accumulate, stream, 1);
}

extern "C" int cs_embedding_backward_fused(const void *dout, const void *indices, void *dwte,
                                           void *dwpe, void *workspace, size_t workspace_bytes,
                                           int64_t B, int64_t T, int64_t C, int64_t num_weights,
                                           int dtype, int idx_dtype, int accumulate,
                                           void *stream) {
  if (B < 0 || T <= 0 || !dwpe) return CS_ERR_INVALID_ARGUMENT;
  return bwd_dispatch(dout, indices, dwte, dwpe, workspace, workspace_bytes, B * T, C,
                      num_weights, -1, B, T, dtype, idx_dtype, accumulate, stream);
}

extern "C" int cs_embedding_backward_positions(const void *dout, void *dwpe, int64_t B, int64_t T,
                                               int64_t C, int dtype, int accumulate,
                                               void *stream) {
  if (B < 0 || T < 0 || C <= 0) return CS_ERR_INVALID_ARGUMENT;
  const size_t es = dtype_size(dtype);
  if (es == 0) return CS_ERR_UNSUPPORTED;
  if (T == 0) return CS_OK;
  if (!dwpe || (B > 0 && !dout)) return CS_ERR_INVALID_ARGUMENT;
  if (!aligned_to(dwpe, es) || (dout && !aligned_to(dout, es))) return CS_ERR_MISALIGNED;
  hipStream_t s = as_stream(stream);
  const int64_t TC = T * C;
#define CS_POS(T)                                                                                       \
  do {                                                                                                  \
    constexpr int VN = Vec16<T>::n;                                                                     \
    /* an empty batch goes to the scalar kernel, which then writes zeros */                            \
    if (!std::is_same_v<T, double> && B > 0 && C % VN == 0 && is_aligned16(dout) && is_aligned16(dwpe)) { \
      const int log2_slices = position_slices(B);                                                       \
      const int64_t vblocks = ceil_div(TC / VN, (int64_t)(kTile >> log2_slices));                       \
      if (vblocks > 0x7fffffffLL) return CS_ERR_TOO_LARGE;                                              \
      emb_bwd_positions_vec_kernel<T><<<dim3((unsigned)vblocks), dim3(kTile), 0, s>>>(                  \
          (const T *)dout, (T *)dwpe, B, TC, accumulate, log2_slices);                                  \
    } else {                                                                                            \
      int64_t blocks = ceil_div(TC, (int64_t)kThreads);                                                 \
      if (blocks > 65536) blocks = 65536;                                                               \
      emb_bwd_positions_kernel<T><<<dim3((unsigned)blocks), dim3(kThreads), 0, s>>>(                    \
          (const T *)dout, (T *)dwpe, B, TC, accumulate);                                               \
    }                                                                                                   \
  } while (0)
  switch (dtype) {
    case CS_F32: CS_POS(float); break;
    case CS_F64: CS_POS(double); break;
    case CS_F16: CS_POS(f16_t); break;
    case CS_BF16: CS_POS(bf16_t); break;
  }
#undef CS_POS
  return launch_status();
}
