// segment_softmax forward and backward (python/kernels/segment.py:233-280,
// csrc/segment_softmax.cpp:235-343 of the reference; the arithmetic follows
// the oracle chain python/reference/segment.py:63-118).
//
// Per segment and channel, in the base-2 domain:
//   y_e = logit_e * log2(e) + 2 log2(max(env_e, 1e-30))   (env_e > 0; else no mass)
//   m = max(null * log2(e), max_e y_e),  w_e = 2^(y_e - m),  D = 2^(null log2 e - m) + sum_e w_e
//   alpha_e = w_e * (1 / D),  null_alpha = 2^(null log2 e - m) * (1 / D)
// which is the natural-base softmax of the reference with the exponent
// rescaled once; v_exp_f32 / v_log_f32 / v_rcp_f32 evaluate it (relative error
// a few 1e-7, inside the 1e-5 parity bar).
//
// Work decomposition.  Rows of more than two 16-byte chunks are cut into slabs
// of up to 8 chunks, one wave per (segment, slab): see the slab kernels.  Rows
// of one or two aligned chunks (C = 4, 8), of C <= 3, and aligned rows of up to
// 64 chunks at the mean degrees that slabs do not suit (uses_slabs) run lane
// groups:
//   * LC lanes cover one edge row (LC = next power of two >= C / V).
//   * Short segments (degree <= CAP) belong to G-lane groups (G = 32, or 64
//     when LC = 64): the group issues all of its segment's loads at once into
//     RMAX register tiles of PG = G / LC rows, so one memory round trip brings
//     the whole segment in; max, sum and normalisation run on the registers
//     and alpha is written once.
//   * Long segments (degree > CAP) belong to a whole 256-thread workgroup:
//     up to RMAXB tiles of PB = 256 / LC rows are staged in registers (one
//     read); longer segments stream twice (an online max/sum pass, then the
//     write pass).  Partial results of the four waves meet in LDS in a fixed
//     order.
//   * With a plan (dpa4k_segment_softmax_plan: the list of long segments of
//     the CSR, built once per graph), workgroups [0, n_long) take one long
//     segment each and the remaining workgroups take SPB consecutive
//     segments and skip the long ones, so no workgroup runs a long segment
//     after its short ones.  This is the degree-binned schedule.  Without a
//     plan, a workgroup handles its own long segments after its short ones.
//     The slab kernels need no plan (theirs is empty).
// All reductions are DPP / ds_swizzle / ds_bpermute butterflies or fixed LDS
// orders: results are reproducible bit for bit from run to run.
#include "common.h"

namespace dpa4k {
namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
constexpr float kLog2e = 1.4426950408889634f;
// Plan layout (int64 words): [0] short-path capacity the plan was built for,
// [1] n_long, [2, 2 + n_long) ascending ids of the long segments, then
// scratch (one count per tile of segments).
constexpr int64_t kPlanHeader = 2;

// ---------------------------------------------------------------------------
// arithmetic
// ---------------------------------------------------------------------------

// y = logit * log2(e) + 2 log2(max(env, 1e-30)) for env > 0, else -inf.
__device__ __forceinline__ float log2_weight(float logit, float env) {
  return env > 0.0f ? logit * kLog2e + 2.0f * __builtin_amdgcn_logf(fmaxf(env, 1e-30f)) : -INFINITY;
}

__device__ __forceinline__ float exp2_of(float x) { return __builtin_amdgcn_exp2f(x); }

// 2^(y - peak), zero when the segment has no mass (peak = -inf).
__device__ __forceinline__ float weight_of(float y, float peak) {
  return peak > -INFINITY ? exp2_of(y - peak) : 0.0f;
}

// The per-row part of y: 2 log2(max(env, 1e-30)) for env > 0, -inf otherwise.
__device__ __forceinline__ float row_term(float env) {
  return env > 0.0f ? 2.0f * __builtin_amdgcn_logf(fmaxf(env, 1e-30f)) : -INFINITY;
}

// y of one value from its row's term: -inf for a row without mass, whatever
// the logit.
__device__ __forceinline__ float log2_weight_of_row(float logit, float term) {
  return term > -INFINITY ? __builtin_fmaf(logit, kLog2e, term) : -INFINITY;
}

// The exponent shift of a column: its peak, or 0 when it has no mass (every
// y is then -inf and 2^(y - 0) = 0).
__device__ __forceinline__ float shift_of(float peak) { return peak > -INFINITY ? peak : 0.0f; }

// 1 / D, with D = 1 for a segment without mass.
__device__ __forceinline__ float inverse_total(float total) {
  return __builtin_amdgcn_rcpf(total > 0.0f ? total : 1.0f);
}

// d l_e / d env = 2 / env where the clamp of the oracle is inactive, 0 elsewhere.
__device__ __forceinline__ float env_gradient(float row_sum, float env) {
  return env >= 1e-30f ? row_sum * 2.0f / env : 0.0f;
}

// Online (max, sum) state of a base-2 softmax: sum = sum_i 2^(y_i - max).
__device__ __forceinline__ void online_add(float& peak, float& sum, float y) {
  if (y == -INFINITY) return;
  if (y > peak) {
    sum = (peak == -INFINITY ? 0.0f : sum * exp2_of(peak - y)) + 1.0f;
    peak = y;
  } else {
    sum += exp2_of(y - peak);
  }
}

// Compensated accumulation (Neumaier's variant of Kahan summation) for the
// loops that run over a whole long segment in one lane.  Over millions of
// rows a plain fp32 running sum drops the many terms far below its own
// magnitude (each rounds away) and comes out biased low: about 5e-4 for a
// 67M-row segment of N(0, 4) logits.  `carry` keeps what each addition
// rounded off; the caller folds it in once, with sum + carry.
__device__ __forceinline__ void compensated_add(float& sum, float& carry, float x) {
  const float t = sum + x;
  carry += fabsf(sum) >= fabsf(x) ? (sum - t) + x : (x - t) + sum;
  sum = t;
}

// online_add with a compensated sum; a new maximum rescales both parts.
__device__ __forceinline__ void online_add(float& peak, float& sum, float& carry, float y) {
  if (y == -INFINITY) return;
  if (y > peak) {
    const float scale = peak == -INFINITY ? 0.0f : exp2_of(peak - y);
    sum *= scale;
    carry *= scale;
    compensated_add(sum, carry, 1.0f);
    peak = y;
  } else {
    compensated_add(sum, carry, exp2_of(y - peak));
  }
}

// Merges (peak_b, sum_b) into (peak, sum); symmetric in its operands.
__device__ __forceinline__ void online_merge(float& peak, float& sum, float peak_b, float sum_b) {
  const float top = fmaxf(peak, peak_b);
  const float a = peak == -INFINITY ? 0.0f : sum * exp2_of(peak - top);
  const float b = peak_b == -INFINITY ? 0.0f : sum_b * exp2_of(peak_b - top);
  peak = top;
  sum = a + b;
}

// Butterflies over the lane bits [FROM, TO) of the wave.
template <int FROM, int TO>
__device__ __forceinline__ float span_max(float v) {
  if constexpr (FROM <= 1 && TO > 1) v = fmaxf(v, xor_lane<1>(v));
  if constexpr (FROM <= 2 && TO > 2) v = fmaxf(v, xor_lane<2>(v));
  if constexpr (FROM <= 4 && TO > 4) v = fmaxf(v, xor_lane<4>(v));
  if constexpr (FROM <= 8 && TO > 8) v = fmaxf(v, xor_lane<8>(v));
  if constexpr (FROM <= 16 && TO > 16) v = fmaxf(v, xor_lane<16>(v));
  if constexpr (FROM <= 32 && TO > 32) v = fmaxf(v, xor_lane<32>(v));
  return v;
}

template <int FROM, int TO, typename T>
__device__ __forceinline__ T span_sum(T v) {
  if constexpr (FROM <= 1 && TO > 1) v += xor_lane<1>(v);
  if constexpr (FROM <= 2 && TO > 2) v += xor_lane<2>(v);
  if constexpr (FROM <= 4 && TO > 4) v += xor_lane<4>(v);
  if constexpr (FROM <= 8 && TO > 8) v += xor_lane<8>(v);
  if constexpr (FROM <= 16 && TO > 16) v += xor_lane<16>(v);
  if constexpr (FROM <= 32 && TO > 32) v += xor_lane<32>(v);
  return v;
}

template <int MASK>
__device__ __forceinline__ void merge_lane(float& peak, float& sum) {
  const float peak_b = xor_lane<MASK>(peak);
  const float sum_b = xor_lane<MASK>(sum);
  online_merge(peak, sum, peak_b, sum_b);
}

template <int FROM, int TO>
__device__ __forceinline__ void span_merge(float& peak, float& sum) {
  if constexpr (FROM <= 1 && TO > 1) merge_lane<1>(peak, sum);
  if constexpr (FROM <= 2 && TO > 2) merge_lane<2>(peak, sum);
  if constexpr (FROM <= 4 && TO > 4) merge_lane<4>(peak, sum);
  if constexpr (FROM <= 8 && TO > 8) merge_lane<8>(peak, sum);
  if constexpr (FROM <= 16 && TO > 16) merge_lane<16>(peak, sum);
  if constexpr (FROM <= 32 && TO > 32) merge_lane<32>(peak, sum);
}

// ---------------------------------------------------------------------------
// geometry
// ---------------------------------------------------------------------------

// Short-path capacity (rows) for rows of LC lanes: 24 / V tiles of a
// 32-lane group.  Forward and backward share it, so one plan serves both.
constexpr int short_capacity(int v, int lc) { return (24 / v) * ((lc > 32 ? lc : 32) / lc); }

// Lanes per short group: 32, or LC when a row is wider.  (16-lane groups
// with twice the tiles fit a config-2-like graph into one dispatch round
// but need over 96 VGPRs, which halves the occupancy, and ran slower.)
constexpr int short_group_log(int log_lc) { return log_lc > 5 ? log_lc : 5; }

template <int V, int LOG_LC>
struct Geo {
  static constexpr int LC = 1 << LOG_LC;               // lanes per edge row
  static constexpr int LOG_G = short_group_log(LOG_LC);
  static constexpr int G = 1 << LOG_G;                 // lanes per short segment
  static constexpr int GPW = 64 / G;                   // short segments per wave
  static constexpr int PG = G / LC;                    // rows per group load
  static constexpr int SPB = kBlock / G;               // segments per short workgroup
  static constexpr int PB = kBlock / LC;               // rows per workgroup load
  static constexpr int CAP = short_capacity(V, LC);    // longest short segment
  static constexpr int RMAX = CAP / PG;                // register tiles, short path
  static constexpr int RMAXB = 16 / V;                 // register tiles, staged long path
  static constexpr int UNROLL = 2;                     // loads in flight per thread, streaming path
};

// Register tiles of rows: tile i holds, for this lane, the row of CSR slot
// first + i * STEP + row_lane when that slot is below `end` and the lane is
// live (its column lies inside the row).
//
// Natural order (slot = edge): rows are read and written through buffer
// views rebased at `base` (wave-uniform, at most the lowest slot of the
// active lanes), and a lane without a row uses kNoRow; callers keep every
// slot of the window within 2^31 bytes of `base`.  No load sits in a branch.
// With an order: the order entries of every tile are loaded first (at slot 0
// for lanes without a row), then the rows they name at a clamped index; `e`
// keeps the edge id, or -1 where there is no row.  Callers guard the ordered
// loads with n_edges > 0, so index 0 exists.  A lane that is not live reads
// column 0 instead of its own (null rows included); its results are neither
// stored nor reduced into the live lanes' results.
template <int R, int STEP, bool kOrdered>
struct Tiles {
  int64_t first, base;
  int32_t rows_left;  // min(end - first, 2^31 - 1)
  int row_lane;
  bool live;
  uint32_t row_bytes, col_bytes;
  int64_t e[kOrdered ? R : 1];

  __device__ __forceinline__ Tiles(int64_t first_, int64_t end, int64_t base_, int row_lane_, bool live_,
                                   int64_t column, int64_t channels)
      : first(first_), base(kOrdered ? 0 : base_), row_lane(row_lane_), live(live_) {
    const int64_t left = end - first_;
    rows_left = static_cast<int32_t>(left < 0 ? 0 : (left > 0x7fffffff ? 0x7fffffff : left));
    row_bytes = static_cast<uint32_t>(channels) * 4u;
    col_bytes = static_cast<uint32_t>(column) * 4u;
  }
  __device__ __forceinline__ bool row(int i) const { return live & (i * STEP + row_lane < rows_left); }
  // kNoRow without a row, 0 with one; folded into offsets by an OR, which keeps
  // the offset arithmetic free of selects (a select here becomes a branch).
  __device__ __forceinline__ uint32_t miss(int i) const { return (static_cast<uint32_t>(row(i)) - 1u) & kNoRow; }
  __device__ __forceinline__ int64_t slot(int i) const { return first + static_cast<int64_t>(i) * STEP + row_lane; }
  // natural order: byte offsets of this lane's chunk and of its row's scalar
  __device__ __forceinline__ uint32_t rel(int i) const {
    return static_cast<uint32_t>(first - base) + static_cast<uint32_t>(i * STEP + row_lane);
  }
  __device__ __forceinline__ uint32_t at(int i) const { return (rel(i) * row_bytes + col_bytes) | miss(i); }
  __device__ __forceinline__ uint32_t scalar_at(int i) const { return (rel(i) * 4u) | miss(i); }
  // ordered: edge ids of every tile
  __device__ __forceinline__ void gather_ids(const int64_t* __restrict__ order, int64_t n_edges) {
    if constexpr (kOrdered) {
#pragma unroll
      for (int i = 0; i < R; ++i) e[i] = order[row(i) ? slot(i) : 0];
#pragma unroll
      for (int i = 0; i < R; ++i) e[i] = row(i) && e[i] >= 0 && e[i] < n_edges ? e[i] : -1;
    }
  }
  __device__ __forceinline__ void clear_ids() {
    if constexpr (kOrdered)
#pragma unroll
      for (int i = 0; i < R; ++i) e[i] = -1;
  }
};

// Lane roles inside a workgroup for rows of LC lanes.
template <int V, int LOG_LC>
struct Lanes {
  using S = Geo<V, LOG_LC>;
  int lane, wave, k, p, pb, gidx;
  bool live;
  int64_t column;
  __device__ Lanes(int64_t chunks) {
    lane = threadIdx.x & 63;
    wave = threadIdx.x >> 6;
    k = lane & (S::LC - 1);
    p = (threadIdx.x & (S::G - 1)) >> LOG_LC;
    pb = threadIdx.x >> LOG_LC;
    gidx = threadIdx.x >> S::LOG_G;
    live = k < chunks;
    column = static_cast<int64_t>(k) * V;
  }
};

// Segment bounds of the SPB segments [first, first + SPB) held by lanes
// 0..SPB of every wave (one vector load); lane i gets segment first + i.
struct BlockBounds {
  int64_t lo, hi;
};

template <int SPB>
__device__ __forceinline__ BlockBounds block_bounds(const int64_t* __restrict__ offsets, int64_t first,
                                                    int64_t n_nodes, int64_t n_edges) {
  const int lane = threadIdx.x & 63;
  const int64_t last = first + SPB < n_nodes ? first + SPB : n_nodes;
  const int64_t index = first + lane < last ? first + lane : last;
  int64_t lo = offsets[index];
  lo = lo < 0 ? 0 : (lo > n_edges ? n_edges : lo);
  int64_t hi = __shfl_down(lo, 1);
  if (hi < lo || first + lane >= last) hi = lo;
  return {lo, hi};
}

// Bounds of this lane's group among the 64 / G consecutive segments of its
// wave (segments first + wave * 64 / G + j), read with scalar loads: the
// addresses are wave-uniform, so no vector load and no lane shuffle stands
// between the kernel's start and the first row loads.
template <int LOG_G>
__device__ __forceinline__ void group_bounds(const int64_t* __restrict__ offsets, int64_t first, int64_t n_nodes,
                                             int64_t n_edges, int64_t& begin, int64_t& end) {
  constexpr int GPW = 64 >> LOG_G;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int64_t s0 = first + static_cast<int64_t>(wave) * GPW;
  int64_t o[GPW + 1];
#pragma unroll
  for (int j = 0; j <= GPW; ++j) o[j] = offsets[s0 + j < n_nodes ? s0 + j : n_nodes];
  __builtin_amdgcn_sched_barrier(0);  // the loads above overlap; clamps follow
#pragma unroll
  for (int j = 0; j <= GPW; ++j) o[j] = o[j] < 0 ? 0 : (o[j] > n_edges ? n_edges : o[j]);
  const int g = static_cast<int>(threadIdx.x & 63) >> LOG_G;
  begin = o[0];
  end = o[1];
#pragma unroll
  for (int j = 1; j < GPW; ++j)
    if (g == j) {
      begin = o[j];
      end = o[j + 1];
    }
  if (end < begin) end = begin;
}

// ---------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------

struct ForwardArgs {
  const float* logit;
  const float* env;
  const int64_t* offsets;
  const float* null_logit;
  const int64_t* order;
  float* alpha;
  float* null_alpha;
  int64_t n_edges, n_nodes, channels;
};

// Loads tile i of the forward input for this lane: the logit chunk and the
// envelope (0, hence no mass, where the lane has no row).  Natural order
// reads through the views; with an order the caller has gathered the ids.
template <int V, int R, int STEP, bool kOrdered>
__device__ __forceinline__ void forward_loads(const ForwardArgs& a, const Tiles<R, STEP, kOrdered>& t,
                                              int64_t column, float (&value)[R][V], float (&envelope)[R]) {
  if constexpr (!kOrdered) {
    const BufferView logit = row_view(a.logit, t.base, a.n_edges, a.channels);
    const BufferView env = row_view(a.env, t.base, a.n_edges, 1);
    // Logit rows are read once and loaded non-temporally (config 2: 14.3 ->
    // 13.7 us, 2R: 138 -> 127 us); the envelope loads keep the default
    // policy, which was faster for them.
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const fvec<V> x = buffer_load_vec<V, kNonTemporal>(logit, t.at(i));
      envelope[i] = buffer_load_f32(env, t.scalar_at(i));
#pragma unroll
      for (int v = 0; v < V; ++v) value[i][v] = x.v[v];
    }
    __builtin_amdgcn_sched_barrier(0);  // every load above is issued before any use
  } else {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int64_t e = t.e[i] >= 0 ? t.e[i] : 0;
      const fvec<V> x = load_vec_stream<V>(a.logit + e * a.channels + column);
      const float env = a.env[e];
      envelope[i] = t.e[i] >= 0 ? env : 0.0f;
#pragma unroll
      for (int v = 0; v < V; ++v) value[i][v] = x.v[v];
    }
  }
}

// Stores alpha of tile i where the lane has a row (tiles [0, tiles) hold
// every row of the lane).
template <int V, int R, int STEP, bool kOrdered>
__device__ __forceinline__ void forward_stores(const ForwardArgs& a, const Tiles<R, STEP, kOrdered>& t,
                                               int64_t column, const float (&alpha)[R][V], int tiles = R) {
  if constexpr (!kOrdered) {
    const BufferView out = row_view(a.alpha, t.base, a.n_edges, a.channels);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (i >= tiles) continue;
      fvec<V> row;
#pragma unroll
      for (int v = 0; v < V; ++v) row.v[v] = alpha[i][v];
      buffer_store_vec_stream<V>(out, t.at(i), row);
    }
  } else {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (t.e[i] >= 0) {
        fvec<V> row;
#pragma unroll
        for (int v = 0; v < V; ++v) row.v[v] = alpha[i][v];
        store_vec_stream<V>(a.alpha + t.e[i] * a.channels + column, row);
      }
    }
  }
}

// Tiles of [first, end) with every load issued before any arithmetic.
template <int V, int R, int STEP, bool kOrdered>
__device__ __forceinline__ Tiles<R, STEP, kOrdered> forward_tiles(const ForwardArgs& a, int64_t first, int64_t end,
                                                                  int64_t base, int row_lane, bool live,
                                                                  int64_t column, float (&value)[R][V],
                                                                  float (&envelope)[R]) {
  Tiles<R, STEP, kOrdered> t(first, end, base, row_lane, live, column, a.channels);
#pragma unroll
  for (int i = 0; i < R; ++i) {
    envelope[i] = 0.0f;
#pragma unroll
    for (int v = 0; v < V; ++v) value[i][v] = 0.0f;
  }
  if constexpr (kOrdered) {
    t.clear_ids();
    if (a.n_edges > 0) {
      t.gather_ids(a.order, a.n_edges);
      forward_loads<V>(a, t, column, value, envelope);
    }
  } else {
    forward_loads<V>(a, t, column, value, envelope);
  }
  return t;
}

// One long segment [begin, end) of `segment`, processed by the whole workgroup.
template <int V, int LOG_LC, bool kNull, bool kOrdered>
__device__ void forward_long(const ForwardArgs& a, int64_t segment, int64_t begin, int64_t end,
                             float (*partial)[2][Geo<V, LOG_LC>::LC * V]) {
  using S = Geo<V, LOG_LC>;
  begin = uniform_i64(begin);  // one segment per workgroup
  end = uniform_i64(end);
  constexpr int LC = S::LC, PB = S::PB, RMAXB = S::RMAXB;
  const Lanes<V, LOG_LC> L(a.channels / V);
  const int64_t column = L.live ? L.column : 0;
  const int64_t degree = end - begin;
  fvec<V> n0;
#pragma unroll
  for (int v = 0; v < V; ++v) n0.v[v] = -INFINITY;
  if constexpr (kNull) n0 = load_vec<V>(a.null_logit + segment * a.channels + column);
  float nv[V];
#pragma unroll
  for (int v = 0; v < V; ++v) nv[v] = n0.v[v] * kLog2e;
  float peak[V], total[V];
  if (degree <= RMAXB * PB) {
    // staged: every row of the segment in registers, one read
    float value[RMAXB][V], envelope[RMAXB];
    const auto t = forward_tiles<V, RMAXB, PB, kOrdered>(a, begin, end, begin, L.pb, L.live, column, value, envelope);
#pragma unroll
    for (int v = 0; v < V; ++v) peak[v] = -INFINITY;
#pragma unroll
    for (int i = 0; i < RMAXB; ++i)
#pragma unroll
      for (int v = 0; v < V; ++v) {
        value[i][v] = log2_weight(value[i][v], envelope[i]);
        peak[v] = fmaxf(peak[v], value[i][v]);
      }
#pragma unroll
    for (int v = 0; v < V; ++v) peak[v] = span_max<LC, 64>(peak[v]);
    if ((L.lane >> LOG_LC) == 0)
#pragma unroll
      for (int v = 0; v < V; ++v) partial[L.wave][0][L.k * V + v] = peak[v];
    __syncthreads();
#pragma unroll
    for (int v = 0; v < V; ++v) {
      float m = partial[0][0][L.k * V + v];
      for (int q = 1; q < kWaves; ++q) m = fmaxf(m, partial[q][0][L.k * V + v]);
      peak[v] = kNull ? fmaxf(m, nv[v]) : m;
      total[v] = 0.0f;
    }
#pragma unroll
    for (int i = 0; i < RMAXB; ++i)
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const float w = weight_of(value[i][v], peak[v]);
        value[i][v] = w;
        total[v] += w;
      }
#pragma unroll
    for (int v = 0; v < V; ++v) total[v] = span_sum<LC, 64>(total[v]);
    if ((L.lane >> LOG_LC) == 0)
#pragma unroll
      for (int v = 0; v < V; ++v) partial[L.wave][1][L.k * V + v] = total[v];
    __syncthreads();
    float nw[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
      float sum = partial[0][1][L.k * V + v];
      for (int q = 1; q < kWaves; ++q) sum = sum + partial[q][1][L.k * V + v];
      nw[v] = kNull ? weight_of(nv[v], peak[v]) : 0.0f;
      total[v] = inverse_total(sum + nw[v]);
    }
#pragma unroll
    for (int i = 0; i < RMAXB; ++i)
#pragma unroll
      for (int v = 0; v < V; ++v) value[i][v] *= total[v];
    forward_stores<V>(a, t, column, value);
    if (kNull && threadIdx.x < LC && L.live) {
      fvec<V> out;
#pragma unroll
      for (int v = 0; v < V; ++v) out.v[v] = nw[v] * total[v];
      store_vec<V>(a.null_alpha + segment * a.channels + L.column, out);
    }
    __syncthreads();  // partial[] is reused by the next long segment
    return;
  }

  // streaming: online max/sum pass, then the write pass
  float run_sum[V], carry[V];
#pragma unroll
  for (int v = 0; v < V; ++v) {
    peak[v] = -INFINITY;
    run_sum[v] = 0.0f;
    carry[v] = 0.0f;
  }
  for (int64_t base = begin; base < end; base += S::UNROLL * PB) {
    float value[S::UNROLL][V], envelope[S::UNROLL];
    forward_tiles<V, S::UNROLL, PB, kOrdered>(a, base, end, base, L.pb, L.live, column, value, envelope);
#pragma unroll
    for (int u = 0; u < S::UNROLL; ++u)
#pragma unroll
      for (int v = 0; v < V; ++v) online_add(peak[v], run_sum[v], carry[v], log2_weight(value[u][v], envelope[u]));
  }
#pragma unroll
  for (int v = 0; v < V; ++v) {
    run_sum[v] = run_sum[v] + carry[v];
    span_merge<LC, 64>(peak[v], run_sum[v]);
  }
  if ((L.lane >> LOG_LC) == 0)
#pragma unroll
    for (int v = 0; v < V; ++v) {
      partial[L.wave][0][L.k * V + v] = peak[v];
      partial[L.wave][1][L.k * V + v] = run_sum[v];
    }
  __syncthreads();
  float nw[V];
#pragma unroll
  for (int v = 0; v < V; ++v) {
    float m = partial[0][0][L.k * V + v];
    float s = partial[0][1][L.k * V + v];
    for (int q = 1; q < kWaves; ++q) online_merge(m, s, partial[q][0][L.k * V + v], partial[q][1][L.k * V + v]);
    if (kNull) online_add(m, s, nv[v]);
    peak[v] = m;
    nw[v] = kNull ? weight_of(nv[v], m) : 0.0f;
    total[v] = inverse_total(s);
  }
  for (int64_t base = begin; base < end; base += S::UNROLL * PB) {
    float value[S::UNROLL][V], envelope[S::UNROLL];
    const auto t = forward_tiles<V, S::UNROLL, PB, kOrdered>(a, base, end, base, L.pb, L.live, column, value, envelope);
#pragma unroll
    for (int u = 0; u < S::UNROLL; ++u)
#pragma unroll
      for (int v = 0; v < V; ++v) value[u][v] = weight_of(log2_weight(value[u][v], envelope[u]), peak[v]) * total[v];
    forward_stores<V>(a, t, column, value);
  }
  if (kNull && threadIdx.x < LC && L.live) {
    fvec<V> out;
#pragma unroll
    for (int v = 0; v < V; ++v) out.v[v] = nw[v] * total[v];
    store_vec<V>(a.null_alpha + segment * a.channels + L.column, out);
  }
  __syncthreads();
}

// Short segment of this lane's group (degree <= CAP), all in registers; rows
// are addressed from `base` (see Tiles).
template <int V, int LOG_LC, bool kNull, bool kOrdered>
__device__ __forceinline__ void forward_short(const ForwardArgs& a, int64_t segment, int64_t begin, int64_t end,
                                              int64_t base) {
  using S = Geo<V, LOG_LC>;
  constexpr int LC = S::LC, G = S::G, PG = S::PG, RMAX = S::RMAX;
  const Lanes<V, LOG_LC> L(a.channels / V);
  const int64_t column = L.live ? L.column : 0;
  const int64_t degree = end - begin;
  fvec<V> n0;
#pragma unroll
  for (int v = 0; v < V; ++v) n0.v[v] = -INFINITY;
  if constexpr (kNull) n0 = load_vec<V>(a.null_logit + segment * a.channels + column);
  float value[RMAX][V], envelope[RMAX];
  const auto t = forward_tiles<V, RMAX, PG, kOrdered>(a, begin, end, base, L.p, L.live, column, value, envelope);
  // Only the tiles that hold rows of the group are computed (the wave runs
  // the larger count of its groups).
  const int tiles = static_cast<int>((degree + PG - 1) / PG);
  float nv[V], peak[V];
#pragma unroll
  for (int v = 0; v < V; ++v) {
    nv[v] = n0.v[v] * kLog2e;
    peak[v] = -INFINITY;
  }
#pragma unroll
  for (int i = 0; i < RMAX; ++i) {
    if (i < tiles) {
      const float term = row_term(envelope[i]);
#pragma unroll
      for (int v = 0; v < V; ++v) {
        value[i][v] = log2_weight_of_row(value[i][v], term);
        peak[v] = fmaxf(peak[v], value[i][v]);
      }
    }
  }
  float total[V], nw[V], shift[V];
#pragma unroll
  for (int v = 0; v < V; ++v) {
    peak[v] = span_max<LC, G>(peak[v]);
    if (kNull) peak[v] = fmaxf(peak[v], nv[v]);
    shift[v] = shift_of(peak[v]);
    total[v] = 0.0f;
  }
#pragma unroll
  for (int i = 0; i < RMAX; ++i) {
    if (i < tiles) {
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const float w = exp2_of(value[i][v] - shift[v]);
        value[i][v] = w;
        total[v] += w;
      }
    }
  }
#pragma unroll
  for (int v = 0; v < V; ++v) {
    total[v] = span_sum<LC, G>(total[v]);
    nw[v] = kNull ? exp2_of(nv[v] - shift[v]) : 0.0f;
    total[v] = inverse_total(total[v] + nw[v]);
  }
#pragma unroll
  for (int i = 0; i < RMAX; ++i)
    if (i < tiles)
#pragma unroll
      for (int v = 0; v < V; ++v) value[i][v] *= total[v];
  forward_stores<V>(a, t, column, value, tiles);
  if (kNull && L.p == 0 && L.live) {
    fvec<V> out;
#pragma unroll
    for (int v = 0; v < V; ++v) out.v[v] = nw[v] * total[v];
    store_vec<V>(a.null_alpha + segment * a.channels + L.column, out);
  }
}

// Planned: workgroups [0, n_long) take the listed long segments, the others
// SPB consecutive segments each, skipping the long ones.  Unplanned: every
// workgroup takes SPB consecutive segments and runs its own long segments
// after its short ones.
template <int V, int LOG_LC, bool kNull, bool kOrdered, bool kPlanned>
__global__ __launch_bounds__(kBlock) void softmax_forward_kernel(ForwardArgs a, const int64_t* __restrict__ plan,
                                                                 int64_t n_long) {
  using S = Geo<V, LOG_LC>;
  __shared__ float partial[kWaves][2][S::LC * V];
  constexpr bool planned = kPlanned;
  const int64_t block = block_index();
  if (planned && block < n_long) {
    const int64_t segment = plan[kPlanHeader + block];
    if (static_cast<uint64_t>(segment) >= static_cast<uint64_t>(a.n_nodes)) return;
    int64_t begin, end;
    segment_bounds(a.offsets, segment, a.n_edges, begin, end);
    forward_long<V, LOG_LC, kNull, kOrdered>(a, segment, begin, end, partial);
    return;
  }
  const int64_t first = (block - (planned ? n_long : 0)) * S::SPB;
  const int gidx = threadIdx.x >> S::LOG_G;
  const int64_t segment = first + gidx;
  {
    int64_t begin, end;
    group_bounds<S::LOG_G>(a.offsets, first, a.n_nodes, a.n_edges, begin, end);
    // The rows of a wave's short groups (at most two) lie within 2 CAP slots
    // of the lowest short group's begin: one buffer window serves the wave.
    static_assert(S::GPW <= 2, "one row window per wave needs at most two short groups per wave");
    if (segment < a.n_nodes && end - begin <= S::CAP)
      forward_short<V, LOG_LC, kNull, kOrdered>(a, segment, begin, end, uniform_i64(begin));
  }
  if constexpr (planned) return;
  const BlockBounds bb = block_bounds<S::SPB>(a.offsets, first, a.n_nodes, a.n_edges);
  // no plan: this workgroup's long segments, one at a time
  const int lane = threadIdx.x & 63;
  unsigned long long longs =
      __ballot(lane < S::SPB && first + lane < a.n_nodes && bb.hi - bb.lo > S::CAP);
  while (longs != 0ull) {
    const int s = __ffsll(static_cast<long long>(longs)) - 1;
    longs &= longs - 1ull;
    forward_long<V, LOG_LC, kNull, kOrdered>(a, first + s, __shfl(bb.lo, s), __shfl(bb.hi, s), partial);
  }
}

// ---------------------------------------------------------------------------
// backward
// ---------------------------------------------------------------------------

struct BackwardArgs {
  const float* alpha;
  const float* grad_alpha;
  const float* env;
  const int64_t* offsets;
  const float* null_alpha;
  const float* grad_null_alpha;
  const int64_t* order;
  float* grad_logit;
  float* grad_null_logit;
  float* grad_env;
  int64_t n_edges, n_nodes, channels;
};

// Tiles of [first, end) for the backward: alpha, grad_alpha and the envelope
// of every row (zeros without a row), every load issued before any arithmetic.
template <int V, int R, int STEP, bool kOrdered>
__device__ __forceinline__ Tiles<R, STEP, kOrdered> backward_tiles(const BackwardArgs& a, int64_t first, int64_t end,
                                                                   int64_t base, int row_lane, bool live,
                                                                   int64_t column, float (&x)[R][V],
                                                                   float (&g)[R][V], float (&envelope)[R]) {
  Tiles<R, STEP, kOrdered> t(first, end, base, row_lane, live, column, a.channels);
#pragma unroll
  for (int i = 0; i < R; ++i) {
    envelope[i] = 0.0f;
#pragma unroll
    for (int v = 0; v < V; ++v) x[i][v] = g[i][v] = 0.0f;
  }
  if constexpr (!kOrdered) {
    const BufferView alpha = row_view(a.alpha, t.base, a.n_edges, a.channels);
    const BufferView grad = row_view(a.grad_alpha, t.base, a.n_edges, a.channels);
    const BufferView env = row_view(a.env, t.base, a.n_edges, 1);
    // envelopes first: they are consumed last, after the row sums.  The rows
    // are read once and loaded non-temporally (config 2R: 222 -> 200 us).
#pragma unroll
    for (int i = 0; i < R; ++i) envelope[i] = buffer_load_f32(env, t.scalar_at(i));
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const fvec<V> xv = buffer_load_vec<V, kNonTemporal>(alpha, t.at(i));
      const fvec<V> gv = buffer_load_vec<V, kNonTemporal>(grad, t.at(i));
#pragma unroll
      for (int v = 0; v < V; ++v) {
        x[i][v] = xv.v[v];
        g[i][v] = gv.v[v];
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // every load above is issued before any use
  } else {
    t.clear_ids();
    if (a.n_edges > 0) {
      t.gather_ids(a.order, a.n_edges);
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const int64_t e = t.e[i] >= 0 ? t.e[i] : 0;
        const fvec<V> xv = load_vec_stream<V>(a.alpha + e * a.channels + column);
        const fvec<V> gv = load_vec_stream<V>(a.grad_alpha + e * a.channels + column);
        const float env = a.env[e];
        const bool has = t.e[i] >= 0;
        envelope[i] = has ? env : 0.0f;
#pragma unroll
        for (int v = 0; v < V; ++v) {
          x[i][v] = has ? xv.v[v] : 0.0f;
          g[i][v] = has ? gv.v[v] : 0.0f;
        }
      }
    }
  }
  return t;
}

// grad_logit rows of the tiles from alpha, grad_alpha and the segment's S;
// grad_env of each row from the row sum over the LC lanes of the row.
template <int V, int LOG_LC, int R, int STEP, bool kOrdered>
__device__ __forceinline__ void backward_rows(const BackwardArgs& a, const Lanes<V, LOG_LC>& L,
                                              const Tiles<R, STEP, kOrdered>& t, int64_t column,
                                              const float (&x)[R][V], const float (&g)[R][V],
                                              const float (&expect)[V], const float (&envelope)[R],
                                              int tiles = R) {
  // natural order only (unused, and dropped by the compiler, with an order)
  const BufferView grad_logit = row_view(a.grad_logit, t.base, a.n_edges, a.channels);
  const BufferView grad_env = row_view(a.grad_env, t.base, a.n_edges, 1);
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (i >= tiles) continue;  // no row of the lane's group in this tile or later ones
    const bool has = kOrdered ? t.e[i] >= 0 : t.row(i);
    fvec<V> out;
    float row = 0.0f;
#pragma unroll
    for (int v = 0; v < V; ++v) {
      out.v[v] = x[i][v] * (g[i][v] - expect[v]);
      row += out.v[v];
    }
    row = span_sum<1, Geo<V, LOG_LC>::LC>(has ? row : 0.0f);
    const float d_env = env_gradient(row, envelope[i]);
    if constexpr (!kOrdered) {
      buffer_store_vec_stream<V>(grad_logit, t.at(i), out);
      buffer_store_f32(grad_env, L.k == 0 ? t.scalar_at(i) : kNoRow, d_env);
    } else {
      if (has) {
        store_vec_stream<V>(a.grad_logit + t.e[i] * a.channels + column, out);
        if (L.k == 0) a.grad_env[t.e[i]] = d_env;
      }
    }
  }
}

template <int V, int LOG_LC, bool kNull, bool kOrdered>
__device__ void backward_long(const BackwardArgs& a, int64_t segment, int64_t begin, int64_t end,
                              float (*partial)[2][Geo<V, LOG_LC>::LC * V]) {
  using S = Geo<V, LOG_LC>;
  begin = uniform_i64(begin);  // one segment per workgroup
  end = uniform_i64(end);
  constexpr int LC = S::LC, PB = S::PB, RMAXB = S::RMAXB;
  const Lanes<V, LOG_LC> L(a.channels / V);
  const int64_t column = L.live ? L.column : 0;
  const int64_t degree = end - begin;
  float a0[V], g0[V], expect[V];
#pragma unroll
  for (int v = 0; v < V; ++v) a0[v] = g0[v] = expect[v] = 0.0f;
  if constexpr (kNull) {
    const fvec<V> x = load_vec<V>(a.null_alpha + segment * a.channels + column);
    const fvec<V> g = load_vec<V>(a.grad_null_alpha + segment * a.channels + column);
#pragma unroll
    for (int v = 0; v < V; ++v) {
      a0[v] = x.v[v];
      g0[v] = g.v[v];
    }
  }
  if (degree <= RMAXB * PB) {
    // staged: every row of the segment in registers, one read
    float xs[RMAXB][V], gs[RMAXB][V], envs[RMAXB];
    const auto t = backward_tiles<V, RMAXB, PB, kOrdered>(a, begin, end, begin, L.pb, L.live, column, xs, gs, envs);
#pragma unroll
    for (int i = 0; i < RMAXB; ++i)
#pragma unroll
      for (int v = 0; v < V; ++v) expect[v] = expect[v] + xs[i][v] * gs[i][v];
#pragma unroll
    for (int v = 0; v < V; ++v) expect[v] = span_sum<LC, 64>(expect[v]);
    if ((L.lane >> LOG_LC) == 0)
#pragma unroll
      for (int v = 0; v < V; ++v) partial[L.wave][0][L.k * V + v] = expect[v];
    __syncthreads();
#pragma unroll
    for (int v = 0; v < V; ++v) {
      float sum = partial[0][0][L.k * V + v];
      for (int q = 1; q < kWaves; ++q) sum = sum + partial[q][0][L.k * V + v];
      expect[v] = kNull ? sum + a0[v] * g0[v] : sum;
    }
    backward_rows<V, LOG_LC>(a, L, t, column, xs, gs, expect, envs);
  } else {
    // streaming: the dot-product pass (compensated), then the gradient pass
    float carry[V];
#pragma unroll
    for (int v = 0; v < V; ++v) carry[v] = 0.0f;
    for (int64_t base = begin; base < end; base += S::UNROLL * PB) {
      float x[S::UNROLL][V], g[S::UNROLL][V], envs[S::UNROLL];
      backward_tiles<V, S::UNROLL, PB, kOrdered>(a, base, end, base, L.pb, L.live, column, x, g, envs);
#pragma unroll
      for (int u = 0; u < S::UNROLL; ++u)
#pragma unroll
        for (int v = 0; v < V; ++v) compensated_add(expect[v], carry[v], x[u][v] * g[u][v]);
    }
#pragma unroll
    for (int v = 0; v < V; ++v) expect[v] = span_sum<LC, 64>(expect[v] + carry[v]);
    if ((L.lane >> LOG_LC) == 0)
#pragma unroll
      for (int v = 0; v < V; ++v) partial[L.wave][0][L.k * V + v] = expect[v];
    __syncthreads();
#pragma unroll
    for (int v = 0; v < V; ++v) {
      float sum = partial[0][0][L.k * V + v];
      for (int q = 1; q < kWaves; ++q) sum = sum + partial[q][0][L.k * V + v];
      expect[v] = kNull ? sum + a0[v] * g0[v] : sum;
    }
    for (int64_t base = begin; base < end; base += S::UNROLL * PB) {
      float x[S::UNROLL][V], g[S::UNROLL][V], envs[S::UNROLL];
      const auto t = backward_tiles<V, S::UNROLL, PB, kOrdered>(a, base, end, base, L.pb, L.live, column, x, g, envs);
      backward_rows<V, LOG_LC>(a, L, t, column, x, g, expect, envs);
    }
  }
  if (kNull && threadIdx.x < LC && L.live) {
    fvec<V> out;
#pragma unroll
    for (int v = 0; v < V; ++v) out.v[v] = a0[v] * (g0[v] - expect[v]);
    store_vec<V>(a.grad_null_logit + segment * a.channels + L.column, out);
  }
  __syncthreads();
}

template <int V, int LOG_LC, bool kNull, bool kOrdered>
__device__ __forceinline__ void backward_short(const BackwardArgs& a, int64_t segment, int64_t begin, int64_t end,
                                               int64_t base) {
  using S = Geo<V, LOG_LC>;
  constexpr int LC = S::LC, G = S::G, PG = S::PG, RMAX = S::RMAX;
  const Lanes<V, LOG_LC> L(a.channels / V);
  const int64_t column = L.live ? L.column : 0;
  float a0[V], g0[V], expect[V];
#pragma unroll
  for (int v = 0; v < V; ++v) a0[v] = g0[v] = expect[v] = 0.0f;
  if constexpr (kNull) {
    const fvec<V> x = load_vec<V>(a.null_alpha + segment * a.channels + column);
    const fvec<V> g = load_vec<V>(a.grad_null_alpha + segment * a.channels + column);
#pragma unroll
    for (int v = 0; v < V; ++v) {
      a0[v] = x.v[v];
      g0[v] = g.v[v];
    }
  }
  float xs[RMAX][V], gs[RMAX][V], envs[RMAX];
  const auto t = backward_tiles<V, RMAX, PG, kOrdered>(a, begin, end, base, L.p, L.live, column, xs, gs, envs);
  const int tiles = static_cast<int>((end - begin + PG - 1) / PG);
#pragma unroll
  for (int i = 0; i < RMAX; ++i)
    if (i < tiles)
#pragma unroll
      for (int v = 0; v < V; ++v) expect[v] = expect[v] + xs[i][v] * gs[i][v];
#pragma unroll
  for (int v = 0; v < V; ++v) {
    expect[v] = span_sum<LC, G>(expect[v]);
    if (kNull) expect[v] = expect[v] + a0[v] * g0[v];
  }
  backward_rows<V, LOG_LC>(a, L, t, column, xs, gs, expect, envs, tiles);
  if (kNull && L.p == 0 && L.live) {
    fvec<V> out;
#pragma unroll
    for (int v = 0; v < V; ++v) out.v[v] = a0[v] * (g0[v] - expect[v]);
    store_vec<V>(a.grad_null_logit + segment * a.channels + L.column, out);
  }
}

template <int V, int LOG_LC, bool kNull, bool kOrdered, bool kPlanned>
__global__ __launch_bounds__(kBlock) void softmax_backward_kernel(BackwardArgs a, const int64_t* __restrict__ plan,
                                                                  int64_t n_long) {
  using S = Geo<V, LOG_LC>;
  __shared__ float partial[kWaves][2][S::LC * V];
  constexpr bool planned = kPlanned;
  const int64_t block = block_index();
  if (planned && block < n_long) {
    const int64_t segment = plan[kPlanHeader + block];
    if (static_cast<uint64_t>(segment) >= static_cast<uint64_t>(a.n_nodes)) return;
    int64_t begin, end;
    segment_bounds(a.offsets, segment, a.n_edges, begin, end);
    backward_long<V, LOG_LC, kNull, kOrdered>(a, segment, begin, end, partial);
    return;
  }
  const int64_t first = (block - (planned ? n_long : 0)) * S::SPB;
  const int gidx = threadIdx.x >> S::LOG_G;
  const int64_t segment = first + gidx;
  {
    int64_t begin, end;
    group_bounds<S::LOG_G>(a.offsets, first, a.n_nodes, a.n_edges, begin, end);
    // The rows of a wave's short groups (at most two) lie within 2 CAP slots
    // of the lowest short group's begin: one buffer window serves the wave.
    static_assert(S::GPW <= 2, "one row window per wave needs at most two short groups per wave");
    if (segment < a.n_nodes && end - begin <= S::CAP)
      backward_short<V, LOG_LC, kNull, kOrdered>(a, segment, begin, end, uniform_i64(begin));
  }
  if constexpr (planned) return;
  const BlockBounds bb = block_bounds<S::SPB>(a.offsets, first, a.n_nodes, a.n_edges);
  const int lane = threadIdx.x & 63;
  unsigned long long longs =
      __ballot(lane < S::SPB && first + lane < a.n_nodes && bb.hi - bb.lo > S::CAP);
  while (longs != 0ull) {
    const int s = __ffsll(static_cast<long long>(longs)) - 1;
    longs &= longs - 1ull;
    backward_long<V, LOG_LC, kNull, kOrdered>(a, first + s, __shfl(bb.lo, s), __shfl(bb.hi, s), partial);
  }
}

// ---------------------------------------------------------------------------
// rows of more than two chunks: a wave per (segment, slab of columns)
// ---------------------------------------------------------------------------
//
// Columns are independent in the forward, and in the backward until the row
// sums of grad_env.  So a row is cut into slabs of LS chunks (LS = 2, 4 or 8:
// 8 chunks are one 128-byte line), and one wave takes one slab of one
// segment: 64 / LS rows per load, up to R loads, all issued before any
// arithmetic.  A segment of up to CAP = R * 64 / LS rows is then read once,
// whatever its width, where a workgroup that stages whole rows in registers
// holds 16 rows at C = 256 and reads everything longer twice.  R follows the
// graph's mean degree (slab_rows).  Longer segments are streamed by the same
// wave: an online max/sum pass, then the write pass.  The sums over the rows
// are kept in 64 bits: they are few instructions beside the row streams, and
// alpha and the gradients come out closer to the exact values for it.
//
// The forward has no barrier.  In the backward, up to 8 waves of a workgroup
// take the slabs of one segment and leave each row's partial sum in LDS; after
// one barrier thread t adds those of row t in slab order and writes grad_env.
// Rows of more than 8 slabs repeat this, grad_env keeping the raw sum until
// the last round (thread t reads back only what it wrote itself).
//
// Any C >= 4 and any 4-byte alignment: the row's last chunk starts at column
// C - 4, so it repeats up to three columns of its neighbour, which compute and
// store the same bits in both lanes and are left out of the row sums (`skip`).
// Where outputs lie on inputs, both lanes must be of one wave, which loads a
// row before it stores it: a row whose last chunk would be alone in its slab is
// then cut `shift` chunks earlier (slab_shift).
//
// Bound by the row streams: C = 256 over 741k edges of 8,192 segments takes
// 274 us forward (5.6 TB/s) and 380 us backward (6.0), where staging whole rows
// took 426 and 700 us; C = 128, 991k edges 419 against 707 us for both; C = 64,
// 182k edges 49 against 61 us; C = 16, 1.48M edges 88 against 109 us.  Scattered
// rows (through an order): C = 128 545 against 819 us, C = 16 unchanged
// (208 us, bound by the 64-byte gathers).  A streamed round takes its maximum
// first: an online update per value kept a wave of 512 rows busy for 53 us,
// this form for 25 us.  Errors against 64 bits (C = 16 to 256, degree 70 with
// hubs): alpha 1.1e-7 -> 7e-8, grad_logit 2.8-3.3e-7 -> 1.1e-7.

constexpr int kSlabWaves = 8;  // most slabs of one segment side by side in a backward workgroup

// How a wave finds its rows: natural order through buffer views, or edge ids
// (from `order`, or the slot itself) and 64-bit addresses, the ids kept in 32
// bits where they fit.  Rows are read and written once and go non-temporally,
// except the first reading of a segment that is streamed (kKeep; C = 32, segments of
// 90 rows among twice as many empty ones: 56 -> 46 us), and (SharedViews) where slabs of 128 bytes do not fall on cache lines, so
// that two waves share most lines: there the default policy keeps a line until
// its other half comes (C = 191, 991k edges: 1,364 -> 961 us; C = 256 the
// other way round: 659 against 726 us).
struct Views {};
struct SharedViews {};
template <typename Id>
constexpr bool kUsesViews = __is_same(Id, Views) || __is_same(Id, SharedViews);
template <typename Id>
constexpr int kRowPolicy = __is_same(Id, SharedViews) ? 0 : kNonTemporal;

// Rows [first, first + CAP) of a segment that ends at `end`, as R tiles of PR
// rows; lane (p, k) holds row i * PR + p, columns [column, column + 4).  The
// views end with the rows, so a tile's offset is the lane's own plus a
// multiple of i, with no test per tile; a lane without a column starts past
// the end (2^31) and stays there (CAP rows are under 2^30 bytes).
template <int LOG_LS, int R, typename Id>
struct SlabRows {
  static constexpr int LS = 1 << LOG_LS;
  static constexpr int PR = 64 >> LOG_LS;
  static constexpr int CAP = R * PR;
  int64_t first;   // wave-uniform
  int rows, p;     // rows below `end`, at most CAP
  bool live;
  uint32_t row_bytes, lane_at;
  Id id[kUsesViews<Id> ? 1 : R];

  __device__ __forceinline__ SlabRows(int64_t first_, int64_t end, bool live_, int64_t column, int64_t channels)
      : first(first_), live(live_) {
    const int64_t left = end - first_;
    rows = static_cast<int>(left < CAP ? left : CAP);
    p = static_cast<int>(threadIdx.x & 63) >> LOG_LS;
    row_bytes = static_cast<uint32_t>(channels) * 4u;
    lane_at = live ? static_cast<uint32_t>(p) * row_bytes + static_cast<uint32_t>(column) * 4u : kNoRow;
  }
  __device__ __forceinline__ bool row(int i) const { return live & (i * PR + p < rows); }
  __device__ __forceinline__ uint32_t at(int i) const { return lane_at + static_cast<uint32_t>(i * PR) * row_bytes; }
  __device__ __forceinline__ uint32_t scalar_at(int i) const { return static_cast<uint32_t>(p + i * PR) * 4u; }
  // These rows of a row-major [n_edges, channels] array.
  __device__ __forceinline__ BufferView view(const float* base, int64_t channels) const {
    return buffer_view(base + first * channels, static_cast<int64_t>(rows) * channels * 4);
  }
  // Ids of every tile; a lane without a row (or with an order entry out of
  // range) keeps kNone and reads edge `first` instead.
  static constexpr uint64_t kNone = ~uint64_t(0);
  __device__ __forceinline__ void find(const int64_t* __restrict__ order, int64_t n_edges) {
    if constexpr (!kUsesViews<Id>) {
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const int64_t slot = first + (row(i) ? i * PR + p : 0);
        const int64_t e = order != nullptr ? order[slot] : slot;
        id[i] = row(i) && static_cast<uint64_t>(e) < static_cast<uint64_t>(n_edges) ? static_cast<Id>(e)
                                                                                     : static_cast<Id>(kNone);
      }
    }
  }
  __device__ __forceinline__ bool has(int i) const {
    if constexpr (kUsesViews<Id>) return row(i);
    else return id[i] != static_cast<Id>(kNone);
  }
  __device__ __forceinline__ int64_t edge(int i) const {  // a valid edge also where there is no row
    if constexpr (kUsesViews<Id>) return first + i * PR + p;
    else return has(i) ? static_cast<int64_t>(id[i]) : first;
  }
};

// The logit chunks and envelopes of every tile, all loads issued before any use.
template <int LOG_LS, int R, bool kKeep = false, typename Id>
__device__ __forceinline__ void slab_forward_loads(const ForwardArgs& a, SlabRows<LOG_LS, R, Id>& t, int64_t column,
                                                   float (&value)[R][4], float (&envelope)[R]) {
  t.find(a.order, a.n_edges);
  if constexpr (kUsesViews<Id>) {
    const BufferView logit = t.view(a.logit, a.channels);
    const BufferView env = t.view(a.env, 1);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const fvec<4> x = buffer_load_vec<4, kKeep ? 0 : kRowPolicy<Id>>(logit, t.at(i));
      envelope[i] = buffer_load_f32(env, t.scalar_at(i));
#pragma unroll
      for (int v = 0; v < 4; ++v) value[i][v] = x.v[v];
    }
  } else {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int64_t e = t.edge(i);
      const float* row = a.logit + e * a.channels + column;
      const fvec<4> x = kKeep ? load_chunk(row) : load_chunk_stream(row);
      envelope[i] = a.env[e];
#pragma unroll
      for (int v = 0; v < 4; ++v) value[i][v] = x.v[v];
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (!kUsesViews<Id>)
#pragma unroll
    for (int i = 0; i < R; ++i) envelope[i] = t.has(i) ? envelope[i] : 0.0f;
}

// 1 / D rounded once (a Newton step on v_rcp_f32 in 64 bits), with D = 1 for a
// segment without mass.
__device__ __forceinline__ float inverse_of(double total) {
  const double d = total > 0.0 ? total : 1.0;
  const double r = static_cast<double>(__builtin_amdgcn_rcpf(static_cast<float>(d)));
  return static_cast<float>(__builtin_fma(r, __builtin_fma(-d, r, 1.0), r));
}

template <int LOG_LS, int R, typename Id>
__device__ __forceinline__ void slab_forward_stores(const ForwardArgs& a, const SlabRows<LOG_LS, R, Id>& t,
                                                    int64_t column, const float (&alpha)[R][4], int tiles) {
  const BufferView out = t.view(a.alpha, a.channels);
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (i >= tiles) continue;
    const fvec<4> row{{alpha[i][0], alpha[i][1], alpha[i][2], alpha[i][3]}};
    if constexpr (kUsesViews<Id>) buffer_store_chunk<kRowPolicy<Id>>(out, t.at(i), row);
    else if (t.has(i)) store_chunk_stream(a.alpha + t.edge(i) * a.channels + column, row);
  }
}

template <int LOG_LS, int R, typename Id>
__global__ __launch_bounds__(kBlock) void softmax_forward_slab_kernel(ForwardArgs a, int64_t slabs, int shift) {
  using T = SlabRows<LOG_LS, R, Id>;
  constexpr int LS = T::LS, PR = T::PR, CAP = T::CAP;
  const int64_t unit = uniform_i64(block_index() * kWaves + (threadIdx.x >> 6));
  const int64_t segment = unit / slabs;
  if (segment >= a.n_nodes) return;
  const int64_t slab = unit - segment * slabs;
  const int lane = threadIdx.x & 63;
  const int64_t chunk = slab * LS + (lane & (LS - 1)) - shift;
  const bool live = chunk >= 0 && chunk * 4 < a.channels;
  const int64_t column = live ? (chunk * 4 + 4 <= a.channels ? chunk * 4 : a.channels - 4) : 0;
  const bool has_null = a.null_logit != nullptr;
  int64_t begin, end;
  segment_bounds(a.offsets, segment, a.n_edges, begin, end);
  float nv[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) nv[v] = -INFINITY;
  if (has_null) {
    const fvec<4> n0 = load_chunk(a.null_logit + segment * a.channels + column);
#pragma unroll
    for (int v = 0; v < 4; ++v) nv[v] = n0.v[v] * kLog2e;
  }
  float total[4], nw[4];
  if (end - begin <= CAP) {
    T t(begin, end, live, column, a.channels);
    float value[R][4], envelope[R];
    if (begin < end) slab_forward_loads(a, t, column, value, envelope);
    const int tiles = (t.rows + PR - 1) / PR;
    float peak[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) peak[v] = -INFINITY;
#pragma unroll
    for (int i = 0; i < R; ++i)
      if (i < tiles) {
        const float term = row_term(envelope[i]);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          value[i][v] = log2_weight_of_row(value[i][v], term);
          peak[v] = fmaxf(peak[v], value[i][v]);
        }
      }
    float shift[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      peak[v] = fmaxf(span_max<LS, 64>(peak[v]), nv[v]);
      shift[v] = shift_of(peak[v]);
    }
    double sum[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < R; ++i)
      if (i < tiles)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          value[i][v] = exp2_of(value[i][v] - shift[v]);
          sum[v] += static_cast<double>(value[i][v]);
        }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      nw[v] = exp2_of(nv[v] - shift[v]);
      total[v] = inverse_of(span_sum<LS, 64>(sum[v]) + static_cast<double>(nw[v]));
    }
#pragma unroll
    for (int i = 0; i < R; ++i)
      if (i < tiles)
#pragma unroll
        for (int v = 0; v < 4; ++v) value[i][v] *= total[v];
    if (begin < end) slab_forward_stores(a, t, column, value, tiles);
  } else {
    float peak[4];
    double sum[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int v = 0; v < 4; ++v) peak[v] = -INFINITY;
    for (int64_t base = begin; base < end; base += CAP) {
      T t(base, end, live, column, a.channels);
      float value[R][4], envelope[R];
      slab_forward_loads<LOG_LS, R, true>(a, t, column, value, envelope);
      // a round's maximum first, then one rescale and the round's terms
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const float term = row_term(envelope[i]);
#pragma unroll
        for (int v = 0; v < 4; ++v) value[i][v] = log2_weight_of_row(value[i][v], term);
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float top = peak[v];
#pragma unroll
        for (int i = 0; i < R; ++i) top = fmaxf(top, value[i][v]);
        const float shift = shift_of(top);
        sum[v] *= static_cast<double>(exp2_of(peak[v] - shift));  // by 0 while the column has no mass
#pragma unroll
        for (int i = 0; i < R; ++i) sum[v] += static_cast<double>(exp2_of(value[i][v] - shift));
        peak[v] = top;
      }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float top = fmaxf(span_max<LS, 64>(peak[v]), nv[v]);
      const float shift = shift_of(top);
      const double part = sum[v] * static_cast<double>(exp2_of(peak[v] - shift));
      peak[v] = shift;
      nw[v] = exp2_of(nv[v] - shift);
      total[v] = inverse_of(span_sum<LS, 64>(part) + static_cast<double>(nw[v]));
    }
    for (int64_t base = begin; base < end; base += CAP) {
      T t(base, end, live, column, a.channels);
      float value[R][4], envelope[R];
      slab_forward_loads(a, t, column, value, envelope);
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const float term = row_term(envelope[i]);
#pragma unroll
        for (int v = 0; v < 4; ++v)
          value[i][v] = exp2_of(log2_weight_of_row(value[i][v], term) - peak[v]) * total[v];
      }
      slab_forward_stores(a, t, column, value, R);
    }
  }
  if (has_null && live && lane < LS)
    store_chunk(a.null_alpha + segment * a.channels + column,
                fvec<4>{{nw[0] * total[0], nw[1] * total[1], nw[2] * total[2], nw[3] * total[3]}});
}

// alpha and grad_alpha chunks of every tile (zeros without a row).
template <int LOG_LS, int R, bool kKeep = false, typename Id>
__device__ __forceinline__ void slab_backward_loads(const BackwardArgs& a, SlabRows<LOG_LS, R, Id>& t,
                                                    int64_t column, float (&x)[R][4], float (&g)[R][4]) {
  t.find(a.order, a.n_edges);
  if constexpr (kUsesViews<Id>) {
    const BufferView alpha = t.view(a.alpha, a.channels);
    const BufferView grad = t.view(a.grad_alpha, a.channels);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const fvec<4> xv = buffer_load_vec<4, kKeep ? 0 : kRowPolicy<Id>>(alpha, t.at(i));
      const fvec<4> gv = buffer_load_vec<4, kKeep ? 0 : kRowPolicy<Id>>(grad, t.at(i));
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        x[i][v] = xv.v[v];
        g[i][v] = gv.v[v];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  } else {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int64_t e = t.edge(i);
      const float *alpha = a.alpha + e * a.channels + column, *grad = a.grad_alpha + e * a.channels + column;
      const fvec<4> xv = kKeep ? load_chunk(alpha) : load_chunk_stream(alpha);
      const fvec<4> gv = kKeep ? load_chunk(grad) : load_chunk_stream(grad);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        x[i][v] = xv.v[v];
        g[i][v] = gv.v[v];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        x[i][v] = t.has(i) ? x[i][v] : 0.0f;
        g[i][v] = t.has(i) ? g[i][v] : 0.0f;
      }
  }
}

// SW waves share a segment (SW > 1), or every wave has a segment of its own
// (SW = 1, rows of one slab).
template <int LOG_LS, int R, int SW, typename Id>
__global__ __launch_bounds__(SW == 1 ? kBlock : SW * 64) void softmax_backward_slab_kernel(
    BackwardArgs a, int64_t slabs, int shift) {
  using T = SlabRows<LOG_LS, R, Id>;
  constexpr int LS = T::LS, PR = T::PR, CAP = T::CAP;
  constexpr int kSegments = SW == 1 ? kWaves : 1;  // segments per workgroup
  __shared__ float row_sum[kSegments][CAP][SW];
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int64_t segment = block_index() * kSegments + (SW == 1 ? wave : 0);
  if (segment >= a.n_nodes) return;  // the whole workgroup, or a wave that shares nothing
  auto& sums = row_sum[SW == 1 ? wave : 0];
  const int part = SW == 1 ? 0 : wave;
  const int lane = threadIdx.x & 63;
  const int member = SW == 1 ? lane : static_cast<int>(threadIdx.x);  // among the SW * 64 threads of the segment
  const bool has_null = a.null_alpha != nullptr;
  int64_t begin, end;
  segment_bounds(a.offsets, segment, a.n_edges, begin, end);

  for (int64_t round = 0; round < slabs; round += SW) {
    const int64_t chunk = (round + part) * LS + (lane & (LS - 1)) - shift;
    const bool live = chunk >= 0 && chunk * 4 < a.channels;
    const int64_t column = live ? (chunk * 4 + 4 <= a.channels ? chunk * 4 : a.channels - 4) : 0;
    const int skip = live ? static_cast<int>(chunk * 4 - column) : 4;  // columns a neighbour accounts for
    const bool last = round + SW >= slabs;
    float a0[4], g0[4], expect[4], rest[4];  // S = expect + rest
    double dot[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int v = 0; v < 4; ++v) a0[v] = g0[v] = 0.0f;
    // S of each column from the lanes' partial dot products
    const auto split = [&]() {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const double total = __builtin_fma(static_cast<double>(a0[v]), static_cast<double>(g0[v]),
                                           span_sum<LS, 64>(dot[v]));
        expect[v] = static_cast<float>(total);
        // no remainder of an infinite S, whose gradients stay infinities
        rest[v] = __builtin_isfinite(expect[v]) ? static_cast<float>(total - static_cast<double>(expect[v])) : 0.0f;
      }
    };
    const auto add_products = [&](const float(&xs)[R][4], const float(&gs)[R][4], int tiles) {
#pragma unroll
      for (int i = 0; i < R; ++i)
        if (i < tiles)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            dot[v] = __builtin_fma(static_cast<double>(xs[i][v]), static_cast<double>(gs[i][v]), dot[v]);
    };
    if (has_null) {
      const fvec<4> xv = load_chunk(a.null_alpha + segment * a.channels + column);
      const fvec<4> gv = load_chunk(a.grad_null_alpha + segment * a.channels + column);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        a0[v] = xv.v[v];
        g0[v] = gv.v[v];
      }
    }
    float x[R][4], g[R][4];
    // edge and envelope of the rows this thread finishes, loaded ahead of the rows
    constexpr int kOwn = (CAP + SW * 64 - 1) / (SW * 64);
    int64_t own_edge[kOwn];
    float own_env[kOwn];
    const auto own_rows = [&](const T& t) {
#pragma unroll
      for (int q = 0; q < kOwn; ++q) {
        const int r = member + q * SW * 64;
        const int64_t slot = t.first + (r < t.rows ? r : 0);
        const int64_t e = a.order != nullptr ? a.order[slot] : slot;
        const bool ok = r < t.rows && static_cast<uint64_t>(e) < static_cast<uint64_t>(a.n_edges);
        own_edge[q] = ok ? e : -1;
        own_env[q] = a.env[ok ? e : t.first];
      }
    };
    const auto finish = [&](const T& t) {
      const BufferView out_view = t.view(a.grad_logit, a.channels);
#pragma unroll
      for (int i = 0; i < R; ++i) {
        if (i * PR >= t.rows) continue;  // wave-uniform
        fvec<4> out;
        float row = 0.0f;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          out.v[v] = x[i][v] * ((g[i][v] - expect[v]) - rest[v]);
          row += v >= skip ? out.v[v] : 0.0f;
        }
        row = span_sum<1, LS>(row);
        if constexpr (kUsesViews<Id>) buffer_store_chunk<kRowPolicy<Id>>(out_view, t.at(i), out);
        else if (t.has(i) && live) store_chunk_stream(a.grad_logit + t.edge(i) * a.channels + column, out);
        if ((lane & (LS - 1)) == 0) sums[i * PR + t.p][part] = row;
      }
      if constexpr (SW > 1) __syncthreads();
      else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int q = 0; q < kOwn; ++q) {
        if (own_edge[q] < 0) continue;
        float sum = round > 0 ? a.grad_env[own_edge[q]] : 0.0f;
#pragma unroll
        for (int w = 0; w < SW; ++w) sum += sums[member + q * SW * 64][w];
        a.grad_env[own_edge[q]] = last ? env_gradient(sum, own_env[q]) : sum;
      }
    };
    if (end - begin <= CAP) {
      if (begin < end) {
        T t(begin, end, live, column, a.channels);
        own_rows(t);
        slab_backward_loads(a, t, column, x, g);
        add_products(x, g, (t.rows + PR - 1) / PR);
        split();
        finish(t);
      } else {
        split();
      }
    } else {
      for (int64_t base = begin; base < end; base += CAP) {
        T t(base, end, live, column, a.channels);
        slab_backward_loads<LOG_LS, R, true>(a, t, column, x, g);
        add_products(x, g, R);
      }
      split();
      for (int64_t base = begin; base < end; base += CAP) {
        T t(base, end, live, column, a.channels);
        own_rows(t);
        slab_backward_loads(a, t, column, x, g);
        finish(t);
        if constexpr (SW > 1) __syncthreads();  // the row sums are read before the next rows overwrite them
        else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
    }
    if (has_null && live && lane < LS)
      store_chunk(a.grad_null_logit + segment * a.channels + column,
                  fvec<4>{{a0[0] * ((g0[0] - expect[0]) - rest[0]), a0[1] * ((g0[1] - expect[1]) - rest[1]),
                           a0[2] * ((g0[2] - expect[2]) - rest[2]), a0[3] * ((g0[3] - expect[3]) - rest[3])}});
    if constexpr (SW > 1) {
      if (!last) __syncthreads();
    }
  }
}

// ---------------------------------------------------------------------------
// plan: ascending list of the segments longer than the short-path capacity
// ---------------------------------------------------------------------------

constexpr int kPlanThreads = 256;
constexpr int kPlanItems = 16;
constexpr int64_t kPlanTile = kPlanThreads * kPlanItems;

__device__ __forceinline__ bool is_long(const int64_t* __restrict__ offsets, int64_t segment, int64_t n_edges,
                                        int64_t capacity) {
  int64_t begin, end;
  segment_bounds(offsets, segment, n_edges, begin, end);
  return end - begin > capacity;
}

__device__ int64_t plan_block_scan(int64_t value, int64_t* lds) {
  const int t = threadIdx.x;
  lds[t] = value;
  __syncthreads();
  for (int offset = 1; offset < kPlanThreads; offset <<= 1) {
    const int64_t add = t >= offset ? lds[t - offset] : 0;
    __syncthreads();
    lds[t] += add;
    __syncthreads();
  }
  const int64_t result = lds[t];
  __syncthreads();
  return result;
}

__global__ __launch_bounds__(kPlanThreads) void plan_count_kernel(const int64_t* __restrict__ offsets,
                                                                  int64_t n_nodes, int64_t n_edges,
                                                                  int64_t capacity, int64_t* __restrict__ counts) {
  __shared__ int64_t lds[kPlanThreads];
  const int64_t tile = block_index();
  if (tile * kPlanTile >= n_nodes) return;
  const int64_t base = tile * kPlanTile + static_cast<int64_t>(threadIdx.x) * kPlanItems;
  int64_t count = 0;
  for (int i = 0; i < kPlanItems; ++i)
    if (base + i < n_nodes && is_long(offsets, base + i, n_edges, capacity)) ++count;
  const int64_t inclusive = plan_block_scan(count, lds);
  if (threadIdx.x == kPlanThreads - 1) counts[tile] = inclusive;
}

// Exclusive scan of the tile counts in place (one workgroup); writes the
// header of the plan.
__global__ __launch_bounds__(kPlanThreads) void plan_scan_kernel(int64_t* __restrict__ counts, int64_t tiles,
                                                                 int64_t capacity, int64_t* __restrict__ plan) {
  __shared__ int64_t lds[kPlanThreads];
  const int64_t per_thread = (tiles + kPlanThreads - 1) / kPlanThreads;
  const int64_t begin = static_cast<int64_t>(threadIdx.x) * per_thread;
  const int64_t end = begin + per_thread < tiles ? begin + per_thread : tiles;
  int64_t sum = 0;
  for (int64_t i = begin; i < end; ++i) sum += counts[i];
  const int64_t inclusive = plan_block_scan(sum, lds);
  int64_t running = inclusive - sum;
  for (int64_t i = begin; i < end; ++i) {
    const int64_t value = counts[i];
    counts[i] = running;
    running += value;
  }
  if (threadIdx.x == kPlanThreads - 1) {
    plan[0] = capacity;
    plan[1] = inclusive;
  }
}

__global__ __launch_bounds__(kPlanThreads) void plan_write_kernel(const int64_t* __restrict__ offsets,
                                                                  int64_t n_nodes, int64_t n_edges,
                                                                  int64_t capacity,
                                                                  const int64_t* __restrict__ tile_prefix,
                                                                  int64_t* __restrict__ list) {
  __shared__ int64_t lds[kPlanThreads];
  const int64_t tile = block_index();
  if (tile * kPlanTile >= n_nodes) return;
  const int64_t base = tile * kPlanTile + static_cast<int64_t>(threadIdx.x) * kPlanItems;
  bool flag[kPlanItems];
  int64_t count = 0;
#pragma unroll
  for (int i = 0; i < kPlanItems; ++i) {
    flag[i] = base + i < n_nodes && is_long(offsets, base + i, n_edges, capacity);
    count += flag[i] ? 1 : 0;
  }
  const int64_t inclusive = plan_block_scan(count, lds);
  int64_t position = tile_prefix[tile] + inclusive - count;
#pragma unroll
  for (int i = 0; i < kPlanItems; ++i)
    if (flag[i]) list[position++] = base + i;
}

int64_t plan_tiles(int64_t n_nodes) { return (n_nodes + kPlanTile - 1) / kPlanTile; }

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

int lanes_log_for(int64_t chunks) {
  int log = 0;
  while ((int64_t(1) << log) < chunks) ++log;
  return log;
}

// Mean degree of a graph with at least one segment.
double mean_degree(int64_t n_edges, int64_t n_nodes) {
  return static_cast<double>(n_edges) / static_cast<double>(n_nodes);
}

// Whether the slab kernels run these rows.  Aligned rows of two chunks (C = 8) and rows of up to four
// columns run the lane-group kernels, rows past 256 columns and rows that are not whole aligned chunks the slab kernels.
// Between, the lane groups take the mean degrees at which slabs are mostly empty or re-read their segments.  Lane
// groups against slabs, forward / backward, 96 MB of logits, us:
//   C = 16   degree 8 54 / 78 and 70 / 115, 12 44 / 61 and 70 / 92, 20 35 / 50 and 50 / 64 (gathered 81 / 129 and 81 / 129),
//            60 66 / 84 and 36 / 54, 90 47 / 63 and 35 / 52, 150 36 / 50 and 43 / 60, 200 35 / 48 and 44 / 65
//   C = 32   8 35 / 52 and 60 / 100, 12 35 / 49 and 44 / 70, 20 43 / 59 and 35 / 52, 30 61 / 79 and 38 / 53, 60 36 / 53 and
//            34 / 53, 90 34 / 47 and 37 / 53, 150 52 / 78 and 42 / 62, 300 55 / 81 and 47 / 73
//   C = 128  5 53 / 67 and 83 / 138, 12 52 / 62 and 44 / 68, 16 41 / 53 and 37 / 56, 30 46 / 63 and 37 / 53, 90 60 / 84 and
//            37 / 52, 200 62 / 86 and 40 / 68
// 64 segments of 12,000 rows and more take twice as long as slabs up to 32 columns, and half as long past that.  At
// degrees of 20 to 100 the sums stay in 64 bits also where lane groups, whose sums have 32, would be up to 1.4 times as
// fast (C = 16, degree 20).
bool uses_slabs(int64_t channels, bool vec4, int64_t n_edges, int64_t n_nodes) {
  if (channels <= 4 || (vec4 && channels == 8)) return false;
  if (!vec4 || channels > 256) return true;
  const double degree = mean_degree(n_edges, n_nodes);
  if (channels <= 16) return degree >= 20.0 && degree <= 112.0;
  if (channels <= 32) return degree >= 18.0 && (degree <= 130.0 || (degree <= 1000.0 && n_nodes >= 1024));
  return degree >= 14.0;
}

// Short-path capacity of the lane-group kernel that runs `channels` with
// (vec4) or without 128-bit rows; 0 for the slab kernels (no plan use).
int64_t capacity_for(int64_t channels, bool vec4, int64_t n_edges, int64_t n_nodes) {
  if (uses_slabs(channels, vec4, n_edges, n_nodes)) return 0;
  return short_capacity(vec4 ? 4 : 1, 1 << lanes_log_for(vec4 ? channels / 4 : channels));
}

int64_t short_blocks(int64_t n_nodes, int log_lc) {
  const int64_t per_block = kBlock >> short_group_log(log_lc);
  return (n_nodes + per_block - 1) / per_block;
}

template <int V, int LOG_LC>
int launch_forward(const ForwardArgs& a, const int64_t* plan, int64_t n_long, hipStream_t stream) {
  const dim3 grid = launch_grid((plan != nullptr ? n_long : 0) + short_blocks(a.n_nodes, LOG_LC), kBlock);
#define DPA4K_SOFTMAX_FWD(NULLV, ORD)                                                                      \
  (plan != nullptr                                                                                        \
       ? softmax_forward_kernel<V, LOG_LC, NULLV, ORD, true>                                               \
       : softmax_forward_kernel<V, LOG_LC, NULLV, ORD, false>)<<<grid, kBlock, 0, \
                                                                 stream>>>(a, plan, n_long)
  if (a.null_logit != nullptr) {
    if (a.order != nullptr) DPA4K_SOFTMAX_FWD(true, true); else DPA4K_SOFTMAX_FWD(true, false);
  } else {
    if (a.order != nullptr) DPA4K_SOFTMAX_FWD(false, true); else DPA4K_SOFTMAX_FWD(false, false);
  }
#undef DPA4K_SOFTMAX_FWD
  return launched("softmax_forward_kernel");
}

template <int V, int LOG_LC>
int launch_backward(const BackwardArgs& a, const int64_t* plan, int64_t n_long, hipStream_t stream) {
  const dim3 grid = launch_grid((plan != nullptr ? n_long : 0) + short_blocks(a.n_nodes, LOG_LC), kBlock);
#define DPA4K_SOFTMAX_BWD(NULLV, ORD)                                                                       \
  (plan != nullptr                                                                                         \
       ? softmax_backward_kernel<V, LOG_LC, NULLV, ORD, true>                                               \
       : softmax_backward_kernel<V, LOG_LC, NULLV, ORD, false>)<<<grid, kBlock, 0, \
                                                                  stream>>>(a, plan, n_long)
  if (a.null_alpha != nullptr) {
    if (a.order != nullptr) DPA4K_SOFTMAX_BWD(true, true); else DPA4K_SOFTMAX_BWD(true, false);
  } else {
    if (a.order != nullptr) DPA4K_SOFTMAX_BWD(false, true); else DPA4K_SOFTMAX_BWD(false, false);
  }
#undef DPA4K_SOFTMAX_BWD
  return launched("softmax_backward_kernel");
}

// Rows a slab wave holds in registers: the mean degree and 3.5 of its standard
// deviations (Poisson), or nearly, so that only outliers are streamed.  Every
// tile costs instructions also where it holds no rows (C = 64, degree 16: 37 /
// 56 us with 32 rows, 54 / 74 with 64), so the rows are not more than needed.  Slabs of four chunks have
// registers for 256 rows (C = 13, degree 200 through an order), of two for 512;
// slabs of four take 128 from a degree of 48 on (C = 16, two populations of
// degree 20 and 100 through an order: 110 / 171 us with 96, 83 / 130 with 128).
int slab_rows(int64_t n_edges, int64_t n_nodes, int log_ls) {
  const double mean = mean_degree(n_edges, n_nodes);
  const double rows = mean + 3.5 * sqrt(mean);
  if (rows <= 40.0) return 32;
  if (rows <= 72.0) return 64;
  if (rows <= 100.0 && log_ls >= 2) return log_ls == 2 ? 128 : 96;
  if (rows <= 140.0 || log_ls == 3) return 128;
  return rows <= 300.0 || log_ls == 2 ? 256 : 512;
}

// Natural order through 32-bit view offsets, edge ids in 32 bits, or in 64.
enum class RowIds { kViews, kSharedViews, kNarrow, kWide };
RowIds row_ids(const int64_t* order, int64_t n_edges, int64_t channels) {
  if (channels > (int64_t(1) << 20)) return RowIds::kWide;  // 128 rows stay within 2^30 bytes
  if (order == nullptr) return channels % 32 == 0 || channels < 32 ? RowIds::kViews : RowIds::kSharedViews;
  return n_edges < 0xffffffffLL ? RowIds::kNarrow : RowIds::kWide;
}

int slab_lanes_log(int64_t channels) { return channels <= 8 ? 1 : (channels <= 16 ? 2 : 3); }

template <int LOG_LS, typename Id>
int launch_forward_slabs(const ForwardArgs& a, int rows, int64_t slabs, int shift, hipStream_t stream) {
  constexpr int PR = 64 >> LOG_LS;
  const dim3 grid = launch_grid((a.n_nodes * slabs + kWaves - 1) / kWaves, kBlock);
  if constexpr (!__is_same(Id, int64_t)) {
    if (rows == 32) softmax_forward_slab_kernel<LOG_LS, 32 / PR, Id><<<grid, kBlock, 0, stream>>>(a, slabs, shift);
    if (rows == 64) softmax_forward_slab_kernel<LOG_LS, 64 / PR, Id><<<grid, kBlock, 0, stream>>>(a, slabs, shift);
    if constexpr (LOG_LS == 3)
      if (rows == 96) softmax_forward_slab_kernel<LOG_LS, 96 / PR, Id><<<grid, kBlock, 0, stream>>>(a, slabs, shift);
    if constexpr (LOG_LS == 1)
      if (rows == 512) softmax_forward_slab_kernel<LOG_LS, 512 / PR, Id><<<grid, kBlock, 0, stream>>>(a, slabs, shift);
    if constexpr (LOG_LS < 3)
      if (rows == 256) softmax_forward_slab_kernel<LOG_LS, 256 / PR, Id><<<grid, kBlock, 0, stream>>>(a, slabs, shift);
    if (rows != 128) return launched("softmax_forward_slab_kernel");
  }
  softmax_forward_slab_kernel<LOG_LS, 128 / PR, Id><<<grid, kBlock, 0, stream>>>(a, slabs, shift);
  return launched("softmax_forward_slab_kernel");
}

template <int LOG_LS, int SW, typename Id>
int launch_backward_slabs_of(const BackwardArgs& a, int rows, int64_t slabs, int shift, hipStream_t stream) {
  constexpr int PR = 64 >> LOG_LS;
  constexpr int kThreads = SW == 1 ? kBlock : SW * 64;
  const dim3 grid = launch_grid(SW == 1 ? (a.n_nodes + kWaves - 1) / kWaves : a.n_nodes, kThreads);
  if constexpr (!__is_same(Id, int64_t)) {
    if (rows == 32) softmax_backward_slab_kernel<LOG_LS, 32 / PR, SW, Id><<<grid, kThreads, 0, stream>>>(a, slabs, shift);
    if (rows == 64) softmax_backward_slab_kernel<LOG_LS, 64 / PR, SW, Id><<<grid, kThreads, 0, stream>>>(a, slabs, shift);
    if constexpr (LOG_LS == 3)
      if (rows == 96) softmax_backward_slab_kernel<LOG_LS, 96 / PR, SW, Id><<<grid, kThreads, 0, stream>>>(a, slabs, shift);
    if constexpr (LOG_LS == 1)
      if (rows == 512) softmax_backward_slab_kernel<LOG_LS, 512 / PR, SW, Id><<<grid, kThreads, 0, stream>>>(a, slabs, shift);
    if constexpr (LOG_LS < 3)
      if (rows == 256) softmax_backward_slab_kernel<LOG_LS, 256 / PR, SW, Id><<<grid, kThreads, 0, stream>>>(a, slabs, shift);
    if (rows != 128) return launched("softmax_backward_slab_kernel");
  }
  softmax_backward_slab_kernel<LOG_LS, 128 / PR, SW, Id><<<grid, kThreads, 0, stream>>>(a, slabs, shift);
  return launched("softmax_backward_slab_kernel");
}

template <int LOG_LS, typename Id>
int launch_backward_slabs(const BackwardArgs& a, int rows, int64_t slabs, int shift, hipStream_t stream) {
  if constexpr (LOG_LS == 3) {
    if (slabs > 4) return launch_backward_slabs_of<LOG_LS, kSlabWaves, Id>(a, rows, slabs, shift, stream);
    if (slabs > 2) return launch_backward_slabs_of<LOG_LS, 4, Id>(a, rows, slabs, shift, stream);
    if (slabs > 1) return launch_backward_slabs_of<LOG_LS, 2, Id>(a, rows, slabs, shift, stream);
  }
  return launch_backward_slabs_of<LOG_LS, 1, Id>(a, rows, slabs, shift, stream);
}

#define DPA4K_SLABS(LAUNCH, ID)                                                         \
  (log_ls == 1 ? LAUNCH<1, ID>(a, rows, slabs, shift, stream)                                   \
               : (log_ls == 2 ? LAUNCH<2, ID>(a, rows, slabs, shift, stream) : LAUNCH<3, ID>(a, rows, slabs, shift, stream)))

// Whether [a, a + floats) and [b, b + floats) share memory.
bool overlap(const float* a, const float* b, int64_t floats) {
  const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
  const uintptr_t bytes = static_cast<uintptr_t>(floats) * 4u;
  return a != nullptr && b != nullptr && x < y + bytes && y < x + bytes;
}

// Chunks by which the slabs of a call in place start early: half a slab where the last chunk repeats columns of the
// slab before it.
int slab_shift(int64_t channels, bool in_place) {
  return in_place && channels > 32 && channels % 32 >= 1 && channels % 32 <= 3 ? 4 : 0;
}

int forward_slabs(const ForwardArgs& a, hipStream_t stream) {
  const int shift = slab_shift(a.channels, overlap(a.alpha, a.logit, a.n_edges * a.channels) ||
                                               overlap(a.null_alpha, a.null_logit, a.n_nodes * a.channels));
  const int log_ls = slab_lanes_log(a.channels);
  const int64_t slabs = ((a.channels + 3) / 4 + shift + (1 << log_ls) - 1) >> log_ls;
  const int rows = slab_rows(a.n_edges, a.n_nodes, log_ls);
  if (!grid_fits(a.n_nodes * slabs, kBlock)) return fail(DPA4K_EINVAL, "segment softmax: grid too large");
  switch (row_ids(a.order, a.n_edges, a.channels)) {
    case RowIds::kViews: return DPA4K_SLABS(launch_forward_slabs, Views);
    case RowIds::kSharedViews: return launch_forward_slabs<3, SharedViews>(a, rows, slabs, shift, stream);
    case RowIds::kNarrow: return DPA4K_SLABS(launch_forward_slabs, uint32_t);
    default: return DPA4K_SLABS(launch_forward_slabs, int64_t);
  }
}

int backward_slabs(const BackwardArgs& a, hipStream_t stream) {
  const int64_t elements = a.n_edges * a.channels, null_elements = a.n_nodes * a.channels;
  const int shift =
      slab_shift(a.channels, overlap(a.grad_logit, a.grad_alpha, elements) || overlap(a.grad_logit, a.alpha, elements) ||
                                 overlap(a.grad_null_logit, a.grad_null_alpha, null_elements) ||
                                 overlap(a.grad_null_logit, a.null_alpha, null_elements));
  const int log_ls = slab_lanes_log(a.channels);
  const int64_t slabs = ((a.channels + 3) / 4 + shift + (1 << log_ls) - 1) >> log_ls;
  const int rows = slab_rows(a.n_edges, a.n_nodes, log_ls);
  switch (row_ids(a.order, a.n_edges, a.channels)) {
    case RowIds::kViews: return DPA4K_SLABS(launch_backward_slabs, Views);
    case RowIds::kSharedViews: return launch_backward_slabs<3, SharedViews>(a, rows, slabs, shift, stream);
    case RowIds::kNarrow: return DPA4K_SLABS(launch_backward_slabs, uint32_t);
    default: return DPA4K_SLABS(launch_backward_slabs, int64_t);
  }
}
#undef DPA4K_SLABS

int check_common(int64_t n_edges, int64_t n_nodes, int64_t channels, const char* what) {
  if (n_edges < 0 || n_nodes < 0) return fail(DPA4K_EINVAL, "%s: negative sizes", what);
  if (channels <= 0) return fail(DPA4K_EINVAL, "%s requires at least one channel", what);
  if (!grid_fits(n_nodes, kBlock)) return fail(DPA4K_EINVAL, "%s: segment count too large", what);
  return DPA4K_OK;
}

int softmax_forward(const float* logit, const float* env, const int64_t* offsets, const float* null_logit,
                    const int64_t* order, float* alpha, float* null_alpha, int64_t n_edges, int64_t n_nodes,
                    int64_t channels, const void* plan, int64_t n_long, int64_t plan_capacity,
                    dpa4k_stream_t stream_handle) {
  if (int s = check_common(n_edges, n_nodes, channels, "segment softmax")) return s;
  if (plan != nullptr && (n_long < 0 || n_long > n_nodes))
    return fail(DPA4K_EINVAL, "segment softmax: n_long outside [0, n_nodes]");
  if (n_nodes == 0) return DPA4K_OK;
  if (offsets == nullptr || (n_edges > 0 && (logit == nullptr || env == nullptr || alpha == nullptr)))
    return fail(DPA4K_EINVAL, "segment softmax: null pointer");
  if ((null_logit == nullptr) != (null_alpha == nullptr))
    return fail(DPA4K_EINVAL, "segment softmax: null_logit and null_alpha go together");
  hipStream_t stream = as_stream(stream_handle);
  const bool vec4 = channels % 4 == 0 && aligned16(logit) && aligned16(alpha) &&
                    (null_logit == nullptr || (aligned16(null_logit) && aligned16(null_alpha)));
  const ForwardArgs a{logit, env, offsets, null_logit, order, alpha, null_alpha, n_edges, n_nodes, channels};
  if (uses_slabs(channels, vec4, n_edges, n_nodes)) return forward_slabs(a, stream);
  // a plan applies only to the geometry it was built for; otherwise run unplanned
  const bool use_plan = plan != nullptr && plan_capacity == capacity_for(channels, vec4, n_edges, n_nodes);
  const int64_t* words = use_plan ? static_cast<const int64_t*>(plan) : nullptr;
  const int64_t listed = use_plan ? n_long : 0;
  if (vec4) {
    switch (lanes_log_for(channels / 4)) {
      case 0: return launch_forward<4, 0>(a, words, listed, stream);
      case 1: return launch_forward<4, 1>(a, words, listed, stream);
      case 2: return launch_forward<4, 2>(a, words, listed, stream);
      case 3: return launch_forward<4, 3>(a, words, listed, stream);
      case 4: return launch_forward<4, 4>(a, words, listed, stream);
      case 5: return launch_forward<4, 5>(a, words, listed, stream);
      default: return launch_forward<4, 6>(a, words, listed, stream);
    }
  }
  if (channels == 1) return launch_forward<1, 0>(a, words, listed, stream);
  if (channels == 2) return launch_forward<1, 1>(a, words, listed, stream);
  return launch_forward<1, 2>(a, words, listed, stream);
}

int softmax_backward(const float* alpha, const float* grad_alpha, const float* env, const int64_t* offsets,
                     const float* null_alpha, const float* grad_null_alpha, const int64_t* order,
                     float* grad_logit, float* grad_null_logit, float* grad_env, int64_t n_edges,
                     int64_t n_nodes, int64_t channels, const void* plan, int64_t n_long,
                     int64_t plan_capacity, dpa4k_stream_t stream_handle) {
  if (int s = check_common(n_edges, n_nodes, channels, "segment softmax backward")) return s;
  if (plan != nullptr && (n_long < 0 || n_long > n_nodes))
    return fail(DPA4K_EINVAL, "segment softmax backward: n_long outside [0, n_nodes]");
  if (n_nodes == 0) return DPA4K_OK;
  if (offsets == nullptr ||
      (n_edges > 0 && (alpha == nullptr || grad_alpha == nullptr || env == nullptr ||
                       grad_logit == nullptr || grad_env == nullptr)))
    return fail(DPA4K_EINVAL, "segment softmax backward: null pointer");
  const bool has_null = null_alpha != nullptr;
  if (has_null != (grad_null_alpha != nullptr) || has_null != (grad_null_logit != nullptr))
    return fail(DPA4K_EINVAL, "segment softmax requires null_alpha and grad_null_alpha together");
  hipStream_t stream = as_stream(stream_handle);
  const bool vec4 = channels % 4 == 0 && aligned16(alpha) && aligned16(grad_alpha) && aligned16(grad_logit) &&
                    (!has_null || (aligned16(null_alpha) && aligned16(grad_null_alpha) &&
                                   aligned16(grad_null_logit)));
  const BackwardArgs a{alpha, grad_alpha, env, offsets, null_alpha, grad_null_alpha, order,
                       grad_logit, grad_null_logit, grad_env, n_edges, n_nodes, channels};
  if (uses_slabs(channels, vec4, n_edges, n_nodes)) return backward_slabs(a, stream);
  // a plan applies only to the geometry it was built for; otherwise run unplanned
  const bool use_plan = plan != nullptr && plan_capacity == capacity_for(channels, vec4, n_edges, n_nodes);
  const int64_t* words = use_plan ? static_cast<const int64_t*>(plan) : nullptr;
  const int64_t listed = use_plan ? n_long : 0;
  if (vec4) {
    switch (lanes_log_for(channels / 4)) {
      case 0: return launch_backward<4, 0>(a, words, listed, stream);
      case 1: return launch_backward<4, 1>(a, words, listed, stream);
      case 2: return launch_backward<4, 2>(a, words, listed, stream);
      case 3: return launch_backward<4, 3>(a, words, listed, stream);
      case 4: return launch_backward<4, 4>(a, words, listed, stream);
      case 5: return launch_backward<4, 5>(a, words, listed, stream);
      default: return launch_backward<4, 6>(a, words, listed, stream);
    }
  }
  if (channels == 1) return launch_backward<1, 0>(a, words, listed, stream);
  if (channels == 2) return launch_backward<1, 1>(a, words, listed, stream);
  return launch_backward<1, 2>(a, words, listed, stream);
}

}  // namespace
}  // namespace dpa4k

using namespace dpa4k;

extern "C" int dpa4k_segment_softmax_forward(const float* logit, const float* env, const int64_t* offsets,
                                             const float* null_logit, const int64_t* order, float* alpha,
                                             float* null_alpha, int64_t n_edges, int64_t n_nodes,
                                             int64_t channels, dpa4k_stream_t stream) {
  clear_error();
  return softmax_forward(logit, env, offsets, null_logit, order, alpha, null_alpha, n_edges, n_nodes, channels,
                         nullptr, 0, 0, stream);
}

extern "C" int dpa4k_segment_softmax_backward(const float* alpha, const float* grad_alpha, const float* env,
                                              const int64_t* offsets, const float* null_alpha,
                                              const float* grad_null_alpha, const int64_t* order,
                                              float* grad_logit, float* grad_null_logit, float* grad_env,
                                              int64_t n_edges, int64_t n_nodes, int64_t channels,
                                              dpa4k_stream_t stream) {
  clear_error();
  return softmax_backward(alpha, grad_alpha, env, offsets, null_alpha, grad_null_alpha, order, grad_logit,
                          grad_null_logit, grad_env, n_edges, n_nodes, channels, nullptr, 0, 0, stream);
}

extern "C" size_t dpa4k_segment_softmax_plan_size(int64_t n_nodes) {
  if (n_nodes < 0) return 0;
  return round_up_256(static_cast<size_t>(kPlanHeader + n_nodes + plan_tiles(n_nodes)) * sizeof(int64_t));
}

extern "C" int dpa4k_segment_softmax_plan(const int64_t* offsets, int64_t n_edges, int64_t n_nodes,
                                          int64_t channels, void* plan, size_t plan_bytes, int64_t* n_long,
                                          int64_t* plan_capacity, dpa4k_stream_t stream_handle) {
  clear_error();
  if (int s = check_common(n_edges, n_nodes, channels, "segment softmax plan")) return s;
  if (offsets == nullptr || plan == nullptr || n_long == nullptr || plan_capacity == nullptr)
    return fail(DPA4K_EINVAL, "segment softmax plan: null pointer");
  if (plan_bytes < dpa4k_segment_softmax_plan_size(n_nodes))
    return fail(DPA4K_EWORKSPACE, "segment softmax plan: %zu bytes given, %zu needed", plan_bytes,
                dpa4k_segment_softmax_plan_size(n_nodes));
  hipStream_t stream = as_stream(stream_handle);
  // The plan is for the 128-bit row kernel when C % 4 == 0 (operands from
  // torch's allocator are 16-byte aligned), for the scalar one otherwise.
  const int64_t capacity = capacity_for(channels, channels % 4 == 0, n_edges, n_nodes > 0 ? n_nodes : 1);
  int64_t* words = static_cast<int64_t*>(plan);
  // The slab kernels need no plan: an empty one, and no host synchronisation.
  const int64_t tiles = capacity > 0 ? plan_tiles(n_nodes) : 0;
  int64_t* counts = words + kPlanHeader + n_nodes;
  if (tiles > 0) {
    plan_count_kernel<<<launch_grid(tiles, kPlanThreads), kPlanThreads, 0, stream>>>(offsets, n_nodes, n_edges,
                                                                                     capacity, counts);
    if (int s = launched("plan_count_kernel")) return s;
  }
  plan_scan_kernel<<<1, kPlanThreads, 0, stream>>>(counts, tiles, capacity, words);
  if (int s = launched("plan_scan_kernel")) return s;
  if (capacity == 0) {
    *n_long = 0;
    *plan_capacity = 0;
    return DPA4K_OK;
  }
  if (tiles > 0) {
    plan_write_kernel<<<launch_grid(tiles, kPlanThreads), kPlanThreads, 0, stream>>>(
        offsets, n_nodes, n_edges, capacity, counts, words + kPlanHeader);
    if (int s = launched("plan_write_kernel")) return s;
  }
  int64_t header[2] = {0, 0};
  if (int s = hip_status(hipMemcpyAsync(header, words, sizeof(header), hipMemcpyDeviceToHost, stream),
                         "hipMemcpyAsync(plan header)"))
    return s;
  if (int s = hip_status(hipStreamSynchronize(stream), "hipStreamSynchronize")) return s;
  *n_long = header[1];
  *plan_capacity = header[0];
  return DPA4K_OK;
}

extern "C" int dpa4k_segment_softmax_forward_planned(const float* logit, const float* env, const int64_t* offsets,
                                                     const float* null_logit, const int64_t* order, float* alpha,
                                                     float* null_alpha, int64_t n_edges, int64_t n_nodes,
                                                     int64_t channels, const void* plan, int64_t n_long,
                                                     int64_t plan_capacity, dpa4k_stream_t stream) {
  clear_error();
  return softmax_forward(logit, env, offsets, null_logit, order, alpha, null_alpha, n_edges, n_nodes, channels,
                         plan, n_long, plan_capacity, stream);
}

extern "C" int dpa4k_segment_softmax_backward_planned(const float* alpha, const float* grad_alpha, const float* env,
                                                      const int64_t* offsets, const float* null_alpha,
                                                      const float* grad_null_alpha, const int64_t* order,
                                                      float* grad_logit, float* grad_null_logit, float* grad_env,
                                                      int64_t n_edges, int64_t n_nodes, int64_t channels,
                                                      const void* plan, int64_t n_long, int64_t plan_capacity,
                                                      dpa4k_stream_t stream) {
  clear_error();
  return softmax_backward(alpha, grad_alpha, env, offsets, null_alpha, grad_null_alpha, order, grad_logit,
                          grad_null_logit, grad_env, n_edges, n_nodes, channels, plan, n_long, plan_capacity,
                          stream);
}
