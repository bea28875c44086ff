// Row-wise RMSNorm, forward and backward (python/kernels/rmsnorm.py:46-85,
// csrc/rmsnorm.cpp:99-157 of the reference; oracle python/reference/rmsnorm.py:40-52):
//   inv = 1 / sqrt(mean(x^2) + eps),  y = (x * inv) * scale
//   u = grad * scale,  grad_x = inv * u - (x * inv^3) * mean(x * u)
//   grad_scale[w] = sum_rows grad * (x * inv)
//
// A wave, or 16 or 32 of its lanes, per row.  Rows of up to 64 * 16 float4
// chunks (W <= 4096) stay in registers between the sum of squares and the
// scaled store, so x is read once; the row sum is a DPP / swizzle / bpermute
// butterfly.  Wider rows take a two-pass streaming kernel.  The reference
// accumulates grad_scale with one float atomic per (row, column); here each
// lane group keeps per-column partials for its fixed set of rows, the groups
// of a workgroup add theirs in LDS, the workgroup partials go to the workspace
// and a workgroup per 64 columns sums them (its waves split the rows, each
// load reading 256 contiguous bytes) -- every order fixed.
#include <mutex>
#include <vector>

#include "common.h"

namespace dpa4k {
namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
constexpr int kPartialWaves = 3072;   // waves of the grad_scale backward (resident at 3 per SIMD)
constexpr int64_t kRegisterMaxWidth = 64 * 16 * 4;  // widest row the register kernels hold

// Column partials of dpa4k_rmsnorm_backward_noalloc: one row per workgroup of
// the grad_scale backward (at most kPartialWaves / kWaves of them) of at most
// kRegisterMaxWidth floats, the most the register kernels ever write
// (DPA4K_RMSNORM_NOALLOC_SCRATCH_BYTES); wider rows do not use it.  Every device the library runs on
// holds its own copy until the process ends.  Host code never uses this name
// as an address: it reaches the array through the per-device pointer that
// scratch_for_stream() obtains from hipGetSymbolAddress.
static_assert(int64_t(kPartialWaves / kWaves) * kRegisterMaxWidth * 4 == DPA4K_RMSNORM_NOALLOC_SCRATCH_BYTES,
              "the header's scratch size must match the partial matrix bound");
__device__ __align__(256) float scratch[DPA4K_RMSNORM_NOALLOC_SCRATCH_BYTES / 4];

__device__ __forceinline__ float inverse_rms_of(float sum_squares, int64_t width, float eps) {
  return 1.0f / sqrtf(sum_squares / static_cast<float>(width) + eps);
}

// A row's chunks over a group of LG lanes: chunk j of lane l is V columns of
// the row, from byte at(j).  With V = 4 the row's last chunk starts at width -
// 4, whatever the width and the alignment; where the width is no multiple of 4
// (kTail) its first `skip` columns are the neighbour's, equal in both lanes, and
// count in no sum.  A chunk past the row lies past every view: past the row's
// own view where a wave has one row (LG = 64), else at kNoRow.
template <int V, int LG, int CPL, bool kTail>
struct RowChunks {
  static constexpr bool kOwnView = LG == 64 && !kTail;
  uint32_t first, start[kOwnView ? 1 : CPL];
  int skip[kTail ? CPL : 1];
  __device__ __forceinline__ RowChunks(int lane, int64_t width) {
    first = static_cast<uint32_t>(lane) * (V * 4u);
    if constexpr (!kOwnView)
#pragma unroll
      for (int j = 0; j < CPL; ++j) {
        const int64_t begin = static_cast<int64_t>(lane + LG * j) * V;
        const int64_t column = !kTail || begin + V <= width ? begin : width - V;
        const bool live = begin < width;
        start[j] = live ? static_cast<uint32_t>(column) * 4u : kNoRow;
        if constexpr (kTail) skip[j] = live ? static_cast<int>(begin - column) : V;
      }
  }
  __device__ __forceinline__ uint32_t at(int j) const {
    if constexpr (kOwnView) return first + static_cast<uint32_t>(j * LG * V * 4);
    else return start[j];
  }
  // Stores leave the lanes past the row out by the execution mask: dropped by
  // the view, they still take the lane's turn (two chunks a lane: 200,000 rows
  // of 300 floats, 11 of 64 lanes in the second, 160 -> 137 us with the scale gradient; with one chunk a lane the
  // branch costs more than the lanes).
  __device__ __forceinline__ bool live(int j, int64_t width) const { return at(j) < static_cast<uint32_t>(width) * 4u; }
  __device__ __forceinline__ bool counts(int j, int i) const {
    if constexpr (kTail) return i >= skip[j];
    else return true;
  }
};

// The GPW rows from `first` of a row-major [rows, width] array (none past its end).
template <int GPW>
__device__ __forceinline__ BufferView group_view(const float* p, int64_t first, int64_t rows, int64_t width) {
  const int64_t left = rows - first;
  const int64_t count = left < GPW ? (left < 0 ? 0 : left) : GPW;
  return buffer_view(p + (count > 0 ? first : 0) * width, count * width * 4);
}

// One group of LG lanes per row (LG = 16, 32 or 64: the row's chunks, CPL per
// lane past 64), NR rows per group in flight, so a wave covers 64 / LG * NR
// consecutive rows.  Bound by the two row streams.  A wave per row with one
// chunk a lane left most lanes without a column and little in flight at narrow
// widths: 262,144 rows of 64 took 61 us (2.2 TB/s), now 24 us (5.6); rows of 1,024
// are unchanged (33 us for 24,576 rows, 6.1 TB/s).  Rows whose width is not a
// multiple of 4 were read one float a lane, twice past 1,024 columns: 24,576
// rows of 2,777 took 175 us, now 102 us.
template <int V, int LG, int CPL, int NR, bool kTail>
__global__ __launch_bounds__(kBlock) void rmsnorm_forward_kernel(
    const float* __restrict__ x, const float* __restrict__ scale, float* __restrict__ y,
    float* __restrict__ inverse_rms, int64_t rows, int64_t width, float eps) {
  constexpr int GPW = 64 / LG;
  const int64_t base = uniform_i64((block_index() * kWaves + (threadIdx.x >> 6)) * (GPW * NR));
  if (base >= rows) return;
  const int lane = threadIdx.x & (LG - 1);
  const int group = (threadIdx.x & 63) / LG;
  const uint32_t group_at = static_cast<uint32_t>(group) * (static_cast<uint32_t>(width) * 4u);
  const RowChunks<V, LG, CPL, kTail> chunks(lane, width);
  // The rows and the scale are loaded before the reduction, through views
  // (zeros past the rows), so that no load sits in a branch: a load in a
  // divergent branch is waited for before the branch closes, and the chunk
  // loads would follow one another instead of overlapping.
  const BufferView row_s = buffer_view(scale, scale != nullptr ? width * 4 : 0);
  fvec<V> value[NR][CPL], s[CPL];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const BufferView rows_x = group_view<GPW>(x, base + r * GPW, rows, width);
#pragma unroll
    for (int j = 0; j < CPL; ++j) value[r][j] = buffer_load_vec<V>(rows_x, group_at + chunks.at(j));
  }
#pragma unroll
  for (int j = 0; j < CPL; ++j) s[j] = buffer_load_vec<V>(row_s, chunks.at(j));
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    float sum = 0.0f;
#pragma unroll
    for (int j = 0; j < CPL; ++j)
#pragma unroll
      for (int i = 0; i < V; ++i)
        sum = sum + (chunks.counts(j, i) ? value[r][j].v[i] * value[r][j].v[i] : 0.0f);
    sum = group_sum<LG>(sum);
    const float inv = inverse_rms_of(sum, width, eps);
    const BufferView rows_y = group_view<GPW>(y, base + r * GPW, rows, width);
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      fvec<V> out;
#pragma unroll
      for (int i = 0; i < V; ++i) {
        out.v[i] = value[r][j].v[i] * inv;
        if (scale != nullptr) out.v[i] = out.v[i] * s[j].v[i];
      }
      if (CPL != 2 || chunks.live(j, width)) buffer_store_vec_stream<V>(rows_y, group_at + chunks.at(j), out);
    }
    if (lane == 0 && base + r * GPW + group < rows) inverse_rms[base + r * GPW + group] = inv;
  }
}

// Rows wider than the register kernels hold: a wave per row, two passes.
template <bool kTail>
__global__ __launch_bounds__(kBlock) void rmsnorm_forward_wide_kernel(
    const float* __restrict__ x, const float* __restrict__ scale, float* __restrict__ y,
    float* __restrict__ inverse_rms, int64_t rows, int64_t width, float eps) {
  const int64_t row = block_index() * kWaves + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  const float* xr = x + row * width;
  float* yr = y + row * width;
  float sum = 0.0f;
  for (int64_t c = lane * 4; c < width; c += 256) {
    const int64_t column = !kTail || c + 4 <= width ? c : width - 4;
    const fvec<4> value = load_chunk(xr + column);
#pragma unroll
    for (int i = 0; i < 4; ++i) sum = sum + (!kTail || column + i >= c ? value.v[i] * value.v[i] : 0.0f);
  }
  sum = group_sum<64>(sum);
  const float inv = inverse_rms_of(sum, width, eps);
  for (int64_t c = lane * 4; c < width; c += 256) {
    const int64_t column = !kTail || c + 4 <= width ? c : width - 4;
    const fvec<4> value = load_chunk(xr + column);
    fvec<4> out, s;
    if (scale != nullptr) s = load_chunk(scale + column);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      out.v[i] = value.v[i] * inv;
      if (scale != nullptr) out.v[i] = out.v[i] * s.v[i];
    }
    store_own(yr + column, out, static_cast<int>(c - column));  // y may be x
  }
  if (lane == 0) inverse_rms[row] = inv;
}

// Register path: wave w handles the GPW = 64 / LG rows from w * GPW, then those
// `waves` * GPW further on, and so on, NR of these row sets per round (far
// apart, so that a small grid still spreads over every wave); with `partial`
// non-null the workgroup also stores its per-column sum of grad * (x * inv) as
// its row of the [workgroups, W] partial matrix.  All rows of a round are loaded
// before any is reduced, non-temporally: they are read once (114,688 rows of
// 1,024: 261 -> 247 us).  Bound by the three row streams; against a wave per
// row, 262,144 rows of 64 went from 62 to 33 us; rows of 2,777 from 269 us and 11 ms for
// the scale gradient, a thread per column over all rows, to 130 us with it.
template <int V, int LG, int CPL, int NR, bool kTail>
__global__ __launch_bounds__(kBlock) void rmsnorm_backward_kernel(
    const float* __restrict__ grad, const float* __restrict__ x, const float* __restrict__ scale,
    const float* __restrict__ inverse_rms, float* __restrict__ grad_x, float* __restrict__ partial,
    int64_t rows, int64_t width) {
  constexpr int GPW = 64 / LG;
  const int64_t wave_id = static_cast<int64_t>(blockIdx.x) * kWaves + (threadIdx.x >> 6);
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kWaves * GPW;
  const int lane = threadIdx.x & (LG - 1);
  const int group = (threadIdx.x & 63) / LG;
  const uint32_t group_at = static_cast<uint32_t>(group) * (static_cast<uint32_t>(width) * 4u);
  const RowChunks<V, LG, CPL, kTail> chunks(lane, width);
  const BufferView row_s = buffer_view(scale, scale != nullptr ? width * 4 : 0);

  fvec<V> s[CPL], column[CPL];
#pragma unroll
  for (int j = 0; j < CPL; ++j) {
    s[j] = buffer_load_vec<V>(row_s, chunks.at(j));
#pragma unroll
    for (int i = 0; i < V; ++i) column[j].v[i] = 0.0f;
  }

  for (int64_t base = uniform_i64(wave_id * GPW); base < rows; base += stride * NR) {
    fvec<V> g[NR][CPL], xv[NR][CPL];
    float inv[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int64_t first = base + r * stride;
      const BufferView rows_g = group_view<GPW>(grad, first, rows, width);
      const BufferView rows_x = group_view<GPW>(x, first, rows, width);
      inv[r] = buffer_load_f32(group_view<GPW>(inverse_rms, first, rows, 1), static_cast<uint32_t>(group) * 4u);
#pragma unroll
      for (int j = 0; j < CPL; ++j) {
        g[r][j] = buffer_load_vec<V, kNonTemporal>(rows_g, group_at + chunks.at(j));
        xv[r][j] = buffer_load_vec<V, kNonTemporal>(rows_x, group_at + chunks.at(j));
      }
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      float dot = 0.0f;
#pragma unroll
      for (int j = 0; j < CPL; ++j)
#pragma unroll
        for (int i = 0; i < V; ++i) {
          const float u = scale != nullptr ? g[r][j].v[i] * s[j].v[i] : g[r][j].v[i];
          dot = dot + (chunks.counts(j, i) ? xv[r][j].v[i] * u : 0.0f);
        }
      dot = group_sum<LG>(dot);
      const float mean_dot = dot / static_cast<float>(width);
      const float inv3 = inv[r] * inv[r] * inv[r];
      const BufferView rows_o = group_view<GPW>(grad_x, base + r * stride, rows, width);
#pragma unroll
      for (int j = 0; j < CPL; ++j) {
        fvec<V> out;
#pragma unroll
        for (int i = 0; i < V; ++i) {
          const float u = scale != nullptr ? g[r][j].v[i] * s[j].v[i] : g[r][j].v[i];
          out.v[i] = inv[r] * u - xv[r][j].v[i] * inv3 * mean_dot;
          if (partial != nullptr) column[j].v[i] = column[j].v[i] + g[r][j].v[i] * (xv[r][j].v[i] * inv[r]);
        }
        if (CPL != 2 || chunks.live(j, width)) buffer_store_vec_stream<V>(rows_o, group_at + chunks.at(j), out);
      }
    }
  }
  if (partial != nullptr) {
    // the groups' column sums meet in LDS and are added in group order; the
    // workgroup writes one row of the [workgroups, W] partial matrix (a column
    // that two lanes hold is written twice with the same value)
    extern __shared__ float columns[];  // [kWaves * GPW][CPL * LG * V]
    constexpr int kSpan = CPL * LG * V;
    const int member = (threadIdx.x >> 6) * GPW + group;
#pragma unroll
    for (int j = 0; j < CPL; ++j)
      if (chunks.at(j) < kSpan * 4u)
#pragma unroll
        for (int i = 0; i < V; ++i) columns[member * kSpan + chunks.at(j) / 4 + i] = column[j].v[i];
    __syncthreads();
    for (int64_t c = threadIdx.x; c < width; c += kBlock) {
      float sum = columns[c];
#pragma unroll
      for (int w = 1; w < kWaves * GPW; ++w) sum = sum + columns[w * kSpan + c];
      partial[static_cast<int64_t>(blockIdx.x) * width + c] = sum;
    }
  }
}

// grad_scale[w] = sum over the workgroup partial rows [n, W]: one workgroup
// of kColumnWaves waves per 64 columns, lane l on column 64 b + l.  Wave k
// adds, in order, the rows of its share [k p, (k + 1) p) (p = n / kColumnWaves
// rounded up), so each of its loads reads 256 consecutive bytes of one row;
// the waves' sums are then added in wave order.
constexpr int kColumnWaves = 16;

__global__ __launch_bounds__(kColumnWaves * 64) void partial_columns_kernel(const float* __restrict__ partial,
                                                                            int64_t n, int64_t width,
                                                                            float* __restrict__ grad_scale) {
  __shared__ float wave_sum[kColumnWaves][64];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int64_t column = static_cast<int64_t>(blockIdx.x) * 64 + lane;
  const int64_t per = (n + kColumnWaves - 1) / kColumnWaves;
  const int64_t first = wave * per;
  const int64_t last = first + per < n ? first + per : n;
  float sum = 0.0f;
  if (column < width) {
    const float* source = partial + column;
    int64_t r = first;
    // eight loads in flight, added in row order
    for (; r + 8 <= last; r += 8) {
      float value[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) value[i] = source[(r + i) * width];
#pragma unroll
      for (int i = 0; i < 8; ++i) sum = sum + value[i];
    }
    for (; r < last; ++r) sum = sum + source[r * width];
  }
  wave_sum[wave][lane] = sum;
  __syncthreads();
  if (wave == 0 && column < width) {
    float total = 0.0f;
#pragma unroll
    for (int k = 0; k < kColumnWaves; ++k) total = total + wave_sum[k][lane];
    grad_scale[column] = total;
  }
}

// Streaming grad_x for wide rows: two passes over the row.
template <bool kTail>
__global__ __launch_bounds__(kBlock) void rmsnorm_backward_wide_kernel(
    const float* __restrict__ grad, const float* __restrict__ x, const float* __restrict__ scale,
    const float* __restrict__ inverse_rms, float* __restrict__ grad_x, int64_t rows,
    int64_t width) {
  const int64_t row = block_index() * kWaves + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  const float* gr = grad + row * width;
  const float* xr = x + row * width;
  float dot = 0.0f;
  for (int64_t c = lane * 4; c < width; c += 256) {
    const int64_t column = !kTail || c + 4 <= width ? c : width - 4;
    const fvec<4> g = load_chunk(gr + column);
    const fvec<4> xv = load_chunk(xr + column);
    fvec<4> s;
    if (scale != nullptr) s = load_chunk(scale + column);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      dot = dot + (!kTail || column + i >= c ? xv.v[i] * (scale != nullptr ? g.v[i] * s.v[i] : g.v[i]) : 0.0f);
  }
  dot = group_sum<64>(dot);
  const float mean_dot = dot / static_cast<float>(width);
  const float inv = inverse_rms[row];
  const float inv3 = inv * inv * inv;
  for (int64_t c = lane * 4; c < width; c += 256) {
    const int64_t column = !kTail || c + 4 <= width ? c : width - 4;
    const fvec<4> g = load_chunk(gr + column);
    const fvec<4> xv = load_chunk(xr + column);
    fvec<4> s;
    if (scale != nullptr) s = load_chunk(scale + column);
    fvec<4> out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float u = scale != nullptr ? g.v[i] * s.v[i] : g.v[i];
      out.v[i] = inv * u - xv.v[i] * inv3 * mean_dot;
    }
    store_own(grad_x + row * width + column, out, static_cast<int>(c - column));  // grad_x may be grad or x
  }
}

// grad_scale without a partial matrix, for rows that the register kernels do
// not hold and for calls without a workspace: a workgroup per 32 columns, whose
// kColumnGroups half waves take the rows in turn (128 bytes of one row per load,
// four rows in flight each) and meet in LDS, added in group order.  The sums are
// kept in 64 bits.  A thread per column over all rows took 2.5 ms for 6,000 rows
// of 5,000 floats, this one 78 us; shares of the rows in a partial matrix took
// 48 us, but needed memory that two overlapping calls would share.
constexpr int kColumnGroups = 2 * kColumnWaves;

__global__ __launch_bounds__(kColumnWaves * 64) void rmsnorm_scale_columns_kernel(
    const float* __restrict__ grad, const float* __restrict__ x, const float* __restrict__ inverse_rms,
    float* __restrict__ grad_scale, int64_t rows, int64_t width) {
  constexpr int U = 4;
  __shared__ double group_total[kColumnGroups][32];
  const int lane = threadIdx.x & 31;
  const int group = threadIdx.x >> 5;
  const int64_t column = block_index() * 32 + lane;
  const bool live = column < width;
  double sum = 0.0;
  if (live) {
    int64_t row = group;
    for (; row + (U - 1) * kColumnGroups < rows; row += U * kColumnGroups) {
      float g[U], xv[U], inv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t at = row + u * kColumnGroups;
        g[u] = __builtin_nontemporal_load(grad + at * width + column);
        xv[u] = __builtin_nontemporal_load(x + at * width + column);
        inv[u] = inverse_rms[at];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) sum += static_cast<double>(g[u] * (xv[u] * inv[u]));
    }
    for (; row < rows; row += kColumnGroups)
      sum += static_cast<double>(grad[row * width + column] * (x[row * width + column] * inverse_rms[row]));
  }
  group_total[group][lane] = sum;
  __syncthreads();
  if (group == 0 && live) {
#pragma unroll
    for (int k = 1; k < kColumnGroups; ++k) sum += group_total[k][lane];
    grad_scale[column] = static_cast<float>(sum);
  }
}

// The register kernels' shape for a row of `width` floats: chunks of V floats
// over LG lanes, CPL per lane.  LG lanes cover rows of up to 256 columns with
// one chunk each; wider rows take 64 lanes and CPL chunks.
struct RowShape {
  int v, lanes, per_lane;
};
bool fits_registers(int64_t width) { return width <= kRegisterMaxWidth; }
RowShape shape_for(int64_t width) {
  if (width < 4) return {1, 16, 1};
  const int64_t chunks = (width + 3) / 4;
  if (chunks <= 16) return {4, 16, 1};
  if (chunks <= 32) return {4, 32, 1};
  int cpl = 1;
  while (64 * cpl < chunks) cpl <<= 1;
  return {4, 64, cpl};
}

// Row sets in flight per wave: forward 4 for the lane groups below a wave where
// the grid fills the chip (16 waves on each CU) all the same, else 1 (rows of
// 512 took 25.3 us with two against 23.4 us with one, 32,768 rows).  Backward,
// where a wave has several (with a scale gradient the grid is bounded): 4 for
// the lane groups, 2 for two to eight chunks a lane, 1 for one chunk (300,000 rows of
// 200: 126 us, 141 with two) and where a row alone takes 128 registers (2,048
// columns on: 139 us with two, spilling past the wave's own registers, 120 us
// with one).  Without a scale gradient every wave has one set: 400,000 rows of 66
// floats 55 us, 106 while three sets of four lay past the rows.
constexpr int forward_rows(int lanes) { return lanes < 64 ? 4 : 1; }
constexpr int backward_rows(int lanes, int cpl) { return cpl >= 16 || (lanes == 64 && cpl == 1) ? 1 : (lanes < 64 ? 4 : 2); }
constexpr int64_t kFullGrid = 4096;  // waves

// Calls LAUNCH(V, LG, CPL) for a row shape.
#define DPA4K_ROW_SHAPES(shape, LAUNCH)                   \
  if (shape.v == 1) LAUNCH(1, 16, 1);                     \
  else if (shape.lanes == 16) LAUNCH(4, 16, 1);           \
  else if (shape.lanes == 32) LAUNCH(4, 32, 1);           \
  else if (shape.per_lane == 1) LAUNCH(4, 64, 1);         \
  else if (shape.per_lane == 2) LAUNCH(4, 64, 2);         \
  else if (shape.per_lane == 4) LAUNCH(4, 64, 4);         \
  else if (shape.per_lane == 8) LAUNCH(4, 64, 8);         \
  else LAUNCH(4, 64, 16);

// Workgroups whose waves take `sets` row sets each.
int64_t row_blocks(const RowShape& shape, int sets, int64_t rows) {
  const int64_t per_block = static_cast<int64_t>(kWaves) * (64 / shape.lanes) * sets;
  return (rows + per_block - 1) / per_block;
}

template <int V, int LG, int CPL, int NR>
void launch_forward_rows(const RowShape& shape, const float* x, const float* scale, float* y, float* inverse_rms,
                         int64_t rows, int64_t width, float eps, hipStream_t stream) {
  const dim3 grid = launch_grid(row_blocks(shape, NR, rows), kBlock);
  if (V == 4 && width % 4 != 0)
    rmsnorm_forward_kernel<V, LG, CPL, NR, V == 4><<<grid, kBlock, 0, stream>>>(x, scale, y, inverse_rms, rows,
                                                                                width, eps);
  else
    rmsnorm_forward_kernel<V, LG, CPL, NR, false><<<grid, kBlock, 0, stream>>>(x, scale, y, inverse_rms, rows, width,
                                                                               eps);
}

int launch_forward(const float* x, const float* scale, float* y, float* inverse_rms,
                   int64_t rows, int64_t width, float eps, hipStream_t stream) {
  const RowShape shape = shape_for(width);
  const bool full = row_blocks(shape, forward_rows(shape.lanes), rows) * kWaves >= kFullGrid;
#define DPA4K_RMS_FWD(V, LG, CPL)                                                                               \
  (full ? launch_forward_rows<V, LG, CPL, forward_rows(LG)> : launch_forward_rows<V, LG, CPL, 1>)(             \
      shape, x, scale, y, inverse_rms, rows, width, eps, stream)
  DPA4K_ROW_SHAPES(shape, DPA4K_RMS_FWD)
#undef DPA4K_RMS_FWD
  return launched("rmsnorm_forward_kernel");
}

template <int V, int LG, int CPL, int NR>
void launch_backward_rows(unsigned int grid, const float* grad, const float* x, const float* scale,
                          const float* inverse_rms, float* grad_x, float* partial, int64_t rows, int64_t width,
                          hipStream_t stream) {
  const size_t lds = partial != nullptr ? kWaves * CPL * 64 * V * sizeof(float) : 0;
  if (V == 4 && width % 4 != 0)
    rmsnorm_backward_kernel<V, LG, CPL, NR, V == 4><<<grid, kBlock, lds, stream>>>(grad, x, scale, inverse_rms, grad_x,
                                                                                   partial, rows, width);
  else
    rmsnorm_backward_kernel<V, LG, CPL, NR, false><<<grid, kBlock, lds, stream>>>(grad, x, scale, inverse_rms, grad_x,
                                                                                  partial, rows, width);
}

int launch_backward(unsigned int grid, const float* grad, const float* x,
                    const float* scale, const float* inverse_rms, float* grad_x, float* partial,
                    int64_t rows, int64_t width, hipStream_t stream) {
  const RowShape shape = shape_for(width);
  // one row set per wave: further ones would lie past the rows, and be loaded, reduced and dropped all the same
  const bool single = row_blocks(shape, 1, rows) <= static_cast<int64_t>(grid);
#define DPA4K_RMS_BWD(V, LG, CPL)                                                                               \
  (single ? launch_backward_rows<V, LG, CPL, 1> : launch_backward_rows<V, LG, CPL, backward_rows(LG, CPL)>)(    \
      grid, grad, x, scale, inverse_rms, grad_x, partial, rows, width, stream)
  DPA4K_ROW_SHAPES(shape, DPA4K_RMS_BWD)
#undef DPA4K_RMS_BWD
  return launched("rmsnorm_backward_kernel");
}

// Rows of the partial matrix of the register kernels' scale gradient: the
// backward's workgroups.
unsigned int partial_blocks(int64_t rows, int64_t width) {
  const int64_t cap = kPartialWaves / kWaves;
  const int64_t wanted = row_blocks(shape_for(width), 1, rows);
  return static_cast<unsigned int>(wanted > cap ? cap : (wanted < 1 ? 1 : wanted));
}

// Device address of `scratch` on the device that runs `stream`, looked up once
// per device with that device current (the null stream runs on the current
// device).  Sets `out` or returns an error status.
int scratch_for_stream(hipStream_t stream, float*& out) {
  static std::mutex lock;
  static std::vector<float*> per_device;
  int current = 0;
  if (int s = hip_status(hipGetDevice(&current), "hipGetDevice")) return s;
  int device = current;
  if (stream != nullptr) {
    if (int s = hip_status(hipStreamGetDevice(stream, &device), "hipStreamGetDevice")) return s;
  }
  std::lock_guard<std::mutex> guard(lock);
  if (per_device.empty()) {
    int count = 0;
    if (int s = hip_status(hipGetDeviceCount(&count), "hipGetDeviceCount")) return s;
    per_device.assign(static_cast<size_t>(count > 0 ? count : 1), nullptr);
  }
  if (device < 0 || static_cast<size_t>(device) >= per_device.size())
    return fail(DPA4K_EHIP, "RMSNorm backward: stream on unknown device %d", device);
  if (per_device[device] == nullptr) {
    if (device != current) {
      if (int s = hip_status(hipSetDevice(device), "hipSetDevice")) return s;
    }
    void* address = nullptr;
    const hipError_t found = hipGetSymbolAddress(&address, HIP_SYMBOL(scratch));
    if (device != current) {
      if (int s = hip_status(hipSetDevice(current), "hipSetDevice")) return s;
    }
    if (int s = hip_status(found, "hipGetSymbolAddress(scratch)")) return s;
    if (address == nullptr) return fail(DPA4K_EHIP, "hipGetSymbolAddress(scratch) returned a null address");
    per_device[device] = static_cast<float*>(address);
  }
  out = per_device[device];
  return DPA4K_OK;
}

size_t backward_workspace_bytes(int64_t rows, int64_t width) {
  if (rows <= 0 || width <= 0) return 0;
  if (!fits_registers(width)) return round_up_256(static_cast<size_t>(width) * 4);  // not used: a size grows with the input
  return round_up_256(static_cast<size_t>(partial_blocks(rows, width)) * static_cast<size_t>(width) * 4);
}

// The backward with its column partials in `workspace` (checked against the size the
// shape needs; only the register kernels with a scale gradient use it), or, with
// `static_scratch`, in this device's `scratch` array.
int rmsnorm_backward(const float* grad, const float* x, const float* scale, const float* inverse_rms,
                     float* grad_x, float* grad_scale, int64_t rows, int64_t width, void* workspace,
                     size_t workspace_bytes, bool static_scratch, hipStream_t stream) {
  if (rows < 0) return fail(DPA4K_EINVAL, "RMSNorm: negative row count");
  if (width <= 0) return fail(DPA4K_EINVAL, "RMSNorm feature dimension must be positive");
  if (grad_scale != nullptr && scale == nullptr)
    return fail(DPA4K_EINVAL, "cannot compute a scale gradient when scale is omitted");
  // the scale gradient of register rows takes its columns along one grid row
  if (grad_scale != nullptr && width > 4294967295LL / kBlock * kBlock)
    return fail(DPA4K_EINVAL, "RMSNorm scale gradient: feature dimension exceeds the launch limit");
  if (rows == 0) {
    if (grad_scale != nullptr) return zero_fill(grad_scale, width * sizeof(float), stream);
    return DPA4K_OK;
  }
  if (grad == nullptr || x == nullptr || inverse_rms == nullptr || grad_x == nullptr)
    return fail(DPA4K_EINVAL, "RMSNorm backward: null pointer");
  // Rows of more than 1,024 floats, unless whole aligned chunks, have always been
  // accepted without a workspace (the header asks for one): the columns kernel takes these.
  const bool wide = !fits_registers(width);
  const size_t needed = wide ? 0 : backward_workspace_bytes(rows, width);
  const bool chunked = width % 4 == 0 && aligned16(grad) && aligned16(x) && aligned16(grad_x) && aligned16(scale);
  const bool short_workspace = !static_scratch && (workspace == nullptr || workspace_bytes < needed);
  const bool columns = grad_scale != nullptr && (wide || (short_workspace && width > 1024 && !chunked));
  if (columns) {  // first: grad_x may be grad or x
    rmsnorm_scale_columns_kernel<<<launch_grid((width + 31) / 32, kColumnWaves * 64), kColumnWaves * 64, 0, stream>>>(
        grad, x, inverse_rms, grad_scale, rows, width);
    if (int s = launched("rmsnorm_scale_columns_kernel")) return s;
  }
  if (wide) {
    const dim3 grid = launch_grid((rows + kWaves - 1) / kWaves, kBlock);
    if (width % 4 != 0)
      rmsnorm_backward_wide_kernel<true><<<grid, kBlock, 0, stream>>>(grad, x, scale, inverse_rms, grad_x, rows, width);
    else
      rmsnorm_backward_wide_kernel<false><<<grid, kBlock, 0, stream>>>(grad, x, scale, inverse_rms, grad_x, rows, width);
    return launched("rmsnorm_backward_wide_kernel");
  }
  if (grad_scale == nullptr || columns) {
    // the register kernel strides over rows: one row of blocks covers any count
    const RowShape shape = shape_for(width);
    const int64_t wanted = row_blocks(shape, 1, rows);
    const int64_t limit = row_block_limit(kBlock);
    const unsigned int grid = static_cast<unsigned int>(wanted < limit ? wanted : limit);
    return launch_backward(grid, grad, x, scale, inverse_rms, grad_x, nullptr, rows, width, stream);
  }
  if (static_scratch) {
    if (needed > static_cast<size_t>(DPA4K_RMSNORM_NOALLOC_SCRATCH_BYTES))
      return fail(DPA4K_EINVAL,
                  "RMSNorm backward (no allocation): %zu bytes of column partials exceed the %d-byte scratch",
                  needed, DPA4K_RMSNORM_NOALLOC_SCRATCH_BYTES);
    float* address = nullptr;
    if (int s = scratch_for_stream(stream, address)) return s;
    workspace = address;
  } else if (short_workspace) {
    return fail(DPA4K_EWORKSPACE, "RMSNorm backward: workspace of %zu bytes is smaller than %zu", workspace_bytes,
                needed);
  }
  const unsigned int parts = partial_blocks(rows, width);
  float* partial = static_cast<float*>(workspace);
  if (int s = launch_backward(parts, grad, x, scale, inverse_rms, grad_x, partial, rows, width, stream)) return s;
  partial_columns_kernel<<<static_cast<unsigned int>((width + 63) / 64), kColumnWaves * 64, 0, stream>>>(
      partial, parts, width, grad_scale);
  return launched("partial_columns_kernel");
}

}  // namespace
}  // namespace dpa4k

using namespace dpa4k;

extern "C" int dpa4k_rmsnorm_forward(const float* x, const float* scale, float* y,
                                     float* inverse_rms, int64_t rows, int64_t width, float eps,
                                     dpa4k_stream_t stream_handle) {
  clear_error();
  if (rows < 0) return fail(DPA4K_EINVAL, "RMSNorm: negative row count");
  if (width <= 0) return fail(DPA4K_EINVAL, "RMSNorm feature dimension must be positive");
  if (!(eps > 0.0f) || !(eps < INFINITY))
    return fail(DPA4K_EINVAL, "RMSNorm eps must be a finite positive number");
  if (!grid_fits((rows + kWaves - 1) / kWaves, kBlock))
    return fail(DPA4K_EINVAL, "RMSNorm row count exceeds the launch limit");
  if (rows == 0) return DPA4K_OK;
  if (x == nullptr || y == nullptr || inverse_rms == nullptr)
    return fail(DPA4K_EINVAL, "RMSNorm: null pointer");
  hipStream_t stream = as_stream(stream_handle);
  if (fits_registers(width)) return launch_forward(x, scale, y, inverse_rms, rows, width, eps, stream);
  const dim3 grid = launch_grid((rows + kWaves - 1) / kWaves, kBlock);
  if (width % 4 != 0)
    rmsnorm_forward_wide_kernel<true><<<grid, kBlock, 0, stream>>>(x, scale, y, inverse_rms, rows, width, eps);
  else
    rmsnorm_forward_wide_kernel<false><<<grid, kBlock, 0, stream>>>(x, scale, y, inverse_rms, rows, width, eps);
  return launched("rmsnorm_forward_wide_kernel");
}

extern "C" size_t dpa4k_rmsnorm_backward_workspace_size(int64_t rows, int64_t width) {
  return backward_workspace_bytes(rows, width);
}

extern "C" int dpa4k_rmsnorm_backward(const float* grad, const float* x, const float* scale,
                                      const float* inverse_rms, float* grad_x, float* grad_scale,
                                      int64_t rows, int64_t width, void* workspace,
                                      size_t workspace_bytes, dpa4k_stream_t stream_handle) {
  clear_error();
  return rmsnorm_backward(grad, x, scale, inverse_rms, grad_x, grad_scale, rows, width, workspace,
                          workspace_bytes, false, as_stream(stream_handle));
}

extern "C" int dpa4k_rmsnorm_backward_noalloc(const float* grad, const float* x, const float* scale,
                                              const float* inverse_rms, float* grad_x, float* grad_scale,
                                              int64_t rows, int64_t width, dpa4k_stream_t stream_handle) {
  clear_error();
  return rmsnorm_backward(grad, x, scale, inverse_rms, grad_x, grad_scale, rows, width, nullptr, 0, true,
                          as_stream(stream_handle));
}
