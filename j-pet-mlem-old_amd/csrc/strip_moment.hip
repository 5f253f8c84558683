// Moment-table form of the strip MLEM iteration (kernels + host driver); the
// algorithm is described in strip_moment.hpp.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <string>
#include <tuple>
#include <type_traits>

#include "strip_band.hpp"
#include "strip_band_device.hpp"
#include "strip_device.hpp"
#include "strip_moment.hpp"

namespace strip {
namespace {

constexpr int R = kMomentRows;
constexpr int kGroup = 16;  // pairs of one 1 KiB group

// exp(v) ~ sum c_m v^m, m < NM, on |v| <= V: 8 terms on V = 1, 6 terms on
// V = 0.42.  The vertex may then lie reach * sigma_z from the line,
// 2 (3 / sqrt 2 + reach) reach = V, for |C u delta| <= V on every u of a
// 3-sigma run.  The relative error is a minimax one (linear programs over 4001
// Chebyshev points) weighted by the kernel value that v goes with, but by no
// less than 0.2, with its mean over a run's kernel values and over their
// products with u^2 held at zero (2e-10 with the rounded coefficients): the
// sigma derivatives are small differences of such sums.  At most 4.9e-7
// (6 terms 7.8e-7) at a run's far ends, 1e-7 (2.2e-7) for |v| < 0.3 V.
template <int NM>
struct ExpPoly;
template <>
struct ExpPoly<8> {
  static constexpr double reach = 0.2141;
  static constexpr float c[8] = {1.0f,           0.999999762f,   0.500000596f,
                                 0.166664779f,   0.0416531637f,  0.008342674f,
                                 0.00142612169f, 0.000193406566f};
};
template <>
struct ExpPoly<6> {
  static constexpr double reach = 0.0948;
  static constexpr float c[6] = {1.0f,         1.00000179f,  0.499997377f,
                                 0.166656896f, 0.0419010967f, 0.00834288821f};
};
constexpr double kRunHalf = 2.1213203435596424;  // 3 / sqrt 2, in sigma_z

typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));

// Half of the moments of one (row, side, position): one LDS access.  A cell
// (side, position) is two halves of 16 rows each, so the 16 lanes of a band
// read consecutive bytes.
template <int NM>
struct HalfCell {
  static constexpr int W = NM / 2;
  float w[W];
  __device__ static HalfCell load(const float* p) {
    HalfCell v;
    if constexpr (W == 4) {
      const float4v x = *reinterpret_cast<const float4v*>(p);
      v.w[0] = x.x;
      v.w[1] = x.y;
      v.w[2] = x.z;
      v.w[3] = x.w;
    } else {
      __builtin_memcpy(v.w, p, sizeof(v.w));
    }
    return v;
  }
  __device__ void store(float* p) const {
    if constexpr (W == 4)
      *reinterpret_cast<float4v*>(p) = float4v{w[0], w[1], w[2], w[3]};
    else
      __builtin_memcpy(p, w, sizeof(w));
  }
  __device__ static constexpr int half_words() { return R * W; }
  __device__ static constexpr int cell_words() { return 2 * R * W; }
  // Words of one side.  Rows of three words (6 terms) touch 16 of the 32
  // banks; 16 words more put the other side's rows on the other 16, so lane
  // groups working on opposite sides do not conflict.
  __device__ static int side_words(int positions) {
    return (positions + 1) * cell_words() + (W == 3 ? 16 : 0);
  }
};

// A bin's line: z = xc at the band's middle row, slope tc.  Bins count
// band-major, then the vertex, then tan.
struct BinLine {
  float xc, tc;
  int band;
};

__device__ inline BinLine bin_line(const MomentInstance& d, int bin) {
#pragma clang fp contract(off)
  const int jt = bin % d.nt, rest = bin / d.nt;
  BinLine l;
  l.xc = d.x_lo + ((float)(rest % d.nx) + 0.5f) * d.dx;
  l.tc = d.t_lo + ((float)jt + 0.5f) * d.dt;
  l.band = rest / d.nx;
  return l;
}

// The line on one row of its band and its column, evaluated alike in every
// kernel (contraction off): runs are stored relative to `column`.
struct LineRow {
  float x;     // z coordinate
  int column;  // nearest column, inside the columns a clamped bbox can hold
};

__device__ inline LineRow line_row(const DeviceGeometry& g, float xc, float tc,
                                   int row) {
#pragma clang fp contract(off)
  LineRow l;
  l.x = xc - tc * (((float)row - 0.5f * (R - 1)) * g.pixel_height);
  const float col = rintf((l.x - g.tl_z_half_w) * g.inv_pixel_width);
  l.column = (int)fminf(fmaxf(col, 0.0f), (float)max(g.n_z - 2, 0));
  return l;
}

// lane i of each row of 16 lanes, in all of them (a DPP operand)
template <int I>
__device__ inline float row_lane(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x150 + I,
                                      0xF, 0xF, true));
}
template <int I>
__device__ inline int row_lane(uint32_t v) {
  return __builtin_amdgcn_mov_dpp((int)v, 0x150 + I, 0xF, 0xF, true);
}

// Has a value computed before what follows in program order (an empty
// statement that claims to change it).
template <typename T>
__device__ inline void computed(T& v) {
  asm volatile("" : "+v"(v));
}

// Keeps LDS accesses of one wavefront in program order across lanes: the
// hardware executes them in order, so only the compiler must not move them.
__device__ inline void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// ---------------------------------------------------------------------------
// plan
// ---------------------------------------------------------------------------

struct PlanStats {
  unsigned long long pairs;
  int max_bands;
  int max_tan;        // bit pattern of a non-negative float
  int max_extent[2];  // widest box, most rows of a span-table slot
  int max_group[2];   // moment_groups_kernel: two bands, one
  int status;         // moment_pack_kernel
  int occupied;       // moment_marked_kernel
};

__device__ inline int box_bands(const uint2 box) {
  const int x0 = box.x & 0xffff, x1 = box.x >> 16;
  const int y0 = box.y & 0xffff, y1 = box.y >> 16;
  return (x1 > x0 && y1 > y0) ? (y1 - 1) / R - y0 / R + 1 : 0;
}

// What the choice between the forms and the sizes of either plan depend on.
__global__ __launch_bounds__(256) void moment_stats_kernel(
    const uint2* __restrict__ box, const float4* __restrict__ a, int64_t n,
    PlanStats* __restrict__ stats) {
  unsigned long long pairs = 0;
  int most[4] = {0, 0, 0, 0};  // bands, |tan| as bits, box width, slot rows
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
       e += (int64_t)gridDim.x * blockDim.x) {
    const uint2 b = box[e];
    const int c = box_bands(b);
    pairs += (unsigned long long)c;
    most[0] = max(most[0], c);
    most[2] = max(most[2], box_width(b.x));
    most[3] = max(most[3], box_slot_rows(b.y));
    // (a NaN stays out: such an event's box is empty or its bin is clamped)
    if (c)
      most[1] =
          max(most[1], __builtin_bit_cast(int, fmaxf(0.0f, fabsf(a[e].z))));
  }
  for (int o = 32; o > 0; o >>= 1) {
    pairs += __shfl_xor(pairs, o);
#pragma unroll
    for (int i = 0; i < 4; ++i) most[i] = max(most[i], __shfl_xor(most[i], o));
  }
  __shared__ unsigned long long sp[4];
  __shared__ int sm[4][4];
  if ((threadIdx.x & 63) == 0) {
    const int w = threadIdx.x >> 6;
    sp[w] = pairs;
#pragma unroll
    for (int i = 0; i < 4; ++i) sm[w][i] = most[i];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) {
      pairs += sp[w];
#pragma unroll
      for (int i = 0; i < 4; ++i) most[i] = max(most[i], sm[w][i]);
    }
    atomicAdd(&stats->pairs, pairs);
    atomicMax(&stats->max_bands, most[0]);
    atomicMax(&stats->max_tan, most[1]);
    atomicMax(&stats->max_extent[0], most[2]);
    atomicMax(&stats->max_extent[1], most[3]);
  }
}

// The most pairs, among every step-th event's, of a group that the row-band
// lists cut their tasks from: a band (two for the forward lists) and the bucket
// of columns in which a pair's runs begin, about half_run columns and the line's
// shear over half a band left of the vertex.  One workgroup counts them in LDS
// (in global memory the additions to the same few words, from all over the card,
// take 0.1 to 0.5 ms); grids of more groups than kGroupWords share words.
constexpr int kBucket = 8;
constexpr int kGroupWords = 1 << 14;
constexpr int kSampled = 1 << 12;

__global__ __launch_bounds__(1024) void moment_groups_kernel(
    DeviceGeometry g, const uint2* __restrict__ box,
    const float4* __restrict__ a, int64_t n, int64_t step, int buckets,
    int words, float half_run, PlanStats* __restrict__ stats) {
  __shared__ int group[kGroupWords];
  for (int i = threadIdx.x; i < words; i += 1024) group[i] = 0;
  __syncthreads();
  for (int64_t e = threadIdx.x * step; e < n; e += 1024 * step) {
    const uint2 b = box[e];
    const int c = box_bands(b);
    if (!c) continue;
    const float4 ev = a[e];  // z, y, tan
    const float shear = 0.5f * R * g.pixel_height * ev.z;
    const float lo = (float)(b.x & 0xffff), hi = (float)(b.x >> 16) - 1.0f;
    for (int k = 0; k < c; ++k) {
      const int band = (int)(b.y & 0xffff) / R + k;
      const float y = g.tl_y_half_h - ((float)band + 0.5f) * R * g.pixel_height;
      const float z = ev.x + ev.z * (y - ev.y) - fabsf(shear) - g.tl_z_half_w;
      const float col = fminf(fmaxf(z * g.inv_pixel_width - half_run, lo), hi);
      atomicAdd(&group[(band * buckets + (int)col / kBucket) % words], 1);
    }
  }
  __syncthreads();
  int two = 0, one = 0;
  for (int i = threadIdx.x; i < words; i += 1024) {
    const int c = group[i];
    const int next = i + buckets < words ? group[i + buckets] : 0;
    one = max(one, c);
    if (!(i / buckets & 1)) two = max(two, c + next);
  }
  for (int o = 32; o > 0; o >>= 1) {
    two = max(two, __shfl_xor(two, o));
    one = max(one, __shfl_xor(one, o));
  }
  if ((threadIdx.x & 63) == 0) {
    atomicMax(&stats->max_group[0], two);
    atomicMax(&stats->max_group[1], one);
  }
}

__global__ __launch_bounds__(256) void fill_words_kernel(uint32_t* p, int64_t n,
                                                         uint32_t v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

__device__ inline int tan_bin(const MomentInstance& d, float t) {
  const float j = floorf((t - d.t_lo) / d.dt);
  return (int)fminf(fmaxf(j, 0.0f), (float)(d.nt - 1));
}

// event order: eighths of a tan bin, then the band of the bbox top, then the
// vertex line's crossing of the axis y = 0: the pairs of a bin then come from
// short runs of nearly consecutive records, so that the wavefronts' accesses to
// the per-record arrays (partial sums, weights) share cache lines.  (With
// whole tan bins and the bbox column instead, neighbouring pairs of a bin lay
// 17 records apart, and their partial sums cost half the forward pass.)
__global__ __launch_bounds__(256) void moment_order_kernel(
    MomentInstance d, const uint2* __restrict__ box,
    const float4* __restrict__ a, int64_t n, uint32_t* __restrict__ keys,
    int* __restrict__ values) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const float4 ev = a[e];  // z, y, tan
  const float t = floorf((ev.z - d.t_lo) * (8.0f / d.dt));
  const float x = (ev.x - ev.z * ev.y - d.x_lo) / ((float)d.nx * d.dx);
  keys[e] = ((uint32_t)fminf(fmaxf(t, 0.0f), 511.0f) << 23) |
            (((box[e].y & 0xffff) / R) << 12) |
            (uint32_t)(fminf(fmaxf(x, 0.0f), 1.0f) * 4095.0f);
  values[e] = (int)e;
}

// records in that order, and their band counts
__global__ __launch_bounds__(256) void moment_records_kernel(
    EventSoA ev, const int* __restrict__ order, int64_t n,
    BandRecord* __restrict__ rec, int* __restrict__ counts) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int e = order[i];
  const float4 a = ev.a[e], b = ev.b[e], c = ev.c[e];
  const uint2 box = ev.box[e];
  BandRecord r;
  r.cz = a.x;
  r.cy = a.y;
  r.A = b.x;
  r.B = b.y;
  r.P = c.x;
  r.Q0 = c.y;
  r.bx = box.x;
  r.by = box.y;
  rec[i] = r;
  counts[i] = box_bands(box);
}

// The bin of a pair: the line z = cz + t (y - cy) at the middle of band b.
__device__ inline int pair_bin(const MomentInstance& d, float cz, float cy,
                               float t, int jt, int b) {
  const float yc = d.g.tl_y_half_h -
                   ((float)(b * R) + 0.5f * (R - 1)) * d.g.pixel_height;
  const float x = cz + t * (yc - cy);
  const float f = floorf((x - d.x_lo) / d.dx);
  const int ix = (int)fminf(fmaxf(f, 0.0f), (float)(d.nx - 1));
  return (b * d.nx + ix) * d.nt + jt;
}

// occupied[bin] = 1 for every bin that has pairs
__global__ __launch_bounds__(256) void moment_mark_kernel(
    MomentInstance d, const uint2* __restrict__ box,
    const float4* __restrict__ a, int64_t n, uint8_t* __restrict__ occupied) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int c = box_bands(box[i]);
  if (!c) return;
  const float4 ev = a[i];  // z, y, tan
  const int jt = tan_bin(d, ev.z);
  const int b0 = (int)(box[i].y & 0xffff) / R;
  for (int k = 0; k < c; ++k)
    occupied[pair_bin(d, ev.x, ev.y, ev.z, jt, b0 + k)] = 1;
}

// *total += occupied bins (four to a word)
__global__ __launch_bounds__(256) void moment_marked_kernel(
    const uint32_t* __restrict__ occupied, int n_words,
    int* __restrict__ total) {
  int c = 0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n_words;
       i += gridDim.x * blockDim.x)
    c += __popc(occupied[i]);
  c = wave_sum_int(c);
  if ((threadIdx.x & 63) == 0 && c) atomicAdd(total, c);
}

// (bin, record) of every pair
__global__ __launch_bounds__(256) void moment_emit_kernel(
    MomentInstance d, const BandRecord* __restrict__ rec,
    const int* __restrict__ counts, const int* __restrict__ offsets, int64_t n,
    uint32_t* __restrict__ keys, int* __restrict__ values) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int c = counts[i];
  if (!c) return;
  const BandRecord r = rec[i];
  const float t = -r.B * d.g.inv_2c;
  const int jt = tan_bin(d, t);
  const int b0 = (int)(r.by & 0xffff) / R;
  const int at = offsets[i];
  for (int k = 0; k < c; ++k) {
    keys[at + k] = (uint32_t)pair_bin(d, r.cz, r.cy, t, jt, b0 + k);
    values[at + k] = (int)i;
  }
}

// first / end pair of every bin that has pairs
__global__ __launch_bounds__(256) void moment_bins_kernel(
    const uint32_t* __restrict__ keys, int64_t n, int* __restrict__ first,
    int* __restrict__ end) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t k = keys[i];
  if (i == 0 || keys[i - 1] != k) first[k] = (int)i;
  if (i == n - 1 || keys[i + 1] != k) end[k] = (int)i + 1;
}

// pieces of `chunk` pairs each bin is cut into (0 at n_bins)
__global__ __launch_bounds__(256) void moment_piece_count_kernel(
    const int* __restrict__ first, const int* __restrict__ end, int n_bins,
    int chunk, int* __restrict__ counts) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i <= n_bins)
    counts[i] = i < n_bins ? (end[i] - first[i] + chunk - 1) / chunk : 0;
}

// the 16-pair groups of every bin, and their first pairs
__global__ __launch_bounds__(256) void moment_group_emit_kernel(
    MomentInstance d, const int* __restrict__ first,
    const int* __restrict__ end, int n_bins, const int* __restrict__ group_of,
    MomentGroup* __restrict__ groups, int* __restrict__ group_pair) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_bins || first[i] == end[i]) return;
  const BinLine line = bin_line(d, i);
  int k = group_of[i];
  for (int p = first[i]; p < end[i]; p += kGroup, ++k) {
    groups[k] = MomentGroup{line.xc, line.tc, i, min(kGroup, end[i] - p)};
    group_pair[k] = p;
  }
}

// Blocks of bins for merged tasks: x_block vertex bins of one band with all
// their tan bins, whose groups lie together.  counts[b] = tasks of at most
// `chunk` groups in block b (0 at n_blocks).
__device__ inline int2 block_groups(const MomentInstance& d, int block,
                                    int x_block, int n_x_blocks,
                                    const int* __restrict__ group_of) {
  const int band = block / n_x_blocks, q = block % n_x_blocks;
  const int lo = (band * d.nx + q * x_block) * d.nt;
  const int hi = (band * d.nx + min((q + 1) * x_block, d.nx)) * d.nt;
  return make_int2(group_of[lo], group_of[hi]);
}

__global__ __launch_bounds__(256) void moment_block_count_kernel(
    MomentInstance d, const int* __restrict__ group_of, int n_blocks,
    int x_block, int n_x_blocks, int chunk, int* __restrict__ counts) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i > n_blocks) return;
  int c = 0;
  if (i < n_blocks) {
    const int2 g = block_groups(d, i, x_block, n_x_blocks, group_of);
    c = (g.y - g.x + chunk - 1) / chunk;
  }
  counts[i] = c;
}

// Merged tasks of a block: its groups in nearly equal parts, with the first
// column any of the block's lines can reach (max_shear: the most a line moves
// from the band's middle row to its ends).
__global__ __launch_bounds__(256) void moment_block_emit_kernel(
    MomentInstance d, const int* __restrict__ group_of, int n_blocks,
    int x_block, int n_x_blocks, int chunk, float max_shear,
    const int* __restrict__ offsets, MomentTask* __restrict__ tasks) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_blocks) return;
  const int2 g = block_groups(d, i, x_block, n_x_blocks, group_of);
  const int total = g.y - g.x, parts = (total + chunk - 1) / chunk;
  const float x = d.x_lo + (float)((i % n_x_blocks) * x_block) * d.dx -
                  max_shear;
  const float col = floorf((x - d.g.tl_z_half_w) * d.g.inv_pixel_width);
  const int first =
      (int)fminf(fmaxf(col, 0.0f), (float)max(d.g.n_z - 2, 0)) - d.positions;
  for (int k = 0; k < parts; ++k) {
    const int lo = g.x + (int)((int64_t)total * k / parts);
    const int hi = g.x + (int)((int64_t)total * (k + 1) / parts);
    MomentTask t;
    t.xc = t.tc = 0.0f;  // (each group has its own)
    t.band = i / n_x_blocks;
    t.instance = 0;
    t.group = lo;
    t.pairs = hi - lo;  // groups
    t.first_column = first;
    t.pad = 0;
    tasks[offsets[i] + k] = t;
  }
}

// tasks of a bin: its groups in nearly equal parts of at most `chunk` pairs
__global__ __launch_bounds__(256) void moment_task_emit_kernel(
    MomentInstance d, const int* __restrict__ first, const int* __restrict__ end, int n_bins,
    int chunk, const int* __restrict__ group_of,
    const int* __restrict__ offsets, MomentTask* __restrict__ tasks) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_bins) return;
  const int total = end[i] - first[i];
  const int groups = (total + kGroup - 1) / kGroup;
  const int parts = (total + chunk - 1) / chunk;
  const BinLine line = bin_line(d, i);
  for (int k = 0; k < parts; ++k) {
    const int lo = (int)((int64_t)groups * k / parts);
    const int hi = (int)((int64_t)groups * (k + 1) / parts);
    MomentTask t;
    t.xc = line.xc;
    t.tc = line.tc;
    t.band = line.band;
    t.instance = 0;
    t.group = group_of[i] + lo;
    t.pairs = min(total, hi * kGroup) - lo * kGroup;
    t.first_column = t.pad = 0;
    tasks[offsets[i] + k] = t;
  }
}

// The pairs' data in groups of 16 pairs of one bin, 1 KiB each, laid out as a
// wavefront reads it: one 16-byte load per lane holds four steps of four pairs
// (pair 4 s + g belongs to lane group g = lane / 16 of step s).  With i =
// lane % 16:
//   word s / 2, lanes i = 8 (s % 2) + k: field k of the pair of step s:
//     cz, cy, tan, 4 id sec^2 (times the exp2 scale), P', Q0' of the record,
//     the record's index and the index of its partial sum for this band;
//   half-word s of words 2 and 3: the run of band row i: a | b << 8, a columns
//     left of the line's column and b from it on, or, for a run that misses
//     the line's column, 0x8000 | n << 8 | (offset + positions / 2), n
//     columns, the first at the line's column + offset (both parts at most
//     `positions`, so that either form addresses cells that exist).
// Missing pairs of a last group repeat the bin's last pair with empty runs and
// the index of a spare partial sum, so a wavefront need not tell them apart.
__global__ __launch_bounds__(256) void moment_pack_kernel(
    MomentInstance d, const BandRecord* __restrict__ rec,
    const MomentGroup* __restrict__ groups,
    const int* __restrict__ group_pair, const int* __restrict__ values,
    int n_groups, int n_records, int spare,
    uint4* __restrict__ blocks, int* __restrict__ status) {
  __shared__ uint32_t words[kGroup * 16];
  const int pair = threadIdx.x >> 4, row = threadIdx.x & 15;
  const int step = pair >> 2, grp = pair & 3;
  for (int k = blockIdx.x; k < n_groups; k += gridDim.x) {
    const MomentGroup group = groups[k];
    const int p = group_pair[k] + min(pair, group.pairs - 1);
    const bool missing = pair >= group.pairs;
    uint32_t word = 0, field = 0;
    const int e = values[p];
    const BandRecord r = rec[e];
    int x0, x1, y0, y1;
    record_box(r, x0, x1, y0, y1);
    const int band = group.bin / (d.nt * d.nx);
    const LineRow l = line_row(d.g, group.xc, group.tc, row);
    const RowSpan s = row_span(d.g, r.cz, r.cy, r.A, r.B, r.P, r.Q0, x0, x1,
                               y0, y1, band * R + row);
    if (s.n > 0 && !missing) {
      const int a = l.column - s.lo, b = s.lo + s.n - l.column;
      const int off = s.lo - l.column + d.positions / 2;
      if (a >= 0 && b >= 0 && a <= d.positions && b <= d.positions)
        word = (uint32_t)(a | (b << 8));
      else if (s.n <= d.positions && off >= 0 && off <= d.positions)
        word = 0x8000u | ((uint32_t)s.n << 8) | (uint32_t)off;
      else
        *status = 1;  // does not fit: the host falls back
    }
    const float t = -r.B * d.g.inv_2c;
    const float ad = 4.0f * d.g.inv_pow_sigma_dl * __builtin_fmaf(t, t, 1.0f);
    switch (row) {
      case 0: field = __builtin_bit_cast(uint32_t, r.cz); break;
      case 1: field = __builtin_bit_cast(uint32_t, r.cy); break;
      case 2: field = __builtin_bit_cast(uint32_t, t); break;
      case 3: field = __builtin_bit_cast(uint32_t, ad * kExp2Scale); break;
      case 4: field = __builtin_bit_cast(uint32_t, r.P); break;
      case 5: field = __builtin_bit_cast(uint32_t, r.Q0); break;
      case 6: field = (uint32_t)e; break;
      case 7:
        field = (uint32_t)(missing ? spare
                                   : (band - y0 / R) * n_records + e);
        break;
      default: break;
    }
    __syncthreads();  // the previous group has been written out
    if (row < 8)
      words[(grp * 16 + (step & 1) * 8 + row) * 4 + (step >> 1)] = field;
    reinterpret_cast<uint16_t*>(words)[(grp * 16 + row) * 8 + 4 + step] =
        (uint16_t)word;
    __syncthreads();
    if (threadIdx.x < 64)
      blocks[(int64_t)k * 64 + threadIdx.x] =
          reinterpret_cast<const uint4*>(words)[threadIdx.x];
  }
}

// ---------------------------------------------------------------------------
// iteration
// ---------------------------------------------------------------------------

// Row terms of a pair on this lane.
struct RowTerms {
  float delta;   // vertex - line
  float qa;      // exponent at the vertex
  float pre;     // row prefactor
  float w;       // pre exp2(exponent on the line): the polynomial's factor
  uint32_t run;  // run word
};

// of step S of a group
template <int S>
__device__ inline RowTerms row_terms(const uint4v& v, float y, float y2,
                                     float x, float qc) {
  constexpr int F = 8 * (S & 1);
  const uint32_t fields = S < 2 ? v.x : v.y, runs = S < 2 ? v.z : v.w;
  const float f = __builtin_bit_cast(float, fields);
  RowTerms r;
  const float dy = y - row_lane<F + 1>(f);
  r.delta = __builtin_fmaf(row_lane<F + 2>(f), dy, row_lane<F>(f) - x);
  r.qa = row_lane<F + 3>(f) * dy * dy;
  r.pre = __builtin_amdgcn_rsqf(
      __builtin_fmaf(row_lane<F + 4>(f), y2, row_lane<F + 5>(f)));
  const float q = __builtin_fmaf(qc * r.delta, r.delta, r.qa);
  r.w = r.pre * __builtin_amdgcn_exp2f(q);
  r.run = (S & 1) ? runs >> 16 : runs & 0xffff;
  return r;
}

// Whether a lane's row of the group's four pairs has a run that misses the
// line's column.
__device__ inline bool any_direct(const uint4v& v) {
  return ((v.z | v.w) & 0x80008000u) != 0;
}

// Whether any lane of the wavefront has it: the row terms read their fields
// from other lanes, so branches around them are taken by whole wavefronts.
__device__ inline bool wave_any(bool v) {
  return __builtin_amdgcn_ballot_w64(v) != 0;
}

// Forward projection of one task: the workgroup tabulates the image around
// the bin's line, then every wavefront step takes four pairs, 16 lanes each.
// Bound by VALU issue (58 instructions per step of 64 rows, whatever the runs'
// lengths).  2e7 events, 1000 x 400 at 1 mm: 3.6 ms (6.4 ms while neighbouring
// pairs' partial sums shared no cache lines), against 12.4 ms for the kernel that
// walks the runs' pixels (33 columns per row, 6.9 lane operations each).
template <int NM, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void moment_forward_kernel(
    const MomentInstance* __restrict__ desc, const MomentTask* __restrict__ tasks) {
  using Half = HalfCell<NM>;
  constexpr int W = Half::W, HALF = Half::half_words(),
                CELL = Half::cell_words();
  extern __shared__ float4v table4[];
  float* const table = reinterpret_cast<float*>(table4);
  const MomentTask task = tasks[blockIdx.x];
  const MomentInstance& d = desc[task.instance];
  const int lane = threadIdx.x & 63;
  const int row = lane & (R - 1);
  const int grp = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int P = d.positions;
  const int n_y = d.g.n_y, n_z = d.g.n_z;
  const float w_px = d.g.pixel_width;
  const int iy = task.band * R + row;
  const LineRow l = line_row(d.g, task.xc, task.tc, row);
  const float qc = d.g.C * kExp2Scale;
  const float* __restrict__ rhoT = d.rhoT;
  const int n_here = task.pairs;
  const uint4v* __restrict__ base =
      reinterpret_cast<const uint4v*>(d.blocks) + (int64_t)task.group * 64;
  const int last = (n_here - 1) / kGroup;
  uint4v next = gload(base + min(wave, last) * 64 + lane);
  {
    // thread = (row, side, MG consecutive moments); cell k of a side holds
    // the sums over its first k columns outward from the line
    constexpr int MG = (NM + 2 * WAVES - 1) / (2 * WAVES);
    static_assert(W % MG == 0, "a thread's moments stay in one half");
    const int side = grp & 1;
    const int m0 = (int)(threadIdx.x >> 5) * MG;
    if (m0 < NM) {
      float* cell = table + side * Half::side_words(P) + (m0 / W) * HALF +
                    row * W + m0 % W;
      float acc[MG], cm[MG];
#pragma unroll
      for (int i = 0; i < MG; ++i) {
        acc[i] = 0.0f;
        cm[i] = ExpPoly<NM>::c[m0 + i];
        cell[i] = 0.0f;
      }
      const int dir = side ? 1 : -1;
      int col = side ? l.column : l.column - 1;
      const bool row_in = iy < n_y;
      const float du = side ? w_px : -w_px;
      const float inv_s = d.inv_s;
      const float u0 = __builtin_fmaf((float)col, w_px, d.g.tl_z_half_w) - l.x;
      // eight columns' pixels are in flight together
      for (int k0 = 0; k0 < P; k0 += 8) {
        float rho[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int x = col + k * dir;
          const bool in = row_in && x >= 0 && x < n_z;
          const float v = gload(rhoT + (in ? (int64_t)x * n_y + iy : 0));
          rho[k] = in ? v : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          if (k0 + k >= P) break;
          cell += CELL;
          const float u = __builtin_fmaf((float)(k0 + k), du, u0);
          const float v = u * inv_s;
          float t = __builtin_amdgcn_exp2f(qc * u * u) * rho[k];
          // (u / s)^m0
          if constexpr (MG < NM) {
            const float v2 = v * v;
            if (MG % 2 == 1 && (m0 & 1)) t *= v;
            if (MG % 4 != 0 && (m0 & 2)) t *= v2;
            if (m0 & 4) t *= v2 * v2;
          }
#pragma unroll
          for (int i = 0; i < MG; ++i) {
            acc[i] = __builtin_fmaf(cm[i], t, acc[i]);
            cell[i] = acc[i];
            t *= v;
          }
        }
        col += 8 * dir;
      }
    }
  }
  __syncthreads();
  const float y = pixel_center_y(d.g, iy);
  const float y2 = y * y;
  const float cs = d.cs;
  float* __restrict__ partial = d.partial;
  const float* const left = table + row * W;
  const int side_words = Half::side_words(P);
  const bool odd = grp & 1;
  auto row_sum = [&](auto tag, const uint4v& v) {
    constexpr int S = decltype(tag)::value;
    const RowTerms r = row_terms<S>(v, y, y2, l.x, qc);
    const float eta = cs * r.delta;
    const int a = (int)(r.run & 0xff), b = (int)((r.run >> 8) & 0x7f);
    const float* pl = left + a * CELL;
    const float* pr = left + b * CELL + side_words;
    if (W == 3) {  // opposite sides first in neighbouring lane groups
      const float* first = odd ? pr : pl;
      pr = odd ? pl : pr;
      pl = first;
    }
    const Half l0 = Half::load(pl), l1 = Half::load(pl + HALF);
    const Half r0 = Half::load(pr), r1 = Half::load(pr + HALF);
    float t = l1.w[W - 1] + r1.w[W - 1];
#pragma unroll
    for (int i = W - 2; i >= 0; --i)
      t = __builtin_fmaf(t, eta, l1.w[i] + r1.w[i]);
#pragma unroll
    for (int i = W - 1; i >= 0; --i)
      t = __builtin_fmaf(t, eta, l0.w[i] + r0.w[i]);
    return t * r.w;
  };
  // a run pixel by pixel
  auto walk = [&](auto tag, const uint4v& v, float s) {
    constexpr int S = decltype(tag)::value;
    const RowTerms r = row_terms<S>(v, y, y2, l.x, qc);
    const bool direct = r.run >= 0x8000u;
    if (!direct && __builtin_fabsf(s) < __builtin_inff()) return s;
    const int a = (int)(r.run & 0xff), b = (int)((r.run >> 8) & 0x7f);
    const int n = direct ? b : a + b;
    const int col = l.column + (direct ? a - P / 2 : -a);
    float dz = (__builtin_fmaf((float)col, w_px, d.g.tl_z_half_w) - l.x) -
               r.delta;
    float acc = 0.0f;
    const float* src = rhoT + (int64_t)col * n_y + iy;
    for (int k = 0; k < n; ++k) {
      acc = __builtin_fmaf(
          __builtin_amdgcn_exp2f(__builtin_fmaf(qc * dz, dz, r.qa)),
          gload(src), acc);
      src += n_y;
      dz += w_px;
    }
    return n > 0 ? r.pre * acc : 0.0f;
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  using S2 = std::integral_constant<int, 2>;
  using S3 = std::integral_constant<int, 3>;
  for (int k = wave; k <= last; k += WAVES) {
    const uint4v cur = next;
    next = gload(base + min(k + WAVES, last) * 64 + lane);
    // a group's four steps at once; a last group's empty steps are left out
    const int steps = min((n_here - k * kGroup + 3) / 4, 4);
    float s0 = row_sum(S0{}, cur), s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
    if (steps == 4) {
      s1 = row_sum(S1{}, cur);
      s2 = row_sum(S2{}, cur);
      s3 = row_sum(S3{}, cur);
    } else {
      if (steps > 1) s1 = row_sum(S1{}, cur);
      if (steps > 2) s2 = row_sum(S2{}, cur);
    }
    // runs that miss the line's column, and rows whose sum is not finite (an
    // infinite pixel times powers of both signs)
    if (wave_any(any_direct(cur) ||
                 !(__builtin_fabsf(s0) + __builtin_fabsf(s1) +
                       __builtin_fabsf(s2) + __builtin_fabsf(s3) <
                   __builtin_inff()))) {
      s0 = walk(S0{}, cur, s0);
      s1 = walk(S1{}, cur, s1);
      s2 = walk(S2{}, cur, s2);
      s3 = walk(S3{}, cur, s3);
    }
    s0 = group_total<R>(s0);
    s1 = group_total<R>(s1);
    s2 = group_total<R>(s2);
    s3 = group_total<R>(s3);
    // the next group is waited for here, not behind this group's stores
    computed(next);
    // lanes 7 and 15 of a row hold the partials' indices
    if ((row & 7) == 7) {
      gstore(partial + (int)cur.x, row == 7 ? s0 : s1);
      gstore(partial + (int)cur.y, row == 7 ? s2 : s3);
    }
  }
}

// Sums of one pair for the sigma derivatives, as band_moments_kernel forms
// them: out[stride * (partial index) + {0, 1, 2}] =
//   sum K x, sum K x Q, sum K x (w - Qd)   over the band's pixels,
// for the column-major image xT.  The same tables and steps as the forward
// projection with ten plain moments M_m = sum x exp(-(C/2) u^2) (u / s)^m:
//   sum x exp(-(C/2)(u - delta)^2) (u / s)^k ~ sum_m c_m eta^m M_{m+k},
// k = 0, 1, 2, and Q = C (u - delta)^2 + Qd.  118 VALU instructions per step
// of 64 rows.  2e6 events, 512 x 256 at 1 mm, sigma_z 14 mm: 1.4 ms, against
// 4.8 ms for the kernel that walks the runs' pixels.
constexpr int kGradMoments = 10;
constexpr int kGradCell = R * kGradMoments;

// word of moment m of a row in a cell: rows of four, four and two moments
__device__ inline int grad_word(int m, int row) {
  return m < 8 ? (m >> 2) * (R * 4) + row * 4 + (m & 3)
               : R * 8 + row * 2 + (m & 1);
}

template <int WAVES>
__global__ __launch_bounds__(64 * WAVES) void moment_gradient_kernel(
    const MomentInstance* __restrict__ desc, const MomentTask* __restrict__ tasks,
    const float* __restrict__ xT, int stride, float* __restrict__ out) {
  extern __shared__ float4v table4[];
  float* const table = reinterpret_cast<float*>(table4);
  const MomentTask task = tasks[blockIdx.x];
  const MomentInstance& d = desc[task.instance];
  const int lane = threadIdx.x & 63;
  const int row = lane & (R - 1);
  const int grp = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int P = d.positions;
  const int n_y = d.g.n_y, n_z = d.g.n_z;
  const float w_px = d.g.pixel_width;
  const int iy = task.band * R + row;
  const LineRow l = line_row(d.g, task.xc, task.tc, row);
  const float C = d.g.C;
  // (the part of C * scale that qc rounds off: with it left out every Q is off
  // by the same factor, up to 6e-8, which the sums over all events show)
  const float qc = C * kExp2Scale;
  const float qc_low =
      (float)((double)C * (-0.5 * 1.4426950408889634) - (double)qc);
  const float inv_s = d.inv_s;
  const int n_here = task.pairs;
  const uint4v* __restrict__ base =
      reinterpret_cast<const uint4v*>(d.blocks) + (int64_t)task.group * 64;
  const int last = (n_here - 1) / kGroup;
  uint4v next = gload(base + min(wave, last) * 64 + lane);
  {
    // thread = (row, side, two consecutive moments)
    const int side = grp & 1;
    const int dir = side ? 1 : -1;
    const int col0 = side ? l.column : l.column - 1;
    const bool row_in = iy < n_y;
    const float du = side ? w_px : -w_px;
    const float u0 = __builtin_fmaf((float)col0, w_px, d.g.tl_z_half_w) - l.x;
    for (int m0 = (int)(threadIdx.x >> 5) * 2; m0 < kGradMoments;
         m0 += 4 * WAVES) {
      float* cell = table + side * (P + 1) * kGradCell + grad_word(m0, row);
      float a0 = 0.0f, a1 = 0.0f;
      cell[0] = 0.0f;
      cell[1] = 0.0f;
      for (int k0 = 0; k0 < P; k0 += 8) {
        float x[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int c = col0 + (k0 + k) * dir;
          const bool in = row_in && c >= 0 && c < n_z;
          const float v = gload(xT + (in ? (int64_t)c * n_y + iy : 0));
          x[k] = in ? v : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          if (k0 + k >= P) break;
          cell += kGradCell;
          const float u = __builtin_fmaf((float)(k0 + k), du, u0);
          const float v = u * inv_s, v2 = v * v, v4 = v2 * v2;
          const float u2 = u * u;
          float t = __builtin_amdgcn_exp2f(
                        __builtin_fmaf(qc, u2, qc_low * u2)) * x[k];
          if (m0 & 2) t *= v2;
          if (m0 & 4) t *= v4;
          if (m0 & 8) t *= v4 * v4;
          a0 += t;
          a1 = __builtin_fmaf(t, v, a1);
          cell[0] = a0;
          cell[1] = a1;
        }
      }
    }
  }
  __syncthreads();
  const float y = pixel_center_y(d.g, iy);
  const float y2 = y * y;
  const float cs = d.cs;
  const float s2 = C / (inv_s * inv_s);  // C s^2
  const float w_row =
      __builtin_fmaf(y2, 1.0f / (d.g.radius * d.g.radius), 1.0f);
  const float* const left = table + grad_word(0, row);
  const int right_words = (P + 1) * kGradCell;
  struct Sums {
    float m[3];
  };
  auto step = [&](auto tag, const uint4v& v) {
    constexpr int S = decltype(tag)::value;
    const RowTerms r = row_terms<S>(v, y, y2, l.x, qc);
    const float eta = cs * r.delta;
    const int a = (int)(r.run & 0xff), b = (int)((r.run >> 8) & 0x7f);
    const float* pl = left + a * kGradCell;
    const float* pr = left + b * kGradCell + right_words;
    typedef float float2v __attribute__((ext_vector_type(2)));
    const float4v t0 = *reinterpret_cast<const float4v*>(pl) +
                       *reinterpret_cast<const float4v*>(pr);
    const float4v t1 = *reinterpret_cast<const float4v*>(pl + R * 4) +
                       *reinterpret_cast<const float4v*>(pr + R * 4);
    const float2v t2 =
        *reinterpret_cast<const float2v*>(pl + R * 8 - row * 2) +
        *reinterpret_cast<const float2v*>(pr + R * 8 - row * 2);
    const float M[kGradMoments] = {t0.x, t0.y, t0.z, t0.w, t1.x,
                                   t1.y, t1.z, t1.w, t2.x, t2.y};
    float e0 = 0.0f, e1 = 0.0f, e2 = 0.0f, power = 1.0f;
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const float c = ExpPoly<8>::c[m] * power;
      e0 = __builtin_fmaf(c, M[m], e0);
      e1 = __builtin_fmaf(c, M[m + 1], e1);
      e2 = __builtin_fmaf(c, M[m + 2], e2);
      power *= eta;
    }
    // C s^2 sum (u / s - delta / s)^2
    const float ds = r.delta * inv_s;
    float k0 = e0 * r.w;
    float kq = s2 * __builtin_fmaf(ds, __builtin_fmaf(ds, e0, -2.0f * e1), e2) *
               r.w;
    const float qd = r.qa * (1.0f / kExp2Scale);
    const bool direct = r.run >= 0x8000u;
    if (direct || !(__builtin_fabsf(k0) + __builtin_fabsf(kq) <
                    __builtin_inff())) {
      const int n = direct ? b : a + b;
      const int col = l.column + (direct ? a - P / 2 : -a);
      float dz = (__builtin_fmaf((float)col, w_px, d.g.tl_z_half_w) - l.x) -
                 r.delta;
      float acc = 0.0f, accq = 0.0f;
      const float* src = xT + (int64_t)col * n_y + iy;
      for (int k = 0; k < n; ++k) {
        const float z = dz * dz;
        const float t =
            __builtin_amdgcn_exp2f(
                __builtin_fmaf(qc, z, __builtin_fmaf(qc_low, z, r.qa))) *
            gload(src);
        acc += t;
        accq = __builtin_fmaf(t, C * z, accq);
        src += n_y;
        dz += w_px;
      }
      k0 = n > 0 ? r.pre * acc : 0.0f;
      kq = n > 0 ? r.pre * accq : 0.0f;
    }
    // w = Q0' (1 + y^2 / R^2) pre^2
    const float f = __builtin_bit_cast(float, S < 2 ? v.x : v.y);
    const float w = row_lane<8 * (S & 1) + 5>(f) * w_row * r.pre * r.pre;
    Sums o;
    o.m[0] = group_total<R>(k0);
    o.m[1] = group_total<R>(__builtin_fmaf(k0, qd, kq));
    o.m[2] = group_total<R>(k0 * (w - qd));
    return o;
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  using S2 = std::integral_constant<int, 2>;
  using S3 = std::integral_constant<int, 3>;
  for (int k = wave; k <= last; k += WAVES) {
    const uint4v cur = next;
    next = gload(base + min(k + WAVES, last) * 64 + lane);
    // (a last group's empty steps are left out)
    const int steps = min((n_here - k * kGroup + 3) / 4, 4);
    Sums s[4] = {};
    s[0] = step(S0{}, cur);
    if (steps > 1) s[1] = step(S1{}, cur);
    if (steps > 2) s[2] = step(S2{}, cur);
    if (steps > 3) s[3] = step(S3{}, cur);
    // the next group is waited for here, not behind this group's stores
    computed(next);
    // lanes 7 and 15 of a row hold the partials' indices
    if ((row & 7) == 7) {
      float* const o01 = out + (int64_t)(int)cur.x * stride;
      float* const o23 = out + (int64_t)(int)cur.y * stride;
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        gstore(o01 + i, row == 7 ? s[0].m[i] : s[1].m[i]);
        gstore(o23 + i, row == 7 ? s[2].m[i] : s[3].m[i]);
      }
    }
  }
}

// D_e = sum of the record's partials; inv_e = 1 / D_e (guarded or not)
__global__ __launch_bounds__(256) void moment_inverse_kernel(
    const int* __restrict__ counts, int64_t n,
    const float* __restrict__ partial, int guard, float* __restrict__ inv,
    float* __restrict__ denominators) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  float s = 0.0f;
  const int c = counts[e];
  for (int k = 0; k < c; ++k) s += partial[k * n + e];
  if (denominators) denominators[e] = s;
  if (inv) inv[e] = guard ? ((s > 0.0f) ? 1.0f / s : 0.0f) : 1.0f / s;
}

// Back-projection of one task by one wavefront that owns the cells of its
// bin's line in LDS.  A step takes four pairs, 16 lanes each.  A row's 16
// additions (8 terms at the end cell of either side) go in four rounds of one
// 16-byte read-modify-write per lane; in each round the four lane groups work on
// different (side, half) quarters of the cells, so two pairs never meet in a word
// and no atomics are needed.  weights_of / into replace the instance's weights and
// images where they are not null.  Bound by VALU issue (61 instructions per step of
// 64 rows) and the chain of LDS round trips at the six wavefronts per CU (eight
// with 6 terms) that the cells leave room for.  2e7 events, 1000 x 400 at 1 mm:
// 6.9 ms (8 terms 8.5 ms; 9.9 ms with a step's arithmetic not between its LDS
// reads and writes), against 22.0 ms for the kernel that adds pixel by pixel (an
// LDS read and write each).  MERGED: a task holds groups of several bins of a
// band, and their pixels are summed in LDS (merged_columns of 16 rows) before
// they are added to the image: 381 x 203, 3e5 events 0.212 -> 0.192 ms, 100 x
// 100, 2e4 events 0.051 -> 0.032 ms.
template <int NM, bool MERGED>
__global__ __launch_bounds__(64) void moment_backward_kernel(
    const MomentInstance* __restrict__ desc, const MomentTask* __restrict__ tasks,
    const float* __restrict__ weights_of, float* __restrict__ into) {
  using Half = HalfCell<NM>;
  constexpr int W = Half::W, HALF = Half::half_words(),
                CELL = Half::cell_words();
  extern __shared__ float4v cells4[];
  const MomentTask task = tasks[blockIdx.x];
  const MomentInstance& d = desc[task.instance];
  const int lane = threadIdx.x;
  const int row = lane & (R - 1);
  const int grp = lane >> 4;
  const int P = d.positions;
  const int n_y = d.g.n_y, n_z = d.g.n_z;
  const float w_px = d.g.pixel_width;
  const int y_base = task.band * R;
  const int iy = y_base + row;
  LineRow l = line_row(d.g, task.xc, task.tc, row);
  const float qc = d.g.C * kExp2Scale;
  const float cs = d.cs;
  const float y = pixel_center_y(d.g, iy);
  const float y2 = y * y;
  const float* __restrict__ inv = weights_of ? weights_of : d.inv;
  float* __restrict__ bpT =
      into ? into
           : d.bpT + (int64_t)(blockIdx.x % (unsigned)d.bp_images) * n_z * n_y;
  const int side_words = Half::side_words(P);
  const int merged_columns = MERGED ? d.merged_columns : 0;
  for (int i = lane; i < side_words / 2; i += 64)
    cells4[i] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
  const uint4v* __restrict__ base =
      reinterpret_cast<const uint4v*>(d.blocks) + (int64_t)task.group * 64;
  const int n_here = task.pairs;
  const int last = MERGED ? n_here - 1 : (n_here - 1) / kGroup;
  // MERGED: the pixels of the task's bins, [column][row]
  float* const pixels = reinterpret_cast<float*>(cells4) + 2 * side_words;
  const MomentGroup* __restrict__ groups = d.groups + task.group;
  if (MERGED)
    for (int i = lane; i < merged_columns * (R / 4); i += 64)
      cells4[side_words / 2 + i] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
  float* const mine = reinterpret_cast<float*>(cells4) + row * W;
  const bool odd = grp & 1, high = grp & 2;
  const int h0 = high ? HALF : 0;
  const int h1 = HALF - h0;
  // the weights of a group's pairs: the lanes that hold a record's index
  // fetch its weight (word 0: steps 0 and 1, word 1: steps 2 and 3)
  struct Weights {
    float w01, w23;
  };
  auto weights = [&](const uint4v& v) {
    const bool index = (row & 7) == 6;
    Weights w;
    w.w01 = gload(inv + (index ? (int)v.x : 0));
    w.w23 = gload(inv + (index ? (int)v.y : 0));
    return w;
  };
  struct Terms {
    Half v0, v1;  // the moments of this lane's first and second half
    float* p0;    // the cells its run ends in, this lane's first side first
    float* p1;
  };
  auto terms = [&](auto tag, const uint4v& v, const Weights& wt) {
    constexpr int S = decltype(tag)::value;
    const RowTerms r = row_terms<S>(v, y, y2, l.x, qc);
    const float eta = cs * r.delta;
    float m[NM];
    m[0] = r.w * row_lane<6 + 8 * (S & 1)>(S < 2 ? wt.w01 : wt.w23);
    // (a run that misses the line's column adds nothing here)
    if (r.run >= 0x8000u) m[0] = 0.0f;
#pragma unroll
    for (int i = 1; i < NM; ++i) m[i] = m[i - 1] * eta;
    Terms t;
#pragma unroll
    for (int i = 0; i < W; ++i) {
      t.v0.w[i] = high ? m[W + i] : m[i];
      t.v1.w[i] = high ? m[i] : m[W + i];
    }
    const int a = (int)(r.run & 0xff) * CELL;
    const int b = (int)((r.run >> 8) & 0x7f) * CELL + side_words;
    t.p0 = mine + (odd ? b : a);
    t.p1 = mine + (odd ? a : b);
    return t;
  };
  auto add_to = [](float* p, Half x, const Half& v) {
#pragma unroll
    for (int i = 0; i < W; ++i) x.w[i] += v.w[i];
    x.store(p);
    lds_order();
  };
  auto add = [&](const Terms& t) {
    add_to(t.p0 + h0, Half::load(t.p0 + h0), t.v0);
    add_to(t.p1 + h0, Half::load(t.p1 + h0), t.v0);
    add_to(t.p0 + h1, Half::load(t.p0 + h1), t.v1);
    add_to(t.p1 + h1, Half::load(t.p1 + h1), t.v1);
  };
  // add(t), and the terms of step S of v a quarter at a time between each LDS
  // read and its write: the arithmetic hides the reads' latency (the scheduler
  // barriers keep it there)
  auto add_and_form = [&](auto tag, const Terms& t, const uint4v& v,
                          const Weights& wt) {
    constexpr int S = decltype(tag)::value;
    constexpr int F = 8 * (S & 1);
    Half x = Half::load(t.p0 + h0);
    __builtin_amdgcn_sched_barrier(0);
    RowTerms r = row_terms<S>(v, y, y2, l.x, qc);
    computed(r.delta);
    computed(r.w);
    __builtin_amdgcn_sched_barrier(0);
    add_to(t.p0 + h0, x, t.v0);
    x = Half::load(t.p1 + h0);
    __builtin_amdgcn_sched_barrier(0);
    const float eta = cs * r.delta;
    float m[NM];
    m[0] = r.w * row_lane<6 + F>(S < 2 ? wt.w01 : wt.w23);
    if (r.run >= 0x8000u) m[0] = 0.0f;
#pragma unroll
    for (int i = 1; i < NM; ++i) m[i] = m[i - 1] * eta;
#pragma unroll
    for (int i = 0; i < NM; ++i) computed(m[i]);
    __builtin_amdgcn_sched_barrier(0);
    add_to(t.p1 + h0, x, t.v0);
    x = Half::load(t.p0 + h1);
    __builtin_amdgcn_sched_barrier(0);
    Terms u;
#pragma unroll
    for (int i = 0; i < W; ++i) {
      u.v0.w[i] = high ? m[W + i] : m[i];
      u.v1.w[i] = high ? m[i] : m[W + i];
      computed(u.v0.w[i]);
      computed(u.v1.w[i]);
    }
    __builtin_amdgcn_sched_barrier(0);
    add_to(t.p0 + h1, x, t.v1);
    x = Half::load(t.p1 + h1);
    __builtin_amdgcn_sched_barrier(0);
    const int a = (int)(r.run & 0xff) * CELL;
    const int b = (int)((r.run >> 8) & 0x7f) * CELL + side_words;
    int first = odd ? b : a, second = odd ? a : b;
    computed(first);
    computed(second);
    u.p0 = mine + first;
    u.p1 = mine + second;
    __builtin_amdgcn_sched_barrier(0);
    add_to(t.p1 + h1, x, t.v1);
    return u;
  };
  // a run that misses the line's column, pixel by pixel
  auto walk = [&](auto tag, const uint4v& v, const Weights& wt) {
    constexpr int S = decltype(tag)::value;
    const RowTerms r = row_terms<S>(v, y, y2, l.x, qc);
    const float weight = row_lane<6 + 8 * (S & 1)>(S < 2 ? wt.w01 : wt.w23);
    if (r.run < 0x8000u || weight == 0.0f) return;
    const int n = (int)((r.run >> 8) & 0x7f);
    const int col = l.column + (int)(r.run & 0xff) - P / 2;
    float dz = (__builtin_fmaf((float)col, w_px, d.g.tl_z_half_w) - l.x) -
               r.delta;
    float* dst = bpT + (int64_t)col * n_y + iy;
    const float f = r.pre * weight;
    for (int k = 0; k < n; ++k) {
      gatomic_add(dst, f * __builtin_amdgcn_exp2f(
                               __builtin_fmaf(qc * dz, dz, r.qa)));
      dst += n_y;
      dz += w_px;
    }
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  using S2 = std::integral_constant<int, 2>;
  using S3 = std::integral_constant<int, 3>;
  // Inward sums, cell by cell: lane = (row, side, half); put(k, column, u, t)
  // takes the half's part t of the value of cell k's pixel.
  const int side = grp & 1, half = grp >> 1;
  float* const half_cell = mine + side * side_words + half * HALF;
  auto expand = [&](auto put) {
    float s[W] = {}, c[W];
#pragma unroll
    for (int i = 0; i < W; ++i)
      c[i] = half ? ExpPoly<NM>::c[W + i] : ExpPoly<NM>::c[i];
    const float inv_s = d.inv_s;
    const int dir = side ? 1 : -1;
    const int col0 = side ? l.column - 1 : l.column;  // + dir k: cell k
    // four cells' words are in flight together
    constexpr int B = 4;
    for (int k0 = P; k0 >= 1; k0 -= B) {
      Half x[B];
#pragma unroll
      for (int i = 0; i < B; ++i)
        x[i] = Half::load(half_cell + max(k0 - i, 0) * CELL);
      float t[B];
#pragma unroll
      for (int i = 0; i < B; ++i) {
#pragma unroll
        for (int w = 0; w < W; ++w) s[w] += x[i].w[w];
        const float u = __builtin_fmaf((float)(col0 + dir * (k0 - i)), w_px,
                                       d.g.tl_z_half_w) - l.x;
        const float v = u * inv_s;
        t[i] = s[W - 1] * c[W - 1];
#pragma unroll
        for (int w = W - 2; w >= 0; --w)
          t[i] = __builtin_fmaf(t[i], v, s[w] * c[w]);
        const float v2 = v * v;
        if (half) t[i] *= v2 * (W == 4 ? v2 : v);
        t[i] *= __builtin_amdgcn_exp2f(qc * u * u);
      }
      put(k0, col0 + dir * k0, t);
    }
  };
  uint4v cur = gload(base + lane);
  uint4v next = gload(base + min(1, last) * 64 + lane);
  Weights wt = weights(cur);
  if constexpr (MERGED) {
    // Bin after bin: a bin's cells are expanded into the task's pixels and
    // cleared when the next one begins.
    MomentGroup group = groups[0];
    l = line_row(d.g, group.xc, group.tc, row);
    auto merge = [&]() {
      expand([&](int k0, int column, const float(&t)[4]) {
        float* at[4];
        float sum[4], have[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const auto both = __builtin_amdgcn_permlane32_swap(
              __builtin_bit_cast(uint32_t, t[i]),
              __builtin_bit_cast(uint32_t, t[i]), false, false);
          const uint32_t lo = both[0], hi = both[1];
          sum[i] = __builtin_bit_cast(float, lo) +
                   __builtin_bit_cast(float, hi);
          Half zero = {};
          zero.store(half_cell + max(k0 - i, 0) * CELL);
          at[i] = pixels +
                  (column - (side ? i : -i) - task.first_column) * R + row;
          have[i] = (k0 - i >= 1 && !half) ? *at[i] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (k0 - i >= 1 && !half) *at[i] = have[i] + sum[i];
      });
      lds_order();
    };
    lds_order();
    for (int k = 0; k <= last; ++k) {
      const uint4v next2 = gload(base + min(k + 2, last) * 64 + lane);
      const Weights wt_next = weights(next);
      const MomentGroup group_next = groups[min(k + 1, last)];
      Terms t = terms(S0{}, cur, wt);
      if (group.pairs > 12) {
        t = add_and_form(S1{}, t, cur, wt);
        t = add_and_form(S2{}, t, cur, wt);
        t = add_and_form(S3{}, t, cur, wt);
        add(t);
      } else {
        add(t);
        if (group.pairs > 4) add(terms(S1{}, cur, wt));
        if (group.pairs > 8) add(terms(S2{}, cur, wt));
      }
      if (wave_any(any_direct(cur))) {
        walk(S0{}, cur, wt);
        walk(S1{}, cur, wt);
        walk(S2{}, cur, wt);
        walk(S3{}, cur, wt);
      }
      if (k == last || group_next.bin != group.bin) {
        merge();
        l = line_row(d.g, group_next.xc, group_next.tc, row);
      }
      cur = next;
      next = next2;
      wt = wt_next;
      group = group_next;
    }
    // lane = (row, column of four)
    for (int c = grp; c < merged_columns; c += 4) {
      const int x = task.first_column + c;
      const float val = pixels[c * R + row];
      if (val != 0.0f && x >= 0 && x < n_z && iy < n_y)
        gatomic_add(bpT + (int64_t)x * n_y + iy, val);
    }
    return;
  }
  // groups two ahead, weights one ahead, and a step's terms formed between the
  // LDS accesses of the step before it
  lds_order();
  Terms t = terms(S0{}, cur, wt);
  for (int k = 0; k <= last; ++k) {
    const uint4v next2 = gload(base + min(k + 2, last) * 64 + lane);
    const Weights wt_next = weights(next);
    const int here = n_here - k * kGroup;
    if (here > 12) {
      t = add_and_form(S1{}, t, cur, wt);
      t = add_and_form(S2{}, t, cur, wt);
      t = add_and_form(S3{}, t, cur, wt);
      t = add_and_form(S0{}, t, next, wt_next);
    } else {
      // a last group's empty steps are left out
      add(t);
      if (here > 4) add(terms(S1{}, cur, wt));
      if (here > 8) add(terms(S2{}, cur, wt));
    }
    if (wave_any(any_direct(cur))) {
      walk(S0{}, cur, wt);
      walk(S1{}, cur, wt);
      walk(S2{}, cur, wt);
      walk(S3{}, cur, wt);
    }
    cur = next;
    next = next2;
    wt = wt_next;
  }
  lds_order();
  // a half's part of a pixel's value replaces word 0 of its half cell (past
  // the last cell: of the unused cell 0)
  expand([&](int k0, int, const float(&t)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) half_cell[max(k0 - i, 0) * CELL] = t[i];
  });
  lds_order();
  // column by column into the image: lane = (row, column of four)
  int x_lo = l.column - P, x_hi = l.column + P;
  for (int o = 1; o < R; o <<= 1) {
    x_lo = min(x_lo, __shfl_xor(x_lo, o));
    x_hi = max(x_hi, __shfl_xor(x_hi, o));
  }
  x_lo = max(__builtin_amdgcn_readfirstlane(x_lo), 0);
  x_hi = min(__builtin_amdgcn_readfirstlane(x_hi), n_z);
  constexpr int B = 4;
  for (int x0 = x_lo + grp; x0 < x_hi; x0 += 4 * B) {
    float val[B];
#pragma unroll
    for (int i = 0; i < B; ++i) {
      const int k = x0 + 4 * i - l.column;
      const int cell = k >= 0 ? k + 1 : -k;
      const bool in = cell <= P && x0 + 4 * i < x_hi && iy < n_y;
      const float* at = mine + (k >= 0 ? side_words : 0) +
                        (in ? cell : 0) * CELL;
      const float sum = at[0] + at[HALF];
      val[i] = in ? sum : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < B; ++i)
      if (val[i] != 0.0f)
        gatomic_add(bpT + (int64_t)(x0 + 4 * i) * n_y + iy, val[i]);
  }
}

// out = or += the sum of the images, which are cleared
__global__ __launch_bounds__(256) void moment_fold_kernel(
    int64_t n, int images, int add, float* __restrict__ bp,
    float* __restrict__ out) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    float sum = 0.0f;
    for (int k = 0; k < images; ++k) {
      sum += bp[k * n + i];
      bp[k * n + i] = 0.0f;
    }
    out[i] = add ? out[i] + sum : sum;
  }
}

// total += columns of every stored run
__global__ __launch_bounds__(256) void moment_count_kernel(
    const uint32_t* __restrict__ blocks, int64_t n_lanes,
    unsigned long long* __restrict__ total) {
  unsigned long long mine = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
       i < 2 * n_lanes; i += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t w = blocks[(i >> 1) * 4 + 2 + (i & 1)];
    for (int k = 0; k < 2; ++k) {
      const uint32_t run = (w >> (16 * k)) & 0xffff;
      const uint32_t b = (run >> 8) & 0x7f;
      mine += (run & 0x8000u) ? b : (run & 0xff) + b;
    }
  }
  for (int o = 32; o > 0; o >>= 1) mine += __shfl_xor(mine, o);
  if ((threadIdx.x & 63) == 0 && mine) atomicAdd(total, mine);
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------

constexpr size_t kLds = 160 * 1024;
// Runs of a smaller sigma_z (in pixels) are a few columns long, and how their
// offsets round decides their kernel values.
constexpr double kMinSigmaPixels = 1.4;
constexpr int kFwdChunk = 2048;  // pairs of a forward workgroup's task
// back-projection tasks of several bins (merge_bins says when)
constexpr int kMergedPositions = 16;
constexpr int kMergedBins = 10500;
constexpr double kMergedSpan = 6.0;  // columns of a merged task's vertices
constexpr int kMergedTasks = 4096;   // tasks aimed at, of 8 to 64 groups
constexpr int kBwdChunk = 1024;  // pairs of a back-projection wavefront's task
// images that the back-projection adds to (images_for says when)
constexpr int kMaxImages = 4;

unsigned grid_of(int64_t n) { return (unsigned)((n + 255) / 256); }

// Cells per row and side: a run reaches at most its half length plus the
// vertex's distance from the line plus half a column (the line's distance from
// its column) to either side, and its columns from the line's on count that
// column too.
int positions_for(const DeviceGeometry& g, double reach) {
  const double sigma_px = 1.0 / std::sqrt((double)g.inv_pow_sigma_z) /
                          g.pixel_width;
  const double p = (kRunHalf + reach) * sigma_px + 1.55;
  return p < 1e6 ? (int)std::floor(p) : 1000000;
}

size_t table_bytes(int positions, int terms) {
  return sizeof(float) *
         (2 * (size_t)(positions + 1) * R * terms + (terms == 6 ? 32 : 0));
}

// Whether back-projection tasks hold several bins (of 8 terms).  Their pixels are
// summed in LDS first: 16 x 2 cells per bin added to the images one by one
// outweigh a few pairs' own work.  It takes bins for full tasks, and short lines,
// as the pixels' LDS comes on top of the cells'; with more pairs to a bin the
// wavefronts that this LDS costs count for more.  An iteration with one bin to a
// task and merged (cells, bins, pairs per bin):
//   5, 18100, 3.3: 42, 41 us       5, 25800, 15: 66, 65 us    5, 27800, 29: 82, 94
//   7, 6400, 1.2: 24, 30 us        7, 32700, 16: 95, 94 us    7, 34300, 30: 115, 137
//   9, 15000, 1.1: 66, 53 us       9, 147000, 15: 588, 471    9, 157000, 35: 753, 736
//   10, 10300, 3.2: 46, 45 us      10, 12500, 7.9: 54, 53     10, 13500, 24: 66, 78
//   13, 5600, 8.3: 40, 48 us       13, 98000, 18: 592, 472    13, 105000, 41: 753, 749
//   15, 10400, 1.6: 68, 55 us      15, 27400, 21: 190, 161    15, 29500, 77: 274, 339
//   19, 57700, 4.1: 342, 322 us    20, 30700, 21: 224, 246 us
bool merge_bins(int positions, double pairs, double bins) {
  return positions <= kMergedPositions && bins >= kMergedBins &&
         pairs < std::min(bins / 1000.0, 2.4 * positions) * bins;
}

// What the time of an iteration in either form depends on.
struct FormSizes {
  int positions;
  double pairs;
  double fwd_group, bwd_group;  // most pairs of a list task
  double slope;                 // largest |tan|, columns per row
  bool wide;                    // no span table for the lists
  double pixels;
};

// Whether the row-band lists do an iteration in less time than the moment form.
// Where the bins hold few pairs, tabulating and expanding their lines costs more
// than walking the runs' pixels, and more so the more cells a line has: it takes
// longer, and its LDS leaves fewer wavefronts to a CU.  The lists take as long as
// all their pairs at full throughput or as the chains of their largest tasks,
// which are short where events are few to a band and bucket, and longer where they
// solve every row's run anew.  Times in us, fitted to 1880 contexts (20 to 1600
// by 24 to 800 pixels of 0.5 to 2.5 mm, sigma_z 5 to 14 mm, 3 to 1e6 events); for
// 1810 others, at 5 and 95 %, the lists' lie at 0.87 and 1.18 of those measured
// and the moments' at 0.86 and 1.14.  There the moment form is taken 1240 times,
// 18 times where it is more than 3 % slower (at most 1.20 times), and the lists
// where they are more than 10 % slower 8 times (at most 1.44 times).  Some of them
// (cells, pairs, occupied bins: lists, moments):
//   24, 3997, 3335: 25, 60 us            57, 1022, 683: 26, 58 us
//   32, 1.2e5, 1.8e4: 189, 311 us        17, 1.8e5, 4.2e4: 237, 338 us
//   45, 9056, 589: 420, 29 us            24, 1.2e6, 3.4e4: 488, 375 us
//   13, 9.5e5, 5.2e4: 323, 256 us        24, 2.9e6, 8.5e4: 3433, 1025 us (wide)
// The moment form's plan is made in half to a third of the time of the lists':
// it is taken where the two are alike, on the shortest lines too, where a few
// events take either form the time of four launches.
// In a batch the members' tasks share the card, so nobody waits for the chains,
// and the moment form has to be a seventh faster.  24 members of 1e4 to 3e5 events,
// whose bins hold 2 to 186 pairs, ten iterations with all copies: 27.4 ms on the
// lists, 43.1 ms with 22 members in the moment form, 26.0 ms with this rule.
bool lists_faster(const FormSizes& s, double bins, bool batch) {
  const double P = s.positions;
  if (batch)
    return 1.15 * (s.pairs * 0.07 + bins * 8.0 * std::pow(P / 24.0, 1.6)) >
           s.pairs * (0.04 + 0.0065 * P);
  const double wide = s.wide ? 1.0 : 0.0;
  const double line = std::max(P - 7.0, 0.0);
  const double chain =
      s.fwd_group * (0.0342 + 0.00323 * P + 0.135 * wide) +
      s.bwd_group * (0.00641 * (P + 8.0 * s.slope) + 0.135 * wide);
  const double work = s.pairs * (9.67e-5 + 6.62e-6 * P +
                                 (5.9e-5 + 2.58e-4 * s.slope) * wide);
  const double lists = 12.4 + 0.0955 * line + 5.54e-6 * s.pixels +
                       std::hypot(chain, work);
  // a bin's line at the wavefronts that its cells leave room for; the chain of
  // the fullest bin
  const double room = std::max(std::floor(160.0 / (P + 1.0)), 1.0);
  const double per_bin = (0.0378 + 8.67e-4 * P) / room *
                         (merge_bins(s.positions, s.pairs, bins) ? 0.79 : 1.0);
  const double one = 0.298 * line + 0.085 * std::min(4.0 * s.pairs / bins, 1024.0);
  const double all = bins * per_bin + s.pairs * (5.35e-5 + 1.15e-6 * P);
  const double moments = 12.4 + 7.73e-6 * s.pixels + std::hypot(one, all);
  return moments > (lists > 60.0 || P <= 7.0 ? 1.05 : 0.95) * lists;
}

// Images that a plan's back-projection adds to.  Every task adds its cells to
// the image with FP32 atomics, and the running sum rounds at each addition: over
// k images it does so at a k-th of the size and of the number.  The error of
// the image derivative of a log-likelihood against 64 bits (both with the FP32
// support), pixel-by-pixel lists and moments with 1, 2, 4, 8 images:
//   203 x 56, 96151 events, 330 additions a pixel:
//     1.9e-7 | 3.2e-7, 2.0e-7, 1.3e-7, 1.2e-7
//   476 x 197, 329679 events, 180: 1.8e-7 | 2.3e-7, 1.4e-7, 1.0e-7, 1.0e-7
//   335 x 185, unrolled, 52 (merged): 9.7e-7 | 1.7e-6, 0.9e-6, 0.6e-6, 0.5e-6
// Few additions need no second image, whose sum and clearing would cost a short
// list on a large grid more than its own work.
int images_for(double additions) {
  return additions < 8.0 ? 1 : additions < 64.0 ? 2 : kMaxImages;
}

// A dispatch counts its work-items in 32 bits: tasks of one launch.
constexpr int64_t kLaunchItems = (int64_t)1 << 31;
int64_t tasks_per_launch(int waves) { return kLaunchItems / (64 * waves); }

int launch_forward(int terms, int waves, size_t lds, const MomentInstance* desc,
                   const MomentTask* tasks, int n_tasks, hipStream_t stream,
                   std::string* err) {
  auto kern = terms == 8 ? (waves == 4 ? moment_forward_kernel<8, 4>
                                       : moment_forward_kernel<8, 1>)
                         : (waves == 4 ? moment_forward_kernel<6, 4>
                                       : moment_forward_kernel<6, 1>);
  const int64_t most = tasks_per_launch(waves);
  for (int64_t at = 0; at < n_tasks; at += most) {
    hipLaunchKernelGGL(kern, dim3((unsigned)std::min(most, n_tasks - at)),
                       dim3(64 * waves), lds, stream, desc, tasks + at);
    BAND_TRY(hipGetLastError());
  }
  return 0;
}

int launch_backward(int terms, bool merged, size_t lds,
                    const MomentInstance* desc, const MomentTask* tasks,
                    int n_tasks, const float* weights, float* into,
                    hipStream_t stream, std::string* err) {
  auto kern = terms == 6 ? moment_backward_kernel<6, false>
              : merged   ? moment_backward_kernel<8, true>
                         : moment_backward_kernel<8, false>;
  const int64_t most = tasks_per_launch(1);
  for (int64_t at = 0; at < n_tasks; at += most) {
    hipLaunchKernelGGL(kern, dim3((unsigned)std::min(most, n_tasks - at)),
                       dim3(64), lds, stream, desc, tasks + at, weights, into);
    BAND_TRY(hipGetLastError());
  }
  return 0;
}

// dst = src as tasks of the batch's instance
__global__ __launch_bounds__(256) void moment_tag_kernel(
    const MomentTask* __restrict__ src, int n, int instance,
    MomentTask* __restrict__ dst) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  MomentTask t = src[i];
  t.instance = instance;
  dst[i] = t;
}

// Device memory handed out from one allocation, in 256-byte steps.
struct Arena {
  size_t used = 0;
  template <typename T>
  size_t take(int64_t n) {
    const size_t at = used;
    used += (sizeof(T) * (size_t)std::max<int64_t>(n, 1) + 255) & ~(size_t)255;
    return at;
  }
};

}  // namespace

bool moment_supported(const DeviceGeometry& g) {
  const double sigma_px = 1.0 / std::sqrt((double)g.inv_pow_sigma_z) /
                          g.pixel_width;
  const int p = positions_for(g, ExpPoly<8>::reach);
  return sigma_px >= kMinSigmaPixels && p <= 120 &&
         table_bytes(p, kGradMoments) <= kLds &&
         g.n_z >= 4 && g.n_y >= 1;
}

void moment_release(MomentPlan& plan) {
  if (plan.arena) (void)hipFree(plan.arena);
  if (plan.lists) (void)hipFree(plan.lists);
  plan = MomentPlan{};
}

int moment_prepare(MomentPlan& plan, const DeviceGeometry& g,
                   const EventSoA& ev, int64_t n, float* const rhoT[2],
                   float* bpT, bool batch, hipStream_t stream, bool* built,
                   int max_extent[2], std::string* err) {
  *built = false;
  moment_release(plan);
  if (n <= 0 || n > 0x3fffffff || !moment_supported(g)) return 0;
  struct Scratch {
    void* p = nullptr;
    ~Scratch() {
      if (p) (void)hipFree(p);
    }
  } stats_mem, temp;
  // what the choice and the sizes of the plan depend on
  const int n_bands = (g.n_y + R - 1) / R;
  const int buckets = (g.n_z + kBucket - 1) / kBucket;
  const int64_t step = (n + kSampled - 1) / kSampled;
  const double sigma = 1.0 / std::sqrt((double)g.inv_pow_sigma_z);
  if (hipMalloc(&stats_mem.p, sizeof(PlanStats)) != hipSuccess) {
    stats_mem.p = nullptr;
    (void)hipGetLastError();
    return 0;
  }
  PlanStats* d_stats = static_cast<PlanStats*>(stats_mem.p);
  hipLaunchKernelGGL(fill_words_kernel, dim3(1), dim3(256), 0, stream,
                     (uint32_t*)d_stats, (int64_t)(sizeof(PlanStats) / 4), 0u);
  hipLaunchKernelGGL(moment_stats_kernel,
                     dim3(std::min<unsigned>(grid_of(n), 1024)), dim3(256), 0,
                     stream, ev.box, ev.a, n, d_stats);
  if (!batch)
    hipLaunchKernelGGL(moment_groups_kernel, dim3(1), dim3(1024), 0, stream, g,
                       ev.box, ev.a, n, step, buckets,
                       std::min(n_bands * buckets, kGroupWords),
                       (float)(kRunHalf * sigma / g.pixel_width), d_stats);
  BAND_TRY(hipGetLastError());
  PlanStats st{};
  BAND_TRY(hipMemcpyAsync(&st, d_stats, sizeof(st), hipMemcpyDeviceToHost,
                          stream));
  BAND_TRY(hipStreamSynchronize(stream));
  for (int i = 0; i < 2; ++i) max_extent[i] = std::max(st.max_extent[i], 1);
  const int64_t n_pairs = (int64_t)st.pairs;
  const double max_tan = (double)__builtin_bit_cast(float, st.max_tan);
  if (n_pairs <= 0 || n_pairs > 0x3fffffff || !(max_tan < 1e3) ||
      (double)n * st.max_bands > 2e9)
    return 0;

  // bins: half the reach for the vertex, half for the shear over a band
  const double iz = g.inv_pow_sigma_z, id = g.inv_pow_sigma_dl;
  const double k = 8.0 * iz * id / (4.0 * id + 2.0 * iz);
  const double half_width = 3.0 / std::sqrt(k);
  MomentInstance d{};
  d.g = g;
  d.max_bands = std::max(st.max_bands, 1);
  d.n_events = n;
  int terms = 8;
  double n_bins_f = 0.0;
  auto set_bins = [&]() {
    const double reach_of = terms == 8 ? ExpPoly<8>::reach : ExpPoly<6>::reach;
    const double reach = reach_of * sigma * 0.995;
    const double dx = reach;
    const double dt = reach / (0.5 * (R - 1) * (double)g.pixel_height);
    const double margin = 2.0 * half_width + 4.0 * g.pixel_width +
                          0.5 * R * g.pixel_height * max_tan + dx;
    const double z_span = (double)g.n_z * g.pixel_width + 2.0 * margin;
    const double nt = std::ceil(2.0 * max_tan / dt) + 1.0;
    const double nx = std::ceil(z_span / dx) + 1.0;
    n_bins_f = nx * nt * n_bands;
    if (!(nt <= 4096.0) || !(n_bins_f <= (double)(1 << 24))) return false;
    d.nx = (int)nx;
    d.nt = (int)nt;
    d.x_lo = (float)((double)g.tl_z - margin);
    d.dx = (float)dx;
    d.t_lo = (float)(-0.5 * nt * dt);
    d.dt = (float)dt;
    d.positions = positions_for(g, reach_of);
    // (a power of two near the largest |u|: no rounding in u / s and C s)
    const double s =
        std::exp2(std::round(std::log2((kRunHalf + reach_of) * sigma)));
    d.inv_s = (float)(1.0 / s);
    d.cs = (float)((double)g.C * s);
    return true;
  };
  if (!set_bins()) return 0;
  // Six terms about lines 2.3 times closer leave room for eight instead of six
  // back-projection wavefronts per CU (24 cells) and save arithmetic, but make
  // five times the bins, each with its table and its expansion: taken where
  // the bins stay full.  An iteration with 8 and 6 terms (cells, pairs per bin,
  // occupied or not):
  //   13, 100: 0.357, 0.361 ms    13, 300: 0.905, 0.866 ms  15, 354: 2.16, 2.35 ms
  //   24, 142: 1.99, 2.43 ms      24, 285: 3.74, 3.84 ms    24, 947: 12.1, 10.8 ms
  //   34, 256: 1.21, 1.17 ms      34, 767: 3.17, 2.59 ms    36, 703: 0.113, 0.119
  //   48, 155: 0.74, 0.94 ms      48, 517: 1.94, 1.82 ms    66, 447: 0.78, 0.63 ms
  if ((double)n_pairs >= 400.0 * n_bins_f) {
    terms = 6;
    if (!set_bins()) {
      terms = 8;
      if (!set_bins()) return 0;
    }
  }
  const int n_bins = d.nx * d.nt * n_bands;

  // Only where the occupied bins decide it are they counted, before anything is
  // sorted.
  const FormSizes sizes{
      d.positions,
      (double)n_pairs,
      std::min((double)(st.max_group[0] * step), 2048.0),
      std::min((double)(st.max_group[1] * step), 512.0),
      max_tan * (double)g.pixel_height / (double)g.pixel_width,
      st.max_extent[0] > 255,
      (double)g.n_z * g.n_y};
  if (lists_faster(sizes, (double)std::min<int64_t>(n_bins, n_pairs), batch)) {
    // (a few pairs lie in nearly as many bins)
    if (n_pairs <= 256) return 0;
    Scratch marks;
    const int n_words = (n_bins + 3) / 4;
    if (hipMalloc(&marks.p, sizeof(uint32_t) * (size_t)n_words) !=
        hipSuccess) {
      marks.p = nullptr;
      (void)hipGetLastError();
      return 0;
    }
    hipLaunchKernelGGL(fill_words_kernel, dim3(256), dim3(256), 0, stream,
                       (uint32_t*)marks.p, (int64_t)n_words, 0u);
    hipLaunchKernelGGL(moment_mark_kernel, dim3(grid_of(n)), dim3(256), 0,
                       stream, d, ev.box, ev.a, n, (uint8_t*)marks.p);
    hipLaunchKernelGGL(moment_marked_kernel, dim3(256), dim3(256), 0, stream,
                       (const uint32_t*)marks.p, n_words, &d_stats->occupied);
    BAND_TRY(hipGetLastError());
    int occupied = 0;
    BAND_TRY(hipMemcpyAsync(&occupied, &d_stats->occupied, sizeof(int),
                            hipMemcpyDeviceToHost, stream));
    BAND_TRY(hipStreamSynchronize(stream));
    if (lists_faster(sizes, (double)occupied, batch)) return 0;
  }

  // what building the plan needs
  Arena work;
  const int64_t sort_n = std::max<int64_t>(n, n_pairs);
  const int64_t bins1 = (int64_t)n_bins + 1;
  const size_t w_keys = work.take<uint32_t>(sort_n);
  const size_t w_keys2 = work.take<uint32_t>(sort_n);
  const size_t w_vals = work.take<int>(sort_n);
  const size_t w_vals2 = work.take<int>(sort_n);
  const size_t w_rec = work.take<BandRecord>(n);
  const size_t w_offsets = work.take<int>(n);
  const size_t w_first = work.take<int>(bins1);
  const size_t w_end = work.take<int>(bins1);
  const size_t w_count = work.take<int>(bins1);
  const size_t w_pieces = work.take<int>(3 * bins1);
  size_t cub = 0;
  {
    size_t b = 0;
    hipcub::DoubleBuffer<uint32_t> kb(nullptr, nullptr);
    hipcub::DoubleBuffer<int> vb(nullptr, nullptr);
    BAND_TRY(hipcub::DeviceRadixSort::SortPairs(nullptr, b, kb, vb,
                                                (int)sort_n, 0, 32, stream));
    cub = std::max(cub, b);
    BAND_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, b, (int*)nullptr,
                                              (int*)nullptr, (int)n, stream));
    cub = std::max(cub, b);
    BAND_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, b, (int*)nullptr,
                                              (int*)nullptr, (int)bins1,
                                              stream));
    cub = std::max(cub, b);
  }
  const size_t w_cub = work.take<char>((int64_t)cub);
  // the plan's per-event memory; its groups and tasks are sized below
  Arena own;
  const size_t o_partial = own.take<float>(n * d.max_bands + 1);
  const size_t o_inv = own.take<float>(n);
  const size_t o_counts = own.take<int>(n);
  const size_t o_order = own.take<int>(n);
  const size_t o_desc = own.take<MomentInstance>(2);
  size_t free_bytes = 0, total_bytes = 0;
  BAND_TRY(hipMemGetInfo(&free_bytes, &total_bytes));
  if (64 * (size_t)n_pairs + own.used > free_bytes / 2 ||
      80 * (size_t)n_pairs + own.used + work.used > free_bytes)
    return 0;
  // out of memory or unsuited events: the row-band lists take over
  auto give_up = [&]() {
    (void)hipGetLastError();
    moment_release(plan);
    return 0;
  };
  if (hipMalloc(&plan.arena, own.used) != hipSuccess) {
    plan.arena = nullptr;
    return give_up();
  }
  if (hipMalloc(&temp.p, work.used) != hipSuccess) {
    temp.p = nullptr;
    return give_up();
  }
  char* A = static_cast<char*>(plan.arena);
  char* W = static_cast<char*>(temp.p);
  plan.partial = reinterpret_cast<float*>(A + o_partial);
  plan.inv = reinterpret_cast<float*>(A + o_inv);
  plan.counts = reinterpret_cast<int*>(A + o_counts);
  plan.order = reinterpret_cast<int*>(A + o_order);
  plan.desc = reinterpret_cast<MomentInstance*>(A + o_desc);
  uint32_t* keys = reinterpret_cast<uint32_t*>(W + w_keys);
  uint32_t* keys2 = reinterpret_cast<uint32_t*>(W + w_keys2);
  int* vals = reinterpret_cast<int*>(W + w_vals);
  int* vals2 = reinterpret_cast<int*>(W + w_vals2);
  BandRecord* rec = reinterpret_cast<BandRecord*>(W + w_rec);
  int* offsets = reinterpret_cast<int*>(W + w_offsets);
  int* first = reinterpret_cast<int*>(W + w_first);
  int* end = reinterpret_cast<int*>(W + w_end);
  int* piece_count = reinterpret_cast<int*>(W + w_count);
  int* pieces[3];  // first group, forward and back-projection task of each bin
  for (int i = 0; i < 3; ++i)
    pieces[i] = reinterpret_cast<int*>(W + w_pieces) + i * bins1;
  void* cub_mem = W + w_cub;

  // events in bin-friendly order, their records, their pairs by bin
  hipLaunchKernelGGL(moment_order_kernel, dim3(grid_of(n)), dim3(256), 0,
                     stream, d, ev.box, ev.a, n, keys, vals);
  BAND_TRY(hipGetLastError());
  {
    hipcub::DoubleBuffer<uint32_t> kb(keys, keys2);
    hipcub::DoubleBuffer<int> vb(vals, vals2);
    size_t b = cub;
    BAND_TRY(hipcub::DeviceRadixSort::SortPairs(cub_mem, b, kb, vb, (int)n, 0,
                                                32, stream));
    BAND_TRY(hipMemcpyAsync(plan.order, vb.Current(), sizeof(int) * n,
                            hipMemcpyDeviceToDevice, stream));
  }
  hipLaunchKernelGGL(moment_records_kernel, dim3(grid_of(n)), dim3(256), 0,
                     stream, ev, plan.order, n, rec, plan.counts);
  BAND_TRY(hipGetLastError());
  {
    size_t b = cub;
    BAND_TRY(hipcub::DeviceScan::ExclusiveSum(cub_mem, b, plan.counts, offsets,
                                              (int)n, stream));
  }
  hipLaunchKernelGGL(moment_emit_kernel, dim3(grid_of(n)), dim3(256), 0,
                     stream, d, rec, plan.counts, offsets, n, keys, vals);
  BAND_TRY(hipGetLastError());
  int end_bit = 1;
  while (end_bit < 32 && (1 << end_bit) < n_bins) ++end_bit;
  hipcub::DoubleBuffer<uint32_t> kb(keys, keys2);
  hipcub::DoubleBuffer<int> vb(vals, vals2);
  {
    size_t b = cub;
    BAND_TRY(hipcub::DeviceRadixSort::SortPairs(cub_mem, b, kb, vb,
                                                (int)n_pairs, 0, end_bit,
                                                stream));
  }
  // the bins' groups and tasks
  hipLaunchKernelGGL(fill_words_kernel, dim3(1024), dim3(256), 0, stream,
                     (uint32_t*)first, (int64_t)(w_count - w_first) / 4, 0u);
  hipLaunchKernelGGL(moment_bins_kernel, dim3(grid_of(n_pairs)), dim3(256), 0,
                     stream, kb.Current(), n_pairs, first, end);
  BAND_TRY(hipGetLastError());
  const int chunks[3] = {kGroup, kFwdChunk, kBwdChunk};
  int totals[3] = {0, 0, 0};
  for (int i = 0; i < 3; ++i) {
    hipLaunchKernelGGL(moment_piece_count_kernel, dim3(grid_of(bins1)),
                       dim3(256), 0, stream, first, end, n_bins, chunks[i],
                       piece_count);
    size_t b = cub;
    BAND_TRY(hipcub::DeviceScan::ExclusiveSum(cub_mem, b, piece_count,
                                              pieces[i], (int)bins1, stream));
    BAND_TRY(hipMemcpyAsync(&totals[i], pieces[i] + n_bins, sizeof(int),
                            hipMemcpyDeviceToHost, stream));
  }
  BAND_TRY(hipStreamSynchronize(stream));
  const int n_groups = totals[0];
  int merged_chunk = 0;
  const double row_step = 0.5 * (R - 1) * (double)g.pixel_height;
  const float max_shear =
      (float)(row_step * ((double)d.nt * 0.5) * (double)d.dt);
  const int x_block = std::max(
      1, (int)std::floor(kMergedSpan * (double)g.pixel_width / (double)d.dx));
  const int merged_columns = std::min<int>(
      2 * d.positions + 4 +
          (int)std::ceil((x_block * (double)d.dx + 2.0 * max_shear) /
                         (double)g.pixel_width),
      g.n_z + 2 * d.positions);
  const size_t merged_bytes = sizeof(float) * R * (size_t)merged_columns;
  const bool merged =
      terms == 8 &&
      merge_bins(d.positions, (double)n_pairs, (double)totals[1]) &&
      table_bytes(d.positions, terms) + merged_bytes <= kLds;
  const int n_x_blocks = (d.nx + x_block - 1) / x_block;
  const int n_blocks = n_bands * n_x_blocks;
  if (merged) {
    const int chunk = std::max(8, std::min(64, n_groups / kMergedTasks));
    hipLaunchKernelGGL(moment_block_count_kernel, dim3(grid_of(n_blocks + 1)),
                       dim3(256), 0, stream, d, pieces[0], n_blocks, x_block,
                       n_x_blocks, chunk, piece_count);
    size_t b = cub;
    BAND_TRY(hipcub::DeviceScan::ExclusiveSum(cub_mem, b, piece_count,
                                              pieces[2], n_blocks + 1,
                                              stream));
    BAND_TRY(hipMemcpyAsync(&totals[2], pieces[2] + n_blocks, sizeof(int),
                            hipMemcpyDeviceToHost, stream));
    BAND_TRY(hipStreamSynchronize(stream));
    merged_chunk = chunk;
  }
  const int64_t n_pixels = (int64_t)g.n_z * g.n_y;
  plan.bp_images = images_for(
      (double)totals[2] * R * (merged ? merged_columns : 2 * d.positions + 1) /
      (double)n_pixels);
  Arena lists;
  const size_t o_images =
      lists.take<float>(plan.bp_images > 1 ? n_pixels * plan.bp_images : 0);
  const size_t o_blocks = lists.take<uint4>((int64_t)n_groups * 64);
  const size_t o_groups = lists.take<MomentGroup>(n_groups);
  const size_t o_fwd = lists.take<MomentTask>(totals[1]);
  const size_t o_bwd = lists.take<MomentTask>(totals[2]);
  if (hipMalloc(&plan.lists, lists.used) != hipSuccess) {
    plan.lists = nullptr;
    return give_up();
  }
  char* L = static_cast<char*>(plan.lists);
  plan.bpT = bpT;
  if (plan.bp_images > 1) {
    plan.bpT = reinterpret_cast<float*>(L + o_images);
    hipLaunchKernelGGL(fill_words_kernel, dim3(1024), dim3(256), 0, stream,
                       (uint32_t*)plan.bpT, n_pixels * plan.bp_images, 0u);
  }
  plan.blocks = reinterpret_cast<uint32_t*>(L + o_blocks);
  plan.fwd_tasks = reinterpret_cast<MomentTask*>(L + o_fwd);
  plan.bwd_tasks = reinterpret_cast<MomentTask*>(L + o_bwd);
  MomentGroup* groups = reinterpret_cast<MomentGroup*>(L + o_groups);
  // (the sorted keys are no longer needed)
  int* group_pair = reinterpret_cast<int*>(kb.Current());
  hipLaunchKernelGGL(moment_group_emit_kernel, dim3(grid_of(n_bins)),
                     dim3(256), 0, stream, d, first, end, n_bins, pieces[0],
                     groups, group_pair);
  for (int pass = 0; pass < (merged ? 1 : 2); ++pass)
    hipLaunchKernelGGL(moment_task_emit_kernel, dim3(grid_of(n_bins)),
                       dim3(256), 0, stream, d, first, end, n_bins,
                       chunks[1 + pass], pieces[0], pieces[1 + pass],
                       pass ? plan.bwd_tasks : plan.fwd_tasks);
  if (merged)
    hipLaunchKernelGGL(moment_block_emit_kernel, dim3(grid_of(n_blocks)),
                       dim3(256), 0, stream, d, pieces[0], n_blocks, x_block,
                       n_x_blocks, merged_chunk, max_shear, pieces[2],
                       plan.bwd_tasks);
  int* d_status = &d_stats->status;
  hipLaunchKernelGGL(moment_pack_kernel,
                     dim3((unsigned)std::min(n_groups, 1 << 20)), dim3(256), 0,
                     stream, d, rec, groups, group_pair, vb.Current(),
                     n_groups,
                     (int)n, (int)(n * d.max_bands),
                     reinterpret_cast<uint4*>(plan.blocks), d_status);
  BAND_TRY(hipGetLastError());
  int status = 0;
  BAND_TRY(hipMemcpyAsync(&status, d_status, sizeof(int),
                          hipMemcpyDeviceToHost, stream));
  d.blocks = plan.blocks;
  d.partial = plan.partial;
  d.counts = plan.counts;
  d.groups = groups;
  d.merged_columns = merged_columns;
  d.inv = plan.inv;
  d.bpT = plan.bpT;
  d.bp_images = plan.bp_images;
  MomentInstance both[2] = {d, d};
  for (int c = 0; c < 2; ++c) {
    both[c].rhoT = rhoT[c];
    both[c].rho_next = rhoT[c ^ 1];
  }
  BAND_TRY(hipMemcpyAsync(plan.desc, both, sizeof(both), hipMemcpyHostToDevice,
                          stream));
  BAND_TRY(hipStreamSynchronize(stream));
  if (status) {
    moment_release(plan);
    return 0;
  }
  plan.inst = both[0];
  plan.n_events = n;
  plan.n_pairs = n_pairs;
  plan.n_groups = n_groups;
  plan.n_bins = n_bins;
  plan.n_fwd = totals[1];
  plan.n_bwd = totals[2];
  plan.terms = terms;
  plan.merged = merged;
  plan.fwd_lds = table_bytes(d.positions, terms);
  plan.bwd_lds = plan.fwd_lds + (merged ? merged_bytes : 0);
  plan.fwd_waves = n_pairs / std::max(plan.n_fwd, 1) >= 100 ? 4 : 1;
  for (const void* kern :
       {reinterpret_cast<const void*>(moment_forward_kernel<8, 1>),
        reinterpret_cast<const void*>(moment_forward_kernel<8, 4>),
        reinterpret_cast<const void*>(moment_forward_kernel<6, 1>),
        reinterpret_cast<const void*>(moment_forward_kernel<6, 4>),
        reinterpret_cast<const void*>(moment_backward_kernel<6, false>),
        reinterpret_cast<const void*>(moment_gradient_kernel<1>),
        reinterpret_cast<const void*>(moment_gradient_kernel<4>),
        reinterpret_cast<const void*>(moment_backward_kernel<8, true>),
        reinterpret_cast<const void*>(moment_backward_kernel<8, false>)})
    BAND_TRY(hipFuncSetAttribute(
        kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds));
  plan.ready = true;
  *built = true;
  return 0;
}

int moment_forward(MomentPlan& plan, int cur, hipStream_t stream,
                   std::string* err) {
  return launch_forward(plan.terms, plan.fwd_waves, plan.fwd_lds,
                        plan.desc + cur, plan.fwd_tasks, plan.n_fwd, stream,
                        err);
}

int moment_inverse(MomentPlan& plan, int guard, float* inv, float* denominators,
                   hipStream_t stream, std::string* err) {
  hipLaunchKernelGGL(moment_inverse_kernel, dim3(grid_of(plan.n_events)),
                     dim3(256), 0, stream, plan.counts, plan.n_events,
                     plan.partial, guard, inv,
                     denominators);
  BAND_TRY(hipGetLastError());
  return 0;
}

int moment_backward(MomentPlan& plan, int cur, hipStream_t stream,
                    std::string* err) {
  return launch_backward(plan.terms, plan.merged, plan.bwd_lds,
                         plan.desc + cur, plan.bwd_tasks, plan.n_bwd, nullptr,
                         nullptr, stream, err);
}

int moment_fold(MomentPlan& plan, float* into, bool add, hipStream_t stream,
                std::string* err) {
  if (plan.bpT == into) return 0;
  const int64_t n = (int64_t)plan.inst.g.n_z * plan.inst.g.n_y;
  hipLaunchKernelGGL(moment_fold_kernel,
                     dim3((unsigned)std::min<int64_t>((n + 255) / 256, 4096)),
                     dim3(256), 0, stream, n, plan.bp_images, add ? 1 : 0,
                     plan.bpT, into);
  BAND_TRY(hipGetLastError());
  return 0;
}

int moment_backward_into(MomentPlan& plan, const float* weights, float* into,
                         bool add, hipStream_t stream, std::string* err) {
  const bool direct = plan.bp_images == 1;
  if (direct && !add)
    hipLaunchKernelGGL(
        fill_words_kernel, dim3(1024), dim3(256), 0, stream, (uint32_t*)into,
        (int64_t)plan.inst.g.n_z * plan.inst.g.n_y, 0u);
  if (launch_backward(plan.terms, plan.merged, plan.bwd_lds, plan.desc,
                      plan.bwd_tasks, plan.n_bwd, weights,
                      direct ? into : nullptr, stream, err))
    return -1;
  return direct ? 0 : moment_fold(plan, into, add, stream, err);
}

int moment_gradient(MomentPlan& plan, const float* xT, int stride, float* out,
                    hipStream_t stream, std::string* err) {
  if (plan.n_fwd == 0) return 0;
  auto kern = plan.fwd_waves == 4 ? moment_gradient_kernel<4>
                                  : moment_gradient_kernel<1>;
  hipLaunchKernelGGL(kern, dim3(plan.n_fwd), dim3(64 * plan.fwd_waves),
                     table_bytes(plan.inst.positions, kGradMoments), stream,
                     plan.desc, plan.fwd_tasks, xT, stride, out);
  BAND_TRY(hipGetLastError());
  return 0;
}

void moment_batch_release(MomentBatch& batch) {
  for (MomentInstance* d : batch.desc)
    if (d) (void)hipFree(d);
  if (batch.tasks) (void)hipFree(batch.tasks);
  batch = MomentBatch{};
}

int moment_batch_build(MomentBatch& batch,
                       const std::vector<const MomentPlan*>& plans,
                       hipStream_t stream, std::string* err) {
  moment_batch_release(batch);
  if (plans.empty()) return 0;
  const int n = (int)plans.size();
  std::vector<MomentInstance> inst(n);
  for (int c = 0; c < 2; ++c) {
    for (int i = 0; i < n; ++i) {
      inst[i] = plans[i]->inst;
      if (c) {
        float* next = const_cast<float*>(inst[i].rhoT);
        inst[i].rhoT = inst[i].rho_next;
        inst[i].rho_next = next;
      }
    }
    BAND_TRY(hipMalloc(&batch.desc[c], sizeof(MomentInstance) * n));
    BAND_TRY(hipMemcpy(batch.desc[c], inst.data(), sizeof(MomentInstance) * n,
                       hipMemcpyHostToDevice));
  }
  // parts: a plan's forward or back-projection tasks; those of one launch are
  // put next to each other, the plans with most pairs first
  struct Part {
    MomentBatch::Launch kind;
    int plan;
  };
  std::vector<Part> parts;
  int64_t total = 0;
  for (int i = 0; i < n; ++i) {
    const MomentPlan& p = *plans[i];
    const Part fwd{{false, p.terms, p.fwd_waves, false, p.fwd_lds, 0, p.n_fwd},
                   i};
    const Part bwd{{true, p.terms, 1, p.merged, p.bwd_lds, 0, p.n_bwd}, i};
    for (const Part& part : {fwd, bwd})
      if (part.kind.n) {
        parts.push_back(part);
        total += part.kind.n;
      }
  }
  if (total > 0x7fffffff) {
    if (err) *err = "too many tasks in one batch";
    return -1;
  }
  auto key = [](const MomentBatch::Launch& l) {
    const int residents = (int)std::min<size_t>(kLds / std::max<size_t>(l.lds, 1), 16);
    return std::make_tuple(l.backward, l.terms, l.waves, l.merged, residents);
  };
  std::stable_sort(parts.begin(), parts.end(),
                   [&](const Part& a, const Part& b) {
                     const auto ka = key(a.kind), kb = key(b.kind);
                     if (ka != kb) return ka < kb;
                     return plans[a.plan]->n_pairs > plans[b.plan]->n_pairs;
                   });
  BAND_TRY(hipMalloc(&batch.tasks,
                     sizeof(MomentTask) * std::max<int64_t>(total, 1)));
  int at = 0;
  for (const Part& part : parts) {
    const MomentPlan& p = *plans[part.plan];
    hipLaunchKernelGGL(moment_tag_kernel, dim3(grid_of(part.kind.n)), dim3(256),
                       0, stream,
                       part.kind.backward ? p.bwd_tasks : p.fwd_tasks,
                       part.kind.n, part.plan, batch.tasks + at);
    BAND_TRY(hipGetLastError());
    if (batch.launches.empty() ||
        key(batch.launches.back()) != key(part.kind)) {
      batch.launches.push_back(part.kind);
      batch.launches.back().first = at;
    } else {
      batch.launches.back().n += part.kind.n;
      batch.launches.back().lds =
          std::max(batch.launches.back().lds, part.kind.lds);
    }
    at += part.kind.n;
  }
  BAND_TRY(hipStreamSynchronize(stream));
  return 0;
}

int moment_batch_launch(const MomentBatch& batch, int c, bool backward,
                        hipStream_t stream, std::string* err) {
  for (const MomentBatch::Launch& l : batch.launches) {
    if (l.backward != backward) continue;
    const MomentTask* tasks = batch.tasks + l.first;
    if (backward ? launch_backward(l.terms, l.merged, l.lds, batch.desc[c],
                                   tasks, l.n, nullptr, nullptr, stream, err)
                 : launch_forward(l.terms, l.waves, l.lds, batch.desc[c], tasks,
                                  l.n, stream, err))
      return -1;
  }
  return 0;
}

int moment_count(MomentPlan& plan, unsigned long long* total,
                 hipStream_t stream, std::string* err) {
  hipLaunchKernelGGL(moment_count_kernel, dim3(2048), dim3(256), 0, stream,
                     plan.blocks, (int64_t)plan.n_groups * 64, total);
  BAND_TRY(hipGetLastError());
  return 0;
}

}  // namespace strip
