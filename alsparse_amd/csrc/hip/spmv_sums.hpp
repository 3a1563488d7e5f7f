// Tiled two-phase CSR SpMV whose first phase adds up (gfx950, wave64): for rows that put several entries into one
// column block -- long rows, power-law graphs, whose popular columns sit side by side.
//
// The tiled pair (spmv_tiled.hpp) writes one product per entry and reads it back.  Where a row meets a column block
// more than once those products belong to the same sum, and in tile order (column block, row block, then CSR order)
// they are neighbours: here the wave that forms them adds them up in registers and writes ONE value per (row, column
// block).  On a power-law graph (8 M rows, rows up to 200 000 entries, R-MAT columns, 96 M entries) that leaves 37 M
// values, no tile longer than its rows, and no two values of one run for the same row: the second phase has neither
// long tiles nor equal rows to combine.  531 us with merge-path and the popular columns in LDS -> 232 us here (162 for
// phase 1, 5.4 TB/s through the L2; 70 for phase 2).
//
//   phase 1  sums_products_kernel   one workgroup per chunk of a column block, the block's x slice in LDS (128 KiB).  A
//            wave takes spans of 2048 consecutive entries, 1024 at a time: 128-bit pieces of values, the 16-bit local
//            columns, whose highest bit marks the last entry of a sum.  A lane adds up its consecutive entries, a
//            segmented scan on DPP moves carries open sums from lane to lane, and the finished sums leave through a
//            staging area in LDS as one unit-stride run.  Sums end with their span, so a wave needs nothing from its
//            neighbours; a row that crosses spans leaves one value in each.
//   phase 2  tiled_reduce_kernel    the one of the tiled pair, over a list of runs of at most 64 values per row
//            block instead of a table of tiles: empty tiles are not visited, long ones are several runs.
//
// Traffic per fp32 entry: 6 bytes + 10 per sum.  The order of every addition is fixed by the layout.  The reference
// has no counterpart; its one kernel is a lane group per row (src/kernel/dcu/level2/mv/csrmv/dcu_gemv_vector.h:14-57).
#pragma once

#include "spmv_tiled.hpp"

namespace asamd {

constexpr int kSumsSliceBytes = 128 * 1024;  // x slice; with 4-byte values 32 768 columns, which leaves bit 15 free
constexpr unsigned kSumsLast = 0x8000u;      // in a local column: the entry is the last one of its sum
constexpr int kSumsWaves = kProdThreads / kWave;
constexpr int kSumsStageBytes = (kLdsPerCu - kSumsSliceBytes) / kSumsWaves;  // a wave's staging area

template <typename T>
struct SumsDims {
  static constexpr int cols = kSumsSliceBytes / (int)sizeof(T);  // width of every column block
  // A lane holds this many CONSECUTIVE entries of a trip: the sums inside a lane cost an addition each, and only one scan
  // over the lanes is needed per trip (one per 256 entries, with four entries per lane: 172 us for phase 1 on the graph
  // above where this form took 166).
  static constexpr int lane = sizeof(T) == 16 ? 8 : 16;
  static constexpr int trip = lane * kWave;  // slots a wave takes at a time
  // Open sums pass from trip to trip in registers and end with the span.  A row with thousands of entries in one column
  // block leaves a value per span, and a run of its own for each: with spans of one trip the waves of phase 2 that hold
  // the longest rows end last by two thirds (75 us against 70; four trips: 69, but phase 1 loses as much, its waves less
  // even at the ends of the column blocks).
  static constexpr int trips = 2;
  static constexpr int span = trip * trips;
  static constexpr int stage = kSumsStageBytes / (int)sizeof(T);
  static_assert(cols <= (int)kSumsLast, "a local column and the mark share 16 bits");
};
constexpr int log2_of(int v) { return v <= 1 ? 0 : 1 + log2_of(v / 2); }

// Where a span keeps its slots, trip by trip: lane l of the wave holds slots l * lane ... of a trip, and its i-th 128-bit
// piece of values lies beside the other lanes' i-th pieces, so that a load instruction moves 1 KiB of consecutive bytes.  (The columns go
// the same way, in the same pieces of Piece<T>::n.)
template <typename T>
__host__ __device__ __forceinline__ int sums_place(int slot) {
  constexpr int kPer = Piece<T>::n;
  const int l = slot % SumsDims<T>::trip / SumsDims<T>::lane, j = slot % SumsDims<T>::lane;
  return slot / SumsDims<T>::trip * SumsDims<T>::trip + (j / kPer * kWave + l) * kPer + j % kPer;
}

struct SumsChunk {
  int col0, ncols;   // the chunk's column block
  int span0;         // its first span
  int slots;         // entries
};

// ---- analysis ----------------------------------------------------------------
// count[g] = sums that the rows 64 g .. 64 g + 63 leave: changes of column block along their entries.  Exact for
// ascending columns (apart from sums cut at span ends), an upper bound otherwise.  One workgroup per group.
static __global__ __launch_bounds__(256) void sums_count_kernel(int m, const int* __restrict__ row_ptr,
                                                                const int* __restrict__ col_ind, int base, int shift,
                                                                int* __restrict__ count) {
  __shared__ int s_n[256 / kWave];
  const int64_t r0 = (int64_t)blockIdx.x << kRowGroupLog2;
  const int rows = (int)(m - r0 < (1 << kRowGroupLog2) ? m - r0 : (1 << kRowGroupLog2));
  const int lo = row_ptr[r0] - base, hi = row_ptr[r0 + rows] - base;
  int n = 0;
#pragma unroll 4
  for (int64_t k = (int64_t)lo + threadIdx.x; k < hi; k += 256)
    n += k == lo || ((col_ind[k] - base) >> shift) != ((col_ind[k - 1] - base) >> shift);
  if ((int)threadIdx.x < rows) {
    const int s = row_ptr[r0 + threadIdx.x] - base, e = row_ptr[r0 + threadIdx.x + 1] - base;
    if (s < e && s > lo && ((col_ind[s] - base) >> shift) == ((col_ind[s - 1] - base) >> shift)) ++n;
  }
  for (int d = kWave / 2; d > 0; d >>= 1) n += __shfl_down(n, d, kWave);
  if (threadIdx.x % kWave == 0) s_n[threadIdx.x / kWave] = n;
  __syncthreads();
  if (threadIdx.x == 0) count[blockIdx.x] = s_n[0] + s_n[1] + s_n[2] + s_n[3];
}

// key and payload of every entry, as tile_keys_payload_kernel; the column blocks are all equally wide
static __global__ __launch_bounds__(256) void sums_keys_kernel(int nnz, const int* __restrict__ coo_row,
                                                               const int* __restrict__ col_ind, int base, int shift,
                                                               const int* __restrict__ row_group_block,
                                                               const int* __restrict__ row_block_start, int row_blocks,
                                                               unsigned* __restrict__ key,
                                                               unsigned long long* __restrict__ payload) {
  for (int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x; k < nnz; k += (int64_t)gridDim.x * 256) {
    const int col = col_ind[k] - base, row = coo_row[k] - base;
    const int rb = row_group_block[row >> kRowGroupLog2];
    key[k] = (unsigned)(col >> shift) * (unsigned)row_blocks + (unsigned)rb;
    payload[k] = ((unsigned long long)(unsigned)k << 32) | ((unsigned)(col & ((1 << shift) - 1)) << 16) |
                 (unsigned)(row - row_block_start[rb]);
  }
}

// The entries [lo, hi) (in sorted order) of a span: column block c has the spans from col_span[c] on, the entries from
// col_ptr[c] on.
struct SpanEntries {
  int lo, hi;
};
static __device__ __forceinline__ SpanEntries span_entries(int span, int span_slots, int col_blocks,
                                                           const int* __restrict__ col_span,
                                                           const int* __restrict__ col_ptr) {
  int c = 0, above = col_blocks;  // the last column block whose first span is <= span
  while (above - c > 1) {
    const int mid = (c + above) / 2;
    if (col_span[mid] <= span) c = mid;
    else above = mid;
  }
  const int64_t lo = (int64_t)col_ptr[c] + (int64_t)(span - col_span[c]) * span_slots;
  const int64_t end = col_ptr[c + 1];
  return {(int)lo, (int)(lo + span_slots < end ? lo + span_slots : end)};
}

// count[span] = sums of a span: its entries that are followed by another row, tile or span.  One wave per span.
static __global__ __launch_bounds__(256) void sums_span_count_kernel(int spans, int span_slots, int col_blocks,
                                                                     const int* __restrict__ col_span,
                                                                     const int* __restrict__ col_ptr,
                                                                     const unsigned* __restrict__ key,
                                                                     const unsigned long long* __restrict__ payload,
                                                                     int* __restrict__ count) {
  const int lane = threadIdx.x % kWave;
  const int span = blockIdx.x * (256 / kWave) + threadIdx.x / kWave;
  if (span >= spans) return;  // wave-uniform
  const SpanEntries at = span_entries(span, span_slots, col_blocks, col_span, col_ptr);
  int n = 0;
  for (int64_t k = (int64_t)at.lo + lane; k < at.hi; k += kWave)
    n += k + 1 == at.hi || key[k + 1] != key[k] || (unsigned short)payload[k + 1] != (unsigned short)payload[k];
  for (int d = kWave / 2; d > 0; d >>= 1) n += __shfl_down(n, d, kWave);
  if (lane == 0) count[span] = n;
}

// Lays out the spans: columns with their marks, CSR positions (-1 where a span has no entry; in place, like the
// columns), and per sum its row; first_sum[entry] = sums that end before it.  One wave per span.
template <typename T>
__global__ __launch_bounds__(256) void sums_spans_kernel(int spans, int col_blocks, const int* __restrict__ col_span,
                                                         const int* __restrict__ col_ptr, const int* __restrict__ span_sum,
                                                         const unsigned* __restrict__ key,
                                                         const unsigned long long* __restrict__ payload,
                                                         unsigned short* __restrict__ t_col, unsigned* __restrict__ t_perm,
                                                         unsigned short* __restrict__ s_row, int* __restrict__ first_sum) {
  const int lane = threadIdx.x % kWave;
  const int span = blockIdx.x * (256 / kWave) + threadIdx.x / kWave;
  if (span >= spans) return;  // wave-uniform
  constexpr int kSpan = SumsDims<T>::span;
  const SpanEntries at = span_entries(span, kSpan, col_blocks, col_span, col_ptr);
  const int64_t home = (int64_t)span * kSpan;
  int before = span_sum[span];
  for (int s0 = 0; s0 < kSpan; s0 += kWave) {
    const int s = s0 + lane;
    const int64_t k = (int64_t)at.lo + s;
    const bool ok = k < at.hi;
    const unsigned long long w = ok ? payload[k] : 0ull;
    const bool last = ok && (k + 1 == at.hi || key[k + 1] != key[k] || (unsigned short)payload[k + 1] != (unsigned short)w);
    const uint64_t ends = __builtin_amdgcn_ballot_w64(last);
    const int mine = before + __builtin_popcountll(ends & (((uint64_t)1 << lane) - 1));
    const int64_t q = home + sums_place<T>(s);
    t_col[q] = (unsigned short)((unsigned)(w >> 16) & (kSumsLast - 1) | (last ? kSumsLast : 0u));
    t_perm[q] = ok ? (unsigned)(w >> 32) : ~0u;
    if (ok) first_sum[k] = mine;
    if (last) s_row[mine] = (unsigned short)w;
    before += __builtin_popcountll(ends);
  }
}

// t_val[q] = val[t_perm[q]], zero where a span has no entry.  One workgroup per span at a time; `order` lists the spans so
// that those of all column blocks that hold the same rows follow each other, and every XCD takes a stretch of that list:
// what it works on at one time picks from one stretch of val.  gate as for gather_values_kernel; gridDim.x: a multiple of
// the XCDs.
template <typename T>
__global__ __launch_bounds__(256) void sums_values_kernel(int spans, const int* __restrict__ order,
                                                          const unsigned* __restrict__ t_perm, const T* __restrict__ val,
                                                          T* __restrict__ t_val, GuardGate gate) {
  if (!guard_open(gate)) return;
  constexpr int kSpan = SumsDims<T>::span, kU = kSpan / 256;
  static_assert(kSpan % 256 == 0, "whole workgroups");
  const int xcd = blockIdx.x % kXcds, per = (spans + kXcds - 1) / kXcds;
  const int end = (xcd + 1) * per < spans ? (xcd + 1) * per : spans;
  for (int i = xcd * per + (int)(blockIdx.x / kXcds); i < end; i += (int)(gridDim.x / kXcds)) {
    const int64_t q = (int64_t)order[i] * kSpan + threadIdx.x;
    unsigned k[kU];
    T v[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) k[u] = nt_load(t_perm + q + u * 256);
#pragma unroll
    for (int u = 0; u < kU; ++u) v[u] = k[u] != ~0u ? val[k[u]] : T(0);
#pragma unroll
    for (int u = 0; u < kU; ++u) nt_store(v[u], t_val + q + u * 256);
  }
}

// The runs of row block rb, at most 64 sums each and none with two sums of one row (a row whose entries cross spans), in
// column block order: counted (runs == nullptr), or written from run_ptr[rb] on.  One lane per row block: neighbouring
// lanes read neighbouring tiles.
static __global__ __launch_bounds__(64) void sums_runs_kernel(int row_blocks, int col_blocks, int nnz, int sums,
                                                              int span_slots, const int* __restrict__ col_span,
                                                              const int* __restrict__ col_ptr,
                                                              const int* __restrict__ span_sum,
                                                              const unsigned short* __restrict__ s_row,
                                                              const int* __restrict__ tile_ptr,
                                                              const int* __restrict__ first_sum,
                                                              const int* __restrict__ run_ptr, int* __restrict__ count,
                                                              TileRange* __restrict__ runs) {
  const int rb = blockIdx.x * 64 + threadIdx.x;
  if (rb >= row_blocks) return;
  int at = runs ? run_ptr[rb] : 0;
  for (int c = 0; c < col_blocks; ++c) {
    const int64_t t = (int64_t)c * row_blocks + rb;
    const int s0 = tile_ptr[t], s1 = tile_ptr[t + 1];
    if (s0 == s1) continue;
    const int hi = s1 < nnz ? first_sum[s1] : sums;
    int lo = first_sum[s0];
    int span = (s0 - col_ptr[c]) / span_slots + 1;  // the next span that begins, in this column block
    while (lo < hi) {
      int cut = hi;  // the tile's sums up to the next span that begins with the row the one before ended with
      for (; cut == hi && (int64_t)col_ptr[c] + (int64_t)span * span_slots < s1; ++span) {
        const int p = span_sum[col_span[c] + span];
        if (p > lo && p < hi && s_row[p] == s_row[p - 1]) cut = p;
      }
      if (runs) {
        for (int b = lo; b < cut; b += kWave) {
          runs[at].begin = b;
          runs[at].end = b + kWave < cut ? b + kWave : cut;
          ++at;
        }
      } else {
        at += (cut - lo + kWave - 1) / kWave;
      }
      lo = cut;
    }
  }
  if (!runs) count[rb] = at;
}

// ---- phase 1 -------------------------------------------------------------------
// Bounds: the streams, 6 bytes per fp32 entry in and 4 per sum out.  The next trip's loads are in flight while one is
// worked on.  A span without all its entries ends in slots that no mark follows: what they form is never stored.
// NTS: the sums are stored past the memory-side cache; NTL: the values and columns are loaded past it (asamd_spmv_sums).
template <typename T, bool NTS, bool NTL>
__global__ __launch_bounds__(kProdThreads) void sums_products_kernel(
    const SumsChunk* __restrict__ chunks, const int* __restrict__ span_sum, const T* __restrict__ t_val,
    const unsigned short* __restrict__ t_col, const T* __restrict__ x, T* __restrict__ out) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int kPer = Piece<T>::n, kLane = SumsDims<T>::lane, kTrip = SumsDims<T>::trip, kPieces = kLane / kPer;
  constexpr int kStage = SumsDims<T>::stage;
  T* xs = reinterpret_cast<T*>(smem);
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  T* stage = xs + SumsDims<T>::cols + wave * kStage;
  const SumsChunk ch = chunks[blockIdx.x];
  struct alignas(2 * kPer) ColPiece {
    unsigned short c[kPer];
  };
  Piece<T> v[kPieces];
  ColPiece c[kPieces];
  // the wave's slots of the chunk, a trip at a time: spans wave, wave + 16, ...
  int at = wave * SumsDims<T>::span;
  auto load = [&](int first) {
    const int64_t q = (int64_t)ch.span0 * SumsDims<T>::span + first + lane * kPer;
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const auto* pv = reinterpret_cast<const Piece<T>*>(t_val + q + i * kWave * kPer);
      const auto* pc = reinterpret_cast<const ColPiece*>(t_col + q + i * kWave * kPer);
      if constexpr (NTL) {
        v[i] = nt_load_object(pv);
        c[i] = nt_load_object(pc);
      } else {
        v[i] = *pv;
        c[i] = *pc;
      }
    }
  };
  if (at < ch.slots) load(at);
  {
    // x slice -> LDS, all of a thread's loads in flight before the first LDS write (as in tiled_products_kernel)
    constexpr int kSlicePieces = SumsDims<T>::cols / kPer / kProdThreads;
    static_assert(kSlicePieces >= 1 && SumsDims<T>::cols % (kPer * kProdThreads) == 0, "slice layout");
    const T* xsrc = x + (int64_t)ch.col0;
    const int whole = ch.ncols / kPer;
    LoosePiece<T> tmp[kSlicePieces];
#pragma unroll
    for (int u = 0; u < kSlicePieces; ++u) {
      const int q = threadIdx.x + u * kProdThreads;
      if (q < whole) tmp[u] = *reinterpret_cast<const LoosePiece<T>*>(xsrc + q * kPer);
    }
#pragma unroll
    for (int u = 0; u < kSlicePieces; ++u) {
      const int q = threadIdx.x + u * kProdThreads;
      if (q < whole) {
        unsigned* dst = reinterpret_cast<unsigned*>(xs + q * kPer);
#pragma unroll
        for (int i = 0; i < 4; ++i) dst[i] = tmp[u].w[i];
      }
    }
    const int rest = whole * kPer + threadIdx.x;
    if (rest < ch.ncols) xs[rest] = xsrc[rest];
  }
  __syncthreads();
  int64_t dst = 0;
  T open = T(0);  // the sum that the trip before left open
  while (at < ch.slots) {
    if (at % SumsDims<T>::span == 0) {
      dst = span_sum[ch.span0 + at / SumsDims<T>::span];
      open = T(0);
    }
    int next = at + kTrip;
    if (next % SumsDims<T>::span == 0) next += (kSumsWaves - 1) * SumsDims<T>::span;
    // running sums of the lane's entries: res[e] is complete where entry e ends a sum
    T res[kLane];
    unsigned marks = 0;  // bit e: entry e ends a sum
    T sum = T(0);
#pragma unroll
    for (int e = 0; e < kLane; ++e) {
      const unsigned cc = c[e / kPer].c[e % kPer];
      sum = sum + v[e / kPer].e[e % kPer] * xs[cc & (kSumsLast - 1)];
      res[e] = sum;
      const bool last = (cc & kSumsLast) != 0;
      marks |= last ? 1u << e : 0u;
      sum = last ? T(0) : sum;
    }
    if (next < ch.slots) load(next);
    // open sums travel from lane to lane: a lane with an end starts afresh behind it
    if (lane == 0 && marks == 0) sum = open + sum;
    const T run = segmented_scan(sum, marks != 0);
    T in = dpp_mov<0x138>(run);  // wave_shr:1: what the lanes below left open
    if (lane == 0) in = open;
    open = lane_bcast(run, kWave - 1);
    const int mine = __builtin_popcount(marks);
    const int upto = wave_sum_scan(mine);  // sums that end in this lane and below
    const int n = lane_bcast(upto, kWave - 1);
    // through LDS, so that they leave side by side; more than the area holds in several turns
    for (int base = 0; base < n; base += kStage) {
      int to = upto - mine - base;
      bool first = true;
#pragma unroll
      for (int e = 0; e < kLane; ++e)
        if ((marks >> e) & 1) {
          if ((unsigned)to < (unsigned)kStage) stage[to] = first ? in + res[e] : res[e];
          first = false;
          ++to;
        }
      wave_lds_fence();
      const int here = n - base < kStage ? n - base : kStage;
      for (int u = lane; u < here; u += kWave) {
        if constexpr (NTS) nt_store(stage[u], out + dst + base + u);
        else out[dst + base + u] = stage[u];
      }
      wave_lds_fence();
    }
    dst += n;
    at = next;
  }
}

}  // namespace asamd
