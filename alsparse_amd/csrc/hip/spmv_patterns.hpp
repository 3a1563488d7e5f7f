// CSR SpMV for matrices whose rows follow few patterns, for gfx950 (wave64): the distances (column - row) of a row's
// entries are one of at most kPatternSlots lists.  A discretisation on a grid has one list for its interior and a few
// for its boundary rows (5-point Laplacian: 9; 27-point stencil: 27), whatever the grid's size.
//
// The staged row blocks (spmv_rows.hpp) are bound by the bytes they stream, and a third to a half of those are column
// numbers.  With a pattern per row the columns cost ONE byte per row instead of four per entry, and the gathers of x
// no longer wait for a stream: a lane knows its columns as soon as its row's pattern is there, so they are
// issued beside the loads of the values, and lanes on neighbouring rows of one pattern read neighbouring elements of x.
// The structure is promised fixed (analysed matrices only); values stay in the caller's array.
//
// Bound by memory.  us per multiply over four matrices in turn, before (32-bit columns, 16-bit distances or the ELL copy,
// whichever the analysis kept) and now: 5-point Laplacian 2048^2 fp64 67.4 -> 47.0 (239 MB moved, 5.1 TB/s), fp32
// 49.6 -> 27.7; 27-point stencil of 101 x 100 x 97 points complex64 72.5 -> 48.6, fp64 69.9 -> 49.0; of 160^3 points fp32
// 179 -> 101; of 60 x 50 x 47 points fp32 10.7 -> 6.2.  Rows far shorter than the longest, and small matrices, stay with
// the columns (patterns_pay in plan.c).  16-byte values: the ELL copy stays
// ahead (5-point Laplacian of 2.1 M rows 58.7 against 84.4).
//
// The reference has no counterpart (src/kernel/dcu/level2/mv/csrmv/dcu_gemv_vector.h:14-57 reads every column).
#pragma once

#include "device_utils.hpp"
#include "spmv_rows.hpp"

namespace asamd {

constexpr int kPatternSlots = 256;   // a pattern's number is one byte
constexpr int kPatternWaves = kStreamRows / kWave;  // waves of a workgroup
constexpr int kPatternMaxLen = 64;   // entries per row; 64 KiB of distances at most, of which a matrix touches a few lines

// What the builder leaves in one allocation besides the rows' pattern numbers.
struct PatternScratch {
  unsigned long long key[kPatternSlots];  // hash of the slot's pattern, 0: free
  int row[kPatternSlots];                 // a row that has it
  int len[kPatternSlots];
  int fail;                               // set where some row found no slot, or differs from its slot's pattern
  int pad[3];
};

// One thread per row: the row's distances from LDS (the block's entries are one contiguous range, read with unit stride),
// hashed, and the hash looked up in an open-addressed table of 256 slots, entered where it is new.  Which slot a pattern
// gets depends on the order of arrival; nothing that a multiply computes does.  All slots are probed before the matrix is
// taken to have too many patterns: which of them a shorter search still reaches depends on the order of arrival as well.
static __global__ __launch_bounds__(kStreamRows) void pattern_rows_kernel(int m, int base, int rows_per_group,
                                                                          int max_len, const int* __restrict__ row_ptr,
                                                                          const int* __restrict__ col_ind,
                                                                          PatternScratch* __restrict__ tab,
                                                                          unsigned char* __restrict__ pid,
                                                                          int* __restrict__ block_off,
                                                                          int* __restrict__ wave_off) {
  extern __shared__ int s_col[];
  if (__atomic_load_n(&tab->fail, __ATOMIC_RELAXED)) return;
  const int64_t row0 = (int64_t)blockIdx.x * rows_per_group;
  int64_t row_last = row0 + rows_per_group;
  if (row_last > m) row_last = m;
  const int64_t lo = (int64_t)row_ptr[row0] - base;
  const int64_t n = (int64_t)row_ptr[row_last] - base - lo;
  if (n < 0 || n > (int64_t)rows_per_group * max_len) {  // (not the offsets that the row statistics were taken from)
    if (threadIdx.x == 0) atomicOr(&tab->fail, 1);
    return;
  }
  if (threadIdx.x == 0) {
    block_off[blockIdx.x] = (int)lo;
    if (row_last == m) block_off[blockIdx.x + 1] = (int)(lo + n);
  }
  if ((int)threadIdx.x < kPatternWaves) {
    const int64_t r = row0 + (int64_t)threadIdx.x * (rows_per_group / kPatternWaves);
    wave_off[(int64_t)blockIdx.x * kPatternWaves + threadIdx.x] = r < m ? row_ptr[r] - base : (int)(lo + n);
    if (row_last == m && threadIdx.x == 0) wave_off[((int64_t)blockIdx.x + 1) * kPatternWaves] = (int)(lo + n);
  }
  for (int k = threadIdx.x; k < (int)n; k += kStreamRows) s_col[k] = col_ind[lo + k];
  __syncthreads();
  const int64_t row = row0 + threadIdx.x;
  if ((int)threadIdx.x >= rows_per_group || row >= m) return;
  const int64_t first = (int64_t)row_ptr[row] - base - lo, last = (int64_t)row_ptr[row + 1] - base - lo;
  const int len = (int)(last - first);
  if (first < 0 || last > n || len < 1 || len > max_len) {
    atomicOr(&tab->fail, 1);
    return;
  }
  unsigned long long h = 0x9E3779B97F4A7C15ull * (unsigned)len;
  for (int s = 0; s < len; ++s) {
    const unsigned d = (unsigned)(s_col[first + s] - base - (int)row);
    h = (h ^ d) * 0xFF51AFD7ED558CCDull;
    h ^= h >> 32;
  }
  const unsigned long long key = h | 1;  // never 0
  int slot = (int)(h >> 56);
  for (int p = 0; p < kPatternSlots; ++p, slot = (slot + 1) % kPatternSlots) {
    if (p % 32 == 31 && __atomic_load_n(&tab->fail, __ATOMIC_RELAXED)) return;  // (a table that others found full)
    unsigned long long seen = __atomic_load_n(&tab->key[slot], __ATOMIC_RELAXED);
    if (seen == 0) {
      seen = atomicCAS(&tab->key[slot], 0ull, key);
      if (seen == 0) {
        tab->row[slot] = (int)row;
        tab->len[slot] = len;
        seen = key;
      }
    }
    if (seen == key) {
      pid[row] = (unsigned char)slot;
      return;
    }
  }
  atomicOr(&tab->fail, 1);
}

// dist[slot * stride + s] = the s-th distance of the slot's pattern (its last one repeated up to the stride), and behind
// all of them the patterns' lengths.  A workgroup of one wave per slot.
static __global__ __launch_bounds__(kWave) void pattern_table_kernel(int base, int stride, const int* __restrict__ row_ptr,
                                                                     const int* __restrict__ col_ind,
                                                                     const PatternScratch* __restrict__ tab,
                                                                     int* __restrict__ dist) {
  const int slot = blockIdx.x;
  if (tab->fail || tab->key[slot] == 0) return;
  const int row = tab->row[slot], len = tab->len[slot];
  const int64_t begin = (int64_t)row_ptr[row] - base;
  for (int s = threadIdx.x; s < stride; s += kWave)
    dist[slot * stride + s] = col_ind[begin + (s < len ? s : len - 1)] - base - row;
  if (threadIdx.x == 0) dist[kPatternSlots * stride + slot] = len;
}

// Every row against its pattern, entry by entry: the table is exact, whatever the hashes did.
static __global__ __launch_bounds__(kStreamRows) void pattern_verify_kernel(int m, int base, int rows_per_group, int stride,
                                                                            const int* __restrict__ row_ptr,
                                                                            const int* __restrict__ col_ind,
                                                                            const unsigned char* __restrict__ pid,
                                                                            const int* __restrict__ dist,
                                                                            PatternScratch* __restrict__ tab) {
  extern __shared__ int s_col[];
  if (__atomic_load_n(&tab->fail, __ATOMIC_RELAXED)) return;
  const int64_t row0 = (int64_t)blockIdx.x * rows_per_group;
  int64_t row_last = row0 + rows_per_group;
  if (row_last > m) row_last = m;
  const int64_t lo = (int64_t)row_ptr[row0] - base;
  const int n = (int)((int64_t)row_ptr[row_last] - base - lo);  // (in range: pattern_rows_kernel looked)
  for (int k = threadIdx.x; k < n; k += kStreamRows) s_col[k] = col_ind[lo + k];
  __syncthreads();
  const int64_t row = row0 + threadIdx.x;
  if ((int)threadIdx.x >= rows_per_group || row >= m) return;
  const int first = (int)((int64_t)row_ptr[row] - base - lo), len = row_ptr[row + 1] - row_ptr[row];
  const int slot = pid[row];
  bool same = len == tab->len[slot];
  for (int s = 0; same && s < len; ++s) same = s_col[first + s] - base - (int)row == dist[slot * stride + s];
  if (!same) atomicOr(&tab->fail, 1);
}

// y = alpha*A*x + beta*y.  256 / G rows per workgroup as in the staged row blocks: their values are one contiguous range,
// streamed into LDS with 128-bit loads that are all in flight at once, G lanes sum a row.  U: entries per lane (rows of at
// most U * G entries), dist, lens: `stride` distances and a length per pattern, wave_off: where every wave's entries
// begin -- words that the neighbours' loads have brought to the L2, so that the values wait for nothing from memory.
// Where a row begins inside its wave's entries is the sum of the lengths before it, and row_ptr is not read.  us with it /
// without, three sets of arrays in turn: 5-point Laplacian 2048^2 fp64 50.8 / 46.8, 3000 x 3001 fp64 108 / 97.4; 27-point
// stencil 101 x 100 x 97 complex64 51.6 / 48.6, 160^3 fp32 107.9 / 102 (a length in front of its distances: 48.5 and 50.3
// for the first and the third; workgroups that take several blocks and load the next one's values while they add one up:
// 54 and 56).  NTV: the values bypass the caches.  val 16-byte aligned.
// EARLY: for matrices that the caches hold, where the chain pattern - distances - x counts and not the bytes: the pattern's
// number is asked for in front of the wait for the starts, and nothing on the way to x waits for a load of its own.  us,
// without / with: 27-point stencil 50 x 51 x 48 fp64 8.2 / 7.7, 64 x 65 x 62 fp64 13.1 / 12.4, fp32 7.8 / 7.4, 5-point Laplacian
// 2048^2 fp32 (138 MB) 29.9 / 27.4; beyond the caches the values' requests, which then stand behind the distances' and x',
// are what counts: stencil 90 x 91 x 88 fp64 (163 MB) 36.3 / 36.3, 101 x 100 x 97 complex64 48.1 / 48.4, Laplacian 2600 x 2601
// fp64 73.7 / 75.5.
template <typename T, int U, int G, bool NTV, bool EARLY>
__global__ __launch_bounds__(kStreamRows) void spmv_pattern_kernel(
    int m, T alpha, const T* __restrict__ val, const unsigned char* __restrict__ pid, const int* __restrict__ dist, int stride,
    const int* __restrict__ lens, const int* __restrict__ wave_off, const T* __restrict__ x, T beta, T* __restrict__ y) {
  constexpr int kRows = kStreamRows / G;
  constexpr int kPer = 16 / (int)sizeof(T);       // values per 128-bit piece
  constexpr int kStaged = kStreamRows * U / kPer + 1;  // pieces of a block: one more for the values in front of its first
  constexpr int kPieces = (kStaged + kStreamRows - 1) / kStreamRows;
  __shared__ Int4 s_words[kStaged];
  const unsigned bid = xcd_contiguous_id(blockIdx.x, gridDim.x);
  const int64_t row0 = (int64_t)bid * kRows;
  const int lane = threadIdx.x % G;
  const int64_t row = row0 + threadIdx.x / G;
  const int64_t my_row = row < m ? row : (int64_t)m - 1;
  const int* __restrict__ starts = wave_off + (int64_t)bid * kPatternWaves;
  const int e0 = starts[0], e1 = starts[kPatternWaves];  // at most kStreamRows * U apart: the builder looked
  const int mine0 = starts[__builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave)];
  const int pattern = pid[my_row];
  if constexpr (EARLY) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::"s"(mine0));  // (left alone, the compiler loads it behind the barrier, where it is needed)
  }
  // The values through a buffer resource that ends with the block: the pieces past its end come back as zeros without a
  // request and without a condition, so that all loads are in flight before the first wait.
  const int a0 = e0 & ~(kPer - 1);
  const BufferRsrc block = make_rsrc(val + a0, (e1 - a0) * (int)sizeof(T));
  Int4 v[kPieces];
#pragma unroll
  for (int s = 0; s < kPieces; ++s) v[s] = buffer_load<Int4, NTV ? 2 : 0>(block, 16 * (threadIdx.x + s * kStreamRows));
  __builtin_amdgcn_sched_barrier(0);  // (left alone, the compiler waits for the pattern's number first)
  // The row's columns, without a condition too: a lane past its row's end takes the last distance again, and what it
  // reads with it is not added below.
  const int* __restrict__ d = dist + pattern * stride;
  const T* __restrict__ xr = x + my_row;
  int len;
  if constexpr (EARLY) {
    const int pattern_len = lens[pattern];  // (no load under a condition: the loads behind it would wait for the branch)
    len = row < m ? pattern_len : 0;
  } else {
    len = row < m ? lens[pattern] : 0;
  }
  int off[U];
  T xv[U];
#pragma unroll
  for (int u = 0; u < U; ++u) off[u] = d[lane + u * G < stride ? lane + u * G : stride - 1];
#pragma unroll
  for (int u = 0; u < U; ++u) xv[u] = xr[off[u]];
#pragma unroll
  for (int s = 0; s < kPieces; ++s) {
    if constexpr (EARLY) asm volatile("" ::"v"(v[s].x));  // (not loaded under the condition either)
    if (threadIdx.x + s * kStreamRows < kStaged) s_words[threadIdx.x + s * kStreamRows] = v[s];
  }
  const int first = mine0 + wave_sum_scan(lane == 0 ? len : 0) - len;
  __syncthreads();
  if (row >= m) return;  // whole lane groups leave together
  const T* mine = reinterpret_cast<const T*>(s_words) + (first - a0);
  T mv[U];
#pragma unroll
  for (int u = 0; u < U; ++u) mv[u] = mine[lane + u * G < len ? lane + u * G : 0];
  T sum = T(0);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const T next = fma_t(mv[u], xv[u], sum);
    sum = lane + u * G < len ? next : sum;
  }
  if constexpr (G > 1) sum = group_sum<G>(sum);
  if (lane == 0) store_axpby(y, row, alpha, sum, beta);
}

}  // namespace asamd
