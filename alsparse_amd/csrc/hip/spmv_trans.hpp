// Transposed CSR SpMV, y = alpha*A^T*x + beta*y (A is m x n: x has m entries, y has n).
//
// Two routes:
//   * a CSR copy of A^T built once by the analysis (stable radix sort of the
//     entries by column, so rows stay ascending inside every column and the
//     layout is deterministic); multiplies then run the ordinary row kernels on
//     that copy: same bytes, same rooflines, bit-reproducible.
//   * without such a copy, the scatter below: y is scaled by beta, then every
//     entry adds alpha*val*x[row] to y[col] with a hardware float atomic.  This
//     is what the reference always does, one lane per row
//     (src/kernel/dcu/level2/mv/csrmv/dcu_gemv_x_csr_trans.cpp:11-45; its beta
//     pass covers m elements of y where n are meant, :61-64); here W lanes share
//     a row so that the entry loads coalesce.  CONJ conjugates the values on
//     the way: y = alpha*A^H*x + beta*y, the reference's
//     csr_gemv_conj_scalar_atomicadd (dcu_gemv_c_csr_conj.cpp:22-48).
#pragma once

#include "device_utils.hpp"

namespace asamd {

// key[k] = zero-based column of entry k, idx[k] = k
static __global__ __launch_bounds__(256) void transpose_keys_kernel(int nnz, const int* __restrict__ col_ind, int base,
                                                             unsigned* __restrict__ key,
                                                             unsigned* __restrict__ idx) {
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < nnz;
       k += (int64_t)gridDim.x * blockDim.x) {
    key[k] = (unsigned)(col_ind[k] - base);
    idx[k] = (unsigned)k;
  }
}

// entries of A^T in column-sorted order: zero-based row of A as the new column index
// (CONJ: values conjugated, which makes the copy A^H)
template <typename T, bool CONJ>
__global__ __launch_bounds__(256) void transpose_gather_kernel(int nnz, const unsigned* __restrict__ perm,
                                                               const int* __restrict__ coo_row,
                                                               const T* __restrict__ val, int base,
                                                               int* __restrict__ t_col, T* __restrict__ t_val) {
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < nnz;
       q += (int64_t)gridDim.x * blockDim.x) {
    const unsigned k = perm[q];
    t_col[q] = coo_row[k] - base;
    t_val[q] = CONJ ? conj_t(val[k]) : val[k];
  }
}

// y <- beta*y over n elements (beta == 0 stores zeros without reading)
template <typename T>
__global__ __launch_bounds__(256) void scale_vec_kernel(int n, T beta, T* __restrict__ y) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  y[i] = beta == T(0) ? T(0) : y[i] * beta;
}

// Sums in LDS are held in double precision whatever the values are: an LDS atomic on doubles is several times as fast as
// one on floats (the same 7 000 entries in one workgroup: 4 us against 9), and rounds less.
template <typename T>
using LdsSum = std::conditional_t<kIsReal<T>, double, Cx<double>>;
__device__ __forceinline__ double widened(float a) { return a; }
__device__ __forceinline__ double widened(double a) { return a; }
template <typename R>
__device__ __forceinline__ Cx<double> widened(Cx<R> a) { return Cx<double>(a.re, a.im); }
template <typename T>
__device__ __forceinline__ T narrowed(double a) { return T(a); }
template <typename T>
__device__ __forceinline__ T narrowed(Cx<double> a) { return T(a.re, a.im); }

// ---- without a copy: a scatter whose workgroups add up a column's entries before they leave the compute unit ----------
// What bounds a scatter is its atomics: they are carried out in memory, a line's one after another.  W lanes share a row,
// K rows of a lane group are in flight, and every entry goes to its column's slot of a table in LDS (a slot takes the
// first column that comes; another one's entries go straight to y).  Neighbouring rows of a discretisation share columns,
// and what is left leaves as neighbouring columns of one instruction.  Without TABLE every entry goes straight to y.
// `blocks` is the grid: a kernel that asks gridDim brings 256 bytes of hidden arguments, which the host writes on every
// launch, and small products are launches alone (A^T of the 5-point Laplacian on 70 x 90 points, fp32: 7.2 us a call with
// gridDim, 6.7 without).
constexpr int kTransThreads = 256;

template <typename T, int W, int K, bool CONJ, bool TABLE = true>
__global__ __launch_bounds__(kTransThreads) void csrmv_trans_scatter_kernel(
    int m, int n, T alpha, const T* __restrict__ val, const int* __restrict__ row_ptr,
    const int* __restrict__ col_ind, const T* __restrict__ x, T* __restrict__ y, int base, unsigned blocks) {
  constexpr int kGroups = kTransThreads / W;
  constexpr int kSlots = TABLE ? 512 * K : 1;
  __shared__ int s_key[kSlots];
  __shared__ LdsSum<T> s_sum[kSlots];
  const int64_t row0 = (int64_t)xcd_contiguous_id(blockIdx.x, blocks) * (kGroups * K) + threadIdx.x / W;
  const int sub = threadIdx.x % W;
  int64_t b[K], e[K];
  T t[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int64_t r = row0 + k * kGroups;
    b[k] = (int64_t)row_ptr[r < m ? r : m] - base + sub;
    e[k] = (int64_t)row_ptr[r < m ? r + 1 : m] - base;
    t[k] = x[r < m ? r : 0];
  }
  if constexpr (TABLE) {
    for (int i = threadIdx.x; i < kSlots; i += kTransThreads) {
      s_key[i] = -1;
      s_sum[i] = LdsSum<T>(0);
    }
  }
  int c[K];
  T v[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {  // a lane's first entry of every row, all in flight
    c[k] = b[k] < e[k] ? col_ind[b[k]] - base : -1;
    v[k] = b[k] < e[k] ? val[b[k]] : T(0);
    t[k] = alpha * t[k];
  }
  if constexpr (TABLE) __syncthreads();
  auto add = [&](int col, T a, T tk) __attribute__((always_inline)) {
    if ((unsigned)col >= (unsigned)n) return;
    const T p = (CONJ ? conj_t(a) : a) * tk;
    if constexpr (!TABLE) {
      atomic_add(&y[col], p);
      return;
    }
    const int slot = col & (kSlots - 1);
    const int there = atomicCAS(&s_key[slot], -1, col);
    if (there == -1 || there == col) atomic_add(&s_sum[slot], widened(p));
    else atomic_add(&y[col], p);
  };
#pragma unroll
  for (int k = 0; k < K; ++k) add(c[k], v[k], t[k]);
#pragma unroll
  for (int k = 0; k < K; ++k)
    for (int64_t j = b[k] + W; j < e[k]; j += W) add(col_ind[j] - base, val[j], t[k]);
  if constexpr (!TABLE) return;
  __syncthreads();
  for (int i = threadIdx.x; i < kSlots; i += kTransThreads) {
    const int col = s_key[i];
    if (col >= 0) atomic_add(&y[col], narrowed<T>(s_sum[i]));
  }
}

// ---- without a copy: the columns in slices, a slice's sums in LDS -------------------------------------------------
// What bounds the scatter is its atomics: they are carried out in memory, a line's one after another, and a popular
// column's line gets most of them; and a lane group per row walks the longest row alone.  Here a workgroup takes one of
// `parts` equal pieces of the ENTRIES, however the rows cut them, and one of the slices of the columns: it reads every
// column number of its piece, multiplies what falls into its slice with alpha * x[row] and adds it to the column's sum in
// LDS.  With one part it writes y itself, else its sums go to partials + part * n and trans_partials_sum_kernel adds the
// parts in order.  Entries are read once per slice: a part's slices run on one XCD (parts a multiple of eight) and meet
// in its L2.
//
// Rows that start in a chunk mark their place, a running maximum names every entry's row.  That walk takes 0.86 us for
// 1 024 rows, and all rows of a run of empty ones fall to one part.  With GAPS the rows of a chunk are counted after
// kSliceWalk of them; more than kSliceLook are not walked (the walk to there takes what follows): the chunk's entries look
// their rows up, a thread its first one's among all, the others' between that and the next thread's.  us, scatter / without /
// with: 4 M rows, all 400 000 entries in the last 100 000 of them 78 / 3 300 / 37; 1 M rows, the second half of two entries
// each, 79 / 431 / 44; 20 M rows, every fortieth of two, 147 / 84 / 103; 200 000 rows, every second of eight, 62 / 18.5 / 19.3.
constexpr int kSliceThreads = 1024;
constexpr int kSlicePer = 8;  // entries per thread and chunk
constexpr int kSliceChunk = kSliceThreads * kSlicePer;
constexpr int kSliceWaves = kSliceThreads / kWave;
constexpr int kSliceWalk = 24 * kSliceThreads;
constexpr int kSliceLook = 40 * kSliceThreads;
constexpr int kSliceLdsFixed = (kSliceChunk + 2 * kSliceWaves) * (int)sizeof(int);
// largest r in [0, m) with row_ptr[r] - base <= k (0 if there is none): a whole wave, 64 probes at a time
static __device__ __forceinline__ int row_of_entry(int m, const int* __restrict__ row_ptr, int base, int64_t k) {
  const int lane = threadIdx.x % kWave;
  int64_t lo = 0, hi = m - 1;
  while (lo < hi) {
    const int64_t step = (hi - lo + kWave - 1) / kWave;
    const int64_t p = lo + (lane + 1) * step;
    const bool not_after = p <= hi && (int64_t)row_ptr[p <= hi ? p : hi] - base <= k;
    lo += __popcll(__builtin_amdgcn_ballot_w64(not_after)) * step;
    hi = lo + step - 1 < hi ? lo + step - 1 : hi;
  }
  return (int)lo;
}

template <typename T, bool CONJ, bool GAPS>
__global__ __launch_bounds__(kSliceThreads) void csrmv_trans_slices_kernel(
    int m, int n, int parts, int slice_cols, T alpha, const T* __restrict__ val, const int* __restrict__ row_ptr,
    const int* __restrict__ col_ind, const T* __restrict__ x, T beta, T* __restrict__ y, T* __restrict__ partials, int base) {
  extern __shared__ __align__(16) unsigned char slice_bytes[];
  int* __restrict__ s_row = reinterpret_cast<int*>(slice_bytes);
  int* __restrict__ s_part = s_row + kSliceChunk;  // a wave's largest mark
  int* __restrict__ s_first = s_part + kSliceWaves;
  int* __restrict__ s_more = s_first + 1;  // more rows start over the chunk than were walked
  using S = LdsSum<T>;
  S* __restrict__ s_sum = reinterpret_cast<S*>(slice_bytes + kSliceLdsFixed);

  const int tid = threadIdx.x, wave = tid / kWave;
  const int part = (int)(blockIdx.x % (unsigned)parts);
  const int64_t lo_col = (int64_t)(blockIdx.x / (unsigned)parts) * slice_cols;
  const int cols = (int)(lo_col + slice_cols < n ? slice_cols : n - lo_col);
  const int64_t first = (int64_t)row_ptr[0] - base, end = (int64_t)row_ptr[m] - base;
  const int64_t piece = (end - first + parts - 1) / parts;
  const int64_t p0 = first + part * piece;
  const int64_t p1 = p0 + piece < end ? p0 + piece : end;
  if (part > 0 && wave == 0) {
    const int r = row_of_entry(m, row_ptr, base, p0);
    if (tid == 0) *s_first = r;
  }
  for (int i = tid; i < cols; i += kSliceThreads) s_sum[i] = S(0);
  __syncthreads();
  int64_t r0 = part > 0 ? *s_first : 0;  // a row that starts at or before the chunk; none later does

  Int4* mine = reinterpret_cast<Int4*>(s_row + tid * kSlicePer);
  for (int64_t k0 = p0; k0 < p1; k0 += kSliceChunk) {
    const int len = (int)(p1 - k0 < kSliceChunk ? p1 - k0 : kSliceChunk);
    // every load unconditional: threads past the end read the chunk's first entry again
    int c[kSlicePer];
#pragma unroll
    for (int s = 0; s < kSlicePer; ++s) c[s] = col_ind[k0 + (tid + s * kSliceThreads < len ? tid + s * kSliceThreads : 0)];
#pragma unroll
    for (int q = 0; q < kSlicePer / 4; ++q) mine[q] = Int4{0, 0, 0, 0};
    __syncthreads();
    int64_t i = 1 + tid;
    const auto walk = [&](int64_t most) __attribute__((always_inline)) {
      for (; i <= most && r0 + i < m; i += kSliceThreads) {  // ascending offsets: past the chunk, all later ones are too
        const int64_t pos = (int64_t)row_ptr[r0 + i] - base - k0;
        if (pos >= len) break;
        atomicMax(&s_row[pos > 0 ? pos : 0], (int)i);
      }
    };
    walk(GAPS ? kSliceWalk : m);
    if (GAPS && tid == kSliceThreads - 1) *s_more = i > kSliceWalk;  // the thread that walks row r0 + kSliceWalk
    __syncthreads();
    int last = 0, most = 0;
    if (GAPS && *s_more) {
      // the row of the chunk's last entry (at least row r0 + kSliceWalk, where row_ptr ascends)
      const int64_t to = row_of_entry(m, row_ptr, base, k0 + len - 1) - r0;
      most = to > 1 ? (int)to : 1;
      if (most <= kSliceLook) {
        walk(m);
        __syncthreads();
      }
    }
    if (GAPS && most > kSliceLook) {
      auto starts_by = [&](int r, int k) __attribute__((always_inline)) {  // row r0 + r starts at or before entry k0 + k
        return (int64_t)row_ptr[r0 + r] - base - k0 <= k;
      };
      const int k1 = tid * kSlicePer;
      int lo = 0;  // the row of the thread's first entry
      for (int step = 1 << (31 - __builtin_clz(most)); step > 0; step >>= 1) {
        const int r = most - lo >= step ? lo + step : 0;
        if (r > 0 && starts_by(r, k1 < len ? k1 : len - 1)) lo = r;
      }
      s_row[k1] = lo;
      __syncthreads();
      const int hi = tid + 1 < kSliceThreads ? s_row[k1 + kSlicePer] : most;  // the others' lie up to the next thread's
      int at[kSlicePer];
#pragma unroll
      for (int q = 0; q < kSlicePer; ++q) at[q] = lo;
      for (int step = hi > lo ? 1 << (31 - __builtin_clz(hi - lo)) : 0; step > 0; step >>= 1) {
#pragma unroll
        for (int q = 1; q < kSlicePer; ++q) {
          const int r = hi - at[q] >= step ? at[q] + step : lo;
          if (r > at[q] && starts_by(r, k1 + q < len ? k1 + q : len - 1)) at[q] = r;
        }
      }
#pragma unroll
      for (int q = 0; q < kSlicePer / 4; ++q) mine[q] = Int4{at[4 * q], at[4 * q + 1], at[4 * q + 2], at[4 * q + 3]};
      __syncthreads();
      last = s_row[len - 1];
    } else {
      int mk[kSlicePer];
#pragma unroll
      for (int q = 0; q < kSlicePer / 4; ++q) {
        const Int4 w = mine[q];
        mk[4 * q] = w.x, mk[4 * q + 1] = w.y, mk[4 * q + 2] = w.z, mk[4 * q + 3] = w.w;
      }
#pragma unroll
      for (int q = 1; q < kSlicePer; ++q) mk[q] = max(mk[q], mk[q - 1]);
      const int incl = wave_max_scan(mk[kSlicePer - 1]);
      int lead = __builtin_amdgcn_update_dpp(0, incl, 0x138, 0xF, 0xF, true);  // wave_shr:1, lane 0 gets 0
      if (tid % kWave == kWave - 1) s_part[wave] = incl;
      __syncthreads();
#pragma unroll
      for (int w = 0; w < kSliceWaves; ++w) {
        const int pw = s_part[w];
        if (w < wave) lead = max(lead, pw);
        last = max(last, pw);
      }
#pragma unroll
      for (int q = 0; q < kSlicePer / 4; ++q)
        mine[q] = Int4{max(lead, mk[4 * q]), max(lead, mk[4 * q + 1]), max(lead, mk[4 * q + 2]), max(lead, mk[4 * q + 3])};
      __syncthreads();
    }
    T v[kSlicePer], t[kSlicePer];
    bool in[kSlicePer];
#pragma unroll
    for (int s = 0; s < kSlicePer; ++s) {
      const int k = tid + s * kSliceThreads;
      const int64_t at = (int64_t)c[s] - base - lo_col;
      in[s] = k < len && at >= 0 && at < cols;
      c[s] = in[s] ? (int)at : 0;
      v[s] = val[k0 + (in[s] ? k : 0)];
      t[s] = x[r0 + (in[s] ? s_row[k] : 0)];
    }
#pragma unroll
    for (int s = 0; s < kSlicePer; ++s)
      if (in[s]) atomic_add(&s_sum[c[s]], widened((CONJ ? conj_t(v[s]) : v[s]) * (alpha * t[s])));
    r0 += last;
    __syncthreads();  // s_row and s_part are free again
  }
  __syncthreads();
  if (partials) {
    T* __restrict__ out = partials + (int64_t)part * n + lo_col;
    for (int i = tid; i < cols; i += kSliceThreads) out[i] = narrowed<T>(s_sum[i]);
  } else {
    T* __restrict__ out = y + lo_col;
    for (int i = tid; i < cols; i += kSliceThreads) {
      const T sum = narrowed<T>(s_sum[i]);
      out[i] = beta == T(0) ? sum : out[i] * beta + sum;
    }
  }
}

// y = beta * y + (the parts' sums, added in the order of the parts): 32 columns per workgroup, eight lanes per column
// with a run of parts each
constexpr int kPartialCols = 32;
constexpr int kPartialLanes = 256 / kPartialCols;
template <typename T>
__global__ __launch_bounds__(256) void trans_partials_sum_kernel(int n, int parts, const T* __restrict__ partials, T beta,
                                                                 T* __restrict__ y) {
  __shared__ T s_sum[256];
  const int lane = threadIdx.x / kPartialCols;
  const int64_t i = (int64_t)blockIdx.x * kPartialCols + threadIdx.x % kPartialCols;
  const int run = (parts + kPartialLanes - 1) / kPartialLanes;
  const int g0 = lane * run, g1 = g0 + run < parts ? g0 + run : parts;
  T sum = T(0);
  if (i < n) {
#pragma unroll 4
    for (int g = g0; g < g1; ++g) sum += partials[(int64_t)g * n + i];
  }
  s_sum[threadIdx.x] = sum;
  __syncthreads();
  if (threadIdx.x >= kPartialCols || i >= n) return;
#pragma unroll
  for (int l = 1; l < kPartialLanes; ++l) sum += s_sum[l * kPartialCols + threadIdx.x];
  y[i] = beta == T(0) ? sum : y[i] * beta + sum;
}

}  // namespace asamd
