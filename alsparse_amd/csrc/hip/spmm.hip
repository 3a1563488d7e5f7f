// CSR SpMM  C = alpha*A*B + beta*C  for gfx950 (wave64).
//
//   spmm_group_kernel (spmm_group.hpp)   contiguous rows of B (row-major B, or column-major with op(B) = B^T):
//       sixteen lanes per row of A, C in either layout.  Row-major is the layout the reference cannot run on the
//       GPU at all (dcu_gemm_?_csr_row returns NOT_SUPPORTED,
//       src/kernel/dcu/level3/mm/csrmm/dcu_gemm_x_csr_row.cpp:15-36).
//   spmm_short_kernel<T, N, K, W>   the same with short rows of B: a lane multiplies an entry with the whole row.
//   dense_panel_kernel<T>   column-major B (with column-major C the layout the reference's GPU path does run) is laid out
//       in row-major panels in the workspace first.  Gathering column-major B directly costs one 128-byte line per
//       ELEMENT instead of per row (44 ms against 1.3 ms on a 2^20 x 2^20 matrix with 32 entries per row and 64 columns).
//   spmm_strided_kernel<T>      any strides: one lane per (row, dense column),
//       lanes of a wave on consecutive rows, so column-major C is written
//       coalesced and B(:, c) is gathered like an SpMV x.  Stands in for
//       csr_gemm_plain_device (dcu_gemm_csr_col_plain.h:9-39).
//
// Arithmetic follows the row-major plain kernel
// (src/plain/kernel/level3/mm/gemm/gemm_x_csr_row_plain.c:11-19): alpha is
// folded into each value, products are accumulated with fma, then
// C = beta*C + acc.  beta == 0 never reads C.  The strided kernel adds a row's
// products in entry order.  The others deal them out by position -- the short
// kernel to W lanes or, long rows, to the workgroup; the group kernel to 16 / GC
// parts of a lane group (one for chunks of more than 128 bytes) or, long rows, to
// sixteen groups -- and join the partial sums in a fixed order, so the same call
// returns the same bits.

#include <hip/hip_runtime.h>

#include "alsparse_amd_kernels.h"
#include "device_utils.hpp"
#include "spmm_group.hpp"

using namespace asamd;

constexpr int kSpmmBlock = 256;
constexpr int kSpmmWaves = kSpmmBlock / kWave;

// N consecutive elements that are only known to be aligned like a single one: the compiler still fetches them with one
// wide load (global memory takes unaligned wide accesses).
template <typename T, int N>
struct __attribute__((packed, aligned(alignof(T)))) Packed {
  T e[N];
};

// Narrow dense operands (rows of B of at most 64 bytes): W lanes share a row of A and read its entries coalesced, every
// lane multiplies its entries with the whole short row of B -- K loads of N elements, the last of them moved back so that
// it ends with the n-th column -- and the group's sums meet through DPP.
// A row of more than 64 W entries is taken by the whole workgroup (spmm_group.hpp says why): 2 M power-law rows, longest
// 48 946, fp32, n = 5: 1.44 ms with a lane group per row whatever its length, 0.40 ms.
template <typename T, int N, int K>
__device__ __forceinline__ void short_add(T a, const Packed<T, N> (&b)[K], T (&acc)[K * N]) {
#pragma unroll
  for (int k = 0; k < K; ++k) {
#pragma unroll
    for (int i = 0; i < N; ++i) acc[k * N + i] = fma_t(a, b[k].e[i], acc[k * N + i]);
  }
}

template <typename T, int N, int K, int W>
__global__ __launch_bounds__(kSpmmBlock) void spmm_short_kernel(int m, int n, T alpha, const T* __restrict__ val,
                                                               const int* __restrict__ row_ptr,
                                                               const int* __restrict__ col_ind, int base,
                                                               const T* __restrict__ B, int64_t ldb, T beta,
                                                               T* __restrict__ C, int64_t c_row, int64_t c_col) {
  constexpr int kRows = kSpmmBlock / W;
  constexpr int kAcc = K * N;
  constexpr int kU = sizeof(T) * kAcc <= 16 ? 4 : 2;  // entries in flight per lane
  __shared__ T s_part[kSpmmWaves * kAcc];
  __shared__ int s_any[kSpmmWaves];
  const int64_t row0 = (int64_t)xcd_contiguous_id(blockIdx.x, gridDim.x) * kRows;
  const int last = n - N;  // where the last load begins
  // sums the entries first, first + step, ... of [first, end)
  auto load = [&](Packed<T, N>(&b)[K], int col) {
    const T* p = B + (int64_t)col * ldb;
#pragma unroll
    for (int k = 0; k < K; ++k) b[k] = *reinterpret_cast<const Packed<T, N>*>(p + (k + 1 < K ? k * N : last));
  };
  auto walk = [&](int64_t first, int64_t end, int step, T(&acc)[kAcc]) {
    int64_t j = first;
    for (; j + (kU - 1) * (int64_t)step < end; j += kU * (int64_t)step) {
      T a[kU];
      int c[kU];
      Packed<T, N> b[kU][K];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        a[u] = alpha * val[j + u * (int64_t)step];
        c[u] = col_ind[j + u * (int64_t)step] - base;
      }
#pragma unroll
      for (int u = 0; u < kU; ++u) load(b[u], c[u]);
#pragma unroll
      for (int u = 0; u < kU; ++u) short_add<T, N, K>(a[u], b[u], acc);
    }
    for (; j < end; j += step) {
      Packed<T, N> b[K];
      load(b, col_ind[j] - base);
      short_add<T, N, K>(alpha * val[j], b, acc);
    }
  };
  auto put = [&](int64_t row, const T(&acc)[kAcc]) {
    T* c = C + row * c_row;
#pragma unroll
    for (int i = 0; i < kAcc; ++i) {
      // the last load's first columns, where they are also the load before's, are stored once
      const int at = i < (K - 1) * N ? i : last + (i - (K - 1) * N);
      if (i >= (K - 1) * N && at < (K - 1) * N) continue;
      T* o = c + at * c_col;
      *o = beta == T(0) ? acc[i] : *o * beta + acc[i];
    }
  };
  const int lane = threadIdx.x % W;
  const int64_t row = row0 + threadIdx.x / W;
  bool is_long = false;
  if (row < m) {
    const int64_t start = (int64_t)row_ptr[row] - base, end = (int64_t)row_ptr[row + 1] - base;
    is_long = end - start > 64 * W;
    if (!is_long) {
      T acc[kAcc];
#pragma unroll
      for (int i = 0; i < kAcc; ++i) acc[i] = T(0);
      walk(start + lane, end, W, acc);
#pragma unroll
      for (int i = 0; i < kAcc; ++i) acc[i] = group_sum<W>(acc[i]);
      if (lane == 0) put(row, acc);
    }
  }
  // (no __syncthreads_or: the library's takes 8 KB of LDS and two more barriers)
  const uint64_t wave_long = __builtin_amdgcn_ballot_w64(is_long);
  if (threadIdx.x % kWave == 0) s_any[threadIdx.x / kWave] = wave_long != 0;
  __syncthreads();
  int any = 0;
#pragma unroll
  for (int w = 0; w < kSpmmWaves; ++w) any |= s_any[w];
  if (!any) return;
  for (int64_t r = row0; r < row0 + kRows && r < m; ++r) {
    const int64_t start = (int64_t)row_ptr[r] - base, end = (int64_t)row_ptr[r + 1] - base;
    if (end - start <= 64 * W) continue;
    T acc[kAcc];
#pragma unroll
    for (int i = 0; i < kAcc; ++i) acc[i] = T(0);
    walk(start + threadIdx.x, end, kSpmmBlock, acc);
#pragma unroll
    for (int i = 0; i < kAcc; ++i) acc[i] = group_sum<kWave>(acc[i]);
    if (threadIdx.x % kWave == 0) {
#pragma unroll
      for (int i = 0; i < kAcc; ++i) s_part[threadIdx.x / kWave * kAcc + i] = acc[i];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < kSpmmWaves; ++w) {
#pragma unroll
        for (int i = 0; i < kAcc; ++i) acc[i] += s_part[w * kAcc + i];
      }
      put(r, acc);
    }
    __syncthreads();
  }
}

// The caller's column-major B (element (r, c) at r + c * ld) as row-major panels: panel element (r, c) at r * stride + c,
// w <= 64 columns.  A workgroup moves `tile` rows (16 to 32 KB) through LDS, reading along the rows and writing the panel's
// rows, which are one contiguous stretch, end to end.
template <typename T>
__global__ __launch_bounds__(kSpmmBlock) void dense_panel_kernel(int rows, int w_all, int w_panel, const T* __restrict__ in,
                                                                int64_t in_ld, T* __restrict__ out, int stride_log2,
                                                                int64_t panel_elems, int tile_rows) {
  extern __shared__ __align__(16) unsigned char smem[];
  T* tile = reinterpret_cast<T*>(smem);
  const int64_t r0 = (int64_t)blockIdx.x * tile_rows;
  const int c0 = blockIdx.y * w_panel;
  const int w = w_all - c0 < w_panel ? w_all - c0 : w_panel;
  const int nr = rows - r0 < tile_rows ? (int)(rows - r0) : tile_rows;
  const int lane = threadIdx.x % kWave;
  for (int c = threadIdx.x / kWave; c < w; c += kSpmmWaves) {
#pragma unroll 4
    for (int r = lane; r < nr; r += kWave) tile[c * (tile_rows + 1) + r] = nt_load(in + r0 + r + (int64_t)(c0 + c) * in_ld);
  }
  __syncthreads();
  T* o = out + (int64_t)blockIdx.y * panel_elems + (r0 << stride_log2);
  const int all = nr << stride_log2;
#pragma unroll 4
  for (int i = threadIdx.x; i < all; i += kSpmmBlock) {
    const int r = i >> stride_log2, c = i & ((1 << stride_log2) - 1);
    if (c < w) o[i] = tile[c * (tile_rows + 1) + r];
  }
}

// One lane per (row, dense column); blockDim = (64 rows, 4 columns).
template <typename T>
__global__ __launch_bounds__(kSpmmBlock) void spmm_strided_kernel(
    int m, int n, T alpha, const T* __restrict__ val, const int* __restrict__ row_ptr,
    const int* __restrict__ col_ind, int base, const T* __restrict__ B, int64_t sbr, int64_t sbc,
    T beta, T* __restrict__ C, int64_t scr, int64_t scc) {
  const int64_t row = (int64_t)blockIdx.x * kWave + threadIdx.x;
  if (row >= m) return;
  const int64_t start = (int64_t)row_ptr[row] - base;
  const int64_t end = (int64_t)row_ptr[row + 1] - base;
  for (int64_t c = (int64_t)blockIdx.y * blockDim.y + threadIdx.y; c < n;
       c += (int64_t)gridDim.y * blockDim.y) {
    T acc = T(0);
    for (int64_t j = start; j < end; ++j) {
      const int64_t col = (int64_t)col_ind[j] - base;
      acc = fma_t(alpha * val[j], B[col * sbr + c * sbc], acc);
    }
    T* out = C + row * scr + c * scc;
    *out = beta == T(0) ? acc : *out * beta + acc;
  }
}

// column-major B (k x n) next to column-major C (m x n), more than one column:
// B is laid out in row-major panels in the workspace first
static bool colmajor_nn(const asamd_dense_strides* st, int n) {
  return n > 1 && st->b_row_stride == 1 && st->b_col_stride != 1 && st->c_row_stride == 1;
}

// ---- the panels of a column-major B ---------------------------------------------------------------
// What a gathered row of B costs is the 128-byte lines it lies in (they come through the L2-miss path whole), so a
// panel's rows start on line boundaries: as many panels of 256 bytes as fit, and of what is left a panel of 128 bytes and
// a small one of the next power of two, up to 64 -- 17 columns of fp64 are one line and 8 bytes that stay in the L2s,
// where rows of 136 bytes end to end take 2.06 lines each (262 147^2 x 16, n = 17: 0.30 -> 0.13 ms with all of this
// file's column-major path) -- or one of 256 where more than 192 are left.  tight: what is left in panels of its powers of
// two instead, as many elements as B has (17 columns of fp32 are 16 and 1, not rows of 32): for a workspace that has no room
// for more, at one more pass over A per panel.
struct Panel {
  int cols, stride;   // columns, elements from row to row
  int64_t at;         // element offset of the first such panel in the workspace
  int count;          // so many of them, one after the other
  int64_t elems;      // elements from panel to panel
};
struct PanelPlan {
  Panel p[1 + 6];
  int kinds;
  int64_t total;  // elements
};
static PanelPlan plan_panels(int val_size, int n, int64_t k, bool tight) {
  PanelPlan plan{};
  const int full = kGroupBytes / val_size, line = full / 2;
  auto add = [&](int cols, int stride, int count) {
    Panel& p = plan.p[plan.kinds++];
    p.cols = cols;
    p.stride = stride;
    p.count = count;
    p.at = plan.total;
    // (one more 128-bit load's worth behind every panel, and whole lines)
    p.elems = (k * stride + 16 / val_size + full - 1) / full * full;
    plan.total += p.elems * count;
  };
  if (n / full > 0) add(full, full, n / full);
  int rest = n % full;
  for (int cols = line; tight && cols > 0; cols /= 2) {
    if (rest & cols) add(cols, cols, 1);
  }
  if (tight) return plan;
  if (rest > line && (rest - line) * val_size <= 64) {
    add(line, line, 1);
    rest -= line;
  }
  if (rest > 0) {
    int stride = 1;
    while (stride < rest) stride *= 2;
    add(rest, stride, 1);
  }
  return plan;
}

static size_t workspace_bytes(size_t val_size, int n, int k, const asamd_dense_strides* st, bool tight) {
  if (!st || n <= 0 || k <= 0 || !colmajor_nn(st, n)) return 0;
  return (size_t)plan_panels((int)val_size, n, k, tight).total * val_size;
}

// ---- launching -------------------------------------------------------------------------------------
template <typename T>
struct SpmmCall {
  hipStream_t s;
  int m, k;
  int64_t nnz;
  T alpha;
  const T* val;
  const int *rp, *ci;
  int base;
  T beta;
  int64_t c_row, c_col;
};

template <typename T, int N, int K>
static void launch_short(const SpmmCall<T>& a, int n, const T* B, int64_t ldb, T* C) {
  const double mean = (double)a.nnz / (double)a.m;
#define ASAMD_SHORT(W)                                                                                       \
  spmm_short_kernel<T, N, K, W><<<(unsigned)(((int64_t)a.m * W + kSpmmBlock - 1) / kSpmmBlock), kSpmmBlock, 0, a.s>>>( \
      a.m, n, a.alpha, a.val, a.rp, a.ci, a.base, B, ldb, a.beta, C, a.c_row, a.c_col)
  if (mean < 8) ASAMD_SHORT(4);
  else if (mean < 48) ASAMD_SHORT(16);
  else ASAMD_SHORT(64);
#undef ASAMD_SHORT
}

// Which rows of B a lane takes whole: up to 32 bytes, and up to 64 where the rows of A hold a few entries.  Against the
// sixteen-lane groups, us: 5-point Laplacian of 793 260 rows, fp64, n = 5 / 8: 40 / 62 against 89 / 92 (sixteen lanes share
// five entries there); 27-point stencil of 402 402 rows, n = 5 / 8: 70 / 91 against 68 / 68; 60 random columns per row: 69 / 78
// against 51 / 64.
template <typename T>
static bool short_rows(const SpmmCall<T>& a, int n) {
  return n <= 2 * kGroupV<T> || (n <= 4 * kGroupV<T> && a.nnz < 8 * (int64_t)a.m);
}

// rows of B of at most 64 bytes
template <typename T>
static void spmm_short(const SpmmCall<T>& a, int n, const T* B, int64_t ldb, T* C) {
  constexpr int V = kGroupV<T>;
  if (n > 3 * V) return launch_short<T, V, 4>(a, n, B, ldb, C);
  if (n > 2 * V) return launch_short<T, V, 3>(a, n, B, ldb, C);
  if (n > V) return launch_short<T, V, 2>(a, n, B, ldb, C);
  if (n == V) return launch_short<T, V, 1>(a, n, B, ldb, C);
  if constexpr (V == 4) {
    if (n == 3) return launch_short<T, 3, 1>(a, n, B, ldb, C);
    if (n == 2) return launch_short<T, 2, 1>(a, n, B, ldb, C);
  }
  launch_short<T, 1, 1>(a, n, B, ldb, C);
}

// `chunks` chunks of `chunk` columns (the last one ends with column n), chunk_elems elements apart in B; span: the bytes
// that may be read from B on, 0 where they are not known or 2 GiB and more
template <typename T, int GC, bool COLC, int L>
static void launch_group(const SpmmCall<T>& a, int n, int chunk, int chunks, const T* B, int64_t ldb, int64_t chunk_elems,
                         uint64_t span, bool padded, T* C) {
  constexpr int full = COLC ? kWave : kGroupRows;
  const GroupTile tile = group_tile(a.m, chunks, full);
  const dim3 grid((unsigned)(((int64_t)a.m + tile.rows - 1) / tile.rows), (unsigned)chunks);
  // Beyond the memory-side cache together: C, which is touched once, should not push B out of it, and B's rows mostly
  // come from memory (FAR, where rows of sixteen entries and more fill the groups' blocks).
  const bool big = ((double)a.k + (double)a.m) * (double)n * (double)sizeof(T) > 256.0e6;
#define ASAMD_GROUP(NARROW, FAR)                                                                               \
  spmm_group_kernel<T, GC, NARROW, COLC, L, FAR><<<grid, kGroupThreads, 0, a.s>>>(                             \
      a.m, n, a.alpha, a.val, a.rp, a.ci, a.base, B, ldb, chunk_elems * (int64_t)sizeof(T), (unsigned)span, padded, \
      a.beta, C, a.c_row, a.c_col, chunk, tile, big)
  if constexpr (GC == 16) {
    if (span > 0 && tile.rows == full && (big || L == 2) && a.nnz >= 16 * (int64_t)a.m) {
      ASAMD_GROUP(true, true);
      return;
    }
  }
  if (span > 0) ASAMD_GROUP(true, false);
  else ASAMD_GROUP(false, false);
#undef ASAMD_GROUP
}

template <typename T>
static void spmm_group(const SpmmCall<T>& a, int n, int chunk, int chunks, const T* B, int64_t ldb, int64_t chunk_elems,
                       uint64_t span, bool padded, T* C) {
  constexpr int V = kGroupV<T>;
  if (span >= (1ull << 31)) span = 0;
  if (a.c_row == 1 && a.c_col != 1) {
    if (chunk <= 4 * V) launch_group<T, 4, true, 1>(a, n, chunk, chunks, B, ldb, chunk_elems, span, padded, C);
    else if (chunk <= 8 * V) launch_group<T, 8, true, 1>(a, n, chunk, chunks, B, ldb, chunk_elems, span, padded, C);
    else launch_group<T, 16, true, 1>(a, n, chunk, chunks, B, ldb, chunk_elems, span, padded, C);
  } else {
    if (chunk <= 4 * V) launch_group<T, 4, false, 1>(a, n, chunk, chunks, B, ldb, chunk_elems, span, padded, C);
    else if (chunk <= 8 * V) launch_group<T, 8, false, 1>(a, n, chunk, chunks, B, ldb, chunk_elems, span, padded, C);
    else if (chunk <= 16 * V) launch_group<T, 16, false, 1>(a, n, chunk, chunks, B, ldb, chunk_elems, span, padded, C);
    else launch_group<T, 16, false, 2>(a, n, chunk, chunks, B, ldb, chunk_elems, span, padded, C);
  }
}

// rows of B of n contiguous elements, ldb apart: the caller's own
template <typename T>
static void spmm_rows(const SpmmCall<T>& a, int n, int k, const T* B, int64_t ldb, T* C) {
  constexpr int V = kGroupV<T>;
  if (short_rows<T>(a, n)) {
    spmm_short<T>(a, n, B, ldb, C);
    return;
  }
  // Where rows of B are whole cache lines the chunks are, too, of up to 256 bytes: one slice of B is live at a time and no
  // line is fetched for two chunks (300 000 rows of 20 random entries, us, chunks as even as whole loads allow / of whole
  // lines: fp32, n = 96 425 / 324, n = 224 1045 / 724; fp64, n = 48 432 / 330; complex128, n = 40 772 / 559).  Where they
  // are not, every chunk begins and ends inside a line: equal widths (79 columns of fp32 are 40 and 39, not 64 and 15), and
  // 512 bytes, which fetch fewer lines twice (438 520 rows of 21 random entries, fp64, n = 63: 0.80 -> 0.68 ms).
  const bool whole_lines = (ldb * (int64_t)sizeof(T)) % 128 == 0 && (uintptr_t)B % 128 == 0;
  const bool colc = a.c_row == 1 && a.c_col != 1;
  const int full = (whole_lines || colc ? 1 : 2) * kGroupBytes / (int)sizeof(T);
  const GroupChunks g = group_chunks(n, full, whole_lines ? 128 / (int)sizeof(T) : V);
  const unsigned __int128 span = (unsigned __int128)(k > 0 ? k - 1 : 0) * (unsigned __int128)ldb * sizeof(T) + (uint64_t)n * sizeof(T);
  spmm_group<T>(a, n, g.chunk, g.count, B, ldb, g.chunk,
                k > 0 && span < ((unsigned __int128)1 << 31) ? (uint64_t)span : 0, false, C);
}

template <typename T>
static int csrmm_impl(hipStream_t s, int m, int n, int k, int nnz, T alpha, const T* val,
                      const int* rp, const int* ci, int base, const T* B, T beta, T* C,
                      const asamd_dense_strides* st, void* ws, size_t ws_bytes) {
  if (!val || !rp || !ci || !B || !C || !st || m <= 0 || n <= 0) return hipErrorInvalidValue;
  if (((uintptr_t)val | (uintptr_t)B | (uintptr_t)C) % alignof(T)) return hipErrorInvalidValue;
  const SpmmCall<T> a{s, m, k, nnz, alpha, val, rp, ci, base, beta, st->c_row_stride, st->c_col_stride};
  // The row kernels load entry 0 for a lane without one: a matrix without entries is the strided kernel's, which then reads
  // row_ptr only.
  const bool entries = nnz > 0;
  if (entries && (n == 1 || st->b_col_stride == 1)) {
    // rows of op(B) are contiguous; C in either layout (a single dense column has unit stride whatever the layout says)
    if (n == 1 || st->c_col_stride == 1 || st->c_row_stride == 1) {
      spmm_rows<T>(a, n, k, B, st->b_row_stride, C);
      return hipGetLastError();
    }
  } else if (entries && colmajor_nn(st, n) && ws && k > 0 && (uintptr_t)ws % 16 == 0 &&
             (ws_bytes >= workspace_bytes(sizeof(T), n, k, st, false) || ws_bytes >= workspace_bytes(sizeof(T), n, k, st, true))) {
    const PanelPlan plan = plan_panels((int)sizeof(T), n, k, ws_bytes < workspace_bytes(sizeof(T), n, k, st, false));
    int c0 = 0;
    for (int i = 0; i < plan.kinds; ++i) {
      const Panel& p = plan.p[i];
      const int cols = p.cols * p.count;
      T* bt = (T*)ws + p.at;
      int stride_log2 = 0;
      while ((1 << stride_log2) < p.stride) ++stride_log2;
      int tile = kWave;
      while (tile * 2 * p.cols * (int)sizeof(T) <= 16384 && tile < 512) tile *= 2;
      const dim3 grid((unsigned)(((int64_t)k + tile - 1) / tile), (unsigned)p.count);
      dense_panel_kernel<T><<<grid, kSpmmBlock, (size_t)(tile + 1) * p.cols * sizeof(T), s>>>(
          k, cols, p.cols, B + (int64_t)c0 * st->b_col_stride, st->b_col_stride, bt, stride_log2, p.elems, tile);
      c0 += cols;
    }
    c0 = 0;
    for (int i = 0; i < plan.kinds; ++i) {
      const Panel& p = plan.p[i];
      const int cols = p.cols * p.count;
      const T* bt = (const T*)ws + p.at;
      T* c = C + (int64_t)c0 * st->c_col_stride;
      if (short_rows<T>(a, cols)) spmm_short<T>(a, cols, bt, p.stride, c);
      else spmm_group<T>(a, cols, p.cols, p.count, bt, p.stride, p.elems, (uint64_t)p.elems * p.count * sizeof(T), true, c);
      c0 += cols;
    }
    return hipGetLastError();
  }
  const dim3 block(kWave, kSpmmBlock / kWave);
  unsigned gy = (unsigned)((n + block.y - 1) / block.y);
  if (gy > 65535u) gy = 65535u;
  const dim3 grid((unsigned)(((int64_t)m + kWave - 1) / kWave), gy);
  spmm_strided_kernel<T><<<grid, block, 0, s>>>(m, n, alpha, val, rp, ci, base, B, st->b_row_stride, st->b_col_stride,
                                                beta, C, st->c_row_stride, st->c_col_stride);
  return hipGetLastError();
}

extern "C" int asamd_s_csrmm(hipStream_t stream, int32_t m, int32_t n, int32_t k, int32_t nnz,
                             float alpha, const float* val, const int32_t* row_ptr,
                             const int32_t* col_ind, int32_t base, const float* B, float beta,
                             float* C, const asamd_dense_strides* strides) {
  return csrmm_impl<float>(stream, m, n, k, nnz, alpha, val, row_ptr, col_ind, base, B, beta, C,
                           strides, nullptr, 0);
}

extern "C" size_t asamd_csrmm_workspace_bytes(int32_t val_size, int32_t m, int32_t n, int32_t k,
                                              const asamd_dense_strides* strides) {
  (void)m;
  return (val_size == 4 || val_size == 8 || val_size == 16) ? workspace_bytes((size_t)val_size, n, k, strides, false) : 0;
}

extern "C" size_t asamd_csrmm_least_workspace_bytes(int32_t val_size, int32_t n, int32_t k, const asamd_dense_strides* strides) {
  return (val_size == 4 || val_size == 8 || val_size == 16) ? workspace_bytes((size_t)val_size, n, k, strides, true) : 0;
}

extern "C" int asamd_s_csrmm_ws(hipStream_t stream, int32_t m, int32_t n, int32_t k, int32_t nnz, float alpha,
                                const float* val, const int32_t* row_ptr, const int32_t* col_ind, int32_t base,
                                const float* B, float beta, float* C, const asamd_dense_strides* strides,
                                void* workspace, size_t workspace_bytes) {
  return csrmm_impl<float>(stream, m, n, k, nnz, alpha, val, row_ptr, col_ind, base, B, beta, C, strides,
                           workspace, workspace_bytes);
}

extern "C" int asamd_d_csrmm_ws(hipStream_t stream, int32_t m, int32_t n, int32_t k, int32_t nnz, double alpha,
                                const double* val, const int32_t* row_ptr, const int32_t* col_ind, int32_t base,
                                const double* B, double beta, double* C, const asamd_dense_strides* strides,
                                void* workspace, size_t workspace_bytes) {
  return csrmm_impl<double>(stream, m, n, k, nnz, alpha, val, row_ptr, col_ind, base, B, beta, C, strides,
                            workspace, workspace_bytes);
}

extern "C" int asamd_d_csrmm(hipStream_t stream, int32_t m, int32_t n, int32_t k, int32_t nnz,
                             double alpha, const double* val, const int32_t* row_ptr,
                             const int32_t* col_ind, int32_t base, const double* B, double beta,
                             double* C, const asamd_dense_strides* strides) {
  return csrmm_impl<double>(stream, m, n, k, nnz, alpha, val, row_ptr, col_ind, base, B, beta, C,
                            strides, nullptr, 0);
}

// ---- the unanalysed, one-lane-per-element path ("plain"): entries of a row in storage order ---
template <typename T>
static int csrmm_plain_impl(hipStream_t s, int m, int n, T alpha, const T* val, const int* rp, const int* ci,
                            int base, const T* B, T beta, T* C, const asamd_dense_strides* st) {
  if (!val || !rp || !ci || !B || !C || !st || m <= 0 || n <= 0) return hipErrorInvalidValue;
  if (((uintptr_t)val | (uintptr_t)B | (uintptr_t)C) % alignof(T)) return hipErrorInvalidValue;
  const dim3 block(kWave, kSpmmBlock / kWave);
  unsigned gy = (unsigned)((n + block.y - 1) / block.y);
  if (gy > 65535u) gy = 65535u;
  const dim3 grid((unsigned)(((int64_t)m + kWave - 1) / kWave), gy);
  spmm_strided_kernel<T><<<grid, block, 0, s>>>(m, n, alpha, val, rp, ci, base, B, st->b_row_stride,
                                                st->b_col_stride, beta, C, st->c_row_stride, st->c_col_stride);
  return hipGetLastError();
}

extern "C" int asamd_s_csrmm_plain(hipStream_t stream, int32_t m, int32_t n, float alpha, const float* val,
                                   const int32_t* row_ptr, const int32_t* col_ind, int32_t base, const float* B,
                                   float beta, float* C, const asamd_dense_strides* strides) {
  return csrmm_plain_impl<float>(stream, m, n, alpha, val, row_ptr, col_ind, base, B, beta, C, strides);
}

extern "C" int asamd_d_csrmm_plain(hipStream_t stream, int32_t m, int32_t n, double alpha, const double* val,
                                   const int32_t* row_ptr, const int32_t* col_ind, int32_t base, const double* B,
                                   double beta, double* C, const asamd_dense_strides* strides) {
  return csrmm_plain_impl<double>(stream, m, n, alpha, val, row_ptr, col_ind, base, B, beta, C, strides);
}

extern "C" int asamd_c_csrmm_plain(hipStream_t stream, int32_t m, int32_t n, asamd_complex8 alpha,
                                   const asamd_complex8* val, const int32_t* row_ptr, const int32_t* col_ind,
                                   int32_t base, const asamd_complex8* B, asamd_complex8 beta, asamd_complex8* C,
                                   const asamd_dense_strides* strides) {
  using T = Cx<float>;
  return csrmm_plain_impl<T>(stream, m, n, T(alpha.real, alpha.imag), (const T*)val, row_ptr, col_ind, base,
                             (const T*)B, T(beta.real, beta.imag), (T*)C, strides);
}

extern "C" int asamd_z_csrmm_plain(hipStream_t stream, int32_t m, int32_t n, asamd_complex16 alpha,
                                   const asamd_complex16* val, const int32_t* row_ptr, const int32_t* col_ind,
                                   int32_t base, const asamd_complex16* B, asamd_complex16 beta, asamd_complex16* C,
                                   const asamd_dense_strides* strides) {
  using T = Cx<double>;
  return csrmm_plain_impl<T>(stream, m, n, T(alpha.real, alpha.imag), (const T*)val, row_ptr, col_ind, base,
                             (const T*)B, T(beta.real, beta.imag), (T*)C, strides);
}

// ---- complex element types: the same kernels over Cx<float> / Cx<double> -------------------
static_assert(sizeof(asamd_complex8) == sizeof(Cx<float>) && sizeof(asamd_complex16) == sizeof(Cx<double>),
              "complex layouts");

extern "C" int asamd_c_csrmm_ws(hipStream_t stream, int32_t m, int32_t n, int32_t k, int32_t nnz,
                                asamd_complex8 alpha, const asamd_complex8* val, const int32_t* row_ptr,
                                const int32_t* col_ind, int32_t base, const asamd_complex8* B, asamd_complex8 beta,
                                asamd_complex8* C, const asamd_dense_strides* strides, void* workspace,
                                size_t workspace_bytes) {
  using T = Cx<float>;
  return csrmm_impl<T>(stream, m, n, k, nnz, T(alpha.real, alpha.imag), (const T*)val, row_ptr, col_ind, base,
                       (const T*)B, T(beta.real, beta.imag), (T*)C, strides, workspace, workspace_bytes);
}

extern "C" int asamd_z_csrmm_ws(hipStream_t stream, int32_t m, int32_t n, int32_t k, int32_t nnz,
                                asamd_complex16 alpha, const asamd_complex16* val, const int32_t* row_ptr,
                                const int32_t* col_ind, int32_t base, const asamd_complex16* B,
                                asamd_complex16 beta, asamd_complex16* C, const asamd_dense_strides* strides,
                                void* workspace, size_t workspace_bytes) {
  using T = Cx<double>;
  return csrmm_impl<T>(stream, m, n, k, nnz, T(alpha.real, alpha.imag), (const T*)val, row_ptr, col_ind, base,
                       (const T*)B, T(beta.real, beta.imag), (T*)C, strides, workspace, workspace_bytes);
}
