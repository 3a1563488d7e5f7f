// The tiled layout whose first phase adds up (spmv_sums.hpp): builder and launcher (gfx950, wave64).
//
// asamd_sums_build sorts the entries by (column block, row block) as asamd_tiled_build does, with column blocks of one
// width and row blocks cut to even numbers of SUMS, marks where every (row, column block) sum ends, and lists the runs
// of sums that belong to a row block.  The reference has no counterpart (its analysis builds row blocks on the host that
// no kernel reads, src/util_cpp/alphasparse_dcu_x_csrmv_analysis.cpp:58-267).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "alsparse_amd_kernels.h"
#include "launch_utils.hpp"
#include "spmv_sums.hpp"
#include "tile_chunks.hpp"
#include "tile_sort.hpp"

using namespace asamd;

// Spans of a phase-1 chunk, between these (tile_chunks.hpp).  us with chunks of at most 48 spans (96 K slots), whatever the
// matrix, / these: uniform columns, 2 M x 2 M x 16 fp32 131 / 115 (256 chunks of 64 spans; 384 of up to 48), transposed
// 1 M x 16 fp64 106 / 100 (245 of 32; 184), 2 M x 2 M x 20 fp32 135 / 129, fp64 250 / 245; power law of 8 M rows fp32 287 / 285.
// A column block's chunks on one XCD, whose L2 then has the x slice: that transposed product 99 / 96, power law of 4 M rows
// 141 / 138, 2 M x 2 M x 20 complex128 444 / 411.
constexpr int kSumsLeastSpans = 16, kSumsMostSpans = 96, kSumsSpanStep = 4;

// Tallest row block: eight waves' accumulators and dummy rows fill a compute unit's LDS
template <typename T>
constexpr int sums_rows_most() {
  return (kLdsPerCu / kRedWaves / (int)sizeof(T) - kWave) >> kRowGroupLog2 << kRowGroupLog2;
}
template <typename T>
static int sums_red_lds(int rows_cap) { return kRedWaves * (rows_cap + kWave) * (int)sizeof(T); }

// Cuts the groups into blocks of at most max_groups groups that hold at most `target` sums each (one group at least).
static int cut_groups(const std::vector<int64_t>& off, int groups, int max_groups, int64_t target, std::vector<int>* start) {
  int blocks = 0, g = 0;
  while (g < groups) {
    if (start) start->push_back(g);
    int e = g + 1;
    while (e < groups && e - g < max_groups && off[(size_t)e + 1] - off[(size_t)g] <= target) ++e;
    g = e;
    ++blocks;
  }
  if (start) start->push_back(groups);
  return blocks;
}

// counts on the device -> host, through pinned memory and a kernel (the copy engine's first copy after a pause takes
// milliseconds); waits for the stream
static hipError_t counts_to_host(hipStream_t stream, int n, const int* d, int* pinned) {
  strided_gather_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(n, d, 1, pinned);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? hipStreamSynchronize(stream) : e;
}

template <typename T>
static hipError_t build_sums(hipStream_t stream, asamd_sums_layout* L, const int m, const int n, const int nnz, const int base,
                             const int64_t most_sums, const int* row_ptr, const int* col_ind, const T* val) {
  constexpr int kCols = SumsDims<T>::cols, kShift = log2_of(kCols);
  const int cb = (int)(((int64_t)n + kCols - 1) >> kShift);
  const int groups = (int)(((int64_t)m + (1 << kRowGroupLog2) - 1) >> kRowGroupLog2);
  const auto room = [](size_t bytes) { return (bytes + 255) / 256 * 256; };
  constexpr int kSpan = SumsDims<T>::span;
  const int64_t spans_most = (int64_t)nnz / kSpan + cb + 1;
  const size_t cnt_n = (size_t)(spans_most > 2 * (int64_t)groups ? spans_most : 2 * (int64_t)groups) + 1;

  int *d_cnt = nullptr, *d_rgb = nullptr, *d_colptr = nullptr, *h_cnt = nullptr;
  char* d_arena = nullptr;
  int *d_coo = nullptr, *d_first = nullptr, *d_tile_ptr = nullptr;
  unsigned *d_key = nullptr, *d_key2 = nullptr;
  unsigned long long *d_pay = nullptr, *d_pay2 = nullptr;
  std::vector<int64_t> off;
  std::vector<int> rstart, rgb, colptr, colspan;
  int rb = 0, spans = 0;
  int64_t tiles = 0, sums = 0;
  bool suits = true;

  // ---- 1. sums per group of 64 rows -> is it worth it, and the row blocks --------------------------------
  hipError_t e = hipMalloc(&d_cnt, cnt_n * sizeof(int));
  if (e == hipSuccess) e = hipHostMalloc((void**)&h_cnt, cnt_n * sizeof(int), hipHostMallocDefault);
  if (e == hipSuccess) {
    sums_count_kernel<<<(unsigned)groups, 256, 0, stream>>>(m, row_ptr, col_ind, base, kShift, d_cnt);
    e = counts_to_host(stream, groups, d_cnt, h_cnt);
  }
  if (e == hipSuccess) {
    off.resize((size_t)groups + 1);
    off[0] = 0;
    for (int g = 0; g < groups; ++g) off[(size_t)g + 1] = off[(size_t)g] + h_cnt[g];
    suits = off[(size_t)groups] <= most_sums;
  }
  if (e == hipSuccess && suits) {
    // One row block per wave, and the chip holds a fixed number of the second phase's waves: the blocks are as even as
    // their groups allow and fill whole rounds.  Tall blocks make few and long runs.
    constexpr int kMostGroups = sums_rows_most<T>() >> kRowGroupLog2;
    const int64_t slots = (int64_t)device_cus() * kRedWaves;
    const int64_t full = ((int64_t)groups + kMostGroups - 1) / kMostGroups;
    const int64_t want = (full + slots - 1) / slots * slots;
    const int64_t all = off[(size_t)groups];
    int64_t target = all / want + 1;
    for (int i = 0; i < 12 && cut_groups(off, groups, kMostGroups, target, nullptr) > want; ++i) target += target / 64 + 1;
    rb = cut_groups(off, groups, kMostGroups, target, &rstart);
    tiles = (int64_t)cb * rb;
    if (cb > kTiledMaxColBlocks || tiles > kTiledMaxTiles) suits = false;
  }
  if (e != hipSuccess || !suits) {
    if (h_cnt) (void)hipHostFree(h_cnt);
    if (d_cnt) (void)hipFree(d_cnt);
    return e;
  }
  std::vector<int> h_rbs((size_t)rb + 1);
  rgb.resize((size_t)groups);
  L->rows_cap = 0;
  for (int r = 0; r <= rb; ++r) {
    const int64_t v = (int64_t)rstart[(size_t)r] << kRowGroupLog2;
    h_rbs[(size_t)r] = (int)(v < m ? v : m);
    if (r > 0) {
      for (int g = rstart[(size_t)r - 1]; g < rstart[(size_t)r]; ++g) rgb[(size_t)g] = r - 1;
      const int rows = (rstart[(size_t)r] - rstart[(size_t)r - 1]) << kRowGroupLog2;
      if (rows > L->rows_cap) L->rows_cap = rows;
    }
  }
  L->col_blocks = cb;
  L->row_blocks = rb;
  unsigned key_bits = 1;
  while (((int64_t)1 << key_bits) < tiles) ++key_bits;

  // ---- 2. entries in tile order -----------------------------------------------------------------------------
  const size_t N = (size_t)nnz;
  size_t slots = 0;
  e = hipMalloc(&d_rgb, (size_t)groups * sizeof(int));
  if (e == hipSuccess) e = hipMalloc(&d_colptr, 2 * ((size_t)cb + 1) * sizeof(int));
  if (e == hipSuccess) e = hipMalloc(&L->row_block_start, ((size_t)rb + 1) * sizeof(int));
  if (e == hipSuccess) e = hipMemcpy(d_rgb, rgb.data(), (size_t)groups * sizeof(int), hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(L->row_block_start, h_rbs.data(), ((size_t)rb + 1) * sizeof(int), hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMalloc(&d_arena, 3 * room(N * sizeof(int)) + 2 * room(N * sizeof(unsigned long long)));
  if (e == hipSuccess) {
    char* at = d_arena;
    const auto take = [&](size_t bytes) {
      char* p = at;
      at += room(bytes);
      return (void*)p;
    };
    d_coo = (int*)take(N * sizeof(int));
    d_key = (unsigned*)take(N * sizeof(unsigned));
    d_key2 = (unsigned*)take(N * sizeof(unsigned));
    d_pay = (unsigned long long*)take(N * sizeof(unsigned long long));
    d_pay2 = (unsigned long long*)take(N * sizeof(unsigned long long));
    d_first = d_coo;  // the rows are used up by then
  }
  if (e == hipSuccess) e = hipMalloc(&d_tile_ptr, (size_t)(tiles + 1) * sizeof(int));
  // (d_key2 is free until the sort: it serves csr2coo as its table of chunk rows)
  if (e == hipSuccess) e = (hipError_t)asamd_csr2coo_ws(stream, row_ptr, nnz, m, d_coo, base, d_key2, N * sizeof(unsigned));
  if (e == hipSuccess) {
    sums_keys_kernel<<<256 * 32, 256, 0, stream>>>(nnz, d_coo, col_ind, base, kShift, d_rgb, L->row_block_start, rb, d_key,
                                                   d_pay);
    e = sort_pairs_u32_u64(stream, d_key, d_key2, d_pay, d_pay2, N, key_bits);
  }
  if (e == hipSuccess) {
    tile_bounds_kernel<<<(unsigned)((tiles + 1 + 255) / 256), 256, 0, stream>>>(nnz, d_key2, tiles, d_tile_ptr);
    strided_gather_kernel<<<(unsigned)((cb + 1 + 255) / 256), 256, 0, stream>>>(cb + 1, d_tile_ptr, (int64_t)rb, d_cnt);
    e = counts_to_host(stream, cb + 1, d_cnt, h_cnt);
  }

  // ---- 3. spans, their sums, the rows of the sums --------------------------------------------------------------
  if (e == hipSuccess) {
    colptr.assign(h_cnt, h_cnt + cb + 1);
    colspan.resize((size_t)cb + 1);
    for (int c = 0; c < cb; ++c) {
      colspan[(size_t)c] = spans;
      const int b = colptr[(size_t)c], end = colptr[(size_t)c + 1];
      spans += (end - b + kSpan - 1) / kSpan;
    }
    colspan[(size_t)cb] = spans;
    e = hipMemcpy(d_colptr, colptr.data(), ((size_t)cb + 1) * sizeof(int), hipMemcpyHostToDevice);
    if (e == hipSuccess)
      e = hipMemcpy(d_colptr + cb + 1, colspan.data(), ((size_t)cb + 1) * sizeof(int), hipMemcpyHostToDevice);
  }
  if (e == hipSuccess) e = hipMalloc(&L->span_sum, ((size_t)spans + 1) * sizeof(int));
  if (e == hipSuccess) {
    sums_span_count_kernel<<<(unsigned)((spans + 3) / 4), 256, 0, stream>>>(spans, kSpan, cb, d_colptr + cb + 1, d_colptr,
                                                                            d_key2, d_pay2, d_cnt);
    e = counts_to_host(stream, spans, d_cnt, h_cnt);
  }
  if (e == hipSuccess) {
    for (int s = 0; s < spans; ++s) {
      const int c = h_cnt[s];
      h_cnt[s] = (int)sums;
      sums += c;
    }
    h_cnt[spans] = (int)sums;
    slots = (size_t)spans * kSpan;
    e = hipMemcpy(L->span_sum, h_cnt, ((size_t)spans + 1) * sizeof(int), hipMemcpyHostToDevice);
  }
  if (e == hipSuccess) e = hipMalloc(&L->tval, slots * sizeof(T));
  if (e == hipSuccess) e = hipMalloc(&L->tcol, slots * sizeof(short));
  if (e == hipSuccess) e = hipMalloc(&L->tperm, slots * sizeof(unsigned));
  if (e == hipSuccess) e = hipMalloc(&L->srow, ((size_t)sums + 1) * sizeof(short));
  if (e == hipSuccess) e = hipMalloc(&L->run_ptr, ((size_t)rb + 1) * sizeof(int));
  std::vector<int> h_run((size_t)rb + 1);
  if (e == hipSuccess) {
    sums_spans_kernel<T><<<(unsigned)((spans + 3) / 4), 256, 0, stream>>>(spans, cb, d_colptr + cb + 1, d_colptr, L->span_sum,
                                                                          d_key2, d_pay2, L->tcol, L->tperm, L->srow, d_first);
    sums_runs_kernel<<<(unsigned)((rb + 63) / 64), 64, 0, stream>>>(rb, cb, nnz, (int)sums, kSpan, d_colptr + cb + 1, d_colptr,
                                                                    L->span_sum, L->srow, d_tile_ptr, d_first, nullptr, d_cnt,
                                                                    nullptr);
    e = counts_to_host(stream, rb, d_cnt, h_cnt);
    for (int r = 0; r < rb; ++r) {
      h_run[(size_t)r] = L->n_runs;
      L->n_runs += h_cnt[r];
    }
    h_run[(size_t)rb] = L->n_runs;
  }
  if (e == hipSuccess) e = hipMemcpy(L->run_ptr, h_run.data(), ((size_t)rb + 1) * sizeof(int), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMalloc(&L->runs, ((size_t)L->n_runs + 1) * sizeof(TileRange));
  if (e == hipSuccess) e = hipMemsetAsync(L->runs, 0, ((size_t)L->n_runs + 1) * sizeof(TileRange), stream);
  if (e == hipSuccess) {
    sums_runs_kernel<<<(unsigned)((rb + 63) / 64), 64, 0, stream>>>(rb, cb, nnz, (int)sums, kSpan, d_colptr + cb + 1, d_colptr,
                                                                    L->span_sum, L->srow, d_tile_ptr, d_first, L->run_ptr,
                                                                    nullptr, (TileRange*)L->runs);
    e = hipGetLastError();
  }

  // ---- 4. phase-1 work list, the values ---------------------------------------------------------------------------
  std::vector<SumsChunk> h_chunks;
  if (e == hipSuccess) {
    std::vector<int> block_spans((size_t)cb);
    for (int c = 0; c < cb; ++c) block_spans[(size_t)c] = colspan[(size_t)c + 1] - colspan[(size_t)c];
    const int limit = chunk_limit(block_spans, (int64_t)kSpan * ((int64_t)sizeof(T) + 2), kSumsSliceBytes, device_cus(),
                                  kSumsLeastSpans, kSumsMostSpans, kSumsSpanStep);
    for (int c = 0; c < cb; ++c) {
      const int all = block_spans[(size_t)c], pieces = (all + limit - 1) / limit;
      const int64_t entries = colptr[(size_t)c + 1] - colptr[(size_t)c];
      for (int i = 0; i < pieces; ++i) {  // as even as whole spans allow
        const int64_t first = (int64_t)all * i / pieces, end = (int64_t)all * (i + 1) / pieces * kSpan;
        SumsChunk ch;
        ch.col0 = c << kShift;
        ch.ncols = n - ch.col0 < kCols ? n - ch.col0 : kCols;
        ch.span0 = colspan[(size_t)c] + (int)first;
        ch.slots = (int)((end < entries ? end : entries) - first * kSpan);
        h_chunks.push_back(ch);
      }
    }
    std::vector<int> size, block;
    for (const SumsChunk& ch : h_chunks) {
      size.push_back(ch.slots);
      block.push_back(ch.col0 >> kShift);
    }
    const std::vector<int> order = chunk_order(size, block, kXcds);
    std::vector<SumsChunk> ordered;
    for (int i : order) ordered.push_back(h_chunks[(size_t)i]);
    h_chunks.swap(ordered);
    L->n_chunks = (int)h_chunks.size();
    e = hipMalloc(&L->chunks, h_chunks.size() * sizeof(SumsChunk));
    if (e == hipSuccess) e = hipMemcpy(L->chunks, h_chunks.data(), h_chunks.size() * sizeof(SumsChunk), hipMemcpyHostToDevice);
  }
  L->dtype = DtypeOf<T>::value;
  L->m = m;
  L->n = n;
  L->nnz = nnz;
  L->sums = (int)sums;
  L->spans = spans;
  // the order in which the values are gathered: the spans of all column blocks side by side that hold the same rows
  if (e == hipSuccess) {
    constexpr int kSteps = 4096;
    std::vector<int> first(kSteps + 1, 0), order((size_t)spans + 1);
    for (int pass = 0; pass < 2; ++pass)
      for (int c = 0; c < cb; ++c) {
        const int b = colspan[(size_t)c], all = colspan[(size_t)c + 1] - b;
        for (int i = 0; i < all; ++i) {
          const int step = (int)((2 * (int64_t)i + 1) * kSteps / (2 * (int64_t)all));
          if (pass == 0) ++first[(size_t)step + 1];
          else order[(size_t)first[(size_t)step]++] = b + i;
        }
        if (pass == 0 && c + 1 == cb)
          for (int k = 0; k < kSteps; ++k) first[(size_t)k + 1] += first[(size_t)k];
      }
    e = hipMalloc(&L->order, ((size_t)spans + 1) * sizeof(int));
    if (e == hipSuccess) e = hipMemcpy(L->order, order.data(), ((size_t)spans + 1) * sizeof(int), hipMemcpyHostToDevice);
  }
  if (e == hipSuccess) e = (hipError_t)asamd_sums_refresh_values(stream, L, val, nullptr);
  for (const void* f : {(const void*)sums_products_kernel<T, false, false>, (const void*)sums_products_kernel<T, false, true>,
                        (const void*)sums_products_kernel<T, true, true>})
    if (e == hipSuccess) e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsPerCu);
  if (e == hipSuccess)
    e = hipFuncSetAttribute((const void*)tiled_reduce_kernel<T, 1, true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            kLdsPerCu);
  if (e == hipSuccess) e = hipStreamSynchronize(stream);
  if (h_cnt) (void)hipHostFree(h_cnt);
  free_all({d_arena, d_cnt, d_rgb, d_colptr, d_tile_ptr});
  if (e != hipSuccess) {
    asamd_sums_free(L);
    return e;
  }
  L->device_bytes = (int64_t)(slots * (sizeof(T) + 2 + 4) + ((size_t)sums + 1) * 2 + ((size_t)L->n_runs + 1) * 8 +
                              ((size_t)rb + 1) * 8 + ((size_t)spans + 1) * 8 +
                              h_chunks.size() * sizeof(SumsChunk));
  return hipSuccess;
}

extern "C" int asamd_sums_build(hipStream_t stream, int32_t dtype, int32_t m, int32_t n, int32_t nnz, int32_t base,
                                const int32_t* row_ptr, const int32_t* col_ind, const void* val, int64_t most_sums,
                                asamd_sums_layout* out) {
  if (!out) return hipErrorInvalidValue;
  *out = asamd_sums_layout{};
  if (!row_ptr || !col_ind || !val || !asamd_tiled_fits(dtype, m, n, nnz)) return hipErrorInvalidValue;
  if ((uintptr_t)val % (size_t)dtype_size(dtype)) return hipErrorInvalidValue;
  return by_dtype(dtype, [&](auto* tag) -> int {
    using T = std::remove_pointer_t<decltype(tag)>;
    return build_sums<T>(stream, out, m, n, nnz, base, most_sums, row_ptr, col_ind, (const T*)val);
  });
}

extern "C" void asamd_sums_free(asamd_sums_layout* L) {
  if (!L) return;
  free_all({L->tval, (void*)L->tperm, (void*)L->tcol, (void*)L->srow, (void*)L->row_block_start, (void*)L->run_ptr,
            (void*)L->span_sum, (void*)L->order, L->runs, L->chunks});
  *L = asamd_sums_layout{};
}

static int sums_refresh(hipStream_t s, const asamd_sums_layout* L, const void* val, const GuardGate& gate) {
  if (!L || !L->tval || !L->tperm || !val) return hipErrorInvalidValue;
  return by_dtype(L->dtype, [&](auto* tag) -> int {
    using T = std::remove_pointer_t<decltype(tag)>;
    if ((uintptr_t)val % alignof(T)) return hipErrorInvalidValue;
    // few enough workgroups to return quickly where the gate is shut, and a multiple of the XCDs
    const unsigned grid = (unsigned)(L->spans >= 256 * 8 ? 256 * 8 : (L->spans + kXcds - 1) / kXcds * kXcds);
    sums_values_kernel<T><<<grid, 256, 0, s>>>(L->spans, L->order, L->tperm, (const T*)val, (T*)L->tval, gate);
    return hipGetLastError();
  });
}
extern "C" int asamd_sums_refresh_values(hipStream_t s, const asamd_sums_layout* L, const void* val, const int32_t* gate) {
  return sums_refresh(s, L, val, guard_gate(gate));
}
extern "C" int asamd_sums_refresh_checked(hipStream_t s, const asamd_sums_layout* L, const void* val,
                                          const asamd_value_check* check) {
  return sums_refresh(s, L, val, guard_gate(check));
}

extern "C" int asamd_spmv_sums(hipStream_t s, const asamd_spmv_args* a, const asamd_sums_layout* L, void* sums) {
  return asamd_spmv_sums_form(s, a, L, sums, nullptr, -1);
}
extern "C" int asamd_spmv_sums_commit(hipStream_t s, const asamd_spmv_args* a, const asamd_sums_layout* L, void* sums,
                                      const asamd_value_check* commit) {
  return asamd_spmv_sums_form(s, a, L, sums, commit, -1);
}
extern "C" int asamd_spmv_sums_form(hipStream_t s, const asamd_spmv_args* a, const asamd_sums_layout* L, void* sums,
                                    const asamd_value_check* commit, int32_t form) {
  if (!a || !L || !L->tval || !sums || !a->alpha || !a->beta || !a->x || !a->y || form < -1 || form > 2)
    return hipErrorInvalidValue;
  if (a->dtype != L->dtype || a->m != L->m || a->n != L->n || a->nnz != L->nnz) return hipErrorInvalidValue;
  return by_dtype(a->dtype, [&](auto* tag) -> int {
    using T = std::remove_pointer_t<decltype(tag)>;
    if (((uintptr_t)a->x | (uintptr_t)a->y | (uintptr_t)sums) % alignof(T)) return hipErrorInvalidValue;
    const T alpha = scalar_of<T>(a->alpha), beta = scalar_of<T>(a->beta);
    const T* x = (const T*)a->x;
    T* y = (T*)a->y;
    T* mid = (T*)sums;
    const auto products = [&](auto kernel) {
      kernel<<<L->n_chunks, kProdThreads, kLdsPerCu, s>>>((const SumsChunk*)L->chunks, L->span_sum, (const T*)L->tval, L->tcol,
                                                          x, mid);
    };
    // Sums that the memory-side cache could not hold are stored past it, as the tiled pair's products.  Where it holds the
    // sums, but not the values and columns beside them, those are loaded past it, so that the second phase finds the sums
    // there.  us, plain / past it, three matrices in turn and one again and again (which that cache serves where it fits):
    //   power law fp32, 2.1 M rows (167 MB)  59.0 / 55.8  51.9 / 56.6     uniform x 16 fp64, 0.70 M (188 MB)  68.7 / 64.7  57.1 / 60.4
    //     2.6 M (209 MB)  73.0 / 68.8  63.8 / 70.1                          0.85 M (230 MB)   83.2 / 79.4  79.3 / 74.3
    //     3.0 M (243 MB)  83.5 / 78.2  72.6 / 77.6                          0.95 M (259 MB)   90.3 / 87.0  81.4 / 78.7
    //     3.3 M (270 MB)  89.3 / 84.9  80.6 / 81.6                        uniform x 16 fp32, 1.6 M (242 MB)  84.6 / 80.2  75.9 / 76.3
    //     3.8 M (312 MB)  102 / 99.0  100 / 97.6                            1.8 M (274 MB)    96.4 / 94.0  91.5 / 88.5
    //     4.5 M (384 MB)  123 / 118  118 / 110                              4.2 M (656 MB)    230 / 215  229 / 217
    // The line lies where one matrix again and again stops losing.
    const int64_t sum_bytes = (int64_t)L->sums * (int64_t)sizeof(T);
    const int64_t stream_bytes = (int64_t)L->spans * SumsDims<T>::span * ((int64_t)sizeof(T) + 2);
    const int by_size = sum_bytes > ((int64_t)512 << 20) ? 2 : sum_bytes + stream_bytes > (int64_t)256000000 ? 1 : 0;
    switch (form < 0 ? by_size : form) {
      case 0: products(sums_products_kernel<T, false, false>); break;
      case 1: products(sums_products_kernel<T, false, true>); break;
      default: products(sums_products_kernel<T, true, true>);
    }
    const unsigned grid = (unsigned)((L->row_blocks + kRedWaves - 1) / kRedWaves);
    tiled_reduce_kernel<T, 1, true><<<grid, kRedWaves * kWave, sums_red_lds<T>(L->rows_cap), s>>>(
        L->row_blocks, 0, L->rows_cap, L->row_block_start, L->run_ptr, (const TileRange*)L->runs, L->srow, mid, alpha, beta,
        y, nullptr, guard_commit_of(commit));
    return hipGetLastError();
  });
}
