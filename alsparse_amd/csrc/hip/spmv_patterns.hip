// Row patterns of a CSR matrix: the builder and the launcher of the kernel that multiplies with them (spmv_patterns.hpp).

#include <hip/hip_runtime.h>

#include <cstdlib>

#include "alsparse_amd_kernels.h"
#include "launch_utils.hpp"
#include "spmv_patterns.hpp"

using namespace asamd;

__global__ void pattern_clear_kernel(PatternScratch* tab) {
  tab->key[threadIdx.x] = 0;
  if (threadIdx.x == 0) tab->fail = 0;
}

extern "C" int asamd_patterns_build(hipStream_t s, int32_t m, int32_t nnz, int32_t base, int32_t group, int32_t max_len,
                                    const int32_t* row_ptr, const int32_t* col_ind, asamd_pattern_layout* out) {
  if (!out) return hipErrorInvalidValue;
  *out = asamd_pattern_layout{};
  if (!row_ptr || !col_ind || m < 1 || nnz < 1 || max_len < 1) return hipErrorInvalidValue;
  if (group < 1 || group > kStreamMaxGroup || (group & (group - 1)) != 0) return hipErrorInvalidValue;
  if (max_len > kPatternMaxLen) return hipSuccess;
  const int rows_per_group = kStreamRows / group;
  // a workgroup's columns in LDS, as many as its rows can hold: never more than 64 KiB
  const size_t lds = (size_t)rows_per_group * (size_t)max_len * sizeof(int);
  if (lds > (size_t)64 * 1024) return hipSuccess;
  const size_t pid_bytes = ((size_t)m + 255) & ~(size_t)255;
  const size_t dist_bytes = (size_t)kPatternSlots * ((size_t)max_len + 1) * sizeof(int);  // (and the lengths)
  const unsigned grid = (unsigned)(((int64_t)m + rows_per_group - 1) / rows_per_group);
  const size_t off_bytes = ((size_t)grid + 1 + (size_t)grid * kPatternWaves + 1) * sizeof(int);
  char* block = nullptr;
  hipError_t e = hipMalloc((void**)&block, pid_bytes + dist_bytes + sizeof(PatternScratch) + off_bytes);
  if (e != hipSuccess) return e;
  unsigned char* pid = (unsigned char*)block;
  int* dist = (int*)(block + pid_bytes);
  PatternScratch* tab = (PatternScratch*)(block + pid_bytes + dist_bytes);
  int* block_off = (int*)(tab + 1);
  pattern_clear_kernel<<<1, kPatternSlots, 0, s>>>(tab);
  pattern_rows_kernel<<<grid, kStreamRows, lds, s>>>(m, base, rows_per_group, max_len, row_ptr, col_ind, tab, pid,
                                                     block_off, block_off + grid + 1);
  pattern_table_kernel<<<kPatternSlots, kWave, 0, s>>>(base, max_len, row_ptr, col_ind, tab, dist);
  pattern_verify_kernel<<<grid, kStreamRows, lds, s>>>(m, base, rows_per_group, max_len, row_ptr, col_ind, pid, dist, tab);
  int fail = 1;
  e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(&fail, &tab->fail, sizeof(int), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess || fail) {
    (void)hipFree(block);
    return e;
  }
  out->pid = pid;
  out->dist = dist;
  out->block_off = block_off;
  out->stride = max_len;
  out->group = group;
  out->device_bytes = (int64_t)(pid_bytes + dist_bytes + sizeof(PatternScratch) + off_bytes);
  return hipSuccess;
}

extern "C" void asamd_patterns_free(asamd_pattern_layout* layout) {
  if (!layout) return;
  if (layout->pid) (void)hipFree(layout->pid);  // (one allocation holds all of it)
  *layout = asamd_pattern_layout{};
}

extern "C" int asamd_spmv_patterns(hipStream_t s, const asamd_spmv_args* a, const asamd_pattern_layout* L) {
  if (!a || !L || !L->pid || !L->dist || !L->block_off) return hipErrorInvalidValue;
  static const int forced = getenv("ALSPARSE_AMD_STREAM_POLICY") ? atoi(getenv("ALSPARSE_AMD_STREAM_POLICY")) : -1;
  // us per multiply, the same arrays again and again / four sets in turn, values cached against not:
  //   5-point Laplacian 2048^2, fp64 (256 MB)      34 / 47 against 40 / 44     fp32 (138 MB)    20 / 28 against 26 / 26
  //   27-point stencil 101 x 100 x 97, fp64 (231 MB)  35 / 49 against 45 / 46
  //   5-point Laplacian 2900 x 2901, fp32 (278 MB)    40 / 57 against 48 / 56
  //   27-point stencil 110^3, fp64 (314 MB)           60 / 68 against 64 / 65
  //   5-point Laplacian 2300 x 2301, fp64 (323 MB)    51 / 58 against 49 / 59
  //   5-point Laplacian 3000 x 3001, fp64 (549 MB)    94 / 94 against 81 / 94
  //   27-point stencil 160^3, fp32 (489 MB)           105 / 105 against 99 / 101
  // What the memory-side cache holds, or nearly, is left there for the next multiply; more than that only pushes the
  // rest out of it.  (Five bytes a row, a pattern's number and four of row_ptr, which the kernel no longer reads: the lines
  // below were drawn in these bytes.)
  const double bytes = (double)a->nnz * dtype_size(a->dtype) + 5.0 * (double)a->m +
                       ((double)a->m + (double)a->n) * dtype_size(a->dtype);
  const bool ntv = forced >= 0 ? (forced & kStreamNtValues) != 0 : bytes > 280.0e6;
  const bool early = !ntv && bytes <= 150.0e6;  // (the kernel has both sides)
  const int g = L->group;
  const unsigned grid = (unsigned)(((int64_t)a->m * g + kStreamRows - 1) / kStreamRows);
  const int *lens = L->dist + kPatternSlots * L->stride, *wave_off = L->block_off + grid + 1;
  auto go = [&](auto* tag) -> int {
    using T = std::remove_pointer_t<decltype(tag)>;
    if (!args_ok<T>(a)) return hipErrorInvalidValue;
    constexpr int kCap = 64 / (int)sizeof(T);  // 16 KiB of values per workgroup
    if (((uintptr_t)a->val & 15u) != 0 || L->stride > kCap * g) return hipErrorInvalidValue;
    const T alpha = scalar_of<T>(a->alpha), beta = scalar_of<T>(a->beta);
#define ASAMD_PATTERN_LAUNCH_AS(U, G, NTV, EARLY)          \
  spmv_pattern_kernel<T, U, G, NTV, EARLY><<<grid, kStreamRows, 0, s>>>( \
      a->m, alpha, (const T*)a->val, L->pid, L->dist, L->stride, lens, wave_off, (const T*)a->x, beta, (T*)a->y)
#define ASAMD_PATTERN_LAUNCH(U, G)                             \
  do {                                                         \
    if (ntv) ASAMD_PATTERN_LAUNCH_AS(U, G, true, false);       \
    else if (early) ASAMD_PATTERN_LAUNCH_AS(U, G, false, true);\
    else ASAMD_PATTERN_LAUNCH_AS(U, G, false, false);          \
  } while (0)
    // U: as few entries per lane as the longest row needs (each is a gather in flight, useful or not)
    const int u = (L->stride + g - 1) / g;
    auto grouped = [&](auto group) {
      constexpr int G = decltype(group)::value;
      if constexpr (kCap == 16) {
        if (u <= 10) ASAMD_PATTERN_LAUNCH(10, G);
        else if (u <= 12) ASAMD_PATTERN_LAUNCH(12, G);
        else if (u <= 14) ASAMD_PATTERN_LAUNCH(14, G);
        else ASAMD_PATTERN_LAUNCH(16, G);
      } else {
        if (u <= 5) ASAMD_PATTERN_LAUNCH(5, G);
        else if (u <= 6) ASAMD_PATTERN_LAUNCH(6, G);
        else if (u <= 7) ASAMD_PATTERN_LAUNCH(7, G);
        else ASAMD_PATTERN_LAUNCH(8, G);
      }
    };
    if (g == 1) {
      if (u <= 2) ASAMD_PATTERN_LAUNCH(2, 1);
      else if (u <= 3) ASAMD_PATTERN_LAUNCH(3, 1);
      else if (u <= 4) ASAMD_PATTERN_LAUNCH(4, 1);
      else if (kCap == 16 && u > 8) grouped(std::integral_constant<int, 1>{});
      else if (u <= 5) ASAMD_PATTERN_LAUNCH(5, 1);
      else if (u <= 6) ASAMD_PATTERN_LAUNCH(6, 1);
      else if (u <= 7) ASAMD_PATTERN_LAUNCH(7, 1);
      else ASAMD_PATTERN_LAUNCH(8, 1);
    } else if (g == 2) {
      grouped(std::integral_constant<int, 2>{});
    } else if (g == 4) {
      grouped(std::integral_constant<int, 4>{});
    } else if (g == 8) {
      grouped(std::integral_constant<int, 8>{});
    } else {
      grouped(std::integral_constant<int, 16>{});
    }
#undef ASAMD_PATTERN_LAUNCH
#undef ASAMD_PATTERN_LAUNCH_AS
    return hipGetLastError();
  };
  switch (a->dtype) {
    case ASAMD_DTYPE_FLOAT: return go((float*)nullptr);
    case ASAMD_DTYPE_DOUBLE: return go((double*)nullptr);
    case ASAMD_DTYPE_FLOAT_COMPLEX: return go((Cx<float>*)nullptr);
    default: return hipErrorInvalidValue;
  }
}
