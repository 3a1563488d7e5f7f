// The scratch of the value guard and what the kernels behind it read (gfx950, wave64).  The reference has no counterpart: its
// kernels read csr_val on every call (src/kernel/dcu/level2/mv/csrmv/dcu_gemv_vector.h:43-46).
#pragma once

#include "alsparse_amd_kernels.h"
#include "device_utils.hpp"

namespace asamd {

constexpr int kGuardBlocks = 2048;
struct GuardWs {
  unsigned long long partial[kGuardBlocks];
  unsigned long long fp;
  int flag;
};
static_assert(ASAMD_GUARD_WS_BYTES >= sizeof(GuardWs), "guard scratch holds the partial sums, the word and the flag");
static_assert(offsetof(GuardWs, flag) == 8 * kGuardBlocks + 8, "ASAMD_GUARD_FLAG points at the flag");

__host__ __device__ __forceinline__ unsigned long long guard_salt(int64_t total_words) {
  return (unsigned long long)total_words * 0x9E3779B97F4A7C15ull;
}

// sum over the 256 threads of a workgroup, valid in thread 0
__device__ __forceinline__ unsigned long long block_sum_u64(unsigned long long mine) {
  __shared__ unsigned long long s_sum[256 / kWave];
  for (int d = kWave / 2; d > 0; d >>= 1) mine += __shfl_down(mine, d, kWave);
  if (threadIdx.x % kWave == 0) s_sum[threadIdx.x / kWave] = mine;
  __syncthreads();
  unsigned long long total = 0;
  if (threadIdx.x == 0)
    for (int w = 0; w < 256 / kWave; ++w) total += s_sum[w];
  return total;
}

// the fingerprint from the partial sums, valid in thread 0; workgroups of 256
__device__ __forceinline__ unsigned long long guard_fingerprint(const GuardWs* ws, unsigned long long salt) {
  constexpr int kEach = kGuardBlocks / 256;
  unsigned long long part[kEach], mine = 0;
#pragma unroll
  for (int i = 0; i < kEach; ++i) part[i] = ws->partial[threadIdx.x + i * 256];
#pragma unroll
  for (int i = 0; i < kEach; ++i) mine += part[i];
  return block_sum_u64(mine) ^ salt;
}

// What a kernel that refreshes a copy goes by: a flag, or a check that is not settled: the pass over the values has left
// partial sums, and every workgroup adds them up itself (16 KB that all of them find in their L2) instead of waiting for a
// launch that does it once; the first one leaves word and flag for the kernels behind.
struct GuardGate {
  const int* flag;  // zero: the values have not changed
  GuardWs* ws;      // neither this nor a flag: refresh
  const unsigned long long* stored;
  unsigned long long salt;
};
// whether to refresh; all 256 threads of every workgroup come here
__device__ __forceinline__ bool guard_open(const GuardGate& g) {
  if (g.flag) return *g.flag != 0;
  if (!g.ws) return true;
  __shared__ int s_changed;
  const unsigned long long fp = guard_fingerprint(g.ws, g.salt);
  if (threadIdx.x == 0) {
    const int changed = *g.stored != fp;
    s_changed = changed;
    if (blockIdx.x == 0) {
      g.ws->fp = fp;
      g.ws->flag = changed;
    }
  }
  __syncthreads();
  return s_changed != 0;
}

// the new fingerprint is recorded once the copy holds the new values: by a kernel behind those that refresh it
struct GuardCommit {
  const GuardWs* ws;  // null: nothing to record
  unsigned long long* stored;
};
__device__ __forceinline__ void guard_commit(const GuardCommit& c) {
  if (c.ws && blockIdx.x == 0 && threadIdx.x == 0 && c.ws->flag) *c.stored = c.ws->fp;
}

inline GuardGate guard_gate(const int* flag) { return GuardGate{flag, nullptr, nullptr, 0}; }
inline GuardGate guard_gate(const asamd_value_check* c) {
  if (!c || c->settled) return guard_gate(c ? ASAMD_GUARD_FLAG(c->ws) : (const int*)nullptr);
  return GuardGate{nullptr, (GuardWs*)c->ws, (const unsigned long long*)c->stored, guard_salt(c->words)};
}
inline GuardCommit guard_commit_of(const asamd_value_check* c) {
  return c ? GuardCommit{(const GuardWs*)c->ws, (unsigned long long*)c->stored} : GuardCommit{nullptr, nullptr};
}

}  // namespace asamd
