// CSR SpMM in 16-lane groups for gfx950 (wave64): C = alpha*A*B + beta*C with contiguous rows of B.
//
// Sixteen lanes -- one DPP row -- own one row of A and up to 256 bytes of dense columns; a wave takes four rows, so one
// 128-bit load instruction fetches four rows of B.  The group reads sixteen entries of its row with one coalesced
// load; every lane turns its entry's column into the byte offset of that row of B once, and the entries go round
// the group with DPP broadcasts inside the address addition and the multiply-adds -- no LDS crossbar (whose
// ds_bpermutes alone held the kernel this one replaced at 0.31 ms on a 27-point stencil of 2^20 rows, n = 64) and no
// 64-bit address arithmetic in the entry loop.  GC lanes cover the dense columns of a chunk; where they are fewer than
// sixteen the group's 16 / GC parts take every (16 / GC)-th entry and their sums meet at the end.
//
// What bounds it: random columns, the L2-miss path (whole 128-byte lines at about 7 TB/s); columns that neighbouring
// rows share, the L1-to-register path (27-point stencil of 2^20 rows, n = 64: 20 TB/s, 0.63 accesses of 64 bytes per clock
// and compute unit).
#pragma once

#include <utility>

#include "device_utils.hpp"

namespace asamd {

constexpr int kGroupThreads = 256;
constexpr int kGroupRows = kGroupThreads / 16;  // rows of A that a workgroup has in work at one time
constexpr int kGroupBytes = 256;                // dense columns of one chunk, in bytes
// A row of more entries than this is taken by all sixteen groups of the workgroup together: one group would hold the
// workgroup up (a power-law graph of 0.7 M rows, longest row 16 727, complex64, n = 11: 3.55 ms with a lane group per
// row whatever its length).
constexpr int kGroupLongRow = 256;
constexpr unsigned kGroupNoRow = 0x80000000u;  // an offset that the buffer's range check turns away (B within 2 GiB)

template <typename T>
constexpr int kGroupV = 16 / (int)sizeof(T);  // elements of one 128-bit load

template <typename T>
struct GroupVec {
  T e[kGroupV<T>];
};
// the same in memory, where only the element's own alignment is known (wide global accesses may be unaligned)
template <typename T>
struct __attribute__((packed, aligned(alignof(T) < 8 ? alignof(T) : 8))) GroupLoose {
  unsigned w[4];
};

// value of lane J of the caller's part of GC lanes (a DPP row holds 16 / GC parts)
template <int GC, int J>
__device__ __forceinline__ int part_bcast(int v, bool upper) {
  if constexpr (GC == 16) {
    return __builtin_amdgcn_update_dpp(0, v, 0x150 + J, 0xF, 0xF, true);  // row_newbcast:J
  } else if constexpr (GC == 8) {
    const int lo = __builtin_amdgcn_update_dpp(0, v, 0x150 + J, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_update_dpp(0, v, 0x158 + J, 0xF, 0xF, true);
    return upper ? hi : lo;
  } else {
    static_assert(GC == 4, "four, eight or sixteen column lanes");
    return __builtin_amdgcn_update_dpp(0, v, J * 0x55, 0xF, 0xF, true);  // quad_perm:[J,J,J,J]
  }
}
template <int GC, int J, typename T>
__device__ __forceinline__ T part_bcast_t(T v, bool upper) {
  struct Words { int w[sizeof(T) / 4]; };
  Words a = __builtin_bit_cast(Words, v);
#pragma unroll
  for (int i = 0; i < (int)(sizeof(T) / 4); ++i) a.w[i] = part_bcast<GC, J>(a.w[i], upper);
  return __builtin_bit_cast(T, a);
}

// lanes of a wave whose position in their part of GC lanes is in [lo, hi)
template <int GC>
constexpr uint64_t part_lanes(int lo, int hi) {
  uint64_t m = 0;
  for (int l = 0; l < 64; ++l)
    if (l % GC >= lo && l % GC < hi) m |= (uint64_t)1 << l;
  return m;
}

// f(0), f(1), ... with compile-time numbers
template <typename F, int... U>
__device__ __forceinline__ void for_each_const(F& f, std::integer_sequence<int, U...>) {
  (f(std::integral_constant<int, U>{}), ...);
}

// ---- which columns a lane takes (host and device: the arithmetic is checked without a GPU) --------------------
// `count` chunks of `chunk` columns, whole units of v each (a load, or a line), as even as that allows; the last ends with
// column n and may hold fewer columns than a load (n = 961, at most 64 a chunk: fifteen of 64, then one column).
struct GroupChunks {
  int chunk, count;
};
__host__ __device__ constexpr GroupChunks group_chunks(int n, int most, int v) {
  const int even = (int)(((int64_t)n + most - 1) / most);
  const int chunk = (int)((((int64_t)n + even - 1) / even + v - 1) / v * v);
  return {chunk, (int)(((int64_t)n + chunk - 1) / chunk)};
}

// How many rows of A a workgroup takes, and from how many entries on its sixteen groups share a row.  Whole tiles (`most`
// rows) where those make two workgroups per compute unit; fewer rows where the matrix has not so many, down to one: a
// workgroup takes its long rows one after the other, and groups without a row are what shared rows are dealt to.
// us, whole tiles against this: 2 000 rows of 1 500 entries, fp32, n = 64: 168 -> 49; 400 of 4 000, fp64, n = 40: 1 255 -> 83;
// 512 of 8 000, column-major, fp32, n = 16: 1 043 -> 37.  Against four workgroups per compute unit: 4 000 rows of 64, n = 64:
// 5.9 (7.3), 2 000 of 1 500, n = 64: 49 (60), n = 200: 300 (233).
constexpr int kGroupFill = 512;
constexpr int kGroupLongLeast = 64;  // entries: the join of the groups' sums is not worth less (400 rows of 40: the same)
struct GroupTile {
  int rows, long_row;
};
__host__ __device__ constexpr GroupTile group_tile(int m, int chunks, int most) {
  int rows = most;
  while (rows > 1 && ((int64_t)m + rows - 1) / rows * chunks < kGroupFill) rows /= 2;
  const int share = rows < kGroupRows ? kGroupLongRow / kGroupRows * rows : kGroupLongRow;
  return {rows, share < kGroupLongLeast ? kGroupLongLeast : share};
}

// The lane at column c of a chunk of cn columns loads V columns from c0 on and stores all but the first `first` of them.
// Where the chunk ends inside a load it is moved back (what its neighbour has as well is `first`), into the chunk before
// where this one holds fewer than V columns: c0 is negative then, and every row of B has the columns there.  Lanes past the
// end load what is sure to be there and store nothing.  padded: 16 bytes behind a row may be read, nothing is moved.
struct GroupColumns {
  int c0, first;
  bool owns;
};
template <int V>
__host__ __device__ constexpr GroupColumns group_columns(int c, int cn, bool padded) {
  // (in this form a load of one element, V == 1, is seen never to move: 8 registers fewer, complex128)
  if (c >= cn) return {V > 1 && !padded && cn < V ? cn - V : 0, 0, false};
  if (c + V > cn && !padded) return {cn - V, c + V - cn, true};
  return {c, 0, true};
}

// Where that load begins, in bytes: from B's row on (`narrow`: offsets into all of B, never negative there), otherwise from
// the chunk's first column on, which may be negative and stays signed when it is added to a 64-bit address.
__host__ __device__ constexpr int group_lane_bytes(bool narrow, int64_t chunk_bytes, int c0, int size) {
  return (int)((narrow ? chunk_bytes : 0) + (int64_t)c0 * size);
}
__host__ __device__ constexpr int64_t group_far_bytes(int row_hi, unsigned row_lo, int lane_bytes) {
  return (int64_t)(((uint64_t)(unsigned)row_hi << 32) | row_lo) + lane_bytes;
}

// where a lane's L pieces of a row of B lie
template <bool NARROW, int L>
struct GroupB {
  BufferRsrc rsrc;    // NARROW: all of B, within 2 GiB
  const char* p;      // otherwise: the chunk's first column of row 0
  int lane_bytes[L];  // group_lane_bytes of the lane's pieces
  int64_t row_bytes;
};

// One block of sixteen entries of a row, an entry per lane: lane l of a group holds entry part + S * (place in the part),
// so that step j of part p takes entry p + S j of the block.  Kept as loaded until the block is worked on: arithmetic on it
// here would wait for the loads.
template <typename T>
struct GroupBlock {
  T val;
  int col;
  bool live;
};

template <typename T, int GC>
__device__ __forceinline__ GroupBlock<T> group_fetch(unsigned j0, unsigned end, const T* __restrict__ val,
                                                     const int* __restrict__ col_ind) {
  const int l16 = threadIdx.x & 15;
  const unsigned j = j0 + l16 / GC + (16 / GC) * (l16 % GC);
  GroupBlock<T> e;
  e.live = j < end;
  // Every lane loads, the ones past the end entry 0 (there is one): a load under a branch would be waited for where the
  // branches meet.  (Not non-temporally: a block is half a cache line of column numbers, and the line's other half is the
  // row's next block.  2^20 rows of 32 random entries, n = 64: 1.29 -> 1.24 ms.)
  e.col = col_ind[e.live ? j : 0];
  e.val = val[e.live ? j : 0];
  return e;
}

// acc += a block's entries times the lane's columns of B; all lanes of the wave come here together
template <typename T, int GC, bool NARROW, int L, bool FAR>
__device__ __forceinline__ void group_work(const GroupBlock<T>& e, T alpha, int base, const GroupB<NARROW, L>& b,
                                           T (&acc)[L * kGroupV<T>]) {
  constexpr int V = kGroupV<T>;
  const bool upper = GC == 8 && (threadIdx.x & 8);
  const uint64_t mask = __builtin_amdgcn_ballot_w64(e.live);
  const T weight = e.live ? alpha * e.val : T(0);
  unsigned off = kGroupNoRow;
  int off_hi = 0;
  if constexpr (NARROW) {
    if (e.live) off = (unsigned)(e.col - base) * (unsigned)b.row_bytes;
  } else {
    const int64_t o = e.live ? (int64_t)(e.col - base) * b.row_bytes : 0;
    off = (unsigned)o;
    off_hi = (int)(o >> 32);
  }
  auto steps = [&](auto first, auto count) {
    constexpr int J0 = decltype(first)::value, N = decltype(count)::value;
    GroupVec<T> bv[N][L];
    bool has[N];
    auto load = [&](auto u) {
      constexpr int U = decltype(u)::value;
      const unsigned lo = (unsigned)part_bcast<GC, J0 + U>((int)off, upper);
      if constexpr (NARROW) {
#pragma unroll
        for (int q = 0; q < L; ++q) bv[U][q] = buffer_load<GroupVec<T>>(b.rsrc, (int)(lo + (unsigned)b.lane_bytes[q]));
      } else {
        has[U] = part_bcast<GC, J0 + U>((int)e.live, upper) != 0;
        const int hi = part_bcast<GC, J0 + U>(off_hi, upper);
        if (has[U]) {
#pragma unroll
          for (int q = 0; q < L; ++q)
            bv[U][q] = __builtin_bit_cast(
                GroupVec<T>, *reinterpret_cast<const GroupLoose<T>*>(b.p + group_far_bytes(hi, lo, b.lane_bytes[q])));
        }
      }
    };
    auto add = [&](auto u) {
      constexpr int U = decltype(u)::value;
      const T w = part_bcast_t<GC, J0 + U>(weight, upper);
      // (a lane group whose row has ended adds 0 * 0: its offset was turned away)
      if (NARROW || has[U]) {
#pragma unroll
        for (int q = 0; q < L; ++q) {
#pragma unroll
          for (int i = 0; i < V; ++i) acc[q * V + i] = fma_t(w, bv[U][q].e[i], acc[q * V + i]);
        }
      }
    };
    for_each_const(load, std::make_integer_sequence<int, N>{});
    for_each_const(add, std::make_integer_sequence<int, N>{});
  };
  // Loads in flight per wave: four (eight took 20 registers more and were no faster).  FAR: one at a time where most lanes
  // have an entry and neighbouring rows begin far apart: the L2-miss path is full either way, and fewer requests
  // in it go faster (2^20 rows of 32 random entries, fp32, n = 64: 1.26 -> 1.21 ms; chunks
  // of two loads a lane have as many lines in flight by themselves, 438 520 rows of 21 entries, fp64, n = 63: 0.69 -> 0.65;
  // rows of few entries and B within
  // the caches are latency-bound and lose up to a third).
  if constexpr (FAR) {
    const int c0 = __builtin_amdgcn_readlane(e.col, 0), c1 = __builtin_amdgcn_readlane(e.col, 16);
    const int c2 = __builtin_amdgcn_readlane(e.col, 32), c3 = __builtin_amdgcn_readlane(e.col, 48);
    if (__builtin_popcountll(mask) >= 48 && (unsigned)(c1 - c0 + 256) > 512u && (unsigned)(c3 - c2 + 256) > 512u) {
      auto one = [&](auto j) { steps(j, std::integral_constant<int, 1>{}); };
      for_each_const(one, std::make_integer_sequence<int, GC>{});
      return;
    }
  }
  auto four = [&](auto q) {
    constexpr int J = 4 * decltype(q)::value;
    if (mask & part_lanes<GC>(J, J + 4)) steps(std::integral_constant<int, J>{}, std::integral_constant<int, 4>{});
  };
  for_each_const(four, std::make_integer_sequence<int, GC / 4>{});
}

// acc += the blocks of sixteen entries of a row at j0, j0 + step, ... before `end`, every group with blocks of its own; the
// parts' sums are not yet joined.  (Positions are below 2^31, so that an unsigned one a step past the end has not wrapped;
// 64-bit ones took 2 to 14 registers more.)
template <typename T, int GC, bool NARROW, int L, bool FAR>
__device__ __forceinline__ void group_walk(unsigned j0, unsigned end, unsigned step, T alpha, const T* __restrict__ val,
                                           const int* __restrict__ col_ind, int base, const GroupB<NARROW, L>& b,
                                           T (&acc)[L * kGroupV<T>]) {
  GroupBlock<T> cur = group_fetch<T, GC>(j0, end, val, col_ind);
  while (__builtin_amdgcn_ballot_w64(j0 + step < end)) {  // the next sixteen travel while these are worked on
    j0 += step;
    const GroupBlock<T> next = group_fetch<T, GC>(j0, end, val, col_ind);
    group_work<T, GC, NARROW, L, FAR>(cur, alpha, base, b, acc);
    cur = next;
  }
  group_work<T, GC, NARROW, L, FAR>(cur, alpha, base, b, acc);
}

// every part of the group receives the sum over the parts
template <int GC, typename T, int N>
__device__ __forceinline__ void group_join(T (&acc)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    if constexpr (GC <= 8) acc[i] += dpp_mov<0x128>(acc[i]);  // row_ror:8
    if constexpr (GC <= 4) acc[i] += dpp_mov<0x124>(acc[i]);  // row_ror:4
  }
}

typedef int Loose4 __attribute__((ext_vector_type(4), aligned(4)));

// the V columns from c on, but not the first `first` of them; nt: C bypasses the caches
template <typename T>
__device__ __forceinline__ void group_store_row(T* __restrict__ c, int first, const T* acc, T beta, bool nt) {
  constexpr int V = kGroupV<T>;
  if (first == 0) {
    GroupVec<T> out;
    if (beta == T(0)) {
#pragma unroll
      for (int i = 0; i < V; ++i) out.e[i] = acc[i];
    } else {
      const Loose4* p = reinterpret_cast<const Loose4*>(c);
      const GroupVec<T> old = __builtin_bit_cast(GroupVec<T>, nt ? __builtin_nontemporal_load(p) : *p);
#pragma unroll
      for (int i = 0; i < V; ++i) out.e[i] = old.e[i] * beta + acc[i];
    }
    if (nt) __builtin_nontemporal_store(__builtin_bit_cast(Loose4, out), reinterpret_cast<Loose4*>(c));
    else *reinterpret_cast<Loose4*>(c) = __builtin_bit_cast(Loose4, out);
  } else {
#pragma unroll
    for (int i = 1; i < V; ++i)
      if (i >= first) c[i] = beta == T(0) ? acc[i] : c[i] * beta + acc[i];
  }
}

// grid.x: blocks of tile.rows rows, a power of two of at most kGroupRows (COLC: kWave; FAR: exactly that many); grid.y:
// chunks of `chunk` dense columns, chunk y at B + y * b_chunk_bytes (b_bytes: what may be read from B on, NARROW only).  ldb in elements; C element (r, c) at
// r * c_row + c * c_col (one of the two strides is 1: COLC when it is the rows').  b_padded: 16 bytes behind every row of
// B may be read (a layout made here); otherwise n is at least kGroupV<T>.  L: 128-bit loads per lane and row of B, the
// chunk's columns [q * GC * V, (q + 1) * GC * V) in load q.  c_nt: row-major C, which is touched once, bypasses the caches.
// FAR: see group_work.
template <typename T, int GC, bool NARROW, bool COLC, int L, bool FAR>
__global__ __launch_bounds__(kGroupThreads) void spmm_group_kernel(
    int m, int n, T alpha, const T* __restrict__ val, const int* __restrict__ row_ptr, const int* __restrict__ col_ind,
    int base, const T* __restrict__ B, int64_t ldb, int64_t b_chunk_bytes, unsigned b_bytes, bool b_padded, T beta,
    T* __restrict__ C, int64_t c_row, int64_t c_col, int chunk, GroupTile tile, bool c_nt) {
  constexpr int V = kGroupV<T>;
  constexpr int kCols = GC * V;
  constexpr int kTileRows = COLC ? kWave : kGroupRows;
  __shared__ T s_part[kGroupRows * kCols * L];          // the groups' sums of a long row
  __shared__ T s_tile[COLC ? kCols * (kWave + 1) : 1];  // COLC: the rows' sums, column by column
  __shared__ int s_ptr[kTileRows + 1];
  static_assert(!COLC || L == 1, "column-major C with one load per lane");
  const unsigned bid = xcd_contiguous_id(blockIdx.x, gridDim.x);
  // (FAR: constants, runtime values took 30 to 50 registers more and two of six waves per SIMD there)
  const int tile_rows = FAR ? kTileRows : tile.rows;
  const int long_row = FAR ? kGroupLongRow : tile.long_row;
  const int64_t row0 = (int64_t)bid * tile_rows;
  if (row0 >= m) return;
  const int nrows = m - row0 < tile_rows ? (int)(m - row0) : tile_rows;
  if ((int)threadIdx.x <= nrows) s_ptr[threadIdx.x] = row_ptr[row0 + threadIdx.x];
  const int group = threadIdx.x / 16;
  const int lane = threadIdx.x % kWave;
  const int cl = threadIdx.x % GC;
  const int cbeg = blockIdx.y * chunk;
  const int cn = n - cbeg < chunk ? n - cbeg : chunk;
  int c0[L], first[L];
  bool owns[L];
  GroupB<NARROW, L> b;
  if constexpr (NARROW) b.rsrc = make_rsrc(B, (int)b_bytes);
  b.p = reinterpret_cast<const char*>(B) + (int64_t)blockIdx.y * b_chunk_bytes;
  b.row_bytes = ldb * (int64_t)sizeof(T);
#pragma unroll
  for (int q = 0; q < L; ++q) {
    const GroupColumns mine = group_columns<V>(q * kCols + cl * V, cn, b_padded);
    c0[q] = mine.c0;
    first[q] = mine.first;
    owns[q] = mine.owns && threadIdx.x % 16 < GC;
    b.lane_bytes[q] = group_lane_bytes(NARROW, (int64_t)blockIdx.y * b_chunk_bytes, mine.c0, (int)sizeof(T));
  }
  auto put = [&](int r, const T(&acc)[L * V]) {  // the tile's row r: the lanes that own columns
#pragma unroll
    for (int q = 0; q < L; ++q) {
      if (!owns[q]) continue;
      const int have = cn - c0[q] < V ? cn - c0[q] : V;  // (fewer than V with a padded B only)
      if constexpr (COLC) {
#pragma unroll
        for (int i = 0; i < V; ++i)
          if (i >= first[q] && i < have) s_tile[(c0[q] + i) * (kWave + 1) + r] = acc[q * V + i];
      } else {
        T* c = C + (row0 + r) * c_row + cbeg + c0[q];
        if (have == V) {
          group_store_row<T>(c, first[q], &acc[q * V], beta, c_nt);
        } else {
#pragma unroll
          for (int i = 0; i < V; ++i)
            if (i < have) c[i] = beta == T(0) ? acc[q * V + i] : c[i] * beta + acc[q * V + i];
        }
      }
    }
  };
  __syncthreads();
#pragma unroll 1
  for (int pass = 0; pass < kTileRows / kGroupRows; ++pass) {
    if (pass > 0 && pass * kGroupRows >= nrows) break;
    const int r = pass * kGroupRows + group;
    int start = 0, end = 0;
    bool there = r < nrows;
    if (there) {
      start = s_ptr[r] - base;
      end = s_ptr[r + 1] - base;
    }
    if (end - start > long_row) {
      there = false;
      end = start;
    }
    T acc[L * V];
#pragma unroll
    for (int i = 0; i < L * V; ++i) acc[i] = T(0);
    group_walk<T, GC, NARROW, L, FAR>(start, end, 16, alpha, val, col_ind, base, b, acc);
    group_join<GC>(acc);
    if (there) put(r, acc);
  }
  // The workgroup's long rows, one after the other.  The groups take blocks of sixteen in turn, so that a workgroup sweeps the
  // row together: rows of ascending columns then read neighbouring rows of B at one time (a sixteenth of the row each:
  // 2 000 rows of 1 500, fp32, n = 64, 71 us against 49).
  uint64_t long_rows = __builtin_amdgcn_ballot_w64(lane < nrows && s_ptr[lane + 1] - s_ptr[lane] > long_row);
  for (; long_rows; long_rows &= long_rows - 1) {  // (the same in every wave)
    const int r = __builtin_ctzll(long_rows);
    const int start = s_ptr[r] - base, end = s_ptr[r + 1] - base;
    T acc[L * V];
#pragma unroll
    for (int i = 0; i < L * V; ++i) acc[i] = T(0);
    group_walk<T, GC, NARROW, L, FAR>(start + 16 * group, end, 16 * kGroupRows, alpha, val, col_ind, base, b, acc);
    group_join<GC>(acc);
    if (threadIdx.x % 16 < GC) {
#pragma unroll
      for (int i = 0; i < L * V; ++i) s_part[(group * GC + cl) * L * V + i] = acc[i];
    }
    __syncthreads();
    if (group == 0) {
      for (int g = 1; g < kGroupRows; ++g) {
#pragma unroll
        for (int i = 0; i < L * V; ++i) acc[i] += s_part[(g * GC + cl) * L * V + i];
      }
      put(r, acc);
    }
    __syncthreads();
  }
  if constexpr (COLC) {
    __syncthreads();
    if (lane < nrows) {
      for (int c = threadIdx.x / kWave; c < cn; c += kGroupThreads / kWave) {
        T* out = C + row0 + lane + (int64_t)(cbeg + c) * c_col;
        const T sum = s_tile[c * (kWave + 1) + lane];
        nt_store(beta == T(0) ? sum : nt_load(out) * beta + sum, out);
      }
    }
  }
}

}  // namespace asamd
