// TEST INFRASTRUCTURE.  The column arithmetic of the sixteen-lane SpMM groups (spmm_group.hpp), enumerated on the host: for
// every width, element size and chunk width each lane's load lies inside its row of B, in both address forms, and
// every column is stored once; and the rows that a workgroup takes, for every number of rows.  Prints the first violation and returns 1, or returns 0.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <vector>

#include "spmm_group.hpp"

using namespace asamd;

template <int SIZE>
static bool check(int chunk_bytes_most, bool lines) {
  constexpr int V = 16 / SIZE;
  const int most = chunk_bytes_most / SIZE, unit = lines ? 128 / SIZE : V;
  int64_t narrow_chunks = 0;
  for (int n = 2 * V + 1; n <= 36 * most; ++n) {
    const GroupChunks g = group_chunks(n, most, unit);
    std::vector<int> stored(n, 0);
    bool ok = g.chunk >= 1 && g.chunk <= most && g.chunk % unit == 0 && (int64_t)g.chunk * (g.count - 1) < n &&
              (int64_t)g.chunk * g.count >= n;
    for (int y = 0; ok && y < g.count; ++y) {
      const int cbeg = y * g.chunk, cn = n - cbeg < g.chunk ? n - cbeg : g.chunk;
      const int64_t chunk_at = (int64_t)cbeg * SIZE;
      if (cn < V) ++narrow_chunks;
      for (int c = 0; ok && c < most; c += V) {  // (every lane and load that the widest group has)
        const GroupColumns m = group_columns<V>(c, cn, false);
        for (int64_t row : {(int64_t)0, (int64_t)0xFFFFFFF0, (int64_t)0x7FFFFFFF0, (int64_t)n * SIZE * 3}) {
          const int64_t far = chunk_at + group_far_bytes((int)(row >> 32), (unsigned)row, group_lane_bytes(false, chunk_at, m.c0, SIZE)) - row;
          ok = ok && far >= 0 && far + 16 <= (int64_t)n * SIZE && far == chunk_at + (int64_t)m.c0 * SIZE;
        }
        const unsigned near = 4096u + (unsigned)group_lane_bytes(true, chunk_at, m.c0, SIZE);
        ok = ok && near >= 4096u && near - 4096u + 16 <= (unsigned)n * SIZE && near - 4096u == (unsigned)(chunk_at + (int64_t)m.c0 * SIZE);
        if (m.owns)
          for (int i = m.first; ok && i < V; ++i) {
            const int col = cbeg + m.c0 + i;
            ok = col >= 0 && col < n && m.c0 + i >= 0 && m.c0 + i < cn;
            if (ok) ++stored[col];
          }
      }
    }
    for (int c = 0; ok && c < n; ++c) ok = stored[c] == 1;
    if (!ok) {
      printf("element size %d, chunks of at most %d bytes, n = %d: chunk %d, %d of them\n", SIZE, chunk_bytes_most, n, g.chunk, g.count);
      return false;
    }
  }
  // (8- and 4-byte elements have last chunks narrower than a load: the case that has to be moved into the chunk before)
  if (V > 1 && narrow_chunks == 0) printf("element size %d: no chunk narrower than a load\n", SIZE);
  return V == 1 || narrow_chunks > 0;
}

// Every row is one workgroup's: a power of two of rows each, the last workgroup begins before row m.
static bool check_tiles() {
  for (int most : {kGroupRows, (int)kWave})
    for (int chunks : {1, 2, 4, 1000})
      for (int64_t m = 1; m < 2147483647; m = m < 70000 ? m + 1 : m * 3 + 1) {
        const GroupTile t = group_tile((int)m, chunks, most);
        const int64_t grid = (m + t.rows - 1) / t.rows;
        const bool whole = (m + most - 1) / most * chunks >= kGroupFill;
        if (t.rows < 1 || t.rows > most || (t.rows & (t.rows - 1)) || (grid - 1) * t.rows >= m || grid * t.rows < m ||
            t.long_row < kGroupLongLeast || t.long_row > kGroupLongRow || (whole && (t.rows != most || t.long_row != kGroupLongRow))) {
          printf("m = %lld, %d chunks, tiles of at most %d: %d rows, long from %d\n", (long long)m, chunks, most, t.rows, t.long_row);
          return false;
        }
      }
  return true;
}

int main() {
  bool ok = check_tiles();
  for (int bytes : {kGroupBytes, 2 * kGroupBytes})
    for (bool lines : {false, true}) ok = check<4>(bytes, lines) && check<8>(bytes, lines) && check<16>(bytes, lines) && ok;
  return ok ? 0 : 1;
}
