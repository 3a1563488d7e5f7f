// TEST INFRASTRUCTURE.  The chunks of the tiled layouts' first phase (tile_chunks.hpp) on the host: the limit lies in its
// range and finds a full round; every chunk is handed out once, no XCD gets far more than its share, and where column
// blocks and XCDs come out even each block stays on one.
// Prints the first violation and returns 1, or returns 0.
#include <cstdio>
#include <random>

#include "tile_chunks.hpp"

using namespace asamd;

static int fail(const char* what, int at) {
  std::printf("%s (%d)\n", what, at);
  return 1;
}

int main() {
  // 64 equal blocks of 256 units: pieces of 64 are one round of 256, of 32 two, of 48 (six a block) one and a half
  if (chunk_limit(std::vector<int>(64, 256), 12288, 131072, 256, 16, 96, 4) != 64) return fail("limit of a full round", 0);
  if (chunk_limit({}, 12288, 131072, 256, 16, 96, 4) != 16 || chunk_limit({0, 0}, 1, 1, 256, 16, 96, 4) != 16)
    return fail("limit without units", 0);
  std::mt19937 rng(1);
  for (int t = 0; t < 3000; ++t) {
    const int blocks = 1 + (int)(rng() % 60);
    std::vector<int> units((size_t)blocks), size, block;
    for (int& u : units) u = (int)(rng() % 700);
    const int limit = chunk_limit(units, 10240, 131072, 256, 16, 96, 4);
    if (limit < 16 || limit > 96) return fail("limit outside its range", t);
    int most = 0;
    int64_t all = 0;
    for (int c = 0; c < blocks; ++c) {
      const int k = (units[(size_t)c] + limit - 1) / limit * (rng() % 9 == 0 ? 20 : 1);  // (a crowded block now and then)
      for (int i = 0; i < k; ++i) {
        size.push_back(1 + (int)(rng() % 3) + limit);
        block.push_back(c);
        most = std::max(most, size.back());
        all += size.back();
      }
    }
    const std::vector<int> order = chunk_order(size, block, 8);
    std::vector<int> seen(size.size(), 0);
    for (int i : order) ++seen[(size_t)i];
    for (int s : seen)
      if (s != 1) return fail("a chunk that is not handed out once", t);
    if (order.size() != size.size()) return fail("chunks more or less", t);
    int64_t load[8] = {};
    bool even = true;  // the lists are as long as each other but for the last turn
    for (size_t i = 0; i < order.size(); ++i) load[i % 8] += size[(size_t)order[i]];
    for (int64_t l : load) even = even && l * 8 <= all + 16 * (int64_t)most * 8;
    if (!even) return fail("an XCD far above its share", t);
  }
  // eight blocks of equal weight, eight XCDs: each keeps a block
  std::vector<int> size(80, 5), block(80);
  for (int i = 0; i < 80; ++i) block[(size_t)i] = i / 10;
  const std::vector<int> order = chunk_order(size, block, 8);
  for (size_t i = 0; i < 80; ++i)
    if (block[(size_t)order[i]] != block[(size_t)order[i % 8]]) return fail("a block on two XCDs", (int)i);
  return 0;
}
