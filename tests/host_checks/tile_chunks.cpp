// TEST INFRASTRUCTURE.  The chunks of the tiled layouts' first phase (tile_chunks.hpp) on the host: the limit lies in its
// range and finds a full round; every chunk is in one XCD's list, the longest first; no list is longer than its share by more
// than a chunk, a column block is in one list but where a list is full, and the order takes from the lists in turn.
// Prints the first violation and returns 1, or returns 0.
#include <cstdio>
#include <random>
#include <set>

#include "tile_chunks.hpp"

using namespace asamd;

static int fail(const char* what, int at) {
  std::printf("%s (%d)\n", what, at);
  return 1;
}

static int check_lists(const std::vector<int>& size, const std::vector<int>& block, size_t xcds, int t) {
  const std::vector<std::vector<int>> list = chunk_lists(size, block, (int)xcds);
  if (list.size() != xcds) return fail("not a list for every XCD", t);
  std::vector<int> seen(size.size(), 0);
  std::set<int> blocks;
  int64_t all = 0, most = 0;
  size_t shortest = size.size(), pairs = 0;
  for (size_t i = 0; i < size.size(); ++i) {
    all += size[i];
    most = std::max<int64_t>(most, size[i]);
    blocks.insert(block[i]);
  }
  for (const auto& l : list) {
    int64_t load = 0;
    std::set<int> here;
    for (size_t i = 0; i < l.size(); ++i) {
      ++seen[(size_t)l[i]];
      load += size[(size_t)l[i]];
      here.insert(block[(size_t)l[i]]);
      if (i > 0 && size[(size_t)l[i]] > size[(size_t)l[i - 1]]) return fail("a longer chunk behind a shorter one", t);
    }
    // A chunk goes to a list that it does not fill past its share, or to the shortest one, which is at most the share.
    if (load * (int64_t)xcds > all + most * (int64_t)xcds) return fail("an XCD above its share", t);
    shortest = std::min(shortest, l.size());
    pairs += here.size();
  }
  for (int s : seen)
    if (s != 1) return fail("a chunk that is not in one list", t);
  // A block goes on in another list where its list is full.  A full list is within a chunk of its share, and it is the
  // shortest one again only where all are, with at most a chunk a list still to come: few more than one list a block.
  if (pairs > blocks.size() + 3 * xcds) return fail("column blocks over many XCDs", t);
  const std::vector<int> order = chunk_order(size, block, (int)xcds);
  if (order.size() != size.size()) return fail("chunks more or less", t);
  std::set<int> once(order.begin(), order.end());
  if (once.size() != order.size()) return fail("a chunk handed out twice", t);
  for (size_t i = 0; i < shortest * xcds; ++i)
    if (order[i] != list[i % xcds][i / xcds]) return fail("not from the lists in turn", t);
  return 0;
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
    // (sizes of their own, from a whole chunk down to one unit; a crowded block now and then)
    for (int c = 0; c < blocks; ++c) {
      const int k = (units[(size_t)c] + limit - 1) / limit * (rng() % 9 == 0 ? 20 : 1);
      for (int i = 0; i < k; ++i) {
        size.push_back(1 + (int)(rng() % (unsigned)limit));
        block.push_back(c);
      }
    }
    if (const int e = check_lists(size, block, 8, t)) return e;
  }
  // eight blocks of equal weight, eight XCDs: each keeps a block
  std::vector<int> size(80, 5), block(80);
  for (int i = 0; i < 80; ++i) block[(size_t)i] = i / 10;
  const std::vector<int> order = chunk_order(size, block, 8);
  for (size_t i = 0; i < 80; ++i)
    if (block[(size_t)order[i]] != block[(size_t)order[i % 8]]) return fail("a block on two XCDs", (int)i);
  return 0;
}
