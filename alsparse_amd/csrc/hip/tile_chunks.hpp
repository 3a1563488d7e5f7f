// Host side: how the column blocks of the tiled layouts are cut into chunks of the first phase (spmv_tiled.hpp,
// spmv_sums.hpp).  The reference has no counterpart.
#pragma once

#include <algorithm>
#include <cstdint>
#include <functional>
#include <utility>
#include <vector>

namespace asamd {

// The most units (spans, entries) of a chunk, of least, least + step, ... most; sizes[c]: a column block's units, cut into as
// few pieces, as even, as the limit allows.  One workgroup to a compute unit (the x slice fills its LDS), so what counts is
// how full the last round of chunks is, and how often a slice is loaded: the limit whose rounds, each as long as its longest
// chunk, are the shortest together.  A slice mostly comes from an L2 and costs three quarters of its bytes (of none, a half,
// three quarters and all of them the one that puts the limits in the order in which they were measured).
inline int chunk_limit(const std::vector<int>& sizes, int64_t unit_bytes, int64_t slice_bytes, int64_t cus, int least, int most,
                       int step) {
  int best = least;
  int64_t best_cost = -1;
  std::vector<std::pair<int, int>> pieces(sizes.size());  // a block's longest piece, and how many
  for (int limit = least; limit <= most; limit += step) {
    for (size_t c = 0; c < sizes.size(); ++c) {
      const int k = (sizes[c] + limit - 1) / limit;
      pieces[c] = {k > 0 ? (sizes[c] + k - 1) / k : 0, k};
    }
    std::sort(pieces.begin(), pieces.end(), std::greater<>());
    int64_t cost = 0, at = 0, round = 0;  // chunks handed out, first chunk of the next round
    for (const auto& [longest, count] : pieces)
      for (at += count; round < at; round += cus) cost += slice_bytes / 4 * 3 + longest * unit_bytes;
    if (best_cost < 0 || cost < best_cost) {
      best = limit;
      best_cost = cost;
    }
  }
  return best;
}

// A list of chunks for every XCD: a column block's chunks in one list as far as the lists stay even, the longest chunks first
// (the short ones even out the workgroups' ends).  size[i]: chunk i; block[i]: its column block, ascending.
inline std::vector<std::vector<int>> chunk_lists(const std::vector<int>& size, const std::vector<int>& block, int xcds) {
  int64_t all = 0;
  for (int s : size) all += s;
  std::vector<std::vector<int>> list((size_t)xcds);
  std::vector<int64_t> load((size_t)xcds, 0);
  size_t to = 0;
  for (int i = 0; i < (int)size.size(); ++i) {
    if (i == 0 || block[(size_t)i] != block[(size_t)i - 1] || (load[to] + size[(size_t)i]) * xcds > all)
      to = (size_t)(std::min_element(load.begin(), load.end()) - load.begin());
    list[to].push_back(i);
    load[to] += size[(size_t)i];
  }
  for (auto& l : list)
    std::stable_sort(l.begin(), l.end(), [&](int a, int b) { return size[(size_t)a] > size[(size_t)b]; });
  return list;
}

// The order in which chunks are handed to workgroups: workgroup i runs on XCD i % xcds, so the lists' chunks in turn.  Where a
// list has ended, those behind it move up: the last, shortest chunks of the longer lists run on other XCDs than their list's.
inline std::vector<int> chunk_order(const std::vector<int>& size, const std::vector<int>& block, int xcds) {
  const std::vector<std::vector<int>> list = chunk_lists(size, block, xcds);
  std::vector<int> order;
  order.reserve(size.size());
  for (size_t at = 0; order.size() < size.size(); ++at)
    for (const auto& l : list)
      if (at < l.size()) order.push_back(l[at]);
  return order;
}

}  // namespace asamd
