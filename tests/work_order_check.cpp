// Host check of csrc/work_order.hpp (no GPU), built and run by tests/test_work_order.py: over grids of every kind, each (tile, pair, member)
// is taken by exactly one workgroup, and beyond a resident grid the XCDs (workgroup number % 8) get equal shares of causal work, which falls
// linearly from the first tile to the last.  The order that gave each of the last pairs an XCD of its own has to fail.
#include <algorithm>
#include <cstdio>
#include <vector>

#include "work_order.hpp"

using namespace segpt;

namespace {

// the order that left XCDs idle: its grid has a workgroup for every pair of a full round of eight, missing pairs do nothing
Item one_pair_an_xcd(int block, int tiles, int pairs, int members, int64_t) {
  const int per = tiles * members, k = block / kXcds, rest = k % per;
  return {rest / members, kXcds * (k / per) + block % kXcds, rest % members};
}

template <typename F>
const char* check(F order, int tiles, int pairs, int members, int64_t stream, int grid) {
  const int n = tiles * pairs * members;
  std::vector<int> taken(n);
  int64_t work[kXcds] = {};
  for (int block = 0; block < grid; ++block) {
    const Item it = order(block, tiles, pairs, members, stream);
    if (it.pair >= pairs) continue;
    if (it.tile < 0 || it.tile >= tiles || it.pair < 0 || it.member < 0 || it.member >= members) return "out of range";
    if (taken[(it.tile * pairs + it.pair) * members + it.member]++) return "taken twice";
    work[block % kXcds] += tiles - it.tile;
  }
  if (std::count(taken.begin(), taken.end(), 1) != n) return "not taken";
  // up to four groups of pairs, in each of which an XCD takes every at most eighth piece: one piece more or less
  const auto range = std::minmax_element(work, work + kXcds);
  if (n > kPinnedGrid && *range.second - *range.first > 4 * tiles) return "unequal shares";
  return nullptr;
}

}  // namespace

int main() {
  int cases = 0, caught = 0;
  for (int n = 1; n <= 1300; ++n) {
    std::vector<int> plain(n), xcd(n);
    for (int id = 0; id < n; ++id) {
      ++plain.at(work_item(id, n));
      ++xcd.at(work_item_xcd(id, n));
      // whole rounds keep an item's XCD; without that the rounds themselves are mirrored
      if (id / 256 * 256 + 256 <= n && work_item_xcd(id, n) % kXcds != id % kXcds) return 1;
      if (n <= 1024 && id / 256 % 2 && id / 256 * 256 + 256 <= n && work_item(id, n) != id / 256 * 256 + 255 - id % 256) return 1;
    }
    if (std::count(plain.begin(), plain.end(), 1) != n || std::count(xcd.begin(), xcd.end(), 1) != n) return 1;
  }
  for (int tiles : {1, 2, 3, 7, 8, 31, 64, 257})
    for (int pairs = 1; pairs <= 41; ++pairs)
      for (int members : {1, 2, 3, 5, 8, 32})
        for (int64_t stream : {(int64_t)1, kStreamLimit / 3, kStreamLimit * 99}) {
          const int n = tiles * pairs * members;
          if (const char* what = check(split_item, tiles, pairs, members, stream, n)) {
            std::printf("VIOLATION %s: %d tiles, %d pairs, %d members\n", what, tiles, pairs, members);
            return 1;
          }
          ++cases;
          if (n > kPinnedGrid && pairs % kXcds && tiles >= 31 && check(one_pair_an_xcd, tiles, pairs, members, stream, (pairs + 7) / 8 * 8 * tiles * members)) ++caught;
        }
  std::printf("%d grids ok, %d caught\n", cases, caught);
  return caught ? 0 : 1;
}
