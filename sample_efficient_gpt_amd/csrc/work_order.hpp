// Which piece of work a workgroup of the fp32 kernels takes.  Plain C++ (constexpr, so device code too): included by the kernels and
// by tests/work_order_check.cpp, which checks on the host that every piece is taken exactly once and that no XCD idles.
#pragma once

#include <cstdint>

namespace segpt {

// Work items are listed heaviest first.  When the whole grid is resident at once (up to two workgroups on each of 256
// CUs) or nearly so, the CU that got item i also gets item i + 256: every second round of 256 is dealt in reverse, so
// that a heavy item shares its CU with a light one (2 x 8 / 4 heads of 1000 tokens, us: forward 39.7 -> 33.8, backward 121 -> 109).  Larger grids
// balance by themselves and keep the plain order (dK/dV 3 % slower reversed at 9216 items).
__attribute__((always_inline)) constexpr int work_item(int id, int n) {
  const int round = id >> 8;
  if (n > 1024 || !(round & 1)) return id;
  return (round << 8) + 255 < n ? (round << 8) + 255 - (id & 255) : n - 1 - (id & 255);
}
// The same with whole rounds reversed in eights, which keeps an item's XCD: where the items of an XCD share what they stream (split_item).  Three-bf16
// kernels, us, work_item -> this: 2 x 8 / 4 heads of 1000 tokens forward 27.8 -> 26.4, 18 / 6 heads of 512 backward 51.5 -> 47.9.  The fp32 instructions'
// kernels do not gain: backward 109 -> 113.
__attribute__((always_inline)) constexpr int work_item_xcd(int id, int n) {
  const int round = id >> 8;
  if (n > 1024 || !(round & 1)) return id;
  const int x = id & 255;
  return (round << 8) + 255 < n ? (round << 8) + 248 - (x & 248) + (x & 7) : n - 1 - x;
}

// Which tile a workgroup takes: (tile, heaviest first; (batch, kv head); member of the pair: query head or part).  The streamed
// tiles of the pairs that an XCD works on at a time should stay in its L2 (2.4 MB a pair at 2048 keys of 64).
//   * Up to 512 workgroups, resident at once: in work_item_xcd's order; from 256 on with the pairs before the members, so that an XCD
//     sees every eighth pair with all its members (us, members before pairs -> this: forward of 8 x 32 / 4 heads, one query, 4096 keys of 64 148 ->
//     75, fp32 instructions 107; fewer workgroups do not fill the memory side and are 5 % faster spread: 16 / 4 heads, 64 queries, 2048 keys 33.9, 35.2).
//     Up to 1024 the same if what an XCD then streams is no more than a few times its L2: it balances the causal tail (4 x 8 heads of 1000
//     tokens: backward 138, 141 in the order below; forward of 32 x 16 / 4 heads, 64 queries, 2048 keys: 210, 159, fp32 instructions 189).
//   * More: eight pairs at a time, one on each XCD; the last pairs % 8 as four, two and one, each on two, four or all XCDs, so that none idles
//     (us, the last ones on an XCD each -> this: 8 heads on one kv head, 8192 tokens of 64: forward 2273 -> 393, backward 4487 -> 1799; 18 / 6
//     heads, 8192 tokens 1098 -> 856, 3768 -> 3640).
struct Item {
  int tile, pair, member;
};
constexpr int kPinnedGrid = 1024, kResident = 512, kXcds = 8;
constexpr int64_t kL2Bytes = 4 << 20, kStreamLimit = 4 * kL2Bytes;
// `stream`: bytes of the streamed tiles of one pair.  What an XCD streams in work_item_xcd's order:
__attribute__((always_inline)) constexpr int64_t stream_per_xcd(int pairs, int64_t stream) { return stream * (pairs % kXcds ? pairs : pairs / kXcds); }
__attribute__((always_inline)) constexpr Item split_item(int block, int tiles, int pairs, int members, int64_t stream) {
  Item it{};
  const int per = tiles * members;
  const int64_t total = (int64_t)per * pairs;
  if (total <= kResident || (total <= kPinnedGrid && stream_per_xcd(pairs, stream) <= kStreamLimit)) {
    const int n = per * pairs, id = work_item_xcd(block, n), rest = id % (pairs * members);
    it.tile = id / (pairs * members);
    it.pair = n < 256 ? rest / members : rest % pairs;
    it.member = n < 256 ? rest % members : rest / pairs;
    return it;
  }
  int first = 0, at_once = kXcds, left = block;  // the group of pairs the workgroup belongs to: first .. first + at_once - 1
  const int rounds = pairs / kXcds;
  if (left < rounds * kXcds * per) {
    first = left / (kXcds * per) * kXcds;
    left -= first * per;
  } else {
    first = rounds * kXcds;
    left -= first * per;
    for (at_once = kXcds / 2; !(pairs & at_once) || left >= at_once * per; at_once /= 2)
      if (pairs & at_once) { left -= at_once * per; first += at_once; }
  }
  it.pair = first + left % at_once;
  const int rest = left / at_once;
  it.tile = rest / members;
  it.member = rest % members;
  return it;
}

}  // namespace segpt
