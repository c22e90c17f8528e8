// Which launches backproject a batch of slices, and what the autotuner keeps.
// Host code on plain values.
#pragma once

#include <cstdint>
#include <cstring>
#include <map>
#include <numeric>
#include <vector>

namespace ctas {

// Tile kinds: rows x cols of output per 256-thread workgroup. The two small
// ones serve launches of CTAS sampling from float32 storage whose 64x64 tiles
// would leave most of the chip idle; they are not among a caller's choices.
enum TileKind { TK_AUTO = 0, TK_64x64 = 1, TK_128x64 = 2, TK_128x128 = 3, TK_32x32 = 4, TK_16x32 = 5 };
inline int tile_rows(int kind) { return kind == TK_16x32 ? 16 : kind == TK_32x32 ? 32 : kind == TK_64x64 ? 64 : 128; }
inline int tile_cols(int kind) { return kind >= TK_32x32 ? 32 : kind == TK_128x128 ? 128 : 64; }

// What the autotuner found for a class of widths and angle counts: the fastest
// kind and pass length of one slice per workgroup, which uneven batches take,
// and what handles without settings of their own take for such launches: that
// kind where it was faster than the launches below on 64x64 tiles, else those.
struct Tuned {
  int kind = TK_64x64, ac = 32;  // the tuned choice at 512-4096 px on MI355X
  int ac64 = 32;                 // the fastest pass length of 64x64 tiles
  bool beats_plan = false;
  int handle_kind() const { return beats_plan ? kind : TK_64x64; }
  int handle_ac() const { return beats_plan ? ac : ac64; }
};

struct PlanShape {
  int w, N, cus;
  int kind;  // of one-slice launches
  int set_kind, set_ac;  // the tile kind and pass length that the caller set; 0: none
  bool f32;  // CTAS sampling of float32 storage
  bool linear;
  bool mirror;  // on tiles of `kind`, through mirrored angle pairs
};

// One backprojection launch: `items` items from `first`, `group` slices per
// workgroup, on tiles of `kind`.
struct BpLaunch {
  int first, items, group, kind;
};

// The launches that backproject S slices, and the order in which the item
// table holds them (slices of a group lie back to back).
//
// Slices of one centre share their ray coordinates, so CTAS sampling of
// float32 storage, and of 16-bit storage through mirrored angle pairs, takes
// four or two of them per workgroup on 64x64 tiles, where that leaves enough
// workgroups. Measured for 1 to 8 slices of 512 to 4096 px on 256 CUs, four
// win from 448 workgroups (float32; 484 of 1400 px 445 us against 570 with
// two and 768 alone, 288 of 768 px 274 against 258 and 353) and 484 (16-bit;
// 544 of 2048 px 1111 us against 1387 and 1430, 288 of 1024 px 559 against
// 513 and 454), two from 288 (float32; 183 us against 234, 256 workgroups 272
// against 264) and 726 (16-bit; 571 us against 717, 576 workgroups 513
// against 454). What remains is taken one by one; float32 launches of less
// than two 64x64 tiles per CU take 32x32 tiles, and 16x32 ones up to a
// quarter of a tile per CU (backproject.hip). Mirrored launches of few tile
// pairs take quarters of them: LINEAR below four per CU, where whole ones do not
// fill the chip once (144 of 1024 px 165 us against 389, 484 of 1400 px 485
// against 532, 1008 of 1024 px 750 against 773, 1088 of 2048 px 1541 against
// 1520), 16-bit below three (144 113 against 215, 726 of 1400 px 394 against 410). A
// tile kind or a pass length that the caller set is kept for every slice, one
// slice per workgroup.
inline std::vector<BpLaunch> plan_launches(const PlanShape &h, const float *centers, int S, std::vector<int> *order) {
  order->resize(S);
  std::iota(order->begin(), order->end(), 0);
  const int kind = h.kind;
  const bool linear = h.linear, f32 = h.f32, mirror = h.mirror;
  if (h.set_kind != TK_AUTO || h.set_ac != 0 || (!f32 && !mirror) || static_cast<long long>(h.N) * h.w >= (1LL << 30))
    return {{0, S, 1, kind}};
  const long long rows = (h.w + 63) / 64, cols = mirror ? (h.w / 2 + 64) / 64 : rows;
  const long long tiles = rows * cols, cus = h.cus;
  const long long four = (mirror ? 15 : 14) * cus / 8, two = (mirror ? 20 : 9) * cus / 8;
  const long long small = (linear ? 4 : 3) * cus;
  auto single = [&](int first, int n) {
    BpLaunch l{first, n, 1, kind};
    if (f32 && 4 * n * tiles <= cus) l.kind = TK_16x32;
    else if (f32 && n * tiles < 2 * cus) l.kind = TK_32x32;
    else if (mirror && kind == TK_64x64 && n * tiles < small) l.kind = TK_32x32;
    return l;
  };
  if (linear) return {single(0, S)};
  if (f32 && S * tiles < 2 * cus) return {single(0, S)};
  std::map<uint32_t, std::vector<int>> by_centre;
  for (int i = 0; i < S; ++i) {
    uint32_t bits;
    std::memcpy(&bits, centers + i, sizeof bits);
    by_centre[bits].push_back(i);
  }
  std::vector<BpLaunch> launches;
  std::vector<int> at;
  for (const int group : {4, 2}) {
    long long n = 0;
    for (const auto &c : by_centre) n += static_cast<long long>(c.second.size()) / group;
    if (n * tiles < (group == 4 ? four : two)) continue;
    const int first = static_cast<int>(at.size());
    for (auto &c : by_centre) {
      const size_t take = c.second.size() / group * group;
      at.insert(at.end(), c.second.begin(), c.second.begin() + take);
      c.second.erase(c.second.begin(), c.second.begin() + take);
    }
    launches.push_back({first, static_cast<int>(at.size()) - first, group, TK_64x64});
  }
  if (launches.empty()) return {single(0, S)};
  const int first = static_cast<int>(at.size());
  for (const auto &c : by_centre) at.insert(at.end(), c.second.begin(), c.second.end());
  if (first < S) launches.push_back(single(first, S - first));
  *order = at;
  return launches;
}

}  // namespace ctas
