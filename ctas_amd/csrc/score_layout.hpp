// LDS of the score kernel (axis.hip), in floats. Host and device code.
#pragma once

namespace ctas {

constexpr int kScoreTH = 32, kScoreTW = 64;                      // derivatives of a tile
constexpr int kScoreSH = kScoreTH + 4, kScoreSW = kScoreTW + 4;  // smoothed rows and columns: 34 and 66, rounded up to fours

// nt taps: the tile of the slice with the rows and columns that they reach,
// [rows][cols] from 0 (later the smoothed tile, [kScoreSH][kScoreSW]), and at
// `mid`, on a 16-byte boundary for its 16-byte stores, the tile smoothed along
// rows, [rows][kScoreSW].
struct ScoreLayout {
  int reach, rows, cols, mid, floats;
};
constexpr ScoreLayout score_layout(int nt) {
  const int e = nt > 0 ? nt - 1 : 0, rows = kScoreSH + e, cols = kScoreSW + e;
  const int mid = (rows * cols + 3) & ~3;
  return {e, rows, cols, mid, mid + rows * kScoreSW};
}

}  // namespace ctas
