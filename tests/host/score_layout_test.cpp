// The score kernel's LDS for every number of taps: its 16-byte stores lie on
// 16-byte boundaries, and what it indexes lies inside its part.
#include "score_layout.hpp"

#include <cstdio>

int main() {
  int bad = 0;
  for (int nt = 0; nt <= 64; ++nt) {
    const ctas::ScoreLayout l = ctas::score_layout(nt);
    const bool ok = l.mid % 4 == 0 && ctas::kScoreSW % 4 == 0 && ctas::kScoreSH % 4 == 0  //
                    && l.reach >= (nt > 0 ? nt - 1 : 0)                                  // the taps' lines
                    && l.rows * l.cols <= l.mid && l.floats - l.mid >= l.rows * ctas::kScoreSW
                    // four outputs of the last column and row, and the derivatives' border
                    && l.reach + ctas::kScoreSW <= l.cols && l.reach + ctas::kScoreSH <= l.rows
                    && ctas::kScoreSH * ctas::kScoreSW <= l.mid && ctas::kScoreSH >= ctas::kScoreTH + 2
                    && ctas::kScoreSW >= ctas::kScoreTW + 2 && l.floats * 4 <= 160 * 1024 - 64;
    if (!ok) std::printf("failed: %d taps, tile %d x %d, second part at %d\n", nt, l.rows, l.cols, l.mid);
    bad += !ok;
  }
  return bad != 0;
}
