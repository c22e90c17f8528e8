// The launches of plan_launches on 256 compute units, and what handles take of
// the autotuner's findings.
#include "bp_plan.hpp"

#include <cstdio>
#include <set>
#include <string>

using namespace ctas;

namespace {
int g_bad = 0;
void check(bool ok, const std::string &what) {
  if (!ok) std::printf("failed: %s\n", what.c_str());
  g_bad += !ok;
}

enum Mode { F32, F16_MIRROR, F16_PLAIN, LIN_MIRROR, LIN_PLAIN, MODES };
PlanShape shape(Mode m, int w, int set_kind, int set_ac) {
  return {w,      1800,     256, set_kind ? set_kind : TK_64x64,      set_kind, set_ac,
          m == F32, m == LIN_MIRROR || m == LIN_PLAIN, m == F16_MIRROR || m == LIN_MIRROR};
}

// Every slice once, a group's of one centre, one kind of tile that its kernel has.
void plans() {
  for (int m = 0; m < MODES; ++m)
    for (int w : {2, 64, 512, 1400, 2048, 4096})
      for (int S : {1, 2, 3, 7, 32, 257})
        for (int centres : {1, 2, 5, 300}) {
          std::vector<float> c(S);
          for (int i = 0; i < S; ++i) c[i] = 0.25f * static_cast<float>(i * 7 % centres);
          const std::string tag = "mode " + std::to_string(m) + " w " + std::to_string(w) + " slices " +
                                  std::to_string(S) + " centres " + std::to_string(centres);
          std::vector<int> order;
          int at = 0;
          for (const BpLaunch &l : plan_launches(shape(static_cast<Mode>(m), w, 0, 0), c.data(), S, &order)) {
            check(l.first == at && l.items > 0 && l.items % l.group == 0, tag + ": back to back");
            check(l.group == 1 || (l.kind == TK_64x64 && (m == F32 || m == F16_MIRROR)), tag + ": groups");
            check(l.kind != TK_16x32 || m == F32, tag + ": 16x32");
            check(l.kind != TK_32x32 || m == F32 || m == F16_MIRROR || m == LIN_MIRROR, tag + ": 32x32");
            for (int k = 0; k < l.items; ++k)
              check(c[order[l.first + k]] == c[order[l.first + k / l.group * l.group]], tag + ": one centre");
            at += l.items;
          }
          check(at == S && std::set<int>(order.begin(), order.end()).size() == static_cast<size_t>(S), tag + ": all");
        }
}

// A tile kind or a pass length of the caller's: that kind, a slice per workgroup,
// in the caller's order.
void settings() {
  const std::vector<float> c(32, 1.5f);
  for (int m = 0; m < MODES; ++m)
    for (int w : {64, 512, 2048})
      for (int S : {1, 2, 32})
        for (int kind : {0, 1, 2, 3})
          for (int ac : {0, 16, 32}) {
            if (!kind && !ac) continue;
            std::vector<int> order;
            const auto l = plan_launches(shape(static_cast<Mode>(m), w, kind, ac), c.data(), S, &order);
            const std::string tag = "mode " + std::to_string(m) + " kind " + std::to_string(kind) + " pass " + std::to_string(ac);
            check(l.size() == 1 && l[0].first == 0 && l[0].items == S && l[0].group == 1, tag + ": one launch");
            check(l[0].kind == (kind ? kind : TK_64x64), tag + ": the kind");
            for (int i = 0; i < S; ++i) check(order[i] == i, tag + ": the order");
          }
}

// Handles keep 64x64 tiles, on which small and grouped launches build, unless
// another kind was measured against those launches.
void tuned() {
  Tuned t;
  t.kind = TK_128x64;
  t.ac = 32;
  t.ac64 = 16;
  check(t.handle_kind() == TK_64x64 && t.handle_ac() == 16, "not measured against the launches");
  t.beats_plan = true;
  check(t.handle_kind() == TK_128x64 && t.handle_ac() == 32, "measured faster than the launches");
}
}  // namespace

int main() {
  plans();
  settings();
  tuned();
  return g_bad != 0;
}
