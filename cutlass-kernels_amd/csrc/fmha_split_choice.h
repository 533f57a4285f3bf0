// Which calls with e4m3 Q and K have some items' keys cut into units of work of their own (SplitCfg builds of the compiler-scheduled
// kernels, 128 rows), and into how many: host code.
#pragma once
#include <cmath>

#include "fmha_common.h"

namespace cfk {

// about the larger of two times that overlap: the sixth root of the sum of their sixth powers
inline float either(float a, float b) {
  a *= a * a, b *= b * b;
  return cbrtf(sqrtf(a * a + b * b));
}

// Times, us, of a build that has `places` workgroups on a CU.  tile[x]: 64 keys of each of x workgroups on every CU; more of them run in rounds,
// a fifth less unevenly than whole ones where a CU has several places.  round: what a round of workgroups takes besides; cut: what a cut call takes besides (the merge is a
// launch of its own), with its partial results at part_rate MB/us; K, V, Q, O, and partial results pass at 8 MB/us.
struct CutTimes {
  int places;
  float tile[4], round, first, cut, part_rate;
};

// The shapes that a call is cut in are few: all items, or those behind one whole round, into as many units as go round the CUs j times, as
// long as all of a CU's workgroups are there at once.
// Fitted to 1650 drawn calls, N(0,1), each with up to ten cuts (rms of the error 3 to 15 %).  110 other calls that this cuts, about one in 25
// drawn, both in turn: 0.746 of the time that they took whole (geometric mean), worst 1.003.  us, whole -> cut: e4m3 D=128, V
// pre-transposed, 38 heads of 224 rows, 12480 keys 108.2 -> 46.7; D=256, 15 heads of 2624 rows, 7360 keys 229 -> 163; hybrid D=128, 20 heads of 480 rows, 6848 keys
// 82.9 -> 42.6; D=256, 28 heads of 1472, 2944 keys 139.8 -> 115.0.
// No gain, and the rule keeps off: whatever takes less than about 25 us; e4m3 up to head dim 128 below 3072 keys (0.99); items behind more
// than a round of workgroups (0.96 to 1.04: idle CUs leave the others their power).  And calls of the key-split kernel stay there, although
// 20 heads of 256 rows, D=256, 7872 keys would go 88.3 -> 41.2 us: it multiplies V by weights in 16 bits, error against
// float64 2.8e-4 of the size of O where the builds with e4m3 weights have 2.6e-2, and 2.8e-4 against 2.9e-4 in hybrid calls.
inline bool choose_cut(const CutTimes &c, int items, int skv, int step_keys, float mbytes, int head_dim, const FmhaPlan &plan, KeySplit *out) {
  constexpr int kCus = 256;
  const int steps = skv / step_keys;
  const float tiles = skv / 64.f;
  const auto tile_us = [&](float x) {
    const float rounds = ceilf(x / c.places) - 1, y = x - rounds * c.places, full = c.tile[c.places];
    const int i = y < c.places ? (int)y : c.places - 1;
    const float us = rounds * full + c.tile[i] + (c.tile[i + 1] - c.tile[i]) * (y - i);
    return rounds > 0 && c.places > 1 ? 0.8f * us + 0.2f * full * x / c.places : us;
  };
  const float x = (float)items / kCus;
  // (the hand-scheduled and the 256-row builds, taken where they are faster, get less of a lead)
  const float whole_us = (plan.hand || plan.block_m != 128 ? 0.92f : 1.f) * (c.first + either(tiles * tile_us(x) + c.round * ceilf(x / c.places), mbytes / 8.f));
  float best = whole_us;
  bool found = false;
  for (int from : {0, c.places * kCus}) {
    const int cut = items - from;
    for (int j = 1; cut > 0 && j <= c.places; ++j) {
      const int n = j * kCus / cut < 64 ? j * kCus / cut : 64;
      if (n < 2 || 3 * n > steps) continue;
      const float unit = (float)((steps + n - 1) / n) * step_keys / 64.f, part = 4e-6f * n * cut * 128 * head_dim;   // MB
      float us = (from ? tiles * tile_us((float)c.places) + c.round : 0.f) + unit * tile_us((float)n * cut / kCus) + c.round;
      us = c.first + either(us, (mbytes + part) / 8.f) + c.cut + part / c.part_rate;
      if (us < 0.92f * whole_us && us < best) best = us, *out = KeySplit{n, 128, from}, found = true;
    }
  }
  return found;
}

}  // namespace cfk
