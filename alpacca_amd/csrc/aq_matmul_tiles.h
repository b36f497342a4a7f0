// aq_matmul_tiles.h - how the matmul tile kernels choose a tile shape and a
// split of K.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace aq {

// A tile shape: the time (us) of one 64-column stage when every CU has one
// workgroup and when it has two (0: no second one fits beside the first, or
// the shape is not built), by kind of weights, and of the ends of a tile
// (prologue, stores).
struct TileCost {
  int bm, bn;
  float one[3], two[3], ends;
};
struct TileModel {
  const TileCost *tiles;
  int n;
  float low;    // a stage's time on few CUs over its time on all of them
  float us_mb;  // the traffic of a split's partials, us per 10^6 bytes
};

// The shape and split of least estimated time: rounds of one or two
// workgroups per CU, the tiles' ends, and for a split the partials (each
// written and read, the sum written).  K is `units` units of `stages` stages;
// a split has at least min_units of them and there are at most max_splits.
inline void choose_tile(const TileModel &model, int kind, int64_t M, int64_t N, int units,
                        int stages, int min_units, int cus, int max_splits, int &shape,
                        int &splits) {
  float best = 0.f;
  shape = -1;
  for (int t = 0; t < model.n; ++t) {
    const TileCost &c = model.tiles[t];
    if (c.one[kind] == 0.f) continue;
    const int64_t tiles = ((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn);
    for (int want = 1; want <= max_splits; ++want) {
      if (want > 1 && (want * min_units > units || (want - 1) * tiles >= 2 * (int64_t)cus)) break;
      const int per = (units + want - 1) / want, sp = (units + per - 1) / per;
      if (sp != want) continue;
      const int64_t wgs = tiles * sp, ones = (wgs + cus - 1) / cus;
      const float low = model.low + (1.f - model.low) * std::min(1.f, (float)wgs / (float)cus);
      float rounds;  // of a stage's time
      if (c.two[kind] == 0.f) {
        rounds = (float)ones * c.one[kind] * low;
      } else {
        const int64_t full = wgs / (2 * cus), rest = wgs - full * 2 * cus;
        rounds = (float)full * c.two[kind] +
                 (rest > cus ? c.two[kind] : rest > 0 ? c.one[kind] * low : 0.f);
      }
      float us = rounds * (float)(stages * per) + c.ends * (float)ones;
      if (sp > 1) us += 0.2f + (float)((2 * sp + 1) * M * N) * 4e-6f * model.us_mb;
      if (shape < 0 || us < best) {
        best = us;
        shape = t;
        splits = sp;
      }
    }
  }
}

}  // namespace aq
