// Host-side lines between two kernels of one job, as functions of a call's sizes alone.
//
// Plain C++ with no HIP dependency, so the lines can be checked by a host compiler alone.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace lbmoe {

// A call's sizes: Is = 0 when the call has no shared expert.
struct CallSizes {
  int E, H, I, Is;
  int64_t T;
  bool fp8;
  int cus;
};

// Tokens per routed expert from which the LDS-tiled GEMMs replace weight streaming. The streaming
// kernels run two token tiles per pass above 8 tokens per expert and four above 28 (kTiledAlways),
// each step slower; the tiled ones barely depend on the count, but a launch takes whole rounds of the
// CUs (one workgroup each), so what counts is
//   - the share of the last round that idles: gate_up's items are one per expert and 128
//     intermediate channels, the shared expert's one per 256 tokens and 128 channels, and two of
//     those past a whole number of rounds cost a round (bf16 H = 2048, E = 64, I = Is = 512, 13
//     tokens: streaming 91 us, tiled 114; without the shared expert 84 / 85);
//   - down's (rows of 256 output channels, cheaper items);
//   - a launch of less than one round, whose length is its longest item's;
//   - for fp8, a shared expert (its wide item then holds up a short launch) and short k ranges (H =
//     512: four k-tiles per item);
//   - a shared expert wider than the routed ones: the streaming launches' workgroups are laid out by
//     the wider of the two, the routed ones past their own width idle (H = 2048, E = 512, I = 256, Is
//     = 512, 8 tokens: 416 / 316).
// The weights come from 3036 layer calls timed both ways (GPU us, in turn in one process; E = 32..512, I =
// 128..768, Is = 0, 256, 512, H = 512, 1024, 2048, 8 to 27 tokens per expert, uniform routing): the
// side taken is slower than the other by more than 3% in 2% of the bf16 and 6% of the fp8 calls, and
// slower than streaming by more than 3% in 0.5% and 2%, at worst 9%. A line by the routed items
// alone lost more than 3% to streaming in 6% and 15%, up to 25%.
// Skewed routings gain from the tiled kernels earlier: under a Zipf bias the streaming kernels walk a
// popular expert's rows pass after pass (E = 512, 7.5 tokens: 477 / 139).
// Below 0.7 items per CU only the four-tile passes are slower (E = 16, I = 512: 25 tokens 32 / 36).
constexpr double kTiledAlways = 28.0;

inline double tiled_min_tokens(const CallSizes& c) {
  if (static_cast<int64_t>(c.E) * (c.I / 128) * 10 < int64_t{7} * c.cus) return kTiledAlways;
  const bool sh = c.Is > 0;
  const int64_t sh_tiles = sh ? (c.T + 255) / 256 : 0;
  const int64_t gate_up = static_cast<int64_t>(c.E) * (c.I / 128) + sh_tiles * (c.Is / 128);
  const int64_t down = (c.E + sh_tiles) * (c.H / 256);
  // the time a launch's last round idles, in units of its items' time
  auto idle = [&](int64_t items) {
    if (items <= 0) return 1.2;
    const double rounds = static_cast<double>((items + c.cus - 1) / c.cus);
    return std::min(1.2, rounds * c.cus / static_cast<double>(items) - 1.0);
  };
  const bool part = gate_up < c.cus;
  const double wider = sh ? std::clamp(2.0 * (c.Is - c.I) / c.I, 0.0, 1.0) : 0.0;
  double t;
  if (c.fp8) {
    const bool long_item = sh && gate_up * 10 < int64_t{13} * c.cus &&
                           (c.T > 256 || c.T % 256 == 0 || c.T % 256 > 128);
    t = 6.0 + (sh ? 3.0 + 8.0 * idle(gate_up) : 0.0) + (part ? 4.0 : 0.0) + (long_item ? 4.0 : 0.0) +
        (c.H <= 512 ? 5.0 : 0.0) - 4.0 * wider;
    return std::clamp(t, 10.0, kTiledAlways);
  }
  t = 9.0 + 16.0 * idle(gate_up) + 4.0 * idle(down) + (part ? 8.0 : 0.0) - (c.H <= 512 ? 3.0 : 0.0) -
      12.0 * wider;
  return std::clamp(t, 8.0, kTiledAlways);
}

}  // namespace lbmoe
