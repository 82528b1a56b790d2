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
// each step slower, and walk a popular expert's rows pass after pass; the tiled ones barely depend on
// the counts, but a launch takes whole rounds of the CUs (one workgroup each). So what counts in bf16 is
//   - the share of the last round that idles: gate_up's items are one per expert and 128
//     intermediate channels, the shared expert's one per 256 tokens and 128 channels, and two of
//     those past a whole number of rounds cost a round (H = 2048, E = 64, I = Is = 512, 13 tokens:
//     streaming 91 us, tiled 114; without the shared expert 84 / 85);
//   - down's (rows of 256 output channels, cheaper items);
//   - a launch of less than one round, whose length is its longest item's;
//   - a shared expert wider than the routed ones: the streaming launches' workgroups are laid out by
//     the wider of the two, the routed ones past their own width idle (H = 2048, E = 512, I = 256, Is
//     = 512, 8 tokens: 416 / 316);
//   - the experts: the more there are, the more of a skewed routing's rows lie with few of them. Under
//     a Zipf bias tiled takes 0.9 of streaming's time at E = 32 and 13 tokens per expert, 0.6 at 128,
//     0.3 at 512 (Qwen3-30B-A3B with a shared expert, 13 tokens: 142 / 66 us).
// The host cannot see the skew. The weights come from 5420 layer calls timed both ways (GPU us, in turn
// in one process; E = 32..512, I = 128..768, Is = 0, 256, 512, H = 512, 1024, 2048, 8 to 27 tokens per
// expert), for the least expected log time with three uniform calls to one under a Zipf bias: uniform
// calls then lie 0.6% above the faster side, more than 3% above streaming in 2% of the cases, at worst
// 10%. By the routed experts' items alone they lay 1.4% above it, at worst 25% above streaming, and the
// calls under a bias 4% higher.
// fp8 (its streaming kernels stream less per wave) gains more from the tiles under a bias, 0.8 at E = 32
// and 0.25 at 512 and 10 tokens per expert, against up to 16% on uniform calls with a shared expert: 10
// tokens for all is within 0.1% of the best line over its sizes.
// Below 0.7 items per CU only the four-tile passes are slower (E = 16, I = 512: 25 tokens 32 / 36).
constexpr double kTiledAlways = 28.0;

inline double tiled_min_tokens(const CallSizes& c) {
  if (static_cast<int64_t>(c.E) * (c.I / 128) * 10 < int64_t{7} * c.cus) return kTiledAlways;
  if (c.fp8) return 10.0;
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
  const double wider = sh ? std::clamp(2.0 * (c.Is - c.I) / c.I, 0.0, 1.0) : 0.0;
  const double t = 8.0 + 16.0 * idle(gate_up) + 4.0 * idle(down) + (gate_up < c.cus ? 6.0 : 0.0) -
                   8.0 * wider - (c.E >= 128 ? 4.0 : 0.0);
  return std::clamp(t, gate_up >= 4 * c.cus ? 8.0 : 10.0, kTiledAlways);
}

// Whether a batch that fits (kInlineRouteTokens, kInlineRouteEntries) is better routed inside the
// bf16 decode gate_up kernel, by every workgroup for itself, than by a launch of its own. Up to 4
// tokens always: a wave selects one token. With 5 to 8 each wave selects up to two, which a CU repeats
// for every workgroup it runs, and more experts per lane hold more registers, so fewer workgroups are
// resident: the more of them per CU, the more of the saved launch goes. Measured (us per layer,
// separate / inside) around the lines:
//   E <= 256: 5 per CU 43.8 / 42.9, 7.5 71.8 / 71.1 and 33.8 / 33.3, 8 81.7 / 79.7; 8.1 55.5 / 57.2,
//     9 35.7 / 38.0, 10.5 49.7 / 51.9, 12 40.1 / 43.4
//   E <= 512: 2.5 31.1 / 28.2, 4 36.4 / 34.2; 4.6 51.7 / 56.1, 5 30.2 / 31.2, 8 36.1 / 39.4
//   E > 512: 2 30.9 / 29.7, 3 48.6 / 46.9; 3.1 37.7 / 41.3, 3.5 38.9 / 42.2, 7 79.0 / 83.9
inline bool route_in_gate_up_pays(const CallSizes& c, int k) {
  if (c.T <= 4) return true;
  const int64_t rows = std::min<int64_t>(c.T * k, c.E) + (c.Is > 0 ? 1 : 0);
  const int64_t per_cu = c.E <= 256 ? 8 : c.E <= 512 ? 4 : 3;
  return std::max(c.I, c.Is) / 16 * rows <= per_cu * c.cus;
}

// Whether a batch behind the residual add and RMSNorm takes the router that also selects (where the
// plain block does, route_in_router). Behind the norm's own kernel the plain router and the selection
// of their own cost as many launches more as without it, but the selecting router's workgroups each
// compute the shared expert's gate of 64 tokens one after another, and at short rows its launch is
// little shorter (us, plain router / selecting: Qwen3-30B-A3B T=1024 267.5 / 264.1; I = 256: H = 2048,
// E = 96, k = 1, T=4096 with a shared expert of 512 145.5 / 155.4, without one T=6000 135 / 140,
// T=8192 169 / 166; E = 48, k = 4, T=1500 103.5 / 98.7; H = 1024, E = 64, k = 1, shared, T=3000 80.4 /
// 86.1; H = 512, E = 16, k = 2, T=1024 46.2 / 48.5, T=8192 65.7 / 65.3; H = 1024 without a shared
// expert within 2% either way).
inline bool norm_takes_selecting_router(const CallSizes& c) { return c.Is == 0 && c.H >= 1024; }

}  // namespace lbmoe
