// The permutation of a decode-sized batch in one workgroup (perm_single and route_perm_small): the
// same order as the chunked kernels of permute.hip.
#pragma once

#include "common.hpp"
#include "internal.hpp"

namespace lbmoe {

// LDS of perm_single_body: R * 16 virtual waves, experts up to EMAX (128, 256, 512 or 1024).
template <int R, int EMAX>
struct PermSingleLds {
  static constexpr int kW = kPermSingle / kWave;
  static constexpr int kVW = kW * R;                  // virtual waves
  static constexpr int kParts = kPermSingle / EMAX;   // threads per expert in the prefix pass
  static_assert(kVW % kParts == 0 && EMAX * kParts == kPermSingle, "threads cover the count table");
  alignas(16) int cnt[kVW][EMAX];                     // per virtual wave and expert: count, prefix
  int psum[kParts][EMAX];
  int start[EMAX];                                    // first row of each expert
  int wsum[kW];
};

// Whole permutation in one workgroup for decode-sized batches (V <= R * kPermSingle): thread
// tid takes entries v = r * kPermSingle + tid, r < R, so that "virtual wave" vw = v / 64 =
// r * (kPermSingle / 64) + wave covers 64 consecutive entries. Each virtual wave ranks its
// entries among equal experts (ballot match) and records its count per expert; the counts then
// turn into per-virtual-wave prefixes (in v order) and totals, a block scan of the totals gives
// the offsets, and every entry lands at offsets[e] + (entries of e in earlier virtual waves) +
// rank. Bound by latency on its one CU, so the prefix pass spreads an expert's virtual waves over
// kParts threads, each with its counts in registers at once (one thread per expert walking up to
// 64 LDS counts, one after another, took half the launch), and the count table is no wider than
// EMAX.
// The body, for a workgroup of kPermSingle threads that all call it (idx may point to LDS).
template <int IB, int R, int EMAX>
__device__ __forceinline__ void perm_single_body(PermSingleLds<R, EMAX>& lds, const void* idx, int T,
                                                 int k, int E, int nbits, int V, int32_t* counts,
                                                 int32_t* offsets, int32_t* perm_tok,
                                                 int32_t* perm_slot, int32_t* inv) {
  using L = PermSingleLds<R, EMAX>;
  constexpr int kW = L::kW, kVW = L::kVW, kParts = L::kParts, kPer = kVW / kParts;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  u32x4* z = reinterpret_cast<u32x4*>(&lds.cnt[0][0]);
  for (int i = tid; i < kVW * EMAX / 4; i += kPermSingle) z[i] = u32x4{0, 0, 0, 0};
  int e[R], s[R], t[R], rank[R];
  bool valid[R];
  // unconditional loads (entries past V read entry V-1 and are masked); V = 0 reads nothing
#pragma unroll
  for (int r = 0; r < R; ++r) {
    e[r] = -1;
    s[r] = t[r] = 0;
  }
  if (V > 0) {                           // the same for every thread
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int v = min(r * kPermSingle + tid, V - 1);
      s[r] = v / T;
      t[r] = v - s[r] * T;
      e[r] = load_expert<IB>(idx, static_cast<int64_t>(t[r]) * k + s[r]);
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (r * kPermSingle + tid >= V) e[r] = -1;
  }
  uint64_t m[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    valid[r] = (e[r] >= 0) && (e[r] < E);
    m[r] = match_expert(valid[r] ? e[r] : 0, __ballot(valid[r]), nbits);
    rank[r] = mask_rank(m[r]);
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (valid[r] && rank[r] == 0) lds.cnt[r * kW + wave][e[r]] = __popcll(m[r]);
  __syncthreads();
  const int ex = tid & (EMAX - 1), part = tid / EMAX;      // expert, its share of the virtual waves
  int c[kPer], mine = 0;
#pragma unroll
  for (int i = 0; i < kPer; ++i) c[i] = lds.cnt[part * kPer + i][ex];
#pragma unroll
  for (int i = 0; i < kPer; ++i) mine += c[i];
  int run = 0, sum = mine;
  if constexpr (kParts > 1) {
    lds.psum[part][ex] = mine;
    __syncthreads();
    sum = 0;
#pragma unroll
    for (int p = 0; p < kParts; ++p) {
      const int v = lds.psum[p][ex];
      run += p < part ? v : 0;
      sum += v;
    }
  }
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    lds.cnt[part * kPer + i][ex] = run;
    run += c[i];
  }
  const int total = tid < E ? sum : 0;                     // part 0: tid is the expert
  int incl = total;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int y = __shfl_up(incl, o, kWave);
    if (lane >= o) incl += y;
  }
  if (lane == kWave - 1) lds.wsum[wave] = incl;
  __syncthreads();
  int before = 0;
#pragma unroll
  for (int w = 0; w < kW; ++w) {
    const int v = lds.wsum[w];
    before += w < wave ? v : 0;
  }
  const int excl = before + incl - total;
  if (tid < E) {
    lds.start[tid] = excl;
    counts[tid] = total;
    offsets[tid] = excl;
  }
  if (tid == kPermSingle - 1) offsets[E] = before + incl;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r * kPermSingle + tid >= V) continue;
    const int64_t ts = static_cast<int64_t>(t[r]) * k + s[r];
    if (!valid[r]) {
      inv[ts] = -1;
    } else {
      const int pos = lds.start[e[r]] + lds.cnt[r * kW + wave][e[r]] + rank[r];
      perm_tok[pos] = t[r];
      perm_slot[pos] = s[r];
      inv[ts] = pos;
    }
  }
}

}  // namespace lbmoe
