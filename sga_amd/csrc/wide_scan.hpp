// Scans and rank searches of one wide workgroup (16 waves): what the one-workgroup steps of the
// selects are made of.
#pragma once
#include "common.hpp"

namespace sga {

constexpr int kWide = 1024;                       // threads of the one-workgroup kernels
constexpr int kWideWaves = kWide / kWave;         // 16
constexpr int kWideBins = 4096;                   // LDS histogram of a descent level: 12 bits

#ifdef __HIPCC__

// LDS scratch of the workgroup-wide scans.  Consecutive scans alternate between the two halves
// (`turn`), so one scan's last reads and the next one's first writes need no barrier between them.
struct WideScratch {
  uint32_t tot[2][kWideWaves];
  uint32_t hit[2][2][3];
};

// The sixteen waves' totals as every wave sees them: what lies before the calling wave, and all of it.  By
// lanes: sixteen reads and adds a wave are 0.4 us where four waves share a SIMD's issue.
__device__ __forceinline__ uint32_t wide_waves_before(const uint32_t* tot, uint32_t& all) {
  const uint32_t incl = row_incl_scan(tot[lane_id() % kWideWaves]);
  all = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWideWaves - 1);
  const int w = uniform_i32(wave_id());
  return w ? (uint32_t)__builtin_amdgcn_readlane((int)incl, w - 1) : 0u;
}

// Exclusive prefix sum over the workgroup, and the total.  One barrier.
__device__ __forceinline__ uint32_t wide_prefix(uint32_t mine, WideScratch& s, int turn, uint32_t& total) {
  const uint32_t incl = wave_incl_scan(mine);
  if (lane_id() == kWave - 1) s.tot[turn][wave_id()] = incl;
  __syncthreads();
  return incl - mine + wide_waves_before(s.tot[turn], total);
}

// The workgroup's totals of two numbers.  One barrier; takes both halves of the scratch.
__device__ __forceinline__ void wide_totals(uint32_t a, uint32_t b, WideScratch& s, uint32_t& all_a, uint32_t& all_b) {
  a = wave_incl_scan(a);
  b = wave_incl_scan(b);
  if (lane_id() == kWave - 1) { s.tot[0][wave_id()] = a; s.tot[1][wave_id()] = b; }
  __syncthreads();
  wide_waves_before(s.tot[0], all_a);
  wide_waves_before(s.tot[1], all_b);
}

struct RankHit { uint32_t bin, above, count; };
// The bins of an LDS histogram where the count from the top reaches each of NR ranks
// (1-based).  All threads get the answers.  Two barriers, after the one that completes the histogram; look(keys
// above, keys in, counts of the calling thread's bins) runs before the second.
template <int NR, int BINS = kWideBins, class L>
__device__ __forceinline__ void wide_find_rank(const uint32_t* s_hist, const uint32_t (&rank)[NR],
                                               WideScratch& s, int turn, RankHit (&hit)[NR], L&& look) {
  constexpr int PER = BINS / kWide;                // 4 or 8
  static_assert(PER % 4 == 0, "whole quads of bins per thread");
  uint32_t h[PER], mine = 0;
#pragma unroll
  for (int j = 0; j < PER; j += 4) {
    const U4 q = reinterpret_cast<const U4*>(s_hist)[threadIdx.x * (PER / 4) + j / 4];
    h[j] = q.x; h[j + 1] = q.y; h[j + 2] = q.z; h[j + 3] = q.w;
    mine += (q.x + q.y) + (q.z + q.w);
  }
  uint32_t total;
  const uint32_t before = wide_prefix(mine, s, turn, total);
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    uint32_t above = total - before - mine;
    if (above < rank[r] && rank[r] <= above + mine) {
#pragma unroll
      for (int j = PER - 1; j >= 0; --j) {
        if (above < rank[r] && rank[r] <= above + h[j]) {
          s.hit[turn][r][0] = (uint32_t)(threadIdx.x * PER + j);
          s.hit[turn][r][1] = above;
          s.hit[turn][r][2] = h[j];
        }
        above += h[j];
      }
    }
  }
  look(total - before - mine, mine, h);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < NR; ++r) hit[r] = RankHit{s.hit[turn][r][0], s.hit[turn][r][1], s.hit[turn][r][2]};
}
template <int NR>
__device__ __forceinline__ void wide_find_rank(const uint32_t* s_hist, const uint32_t (&rank)[NR],
                                               WideScratch& s, int turn, RankHit (&hit)[NR]) {
  wide_find_rank<NR, kWideBins>(s_hist, rank, s, turn, hit, [](uint32_t, uint32_t, const auto&) {});
}

// Short list of keys in LDS (what one histogram bin holds): `rank` (1-based, from the top) by counting.
// The thread that owns an entry compares it with all of them; the one whose key it is leaves (key,
// keys above, equal keys) in out.  128 entries cost 32 LDS reads of two waves; with 1024 the one LDS
// of the workgroup was busy for 20 us.
constexpr int kWideList = 128;
__device__ __forceinline__ void wide_list_rank(const uint32_t* s_key, uint32_t cnt, uint32_t rank, uint32_t* out) {
  if (threadIdx.x >= cnt) return;
  const uint32_t me = s_key[threadIdx.x];
  uint32_t gt = 0, eq = 0;
  for (uint32_t j = 0; j < cnt; j += kVec) {
    const U4 o = *reinterpret_cast<const U4*>(s_key + j);
    const uint32_t left = cnt - j;
    gt += (o.x > me) + (left > 1 && o.y > me) + (left > 2 && o.z > me) + (left > 3 && o.w > me);
    eq += (o.x == me) + (left > 1 && o.y == me) + (left > 2 && o.z == me) + (left > 3 && o.w == me);
  }
  if (gt < rank && rank <= gt + eq) { out[0] = me; out[1] = gt; out[2] = eq; }   // equal keys write the same
}

// One LDS increment per participating lane; a wave whose lanes all hit one bin (a plateau of equal
// keys) adds once.  For loops of unbounded length only: the 16 to 20 keys per thread of the usual
// passes add plainly (one workgroup's instruction issue is the bound there -- 0.2 us for every
// instruction per key of 24 K keys -- and 64 lanes on one bin cost no more than this test).
__device__ __forceinline__ void wide_hist_add(uint32_t* s_hist, uint32_t bin, bool part) {
  const uint64_t act = ballot64(part);
  if (act == 0) return;
  const uint32_t lead = (uint32_t)__builtin_amdgcn_readlane((int)bin, __ffsll((unsigned long long)act) - 1);
  if (ballot64(part && bin != lead) == 0) {
    if (lane_id() == 0) atomicAdd(&s_hist[lead], (uint32_t)__popcll(act));
  } else if (part) {
    atomicAdd(&s_hist[bin], 1u);
  }
}

#endif  // __HIPCC__
}  // namespace sga
