// Exact k-th-largest select over 31-bit magnitude keys, templated on where
// the keys come from (a score array, raw key buffers, or a fused g+residual
// expression).  Non-negative fp32 values order like their integer patterns,
// so the k-th largest key is found by a three-level radix descent
// (12 + 12 + 7 bits) over LDS-privatised histograms, followed by an ordered
// per-chunk count so that ties at the threshold can be granted in ascending
// index order without any float compare ambiguity.
#pragma once
#include <type_traits>
#include "adam_math.hpp"
#include "sel_state.hpp"
#include "wide_scan.hpp"

namespace sga {

constexpr int kL0Bits = 12, kL1Bits = 12, kL2Bits = 7;
constexpr int kL0Shift = 19, kL1Shift = 7;
constexpr int kBinsBig = 4096, kBinsSmall = 128;
constexpr int kTileScanPer = 16;
constexpr int kTileScanSpan = kBlock * kTileScanPer;  // 4096 tiles / workgroup
constexpr int kMaxTileBlocks = 1024;                  // covers n < 2^32

struct SelWorkspace {
  SelState* st;        // main state (result, bracket)
  SelState* aux;       // aux[0]: state of the descent over dense records (single-sweep step)
  uint32_t* hist;      // 2 sets of 3 levels: [0,4096) [4096,8192) [8192,8320)
  uint32_t* tile_gt;   // n_tiles -> selected-count prefix
  uint32_t* tile_eq;   // n_tiles -> tie-count prefix
  uint32_t* blk_gt;    // kMaxTileBlocks
  uint32_t* blk_eq;    // kMaxTileBlocks
  int32_t* seg_dir;    // kSelDirEntries: tensor directory of segment-keyed sources (adam_math.hpp)
  int64_t n_tiles_cap;
  // sampled-bracket path (null / 0 when the workspace has no room for it)
  uint32_t* sample;    // keys of the coarse sample
  uint32_t* rel;       // kRelWords
  uint32_t* seg_cnt;   // kSegWaves (+1) counts -> offsets
  uint32_t* seg_idx;   // kSegWaves * seg_cap
  uint32_t* seg_key;
  uint32_t* cand_idx;  // dense candidates
  uint32_t* cand_key;
  uint32_t* pbits;     // 32 words per chunk: bit planes of "key above the bracket"
  // one-workgroup path (small_select.hpp): list of the bracket's keys, shares the memory of the
  // segments above
  uint32_t* small_idx;
  uint32_t* small_key;
  int64_t sample_cap;  // keys of the sample the bracket comes from
  int64_t seg_cap;     // per-wave candidate capacity
};

constexpr int kSegWaves = 8192;            // candidate segments the sweep's chunks hash to
constexpr int kSweepParts = 256;            // partial counters of the sweep's two totals
constexpr int64_t kFastMinN = 1 << 20;     // the sampled bracket of the large buckets begins here
constexpr int kSmallTiles = 8192;          // up to this many chunks a bucket takes small_select.hpp
constexpr int kSmallSegs = 16;             // list segments there (one per wave of its finishing workgroup)
constexpr int kSmallSegStride = 64;        // their counters lie 256 bytes apart (see small_geom)
// Histograms of keys relative to a bracket (large buckets): kRelCopies copies of kRelBins bins that the
// sweep's workgroups add to by turns (equal keys would otherwise queue on one word, 11 ns each), and
// one of kWideBins bins with kRelSpread spread counters for the sample.
constexpr int kRelBins = 1024, kRelCopies = 32, kRelSpread = 16;
constexpr int kRelSample = kRelBins * kRelCopies;
constexpr int kRelAbove = kRelSample + kWideBins;
constexpr int kRelWords = kRelAbove + kRelSpread * 64;
// Margin of a bracket that has a way back when it misses, in standard deviations of the sample rank.
constexpr double kBracketSigmas = 5.0;

// Sample: one quad of keys in 512 coordinates, 8 K to 16 K keys (or all).  A thousand more keys cost
// the picking workgroup 0.25 us and a thousand more list entries the finishing one 0.12: at 4 M
// coordinates and 1 % (35 K entries from 16 K keys) the two sum to a flat minimum near these sizes.
constexpr int64_t kSmallSampleMin = 2048, kSmallSampleMax = 4096;
__host__ __device__ static inline int64_t small_sample_vecs(int64_t n) {
  int64_t v = n / 512;
  if (v < kSmallSampleMin) v = kSmallSampleMin;
  if (v > kSmallSampleMax) v = kSmallSampleMax;
  return v < n / 4 ? v : n / 4;
}

static inline int64_t fast_sample_vecs(int64_t n) {
  int64_t v = n / 1024;
  if (v < 16384) v = 16384;
  if (v > (1 << 18)) v = 1 << 18;
  return v;
}
static inline int64_t fast_seg_cap(int64_t n) {
  int64_t c = n / 32 / kSegWaves;
  if (c < 64) c = 64;
  if (c > 8192) c = 8192;
  return c;
}

// Batched chain: every short kernel around a select takes up to kMaxJobs
// independent select problems in one launch (blockIdx.y = job), so that a
// caller with several buckets (or several re-selections of one replay step)
// pays the chain of dependent launches once instead of once per problem.
// The operands travel by value in the kernel arguments.
constexpr int kMaxJobs = 8;
struct ChainJob {
  SelState* st;
  SelState* aux;
  uint32_t* hist;
  uint32_t* tile_gt;
  uint32_t* tile_eq;
  uint32_t* blk_gt;
  uint32_t* blk_eq;
  uint32_t* sample;
  uint32_t* rel;
  uint32_t* seg_cnt;
  uint32_t* seg_idx;
  uint32_t* seg_key;
  uint32_t* cand_idx;
  uint32_t* cand_key;
  uint32_t* seg_fail;          // single-sweep step: per-segment first failed reservation
  uint32_t* small_idx;         // small_select.hpp: list of the bracket's keys
  uint32_t* small_key;
  const F4* seg_rec;           // single-sweep step: records beside the segments' keys
  F4* cand_rec;
  uint32_t* planes;            // where the settlement writes the selection (bit planes) ...
  uint8_t* mask;               // ... or mask bytes
  sga_select_result* result;
  int64_t n, n_tiles, n_sv, n_vec;
  uint32_t k, seg_cap, seed, ovf_cap;
  int tie_all, spec;
  int mask_only;               // no pack: a settled bracket needs no chunk scan
};
struct ChainJobs { ChainJob j[kMaxJobs]; };
template <class Src>
struct SrcPack { Src s[kMaxJobs]; };

// Workspace layout: [fixed: states | level histograms | tile-scan block sums]
// [tile_gt[nt] | tile_eq[nt]] [fast-path buffers sized from nt: sample keys,
// per-wave candidate segments, dense candidates, 128 B of bit planes per
// tile].  nt is derived from the byte size, so every entry point recovers
// the same carve from (ws, ws_bytes) alone.
constexpr int kHistEntries = 2 * kBinsBig + kBinsSmall;      // 8320
constexpr int kHistStride = kHistEntries + 64;               // per-state stride
constexpr int kSelDirEntries = 1 << 15;                        // n < 2^31 in blocks of 2^16
constexpr size_t kSelFixedBytes =
    3 * sizeof(SelState) + (size_t)kHistStride * 2 * 4 + (size_t)kMaxTileBlocks * 4 * 2 + (size_t)kSelDirEntries * 4;

// List entries of the small path: its kSmallSegs segments hold every coordinate of their
// workgroups, and the last one may fall a segment's share short of full.
static inline size_t small_list_entries(int64_t nt) {
  const int64_t t = nt < kSmallTiles + 8 ? nt : kSmallTiles + 8;
  return (size_t)(t + t / kSmallSegs + 4 * kChunksPerBlock) * kChunk;
}
// Bytes the candidate segments (four arrays) and the small path's list (two) share.  Above
// kSmallTiles the list's share stays what it was there, so that the layout grows with nt.
static inline size_t list_bytes_for_tiles(int64_t nt) {
  const size_t segs = nt * kChunk < kFastMinN ? 0 : (size_t)kSegWaves * fast_seg_cap(nt * kChunk) * 16;
  const size_t small = small_list_entries(nt) * 8;
  return segs > small ? segs : small;
}
static inline size_t fast_bytes_for_tiles(int64_t nt) {
  const int64_t n = nt * kChunk;
  const size_t always = (size_t)(kSegWaves + 64) * 4 + list_bytes_for_tiles(nt) + 256;
  return n < kFastMinN ? always : always + (size_t)kSmallSampleMax * 16 + (size_t)kRelWords * 4 + (size_t)nt * 128;
}

static inline size_t sel_ws_bytes(int64_t n) {
  const int64_t nt = cdiv64(n, kChunk) + 8;
  size_t b = kSelFixedBytes + (size_t)nt * 4 * 2 + fast_bytes_for_tiles(nt);
  return (b + 255) & ~(size_t)255;
}

static inline bool sel_ws_carve(void* ws, size_t bytes, int64_t n_tiles_needed,
                                SelWorkspace* out) {
  if (!ws || bytes < kSelFixedBytes || (reinterpret_cast<uintptr_t>(ws) & 15))
    return false;
  // largest nt whose full layout fits (layout size is monotone in nt)
  int64_t lo = 0, hi = (int64_t)((bytes - kSelFixedBytes) / 8);
  while (lo < hi) {
    const int64_t mid = lo + (hi - lo + 1) / 2;
    if (kSelFixedBytes + (size_t)mid * 8 + fast_bytes_for_tiles(mid) <= bytes) lo = mid;
    else hi = mid - 1;
  }
  const int64_t nt = lo;
  if (nt < n_tiles_needed) return false;
  char* p = reinterpret_cast<char*>(ws);
  out->st = reinterpret_cast<SelState*>(p);
  out->aux = out->st + 1;
  p += 3 * sizeof(SelState);
  out->hist = reinterpret_cast<uint32_t*>(p);
  p += (size_t)kHistStride * 2 * 4;
  out->blk_gt = reinterpret_cast<uint32_t*>(p);
  p += (size_t)kMaxTileBlocks * 4;
  out->blk_eq = reinterpret_cast<uint32_t*>(p);
  p += (size_t)kMaxTileBlocks * 4;
  out->seg_dir = reinterpret_cast<int32_t*>(p);
  p += (size_t)kSelDirEntries * 4;
  out->tile_gt = reinterpret_cast<uint32_t*>(p);
  p += (size_t)nt * 4;
  out->tile_eq = reinterpret_cast<uint32_t*>(p);
  p += (size_t)nt * 4;
  out->n_tiles_cap = nt;
  out->sample = out->rel = nullptr;
  out->seg_idx = out->seg_key = out->cand_idx = out->cand_key = nullptr;
  out->pbits = nullptr;
  out->sample_cap = 0;
  out->seg_cap = 0;
  p = reinterpret_cast<char*>((reinterpret_cast<uintptr_t>(p) + 255) & ~(uintptr_t)255);
  out->seg_cnt = reinterpret_cast<uint32_t*>(p);
  p += (size_t)(kSegWaves + 64) * 4;
  out->small_idx = reinterpret_cast<uint32_t*>(p);
  out->small_key = out->small_idx + small_list_entries(nt);
  if (nt * kChunk >= kFastMinN) {
    const int64_t n = nt * kChunk;
    char* q = p;
    out->seg_cap = fast_seg_cap(n);
    const size_t seg_bytes = (size_t)kSegWaves * out->seg_cap * 4;
    out->seg_idx = reinterpret_cast<uint32_t*>(q); q += seg_bytes;
    out->seg_key = reinterpret_cast<uint32_t*>(q); q += seg_bytes;
    out->cand_idx = reinterpret_cast<uint32_t*>(q); q += seg_bytes;
    out->cand_key = reinterpret_cast<uint32_t*>(q);
    p += list_bytes_for_tiles(nt);
    out->sample_cap = fast_sample_vecs(n) * 4;
    out->sample = reinterpret_cast<uint32_t*>(p);
    p += (size_t)kSmallSampleMax * 16;
    out->rel = reinterpret_cast<uint32_t*>(p);
    p += (size_t)kRelWords * 4;
    out->pbits = reinterpret_cast<uint32_t*>(p);
  }
  return true;
}

#ifdef __HIPCC__

// ------------------------------------------------------------ key sources
// A key source yields the 31-bit magnitude keys of 4 consecutive elements.
// load<FULL>: FULL promises i + 4 <= n and vector alignment (see ld_f32).
// The one-sweep select drives a source in three steps instead, so that the
// loads of kAhead slabs of a chunk are in flight before the first key is
// formed: chunk_begin (what is common to the chunk's 1024 elements, held on
// the scalar unit), fetch (loads only), keys (arithmetic only).
struct NoChunk {};
struct SrcF32 {                 // |x| of an fp32 score array
  const float* x;
  bool vec;
  uint32_t neg;                 // this lane has seen a value below zero (callers that promise
                                // non-negative scores are told, without a pass of their own)
  using Raw = F4;
  using Chunk = NoChunk;
  using Cols = NoCols;                                   // see k_sample_pick
  static constexpr bool kHyper = false, kReadAgain = false;
  static constexpr int kSweep = 2;                       // see chain_sweeps
  static constexpr int kAhead = kChunkIters;
  __device__ __forceinline__ Chunk chunk_begin(int64_t) { return Chunk{}; }
  __device__ __forceinline__ void chunk_hyper(int64_t) {}
  __device__ __forceinline__ void slab_hyper(int64_t) {}
  template <bool FULL, bool KEEP = false>
  __device__ __forceinline__ void fetch(const Chunk&, int64_t i, int64_t n, Raw& r) {
    r = ldraw_f32<FULL, KEEP>(x, i, n, vec);
  }
  template <bool FULL, class Now = NoCols>
  __device__ __forceinline__ void keys(const Chunk&, int64_t, int64_t, const Raw& r, uint32_t key[4],
                                       const Now& = Now()) {
    key[0] = abs_key(r.x); key[1] = abs_key(r.y); key[2] = abs_key(r.z); key[3] = abs_key(r.w);
    neg |= (uint32_t)((r.x < 0.0f) | (r.y < 0.0f) | (r.z < 0.0f) | (r.w < 0.0f));
  }
  template <bool FULL = false>
  __device__ __forceinline__ void load(int64_t i, int64_t n, uint32_t key[4]) {
    float v[4];
    ld_f32<FULL>(x, i, n, v, vec);
#pragma unroll
    for (int e = 0; e < 4; ++e) { key[e] = abs_key(v[e]); neg |= (uint32_t)(v[e] < 0.0f); }
  }
};
// What a key source knows about the sign of its inputs (only fp32 score arrays keep track).
template <class Src>
__device__ __forceinline__ uint32_t src_negative(const Src&) { return 0u; }
__device__ __forceinline__ uint32_t src_negative(const SrcF32& s) { return s.neg; }
// Signed scores (`update`) are the rule for some callers: with one OR per wave every wave of the
// sweep queues on this one word, 11 ns each (708 us for a 63 M-element sweep that takes 58 us).
// The flag only ever goes up, so whoever already sees it set leaves it alone; a stale zero costs
// one more OR.
__device__ __forceinline__ void raise_negative(SelState* st) {
  if (__hip_atomic_load(&st->negative, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u)
    atomicOr(&st->negative, 1u);
}
template <class Src>
__device__ __forceinline__ void note_negative(const Src& src, SelState* st) {
  if (ballot64(src_negative(src) != 0u) != 0ull && lane_id() == 0) raise_negative(st);
}

struct SrcU32 {                 // raw keys (sample / candidate buffers)
  const uint32_t* x;
  static constexpr bool vec = true;
  template <bool FULL = false>
  __device__ __forceinline__ void load(int64_t i, int64_t n, uint32_t key[4]) {
    if (FULL || i + 4 <= n) {
      U4 v = *reinterpret_cast<const U4*>(x + i);
      key[0] = v.x; key[1] = v.y; key[2] = v.z; key[3] = v.w;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) key[e] = (i + e < n) ? x[i + e] : 0u;
    }
  }
};

// ------------------------------------------------------------- LDS histogram
// One increment per participating lane; when many lanes of the wave hit the
// bin of the first participating lane (zero-heavy or plateau data) they are
// folded into a single add so same-address LDS atomics do not serialise.
__device__ __forceinline__ void lds_hist_add(uint32_t* s_h, uint32_t bin, bool part) {
  uint64_t act = ballot64(part);
  if (act == 0) return;
  const int leader = __ffsll((unsigned long long)act) - 1;
  const uint32_t lead_bin = __shfl(bin, leader, kWave);
  const uint64_t same = ballot64(part && bin == lead_bin);
  const int ns = __popcll(same);
  if (ns >= 8) {
    if (lane_id() == leader) atomicAdd(&s_h[lead_bin], (uint32_t)ns);
    part = part && bin != lead_bin;
  }
  if (part) atomicAdd(&s_h[bin], 1u);
}

template <int LEVEL>
__device__ __forceinline__ void level_bin(uint32_t key, uint32_t prefix, bool valid,
                                          uint32_t& bin, bool& part) {
  if (LEVEL == 0) { bin = key >> kL0Shift; part = valid; }
  else if (LEVEL == 1) { bin = (key >> kL1Shift) & (kBinsBig - 1); part = valid && (key >> kL0Shift) == prefix; }
  else { bin = key & (kBinsSmall - 1); part = valid && (key >> kL1Shift) == prefix; }
}

// State that other workgroups of the same launch write or read: past the caches of this CU and XCD.
__device__ __forceinline__ uint32_t ld_agent(const uint32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(uint32_t* p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long ld_agent64(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent64(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Every such store and atomic of the workgroup has landed when this returns.
__device__ __forceinline__ void wait_landed() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

// One level of the descent for one state, run by a single workgroup: find
// the bin where the descending cumulative count crosses the remaining rank.
template <int LEVEL>
__device__ __forceinline__ void level_scan_body(SelState* __restrict__ st,
                                                const uint32_t* __restrict__ hist,
                                                uint32_t* s_suf /* kBlock + 1 */) {
  constexpr int NB = LEVEL == 2 ? kBinsSmall : kBinsBig;
  constexpr int PER = NB >= kBlock ? NB / kBlock : 1;
  constexpr int BITS = LEVEL == 2 ? kL2Bits : 12;
  const int t = threadIdx.x;
  // read the incoming rank before any barrier: the one thread that descends
  // overwrites st->krem after the barriers below
  const uint32_t krem = (LEVEL == 0) ? st->k : ld_agent(&st->krem);
  const uint32_t pre_in = (LEVEL == 0) ? 0u : ld_agent(&st->prefix);
  uint32_t loc[PER];
  uint32_t mine = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int b = t * PER + j;
    loc[j] = (b < NB) ? __atomic_load_n(&hist[b], __ATOMIC_RELAXED) : 0u;
    mine += loc[j];
  }
  __syncthreads();
  s_suf[t] = mine;                       // suffix sums over threads
  if (t == 0) s_suf[kBlock] = 0u;
  __syncthreads();
  for (int o = 1; o < kBlock; o <<= 1) {
    uint32_t add = (t + o < kBlock) ? s_suf[t + o] : 0u;
    __syncthreads();
    s_suf[t] += add;
    __syncthreads();
  }
  const uint32_t total = s_suf[0];
  if (LEVEL == 0 && t == 0) {
    st->total = total;
    if (krem < 1 || krem > total) st->status = 1;
  }
  // exponent 255 (Inf / NaN) is bins 0xFF0..0xFFF: exactly the last thread's bins
  static_assert(kBinsBig / kBlock == 16 && (kBlock - 1) * 16 == 0xFF0, "non-finite bins = last thread");
  if (LEVEL == 0 && t == kBlock - 1) st->nonfinite = mine;
  const uint32_t above_me = s_suf[t + 1];
  if (krem >= 1 && above_me < krem && krem <= above_me + mine) {
    uint32_t above = above_me;
#pragma unroll
    for (int j = PER - 1; j >= 0; --j) {
      const int b = t * PER + j;
      if (b < NB) {
        if (above < krem && krem <= above + loc[j]) {
          const uint32_t np = (pre_in << BITS) | (uint32_t)b;
          st->prefix = np;
          st->krem = krem - above;
          if (LEVEL == 2) {
            st->thresh_bits = np;
            st->need = krem - above;
            st->n_eq = loc[j];
            st->n_gt = st->k - (krem - above);
          }
        }
        above += loc[j];
      }
    }
  }
  __syncthreads();
}

template <int LEVEL>
__device__ __forceinline__ uint32_t* level_hist_of(uint32_t* hist_set) {
  return hist_set + (LEVEL == 0 ? 0 : LEVEL == 1 ? kBinsBig : 2 * kBinsBig);
}

// Histogram of one radix level, by workgroup blk of n_blk: LDS bins, flushed to global ones.
template <class Src, int LEVEL>
__device__ __forceinline__ void level_hist_body(Src& src, int64_t n, uint32_t prefix,
                                                uint32_t* __restrict__ gh, uint32_t* s_h /* kBinsBig */,
                                                uint32_t blk, uint32_t n_blk) {
  constexpr int NB = LEVEL == 2 ? kBinsSmall : kBinsBig;
  for (int b = threadIdx.x; b < NB; b += kBlock) s_h[b] = 0u;
  __syncthreads();
  // Raw key buffers (dense records) are short and sit in L2: what their passes cost is load
  // latency, so each lane keeps kQuads 16-byte loads in flight per trip; the passes over the data
  // itself run on a small grid and need them too.
  constexpr int kQuads = 4;
  constexpr int64_t kSlabKeys = (int64_t)kBlock * kVec;
  const int64_t stride = (int64_t)n_blk * kSlabKeys * kQuads;
  // uniform trip count so the wave-level ballots inside lds_hist_add are safe
  const int64_t first = (int64_t)blk * kSlabKeys * kQuads;
  for (int64_t base = first; base < n; base += stride) {
    uint32_t key[kQuads][4];
    bool full[kQuads];
#pragma unroll
    for (int u = 0; u < kQuads; ++u) {
      const int64_t bu = base + u * kSlabKeys;
      const int64_t i = bu + (int64_t)threadIdx.x * kVec;
      key[u][0] = key[u][1] = key[u][2] = key[u][3] = 0u;
      full[u] = src.vec && bu + kSlabKeys <= n;   // whole workgroup span in range
      if (full[u]) src.template load<true>(i, n, key[u]);
      else if (i < n) src.template load<false>(i, n, key[u]);
    }
#pragma unroll
    for (int u = 0; u < kQuads; ++u) {
      const int64_t i = base + u * kSlabKeys + (int64_t)threadIdx.x * kVec;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t bin; bool part;
        level_bin<LEVEL>(key[u][e], prefix, full[u] || i + e < n, bin, part);
        // Raw key buffers are at most a few million keys for 64 workgroups of one wave per
        // SIMD: what a pass costs there is the latency of each key's chain, and the folding of
        // equal bins (two ballots, a cross-lane read and two scalar branches per key) is most of
        // it.  A plain LDS atomic per lane is shorter; on a plateau (every lane on one bin) it
        // serialises 64-fold, which for these few keys is a couple of microseconds.
        if (std::is_same<Src, SrcU32>::value) {
          if (part) atomicAdd(&s_h[bin], 1u);
        } else {
          lds_hist_add(s_h, bin, part);
        }
      }
    }
  }
  __syncthreads();
  for (int b = threadIdx.x; b < NB; b += kBlock) {
    const uint32_t c = s_h[b];
    if (c) atomicAdd(&gh[b], c);
  }
}
// True in the last of a level's n_blk workgroups.  The bins are device-scope atomics and are read by
// atomic loads (level_scan_body): waiting for one's own is enough, no fence.
__device__ __forceinline__ bool level_last(uint32_t* done, uint32_t n_blk, uint32_t* s_last) {
  wait_landed();
  if (threadIdx.x == 0) *s_last = atomicAdd(done, 1u) == n_blk - 1 ? 1u : 0u;
  __syncthreads();
  return *s_last != 0;
}
// Histogram only: several views of a staged select feed one level before its scan.
template <class Src, int LEVEL>
__global__ __launch_bounds__(kBlock) void k_level_hist(SrcPack<Src> srcs, ChainJobs jobs) {
  __shared__ uint32_t s_h[kBinsBig];
  const ChainJob& J = jobs.j[blockIdx.y];
  if (J.st->skip) return;
  Src src = srcs.s[blockIdx.y];
  level_hist_body<Src, LEVEL>(src, J.n, J.st->prefix, level_hist_of<LEVEL>(J.hist), s_h, blockIdx.x, gridDim.x);
}
// over the dense candidate keys of the job (the single-sweep step's records; their count lives on the
// device, state aux[0]).  The last workgroup to finish also runs the level's scan.
template <int LEVEL>
__global__ __launch_bounds__(kBlock) void k_level_hist_raw(ChainJobs jobs) {
  __shared__ uint32_t s_h[kBinsBig], s_suf[kBlock + 1], s_last;
  const ChainJob& J = jobs.j[blockIdx.y];
  SelState* st = J.aux;
  if (st->skip) return;
  const int64_t cap = (int64_t)kSegWaves * J.seg_cap;
  const int64_t n = J.st->cand_count < cap ? J.st->cand_count : cap;
  SrcU32 src{J.cand_key};
  uint32_t* gh = level_hist_of<LEVEL>(J.hist);
  level_hist_body<SrcU32, LEVEL>(src, n, st->prefix, gh, s_h, blockIdx.x, gridDim.x);
  if (!level_last(&st->done[LEVEL], gridDim.x, &s_last)) return;
  level_scan_body<LEVEL>(st, gh, s_suf);
}

// Stand-alone scan (used when one level's histogram is built by several
// launches, one per view).
template <int LEVEL>
__global__ __launch_bounds__(kBlock) void k_level_scan(ChainJobs jobs) {
  __shared__ uint32_t s_suf[kBlock + 1];
  const ChainJob& J = jobs.j[blockIdx.y];
  if (J.st->skip) return;
  level_scan_body<LEVEL>(J.st, level_hist_of<LEVEL>(J.hist), s_suf);
}

// Per-chunk (1024 elements, one wave) counts of keys above / equal to the
// threshold, by wave `wave` of `wstride`.  ROLL: a slab at a time, for kernels with few registers to spare.
template <class Src, bool ROLL = false>
__device__ __forceinline__ void tile_count_body(Src& src, const ChainJob& J, uint32_t T, int64_t tile_base,
                                                int64_t wave, int64_t wstride) {
  const int64_t n = J.n;
  uint32_t* tile_gt = J.tile_gt;
  uint32_t* tile_eq = J.tile_eq;
  const int64_t n_chunks = cdiv64(n, kChunk);
  for (int64_t c = wave; c < n_chunks; c += wstride) {
    uint32_t cg = 0, ce = 0;
    const bool full = src.vec && (c + 1) * kChunk <= n;
    if (!ROLL && full) {
      uint32_t key[kChunkIters][4];
#pragma unroll
      for (int it = 0; it < kChunkIters; ++it)
        src.template load<true>(c * kChunk + it * (kWave * kVec) + lane_id() * kVec, n, key[it]);
#pragma unroll
      for (int it = 0; it < kChunkIters; ++it)
#pragma unroll
        for (int e = 0; e < 4; ++e) { cg += key[it][e] > T; ce += key[it][e] == T; }
    } else {
      constexpr int kUnroll = ROLL ? 1 : kChunkIters;
#pragma unroll kUnroll
      for (int it = 0; it < kChunkIters; ++it) {
        const int64_t i = c * kChunk + it * (kWave * kVec) + lane_id() * kVec;
        uint32_t key[4] = {0, 0, 0, 0};
        if (ROLL && full) src.template load<true>(i, n, key);
        else if (i < n) src.template load<false>(i, n, key);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool valid = i + e < n;
          cg += (valid && key[e] > T);
          ce += (valid && key[e] == T);
        }
      }
    }
    cg = wave_sum(cg);
    ce = wave_sum(ce);
    if (lane_id() == 0) {
      st_agent(&tile_gt[tile_base + c], cg);
      st_agent(&tile_eq[tile_base + c], ce);
    }
  }
  note_negative(src, J.st);
}
template <class Src>
__global__ __launch_bounds__(kBlock) void k_tile_count(SrcPack<Src> srcs, ChainJobs jobs, int64_t tile_base) {
  const ChainJob& J = jobs.j[blockIdx.y];
  if (J.st->skip) return;
  Src src = srcs.s[blockIdx.y];
  tile_count_body(src, J, J.st->thresh_bits, tile_base, (int64_t)blockIdx.x * kChunksPerBlock + wave_id(),
                  (int64_t)gridDim.x * kChunksPerBlock);
}

// Tile scan of a staged select, kernel 1: per-workgroup totals of (gt, eq).
static __global__ __launch_bounds__(kBlock) void k_tile_sums(ChainJobs jobs) {
  __shared__ uint32_t s_g[kChunksPerBlock], s_e[kChunksPerBlock];
  const ChainJob& J = jobs.j[blockIdx.y];
  const int64_t n_tiles = J.n_tiles;
  if ((int64_t)blockIdx.x * kTileScanSpan >= n_tiles) return;     // a job with fewer tiles
  const uint32_t* __restrict__ tile_gt = J.tile_gt;
  const uint32_t* __restrict__ tile_eq = J.tile_eq;
  uint32_t* __restrict__ blk_gt = J.blk_gt;
  uint32_t* __restrict__ blk_eq = J.blk_eq;
  const int64_t base = (int64_t)blockIdx.x * kTileScanSpan + (int64_t)threadIdx.x * kTileScanPer;
  uint32_t g = 0, e = 0;
#pragma unroll
  for (int j = 0; j < kTileScanPer; ++j)
    if (base + j < n_tiles) { g += tile_gt[base + j]; e += tile_eq[base + j]; }
  g = wave_sum(g);
  e = wave_sum(e);
  if (lane_id() == 0) { s_g[wave_id()] = g; s_e[wave_id()] = e; }
  __syncthreads();
  if (threadIdx.x == 0) {
    blk_gt[blockIdx.x] = s_g[0] + s_g[1] + s_g[2] + s_g[3];
    blk_eq[blockIdx.x] = s_e[0] + s_e[1] + s_e[2] + s_e[3];
  }
}

__device__ __forceinline__ uint32_t ties_taken(uint32_t need, uint32_t eq_before, uint32_t eq_here) {
  if (need <= eq_before) return 0u;
  const uint32_t left = need - eq_before;
  return left < eq_here ? left : eq_here;
}

// Block-wide exclusive scan of one uint32 per thread (kBlock threads).
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* s_w4, uint32_t& block_total) {
  const uint32_t incl = wave_incl_scan(v);
  __syncthreads();
  if (lane_id() == kWave - 1) s_w4[wave_id()] = incl;
  __syncthreads();
  uint32_t pre = 0;
  for (int w = 0; w < wave_id(); ++w) pre += s_w4[w];
  block_total = s_w4[0] + s_w4[1] + s_w4[2] + s_w4[3];
  return pre + incl - v;
}

// Tile scan, kernel 2: tile_eq[i] <- ties before tile i; tile_gt[i] <- selected
// coordinates before tile i (ties granted in ascending order until `need`
// is used up; all of them when tie_all).
static __global__ __launch_bounds__(kBlock) void k_tile_apply(ChainJobs jobs) {
  __shared__ uint32_t s_w4[kChunksPerBlock];
  const ChainJob& J = jobs.j[blockIdx.y];
  const int64_t n_tiles = J.n_tiles;
  const int n_blocks = (int)cdiv64(n_tiles, kTileScanSpan);
  if ((int)blockIdx.x >= n_blocks) return;                        // a job with fewer tiles
  uint32_t* __restrict__ tile_gt = J.tile_gt;
  uint32_t* __restrict__ tile_eq = J.tile_eq;
  const uint32_t* __restrict__ blk_gt = J.blk_gt;
  const uint32_t* __restrict__ blk_eq = J.blk_eq;
  const int tie_all = J.tie_all;
  SelState* __restrict__ st = J.st;
  const uint32_t need = tie_all ? 0xFFFFFFFFu : st->need;
  // prefixes of the workgroups before this one (n_blocks <= 1024 -> 4 each)
  uint32_t be[4], bg[4];
  uint32_t mine_e = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int b = threadIdx.x * 4 + j;
    be[j] = (b < n_blocks) ? blk_eq[b] : 0u;
    bg[j] = (b < n_blocks) ? blk_gt[b] : 0u;
    mine_e += be[j];
  }
  uint32_t tot_e;
  uint32_t e_run = block_excl_scan(mine_e, s_w4, tot_e);
  uint32_t sel_before = 0, eq_before = 0;   // contributions of blocks < blockIdx.x
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int b = threadIdx.x * 4 + j;
    if (b < (int)blockIdx.x) {
      sel_before += bg[j] + ties_taken(need, e_run, be[j]);
      eq_before += be[j];
    }
    e_run += be[j];
  }
  uint32_t dummy;
  __syncthreads();
  // reduce sel_before / eq_before across the workgroup via scans' totals
  block_excl_scan(sel_before, s_w4, dummy);
  const uint32_t S0 = dummy;
  __syncthreads();
  block_excl_scan(eq_before, s_w4, dummy);
  const uint32_t E0 = dummy;
  __syncthreads();

  const int64_t base = (int64_t)blockIdx.x * kTileScanSpan + (int64_t)threadIdx.x * kTileScanPer;
  uint32_t g[kTileScanPer], e[kTileScanPer];
  uint32_t my_e = 0;
#pragma unroll
  for (int j = 0; j < kTileScanPer; ++j) {
    const bool ok = base + j < n_tiles;
    g[j] = ok ? tile_gt[base + j] : 0u;
    e[j] = ok ? tile_eq[base + j] : 0u;
    my_e += e[j];
  }
  uint32_t blk_tot_e;
  uint32_t er = E0 + block_excl_scan(my_e, s_w4, blk_tot_e);
  uint32_t my_s = 0;
  uint32_t ebase[kTileScanPer], scount[kTileScanPer];
#pragma unroll
  for (int j = 0; j < kTileScanPer; ++j) {
    ebase[j] = er;
    scount[j] = g[j] + ties_taken(need, er, e[j]);
    my_s += scount[j];
    er += e[j];
  }
  __syncthreads();
  uint32_t blk_tot_s;
  uint32_t sr = S0 + block_excl_scan(my_s, s_w4, blk_tot_s);
#pragma unroll
  for (int j = 0; j < kTileScanPer; ++j) {
    if (base + j < n_tiles) {
      tile_gt[base + j] = sr;
      tile_eq[base + j] = ebase[j];
    }
    sr += scount[j];
  }
  if ((int)blockIdx.x == n_blocks - 1 && threadIdx.x == 0)
    st->n_selected = S0 + blk_tot_s;
}

// Ordered flags for one 256-element slab of a wave's chunk: `sel[e]` says
// whether element e of this lane is selected; `pos` is the number of selected
// elements before this lane's first element (within the whole array).
struct ChunkCursor {
  uint32_t sel_run;   // selected before the current slab
  uint32_t eq_run;    // ties before the current slab
};

// Everything a slab's order needs is on the scalar unit: four ballots each for the ties and the selected
// (a cross-lane scan is six dependent LDS permutes, 0.3 us a slab where nothing hides them).
__device__ __forceinline__ void slab_select(const uint32_t key[4], const bool valid[4],
                                            uint32_t T, uint32_t need, ChunkCursor& cur,
                                            bool sel[4], uint32_t& pos) {
  uint64_t eq[4], any_eq = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    eq[e] = ballot64(valid[e] && key[e] == T);
    any_eq |= eq[e];
    sel[e] = valid[e] && key[e] > T;
  }
  if (any_eq) {                                  // scalar branch
    uint32_t rank = cur.eq_run + lanes_below(eq[0]) + lanes_below(eq[1]) + lanes_below(eq[2]) + lanes_below(eq[3]);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (valid[e] && key[e] == T) sel[e] = rank++ < need;
    cur.eq_run += (uint32_t)(__popcll(eq[0]) + __popcll(eq[1]) + __popcll(eq[2]) + __popcll(eq[3]));
  }
  uint32_t below = 0, total = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint64_t m = ballot64(sel[e]);
    below += lanes_below(m);
    total += (uint32_t)__popcll(m);
  }
  pos = cur.sel_run + below;
  cur.sel_run += total;
}

template <class Src>
__device__ __forceinline__ void write_mask_body(Src& src, const ChainJob& J, uint32_t T, uint32_t need,
                                                int64_t tile_base, uint8_t* __restrict__ mask, uint32_t blk,
                                                uint32_t n_blk) {
  const bool mvec = quads_ok(mask, 1);
  const int64_t n = J.n;
  const int64_t n_chunks = cdiv64(n, kChunk);
  const int64_t wstride = (int64_t)n_blk * kChunksPerBlock;
  for (int64_t c = (int64_t)blk * kChunksPerBlock + wave_id(); c < n_chunks;
       c += wstride) {
    ChunkCursor cur;
    cur.sel_run = (uint32_t)uniform_i32((int)ld_agent(&J.tile_gt[tile_base + c]));
    cur.eq_run = (uint32_t)uniform_i32((int)ld_agent(&J.tile_eq[tile_base + c]));
    const bool full = src.vec && mvec && (c + 1) * kChunk <= n;
    uint32_t key[kChunkIters][4];
#pragma unroll
    for (int it = 0; it < kChunkIters; ++it) {
      const int64_t i = c * kChunk + it * (kWave * kVec) + lane_id() * kVec;
#pragma unroll
      for (int e = 0; e < 4; ++e) key[it][e] = 0u;
      if (full) src.template load<true>(i, n, key[it]);
      else if (i < n) src.template load<false>(i, n, key[it]);
    }
#pragma unroll
    for (int it = 0; it < kChunkIters; ++it) {
      const int64_t i = c * kChunk + it * (kWave * kVec) + lane_id() * kVec;
      bool valid[4], sel[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) valid[e] = full || i + e < n;
      uint32_t pos;
      slab_select(key[it], valid, T, need, cur, sel, pos);
      uint32_t mk[4] = {sel[0], sel[1], sel[2], sel[3]};
      if (full) st_u8<true>(mask, i, n, mk, true);
      else if (i < n) store4_u8(mask, i, n, mk, mvec);
    }
  }
}

template <class Src>
__global__ __launch_bounds__(kBlock) void k_write_mask(SrcPack<Src> srcs, ChainJobs jobs, int64_t tile_base) {
  const ChainJob& J = jobs.j[blockIdx.y];
  Src src = srcs.s[blockIdx.y];
  write_mask_body(src, J, J.st->thresh_bits, J.tie_all ? 0xFFFFFFFFu : J.st->need, tile_base, J.mask, blockIdx.x,
                  gridDim.x);
}

__device__ __forceinline__ void write_result(const ChainJob& J) {
  const SelState* st = J.st;
  sga_select_result* out = J.result;
  if (!out) return;
  st_host(&out->thresh_bits, ld_agent(&st->thresh_bits));
  st_host(&out->need, ld_agent(&st->need));
  st_host(&out->n_gt, ld_agent(&st->n_gt));
  st_host(&out->n_eq, ld_agent(&st->n_eq));
  st_host(&out->n_selected, ld_agent(&st->n_selected));
  st_host(&out->nonfinite, ld_agent(&st->nonfinite));
  st_host(&out->status, ld_agent(&st->status));
  st_host(&out->path, st->path | (ld_agent(&st->negative) ? 0x100u : 0u) | (st->redone ? 0x200u : 0u));
}
static __global__ void k_sel_result(ChainJobs jobs) { write_result(jobs.j[blockIdx.y]); }

// -------------------------------------------------------------- host drivers
// Grid unit of the histogram passes over dense records (the single-sweep step launches three of them;
// the count of the records lives on the device).  What a workgroup costs there is fixed: zeroing and
// flushing its LDS bins, and its ticket.
constexpr unsigned kRawKeyBlocks = 64;
static inline dim3 hist_grid(int64_t n) {
  return dim3(stream_grid(n, (int64_t)kBlock * kVec * 4, 256 * 8));
}

// Host side of a batched chain: up to kMaxJobs select problems that go through every short
// kernel together.  A single select is a batch of one.
struct SelBatch {
  int count = 0;
  ChainJobs jobs;
  SelWorkspace w[kMaxJobs];
  int64_t max_n = 0, max_tiles = 0, max_nsv = 0;
  // true when the job takes the one-workgroup path of small_select.hpp
  static bool small_ok(int64_t n) { return cdiv64(n, kChunk) <= kSmallTiles; }
  // true when the job takes the sampled-bracket path (all jobs of one batch must agree)
  static bool fast_ok(const SelWorkspace& ws, int64_t n) {
    return n >= kFastMinN && ws.sample != nullptr && n < (1ll << 32);
  }
  ChainJob& add(const SelWorkspace& ws, int64_t n, int64_t k, int tie_all) {
    ChainJob& J = jobs.j[count];
    w[count++] = ws;
    J = ChainJob{};
    J.st = ws.st; J.aux = ws.aux; J.hist = ws.hist;
    J.tile_gt = ws.tile_gt; J.tile_eq = ws.tile_eq; J.blk_gt = ws.blk_gt; J.blk_eq = ws.blk_eq;
    J.sample = ws.sample; J.rel = ws.rel; J.seg_cnt = ws.seg_cnt; J.seg_idx = ws.seg_idx; J.seg_key = ws.seg_key;
    J.cand_idx = ws.cand_idx; J.cand_key = ws.cand_key;
    J.small_idx = ws.small_idx; J.small_key = ws.small_key;
    J.n = n; J.n_tiles = cdiv64(n, kChunk);
    J.n_vec = n / 4;
    J.n_sv = ws.sample_cap / 4 < J.n_vec ? ws.sample_cap / 4 : J.n_vec;
    J.k = (uint32_t)k; J.seg_cap = (uint32_t)ws.seg_cap; J.tie_all = tie_all;
    if (n > max_n) max_n = n;
    if (J.n_tiles > max_tiles) max_tiles = J.n_tiles;
    if (J.n_sv > max_nsv) max_nsv = J.n_sv;
    return J;
  }
  dim3 grid(unsigned gx) const { return dim3(gx, (unsigned)count); }
};

// histogram of one radix level over the data, for every job of the batch (staged selects)
template <class Src>
static inline void launch_level_data(const SrcPack<Src>& srcs, const SelBatch& B, int level,
                                     hipStream_t s) {
  const dim3 grid = B.grid(hist_grid(B.max_n).x), block(kBlock);
  if (level == 0) hipLaunchKernelGGL((k_level_hist<Src, 0>), grid, block, 0, s, srcs, B.jobs);
  else if (level == 1) hipLaunchKernelGGL((k_level_hist<Src, 1>), grid, block, 0, s, srcs, B.jobs);
  else hipLaunchKernelGGL((k_level_hist<Src, 2>), grid, block, 0, s, srcs, B.jobs);
}
// the same over the jobs' dense candidate keys
static inline void launch_level_raw(const SelBatch& B, int level, hipStream_t s, unsigned blocks) {
  const dim3 grid = B.grid(blocks), block(kBlock);
  if (level == 0) hipLaunchKernelGGL((k_level_hist_raw<0>), grid, block, 0, s, B.jobs);
  else if (level == 1) hipLaunchKernelGGL((k_level_hist_raw<1>), grid, block, 0, s, B.jobs);
  else hipLaunchKernelGGL((k_level_hist_raw<2>), grid, block, 0, s, B.jobs);
}
static inline void launch_level_scan(int level, const SelBatch& B, hipStream_t s) {
  if (level == 0) hipLaunchKernelGGL((k_level_scan<0>), B.grid(1), dim3(kBlock), 0, s, B.jobs);
  else if (level == 1) hipLaunchKernelGGL((k_level_scan<1>), B.grid(1), dim3(kBlock), 0, s, B.jobs);
  else hipLaunchKernelGGL((k_level_scan<2>), B.grid(1), dim3(kBlock), 0, s, B.jobs);
}

template <class Src>
static inline void launch_tile_count(const SrcPack<Src>& srcs, const SelBatch& B, int64_t tile_base,
                                     hipStream_t s) {
  hipLaunchKernelGGL((k_tile_count<Src>), B.grid(stream_grid(B.max_tiles, kChunksPerBlock)),
                     dim3(kBlock), 0, s, srcs, B.jobs, tile_base);
}

static inline void launch_tile_scan(const SelBatch& B, hipStream_t s) {
  const unsigned nb = (unsigned)cdiv64(B.max_tiles, kTileScanSpan);
  hipLaunchKernelGGL(k_tile_sums, B.grid(nb), dim3(kBlock), 0, s, B.jobs);
  hipLaunchKernelGGL(k_tile_apply, B.grid(nb), dim3(kBlock), 0, s, B.jobs);
}

static inline void launch_result(const SelBatch& B, hipStream_t s) {
  hipLaunchKernelGGL(k_sel_result, B.grid(1), dim3(1), 0, s, B.jobs);
}

// ===================================================== sampled-bracket path
// The k-th largest key is bracketed from a small deterministic sample, so
// the full data needs ONE sweep instead of four: that sweep counts, per
// chunk, the keys above the bracket and collects the few keys inside it;
// the exact threshold is then selected among those candidates only.  The
// result is exact for any sample; if the bracket misses the k-th key (or the
// candidate buffers overflow, e.g. on tie-heavy data) a flag routes the work
// to the radix passes, all on the device.

__device__ __forceinline__ uint32_t mix32(uint32_t x) {
  x ^= x >> 16; x *= 0x7FEB352Du; x ^= x >> 15; x *= 0x846CA68Bu; x ^= x >> 16;
  return x;
}

// Quad j of a sample: one 4-element vector per window, at a hashed offset; the n_sv windows tile ALL
// n_vec vectors (window j = [j n_vec / n_sv, (j + 1) n_vec / n_sv)): a tail that no window covered
// would bias the sample whenever the last tensors score differently from the rest.  `seed` moves the
// offsets (0: the fixed pattern); the select is exact for any of them.
__device__ __forceinline__ int64_t quad_of_window(int64_t j, int64_t n_vec, int64_t n_sv, uint32_t seed) {
  const int64_t w0 = j * n_vec / n_sv, w1 = (j + 1) * n_vec / n_sv;
  return w0 + (int64_t)(mix32((uint32_t)j + seed * 0x9E3779B9u) % (uint32_t)(w1 - w0));
}

// Shift that maps the offsets of [lo, hi) onto at most `bins` (a power of two) bins.
__device__ __forceinline__ int rel_shift(uint32_t lo, uint32_t hi, int bins) {
  const int w = 32 - __clz((int)(hi - 1u - lo)), b = 31 - __clz(bins);     // hi - lo == 1: w = 0
  return w > b ? w - b : 0;
}

// What the kernels of a large bucket's select count in.
__device__ __forceinline__ void clear_large(const ChainJob& J, int t0, int step, bool fast) {
  for (int i = t0; i < kHistStride * 2; i += step) J.hist[i] = 0u;
  if (!fast) return;
  for (int i = t0; i <= kSegWaves + 1; i += step) J.seg_cnt[i] = 0u;     // + overflow count
  for (int i = t0; i < kSweepParts; i += step) { J.blk_gt[i] = 0u; J.blk_eq[i] = 0u; }
  for (int i = t0; i < kRelWords; i += step) J.rel[i] = 0u;
  if (J.seg_fail)
    for (int i = t0; i < kSegWaves; i += step) J.seg_fail[i] = 0u;
}
// The directory of a job's segment table (dirs.j[job].dir null: none wanted).
__device__ __forceinline__ void seg_dirs(const SegDirJobs& dirs, int job, int t0, int step) {
  const auto& D = dirs.j[job];
  if (!D.dir) return;
  const int nb = (int)((D.n + (1ll << kSegDirLog) - 1) >> kSegDirLog);
  for (int b = t0; b < nb; b += step) D.dir[b] = seg_dir_entry(D.segs, D.n_segs, b);
}

// ... and what a select's first kernel carries for the tables' changing columns.
template <class Cols>
__device__ __forceinline__ void keep_tables(const SegDirJobs& dirs, const Cols& cols, int t0, int step) {
  seg_dirs(dirs, blockIdx.y, t0, step);
  if constexpr (std::is_same<Cols, NowCols>::value)
    now_cols_write(cols, blockIdx.y, const_cast<sga_segment*>(dirs.j[blockIdx.y].segs), t0, step);
}
// Small buckets: the bracket on its way from the pick to the sweep, a copy beside each segment counter (on a line of
// its own), either end with the launch's number above it.
__device__ __forceinline__ unsigned long long* small_bracket_copy(const ChainJob& J, int c) {
  return reinterpret_cast<unsigned long long*>(J.seg_cnt + c * kSmallSegStride + kSmallSegStride / 2);
}

// First kernel of a select of the large buckets that goes by radix passes alone.
static __global__ __launch_bounds__(kBlock) void k_chain_begin(ChainJobs jobs, SegDirJobs dirs) {
  const ChainJob& J = jobs.j[blockIdx.y];
  const int t0 = blockIdx.x * kBlock + threadIdx.x, step = gridDim.x * kBlock;
  clear_large(J, t0, step, false);
  seg_dirs(dirs, blockIdx.y, t0, step);
  if (t0 != 0) return;
  SelState z = {};
  z.k = J.k;
  *J.st = z;
}

constexpr int kSmallPick = (int)(kSmallSampleMax / kWide);   // quads per thread of the picking workgroup

// A key source that looks tensors up: without the directory (it is being built while the sample is
// taken) the lookup bisects the table.
template <class S>
__device__ __forceinline__ auto drop_dir(S& s, int) -> decltype(s.sc.dir, void()) { s.sc.dir = nullptr; }
template <class S>
__device__ __forceinline__ void drop_dir(S&, long) {}

// Ranks in a sample of ns keys (1-based from the top) between which the k-th of n lies.
struct RankEnds { double hi, lo; };
__device__ __forceinline__ RankEnds bracket_ranks(double k, double n, double ns, double sigmas) {
  const double frac = k / n, r = frac * ns;
  const double d = sigmas * sqrt(r * (1.0 - frac) + 1.0) + 8.0;
  return RankEnds{floor(r - d), ceil(r + d)};
}

// First kernel of a select by a sampled bracket: the sample, the two ends of the bracket from it, the state.
//
// kSampleGroups workgroups take the sample (one quad per window at a hashed offset, see quad_of_window): one
// alone would be bound by its CU's translation misses (4096 quads of two arrays: 25 us).  A workgroup that has
// left its keys leaves the launch's number beside them and looks at the others': whoever sees all of them picks.
// Nobody waits for anybody, and two that see all numbers at once do the same and write the same.  (Numbers of an
// earlier launch are gone: the pick writes the whole state.  Memory that happens to hold the number spoils the
// sample and no more, see sampled_key.)  As two launches (three with the clearing kernel of the large buckets)
// before -> after, with the bin edges below, selects in a row at 1 %, us: 261 K 28.1 -> 26.1, 3 M 41.0 -> 36.3, 20 M
// 60.4 -> 51.8, 100 M 122 -> 114.
//
// The pick: one LDS histogram of the top 13 bits of all keys.  The ends of the bins that the two ends of the
// bracket fall into will do, rounded outwards, as long as that takes in no more than a quarter of the bracket's
// own ranks in addition and no bin between them stands out: a third of those ranks, and more than both its
// neighbours.  Where they take in more (about 10 % of heavy-tailed scores, where a bin is a fifth of the bracket), the
// two bins are split in 64 by their next six bits, a wave each, and the ends of those parts will do by the same rule
// (selects at 10 %, key ends / ends of parts, us: 1 M scores 40.5 / 36.4, 3 M 55.4 / 48.8, 8 M 96.3 / 90.1).
// Otherwise (plateaus) the next 12 bits of the keys in the two bins go into a histogram each, and what is left in a
// bin then is ranked by counting, or split by the last 6 bits.  A plateau that
// holds both ends shrinks the bracket to its one key that way, whose members nobody lists.  Selects at 1 % with a
// plateau of f times k keys around the k-th, bin edges without a look at the bins between / with: 8.4 M f = 0.9
// 226 / 81 us, 20 M f = 1.6 315 / 156, 100 M f = 0.6 980 / 518; without plateaus the look costs 0.3, and key ends
// everywhere cost 3 more (8 at 10 % of a large bucket).
// kBracketSigmas etc.: the small buckets bracket the k-th key of the data this way.  The large ones
// (coarse) bracket the ends of the bracket that their fine sample (J.n_sv quads) will give, with eight
// sigma of the coarse sample to either side: k_sample_fine then only looks at the keys in between.  Sigma
// is that of independent keys; scores that the four neighbours of a quad share halve it.  Such scores
// missed in 32 of 1000 draws of 40 M coordinates at 10 % with four sigma, and in 12 with eight (the fine
// sample's own five, halved); a wider coarse bracket costs the fine one a few keys of resolution.
//
// COARSE: the large buckets' launch, k_sample_pick; the other one is k_small_front (small_select.hpp), in which others
// wait for the bracket: there the first workgroup clears the state and the segment counters before it leaves its mark,
// so that no pick comes before that, and a pick writes the bracket and its copies alone (a second pick writes the
// same; what others have counted meanwhile stays).
//
// The workgroups behind those of the sample keep house: counters and histograms of the kernels behind this one,
// the directories of the segment tables (dirs.j[job].dir null: none wanted), the tables' changing columns (cols; the
// sample forms its keys with those that it was handed, whatever the tables hold by then).
constexpr int kSampleGroups = 16;
constexpr int kPickBits = 13, kPickShift = 31 - kPickBits;
constexpr uint32_t kHeavyBin = 3;                    // a half misses the 100 M case above
template <class Src, bool COARSE>
__device__ __forceinline__ void sample_pick_body(const SrcPack<Src>& srcs, const ChainJob& J,
                                                 const typename Src::Cols& cols, uint32_t launch, double sigmas) {
  __shared__ __align__(16) uint32_t s_h[2][kBinsBig];
  __shared__ __align__(16) uint32_t s_list[2][kWideList];
  __shared__ uint32_t s_cnt[2], s_out[2][3], s_all, s_heavy, s_rank[2], s_open[2], s_sub[2][kWave];
  __shared__ WideScratch s_scan;
  static_assert(1 << kPickBits == 2 * kBinsBig, "the two small histograms are the first one");
  SelState* st = J.st;
  const int64_t n = J.n;
  const int n_sv = (int)small_sample_vecs(n);
  // small: the histograms, which only a missed bracket needs (the list may be written while a second picks)
  unsigned long long* __restrict__ sample = reinterpret_cast<unsigned long long*>(COARSE ? J.sample : J.hist);
  static_assert(kHistStride * 2 >= kSmallSampleMax * 4, "two keys a word");
  if (!COARSE && blockIdx.x == 0) {
    constexpr uint32_t MARKS = offsetof(SelState, sampled) / 4;
    const uint32_t t = threadIdx.x;
    if (t < kSmallSegs) st_agent(&J.seg_cnt[t * kSmallSegStride], 0u);
    if (t < sizeof(SelState) / 4 && t - MARKS >= kSampleGroups) st_agent(reinterpret_cast<uint32_t*>(st) + t, t == 0 ? J.k : 0u);
  }
  {
    const int per = (n_sv + kSampleGroups - 1) / kSampleGroups, j = (int)blockIdx.x * per + (int)threadIdx.x;
    const bool mine = (int)threadIdx.x < per && j < n_sv;
    // coarse: a subset of the windows of the fine sample, which it then agrees with
    const int64_t all = COARSE ? J.n_sv : n_sv;
    const int64_t i = mine ? quad_of_window(j * all / n_sv, n / 4, all, J.seed) * 4 : 0;
    Src src = srcs.s[blockIdx.y];
    drop_dir(src, 0);
    // A tensor is looked up among the starts in LDS, beside the loads from the arrays: without the directory, which is
    // being built meanwhile, the bisection is eight dependent loads behind them.  Steps by `update`, bisection in memory ->
    // in LDS, us: 261 K coordinates 40.4 -> 39.1, 1.2 M 51.8 -> 50.2, 8.4 M 137 -> 134, twelve buckets of 20 M 295 -> 287.
    if constexpr (Src::kHyper) {
      uint32_t* const start = &s_h[0][0];
      const int ns = src.sc.n_segs;
      const bool fits = ns <= 2 * kBinsBig;
      if (fits)
        for (int e = (int)threadIdx.x; e < ns; e += kWide) start[e] = (uint32_t)src.sc.segs[e].start;
      __syncthreads();
      if (fits && mine) {
        int a = 0, b = ns - 1;
        while (a < b) {
          const int mid = (a + b + 1) >> 1;
          if (start[mid] <= (uint32_t)i) a = mid; else b = mid - 1;
        }
        src.sc.place(a);
      }
      __syncthreads();                                 // the words are a histogram's next
    }
    if (mine) {
      uint32_t key[4];
      if constexpr (std::is_same<typename Src::Cols, NowCols>::value)
        src.template load<false>(i, n, key, ColsOf{&cols, (int)blockIdx.y});
      else
        src.template load<false>(i, n, key);
#pragma unroll
      for (int h = 0; h < 2; ++h)
        st_agent64(&sample[2 * j + h], (unsigned long long)key[2 * h + 1] << 32 | key[2 * h]);
    }
  }
  const uint32_t ns = (uint32_t)(n_sv * 4);
  if (wave_id() == kWideWaves - 1) {                 // takes no sample; double precision, 0.7 us that nobody waits for
    double rh, rl;
    if (COARSE) {
      const double nf = (double)(J.n_sv * 4), to = (double)ns / nf;
      const RankEnds f = bracket_ranks((double)J.k, (double)n, nf, sigmas);
      const double ah = f.hi * to, al = f.lo * to;
      const double m = (double)ns;
      rh = floor(ah - (8.0 * sqrt(fmax(ah * (1.0 - ah / m), 0.0) + 1.0) + 4.0));
      rl = ceil(al + (8.0 * sqrt(fmax(al * (1.0 - al / m), 0.0) + 1.0) + 4.0));
    } else {
      const RankEnds f = bracket_ranks((double)J.k, (double)n, (double)ns, sigmas);
      rh = f.hi;
      rl = f.lo;
    }
    const bool up = rh < 1.0 || ns == 0, down = rl > (double)ns || ns == 0;
    if (lane_id() == 0) {
      s_open[0] = up;
      s_open[1] = down;
      s_rank[0] = up ? 1u : (uint32_t)rh;
      s_rank[1] = down ? ns : (uint32_t)rl;
    }
  }
  const U4 zero{0u, 0u, 0u, 0u};
  reinterpret_cast<U4*>(s_h[0])[threadIdx.x] = zero;
  reinterpret_cast<U4*>(s_h[1])[threadIdx.x] = zero;
  if (threadIdx.x < 2 * kWave) s_sub[threadIdx.x / kWave][threadIdx.x % kWave] = 0u;
  if (threadIdx.x < 2) s_cnt[threadIdx.x] = 0u;
  if (threadIdx.x == 0) s_heavy = 0u;
  wait_landed();
  if (wave_id() == 0) {
    if (lane_id() == 0) st_agent(&st->sampled[blockIdx.x], launch);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                  // it has landed before the others' are read
    const bool there = lane_id() >= kSampleGroups || ld_agent(&st->sampled[lane_id() % kSampleGroups]) == launch;
    const uint32_t all = ballot64(there) == ~0ull;
    if (lane_id() == 0) s_all = all;
  }
  __syncthreads();
  if (!s_all) return;
  uint32_t key[kSmallPick][4];
#pragma unroll
  for (int u = 0; u < kSmallPick; ++u) {
    const int j = u * kWide + (int)threadIdx.x;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const unsigned long long q =
          j < n_sv ? ld_agent64(&sample[2 * j + h]) : 0ull;
      key[u][2 * h] = sampled_key(q, 0);
      key[u][2 * h + 1] = sampled_key(q, 1);
    }
  }
  const bool open_hi = s_open[0] != 0u, open_lo = s_open[1] != 0u;
  const uint32_t rank[2] = {s_rank[0], s_rank[1]};
  uint32_t t_hi = 0x80000000u, t_lo = 0u;
  if (ns) {
    auto each = [&](auto&& f) {
#pragma unroll
      for (int u = 0; u < kSmallPick; ++u) {
        if (u * kWide >= n_sv) break;                           // uniform
        const bool live = u * kWide + (int)threadIdx.x < n_sv;
#pragma unroll
        for (int e = 0; e < 4; ++e) f(key[u][e], live);
      }
    };
    each([&](uint32_t kk, bool live) { if (live) atomicAdd(&s_h[0][kk >> kPickShift], 1u); });
    __syncthreads();
    RankHit hit[2];
    const uint32_t held = rank[1] - rank[0];
    wide_find_rank<2, 2 * kBinsBig>(s_h[0], rank, s_scan, 0, hit, [&](uint32_t above, uint32_t mine, const auto& h) {
      if (kHeavyBin * mine <= held || above >= rank[1] || above + mine < rank[0]) return;
      constexpr int PER = 2 * kBinsBig / kWide, LAST = 2 * kBinsBig - 1;
#pragma unroll
      for (int j = PER - 1; j >= 0; --j) {
        if (kHeavyBin * h[j] > held && above < rank[1] && above + h[j] >= rank[0]) {
          const int b = threadIdx.x * PER + j;
          if (h[j] > (b > 0 ? s_h[0][b - 1] : 0u) + (b < LAST ? s_h[0][b + 1] : 0u)) s_heavy = 1u;
        }
        above += h[j];
      }
    });
    uint32_t bin[2] = {hit[0].bin, hit[1].bin};
    uint32_t rk[2] = {rank[0] - hit[0].above, rank[1] - hit[1].above};
    uint32_t cnt[2] = {hit[0].count, hit[1].count};
    int w = kPickShift, turn = 1;                      // bits of a key below the bins found so far
    const uint32_t more = (open_hi ? 0u : rk[0] - 1u) + (open_lo ? 0u : cnt[1] - rk[1]);
    bool ends = false;
    if (!s_heavy && 4u * more <= held) {
      ends = true;
      if (!open_hi) t_hi = (bin[0] + 1u) << w;
      if (!open_lo) t_lo = bin[1] << w;
    } else if (!s_heavy) {
      constexpr int kSub = 6, SH = kPickShift - kSub;
      static_assert(1 << kSub == kWave, "a bin's part per lane");
      each([&](uint32_t kk, bool live) {
        const uint32_t top = kk >> kPickShift, part = (kk >> SH) & (kWave - 1);
        if (live && top == bin[0]) atomicAdd(&s_sub[0][part], 1u);
        if (live && top == bin[1]) atomicAdd(&s_sub[1][part], 1u);
      });
      __syncthreads();
      if (wave_id() < 2) {
        const int q = wave_id(), l = lane_id();
        const uint32_t c = s_sub[q][kWave - 1 - l], incl = wave_incl_scan(c);              // from the top
        const uint32_t near = (l > 0 ? s_sub[q][kWave - l] : 0u) + (l < kWave - 1 ? s_sub[q][kWave - 2 - l] : 0u);
        const bool one_bin = bin[0] == bin[1];
        const bool between = (q == 1 && !one_bin ? true : incl >= rk[0]) && (q == 0 && !one_bin ? true : incl - c < rk[1]);
        if (between && kHeavyBin * c > held && c > near) s_heavy = 1u;
        const int at = __ffsll((unsigned long long)ballot64(incl >= rk[q])) - 1;
        if (l == at) { s_out[q][0] = (uint32_t)(kWave - 1 - l); s_out[q][1] = incl - c; s_out[q][2] = c; }
      }
      __syncthreads();
      const uint32_t beyond = (open_hi ? 0u : rk[0] - s_out[0][1] - 1u) + (open_lo ? 0u : s_out[1][2] - (rk[1] - s_out[1][1]));
      ends = !s_heavy && 4u * beyond <= held;
      if (ends && !open_hi) t_hi = ((bin[0] << kSub | s_out[0][0]) + 1u) << SH;
      if (ends && !open_lo) t_lo = (bin[1] << kSub | s_out[1][0]) << SH;
    }
    if (!ends) {
      while (w > 0 && (cnt[0] > (uint32_t)kWideList || cnt[1] > (uint32_t)kWideList)) {
        const int sh = w > 12 ? w - 12 : 0, bits = w - sh;
        reinterpret_cast<U4*>(s_h[0])[threadIdx.x] = zero;
        reinterpret_cast<U4*>(s_h[1])[threadIdx.x] = zero;
        __syncthreads();
        each([&](uint32_t kk, bool live) {
          const uint32_t top = kk >> w;
          if (!live || (top != bin[0] && top != bin[1])) return;
          const uint32_t low = (kk >> sh) & ((1u << bits) - 1u);
          if (top == bin[0]) atomicAdd(&s_h[0][low], 1u);
          if (top == bin[1]) atomicAdd(&s_h[1][low], 1u);
        });
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const uint32_t want[1] = {rk[q]};
          RankHit h[1];
          wide_find_rank<1>(s_h[q], want, s_scan, turn, h);
          turn ^= 1;
          bin[q] = (bin[q] << bits) | h[0].bin;
          rk[q] -= h[0].above;
          cnt[q] = h[0].count;
        }
        w = sh;
      }
      if (w > 0) {
        each([&](uint32_t kk, bool live) {
          const uint32_t top = kk >> w;
          if (!live || (top != bin[0] && top != bin[1])) return;
          if (top == bin[0]) s_list[0][atomicAdd(&s_cnt[0], 1u)] = kk;
          if (top == bin[1]) s_list[1][atomicAdd(&s_cnt[1], 1u)] = kk;
        });
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 2; ++q) wide_list_rank(s_list[q], cnt[q], rk[q], s_out[q]);
        __syncthreads();
      }
      // keys equal to the upper sample key stay inside the bracket
      if (!open_hi) t_hi = (w > 0 ? s_out[0][0] : bin[0]) + 1u;
      if (!open_lo) t_lo = w > 0 ? s_out[1][0] : bin[1];
    }
  }
  if (COARSE) {
    if (threadIdx.x < kStateWords)
      st_agent64(reinterpret_cast<unsigned long long*>(st) + threadIdx.x, picked_word(threadIdx.x, J.k, t_lo, t_hi));
  } else {
    if (threadIdx.x < kSmallSegs) {
      unsigned long long* w = small_bracket_copy(J, (int)threadIdx.x);
      st_agent64(w, (unsigned long long)launch << 32 | t_lo);
      st_agent64(w + 1, (unsigned long long)launch << 32 | t_hi);
    }
    if (threadIdx.x == 0)
      st_agent64(reinterpret_cast<unsigned long long*>(st) + kBracketWord, picked_word(kBracketWord, J.k, t_lo, t_hi));
  }
}
template <class Src>
__global__ __launch_bounds__(kWide) void k_sample_pick(SrcPack<Src> srcs, ChainJobs jobs, SegDirJobs dirs,
                                                       typename Src::Cols cols, uint32_t launch, double sigmas) {
  const ChainJob& J = jobs.j[blockIdx.y];
  if (blockIdx.x < kSampleGroups) {
    sample_pick_body<Src, true>(srcs, J, cols, launch, sigmas);
    return;
  }
  const int t0 = (blockIdx.x - kSampleGroups) * kWide + threadIdx.x, step = (gridDim.x - kSampleGroups) * kWide;
  clear_large(J, t0, step, true);
  keep_tables(dirs, cols, t0, step);
}

// The fine sample of a large bucket: only how its keys fall relative to the coarse bracket is kept --
// counts above it, and a histogram of the few inside.  The last workgroup to finish takes the bracket from it, at the
// edges of the histogram's bins (rounded outwards: a few sample keys wide); an end the coarse bracket missed is left
// open.  The tickets go by sixteen words and one: on one word they queue, 11 ns each (1024 workgroups: 8 us of a select
// of 300 M scores), and four quads a thread by a quarter of the workgroups made the sample of `update` 12 us longer.
// The pick as a launch of its own -> here, selects in a row at 1 %, us: 9 M scores 43.0 -> 41.1, 20 M 53.9 -> 52.5,
// 40 M 69.7 -> 68.7, 100 M and more the same.
// What the pick reads of the others' are device-scope atomics, which every wave waits for before its workgroup
// takes its ticket; the ticket is a word of the state that the kernel before has written.
constexpr int kFineSpread = kRelSpread;                // tickets: a word for every sixteenth workgroup, then one for those
template <class Src>
__global__ __launch_bounds__(kBlock) void k_sample_fine(SrcPack<Src> srcs, ChainJobs jobs, double sigmas) {
  __shared__ uint32_t s_w[kChunksPerBlock], s_last, s_hit[2][3], s_bins[kWideBins + kBlock];
  const ChainJob& J = jobs.j[blockIdx.y];
  const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if ((int64_t)blockIdx.x * kBlock >= J.n_sv) return;                 // a smaller job of the batch
  Src src = srcs.s[blockIdx.y];
  const uint32_t c_lo = J.st->t_lo, c_hi = J.st->t_hi;
  const int sh = rel_shift(c_lo, c_hi, kWideBins);
  uint32_t* __restrict__ bins = J.rel + kRelSample;
  uint32_t key[4] = {0u, 0u, 0u, 0u};
  const bool live = j < J.n_sv;
  if (live) src.template load<false>(quad_of_window(j, J.n_vec, J.n_sv, J.seed) * 4, J.n, key);
  uint32_t above = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    above += (uint32_t)__popcll(ballot64(live && key[e] >= c_hi));
    const bool in = live && key[e] >= c_lo && key[e] < c_hi;
    const uint32_t bin = (key[e] - c_lo) >> sh;
    const uint64_t act = ballot64(in);
    if (act == 0) continue;
    // many lanes on one bin (a plateau) add once
    const uint32_t lead = (uint32_t)__builtin_amdgcn_readlane((int)bin, __ffsll((unsigned long long)act) - 1);
    const uint64_t same = ballot64(in && bin == lead);
    const bool fold = __popcll(same) >= 8;
    if (fold && lane_id() == 0) atomicAdd(&bins[lead], (uint32_t)__popcll(same));
    if (in && !(fold && bin == lead)) atomicAdd(&bins[bin], 1u);
  }
  if (lane_id() == 0) s_w[wave_id()] = above;
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t all = s_w[0] + s_w[1] + s_w[2] + s_w[3];
    if (all) atomicAdd(&J.rel[kRelAbove + (blockIdx.x % kRelSpread) * 64], all);
  }
  wait_landed();
  if (threadIdx.x == 0) {
    const uint32_t groups = (uint32_t)cdiv64(J.n_sv, kBlock), w = blockIdx.x % kFineSpread;
    const uint32_t words = groups < (uint32_t)kFineSpread ? groups : (uint32_t)kFineSpread;
    const bool filled = atomicAdd(&J.rel[kRelAbove + w * 64 + 32], 1u) == (groups - w + kFineSpread - 1) / kFineSpread - 1;
    s_last = filled && atomicAdd(&J.st->ticket, 1u) == words - 1u;
  }
  __syncthreads();
  if (!s_last) return;
  constexpr int PER = kWideBins / kBlock;
  const uint32_t part = threadIdx.x < kRelSpread ? ld_agent(&J.rel[kRelAbove + threadIdx.x * 64]) : 0u;
  uint32_t h[PER], mine = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) h[i] = ld_agent(&bins[i * kBlock + threadIdx.x]);
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int at = i * kBlock + (int)threadIdx.x;
    s_bins[at + at / PER] = h[i];                                     // a word between the threads' runs
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < PER; ++i) { h[i] = s_bins[threadIdx.x * (PER + 1) + i]; mine += h[i]; }
  uint32_t total, inside;
  const uint32_t before = block_excl_scan(mine, s_w, inside);
  __syncthreads();
  block_excl_scan(part, s_w, total);
  const double ns = (double)(J.n_sv * 4);
  const RankEnds f = bracket_ranks((double)J.k, (double)J.n, ns, sigmas);
  const bool in_hi = f.hi >= 1.0 && f.hi > (double)total && f.hi <= (double)total + (double)inside;
  const bool in_lo = f.lo <= ns && f.lo > (double)total && f.lo <= (double)total + (double)inside;
  const uint32_t rank[2] = {in_hi ? (uint32_t)f.hi - total : 1u, in_lo ? (uint32_t)f.lo - total : 1u};
  if (threadIdx.x < 2) s_hit[threadIdx.x][0] = s_hit[threadIdx.x][1] = s_hit[threadIdx.x][2] = 0u;
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    uint32_t run = inside - before - mine;                            // keys in the bins above the thread's
    if (run < rank[q] && rank[q] <= run + mine) {
#pragma unroll
      for (int i = PER - 1; i >= 0; --i) {
        if (run < rank[q] && rank[q] <= run + h[i]) {
          s_hit[q][0] = (uint32_t)(threadIdx.x * PER + i);
          s_hit[q][1] = run;
          s_hit[q][2] = h[i];
        }
        run += h[i];
      }
    }
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  uint32_t t_hi = 0x80000000u, t_lo = 0u, in_sample = ~0u;
  if (in_hi) {
    t_hi = c_lo + ((s_hit[0][0] + 1u) << sh);
    if (t_hi > c_hi) t_hi = c_hi;
  }
  if (in_lo) {
    t_lo = c_lo + (s_hit[1][0] << sh);
    in_sample = total + s_hit[1][1] + s_hit[1][2] - (in_hi ? total + s_hit[0][1] : 0u);
  }
  SelState z = {};
  z.k = J.k;
  z.t_hi = t_hi;
  z.t_lo = t_lo;
  z.in_sample = in_sample;
  *J.st = z;
}

// The one sweep over the data: a one-shot grid, one 1024-element chunk per
// wave (a capped grid that strides over the chunks reads 15 % slower).  The
// keys inside the bracket are first gathered, in index order, in the wave's
// LDS buffer; at the end of the chunk the wave reserves room for all of them
// with ONE atomic add on the counter of the candidate segment its chunk
// hashes to (kSegWaves counters, so neighbouring waves hit different
// addresses) and copies them there.  A chunk's candidates therefore stay
// contiguous and index-ordered in the list; the order of the chunks inside a
// segment is arbitrary and nothing downstream depends on it.
constexpr int kWaveCandCap = 256;          // candidates one chunk can hold before the sweep gives up

// LDS of one wave of the sweep.
struct SweepLds {
  uint32_t idx[kWaveCandCap];              // the chunk's candidates, index order
  uint32_t key[kWaveCandCap];
  uint32_t planes[kPlaneWordsPerChunk];    // the chunk's 32 plane words ("key above the bracket")
  uint32_t mbytes[kChunk / 4];             // the chunk's mask bytes in element order (mask-byte sweeps)
};

// The flags of a slab live as four wave ballots (element e of every lane), i.e.
// on the scalar unit: counts are popcounts, "any" is a scalar test, and the
// index-ordered position of a flagged element is the number of mask bits
// below its lane over the four ballots plus the lane's own earlier elements.
struct Ballot4 {
  uint64_t m[4];
  __device__ __forceinline__ uint64_t any() const { return m[0] | m[1] | m[2] | m[3]; }
  __device__ __forceinline__ uint32_t count() const {
    return (uint32_t)(__popcll(m[0]) + __popcll(m[1]) + __popcll(m[2]) + __popcll(m[3]));
  }
  __device__ __forceinline__ uint32_t below_lane() const {
    return lanes_below(m[0]) + lanes_below(m[1]) + lanes_below(m[2]) + lanes_below(m[3]);
  }
  __device__ __forceinline__ bool mine(int e) const { return (m[e] >> lane_id()) & 1ull; }
};

// Appends the flagged elements of one slab in index order: put(pos, e).
template <class F>
__device__ __forceinline__ void ballot_append(const Ballot4& f, uint32_t& count, F&& put) {
  if (f.any() == 0) return;                      // scalar branch
  uint32_t pos = count + f.below_lane();
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (f.mine(e)) { put(pos, e); ++pos; }
  count += f.count();
}

// The slab's four "above" ballots are eight of the chunk's 32 plane words
// (words 8 it + 2 e + h): one lane parks them in the wave's LDS planes, from
// where the chunk's 128 bytes are stored in one piece.
__device__ __forceinline__ void plane_put(const Ballot4& a, int it, uint32_t* lds_planes) {
  if (lane_id() == 0) {
    uint64_t* w = reinterpret_cast<uint64_t*>(lds_planes) + it * 4;
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = a.m[e];
  }
}

// One chunk of the sweep.  chi / tot_nf / mycnt are wave totals (scalar).
// PM: 0 counts only; 1 the provisional selection (keys above the bracket) also goes out as bit
// planes; 2 as mask bytes, straight into the caller's mask (a mask-only select then needs no
// expansion pass: the candidates are settled in the bytes).
// KEEP: a pass behind the select reads the same data again and finds it in the memory-side cache.
template <class Src, bool FULL, int PM, bool KEEP>
__device__ __forceinline__ void bracket_chunk(Src& src, const typename Src::Chunk& ck, int64_t n,
                                              int64_t c, uint32_t T_LO,
                                              uint32_t T_HI, uint32_t& chi, uint32_t& tot_nf,
                                              uint32_t& mycnt, SweepLds& lds,
                                              uint32_t* __restrict__ pbits,
                                              uint8_t* __restrict__ mask_bytes = nullptr,
                                              bool mvec = false, bool m16 = false) {
  // The loads of kAhead slabs (256 elements each) are issued together, then
  // their keys are formed slab by slab: expensive key sources (Adam-normalised
  // scores) look fewer slabs ahead to stay within their register budget.  The
  // ragged path (the last chunk) goes one slab at a time through
  // a rolled loop: it only has to be small.
  constexpr int kAhead = FULL ? Src::kAhead : 1;
  static_assert(kChunkIters % kAhead == 0, "look-ahead divides the slabs of a chunk");
  constexpr int kGroupUnroll = kAhead == kChunkIters ? kChunkIters : 1;
  src.chunk_hyper(c);        // measured: looking the tensor up behind the first loads instead is slower
#pragma unroll kGroupUnroll
  for (int g0 = 0; g0 < kChunkIters; g0 += kAhead) {
    typename Src::Raw raw[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int64_t i = c * kChunk + (g0 + u) * (kWave * kVec) + lane_id() * kVec;
      if (FULL || i < n) src.template fetch<FULL, KEEP>(ck, i, n, raw[u]);
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int it = g0 + u;
      const int64_t i = c * kChunk + it * (kWave * kVec) + lane_id() * kVec;
      uint32_t key[4] = {0u, 0u, 0u, 0u};
      if (FULL || i < n) src.template keys<FULL>(ck, i, n, raw[u], key);
      Ballot4 above, cand;
      uint64_t nf = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint64_t valid = FULL ? ~0ull : ballot64(i + e < n);
        above.m[e] = ballot64(key[e] >= T_HI) & valid;
        cand.m[e] = ballot64(key[e] >= T_LO) & valid & ~above.m[e];
        nf |= ballot64(key[e] >= 0x7F800000u) & valid;
      }
      chi += above.count();
      if (nf) {                                  // rare: count them properly
#pragma unroll
        for (int e = 0; e < 4; ++e)
          tot_nf += (uint32_t)__popcll(ballot64(key[e] >= 0x7F800000u && (FULL || i + e < n)));
      }
      ballot_append(cand, mycnt, [&](uint32_t pos, int e) {
        if (pos < (uint32_t)kWaveCandCap) { lds.idx[pos] = (uint32_t)(i + e); lds.key[pos] = key[e]; }
      });
      // provisional mask as bit planes: everything above the bracket is
      // certainly selected; the few keys inside it are settled after the
      // candidate descent.  One 128-byte store per chunk.
      if (PM == 1) plane_put(above, it, lds.planes);
      if (PM == 2 && (FULL || i < n)) {
        const uint32_t mk[4] = {above.mine(0), above.mine(1), above.mine(2), above.mine(3)};
        // a lane's four bytes per slab are parked in LDS in element order, and the chunk's 1024
        // bytes leave as one 16-byte store per lane (four 4-byte stores per lane otherwise)
        if (FULL && m16) lds.mbytes[it * kWave + lane_id()] = mk[0] | (mk[1] << 8) | (mk[2] << 16) | (mk[3] << 24);
        else if (FULL && mvec) st_u8<true>(mask_bytes, i, n, mk, true);
        else store4_u8(mask_bytes, i, n, mk, mvec);
      }
    }
  }
  if (PM == 1) {
    __builtin_amdgcn_wave_barrier();
    if (lane_id() < kPlaneWordsPerChunk) pbits[c * kPlaneWordsPerChunk + lane_id()] = lds.planes[lane_id()];
  }
  if (PM == 2 && FULL && m16) {
    __builtin_amdgcn_wave_barrier();
    const U4 v = reinterpret_cast<const U4*>(lds.mbytes)[lane_id()];
    *reinterpret_cast<U4*>(mask_bytes + c * kChunk + lane_id() * 16) = v;
  }
}

// A wave's candidates beyond its LDS buffer: a second look at the chunk, slab by slab.
template <class Src, class F>
__device__ __forceinline__ void recollect(Src& src, int64_t n, int64_t c, uint32_t T_LO, uint32_t T_HI, F&& put) {
  src.chunk_hyper(c);
  uint32_t run = 0;
  for (int it = 0; it < kChunkIters; ++it) {
    const int64_t i = c * kChunk + it * (kWave * kVec) + lane_id() * kVec;
    uint32_t key[4] = {0u, 0u, 0u, 0u};
    if (i < n) src.template load<false>(i, n, key);
    Ballot4 in;
#pragma unroll
    for (int e = 0; e < 4; ++e) in.m[e] = ballot64(i + e < n && key[e] >= T_LO && key[e] < T_HI);
    ballot_append(in, run, [&](uint32_t pos, int e) { put(pos, (uint32_t)(i + e), key[e]); });
  }
}

// A bracket of a single key (a plateau of equal keys holds the k-th one) collects nothing: its members
// are ties, counted per chunk (tile_eq) and in bin 0 of the relative histogram.
template <class Src, int PM, bool KEEP = false>
__global__ __launch_bounds__(kBlock) void k_bracket_sweep(
    Src src, int64_t n, SelState* __restrict__ st, uint32_t* __restrict__ rel,
    uint32_t* __restrict__ tile_gt, uint32_t* __restrict__ tile_eq, uint32_t* __restrict__ seg_idx,
    uint32_t* __restrict__ seg_key, uint32_t* __restrict__ seg_cnt, uint32_t seg_cap,
    uint32_t* __restrict__ pbits, uint32_t* __restrict__ hi_part, uint32_t* __restrict__ nf_part,
    uint8_t* __restrict__ mask_bytes = nullptr, bool mvec = false) {
  const bool m16 = PM == 2 && (reinterpret_cast<uintptr_t>(mask_bytes) & 15) == 0;
  __shared__ uint32_t s_hi[kChunksPerBlock], s_nf[kChunksPerBlock], s_eq[kChunksPerBlock];
  __shared__ SweepLds s_lds[kChunksPerBlock];
  const uint32_t T_HI = st->t_hi, T_LO = st->t_lo;
  const bool single = T_HI - T_LO == 1u;
  const int64_t n_chunks = cdiv64(n, kChunk);
  const int64_t c = (int64_t)blockIdx.x * kChunksPerBlock + wave_id();
  uint32_t chi = 0, tot_nf = 0, ties = 0;
  uint32_t* __restrict__ const bins = rel + (blockIdx.x % kRelCopies) * kRelBins;
  if (c < n_chunks) {
    uint32_t mycnt = 0;
    SweepLds& lds = s_lds[wave_id()];
    const typename Src::Chunk ck = src.chunk_begin(c);
    if (src.vec && (c + 1) * kChunk <= n)
      bracket_chunk<Src, true, PM, KEEP>(src, ck, n, c, T_LO, T_HI, chi, tot_nf, mycnt, lds, pbits, mask_bytes, mvec, m16);
    else
      bracket_chunk<Src, false, PM, KEEP>(src, ck, n, c, T_LO, T_HI, chi, tot_nf, mycnt, lds, pbits, mask_bytes, mvec);
    if (single) { ties = mycnt; mycnt = 0; }
    if (lane_id() == 0) { tile_gt[c] = chi; tile_eq[c] = ties; }   // chi / tot_nf are wave totals
    if (mycnt) {                                        // wave-uniform
      const uint32_t seg = (uint32_t)c & (uint32_t)(kSegWaves - 1);
      uint32_t base = 0;
      if (lane_id() == 0) base = atomicAdd(&seg_cnt[seg], mycnt);
      base = __shfl(base, 0, kWave);
      if (base + mycnt > seg_cap) {
        if (lane_id() == 0) atomicOr(&st->overflow, 1u);
      } else {
        const int sh = rel_shift(T_LO, T_HI, kRelBins);
        uint32_t* const g_idx = seg_idx + (int64_t)seg * seg_cap + base;
        uint32_t* const g_key = seg_key + (int64_t)seg * seg_cap + base;
        if (mycnt <= (uint32_t)kWaveCandCap) {
          __builtin_amdgcn_wave_barrier();              // the wave's LDS stores above are read below
          for (uint32_t j = lane_id(); j < mycnt; j += kWave) {
            const uint32_t key = lds.key[j];
            g_idx[j] = lds.idx[j];
            g_key[j] = key;
            atomicAdd(&bins[(key - T_LO) >> sh], 1u);
          }
        } else {
          recollect(src, n, c, T_LO, T_HI, [&](uint32_t pos, uint32_t idx, uint32_t key) {
            g_idx[pos] = idx;
            g_key[pos] = key;
            atomicAdd(&bins[(key - T_LO) >> sh], 1u);
          });
        }
      }
    }
  }
  const bool neg = ballot64(src_negative(src) != 0u) != 0ull;
  if (lane_id() == 0) {
    s_hi[wave_id()] = chi;
    s_eq[wave_id()] = ties;
    s_nf[wave_id()] = tot_nf | (neg ? 0x80000000u : 0u);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t h = s_hi[0] + s_hi[1] + s_hi[2] + s_hi[3];
    const uint32_t t = s_eq[0] + s_eq[1] + s_eq[2] + s_eq[3];
    const uint32_t any_neg = (s_nf[0] | s_nf[1] | s_nf[2] | s_nf[3]) & 0x80000000u;
    const uint32_t f = (s_nf[0] + s_nf[1] + s_nf[2] + s_nf[3]) & 0x7FFFFFFFu;
    if (h) atomicAdd(&hi_part[blockIdx.x & (kSweepParts - 1)], h);
    if (t) atomicAdd(&bins[0], t);
    if (f) atomicAdd(&nf_part[blockIdx.x & (kSweepParts - 1)], f);
    if (any_neg) raise_negative(st);
  }
}

// Settlement of a bracket, one launch for all that lies between the sweep and the chunk scan: exact
// threshold, per-chunk corrections, and the candidates' places in the mask or the planes.
//   1. Every workgroup sums the copies of the sweep's relative histogram and finds the bin where the
//      count from the top reaches k -- each for itself, so nothing has to wait for anything.
//   2. It then walks its share of the candidate segments: keys above the bin are selected, the bin's
//      own go to the edge list (about C / kRelBins of C candidates) and are counted as ties for now.
//   3. The last workgroup to finish ranks the edge list (threshold, ties, which of them are granted:
//      lowest index first) and corrects the counts.  An edge list of one key value needs no ranking
//      whatever its length (gradients on the bf16 grid: a hundred thousand equal keys); the ties of
//      one too long for LDS are placed by k_tail, behind the chunk scan.
// What step 3 reads of the others' is written by device-scope atomics and atomic stores, each wave
// waits for its own (vmcnt) before the workgroup takes its ticket, and the last one reads with atomic
// loads: no cache-wide fence, which costs 65 ns a workgroup here.
// The chain of one-level launches this replaces (check, compaction, three histogram levels, chunk
// counts, mask) took 75 to 150 us.  Now 16 us at 40 M coordinates (48 K candidates), 53 us at 1e9
// (1.25 M candidates: their random mask bytes), 20 us over the bf16 ties of a replayed step.
constexpr int kEdgeCap = 4096;              // edge entries the last workgroup holds in LDS
struct EdgeList {                           // LDS, or global memory when there are more
  const uint32_t* key;
  const uint32_t* idx;
  uint32_t cnt;
  bool lds;
  __device__ __forceinline__ uint32_t key_at(uint32_t j) const {
    return lds ? key[j] : __hip_atomic_load(key + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __device__ __forceinline__ uint32_t idx_at(uint32_t j) const {
    return lds ? idx[j] : __hip_atomic_load(idx + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
};
// `rank`-th (1-based) largest of the w-bit offsets value(j) - lo, by 12-bit levels.  `lo`, `rank`, `eq`
// end as the value, its rank among the equal ones, and their number.
template <class V>
__device__ __forceinline__ void edge_descend(uint32_t cnt, V&& value, uint32_t& lo, int w, uint32_t& rank,
                                             uint32_t& eq, uint32_t* s_hist, WideScratch& s_scan) {
  int turn = 0;
  while (w > 0) {
    const int sh = w > 12 ? w - 12 : 0;
    reinterpret_cast<U4*>(s_hist)[threadIdx.x] = U4{0u, 0u, 0u, 0u};
    __syncthreads();
    constexpr int U = 4;                                 // global lists: loads in flight per thread
    for (uint32_t j0 = 0; j0 < cnt; j0 += U * kWide) {
      uint32_t v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t j = j0 + u * kWide + threadIdx.x;
        v[u] = j < cnt ? value(j) : ~0u;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t off = v[u] - lo;
        wide_hist_add(s_hist, off >> sh, off >> w == 0u);
      }
    }
    __syncthreads();
    const uint32_t want[1] = {rank};
    RankHit h[1];
    wide_find_rank<1>(s_hist, want, s_scan, turn, h);
    turn ^= 1;
    lo += h[0].bin << sh;
    rank -= h[0].above;
    eq = h[0].count;
    w = sh;
  }
  __syncthreads();
}
// The place of a settled coordinate in the job's mask bytes or bit planes (neither: the writing pass
// forms the keys again).
__device__ __forceinline__ void place_selected(const ChainJob& J, uint32_t idx) {
  if (J.mask) {
    J.mask[idx] = 1;
  } else if (J.planes) {
    const uint32_t lane = (idx >> 2) & 63u, e = idx & 3u;
    atomicOr(&J.planes[(idx >> 8) * 8 + 2 * e + (lane >> 5)], 1u << (lane & 31));
  }
}
// The calling wave's share of the candidate segments: f(valid, key, idx, position), by whole waves.  Eight
// segments at a time: their counts in one load, their entries as one run, so that short segments still
// fill the wave and several loads are in flight.
template <class F>
__device__ __forceinline__ void walk_segments(const ChainJob& J, int wave, int waves, F&& f) {
  constexpr int kRun = 8, U = 4;
  for (int w0 = wave * kRun; w0 < kSegWaves; w0 += waves * kRun) {
    const uint32_t cl = lane_id() < kRun ? J.seg_cnt[w0 + lane_id()] : 0u;
    uint32_t off[kRun + 1];
    off[0] = 0;
#pragma unroll
    for (int r = 0; r < kRun; ++r) off[r + 1] = off[r] + (uint32_t)__builtin_amdgcn_readlane((int)cl, r);
    for (uint32_t q0 = 0; q0 < off[kRun]; q0 += U * kWave) {
      uint32_t key[U], idx[U], pos[U];
      bool valid[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t q = q0 + u * kWave + lane_id();
        valid[u] = q < off[kRun];
        uint32_t at = q;                                 // entry q is entry q - off[r] of segment w0 + r
#pragma unroll
        for (int r = 0; r < kRun - 1; ++r) at = q >= off[r + 1] ? q - off[r + 1] + (uint32_t)(r + 1) * J.seg_cap : at;
        pos[u] = (uint32_t)w0 * J.seg_cap + at;          // kSegWaves * seg_cap <= n / 32 rounded up: 27 bits
        key[u] = valid[u] ? J.seg_key[pos[u]] : 0u;
        idx[u] = valid[u] ? J.seg_idx[pos[u]] : 0u;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (q0 + u * kWave >= off[kRun]) break;          // wave-uniform
        f(valid[u], key[u], idx[u], pos[u]);
      }
    }
  }
}
// Adds the wave's flagged entries to their chunks' counters.  A chunk's candidates follow one another
// in the list, so equal neighbours are counted together: one atomic per chunk and 64 entries.
__device__ __forceinline__ void count_by_chunk(uint32_t* __restrict__ tiles, bool flag, uint32_t idx) {
  const uint64_t on = ballot64(flag);
  if (on == 0) return;
  const uint32_t c = idx >> 10;
  const uint32_t left = __shfl_up(c, 1, kWave);
  const uint64_t heads = ballot64(lane_id() == 0 || c != left);       // first lane of every run of one chunk
  if ((heads >> lane_id()) & 1ull) {
    const uint64_t behind = lane_id() == 63 ? 0ull : heads >> (lane_id() + 1) << (lane_id() + 1);
    const uint64_t run = (behind ? (1ull << (__ffsll((unsigned long long)behind) - 1)) - 1ull : ~0ull) &
                         (~0ull << lane_id());
    const uint32_t cnt = (uint32_t)__popcll(on & run);
    if (cnt) atomicAdd(&tiles[c], cnt);
  }
}
static __global__ __launch_bounds__(kWide) void k_settle(ChainJobs jobs) {
  __shared__ __align__(16) uint32_t s_hist[kWideBins];
  __shared__ uint32_t s_key[kEdgeCap], s_idx[kEdgeCap];
  __shared__ uint32_t s_n, s_inv, s_max, s_base, s_last;
  __shared__ WideScratch s_scan;
  const ChainJob& J = jobs.j[blockIdx.y];
  SelState* __restrict__ st = J.st;
  const uint32_t T_LO = st->t_lo, T_HI = st->t_hi, k = J.k;
  const bool single = T_HI - T_LO == 1u;
  const int sh = rel_shift(T_LO, T_HI, kRelBins);
  // ---- 1
  uint32_t mine = 0;
#pragma unroll
  for (int r = 0; r < kRelCopies; ++r) mine += J.rel[r * kRelBins + threadIdx.x];
  static_assert(kRelBins == kWide && kSweepParts <= kWide, "a bin and a partial counter per thread");
  const uint32_t part = threadIdx.x < kSweepParts ? J.blk_gt[threadIdx.x] : 0u;
  if (threadIdx.x == 0) s_n = s_inv = s_max = 0u;
  uint32_t n_hi, n_in;
  wide_prefix(part, s_scan, 0, n_hi);
  const uint32_t before = wide_prefix(mine, s_scan, 1, n_in);
  const bool ok = !st->overflow && n_hi < k && k <= n_hi + n_in;
  const uint32_t above_me = n_in - before - mine, rank0 = k - n_hi;
  if (ok && above_me < rank0 && rank0 <= above_me + mine) {
    s_scan.hit[0][0][0] = threadIdx.x;
    s_scan.hit[0][0][1] = above_me;
    s_scan.hit[0][0][2] = mine;
  }
  __syncthreads();
  const bool first = blockIdx.x == 0;
  if (first) {
    uint32_t n_nf;
    wide_prefix(threadIdx.x < kSweepParts ? J.blk_eq[threadIdx.x] : 0u, s_scan, 0, n_nf);
    if (threadIdx.x == 0) {
      st->n_hi = n_hi;
      st->cand_count = n_in;
      st->bracket_ok = ok && !single ? 1u : 0u;     // a plateau's selection is written by an ordered pass
      st->skip = ok ? 1u : 0u;                      // the radix passes run only when the bracket failed
      st->path = ok && !single ? 1u : 0u;
      st->nonfinite = ok ? n_nf : 0u;               // recounted by the radix passes otherwise
      if (ok && single) {
        st->thresh_bits = T_LO;
        st->need = rank0;
        st->n_eq = n_in;
        st->n_gt = n_hi;
      }
    }
  }
  if (!ok || single) return;
  const uint32_t bin = s_scan.hit[0][0][0], above = s_scan.hit[0][0][1];
  // ---- 2
  const uint32_t e_lo = T_LO + (bin << sh);
  uint32_t e_inv = 0, e_max = 0;
  walk_segments(J, (int)blockIdx.x * kWideWaves + wave_id(), (int)gridDim.x * kWideWaves,
                [&](bool valid, uint32_t key, uint32_t idx, uint32_t) {
    const uint32_t off = key - e_lo;
    const bool sel = valid && (int32_t)off >= 0 && off >> sh != 0u;
    const bool edge = valid && (int32_t)off >= 0 && off >> sh == 0u;
    if (!J.mask_only) count_by_chunk(J.tile_gt, sel, idx);
    if (sel) place_selected(J, idx);
    if (ballot64(edge) == 0) return;
    count_by_chunk(J.tile_eq, edge, idx);
    if (!edge) return;
    e_inv = e_inv > ~key ? e_inv : ~key;
    e_max = e_max > key ? e_max : key;
    const uint32_t at = atomicAdd(&s_n, 1u);
    if (at < (uint32_t)kEdgeCap) {
      s_key[at] = key;
      s_idx[at] = idx;
    } else {                                            // more than a workgroup's share of any but a plateau
      const uint32_t g = atomicAdd(&st->edge_cnt, 1u);
      __hip_atomic_store(&J.cand_key[g], key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(&J.cand_idx[g], idx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  });
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    const uint32_t a = __shfl_xor(e_inv, o, kWave), b = __shfl_xor(e_max, o, kWave);
    e_inv = e_inv > a ? e_inv : a;
    e_max = e_max > b ? e_max : b;
  }
  if (lane_id() == 0 && e_inv) { atomicMax(&s_inv, e_inv); atomicMax(&s_max, e_max); }
  __syncthreads();
  const uint32_t held = s_n < (uint32_t)kEdgeCap ? s_n : (uint32_t)kEdgeCap;
  if (threadIdx.x == 0 && held) {
    s_base = atomicAdd(&st->edge_cnt, held);
    atomicMax(&st->edge_inv, s_inv);
    atomicMax(&st->edge_max, s_max);
  }
  __syncthreads();
  for (uint32_t j = threadIdx.x; j < held; j += kWide) {
    __hip_atomic_store(&J.cand_key[s_base + j], s_key[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&J.cand_idx[s_base + j], s_idx[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  // ---- 3
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // this wave's atomics and stores have landed
  __syncthreads();
  if (threadIdx.x == 0)
    s_last = __hip_atomic_fetch_add(&st->ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
  __syncthreads();
  if (!s_last) return;
  const uint32_t cnt = __hip_atomic_load(&st->edge_cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const uint32_t inv = __hip_atomic_load(&st->edge_inv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const uint32_t top = __hip_atomic_load(&st->edge_max, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const bool one_key = top == ~inv, short_list = cnt <= (uint32_t)kEdgeCap;
  EdgeList L{J.cand_key, J.cand_idx, cnt, false};
  if (short_list) {
    for (uint32_t j = threadIdx.x; j < cnt; j += kWide) { s_key[j] = L.key_at(j); s_idx[j] = L.idx_at(j); }
    L = EdgeList{s_key, s_idx, cnt, true};
    __syncthreads();
  }
  uint32_t T = one_key ? top : e_lo, need = rank0 - above, n_eq = cnt;
  if (!one_key)
    edge_descend(cnt, [&](uint32_t j) { return L.key_at(j); }, T, sh, need, n_eq, s_hist, s_scan);
  const bool places = J.mask || J.planes;
  // of the ties the `need` lowest indices are granted: the last granted one is the need-th from below
  const bool all = J.tie_all || need == n_eq;
  uint32_t last_idx = 0xFFFFFFFFu;
  if (short_list && places && !all) {
    uint32_t lo = 0, r = n_eq - need + 1, eq = 0;         // rank from the top among the ties
    edge_descend(cnt, [&](uint32_t j) { return L.key_at(j) == T ? L.idx_at(j) : ~0u; }, lo, 31, r, eq, s_hist, s_scan);
    last_idx = lo;
  }
  if (!one_key || (short_list && places)) {
    for (uint32_t j = threadIdx.x; j < cnt; j += kWide) {
      const uint32_t key = L.key_at(j), idx = L.idx_at(j);
      if (key != T) {
        atomicSub(&J.tile_eq[idx >> 10], 1u);
        if (key < T) continue;
        atomicAdd(&J.tile_gt[idx >> 10], 1u);
      }
      if (key > T || (short_list && idx <= last_idx)) place_selected(J, idx);
    }
  }
  if (threadIdx.x == 0) {
    st->thresh_bits = T;
    st->need = need;
    st->n_eq = n_eq;
    st->n_gt = k - need;
    st->n_selected = J.tie_all ? k - need + n_eq : k;     // the chunk scan says the same where it runs
    st->ties_left = places && !short_list ? 1u : 0u;
  }
}

// Ties of an edge list that did not fit the last workgroup's LDS, in index order: the chunk scan has
// left the ties before every chunk in tile_eq, so only the one chunk where the quota runs out has to
// rank its ties (a chunk's candidates are contiguous and index-ordered in its segment).
__device__ __forceinline__ void settle_ties_body(const ChainJob& J, uint32_t blk, uint32_t n_blk) {
  const SelState* st = J.st;
  const uint32_t T = st->thresh_bits, n_eq = st->n_eq;
  const uint32_t need = J.tie_all ? 0xFFFFFFFFu : st->need;
  walk_segments(J, (int)blk * kChunksPerBlock + wave_id(), (int)n_blk * kChunksPerBlock,
                [&](bool valid, uint32_t key, uint32_t idx, uint32_t pos) {
    if (!valid || key != T) return;
    bool on = true;
    if (need < n_eq) {
      const uint32_t c = idx >> 10;
      const uint32_t before = ld_agent(&J.tile_eq[c]);     // the scan's, in this launch
      const uint32_t upto = (int64_t)c + 1 < J.n_tiles ? ld_agent(&J.tile_eq[c + 1]) : n_eq;
      if (before >= need) {
        on = false;
      } else if (upto > need) {                           // the quota ends inside this chunk
        uint32_t rank = before;
        const uint32_t begin = pos / J.seg_cap * J.seg_cap;
        for (uint32_t q = pos; q > begin && (J.seg_idx[q - 1] >> 10) == c; --q) rank += J.seg_key[q - 1] == T;
        on = rank < need;
      }
    }
    if (on) place_selected(J, idx);
  });
}

// Single workgroup: segment counts -> offsets, validate the bracket, arm the
// candidate descent (aux) or the radix passes (st->skip == 0).
static __global__ __launch_bounds__(kBlock) void k_bracket_check(ChainJobs jobs) {
  __shared__ uint32_t s_w4[kChunksPerBlock];
  const ChainJob& J = jobs.j[blockIdx.y];
  SelState* __restrict__ st = J.st;
  SelState* __restrict__ aux = J.aux;
  uint32_t* __restrict__ seg_cnt = J.seg_cnt;
  uint32_t* __restrict__ hist = J.hist;
  constexpr int nhist = kHistStride * 2;
  const uint32_t seg_cap = J.seg_cap;
  const uint32_t* __restrict__ hi_part = J.blk_gt;
  const uint32_t* __restrict__ nf_part = J.blk_eq;
  const int spec = J.spec;
  const uint32_t ovf_cap = J.ovf_cap;
  const uint32_t* __restrict__ seg_fail = J.seg_fail;
  constexpr int PER = kSegWaves / kBlock;   // 32
  uint32_t v[PER], mine = 0, over = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    uint32_t cnt = seg_cnt[threadIdx.x * PER + j];
    if (seg_fail && cnt > seg_cap) {
      // single-sweep step: reservations are never taken back, the segment's records end where
      // the first reservation that did not fit began (the later ones went to the overflow list)
      cnt = 0xFFFFFFFFu - seg_fail[threadIdx.x * PER + j];
    }
    over |= cnt > seg_cap;                    // the sweep reserved more than the segment holds
    v[j] = cnt < seg_cap ? cnt : seg_cap;
    mine += v[j];
  }
  uint32_t total;
  uint32_t run = block_excl_scan(mine, s_w4, total);
#pragma unroll
  for (int j = 0; j < PER; ++j) { seg_cnt[threadIdx.x * PER + j] = run; run += v[j]; }
  for (int i = threadIdx.x; i < nhist; i += kBlock) hist[i] = 0u;
  static_assert(kSweepParts == kBlock, "one partial counter per thread");
  uint32_t dummy;
  __syncthreads();
  block_excl_scan(hi_part[threadIdx.x], s_w4, dummy);
  const uint32_t n_hi = dummy;
  __syncthreads();
  block_excl_scan(nf_part[threadIdx.x], s_w4, dummy);
  const uint32_t n_nf = dummy;
  __syncthreads();
  block_excl_scan(over, s_w4, dummy);
  const bool any_over = dummy != 0;
  if (threadIdx.x == 0) {
    seg_cnt[kSegWaves] = total;       // where the overflow list's records go in the dense list
    bool ovf_over = false;
    if (ovf_cap) {                    // single-sweep step: records of the shared overflow list
      const uint32_t oc = seg_cnt[kSegWaves + 1];
      ovf_over = oc > ovf_cap || (uint64_t)total + oc > (uint64_t)kSegWaves * seg_cap;
      total += oc < ovf_cap ? oc : ovf_cap;
    }
    const uint32_t k = st->k;
    const bool ok = !st->overflow && !any_over && !ovf_over && n_hi < k && k <= n_hi + total;
    st->n_hi = n_hi;
    st->cand_count = total;
    // A single-sweep step that went ahead IN PLACE has already committed on the bracket: a miss
    // cannot be repaired by the radix passes, it is reported (status 3) and nothing further
    // runs.  Out of place (spec == 2) the inputs are untouched: the miss is an ordinary failed
    // bracket, the radix passes and the key-forming final sweep redo the step over what the
    // sweep wrote, and `redone` says so.
    const bool missed = spec && st->spec && !ok;
    const bool lost = missed && spec != 2;
    if (missed && spec == 2) { st->spec = 0u; st->redone = 1u; }
    st->bracket_ok = ok ? 1u : 0u;
    st->skip = (ok || lost) ? 1u : 0u;   // the radix passes run only when the bracket failed
    st->path = ok ? (spec ? 2u : 1u) : 0u;
    st->nonfinite = ok ? n_nf : 0u;   // recounted by the radix passes otherwise
    if (!ok) st->status = lost ? 3u : 0u;
    SelState z = {};
    z.k = ok ? k - n_hi : 0u;
    z.skip = ok ? 0u : 1u;
    aux[0] = z;                       // the candidate descent runs on aux[0]
  }
}

// Dense candidate list from the per-wave segments (order: wave, then index).
static __global__ __launch_bounds__(kBlock) void k_cand_compact(ChainJobs jobs) {
  const ChainJob& J = jobs.j[blockIdx.y];
  if (J.aux->skip) return;
  const uint32_t* __restrict__ seg_off = J.seg_cnt;
  const uint32_t* __restrict__ seg_idx = J.seg_idx;
  const uint32_t* __restrict__ seg_key = J.seg_key;
  const uint32_t seg_cap = J.seg_cap;
  uint32_t* __restrict__ cand_idx = J.cand_idx;
  uint32_t* __restrict__ cand_key = J.cand_key;
  const F4* __restrict__ seg_rec = J.seg_rec;
  F4* __restrict__ cand_rec = J.cand_rec;
  for (int w = blockIdx.x * kChunksPerBlock + wave_id(); w < kSegWaves;
       w += gridDim.x * kChunksPerBlock) {
    const uint32_t off = seg_off[w], cnt = seg_off[w + 1] - off;
    for (uint32_t j = lane_id(); j < cnt; j += kWave) {
      cand_idx[off + j] = seg_idx[(int64_t)w * seg_cap + j];
      cand_key[off + j] = seg_key[(int64_t)w * seg_cap + j];
      if (seg_rec) cand_rec[off + j] = seg_rec[(int64_t)w * seg_cap + j];
    }
  }
}

// After the candidate descent: publish the exact threshold and fold each
// candidate into its chunk's (above, equal) counts.
static __global__ __launch_bounds__(kBlock) void k_cand_tiles(ChainJobs jobs) {
  const ChainJob& J = jobs.j[blockIdx.y];
  SelState* __restrict__ st = J.st;
  const SelState* __restrict__ aux = J.aux;
  if (aux->skip) return;
  const uint32_t* __restrict__ cand_idx = J.cand_idx;
  const uint32_t* __restrict__ cand_key = J.cand_key;
  uint32_t* __restrict__ tile_gt = J.tile_gt;
  uint32_t* __restrict__ tile_eq = J.tile_eq;
  const uint32_t T = aux->thresh_bits;
  const uint32_t nc = st->cand_count;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->thresh_bits = T;
    st->need = aux->need;
    st->n_eq = aux->n_eq;
    st->n_gt = st->k - aux->need;
    st->status = aux->status;
  }
  for (uint32_t j = blockIdx.x * kBlock + threadIdx.x; j < nc; j += gridDim.x * kBlock) {
    const uint32_t key = cand_key[j];
    if (key > T) atomicAdd(&tile_gt[cand_idx[j] >> 10], 1u);
    else if (key == T) atomicAdd(&tile_eq[cand_idx[j] >> 10], 1u);
  }
}
static_assert(kChunk == 1024, "candidate -> chunk mapping uses idx >> 10");

// Bit planes of the bracket sweep -> mask bytes (keys above the bracket).
// Each lane expands 16 consecutive bytes: 4 lanes x 4 elements of one slab.
static __global__ __launch_bounds__(kBlock) void k_expand_mask(
    const SelState* __restrict__ st, const uint32_t* __restrict__ pbits, int64_t n,
    uint8_t* __restrict__ mask, bool mvec, const uint32_t* __restrict__ pbits2 = nullptr) {
  if (st && !st->bracket_ok) return;
  const int64_t n_chunks = cdiv64(n, kChunk);
  const int64_t wstride = (int64_t)gridDim.x * kChunksPerBlock;
  const int l = lane_id();
  const int it = l >> 4, sl0 = (l & 15) * 4;        // slab, first slab-lane
  for (int64_t c = (int64_t)blockIdx.x * kChunksPerBlock + wave_id(); c < n_chunks; c += wstride) {
    const U4* pw = reinterpret_cast<const U4*>(pbits + c * 32 + it * 8);
    U4 lo = pw[0], hi = pw[1];
    if (pbits2) {                                   // union of two planes
      const U4* qw = reinterpret_cast<const U4*>(pbits2 + c * 32 + it * 8);
      const U4 l2 = qw[0], h2 = qw[1];
      lo = U4{lo.x | l2.x, lo.y | l2.y, lo.z | l2.z, lo.w | l2.w};
      hi = U4{hi.x | h2.x, hi.y | h2.y, hi.z | h2.z, hi.w | h2.w};
    }
    const uint32_t w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    uint32_t out[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {                   // slab-lane sl0 + j -> 4 bytes
      const int sl = sl0 + j;
      uint32_t v = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v |= (((sl < 32 ? w[2 * e] : w[2 * e + 1]) >> (sl & 31)) & 1u) << (8 * e);
      out[j] = v;
    }
    const int64_t i = c * kChunk + (int64_t)l * 16;
    if (mvec && i + 16 <= n) {
      *reinterpret_cast<U4*>(mask + i) = U4{out[0], out[1], out[2], out[3]};
    } else {
      for (int b = 0; b < 16; ++b)
        if (i + b < n) mask[i + b] = (uint8_t)((out[b >> 2] >> (8 * (b & 3))) & 1u);
    }
  }
}

// Ordered full pass that writes the mask as bit planes: where no bracket was settled (k_settle), or
// none was tried.
template <class Src>
__device__ __forceinline__ void write_bits_body(Src& src, const ChainJob& J, uint32_t T, uint32_t need, uint32_t blk,
                                                uint32_t n_blk) {
  const int64_t n = J.n;
  uint32_t* __restrict__ planes = J.planes;
  const int64_t n_chunks = cdiv64(n, kChunk);
  const int64_t wstride = (int64_t)n_blk * kChunksPerBlock;
  for (int64_t c = (int64_t)blk * kChunksPerBlock + wave_id(); c < n_chunks; c += wstride) {
    ChunkCursor cur;
    cur.sel_run = (uint32_t)uniform_i32((int)ld_agent(&J.tile_gt[c]));
    cur.eq_run = (uint32_t)uniform_i32((int)ld_agent(&J.tile_eq[c]));
    const bool full = src.vec && (c + 1) * kChunk <= n;
    uint32_t word = 0u;
#pragma unroll
    for (int it = 0; it < kChunkIters; ++it) {
      const int64_t i = c * kChunk + it * (kWave * kVec) + lane_id() * kVec;
      uint32_t key[4] = {0u, 0u, 0u, 0u};
      if (full) src.template load<true>(i, n, key);
      else if (i < n) src.template load<false>(i, n, key);
      bool valid[4], sel[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) valid[e] = full || i + e < n;
      uint32_t pos;
      slab_select(key, valid, T, need, cur, sel, pos);
      const uint32_t flag[4] = {sel[0], sel[1], sel[2], sel[3]};
      plane_collect(flag, it, word);
    }
    if (lane_id() < 32) planes[c * kPlaneWordsPerChunk + lane_id()] = word;
  }
}
template <class Src>
__global__ __launch_bounds__(kBlock) void k_write_bits(SrcPack<Src> srcs, ChainJobs jobs) {
  const ChainJob& J = jobs.j[blockIdx.y];
  Src src = srcs.s[blockIdx.y];
  write_bits_body(src, J, J.st->thresh_bits, J.tie_all ? 0xFFFFFFFFu : J.st->need, blockIdx.x, gridDim.x);
}

// All that can be left to do behind a settlement, in one launch: the radix passes over the data and the
// chunk counts (a bracket that failed or was never tried), the chunk scan (callers that pack, plateaus),
// the ties of an edge list too long for LDS, the ordered pass that writes the mask or the planes (OUT:
// 1 planes, 2 mask bytes, 0 the caller forms the keys again), the result.  Usually that is the chunk scan
// or nothing at all, and what a select paid for was nine launches that returned at once, 4.7 us each.
// With them -> in one launch: step of 40 M coordinates 450 -> 424 us, select of 1e9 1097 -> 1034, eight
// buckets of 596 M 4584 -> 4407; the radix passes themselves (sorted scores) 711 -> 324 at 20 M, 994 -> 668
// at 63 M.
//
// The steps are items of one queue: a workgroup takes the next item by its ticket, waits until every
// item of the steps before is finished, and does it.  Whoever waits holds a later ticket than those it
// waits for, which running workgroups hold, so the queue drains with any number of workgroups resident.
// The items of the scan wait for one another's totals the same way (in ticket order), through 64-bit
// words that carry the totals themselves.  All else that crosses workgroups goes by device-scope accesses,
// waited for before an item counts as finished: a cache-wide fence costs 240 ns an item, one after the other
// (the 256 tie items behind a scan, with a fence each: this launch took 59 to 72 us, 32 without, on 74.5 M
// coordinates of bf16 gradients without a residual, where 10 to 20 thousand keys equal the threshold).  The waiting
// ones look at a word of its own, away from the counter that they add to.
constexpr int kTailBlocks = 512;
constexpr int kTailStep = kHistStride + 2 * kMaxTileBlocks + 256;    // that word, in the second histogram set
constexpr int kTailRuns = kTileScanSpan + kBlock;     // a word between the threads' runs: no bank conflicts
struct TailLds {
  uint32_t h[kTailRuns];                              // a level's bins, or a scan's counters on their way
  uint32_t suf[kBlock + 1], w4[kChunksPerBlock], last, ticket;
};
// armed: the chunk counts come from this launch; read_on: items behind the scan read the prefixes in it.
__device__ __forceinline__ void tail_scan(const ChainJob& J, uint32_t b, uint32_t n_blk, bool armed, bool read_on,
                                          TailLds& s) {
  const int64_t n_tiles = J.n_tiles;
  unsigned long long* words = reinterpret_cast<unsigned long long*>(J.hist + kHistStride);
  static_assert(kTailStep < 2 * kHistStride && kHistStride % 2 == 0, "a word per workgroup of the scan");
  static_assert((int64_t)kTileScanSpan * kChunk < (1 << 23), "two totals and a flag in 64 bits");
  // counters come and go a line a wave and instruction, by LDS; a thread scans a run of sixteen.  (By runs straight
  // from and to memory the scan of 18,190 chunks spent 4.5 us on its loads and 7.8 on its stores.)
  const int64_t base = (int64_t)b * kTileScanSpan;
  // Places in LDS by offsets from two numbers that the compiler does not know ahead of the queue's loop: held in registers
  // throughout, the places cost the radix passes of scores that are chains of arithmetic half of their waves (a step by
  // `coi` on 20 M coordinates whose k-th score 0.9 M share: 1,298 us, 997 so).
  int tid = (int)threadIdx.x;
  asm volatile("" : "+v"(tid));
  constexpr int kTurn = kBlock + kBlock / kTileScanPer;
  static_assert(kBlock % kTileScanPer == 0, "word j * kBlock + i lies at j * kTurn + i + i / kTileScanPer");
  uint32_t* const line = s.h + tid + tid / kTileScanPer;
  uint32_t* const mine = s.h + tid * (kTileScanPer + 1);
  uint32_t g[kTileScanPer], e[kTileScanPer], my_g = 0, my_e = 0;
#pragma unroll
  for (int j = 0; j < kTileScanPer; ++j) {
    const int64_t at = base + j * kBlock + tid;
    const bool ok = at < n_tiles;
    g[j] = ok ? (armed ? ld_agent(&J.tile_gt[at]) : J.tile_gt[at]) : 0u;
    e[j] = ok ? (armed ? ld_agent(&J.tile_eq[at]) : J.tile_eq[at]) : 0u;
  }
  auto turn = [&](uint32_t (&v)[kTileScanPer]) {      // from a word of every line to a run
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kTileScanPer; ++j) line[j * kTurn] = v[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kTileScanPer; ++j) v[j] = mine[j];
  };
  auto put = [&](const uint32_t (&v)[kTileScanPer], uint32_t* to) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kTileScanPer; ++j) mine[j] = v[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kTileScanPer; ++j) {
      const int64_t at = base + j * kBlock + tid;
      const uint32_t w = line[j * kTurn];
      if (at >= n_tiles) continue;
      if (read_on) st_agent(&to[at], w);
      else to[at] = w;
    }
  };
  turn(g);
  turn(e);
#pragma unroll
  for (int j = 0; j < kTileScanPer; ++j) { my_g += g[j]; my_e += e[j]; }
  uint32_t tot_g, tot_e;
  uint32_t gr = block_excl_scan(my_g, s.w4, tot_g);
  uint32_t er = block_excl_scan(my_e, s.w4, tot_e);
  if (threadIdx.x == 0)
    __hip_atomic_store(&words[b], (1ull << 63) | ((unsigned long long)tot_g << 32) | tot_e, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  uint32_t pg = 0, pe = 0;
  for (uint32_t j = threadIdx.x; j < b; j += kBlock) {
    unsigned long long w;
    while ((w = __hip_atomic_load(&words[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 0ull)
      __builtin_amdgcn_s_sleep(1);
    pg += (uint32_t)(w >> 32) & 0x7FFFFFFFu;
    pe += (uint32_t)w;
  }
  uint32_t G0, E0;
  block_excl_scan(pg, s.w4, G0);
  block_excl_scan(pe, s.w4, E0);
  gr += G0;
  er += E0;
  // ties are granted in index order until `need` is used up: min(need, ties before) of them lie before a chunk
  const uint32_t need = J.tie_all ? 0xFFFFFFFFu : ld_agent(&J.st->need);
#pragma unroll
  for (int j = 0; j < kTileScanPer; ++j) {
    const uint32_t here_g = g[j], here_e = e[j];
    g[j] = gr + (er < need ? er : need);
    e[j] = er;
    gr += here_g;
    er += here_e;
  }
  put(g, J.tile_gt);
  put(e, J.tile_eq);
  // (a settlement that placed a mask has stored the number and kept no selected counts)
  if (b == n_blk - 1 && threadIdx.x == 0 && !(J.mask_only && J.st->bracket_ok)) {
    const uint32_t E = E0 + tot_e;
    st_agent(&J.st->n_selected, G0 + tot_g + (E < need ? E : need));
  }
}
template <class Src, int LEVEL>
__device__ __forceinline__ void tail_level(Src& src, const ChainJob& J, uint32_t blk, uint32_t n_blk, TailLds& s) {
  uint32_t* gh = level_hist_of<LEVEL>(J.hist);
  level_hist_body<Src, LEVEL>(src, J.n, LEVEL == 0 ? 0u : ld_agent(&J.st->prefix), gh, s.h, blk, n_blk);
  if (!level_last(&J.st->done[LEVEL], n_blk, &s.last)) return;
  level_scan_body<LEVEL>(J.st, gh, s.suf);
  __threadfence();
}
template <class Src, int OUT>
__global__ __launch_bounds__(kBlock) void k_tail(SrcPack<Src> srcs, ChainJobs jobs) {
  __shared__ TailLds s;
  const ChainJob& J = jobs.j[blockIdx.y];
  SelState* st = J.st;
  // none of these changes while the queue is worked off
  const bool armed = st->skip == 0, ties = st->ties_left != 0, write = OUT != 0 && !st->bracket_ok;
  const uint32_t G = gridDim.x;
  const uint32_t n_pass = armed ? G : 0u, n_ties = ties ? (G < 256u ? G : 256u) : 0u, n_write = write ? G : 0u;
  const uint32_t n_scan = J.mask_only && st->bracket_ok && !ties ? 0u : (uint32_t)cdiv64(J.n_tiles, kTileScanSpan);
  const uint32_t at_scan = 4u * n_pass, at_ties = at_scan + n_scan, at_write = at_ties + n_ties;
  const uint32_t total = at_write + n_write;
  if (total == 0) {
    if (blockIdx.x == 0 && threadIdx.x == 0) write_result(J);
    return;
  }
  const bool once = !armed && !write && total <= G;                   // a workgroup per item is enough
  if (once && blockIdx.x >= total) return;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) s.ticket = atomicAdd(&st->tail_ticket, 1u);
    __syncthreads();
    const uint32_t t = s.ticket;
    if (t >= total) return;
    const uint32_t first = t >= at_ties ? at_ties : t >= at_scan ? at_scan : t / G * G;
    if (first) {
      if (threadIdx.x == 0)
        while (ld_agent(&J.hist[kTailStep]) < first) __builtin_amdgcn_s_sleep(4);
      __syncthreads();
    }
    Src src = srcs.s[blockIdx.y];
    if (t < at_scan) {
      const uint32_t step = t / G, blk = t - first;
      if (step == 0) tail_level<Src, 0>(src, J, blk, G, s);
      else if (step == 1) tail_level<Src, 1>(src, J, blk, G, s);
      else if (step == 2) tail_level<Src, 2>(src, J, blk, G, s);
      else tile_count_body(src, J, ld_agent(&st->thresh_bits), 0, (int64_t)blk * kChunksPerBlock + wave_id(),
                           (int64_t)G * kChunksPerBlock);
    } else if (t < at_ties) {
      tail_scan(J, t - first, n_scan, armed, at_ties != total, s);
    } else if (t < at_write) {
      settle_ties_body(J, t - first, n_ties);
    } else if (OUT != 0) {
      const uint32_t T = ld_agent(&st->thresh_bits), need = J.tie_all ? 0xFFFFFFFFu : ld_agent(&st->need);
      if (OUT == 1) write_bits_body(src, J, T, need, t - first, n_write);
      else write_mask_body(src, J, T, need, 0, J.mask, t - first, n_write);
    }
    if (t >= at_ties) {                                               // nothing in this launch reads what these wrote
      if (once) return;
      continue;
    }
    wait_landed();
    if (threadIdx.x == 0) {
      const uint32_t done = atomicAdd(&st->tail_done, 1u) + 1u;
      if (done == at_ties) write_result(J);                           // settled with the scan's last item
      if (done == at_ties || (done <= at_scan && done % G == 0)) st_agent(&J.hist[kTailStep], done);
    }
    if (once) return;
  }
}

// Byte mask -> bit planes (chunk-structured, planes sized for cdiv(n, 1024) chunks).
static __global__ __launch_bounds__(kBlock) void k_mask_to_planes(const uint8_t* __restrict__ mask,
                                                                  int64_t n,
                                                                  uint32_t* __restrict__ planes,
                                                                  bool mvec) {
  const int64_t n_chunks = cdiv64(n, kChunk);
  const int64_t wstride = (int64_t)gridDim.x * kChunksPerBlock;
  for (int64_t c = (int64_t)blockIdx.x * kChunksPerBlock + wave_id(); c < n_chunks; c += wstride) {
    uint32_t word = 0u;
#pragma unroll
    for (int it = 0; it < kChunkIters; ++it) {
      const int64_t i = c * kChunk + it * (kWave * kVec) + lane_id() * kVec;
      uint32_t mk[4] = {0u, 0u, 0u, 0u};
      if (i < n) load4_u8(mask, i, n, mk, mvec);
      plane_collect(mk, it, word);
    }
    if (lane_id() < 32) planes[c * kPlaneWordsPerChunk + lane_id()] = word;
  }
}

// The select of every job of a batch: begin -> (sampled-bracket path: coarse sample and pick, fine sample
// and pick, ONE data sweep per job, settlement) -> k_tail.  The short kernels run once for the whole
// batch; only the data sweeps are launched per job.
// Src::kSweep: what the sweep leaves behind -- 0 nothing, 1 the keys above the bracket as bit planes
// (job.planes), 2 as mask bytes (job.mask) -- where the settlement adds the candidates; the tail's
// writing pass over the data then has nothing to do.
// All jobs of a batch take the same path (`fast`: SelBatch::fast_ok for every one of them).
//
// The chain comes in phases so that a batch whose jobs form their keys differently (the
// re-selections of a replay step rank by different scores) still shares every kernel that does
// not form keys: chain_begin and chain_settle take the whole batch; launch_sample_*,
// chain_sweeps and chain_tail are templates of the key source and take the jobs of one kind (a sub-batch
// over the same workspaces).
static inline void chain_begin(const SelBatch& B, const SegDirJobs& dirs, hipStream_t s) {
  static_assert(sizeof(ChainJobs) + sizeof(SegDirJobs) + 64 <= 4096, "operands travel in the kernel arguments");
  hipLaunchKernelGGL(k_chain_begin, B.grid(4), dim3(kBlock), 0, s, B.jobs, dirs);
}
// Number of the next launch that takes a sample: one count for the whole library (select.hip).
uint32_t next_launch();
template <class Src>
static inline void launch_sample_pick(const SrcPack<Src>& srcs, const SelBatch& B, const SegDirJobs& dirs,
                                      const typename Src::Cols& cols, double sigmas, hipStream_t s) {
  static_assert(sizeof(ChainJobs) + sizeof(SrcPack<Src>) + sizeof(SegDirJobs) + sizeof(typename Src::Cols) + 64 <= 4096,
                "the operands of a batched chain kernel travel in its 4 KiB of kernel arguments");
  hipLaunchKernelGGL((k_sample_pick<Src>), B.grid(kSampleGroups + 16), dim3(kWide), 0, s, srcs, B.jobs, dirs, cols,
                     next_launch(), sigmas);
}
template <class Src>
static inline void launch_sample_fine(const SrcPack<Src>& srcs, const SelBatch& B, double sigmas, hipStream_t s) {
  hipLaunchKernelGGL((k_sample_fine<Src>), B.grid((unsigned)cdiv64(B.max_nsv, kBlock)), dim3(kBlock), 0, s, srcs,
                     B.jobs, sigmas);
}
// begin ... bracket, for a batch of one key source
template <class Src>
static inline void chain_bracket(const SrcPack<Src>& srcs, const SelBatch& B, const SegDirJobs& dirs,
                                 const typename Src::Cols& cols, double sigmas, hipStream_t s) {
  launch_sample_pick(srcs, B, dirs, cols, sigmas, s);
  launch_sample_fine(srcs, B, sigmas, s);
}
// keep (sources that a writing pass reads again): see bracket_chunk
template <class Src>
static inline void chain_sweeps(const SrcPack<Src>& srcs, const SelBatch& B, hipStream_t s, bool keep = false) {
  constexpr int PM = Src::kSweep;
  for (int b = 0; b < B.count; ++b) {
    const ChainJob& J = B.jobs.j[b];
    const SelWorkspace& w = B.w[b];
    const unsigned sweep_blocks = (unsigned)cdiv64(J.n_tiles, kChunksPerBlock);
    ProfPair* pp = prof_begin(SGA_PROF_SELECT_SWEEP, s);
    // the sweep's two totals go through 256 partial counters (blk_gt / blk_eq are free until
    // the tile scan, which runs after the settlement has read them)
    auto sweep = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(sweep_blocks), dim3(kBlock), 0, s, srcs.s[b], J.n, w.st, w.rel, w.tile_gt,
                         w.tile_eq, w.seg_idx, w.seg_key, w.seg_cnt, (uint32_t)w.seg_cap,
                         PM == 1 ? J.planes : (uint32_t*)nullptr, w.blk_gt, w.blk_eq,
                         PM == 2 ? J.mask : (uint8_t*)nullptr, true);
    };
    if (Src::kReadAgain && keep) sweep(k_bracket_sweep<Src, PM, Src::kReadAgain>);
    else sweep(k_bracket_sweep<Src, PM>);
    prof_end(pp, s);
  }
}
static inline void chain_settle(const SelBatch& B, hipStream_t s) {
  // The work is the random atomics and stores of about n / 800 candidates: a workgroup per 4 M coordinates,
  // no fewer than hold every segment at once (64; a batch shares them), no more than the chip has CUs.
  const int64_t want = B.max_n >> 22, least = B.count > 1 ? 32 : 64;
  const unsigned wgs = (unsigned)(want < least ? least : want > 256 ? 256 : want);
  hipLaunchKernelGGL(k_settle, B.grid(wgs), dim3(kWide), 0, s, B.jobs);
}
// OUT: what the ordered pass over the data writes where no bracket settled it (k_tail)
template <int OUT, class Src>
static inline void chain_tail(const SrcPack<Src>& srcs, const SelBatch& B, hipStream_t s) {
  const unsigned wgs = stream_grid(B.max_n, kTileScanSpan, kTailBlocks);
  hipLaunchKernelGGL((k_tail<Src, OUT>), B.grid(wgs), dim3(kBlock), 0, s, srcs, B.jobs);
}

template <int OUT, class Src>
static inline void run_select_batch(const SrcPack<Src>& srcs, const SelBatch& B, const SegDirJobs& dirs,
                                    const typename Src::Cols& cols, bool fast, hipStream_t s, bool keep = false) {
  if (fast) {
    chain_bracket(srcs, B, dirs, cols, kBracketSigmas, s);
    chain_sweeps(srcs, B, s, keep);
    chain_settle(B, s);
  } else {
    chain_begin(B, dirs, s);
  }
  chain_tail<OUT>(srcs, B, s);
}

#endif  // __HIPCC__
}  // namespace sga
