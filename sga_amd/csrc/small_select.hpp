// Exact top-k of a bucket of up to kSmallTiles chunks (8.4 M coordinates) in three launches:
//   k_sample_pick     8 K to 16 K sample keys, and the bracket of the k-th key from them (and the
//                     directory of the segment table)
//   k_small_sweep     the one sweep over the data: per-chunk counts above the bracket, and a list
//                     of the few keys inside it
//   k_small_finish    one workgroup: exact threshold from the list, ties to grant, and the
//                     per-chunk (selected, ties) prefixes the writing pass starts from
// followed by the caller's writing pass (final sweep, k_write_mask, k_write_bits), which forms the
// keys again: the whole bucket sits in L2 / Infinity Cache then.
//
// Why not the chain of the large buckets (select_impl.hpp): that is five dependent
// launches beside the sweep (twenty, 150 us, when this path was written) and half-empty grids,
// where the data of a 4 M-element bucket takes 24 us.  One workgroup is enough for what lies
// between the sweeps as long as the chunk counts fit its LDS, which draws the line at kSmallTiles
// (8 M coordinates at 1 %: 30 us in k_small_finish, as much as the sweep and a half).
// Measured through the public entry points, us per call, before -> with this path:
//   fused step, |g + r|, 1 %, 261 K elements bf16   84 -> 55       4.2 M elements fp32   184 -> 91
//   select_topk_flat, 3 M scores, 1 %              168 -> 69
// (Kernels of the 4.2 M step, fp32 gradients, each pass after a wait: sample and pick 12.5 us, sweep 11.4, finish
// 20.6, final sweep 27.2.)
//
// The result is exact for any sample: where the bracket misses the k-th key the finishing launch goes
// over the data itself, with all of its workgroups (small_redo).
#pragma once
#include "select_impl.hpp"

namespace sga {

#ifdef __HIPCC__

// Candidate lists of the small path: the chunks of the sweep share kSmallSegs counters (the segments of
// the list); a segment has room for every coordinate of its chunks, so it never overflows.
// The counters lie 256 bytes apart: atomics on one cache line queue like those on one address (11 ns
// each; 1024 workgroups on 16 adjacent words: the sweep of 4 M elements took 19 us, 8.6 with this).
struct SmallGeom { uint32_t segs, cap; };          // cap: list entries per segment
__host__ __device__ static inline SmallGeom small_geom(int64_t n_tiles, int cpw) {
  SmallGeom s;
  const uint32_t n_wg = (uint32_t)cdiv64(n_tiles, cpw), per = (uint32_t)cdiv64(n_wg, kSmallSegs);
  s.segs = (uint32_t)cdiv64(n_wg, per);
  s.cap = (per * cpw < 2 ? 2 : per * cpw) * (uint32_t)kChunk;      // two chunks hold the head that is read unseen
  return s;
}

// The sweep: a workgroup per chunk and a wave per slab, so that a bucket of a few hundred chunks still
// reaches every SIMD; counts above the bracket, keys inside it to the list (one reservation per chunk).
// Keys equal to the bracket's lower end are counted per chunk and not
// listed: a plateau of equal keys (zeros, momenta that have decayed to the last denormal) puts the
// lower end on itself, and the one workgroup behind the sweep would walk a list as long as the bucket
// (|m| after a thousand sparse steps, 1.7 M coordinates: 889 us, 86 like this).
// Chunks per workgroup (CPW): one up to kSweepTiles chunks and for the scores that are a chain of arithmetic;
// beyond, four, whose loads are in flight together (a reservation per 4096 coordinates, half the waves).
// Step of 261 K coordinates with one / four 36.1 / 38.8 us, 2 M 59.2 / 62.3, 8.3 M 145 / 140; `update`
// 261 K 50.5 / 57.4, 8.3 M 159 / 166; select of 3 M scores 70.4 / 67.4.
constexpr int64_t kSweepTiles = 2048;
template <class Src, int CPW>
__global__ __launch_bounds__(kBlock) void k_small_sweep(SrcPack<Src> srcs, ChainJobs jobs) {
  const ChainJob& J = jobs.j[blockIdx.y];
  const int64_t n = J.n, n_chunks = J.n_tiles, c0 = (int64_t)blockIdx.x * CPW;
  if (c0 >= n_chunks) return;                         // a smaller job of the batch
  __shared__ uint32_t s_hi[CPW][kChunkIters], s_eq[CPW][kChunkIters], s_cnt[kChunkIters], s_nf[kChunkIters], s_base;
  static_assert(kChunkIters == kChunksPerBlock && CPW <= kWave, "a wave per slab");
  SelState* __restrict__ st = J.st;
  if (blockIdx.x == 0 && threadIdx.x < kSampleGroups) st->sampled[threadIdx.x] = 0u;      // see launch_number
  Src src = srcs.s[blockIdx.y];
  const int64_t i0 = c0 * kChunk + uniform_i32(wave_id()) * (kWave * kVec);
  typename Src::Raw raw[CPW];
#pragma unroll
  for (int u = 0; u < CPW; ++u) {
    const typename Src::Chunk ck = src.chunk_begin(c0 + u);
    const int64_t i = i0 + u * kChunk + lane_id() * kVec;
    if (src.vec && (c0 + u + 1) * kChunk <= n) src.template fetch<true, true>(ck, i, n, raw[u]);  // read again soon
    else if (i < n) src.template fetch<false>(ck, i, n, raw[u]);
  }
  src.slab_hyper(i0);
  const uint32_t T_LO = st->t_lo, T_HI = st->t_hi;
  uint32_t key[CPW][4], cnt = 0, nf = 0;
  Ballot4 cand[CPW];
#pragma unroll
  for (int u = 0; u < CPW; ++u) {
    const typename Src::Chunk ck = src.chunk_begin(c0 + u);
    const int64_t i = i0 + u * kChunk + lane_id() * kVec;
    const bool full = src.vec && (c0 + u + 1) * kChunk <= n;
    if (u > 0) src.slab_hyper(i0 + u * kChunk);
    key[u][0] = key[u][1] = key[u][2] = key[u][3] = 0u;
    if (full) src.template keys<true>(ck, i, n, raw[u], key[u]);
    else if (i < n) src.template keys<false>(ck, i, n, raw[u], key[u]);
    uint32_t hi = 0, eq = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint64_t valid = full ? ~0ull : ballot64(i + e < n);
      const uint64_t above = ballot64(key[u][e] >= T_HI) & valid;
      cand[u].m[e] = ballot64(key[u][e] > T_LO) & valid & ~above;
      hi += (uint32_t)__popcll(above);
      eq += (uint32_t)__popcll(ballot64(key[u][e] == T_LO) & valid);
      nf += (uint32_t)__popcll(ballot64(key[u][e] >= 0x7F800000u) & valid);
    }
    cnt += cand[u].count();
    if (lane_id() == 0) { s_hi[u][wave_id()] = hi; s_eq[u][wave_id()] = eq; }
  }
  const bool neg = ballot64(src_negative(src) != 0u) != 0ull;
  if (lane_id() == 0) {
    s_cnt[wave_id()] = cnt;
    s_nf[wave_id()] = nf | (neg ? 0x80000000u : 0u);
  }
  __syncthreads();
  const SmallGeom geo = small_geom(n_chunks, CPW);
  const uint32_t seg = blockIdx.x % geo.segs;
  if (threadIdx.x < CPW && c0 + (int)threadIdx.x < n_chunks) {
    const uint32_t* h = s_hi[threadIdx.x];
    const uint32_t* q = s_eq[threadIdx.x];
    J.tile_gt[c0 + threadIdx.x] = h[0] + h[1] + h[2] + h[3];
    J.tile_eq[c0 + threadIdx.x] = q[0] + q[1] + q[2] + q[3];
  }
  if (threadIdx.x == 0) {
    const uint32_t all = s_cnt[0] + s_cnt[1] + s_cnt[2] + s_cnt[3];
    const uint32_t f = (s_nf[0] + s_nf[1] + s_nf[2] + s_nf[3]) & 0x7FFFFFFFu;
    if (all) s_base = atomicAdd(&J.seg_cnt[seg * kSmallSegStride], all);
    if (f) atomicAdd(&st->nonfinite, f);
    if ((s_nf[0] | s_nf[1] | s_nf[2] | s_nf[3]) & 0x80000000u) raise_negative(st);
  }
  __syncthreads();
  uint32_t run = seg * geo.cap + s_base;
  for (int w = 0; w < wave_id(); ++w) run += s_cnt[w];
#pragma unroll
  for (int u = 0; u < CPW; ++u)
    ballot_append(cand[u], run, [&](uint32_t pos, int e) {
      J.small_idx[pos] = (uint32_t)(i0 + u * kChunk + lane_id() * kVec + e);
      J.small_key[pos] = key[u][e];
    });
}

// The candidate list as the finishing workgroup sees it: wave w owns segment w (kSmallSegs ==
// kWideWaves).  The first kSmallHead quads per lane of every segment are requested before anything is
// known about it -- together with the counters they are then one memory latency instead of three --
// and stay in registers for both passes; a longer segment is read on from L2.  Entries past the
// segment's count become the key ~0: its offset from any bracket end has the top bit set, like that of
// a key below the bracket, and no pass takes it.
constexpr int kSmallHead = 5;                         // 16 waves x 64 lanes x 5 x 4 = 20 K entries
struct SmallList {
  const U4* keys;
  const U4* idxs;
  uint32_t cnt;
  U4 key[kSmallHead], idx[kSmallHead];
  __device__ __forceinline__ void request(const ChainJob& J, const SmallGeom& geo) {
    static_assert(kSmallSegs == kWideWaves, "one list segment per wave");
    keys = reinterpret_cast<const U4*>(J.small_key + (int64_t)wave_id() * geo.cap);
    idxs = reinterpret_cast<const U4*>(J.small_idx + (int64_t)wave_id() * geo.cap);
    const bool mine = (uint32_t)wave_id() < geo.segs;   // a segment has room for 2048 entries at least
#pragma unroll
    for (int u = 0; u < kSmallHead; ++u)
      if (mine) { key[u] = keys[u * kWave + lane_id()]; idx[u] = idxs[u * kWave + lane_id()]; }
  }
  static __device__ __forceinline__ void trim(U4& k, uint32_t j, uint32_t cnt) {
    k.x = j < cnt ? k.x : ~0u;
    k.y = j + 1 < cnt ? k.y : ~0u;
    k.z = j + 2 < cnt ? k.z : ~0u;
    k.w = j + 3 < cnt ? k.w : ~0u;
  }
  __device__ __forceinline__ void counted(uint32_t c) {
    cnt = c;
#pragma unroll
    for (int u = 0; u < kSmallHead; ++u) trim(key[u], (uint32_t)(u * kWave + lane_id()) * kVec, c);
  }
  // head(key, idx) over the entries in registers, tail(keys, idxs) over rounds of quads of the rest (whole waves).
  // IDX: the index is wanted; without it twice as many keys are in flight.  The rest comes from other XCDs' stores, a microsecond
  // a round of loads, so the next round is on its way while one is worked off.
  template <bool IDX, class H, class T>
  __device__ __forceinline__ void visit(H&& head, T&& tail) const {
#pragma unroll
    for (int u = 0; u < kSmallHead; ++u) {
      if ((uint32_t)(u * kWave * kVec) >= cnt) return;  // wave-uniform
      head(key[u].x, idx[u].x); head(key[u].y, idx[u].y); head(key[u].z, idx[u].z); head(key[u].w, idx[u].w);
    }
    visit_tail<IDX>(tail);
  }
  template <bool IDX, class T>
  __device__ __forceinline__ void visit_tail(T&& tail) const {
    constexpr int U = IDX ? 2 : 4;
    U4 k2[U], i2[U];
    auto request_from = [&](uint32_t q0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t q = q0 + u * kWave + lane_id();
        k2[u] = U4{~0u, ~0u, ~0u, ~0u};
        if (q * kVec < cnt) { k2[u] = keys[q]; if (IDX) i2[u] = idxs[q]; }
      }
    };
    constexpr uint32_t q_first = kSmallHead * kWave;
    if (q_first * kVec < cnt) request_from(q_first);
    for (uint32_t q0 = q_first; q0 * kVec < cnt; q0 += U * kWave) {
      U4 k[U], i[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        k[u] = k2[u];
        i[u] = IDX ? i2[u] : U4{0u, 0u, 0u, 0u};
        trim(k[u], (q0 + u * kWave + lane_id()) * kVec, cnt);
      }
      if ((q0 + U * kWave) * kVec < cnt) request_from(q0 + U * kWave);
      tail(k, i);
    }
  }
  template <int U, class F>
  static __device__ __forceinline__ void each(const U4 (&k)[U], const U4 (&i)[U], F&& f) {
#pragma unroll
    for (int u = 0; u < U; ++u) { f(k[u].x, i[u].x); f(k[u].y, i[u].y); f(k[u].z, i[u].z); f(k[u].w, i[u].w); }
  }
  // quad(key, idx) over all entries, four of a lane at a time.
  template <class F>
  __device__ __forceinline__ void visit_quads(F&& quad) const {
#pragma unroll
    for (int u = 0; u < kSmallHead; ++u) {
      if ((uint32_t)(u * kWave * kVec) >= cnt) return;  // wave-uniform
      quad(key[u], idx[u]);
    }
    visit_tail<true>([&](const auto& k, const auto& i) {
#pragma unroll
      for (int u = 0; u < (int)(sizeof(k) / sizeof(k[0])); ++u) quad(k[u], i[u]);
    });
  }
};
// Adds the numbers of a lane's four neighbouring entries to their chunks' words.  A chunk's entries follow one
// another in the list, eleven and more of them, so the four mostly share a chunk, and two at most all but always;
// an add per entry queues on the word that its neighbours add to: selects in a row, an add per entry / this, us: 3 M
// scores at 1 % (25 K entries) 36.6 / 35.3, 8 M (79 K) 62.8 / 58.4, 10 % (206 K) 105.7 / 96.3.  A number of zero has
// no index to speak of.
__device__ __forceinline__ void quad_add(uint32_t* s_tile, const U4& idx, const U4& num) {
  const uint32_t c0 = idx.x >> 10, c1 = idx.y >> 10, c2 = idx.z >> 10, c3 = idx.w >> 10;
  const bool a1 = c1 == c0, a2 = c2 == c0, a3 = c3 == c0, b1 = !a1 && c1 == c3, b2 = !a2 && c2 == c3;
  const uint32_t first = num.x + (a1 ? num.y : 0u) + (a2 ? num.z : 0u) + (a3 ? num.w : 0u);
  const uint32_t last = (a3 ? 0u : num.w) + (b1 ? num.y : 0u) + (b2 ? num.z : 0u);
  if (first) atomicAdd(&s_tile[c0], first);
  if (last) atomicAdd(&s_tile[c3], last);
  if (!a1 && !b1 && num.y) atomicAdd(&s_tile[c1], num.y);
  if (!a2 && !b2 && num.z) atomicAdd(&s_tile[c2], num.z);
}
static_assert(kSmallHead * kWave * kVec <= 2 * kChunk, "the head never reaches past a segment");

// A bracket that missed: the radix descent and the chunk counts over the data itself, as items of one
// queue that every workgroup of the launch works on (the way of k_tail: whoever waits holds a later
// ticket than those it waits for, so any number of resident workgroups will do).  True in the workgroup
// that finished the last item: it finds the threshold in the state and the counts per chunk in tile_gt /
// tile_eq.
// The margin is five sigma of independent keys, but the sample is drawn by quads: scores that neighbours
// share miss about once in a hundred times.  One workgroup alone took 5.9 ms for such a select of 8.4 M
// coordinates, the launch takes 0.21 (a bracket that holds: 0.10).
constexpr int kRedoGroups = 64;                       // at most; one per kRedoTiles chunks
constexpr int kRedoTiles = 32;
constexpr uint32_t kCrowdedList = 1 << 16;            // shorter lists are walked in less time than the passes take
                                                      // (0.9 us a thousand keys of a plateau, 50 to 190 us the passes)
template <class Src>
__device__ __forceinline__ bool small_redo(Src& src, const ChainJob& J, uint32_t* s_hist, WideScratch& s_scan,
                                           uint32_t* s_word) {
  SelState* st = J.st;
  const int64_t n = J.n;
  const uint32_t G = gridDim.x;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) *s_word = atomicAdd(&st->tail_ticket, 1u);
    __syncthreads();
    const uint32_t t = *s_word, step = t / G, blk = t % G;
    if (step > 3) return false;
    if (step) {
      if (threadIdx.x == 0)
        while (ld_agent(&st->redo_step) < step) __builtin_amdgcn_s_sleep(16);
      __syncthreads();
    }
    const uint32_t prefix = step ? ld_agent(&st->prefix) : 0u;
    const int shift = step == 0 ? kL0Shift : step == 1 ? kL1Shift : 0;
    const int above = step == 0 ? 31 : step == 1 ? kL0Shift : kL1Shift, bits = above - shift;
    uint32_t* gh = J.hist + (step == 0 ? 0 : step == 1 ? kBinsBig : 2 * kBinsBig);
    if (step == 3) {
      tile_count_body(src, J, prefix, 0, (int64_t)blk * kWideWaves + wave_id(), (int64_t)G * kWideWaves);
    } else {
      reinterpret_cast<U4*>(s_hist)[threadIdx.x] = U4{0u, 0u, 0u, 0u};
      __syncthreads();
      constexpr int U = 4;                            // quads in flight per thread
      constexpr int64_t kSlab = (int64_t)kWide * kVec;
      for (int64_t base = (int64_t)blk * kSlab * U; base < n; base += (int64_t)G * kSlab * U) {
        uint32_t key[U][4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int64_t b = base + u * kSlab, i = b + (int64_t)threadIdx.x * kVec;
          key[u][0] = key[u][1] = key[u][2] = key[u][3] = 0u;
          if (src.vec && b + kSlab <= n) src.template load<true>(i, n, key[u]);
          else if (i < n) src.template load<false>(i, n, key[u]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int64_t i = base + u * kSlab + (int64_t)threadIdx.x * kVec;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            wide_hist_add(s_hist, (key[u][e] >> shift) & ((1u << bits) - 1u),
                          i + e < n && (key[u][e] >> above) == prefix);
        }
      }
      __syncthreads();
      for (int b = threadIdx.x; b < (1 << bits); b += kWide)
        if (const uint32_t c = s_hist[b]) atomicAdd(&gh[b], c);
    }
    wait_landed();
    if (threadIdx.x == 0) *s_word = atomicAdd(&st->tail_done, 1u) + 1u;
    __syncthreads();
    if (*s_word != (step + 1u) * G) continue;
    if (step == 3) return true;
    for (int b = threadIdx.x; b < kWideBins; b += kWide) s_hist[b] = b < (1 << bits) ? ld_agent(&gh[b]) : 0u;
    const uint32_t want[1] = {step ? ld_agent(&st->krem) : J.k};
    __syncthreads();
    RankHit h[1];
    wide_find_rank<1>(s_hist, want, s_scan, (int)(step & 1u), h);
    if (threadIdx.x == 0) {
      st_agent(&st->prefix, (prefix << bits) | h[0].bin);
      st_agent(&st->krem, want[0] - h[0].above);
      st_agent(&st->n_eq, h[0].count);
    }
    wait_landed();
    if (threadIdx.x == 0) st_agent(&st->redo_step, step + 1u);
  }
}

template <class Src>
__global__ __launch_bounds__(kWide) void k_small_finish(SrcPack<Src> srcs, ChainJobs jobs, int cpw) {
  __shared__ __align__(16) uint32_t s_hist[kBinsBig];
  __shared__ __align__(16) uint32_t s_tile[kSmallTiles];          // above | ties << 16, at most 1024 each
  __shared__ __align__(16) uint32_t s_key[kWideList];
  __shared__ uint32_t s_idx[kWideList];
  __shared__ uint32_t s_seg[kWideWaves], s_cnt, s_out[3], s_word;
  __shared__ WideScratch s_scan;
  const ChainJob& J = jobs.j[blockIdx.y];
  SelState* st = J.st;
  const int64_t n = J.n;
  const int nt = (int)J.n_tiles;
  const uint32_t k = J.k, T_LO = st->t_lo, T_HI = st->t_hi;
  const bool single = T_HI - T_LO == 1u;
  const SmallGeom geo = small_geom(nt, cpw);
  SmallList list;
  list.request(J, geo);
  constexpr int PER = kSmallTiles / kWide;            // 8
  uint32_t g8[PER], e8[PER], hi = 0, eqs = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int t = j * kWide + threadIdx.x;
    g8[j] = e8[j] = 0u;
    if (j * kWide < nt && t < nt) { g8[j] = J.tile_gt[t]; e8[j] = J.tile_eq[t]; }
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    s_tile[j * kWide + threadIdx.x] = g8[j] | (e8[j] << 16);
    hi += g8[j];
    eqs += e8[j];
  }
  reinterpret_cast<U4*>(s_hist)[threadIdx.x] = U4{0u, 0u, 0u, 0u};
  if (threadIdx.x < kWideWaves)
    s_seg[threadIdx.x] = threadIdx.x < geo.segs ? J.seg_cnt[threadIdx.x * kSmallSegStride] : 0u;
  if (threadIdx.x == 0) {
    s_cnt = 0u;
    s_word = gridDim.x > 1 ? atomicAdd(&st->finish_ticket, 1u) : 0u;
  }
  // The first workgroup to begin judges the bracket and usually does all the rest; the others wait for its
  // word (it is running, so they need not fit the chip beside it) and go.
  __syncthreads();
  const bool judge = s_word == 0u;
  if (!judge) {
    if (threadIdx.x == 0) {
      uint32_t v;
      while ((v = ld_agent(&st->verdict)) == 0u) __builtin_amdgcn_s_sleep(8);
      s_cnt = v;
    }
    __syncthreads();
    if (s_cnt == 1u) return;
  }
  uint32_t n_hi, n_low, n_list;
  wide_totals(hi, eqs, s_scan, n_hi, n_low);
  wide_waves_before(s_seg, n_list);
  list.counted(s_seg[wave_id()]);
  // A list far longer than its margin says holds a plateau that one workgroup should not walk (keys equal
  // to the upper end are listed): two values, k near where they change, 8.4 M coordinates: half of them
  // on the upper one 5.7 ms, a tenth 1.06; by passes over the data 0.29 and 0.32.  Independent scores list
  // 1.0 to 1.25 times what the margin says (the bracket ends at bin edges).
  bool crowded = false;
  if (n_list > kCrowdedList) {
    const double ns = (double)(small_sample_vecs(n) * 4);
    const RankEnds f = bracket_ranks((double)k, (double)n, ns, kBracketSigmas);
    crowded = (double)n_list * ns > 2.0 * (f.lo - f.hi) * (double)n;
  }
  const bool ok = judge && !crowded && n_hi < k && k <= n_hi + n_list + n_low;
  if (judge && gridDim.x > 1 && ok && threadIdx.x == 0) st_agent(&st->verdict, 1u);
  const bool low = ok && k > n_hi + n_list;           // the lower end is the threshold
  uint32_t T = T_LO, need = k - n_hi - n_list, n_eq = n_low;
  int turn = 0;
  if (low) {
    list.visit_quads([&](const U4& key, const U4& idx) {
      quad_add(s_tile, idx, U4{key.x != ~0u, key.y != ~0u, key.z != ~0u, key.w != ~0u});
    });
    __syncthreads();
  } else if (ok) {
    // the lower end is below the threshold: its members are no ties
#pragma unroll
    for (int j = 0; j < PER; ++j) s_tile[j * kWide + threadIdx.x] = g8[j];
    // descent over the list inside (T_LO, T_HI): 4096 bins per level, until one bin is left whose
    // keys fit the short list (nearly always after the first level) or are all equal
    uint32_t lo = T_LO + 1u, rank = k - n_hi;
    int w = 32 - __clz((int)(T_HI - 1u - lo));         // bits of the offset (the list is not empty)
    for (;;) {
      const int sh = w > 12 ? w - 12 : 0;
      auto count = [&](uint32_t key, uint32_t) {
        const uint32_t off = key - lo;
        if (off >> w == 0u) atomicAdd(&s_hist[off >> sh], 1u);
      };
      // A plateau in a long list queues on its bin: where sixteen lanes' first keys of a round share one, the lanes
      // of that bin add together.  8.4 M coordinates, plateaus inside the bracket, plain adds / this: at 1 % 256 / 180
      // and 295 / 181 us, at 10 % 564 / 272; without plateaus 96.7 / 96.5 and 132.6 / 133.1 (to ask for every key: 146).
      auto count_round = [&](const auto& k, const auto& i) {
        const uint32_t first = k[0].x - lo, lead = (uint32_t)uniform_i32((int)(first >> sh));
        if (__popcll(ballot64(first >> w == 0u && first >> sh == lead)) < 16) {
          SmallList::each(k, i, count);
        } else {
          SmallList::each(k, i, [&](uint32_t key, uint32_t) {
            const uint32_t off = key - lo;
            const bool in = off >> w == 0u, with = in && off >> sh == lead;
            const uint32_t same = (uint32_t)__popcll(ballot64(with));
            if (same && lane_id() == 0) atomicAdd(&s_hist[lead], same);
            if (in && !with) atomicAdd(&s_hist[off >> sh], 1u);
          });
        }
      };
      list.visit<false>(count, count_round);
      __syncthreads();
      const uint32_t want[1] = {rank};
      RankHit h[1];
      wide_find_rank<1>(s_hist, want, s_scan, turn, h);
      turn ^= 1;
      rank -= h[0].above;
      lo += h[0].bin << sh;
      n_eq = h[0].count;
      w = sh;
      if (sh == 0 || n_eq <= (uint32_t)kWideList) break;
      reinterpret_cast<U4*>(s_hist)[threadIdx.x] = U4{0u, 0u, 0u, 0u};
      __syncthreads();
    }
    // one pass with the indices: keys above the bin are selected, the bin's own go to the short list
    // (a bin of one key value, of any size, are the ties)
    const bool ties_only = w == 0;
    const uint32_t width = 1u << w;
    if (ties_only) {
      auto num = [&](uint32_t key) {
        const uint32_t off = key - lo;
        return (int32_t)off < 0 ? 0u : off < width ? 1u << 16 : 1u;
      };
      list.visit_quads([&](const U4& key, const U4& idx) {
        quad_add(s_tile, idx, U4{num(key.x), num(key.y), num(key.z), num(key.w)});
      });
    } else {
      auto num = [&](uint32_t key) { return (uint32_t)(key - lo - width < 0x80000000u - width); };
      auto keep = [&](uint32_t key, uint32_t idx) {
        if (key - lo >= width) return;
        const uint32_t at = atomicAdd(&s_cnt, 1u);
        s_key[at] = key;
        s_idx[at] = idx;
      };
      list.visit_quads([&](const U4& key, const U4& idx) {
        quad_add(s_tile, idx, U4{num(key.x), num(key.y), num(key.z), num(key.w)});
        keep(key.x, idx.x); keep(key.y, idx.y); keep(key.z, idx.z); keep(key.w, idx.w);
      });
    }
    T = lo;
    need = rank;
    __syncthreads();
    if (!ties_only) {
      const uint32_t cnt = s_cnt;
      wide_list_rank(s_key, cnt, rank, s_out);
      __syncthreads();
      T = s_out[0];
      need = rank - s_out[1];
      n_eq = s_out[2];
      if (threadIdx.x < cnt && s_key[threadIdx.x] >= T)
        atomicAdd(&s_tile[s_idx[threadIdx.x] >> 10], s_key[threadIdx.x] > T ? 1u : 1u << 16);
      __syncthreads();
    }
  }
  if (!ok) {
    if (judge) {
      for (int b = threadIdx.x; b < kHistEntries; b += kWide) st_agent(&J.hist[b], 0u);
      wait_landed();
      if (threadIdx.x == 0) st_agent(&st->verdict, 2u);
    }
    Src src = srcs.s[blockIdx.y];
    if (!small_redo(src, J, s_hist, s_scan, &s_word)) return;
    T = ld_agent(&st->prefix);
    need = ld_agent(&st->krem);
    n_eq = ld_agent(&st->n_eq);
    for (int t = threadIdx.x; t < kSmallTiles; t += kWide)
      s_tile[t] = t < nt ? ld_agent(&J.tile_gt[t]) | (ld_agent(&J.tile_eq[t]) << 16) : 0u;
    __syncthreads();
  }
  // chunk prefixes: ties granted in index order until `need` is used up (all of them: tie_all); where all are,
  // the writing pass need not know how many lie before a chunk
  const uint32_t quota = J.tie_all || need == n_eq ? 0xFFFFFFFFu : need;
  uint32_t tv[PER], my_e = 0, er = 0, total;          // eight consecutive chunks per thread
#pragma unroll
  for (int j = 0; j < PER; j += 4) {
    const U4 q = *reinterpret_cast<const U4*>(s_tile + threadIdx.x * PER + j);
    tv[j] = q.x; tv[j + 1] = q.y; tv[j + 2] = q.z; tv[j + 3] = q.w;
  }
  if (quota != 0xFFFFFFFFu) {
#pragma unroll
    for (int j = 0; j < PER; ++j) my_e += tv[j] >> 16;
    er = wide_prefix(my_e, s_scan, turn, total);
  }
  uint32_t my_s = 0, eb[PER], sc[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    eb[j] = er;
    sc[j] = (tv[j] & 0xFFFFu) + ties_taken(quota, er, tv[j] >> 16);
    my_s += sc[j];
    if (quota != 0xFFFFFFFFu) er += tv[j] >> 16;
  }
  uint32_t selected;
  uint32_t sr = wide_prefix(my_s, s_scan, turn ^ 1, selected);
  if ((int)(threadIdx.x + 1) * PER <= nt) {
#pragma unroll
    for (int j = 0; j < PER; j += 4) {
      U4 q;
      q.x = sr; sr += sc[j];
      q.y = sr; sr += sc[j + 1];
      q.z = sr; sr += sc[j + 2];
      q.w = sr; sr += sc[j + 3];
      st4_u32(J.tile_gt + threadIdx.x * PER + j, q);
      st4_u32(J.tile_eq + threadIdx.x * PER + j, U4{eb[j], eb[j + 1], eb[j + 2], eb[j + 3]});
    }
  } else if ((int)threadIdx.x * PER < nt) {
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int t = threadIdx.x * PER + j;
      if (t < nt) { J.tile_gt[t] = sr; J.tile_eq[t] = eb[j]; }
      sr += sc[j];
    }
  }
  if (threadIdx.x == 0) {
    st->thresh_bits = T;
    st->need = need;
    st->n_eq = n_eq;
    st->n_gt = k - need;
    st->n_selected = selected;
    if (sga_select_result* out = J.result) {
      out->thresh_bits = T;
      out->need = need;
      out->n_gt = k - need;
      out->n_eq = n_eq;
      out->n_selected = selected;
      out->nonfinite = st->nonfinite;
      out->status = 0u;
      // 1 where the bracket decided, but for buckets below 2^20: they report 0 whatever decided (callers
      // know the path of those sizes as 0)
      out->path = (ok && !single && n >= kFastMinN ? 1u : 0u) | (st->negative ? 0x100u : 0u);
    }
  }
}

// The launches for every job of a batch (all of them SelBatch::small_ok).  dirs: segment
// directories to build on the way (the finishing and writing passes read them).
template <class Src>
static inline void run_small_select(const SrcPack<Src>& srcs, const SelBatch& B, const SegDirJobs& dirs,
                                    const typename Src::Cols& cols, hipStream_t s) {
  launch_sample_pick<false>(srcs, B, dirs, cols, kBracketSigmas, s);
  const int cpw = Src::kHyper || B.max_tiles <= kSweepTiles ? 1 : 4;
  if (cpw == 1)
    hipLaunchKernelGGL((k_small_sweep<Src, 1>), B.grid((unsigned)B.max_tiles), dim3(kBlock), 0, s, srcs, B.jobs);
  else
    hipLaunchKernelGGL((k_small_sweep<Src, Src::kHyper ? 1 : 4>), B.grid((unsigned)cdiv64(B.max_tiles, 4)), dim3(kBlock), 0,
                       s, srcs, B.jobs);
  const int64_t wgs = cdiv64(B.max_tiles, kRedoTiles);
  hipLaunchKernelGGL((k_small_finish<Src>), B.grid((unsigned)(wgs < kRedoGroups ? wgs : kRedoGroups)), dim3(kWide), 0,
                     s, srcs, B.jobs, cpw);
}

#endif  // __HIPCC__
}  // namespace sga
