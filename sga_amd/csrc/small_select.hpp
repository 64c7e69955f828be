// Exact top-k of a bucket of up to kSmallTiles chunks (8.4 M coordinates) in two or three launches:
//   k_small_front     8 K to 16 K sample keys, the bracket of the k-th key from them (and the
//                     directory of the segment table), and in the same launch, where its workgroups are all
//                     resident at once, the one sweep over the data: per-chunk counts above the bracket, and a
//                     list of the few keys inside it
//   k_small_sweep     that sweep where they are not
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
// (Kernels of the 4.2 M step, fp32 gradients: front 18, finish 16, final sweep 27.  In the front, us after its start:
// sample loaded 4 to 5, bracket 10, seen by the sweep 10.5, its list reserved 13.5, launch over 17; the finish is
// bound by one workgroup's instruction issue and LDS atomics: loads 3, totals 1, histogram of 35 K entries 4, chunk
// counts 6, edge and prefixes 2.  Adding the list to a histogram in the sweep instead moves its 4 us to 5 of
// device-wide atomics there; counting by a bit per entry is no faster below 8 M.)
//
// The result is exact for any sample: where the bracket misses the k-th key the finishing launch goes
// over the data itself, with all of its workgroups (small_redo).
#pragma once
#include "select_impl.hpp"

namespace sga {

#ifdef __HIPCC__

// Candidate lists of the small path: the chunks of the sweep share kSmallSegs counters (the segments of
// the list), by units of a few chunks that reserve together and go round the segments; a segment has room for every
// coordinate of its chunks, so it never overflows.
// The counters lie 256 bytes apart: atomics on one cache line queue like those on one address (11 ns
// each; 1024 workgroups on 16 adjacent words: the sweep of 4 M elements took 19 us, 8.6 with this).
struct SmallGeom { uint32_t segs, cap; };          // cap: list entries per segment
__host__ __device__ static inline SmallGeom small_geom(int64_t n_tiles, int unit) {
  SmallGeom s;
  const uint32_t units = (uint32_t)cdiv64(n_tiles, unit), per = (uint32_t)cdiv64(units, kSmallSegs);
  s.segs = (uint32_t)cdiv64(units, per);
  s.cap = (per * unit < 2 ? 2 : per * unit) * (uint32_t)kChunk;      // two chunks hold the head that is read unseen
  return s;
}

// Sample, bracket and the one sweep over the data, one launch: the first kSampleGroups workgroups of a job take the
// sample and one of them the bracket (sample_pick_body), one keeps house (directory and columns of the segment
// table), the others sweep.  These request their data and form its keys while the bracket is on its way, and then
// look for it in one of kSmallSegs copies.  Counts above the bracket, keys inside it to the list.  A workgroup reserves
// its entries together; in the front four chunks' entries, so that a workgroup that has all of the list spreads it over
// the segments, each of which is one wave's work in the finish.  Selects at 1 %, a reservation per workgroup / per four
// chunks, us: ascending scores 1.3 M 64 / 46, 3 M 75 / 54, 4.2 M 77 / 59; a fiftieth of the scores high, in one piece
// 49 / 35, 47 / 41, 50 / 44; independent ones the same.
// Keys equal to the bracket's lower end are counted per chunk and not
// listed: a plateau of equal keys (zeros, momenta that have decayed to the last denormal) puts the
// lower end on itself, and the one workgroup behind the sweep would walk a list as long as the bucket
// (|m| after a thousand sparse steps, 1.7 M coordinates: 889 us, 86 like this).
//
// One launch or two: the waiting workgroups hold their registers and LDS, one on a CU, so they go along where they are
// no more than the CUs (kFrontSweeps: 4.2 M coordinates, 1 M of a score that is a chain of arithmetic).  With twice
// as many the ones behind begin when the first are done, which two launches are faster than (`update` 8.4 M one launch
// 155 us, two 136; twelve buckets of 20 M 493 / 291).  Two launches -> one, us: step of 261 K 28.8 -> 27.6, `update`
// 43.6 -> 39.9, 3 M 60.1 -> 56.3, 4.2 M fp32 65.9 -> 62.9; selects of 1 M at 10 % 59.1 -> 54.6, of 3 M 56.6 -> 55.1.
// Slabs per wave (SPW): one up to kFrontTiles chunks (kSweepTiles for a sweep of its own) and for the scores that are a
// chain of arithmetic; beyond, four, whose loads are in flight together.
// In the front a workgroup's entries leave by LDS, whole lines at a time (few lanes of a store hold one: 5 us of the
// front at 4.2 M, 3.5 so); a sweep of its own has other workgroups to fill that time.
//
// Nobody waits for long: a sweeping workgroup looks kBracketLooks times (some milliseconds; those that it waits for
// wait for nobody and come before it in the grid, so that it does not happen) and then says in its chunks' words that
// it had none.  The launch's number makes a copy this launch's; k_small_finish clears copies and marks for recorded
// graphs, which repeat their numbers.  Memory that happens to hold the number may give a workgroup a bracket that is
// not the one in the state, or clear a segment's counter after somebody has added to it: tags and counts then do not
// agree, or a reservation does not fit, and the finish goes over the data itself.
constexpr int64_t kSweepTiles = 2048, kFrontTiles = 1024, kFrontSweeps = 256;
constexpr int kBracketLooks = 4096;
constexpr int kSweepList = 2048;                     // entries of a workgroup that are gathered in LDS
template <class Src, int WAVES, int SPW, bool WAIT, class Now>
__device__ __forceinline__ void small_sweep_body(Src src, const ChainJob& J, const Now& now, uint32_t launch, int64_t blk) {
  constexpr int ROUND = WAVES / kChunkIters, CPW = ROUND * SPW, SLABS = WAVES * SPW;
  constexpr int PARTS = WAIT ? SPW : 1, UNIT = CPW / PARTS;         // chunks of a reservation; slabs u * WAVES + w
  static_assert(SLABS <= kWave, "a lane per slab");
  __shared__ uint32_t s_hi[SLABS], s_eq[SLABS], s_cnt[SLABS], s_nf[SLABS], s_got[3], s_base[PARTS], s_off[PARTS], s_fit;
  __shared__ uint32_t s_lkey[WAIT ? kSweepList : 1], s_lidx[WAIT ? kSweepList : 1];
  const int64_t n = J.n, n_chunks = J.n_tiles, c0 = blk * CPW;
  if (c0 >= n_chunks) return;                         // a smaller job of the batch
  const int w = uniform_i32(wave_id());
  const int64_t c1 = c0 + w / kChunkIters, i1 = c1 * kChunk + (w % kChunkIters) * (kWave * kVec);
  uint32_t left_lo = 0, left_hi = 0;                  // by the launch before
  if (!WAIT) { left_lo = J.st->t_lo; left_hi = J.st->t_hi; }
  typename Src::Raw raw[SPW];
#pragma unroll
  for (int u = 0; u < SPW; ++u) {
    const int64_t c = c1 + u * ROUND, i = i1 + u * ROUND * kChunk + lane_id() * kVec;
    const typename Src::Chunk ck = src.chunk_begin(c);
    if (src.vec && (c + 1) * kChunk <= n) src.template fetch<true, true>(ck, i, n, raw[u]);       // read again soon
    else if (i < n) src.template fetch<false>(ck, i, n, raw[u]);
  }
  uint32_t key[SPW][4], nf[SPW];
#pragma unroll
  for (int u = 0; u < SPW; ++u) {
    const int64_t c = c1 + u * ROUND, i0 = i1 + u * ROUND * kChunk, i = i0 + lane_id() * kVec;
    const typename Src::Chunk ck = src.chunk_begin(c);
    key[u][0] = key[u][1] = key[u][2] = key[u][3] = 0u;
    const bool full = (c + 1) * kChunk <= n;
    src.slab_hyper(i0);
    if constexpr (Src::kHyper) now.into(src.sc.h, src.sc.at);
    if (src.vec && full) src.template keys<true>(ck, i, n, raw[u], key[u], now);
    else if (i < n) src.template keys<false>(ck, i, n, raw[u], key[u], now);
    nf[u] = 0u;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (!full && i + e >= n) key[u][e] = ~0u;       // below every bound, as the signed number it is compared as
      nf[u] += (uint32_t)__popcll(ballot64((int32_t)key[u][e] >= 0x7F800000));
    }
  }
  const uint32_t neg = ballot64(src_negative(src) != 0u) != 0ull ? 0x80000000u : 0u;
  if (WAIT && threadIdx.x == 0) {
    const unsigned long long* from = small_bracket_copy(J, (int)(blk % kSmallSegs));
    unsigned long long lo = 0, hi = 0;
    bool there = false;
    for (int t = 0; t < kBracketLooks && !there; ++t) {
      if (t) __builtin_amdgcn_s_sleep(4);
      lo = ld_agent64(from);
      hi = ld_agent64(from + 1);
      there = (uint32_t)(lo >> 32) == launch && (uint32_t)(hi >> 32) == launch;
    }
    s_got[0] = there ? (uint32_t)lo : 0x7FFFFFFFu;    // without a bracket no key is listed
    s_got[1] = there ? (uint32_t)hi : 0x80000000u;
    s_got[2] = there;
  }
  if (WAIT) __syncthreads();
  const uint32_t T_LO = WAIT ? s_got[0] : left_lo, T_HI = WAIT ? s_got[1] : left_hi;
  const int32_t below = (int32_t)T_LO, top = (int32_t)(T_HI - 1u);
  Ballot4 cand[SPW];
#pragma unroll
  for (int u = 0; u < SPW; ++u) {
    uint32_t hi = 0, eq = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint64_t above = ballot64((int32_t)key[u][e] > top);
      cand[u].m[e] = ballot64((int32_t)key[u][e] > below) & ~above;
      hi += (uint32_t)__popcll(above);
      eq += (uint32_t)__popcll(ballot64(key[u][e] == T_LO));
    }
    if (lane_id() == 0) {
      const int q = u * WAVES + w;
      s_hi[q] = hi; s_eq[q] = eq; s_cnt[q] = cand[u].count(); s_nf[q] = nf[u] | neg;
    }
  }
  __syncthreads();
  // every wave sums the slabs' counts for itself; the first one reserves and writes the chunks' words meanwhile
  const uint32_t mine = lane_id() < SLABS ? s_cnt[lane_id()] : 0u, incl = wave_incl_scan(mine);
  const uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
  // of the part that slab q lies in: where it begins in the workgroup's list (uniform q)
  auto part_off = [&](int p) { return p ? (uint32_t)__builtin_amdgcn_readlane((int)incl, p * (SLABS / PARTS) - 1) : 0u; };
  if (w == 0) {
    const SmallGeom geo = small_geom(n_chunks, UNIT);
    uint32_t base = 0, off = 0, cnt_p = all, seg = (uint32_t)(blk % geo.segs);      // of the lane's part
#pragma unroll
    for (int p = 0; PARTS > 1 && p < PARTS; ++p) {
      const uint32_t from = part_off(p), to = p + 1 < PARTS ? part_off(p + 1) : all;
      if (lane_id() == p) { off = from; cnt_p = to - from; seg = (uint32_t)((blk * PARTS + p) % geo.segs); }
    }
    const bool reserves = lane_id() < PARTS && cnt_p != 0u;
    if (reserves) base = atomicAdd(&J.seg_cnt[seg * kSmallSegStride], cnt_p);
    const uint32_t fits = (uint32_t)ballot64(!reserves || (base <= geo.cap && cnt_p <= geo.cap - base));      // a bit a part
    if (lane_id() < PARTS) { s_base[lane_id()] = seg * geo.cap + base; s_off[lane_id()] = off; }
    if (lane_id() == 0) s_fit = fits;
    if (lane_id() < CPW && c0 + lane_id() < n_chunks) {
      const bool fit = (fits >> (lane_id() / UNIT) & 1u) != 0u;
      uint32_t hi = 0, eq = 0, cnt = 0, bad = 0, minus = 0;
#pragma unroll
      for (int j = 0; j < kChunkIters; ++j) {
        const int q = lane_id() * kChunkIters + j;
        hi += s_hi[q]; eq += s_eq[q]; cnt += s_cnt[q];
        bad += s_nf[q] & 0x7FFFFFFFu; minus |= s_nf[q] >> 31;
      }
      const SmallChunk ch = SmallChunk::of(T_LO, T_HI, hi, cnt, eq, bad, minus != 0u, !fit || (WAIT && s_got[2] == 0u));
      J.tile_gt[c0 + lane_id()] = ch.a;
      J.tile_eq[c0 + lane_id()] = ch.b;
    }
  }
  const bool via_lds = WAIT && all <= (uint32_t)kSweepList;
  if (!via_lds) __syncthreads();                      // uniform; the list goes straight to its place then
#pragma unroll
  for (int u = 0; u < SPW; ++u) {
    const int q = u * WAVES + w, p = PARTS > 1 ? u : 0;
    uint32_t run = (uint32_t)__builtin_amdgcn_readlane((int)(incl - mine), q);
    const uint32_t i = (uint32_t)(i1 + u * ROUND * kChunk + lane_id() * kVec);
    if (via_lds) {
      ballot_append(cand[u], run, [&](uint32_t pos, int e) { s_lidx[pos] = i + e; s_lkey[pos] = key[u][e]; });
    } else if (s_fit >> p & 1u) {
      run += s_base[p] - s_off[p];
      ballot_append(cand[u], run, [&](uint32_t pos, int e) { J.small_idx[pos] = i + e; J.small_key[pos] = key[u][e]; });
    }
  }
  if (!via_lds) return;
  __syncthreads();
  for (uint32_t t = threadIdx.x; t < all; t += WAVES * kWave) {
    int p = 0;
#pragma unroll
    for (int j = 1; j < PARTS; ++j) p += t >= s_off[j];
    if (!(s_fit >> p & 1u)) continue;
    const uint32_t at = s_base[p] + (t - s_off[p]);
    J.small_idx[at] = s_lidx[t];
    J.small_key[at] = s_lkey[t];
  }
}
template <class Src, int SPW>
__global__ __launch_bounds__(kWide) void k_small_front(SrcPack<Src> srcs, ChainJobs jobs, SegDirJobs dirs,
                                                       typename Src::Cols cols, uint32_t launch, double sigmas) {
  const ChainJob& J = jobs.j[blockIdx.y];
  const int64_t sweep = (int64_t)blockIdx.x - kSampleGroups - 1;
  if (blockIdx.x < kSampleGroups) sample_pick_body<Src, false>(srcs, J, cols, launch, sigmas);
  else if (sweep < 0) keep_tables(dirs, cols, threadIdx.x, kWide);
  else if constexpr (std::is_same<typename Src::Cols, NowCols>::value)
    small_sweep_body<Src, kWideWaves, SPW, true>(srcs.s[blockIdx.y], J, ColsOf{&cols, (int)blockIdx.y}, launch, sweep);
  else
    small_sweep_body<Src, kWideWaves, SPW, true>(srcs.s[blockIdx.y], J, NoCols{}, launch, sweep);
}
// The sweep behind a launch that took the sample and the bracket alone.
template <class Src, int SPW>
__global__ __launch_bounds__(kBlock) void k_small_sweep(SrcPack<Src> srcs, ChainJobs jobs) {
  small_sweep_body<Src, kChunksPerBlock, SPW, false>(srcs.s[blockIdx.y], jobs.j[blockIdx.y], NoCols{}, 0u, blockIdx.x);
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
    for (int u = 0; u < kSmallHead; ++u)
      if (c < (uint32_t)(u + 1) * kWave * kVec) trim(key[u], (uint32_t)(u * kWave + lane_id()) * kVec, c);   // uniform
  }
  // head(key, idx) over the entries in registers, tail(keys, idxs) over rounds of quads of the rest (whole waves).
  // IDX: the index is wanted; without it twice as many keys are in flight.  The rest comes from other XCDs' stores, a
  // microsecond a round of loads, so the next round is on its way while one is worked off.
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
  const bool a1 = c1 == c0, a2 = c2 == c0, a3 = c3 == c0;
  const uint32_t first = num.x + (a1 ? num.y : 0u) + (a2 ? num.z : 0u) + (a3 ? num.w : 0u);
  const uint32_t behind = num.x + num.y + num.z + num.w - first;
  if (first) atomicAdd(&s_tile[c0], first);
  if (behind) {
    const bool b1 = c1 == c3, b2 = c2 == c3;          // of c3's chunk, which is not c0's
    const uint32_t last = a3 ? 0u : num.w + (b1 ? num.y : 0u) + (b2 ? num.z : 0u);
    if (last) atomicAdd(&s_tile[c3], last);
    if (behind != last) {
      if (!a1 && (a3 || !b1) && num.y) atomicAdd(&s_tile[c1], num.y);
      if (!a2 && (a3 || !b2) && num.z) atomicAdd(&s_tile[c2], num.z);
    }
  }
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
      tile_count_body<Src, Src::kHyper>(src, J, prefix, 0, (int64_t)blk * kWideWaves + wave_id(), (int64_t)G * kWideWaves);
    } else {
      reinterpret_cast<U4*>(s_hist)[threadIdx.x] = U4{0u, 0u, 0u, 0u};
      __syncthreads();
      constexpr int U = Src::kHyper ? 1 : 4;          // quads in flight per thread (the chains: four of them spill)
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
__global__ __launch_bounds__(kWide) void k_small_finish(SrcPack<Src> srcs, ChainJobs jobs, int unit) {
  __shared__ __align__(16) uint32_t s_hist[kBinsBig + kWave];     // behind the bins, a word per lane for what is in none
  __shared__ __align__(16) uint32_t s_tile[kSmallTiles];          // above | ties << 16, at most 1024 each
  __shared__ __align__(16) uint32_t s_key[kWideList];
  __shared__ uint32_t s_idx[kWideList];
  __shared__ uint32_t s_seg[kWideWaves], s_cnt, s_out[3], s_word, s_listed, s_nf, s_flags;
  __shared__ WideScratch s_scan;
  const ChainJob& J = jobs.j[blockIdx.y];
  SelState* st = J.st;
  const int64_t n = J.n;
  const int nt = (int)J.n_tiles;
  const uint32_t k = J.k, T_LO = st->t_lo, T_HI = st->t_hi;
  const bool single = T_HI - T_LO == 1u;
  const SmallGeom geo = small_geom(nt, unit);
  SmallList list;
  list.request(J, geo);
  constexpr int PER = kSmallTiles / kWide;            // 8
  const SmallChunk none = SmallChunk::none(T_LO, T_HI);
  SmallChunk ch[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int t = j * kWide + threadIdx.x;
    ch[j] = none;
    if (j * kWide < nt && t < nt) { ch[j].a = J.tile_gt[t]; ch[j].b = J.tile_eq[t]; }
  }
  uint32_t sum_a = 0, sum_b = 0, off_a = 0, off_b = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    sum_a += ch[j].a & SmallChunk::kNumbers;
    sum_b += ch[j].b & SmallChunk::kNumbers;
    off_a |= ch[j].a ^ none.a;
    off_b |= ch[j].b ^ none.b;
  }
  const uint32_t hi = sum_a & 0xFFFFu, eqs = sum_b & 0xFFFFu, nonfinite = sum_b >> 16;
  uint32_t listed = sum_a >> 16;
  const bool minus = (off_b & SmallChunk::kNegative) != 0u;
  const bool wrong = SmallChunk::wrong(off_a, off_b);
  reinterpret_cast<U4*>(s_hist)[threadIdx.x] = U4{0u, 0u, 0u, 0u};
  if (threadIdx.x < kWideWaves)
    s_seg[threadIdx.x] = threadIdx.x < geo.segs ? J.seg_cnt[threadIdx.x * kSmallSegStride] : 0u;
  if (blockIdx.x == 0 && threadIdx.x < 4 * kSmallSegs) {             // behind the launch that used them
    reinterpret_cast<uint32_t*>(small_bracket_copy(J, (int)threadIdx.x / 4))[threadIdx.x % 4] = 0u;
    if (threadIdx.x < kSampleGroups) st->sampled[threadIdx.x] = 0u;
  }
  if (threadIdx.x == 0) {
    s_listed = s_nf = s_flags = 0u;
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
  listed = wave_sum(listed);
  if (lane_id() == 0 && listed) atomicAdd(&s_listed, listed);
  if (nonfinite) atomicAdd(&s_nf, nonfinite);
  if (minus | wrong) atomicOr(&s_flags, (minus ? 1u : 0u) | (wrong ? 2u : 0u));
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
  const bool whole = s_listed == n_list && (s_flags & 2u) == 0u;     // of one bracket, and nothing lost
  const bool ok = judge && whole && !crowded && n_hi < k && k <= n_hi + n_list + n_low;
  if (judge && gridDim.x > 1 && ok && threadIdx.x == 0) st_agent(&st->verdict, 1u);
  const bool low = ok && k > n_hi + n_list;           // the lower end is the threshold
  uint32_t T = T_LO, need = k - n_hi - n_list, n_eq = n_low;
  int turn = 0;
  if (ok) {
#pragma unroll
    for (int j = 0; j < PER; ++j)                     // the lower end below the threshold: its members are no ties
      s_tile[j * kWide + threadIdx.x] = (ch[j].a & 0x7FFu) | (low ? (ch[j].b & 0x7FFu) << 16 : 0u);
  }
  if (low) {
    __syncthreads();
    list.visit_quads([&](const U4& key, const U4& idx) {
      quad_add(s_tile, idx, U4{key.x != ~0u, key.y != ~0u, key.z != ~0u, key.w != ~0u});
    });
    __syncthreads();
  } else if (ok) {
    // descent over the list inside (T_LO, T_HI): 4096 bins per level, until one bin is left whose
    // keys fit the short list (nearly always after the first level) or are all equal
    uint32_t lo = T_LO + 1u, rank = k - n_hi;
    int w = 32 - __clz((int)(T_HI - 1u - lo));         // bits of the offset (the list is not empty)
    for (;;) {
      const int sh = w > 12 ? w - 12 : 0;
      const uint32_t bins = 1u << (w - sh), none = kBinsBig + (uint32_t)lane_id();
      auto count = [&](uint32_t key, uint32_t) {
        const uint32_t bin = (key - lo) >> sh;
        atomicAdd(&s_hist[bin < bins ? bin : none], 1u);
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
      const int32_t last = (int32_t)(lo + width - 1u), first = (int32_t)lo;     // of the bin; keys past the list are -1
      auto num = [&](uint32_t key) { return (uint32_t)((int32_t)key > last); };
      auto in = [&](uint32_t key) { return (int32_t)key >= first && (int32_t)key <= last; };
      auto keep = [&](uint32_t key, uint32_t idx) {
        if (!in(key)) return;
        const uint32_t at = atomicAdd(&s_cnt, 1u);
        s_key[at] = key;
        s_idx[at] = idx;
      };
      list.visit_quads([&](const U4& key, const U4& idx) {
        quad_add(s_tile, idx, U4{num(key.x), num(key.y), num(key.z), num(key.w)});
        if (ballot64(in(key.x) | in(key.y) | in(key.z) | in(key.w)) == 0ull) return;
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
      if (threadIdx.x == 0) { st_agent(&st->nonfinite, s_nf); st_agent(&st->negative, s_flags & 1u); }
      wait_landed();
      if (threadIdx.x == 0) st_agent(&st->verdict, 2u);
    }
    Src src = srcs.s[blockIdx.y];
    if (!small_redo(src, J, s_hist, s_scan, &s_word)) return;
    T = ld_agent(&st->prefix);
    need = ld_agent(&st->krem);
    n_eq = ld_agent(&st->n_eq);
    if (threadIdx.x == 0) { s_nf = ld_agent(&st->nonfinite); s_flags = ld_agent(&st->negative); }
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
      st_host(&out->thresh_bits, T);
      st_host(&out->need, need);
      st_host(&out->n_gt, k - need);
      st_host(&out->n_eq, n_eq);
      st_host(&out->n_selected, selected);
      st_host(&out->nonfinite, s_nf);
      st_host(&out->status, 0u);
      // 1 where the bracket decided, but for buckets below 2^20: they report 0 whatever decided (callers
      // know the path of those sizes as 0)
      st_host(&out->path, (ok && !single && n >= kFastMinN ? 1u : 0u) | (s_flags & 1u ? 0x100u : 0u));
    }
  }
}

// The launches for every job of a batch (all of them SelBatch::small_ok).  dirs: segment
// directories to build on the way (the finishing and writing passes read them).
template <class Src>
static inline void run_small_select(const SrcPack<Src>& srcs, const SelBatch& B, const SegDirJobs& dirs,
                                    const typename Src::Cols& cols, hipStream_t s) {
  static_assert(sizeof(ChainJobs) + sizeof(SrcPack<Src>) + sizeof(SegDirJobs) + sizeof(typename Src::Cols) + 64 <= 4096,
                "the operands travel in the kernel arguments");
  constexpr int MANY = Src::kHyper ? 1 : 4, ROUND = kWideWaves / kChunkIters;
  const int64_t t = B.max_tiles;
  int cpw = MANY == 1 || t <= kFrontTiles ? ROUND : ROUND * MANY;
  const bool together = cdiv64(t, cpw) * B.count <= kFrontSweeps;
  const auto front = [&](auto kernel, unsigned sweeps) {
    hipLaunchKernelGGL(kernel, B.grid(kSampleGroups + 1 + sweeps), dim3(kWide), 0, s, srcs, B.jobs, dirs, cols,
                       next_launch(), kBracketSigmas);
  };
  const auto sweep = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, B.grid((unsigned)cdiv64(t, cpw)), dim3(kBlock), 0, s, srcs, B.jobs);
  };
  if (together) {
    if (cpw == ROUND) front(k_small_front<Src, 1>, (unsigned)cdiv64(t, cpw));
    else front(k_small_front<Src, MANY>, (unsigned)cdiv64(t, cpw));
  } else {
    front(k_small_front<Src, 1>, 0u);
    cpw = t <= kSweepTiles ? 1 : MANY;
    if (cpw == 1) sweep(k_small_sweep<Src, 1>);
    else sweep(k_small_sweep<Src, MANY>);
  }
  const int64_t wgs = cdiv64(B.max_tiles, kRedoTiles);
  hipLaunchKernelGGL((k_small_finish<Src>), B.grid((unsigned)(wgs < kRedoGroups ? wgs : kRedoGroups)), dim3(kWide), 0,
                     s, srcs, B.jobs, together ? ROUND : cpw);
}

#endif  // __HIPCC__
}  // namespace sga
