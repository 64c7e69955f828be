// Scheme-agnostic masked ops: pack / scatter / norms / block gather-scatter /
// mask compaction.  All are HBM-bound byte movers; nothing here is a
// contraction.
#include <mutex>

#include "common.hpp"

namespace sga {

// ---------------------------------------------------------------- scatter
__global__ __launch_bounds__(kBlock) void k_scatter(float* __restrict__ dst,
                                                    const int32_t* __restrict__ idx,
                                                    const float* __restrict__ src,
                                                    int64_t k, int64_t n_dst) {
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < k;
       i += (int64_t)gridDim.x * kBlock) {
    const int64_t j = idx[i];
    if (j >= 0 && j < n_dst) dst[j] = src[i];
  }
}

// Up to kParts arrays that hold consecutive ranges of one list: part j is entries [end[j - 1], end[j]).
constexpr int kParts = SGA_MAX_PARTS;
struct Parts {
  float* base[kParts];           // of entry 0, were the part that long
  int64_t end[kParts];
  int count;
  __host__ __device__ __forceinline__ float* at(int64_t i) const {
    float* p = base[0];
    for (int j = 1; j < count; ++j)
      if (i >= end[j - 1]) p = base[j];
    return p + i;
  }
};
// One launch for the slices of a list (two of them: 4.8 us less a step, and a call from the host).
__global__ __launch_bounds__(kBlock) void k_scatter_parts(float* __restrict__ dst, const int32_t* __restrict__ idx,
                                                          Parts src, int64_t k, int64_t n_dst) {
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < k; i += (int64_t)gridDim.x * kBlock) {
    const int64_t j = idx[i];
    if (j >= 0 && j < n_dst) dst[j] = *src.at(i);
  }
}

// ------------------------------------------------------------------- pack
// The calling wave's number of entries of the ascending idx[0, k) below `split`: 64 entries a round of loads.
__device__ __forceinline__ int64_t wave_lower_bound(const int32_t* __restrict__ idx, int64_t k, int64_t split) {
  int64_t lo = 0, hi = k;                            // entries before lo are below, those from hi on are not
  while (lo < hi) {
    const int64_t step = (hi - lo + kWave - 1) / kWave, at = lo + lane_id() * step;
    const uint64_t below = ballot64(at < hi && idx[at] < split);
    const int c = __popcll(below);                   // lanes 0 .. c - 1
    const int64_t from = lo;
    lo = c ? from + (c - 1) * step + 1 : from;
    if (from + c * step < hi) hi = from + c * step;
    if (c == 0) break;
  }
  return uniform_i64(lo);
}
// With `below`, the first workgroup counts the entries under `split` instead: a host that waits for the slices' bound
// in its own memory goes on while the pack runs, where a search of its own and the wait for it came first.
// Index layout, a step on 63 M coordinates, bound with the pack's last workgroup and a copy of it -> so: 360 -> 338 us
// (with the clip's sum in host memory as well), 92 M 579 -> 533, 290 K 97 -> 70.
template <bool BF16, bool SCALE>
__global__ __launch_bounds__(kBlock) void k_pack(float* __restrict__ grad,
                                                 const int32_t* __restrict__ idx,
                                                 void* __restrict__ values,
                                                 float factor, int64_t k,
                                                 int64_t n_grad, int64_t split = 0, int64_t* __restrict__ below = nullptr) {
  const unsigned extra = below ? 1u : 0u, groups = gridDim.x - extra;
  if (blockIdx.x < extra) {
    if (wave_id() == 0) {
      const int64_t c = wave_lower_bound(idx, k, split);
      if (lane_id() == 0) st_host(below, c);
    }
    return;
  }
  for (int64_t i = (int64_t)(blockIdx.x - extra) * kBlock + threadIdx.x; i < k;
       i += (int64_t)groups * kBlock) {
    const int64_t j = idx[i];
    if (j < 0 || j >= n_grad) continue;
    float x = grad[j];
    if (SCALE) x = x * factor;
    if (BF16)
      reinterpret_cast<uint16_t*>(values)[i] = f32_to_bf16(x);
    else
      reinterpret_cast<float*>(values)[i] = x;
    grad[j] = 0.0f;
  }
}

// ------------------------------------------------------------------ norms
// Stage 1: one fp32 partial per workgroup (fixed order: lane-strided sums,
// wave tree, then 4 waves) -- run-to-run deterministic for a given n.
template <bool MASKED>
__global__ __launch_bounds__(kBlock) void k_norm_stage1(
    const float* __restrict__ x, const uint8_t* __restrict__ mask, int64_t n,
    float* __restrict__ partials, bool vec) {
  __shared__ float s_w[kChunksPerBlock];
  float acc = 0.0f;
  const int64_t stride = (int64_t)gridDim.x * kBlock * kVec;
  for (int64_t i = ((int64_t)blockIdx.x * kBlock + threadIdx.x) * kVec; i < n;
       i += stride) {
    float v[4];
    load4_f32(x, i, n, v, vec);
    if (MASKED) {
      uint32_t mk[4];
      load4_u8(mask, i, n, mk, vec);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = mk[e] ? v[e] : 0.0f;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) acc += v[e] * v[e];
  }
  acc = wave_sum(acc);
  if (lane_id() == 0) s_w[wave_id()] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.0f;
    for (int w = 0; w < kChunksPerBlock; ++w) t += s_w[w];
    partials[blockIdx.x] = t;
  }
}

// Stage 2: single workgroup folds the partials in index order.
__global__ __launch_bounds__(kBlock) void k_norm_stage2(
    const float* __restrict__ partials, int64_t np, const float* before, float* total) {
  __shared__ float s_w[kChunksPerBlock];
  float acc = 0.0f;
  for (int64_t i = threadIdx.x; i < np; i += kBlock) acc += partials[i];
  acc = wave_sum(acc);
  if (lane_id() == 0) s_w[wave_id()] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.0f;
    for (int w = 0; w < kChunksPerBlock; ++w) t += s_w[w];
    st_host(total, before ? before[0] + t : t);
  }
}

// ------------------------------------------- clip service over many records
// One workgroup per 4096-element span of one record (sga_span_record): the
// norm and the scale of a step are one launch each, whatever the number of
// parameter tensors (45 tensors of a 1.15 M-element bucket: 90 + 45 launches,
// 0.5 ms of host time, for 4 us of traffic).  A masked record loads its mask
// bytes first and then only the quads that hold a selected coordinate: at 1 %
// three of four 128-byte lines of the gradient are never touched.
struct SpanWork {
  float* g;
  const uint8_t* mask;
  int64_t n, base;
  bool vec, full;
};
__device__ __forceinline__ SpanWork span_work(const sga_span_record* __restrict__ recs, int n_recs) {
  const int64_t span = blockIdx.x;
  const sga_span_record r = recs[find_record(recs, n_recs, span)];
  SpanWork w;
  w.g = r.g; w.mask = r.mask; w.n = r.n;
  w.base = (span - r.first_span) * kBlockSpan;
  w.vec = quads_ok(r.g, 4) && quads_ok(r.mask, 1);
  w.full = w.vec && w.base + kBlockSpan <= r.n;
  return w;
}
constexpr int kSpanIters = kBlockSpan / (kBlock * kVec);   // 4 quads per lane

// the lane's quads of the span; quads without a selected coordinate are not read
template <bool FULL>
__device__ __forceinline__ void span_quads(const SpanWork& w, float v[kSpanIters][4],
                                           uint32_t mk[kSpanIters][4]) {
#pragma unroll
  for (int it = 0; it < kSpanIters; ++it) {
    const int64_t i = w.base + ((int64_t)it * kBlock + threadIdx.x) * kVec;
#pragma unroll
    for (int e = 0; e < 4; ++e) mk[it][e] = 1u;
    if (w.mask) ld_u8<FULL>(w.mask, i, w.n, mk[it], w.vec);
    else if (!FULL) {
#pragma unroll
      for (int e = 0; e < 4; ++e) mk[it][e] = i + e < w.n;
    }
  }
#pragma unroll
  for (int it = 0; it < kSpanIters; ++it) {
    const int64_t i = w.base + ((int64_t)it * kBlock + threadIdx.x) * kVec;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[it][e] = 0.0f;
    if (mk[it][0] | mk[it][1] | mk[it][2] | mk[it][3]) {
      if (FULL) {
        const F4 q = ld4(w.g + i);
        v[it][0] = q.x; v[it][1] = q.y; v[it][2] = q.z; v[it][3] = q.w;
      } else {
        load4_f32(w.g, i, w.n, v[it], w.vec);
      }
    }
  }
}

__global__ __launch_bounds__(kBlock) void k_norm_multi(const sga_span_record* __restrict__ recs,
                                                       int n_recs, float* __restrict__ partials) {
  __shared__ float s_w[kChunksPerBlock];
  const SpanWork w = span_work(recs, n_recs);
  float v[kSpanIters][4];
  uint32_t mk[kSpanIters][4];
  if (w.full) span_quads<true>(w, v, mk);
  else span_quads<false>(w, v, mk);
  float acc = 0.0f;
#pragma unroll
  for (int it = 0; it < kSpanIters; ++it)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x = mk[it][e] ? v[it][e] : 0.0f;
      acc += x * x;
    }
  acc = wave_sum(acc);
  if (lane_id() == 0) s_w[wave_id()] = acc;
  __syncthreads();
  if (threadIdx.x == 0) partials[blockIdx.x] = (s_w[0] + s_w[1]) + (s_w[2] + s_w[3]);
}

// One workgroup folds the spans' partials in a fixed order, in double.
constexpr int kFoldBlock = 1024;
__global__ __launch_bounds__(kFoldBlock) void k_norm_multi_fold(const float* __restrict__ partials,
                                                                int64_t np, float* __restrict__ total) {
  __shared__ double s_w[kFoldBlock / kWave];
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < np; i += kFoldBlock) acc += (double)partials[i];
  acc = wave_sum(acc);
  if (lane_id() == 0) s_w[wave_id()] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < kFoldBlock / kWave; ++w) t += s_w[w];
    st_host(total, (float)t);
  }
}

__global__ __launch_bounds__(kBlock) void k_scale_multi(const sga_span_record* __restrict__ recs,
                                                        int n_recs, float coeff) {
  const SpanWork w = span_work(recs, n_recs);
  float v[kSpanIters][4];
  uint32_t mk[kSpanIters][4];
  if (w.full) span_quads<true>(w, v, mk);
  else span_quads<false>(w, v, mk);
#pragma unroll
  for (int it = 0; it < kSpanIters; ++it) {
    const int64_t i = w.base + ((int64_t)it * kBlock + threadIdx.x) * kVec;
    if (!(mk[it][0] | mk[it][1] | mk[it][2] | mk[it][3])) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[it][e] = mk[it][e] ? v[it][e] * coeff : v[it][e];
    if (w.full) st4(w.g + i, F4{v[it][0], v[it][1], v[it][2], v[it][3]});
    else store4_f32(w.g, i, w.n, v[it], w.vec);
  }
}

// --------------------------------------------------------- block gather
template <bool SCALE>
__global__ __launch_bounds__(kBlock) void k_gather_blocks(
    const float* __restrict__ grad, const uint8_t* __restrict__ mask,
    const int32_t* __restrict__ bidx, float* __restrict__ values, int64_t total,
    int xlog, float factor, int64_t n) {
  for (int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x; t < total;
       t += (int64_t)gridDim.x * kBlock) {
    const int64_t j = t >> xlog;
    const int64_t pos = (int64_t)bidx[j] + (t & ((1 << xlog) - 1));
    float out = 0.0f;
    if (pos >= 0 && pos < n && mask[pos] != 0) {
      out = grad[pos];
      if (SCALE) out = out * factor;
    }
    values[t] = out;
  }
}

__global__ __launch_bounds__(kBlock) void k_scatter_blocks(
    float* __restrict__ dst, const uint8_t* __restrict__ mask,
    const int32_t* __restrict__ bidx, const float* __restrict__ src,
    int64_t total, int xlog, int64_t n) {
  for (int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x; t < total;
       t += (int64_t)gridDim.x * kBlock) {
    const int64_t j = t >> xlog;
    const int64_t pos = (int64_t)bidx[j] + (t & ((1 << xlog) - 1));
    if (pos >= 0 && pos < n && mask[pos] != 0) dst[pos] = src[t];
  }
}

// ------------------------------------------------ block-granular helpers
// A group of L = min(x, 64) lanes cooperates on one x-element block of a
// view (the tail block of a view is short and reduces over its real length).
// MODE 0: mean of |g|, 1: max of |g|  -> float out[block]
template <int MODE>
__global__ __launch_bounds__(kBlock) void k_block_reduce(const float* __restrict__ g, int64_t n,
                                                         int x, int lanes, float* __restrict__ out,
                                                         int64_t n_blocks) {
  const int per_wave = kWave / lanes;
  const int sub = lane_id() / lanes, l = lane_id() % lanes;
  const int64_t wstride = (int64_t)gridDim.x * kChunksPerBlock * per_wave;
  for (int64_t b0 = ((int64_t)blockIdx.x * kChunksPerBlock + wave_id()) * per_wave; b0 < n_blocks;
       b0 += wstride) {
    const int64_t b = b0 + sub;
    float acc = 0.0f;
    int64_t len = 0;
    if (b < n_blocks) {
      const int64_t lo = b * x;
      len = n - lo < x ? n - lo : x;
      for (int64_t j = l; j < len; j += lanes) {
        const float a = fabsf(g[lo + j]);
        acc = MODE == 0 ? acc + a : fmaxf(acc, a);
      }
    }
    for (int o = lanes / 2; o > 0; o >>= 1) {
      const float t = __shfl_xor(acc, o, kWave);
      acc = MODE == 0 ? acc + t : fmaxf(acc, t);
    }
    if (b < n_blocks && l == 0) out[b] = MODE == 0 ? __fdiv_rn(acc, (float)len) : acc;
  }
}

// any_out[b] = 1 when block b of the span has a set byte
__global__ __launch_bounds__(kBlock) void k_block_any(const uint8_t* __restrict__ mask, int64_t n,
                                                      int x, int lanes, uint8_t* __restrict__ any_out,
                                                      int64_t n_blocks) {
  const int per_wave = kWave / lanes;
  const int sub = lane_id() / lanes, l = lane_id() % lanes;
  const int64_t wstride = (int64_t)gridDim.x * kChunksPerBlock * per_wave;
  for (int64_t b0 = ((int64_t)blockIdx.x * kChunksPerBlock + wave_id()) * per_wave; b0 < n_blocks;
       b0 += wstride) {
    const int64_t b = b0 + sub;
    uint32_t acc = 0;
    if (b < n_blocks) {
      const int64_t lo = b * x;
      const int64_t len = n - lo < x ? n - lo : x;
      for (int64_t j = l; j < len; j += lanes) acc |= mask[lo + j];
    }
    for (int o = lanes / 2; o > 0; o >>= 1) acc |= __shfl_xor(acc, o, kWave);
    if (b < n_blocks && l == 0) any_out[b] = acc ? 1 : 0;
  }
}

// out[i] = bmask[i / x]  (repeat_interleave(x)[:n])
__global__ __launch_bounds__(kBlock) void k_expand_blocks(const uint8_t* __restrict__ bmask, int xlog,
                                                          int64_t n, uint8_t* __restrict__ out) {
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kBlock)
    out[i] = bmask[i >> xlog];
}

// ------------------------------------------------------- mask compaction
// Chunk = 1024 consecutive bytes owned by one wave, 16 bytes per lane in one load; four chunks per wave, whose
// loads are in flight together.  Phase 1 counts the non-zero bytes of each chunk; a two-level exclusive scan
// turns counts into offsets; phase 2 rewrites positions in ascending order from the lanes' prefix -- the output
// equals nonzero() for any launch geometry.  With four
// bytes per lane and load, 63 M bytes: count 20.0 -> 10.7 us, fill 24.1 -> 14.2 (5.9 and 4.6 TB/s of the mask and list).
constexpr int kMaskChunks = 4;                  // per wave
// Bit j: byte j of the lane's 16 bytes at i is not zero (past n: zero).
__device__ __forceinline__ uint32_t nonzero_bits(const U4& w) {
  const uint32_t x[4] = {w.x, w.y, w.z, w.w};
  uint32_t bits = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t nz = (((x[j] & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | x[j]) & 0x80808080u;     // top bit of every such byte
    bits |= ((nz >> 7) * 0x10204080u >> 28) << (4 * j);                                 // ... side by side
  }
  return bits;
}
// The lane's bits of the wave's chunks c0 .. c0 + kMaskChunks - 1.
__device__ __forceinline__ void mask_bits(const uint8_t* __restrict__ mask, int64_t n, int64_t c0,
                                          uint32_t (&bits)[kMaskChunks]) {
  typedef uint32_t u4v __attribute__((ext_vector_type(4), aligned(1)));      // a view may begin at any byte
  U4 w[kMaskChunks];
#pragma unroll
  for (int u = 0; u < kMaskChunks; ++u) {
    const int64_t i = (c0 + u) * kChunk + lane_id() * 16;
    w[u] = U4{0u, 0u, 0u, 0u};
    if (i + 16 <= n) {
      const u4v t = *reinterpret_cast<const u4v*>(mask + i);
      w[u] = U4{t.x, t.y, t.z, t.w};
    } else if (i < n) {
      uint32_t x[4] = {0u, 0u, 0u, 0u};
      for (int e = 0; e < 16 && i + e < n; ++e) {
        const uint32_t by = (uint32_t)mask[i + e] << (8 * (e & 3));
        if (e < 4) x[0] |= by; else if (e < 8) x[1] |= by; else if (e < 12) x[2] |= by; else x[3] |= by;
      }
      w[u] = U4{x[0], x[1], x[2], x[3]};
    }
  }
#pragma unroll
  for (int u = 0; u < kMaskChunks; ++u) bits[u] = nonzero_bits(w[u]);
}

__global__ __launch_bounds__(kBlock) void k_mask_count(const uint8_t* __restrict__ mask, int64_t n,
                                                       uint32_t* __restrict__ counts, int64_t n_chunks) {
  const int64_t c0 = ((int64_t)blockIdx.x * kChunksPerBlock + wave_id()) * kMaskChunks;
  if (c0 >= n_chunks) return;
  uint32_t bits[kMaskChunks];
  mask_bits(mask, n, c0, bits);
#pragma unroll
  for (int u = 0; u < kMaskChunks; ++u) {
    const uint32_t cnt = wave_incl_scan((uint32_t)__popc(bits[u]));
    if (lane_id() == kWave - 1 && c0 + u < n_chunks) counts[c0 + u] = cnt;
  }
}

// A chunk's positions leave lane by lane while they are few: a store then touches few lines, if far apart.  From
// kStagedFill on they go through LDS (a word free after every 16, lanes 16 words apart would share a bank) and leave
// as quads in order, because a lane's own sixteen lie up to 64 bytes from its neighbour's.  Compaction of 63 M bytes,
// lane by lane / staged / four bytes per lane and load: a tenth set 67 / 73 / 90 us, 15 % 72 / 69 / 90, a quarter
// 87 / 73 / 91, half 142 / 81 / 102, all 334 / 98 / 140.
constexpr uint32_t kStagedFill = 160;
__global__ __launch_bounds__(kBlock) void k_mask_fill(const uint8_t* __restrict__ mask, int64_t n,
                                                      const uint32_t* __restrict__ offsets, int32_t* __restrict__ idx_out,
                                                      int64_t cap, int64_t n_chunks) {
  __shared__ int32_t s_idx[kChunksPerBlock][kChunk + kChunk / 16];
  const int64_t c0 = ((int64_t)blockIdx.x * kChunksPerBlock + wave_id()) * kMaskChunks;
  if (c0 >= n_chunks) return;
  uint32_t bits[kMaskChunks];
  mask_bits(mask, n, c0, bits);
  int32_t* own = s_idx[wave_id()];
#pragma unroll
  for (int u = 0; u < kMaskChunks; ++u) {
    if (c0 + u >= n_chunks) return;
    const uint32_t mine = (uint32_t)__popc(bits[u]), incl = wave_incl_scan(mine);
    const uint32_t count = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
    const int64_t base = offsets[c0 + u];
    const int32_t i0 = (int32_t)((c0 + u) * kChunk + lane_id() * 16);
    uint32_t at = incl - mine;
    if (count < kStagedFill) {
      for (uint32_t left = bits[u]; left; left &= left - 1u, ++at)
        if (base + at < cap) idx_out[base + at] = i0 + __ffs((int)left) - 1;
      continue;
    }
    for (uint32_t left = bits[u]; left; left &= left - 1u, ++at) own[at + at / 16] = i0 + __ffs((int)left) - 1;
    __builtin_amdgcn_wave_barrier();              // the wave's own LDS: its accesses stay in order
    const int64_t room = cap - base;
    const int put = room < (int64_t)count ? (int)(room < 0 ? 0 : room) : (int)count;
    typedef int32_t i4v __attribute__((ext_vector_type(4), aligned(4)));
    for (int j = lane_id() * kVec; j < put; j += kWave * kVec) {
      const int32_t* q = own + j + j / 16;        // the quad lies in one group of 16
      const int32_t v[4] = {q[0], q[1], q[2], q[3]};
      if (j + kVec <= put) {
        *reinterpret_cast<i4v*>(idx_out + base + j) = i4v{v[0], v[1], v[2], v[3]};
      } else {
        for (int e = 0; j + e < put; ++e) idx_out[base + j + e] = v[e];
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// The compaction around one wait of the host, which needs the count to allocate: before it, the chunks' counts with
// their sums by workgroup (a group of 16 chunks), and one workgroup that turns the sums into offsets and takes the
// totals; behind it, the positions, and with GATHER the values at them.  (Counts, two launches of a scan, a launch for
// the slices' ends, the positions, and a gather for each slice were eight: mask layout, step on 1.15 M coordinates in
// 45 tensors 125 to 139 us, 119 so.)
__global__ __launch_bounds__(kBlock) void k_mask_groups(const uint8_t* __restrict__ mask, int64_t n,
                                                        uint32_t* __restrict__ counts, uint32_t* __restrict__ sums,
                                                        int64_t n_chunks) {
  __shared__ uint32_t s_w[kChunksPerBlock];
  const int64_t c0 = ((int64_t)blockIdx.x * kChunksPerBlock + wave_id()) * kMaskChunks;
  uint32_t bits[kMaskChunks], all = 0;
  mask_bits(mask, n, c0, bits);                       // chunks past the end: zero
#pragma unroll
  for (int u = 0; u < kMaskChunks; ++u) {
    const uint32_t cnt = (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_scan((uint32_t)__popc(bits[u])), kWave - 1);
    if (lane_id() == 0 && c0 + u < n_chunks) counts[c0 + u] = cnt;
    all += cnt;
  }
  if (lane_id() == 0) s_w[wave_id()] = all;
  __syncthreads();
  if (threadIdx.x == 0) sums[blockIdx.x] = s_w[0] + s_w[1] + s_w[2] + s_w[3];
}

constexpr int kGroupChunks = kChunksPerBlock * kMaskChunks;
constexpr int kTotalsBlock = 1024, kTotalsWaves = kTotalsBlock / kWave;
typedef uint32_t q4u __attribute__((ext_vector_type(4), aligned(4)));       // the sums lie behind any number of counts
// out[0] = all set bytes, out[j] = those before j * step (j = 1 .. cuts).  sums become the groups' offsets, PER of them a
// thread and round.  The one workgroup is bound by the latency of a round: up to 1024 groups (16.8 MB of mask) are one
// round of one each (a microsecond less than by runs); more go by runs of 16, and the next round's are on their way
// while one is scanned.  Counting and listing no set byte, by rounds of 1024 / so / with two launches over the chip
// instead of this one, us: 4e8 bytes 103 / 95 / 106, 1.2e9 263 / 233 / 239, 2^31 464 / 399 / 392.
template <int PER>
__global__ __launch_bounds__(kTotalsBlock) void k_mask_totals(const uint8_t* __restrict__ mask, int64_t n,
                                                              const uint32_t* __restrict__ counts,
                                                              uint32_t* __restrict__ sums, int64_t n_groups, int64_t step,
                                                              int cuts, int64_t* __restrict__ out) {
  __shared__ uint32_t s_w[2][kTotalsWaves];
  uint32_t run = 0;                                   // set bytes before the round
  int turn = 0;
  constexpr int64_t kRound = kTotalsBlock * PER;
  uint32_t next[PER];
  const auto request = [&](int64_t g) {
    if constexpr (PER % 4 == 0) {
      if (g + PER <= n_groups) {
#pragma unroll
        for (int j = 0; j < PER; j += 4) {
          const q4u q = *reinterpret_cast<const q4u*>(sums + g + j);
          next[j] = q.x; next[j + 1] = q.y; next[j + 2] = q.z; next[j + 3] = q.w;
        }
        return;
      }
    }
#pragma unroll
    for (int j = 0; j < PER; ++j) next[j] = g + j < n_groups ? sums[g + j] : 0u;
  };
  request((int64_t)threadIdx.x * PER);
  for (int64_t g0 = 0; g0 < n_groups; g0 += kRound, turn ^= 1) {
    const int64_t g = g0 + (int64_t)threadIdx.x * PER;
    uint32_t v[PER], mine = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) { v[j] = next[j]; mine += v[j]; }
    if (g0 + kRound < n_groups) request(g + kRound);  // on its way while this round is scanned
    const uint32_t incl = wave_incl_scan(mine);
    if (lane_id() == kWave - 1) s_w[turn][wave_id()] = incl;
    __syncthreads();
    const uint32_t waves = row_incl_scan(s_w[turn][lane_id() % kTotalsWaves]);
    const int w = uniform_i32(wave_id());
    const uint32_t before = w ? (uint32_t)__builtin_amdgcn_readlane((int)waves, w - 1) : 0u;
    uint32_t at = run + before + incl - mine;
#pragma unroll
    for (int j = 0; j < PER; ++j) { const uint32_t c = v[j]; v[j] = at; at += c; }
    bool put = false;
    if constexpr (PER % 4 == 0) {
      put = g + PER <= n_groups;
#pragma unroll
      for (int j = 0; put && j < PER; j += 4)
        *reinterpret_cast<q4u*>(sums + g + j) = q4u{v[j], v[j + 1], v[j + 2], v[j + 3]};
    }
#pragma unroll
    for (int j = 0; !put && j < PER; ++j)
      if (g + j < n_groups) sums[g + j] = v[j];
    run += (uint32_t)__builtin_amdgcn_readlane((int)waves, kTotalsWaves - 1);
  }
  if (threadIdx.x == 0) st_host(out, (int64_t)run);
  __syncthreads();                                    // the offsets, which the same workgroup wrote
  for (int j = 1 + wave_id(); j <= cuts; j += kTotalsWaves) {
    const int64_t at = (int64_t)j * step, c = at / kChunk;
    if (at >= n) {
      if (lane_id() == 0) st_host(out + j, (int64_t)run);
      continue;
    }
    const int64_t c0 = c / kGroupChunks * kGroupChunks;
    uint32_t cnt = lane_id() < c - c0 ? counts[c0 + lane_id()] : 0u;
    for (int64_t i = c * kChunk + lane_id(); i < at; i += kWave) cnt += mask[i] != 0;
    cnt = wave_sum(cnt);
    if (lane_id() == 0) st_host(out + j, (int64_t)sums[c / kGroupChunks] + cnt);
  }
}

// Positions (and values) of a wave's four chunks.  They go through LDS and leave in order, as whole lines: with few
// set (a hundredth: 41 of 4096) in one piece, whose values are one round of loads in flight together.
template <bool GATHER, bool SCALE>
__global__ __launch_bounds__(kBlock) void k_mask_list(const uint8_t* __restrict__ mask, int64_t n,
                                                      const uint32_t* __restrict__ counts,
                                                      const uint32_t* __restrict__ offsets, int32_t* __restrict__ idx_out,
                                                      int64_t cap, int64_t n_chunks, const float* __restrict__ grad,
                                                      float factor, Parts values) {
  __shared__ int32_t s_idx[kChunksPerBlock][kChunk + kChunk / 16];
  const int64_t g0 = (int64_t)blockIdx.x * kGroupChunks, c0 = g0 + wave_id() * kMaskChunks;
  if (c0 >= n_chunks) return;
  uint32_t bits[kMaskChunks];
  mask_bits(mask, n, c0, bits);
  const uint32_t in_group = lane_id() < kGroupChunks && g0 + lane_id() < n_chunks ? counts[g0 + lane_id()] : 0u;
  const uint32_t upto = row_incl_scan(in_group);      // lane l < 16: set bytes of the group's chunks 0 .. l
  const int first = uniform_i32(wave_id()) * kMaskChunks;
  const uint32_t lead = first ? (uint32_t)__builtin_amdgcn_readlane((int)upto, first - 1) : 0u;
  const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)upto, first + kMaskChunks - 1) - lead;
  int64_t base = (int64_t)offsets[blockIdx.x] + lead;
  int32_t* own = s_idx[wave_id()];
  auto leave = [&](uint32_t have) {                   // the staged positions, in order
    __builtin_amdgcn_wave_barrier();                  // the wave's own LDS: its accesses stay in order
    const int64_t room = cap - base;
    const uint32_t put = room < (int64_t)have ? (uint32_t)(room < 0 ? 0 : room) : have;
    if (GATHER) {
      for (uint32_t j = lane_id(); j < put; j += kWave) {
        const int32_t i = own[j + j / 16];
        idx_out[base + j] = i;
        float v = grad[i];
        if (SCALE) v = v * factor;
        *values.at(base + j) = v;
      }
    } else {
      typedef int32_t i4v __attribute__((ext_vector_type(4), aligned(4)));
      for (uint32_t j = lane_id() * kVec; j < put; j += kWave * kVec) {
        const int32_t* q = own + j + j / 16;          // the quad lies in one group of 16
        const int32_t v[4] = {q[0], q[1], q[2], q[3]};
        if (j + kVec <= put) {
          *reinterpret_cast<i4v*>(idx_out + base + j) = i4v{v[0], v[1], v[2], v[3]};
        } else {
          for (uint32_t e = 0; j + e < put; ++e) idx_out[base + j + e] = v[e];
        }
      }
    }
    base += have;
    __builtin_amdgcn_wave_barrier();
  };
  const bool together = total <= (uint32_t)kChunk;
  uint32_t at0 = 0;
#pragma unroll
  for (int u = 0; u < kMaskChunks; ++u) {
    const uint32_t mine = (uint32_t)__popc(bits[u]), incl = wave_incl_scan(mine);
    const uint32_t count = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
    const int32_t i0 = (int32_t)((c0 + u) * kChunk + lane_id() * 16);
    uint32_t at = at0 + incl - mine;
    for (uint32_t left = bits[u]; left; left &= left - 1u, ++at) own[at + at / 16] = i0 + __ffs((int)left) - 1;
    if (together) at0 += count;
    else leave(count);
  }
  if (together) leave(at0);
}

// out[0] = all set bytes, out[j] = those before j * step (j = 1 .. cuts): a wave per cut, from the offsets.
__global__ __launch_bounds__(kBlock) void k_mask_cuts(const uint8_t* __restrict__ mask, int64_t n,
                                                      const uint32_t* __restrict__ offsets, int64_t step, int cuts,
                                                      int64_t* __restrict__ out) {
  const int j = (int)blockIdx.x * kChunksPerBlock + wave_id() + 1;
  if (j > cuts) return;
  const int64_t at = (int64_t)j * step, c = at / kChunk;
  if (at >= n) {
    if (lane_id() == 0) out[j] = out[0];
    return;
  }
  uint32_t cnt = 0;
  for (int64_t i = c * kChunk + lane_id(); i < at; i += kWave) cnt += mask[i] != 0;
  cnt = wave_sum(cnt);
  if (lane_id() == 0) out[j] = (int64_t)offsets[c] + cnt;
}

}  // namespace sga

using namespace sga;

// Exclusive scan of uint32 counts in place (+ int64 total), shared by the
// compaction-style entry points.  Implemented in scan.hip.
namespace sga {
int exclusive_scan_u32(uint32_t* data, int64_t n, int64_t* total,
                       hipStream_t st);
int64_t scan_scratch_entries(int64_t n);
}

extern "C" int sga_scatter_selected(float* dst, const int32_t* idx,
                                    const float* src, int64_t k, int64_t n_dst,
                                    void* stream) {
  if (k == 0) return SGA_OK;
  if (!dst || !idx || !src || k < 0 || n_dst >= (1ll << 31)) {
    set_error("sga_scatter_selected: bad argument (k=%lld n_dst=%lld, needs < 2^31)",
              (long long)k, (long long)n_dst);
    return SGA_ERR_ARG;
  }
  hipLaunchKernelGGL(k_scatter, dim3(stream_grid(k, kBlock)), dim3(kBlock), 0,
                     (hipStream_t)stream, dst, idx, src, k, n_dst);
  return check_launch("sga_scatter_selected");
}

static int pack_selected(const char* who, float* grad, const int32_t* idx, void* values, int values_dtype, float factor,
                         int64_t k, int64_t n_grad, int64_t split, int64_t* below, void* stream) {
  if (!grad || !idx || !values || k < 0 || n_grad >= (1ll << 31) ||
      (values_dtype != SGA_F32 && values_dtype != SGA_BF16)) {
    set_error("%s: bad argument (k=%lld n_grad=%lld dtype=%d, needs < 2^31)", who, (long long)k, (long long)n_grad,
              values_dtype);
    return SGA_ERR_ARG;
  }
  dim3 grid(stream_grid(k, kBlock) + (below ? 1u : 0u)), block(kBlock);
  hipStream_t st = (hipStream_t)stream;
  const bool scale = factor != 1.0f;
  if (values_dtype == SGA_BF16) {
    if (scale) hipLaunchKernelGGL((k_pack<true, true>), grid, block, 0, st, grad, idx, values, factor, k, n_grad, split, below);
    else hipLaunchKernelGGL((k_pack<true, false>), grid, block, 0, st, grad, idx, values, factor, k, n_grad, split, below);
  } else {
    if (scale) hipLaunchKernelGGL((k_pack<false, true>), grid, block, 0, st, grad, idx, values, factor, k, n_grad, split, below);
    else hipLaunchKernelGGL((k_pack<false, false>), grid, block, 0, st, grad, idx, values, factor, k, n_grad, split, below);
  }
  return check_launch(who);
}

extern "C" int sga_pack_selected(float* grad, const int32_t* idx, void* values,
                                 int values_dtype, float factor, int64_t k,
                                 int64_t n_grad, void* stream) {
  if (k == 0) return SGA_OK;
  return pack_selected("sga_pack_selected", grad, idx, values, values_dtype, factor, k, n_grad, 0, nullptr, stream);
}

extern "C" int sga_pack_selected_split(float* grad, const int32_t* idx, void* values, int values_dtype, float factor,
                                       int64_t k, int64_t n_grad, int64_t split, int64_t* below, void* stream) {
  if (!below || k < 1) {
    set_error("sga_pack_selected_split: bad argument (k=%lld, below is required)", (long long)k);
    return SGA_ERR_ARG;
  }
  return pack_selected("sga_pack_selected_split", grad, idx, values, values_dtype, factor, k, n_grad, split, below,
                       stream);
}

// The parts' arrays as Parts; false (with the error text) where they do not fit together.
static bool parts_of(const char* who, float* const* base, const int64_t* counts, int n_parts, Parts* p, int64_t* total) {
  bool ok = base && counts && n_parts >= 1 && n_parts <= kParts;
  *total = 0;
  p->count = n_parts;
  for (int j = 0; ok && j < n_parts; ++j) {
    ok = counts[j] >= 0 && (base[j] || counts[j] == 0);
    p->base[j] = reinterpret_cast<float*>(reinterpret_cast<uintptr_t>(base[j]) - (uintptr_t)*total * sizeof(float));
    *total += counts[j];
    p->end[j] = *total;
  }
  if (!ok) set_error("%s: bad parts (1 <= n_parts=%d <= %d, counts >= 0)", who, n_parts, kParts);
  return ok;
}

extern "C" int sga_scatter_selected_parts(float* dst, const int32_t* idx, const float* const* src, const int64_t* counts,
                                          int n_parts, int64_t n_dst, void* stream) {
  const char* who = "sga_scatter_selected_parts";
  Parts p = {};
  int64_t k = 0;
  if (!parts_of(who, const_cast<float* const*>(src), counts, n_parts, &p, &k)) return SGA_ERR_ARG;
  if (k == 0) return SGA_OK;
  if (!dst || !idx || n_dst >= (1ll << 31)) {
    set_error("%s: bad argument (n_dst=%lld, needs < 2^31)", who, (long long)n_dst);
    return SGA_ERR_ARG;
  }
  hipLaunchKernelGGL(k_scatter_parts, dim3(stream_grid(k, kBlock)), dim3(kBlock), 0, (hipStream_t)stream, dst, idx, p, k,
                     n_dst);
  return check_launch(who);
}

static const int64_t kNormMaxBlocks = 2048;
// largest k of the allocation-free norm: the int32 index domain of a bucket (kernels.py:154)
static const int64_t kNoAllocNormMaxK = SGA_NOALLOC_NORM_MAX_K;

static int xlog_of(int x);

extern "C" int sga_block_reduce(const float* g, int64_t n, int x, int mode, float* out,
                                void* stream) {
  if (n == 0) return SGA_OK;
  if (!g || !out || n < 0 || xlog_of(x) < 0 || (mode != 0 && mode != 1)) {
    set_error("sga_block_reduce: bad argument (x=%d mode=%d)", x, mode);
    return SGA_ERR_ARG;
  }
  const int64_t nb = cdiv64(n, x);
  const int lanes = x < kWave ? x : kWave;
  dim3 grid(stream_grid(nb, kChunksPerBlock * (kWave / lanes))), block(kBlock);
  if (mode == 0) hipLaunchKernelGGL((k_block_reduce<0>), grid, block, 0, (hipStream_t)stream, g, n, x, lanes, out, nb);
  else hipLaunchKernelGGL((k_block_reduce<1>), grid, block, 0, (hipStream_t)stream, g, n, x, lanes, out, nb);
  return check_launch("sga_block_reduce");
}

extern "C" int sga_block_any(const uint8_t* mask, int64_t n, int x, uint8_t* any_out, void* stream) {
  if (n == 0) return SGA_OK;
  if (!mask || !any_out || n < 0 || xlog_of(x) < 0) {
    set_error("sga_block_any: bad argument (x=%d)", x);
    return SGA_ERR_ARG;
  }
  const int64_t nb = cdiv64(n, x);
  const int lanes = x < kWave ? x : kWave;
  hipLaunchKernelGGL(k_block_any, dim3(stream_grid(nb, kChunksPerBlock * (kWave / lanes))),
                     dim3(kBlock), 0, (hipStream_t)stream, mask, n, x, lanes, any_out, nb);
  return check_launch("sga_block_any");
}

extern "C" int sga_expand_blocks(const uint8_t* bmask, int x, int64_t n, uint8_t* out, void* stream) {
  if (n == 0) return SGA_OK;
  const int xl = xlog_of(x);
  if (!bmask || !out || n < 0 || xl < 0) {
    set_error("sga_expand_blocks: bad argument (x=%d)", x);
    return SGA_ERR_ARG;
  }
  hipLaunchKernelGGL(k_expand_blocks, dim3(stream_grid(n, kBlock)), dim3(kBlock), 0,
                     (hipStream_t)stream, bmask, xl, n, out);
  return check_launch("sga_expand_blocks");
}

extern "C" int64_t sga_norm_partials(int64_t n) {
  return stream_grid(n, (int64_t)kBlock * kVec, kNormMaxBlocks);
}

extern "C" int sga_compact_norm_sq(const float* values, int64_t k,
                                   float* partials, float* total, void* stream) {
  if (k == 0) return SGA_OK;
  if (!values || !partials || !total || k < 0) {
    set_error("sga_compact_norm_sq: bad argument");
    return SGA_ERR_ARG;
  }
  const unsigned nb = (unsigned)sga_norm_partials(k);
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL((k_norm_stage1<false>), dim3(nb), dim3(kBlock), 0, st,
                     values, (const uint8_t*)nullptr, k, partials,
                     quads_ok(values, 4));
  hipLaunchKernelGGL(k_norm_stage2, dim3(1), dim3(kBlock), 0, st, partials,
                     (int64_t)nb, total, total);
  return check_launch("sga_compact_norm_sq");
}

extern "C" int sga_compact_norm_sq_from(const float* values, int64_t k, float* partials, const float* before,
                                        float* total, void* stream) {
  if (!values || !partials || !total || k < 1) {
    set_error("sga_compact_norm_sq_from: bad argument (k=%lld)", (long long)k);
    return SGA_ERR_ARG;
  }
  const unsigned nb = (unsigned)sga_norm_partials(k);
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL((k_norm_stage1<false>), dim3(nb), dim3(kBlock), 0, st, values, (const uint8_t*)nullptr, k,
                     partials, quads_ok(values, 4));
  hipLaunchKernelGGL(k_norm_stage2, dim3(1), dim3(kBlock), 0, st, partials, (int64_t)nb, before, total);
  return check_launch("sga_compact_norm_sq_from");
}

// The stage-1 partials of the allocation-free norm: one array per device,
// held by every GPU the library runs on until the process ends (8 KiB).  In
// host code the array's name is only a stand-in for the symbol; the device
// address is resolved once per device and kept in g_norm_scratch_ptr.
static __device__ __align__(256) float scratch[kNormMaxBlocks];

static const int kNoAllocMaxDevices = 64;
static std::mutex g_norm_scratch_mu;
static float* g_norm_scratch_ptr[kNoAllocMaxDevices] = {};

// Device address of `scratch` on the current device, or null with the error
// text set.  The first call on a device resolves the symbol (no allocation).
static float* norm_scratch_of_current_device(const char* who) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kNoAllocMaxDevices) {
    set_error("%s: cannot name the current device (%s, device %d, at most %d supported)", who,
              hipGetErrorString(e), dev, kNoAllocMaxDevices);
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_norm_scratch_mu);
  if (!g_norm_scratch_ptr[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      set_error("%s: hipGetSymbolAddress(scratch) failed on device %d: %s", who, dev,
                hipGetErrorString(e));
      return nullptr;
    }
    g_norm_scratch_ptr[dev] = static_cast<float*>(ptr);
  }
  return g_norm_scratch_ptr[dev];
}

extern "C" int sga_compact_norm_sq_noalloc(const float* values, int64_t k, float* total,
                                           void* stream) {
  if (k == 0) return SGA_OK;
  if (!values || !total || k < 0) {
    set_error("sga_compact_norm_sq_noalloc: bad argument");
    return SGA_ERR_ARG;
  }
  if (k > kNoAllocNormMaxK) {
    set_error("sga_compact_norm_sq_noalloc: k=%lld exceeds the supported maximum %lld "
              "(use sga_compact_norm_sq with a caller workspace)",
              (long long)k, (long long)kNoAllocNormMaxK);
    return SGA_ERR_ARG;
  }
  float* partials = norm_scratch_of_current_device("sga_compact_norm_sq_noalloc");
  if (!partials) return SGA_ERR_LAUNCH;
  // same two kernels, same grid as sga_compact_norm_sq: the result has the same bits.  Stage 1
  // overwrites the nb slots stage 2 reads, so nothing in the array has to start at zero.
  const unsigned nb = (unsigned)sga_norm_partials(k);
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL((k_norm_stage1<false>), dim3(nb), dim3(kBlock), 0, st, values,
                     (const uint8_t*)nullptr, k, partials, quads_ok(values, 4));
  hipLaunchKernelGGL(k_norm_stage2, dim3(1), dim3(kBlock), 0, st, partials, (int64_t)nb, total, total);
  return check_launch("sga_compact_norm_sq_noalloc");
}

extern "C" int sga_masked_norm_sq(const float* grad, const uint8_t* mask,
                                  int64_t n, float* partials, float* total,
                                  void* stream) {
  if (n == 0) return SGA_OK;
  if (!grad || !mask || !partials || !total || n < 0) {
    set_error("sga_masked_norm_sq: bad argument");
    return SGA_ERR_ARG;
  }
  const unsigned nb = (unsigned)sga_norm_partials(n);
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL((k_norm_stage1<true>), dim3(nb), dim3(kBlock), 0, st, grad,
                     mask, n, partials, quads_ok(grad, 4) && quads_ok(mask, 1));
  hipLaunchKernelGGL(k_norm_stage2, dim3(1), dim3(kBlock), 0, st, partials,
                     (int64_t)nb, total, total);
  return check_launch("sga_masked_norm_sq");
}

// g[i] *= coeff where mask[i] (every i when mask is null): the explicit clip
// scale, one fp32 multiply per touched coordinate.
template <bool MASKED>
__global__ __launch_bounds__(kBlock) void k_scale_masked(float* __restrict__ g,
                                                         const uint8_t* __restrict__ mask,
                                                         int64_t n, float coeff, bool vec) {
  const int64_t stride = (int64_t)gridDim.x * kBlock * kVec;
  for (int64_t i = ((int64_t)blockIdx.x * kBlock + threadIdx.x) * kVec; i < n; i += stride) {
    uint32_t mk[4] = {1u, 1u, 1u, 1u};
    if (MASKED) {
      load4_u8(mask, i, n, mk, vec);
      if (!(mk[0] | mk[1] | mk[2] | mk[3])) continue;   // untouched lanes move no gradient bytes
    }
    float v[4];
    load4_f32(g, i, n, v, vec);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = mk[e] ? v[e] * coeff : v[e];
    store4_f32(g, i, n, v, vec);
  }
}

extern "C" int sga_scale_masked(float* grad, const uint8_t* mask, int64_t n, float coeff,
                                void* stream) {
  if (n == 0) return SGA_OK;
  if (!grad || n < 0) { set_error("sga_scale_masked: bad argument"); return SGA_ERR_ARG; }
  dim3 grid(stream_grid(n, (int64_t)kBlock * kVec, 1 << 22)), block(kBlock);
  const bool vec = quads_ok(grad, 4) && quads_ok(mask, 1);
  if (mask)
    hipLaunchKernelGGL((k_scale_masked<true>), grid, block, 0, (hipStream_t)stream, grad, mask, n, coeff, vec);
  else
    hipLaunchKernelGGL((k_scale_masked<false>), grid, block, 0, (hipStream_t)stream, grad, mask, n, coeff, vec);
  return check_launch("sga_scale_masked");
}

static int span_args(const char* who, const sga_span_record* recs, int n_recs, int64_t total_spans) {
  if (recs && n_recs > 0 && total_spans > 0 && total_spans < (1ll << 31)) return SGA_OK;
  set_error("%s: bad argument (n_recs=%d spans=%lld)", who, n_recs, (long long)total_spans);
  return SGA_ERR_ARG;
}

extern "C" int sga_norm_sq_multi(const sga_span_record* recs, int n_recs, int64_t total_spans,
                                 float* partials, float* total, void* stream) {
  if (int rc = span_args("sga_norm_sq_multi", recs, n_recs, total_spans)) return rc;
  if (!partials || !total) { set_error("sga_norm_sq_multi: bad argument"); return SGA_ERR_ARG; }
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(k_norm_multi, dim3((unsigned)total_spans), dim3(kBlock), 0, st, recs, n_recs, partials);
  hipLaunchKernelGGL(k_norm_multi_fold, dim3(1), dim3(kFoldBlock), 0, st, partials, total_spans, total);
  return check_launch("sga_norm_sq_multi");
}

extern "C" int sga_scale_multi(const sga_span_record* recs, int n_recs, int64_t total_spans,
                               float coeff, void* stream) {
  if (int rc = span_args("sga_scale_multi", recs, n_recs, total_spans)) return rc;
  hipLaunchKernelGGL(k_scale_multi, dim3((unsigned)total_spans), dim3(kBlock), 0, (hipStream_t)stream, recs,
                     n_recs, coeff);
  return check_launch("sga_scale_multi");
}

static int xlog_of(int x) {
  if (x < 1 || x > 1024 || (x & (x - 1))) return -1;
  int l = 0;
  while ((1 << l) < x) ++l;
  return l;
}

extern "C" int sga_gather_selected_blocks(const float* grad, const uint8_t* mask,
                                          const int32_t* block_idx,
                                          float* values, int64_t kb, int x,
                                          float factor, int64_t n_grad,
                                          void* stream) {
  if (kb == 0) return SGA_OK;
  const int xl = xlog_of(x);
  if (!grad || !mask || !block_idx || !values || kb < 0 || xl < 0 ||
      n_grad >= (1ll << 31)) {
    set_error("sga_gather_selected_blocks: bad argument (x=%d must be a power of two in [1,1024]; n < 2^31)", x);
    return SGA_ERR_ARG;
  }
  const int64_t total = kb * x;
  dim3 grid(stream_grid(total, kBlock)), block(kBlock);
  if (factor != 1.0f)
    hipLaunchKernelGGL((k_gather_blocks<true>), grid, block, 0, (hipStream_t)stream, grad, mask, block_idx, values, total, xl, factor, n_grad);
  else
    hipLaunchKernelGGL((k_gather_blocks<false>), grid, block, 0, (hipStream_t)stream, grad, mask, block_idx, values, total, xl, factor, n_grad);
  return check_launch("sga_gather_selected_blocks");
}

extern "C" int sga_scatter_selected_blocks(float* dst, const uint8_t* mask,
                                           const int32_t* block_idx,
                                           const float* src, int64_t kb, int x,
                                           int64_t n_dst, void* stream) {
  if (kb == 0) return SGA_OK;
  const int xl = xlog_of(x);
  if (!dst || !mask || !block_idx || !src || kb < 0 || xl < 0 ||
      n_dst >= (1ll << 31)) {
    set_error("sga_scatter_selected_blocks: bad argument (x=%d)", x);
    return SGA_ERR_ARG;
  }
  const int64_t total = kb * x;
  hipLaunchKernelGGL(k_scatter_blocks, dim3(stream_grid(total, kBlock)),
                     dim3(kBlock), 0, (hipStream_t)stream, dst, mask, block_idx,
                     src, total, xl, n_dst);
  return check_launch("sga_scatter_selected_blocks");
}

// Entries the caller must provide for chunk_counts: one per 1024-byte chunk
// plus the scan's workgroup-sum scratch.
extern "C" int64_t sga_mask_chunks(int64_t n) {
  const int64_t nc = cdiv64(n, kChunk);
  return nc + scan_scratch_entries(nc);
}
static inline int64_t n_chunks_of(int64_t n) { return cdiv64(n, kChunk); }

// total[0], and with cuts > 0 total[j] = set bytes before j * step
static int mask_count(const char* who, const uint8_t* mask, int64_t n, uint32_t* chunk_counts, int64_t* total,
                      int64_t step, int cuts, void* stream) {
  if (!total || n < 0 || n >= (1ll << 31) || (n > 0 && (!mask || !chunk_counts)) || step < 0 || cuts < 0) {
    set_error("%s: bad argument (n=%lld, int32 indices need n < 2^31)", who, (long long)n);
    return SGA_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  const int64_t nc = n_chunks_of(n);
  if (nc > 0)
    hipLaunchKernelGGL(k_mask_count, dim3((unsigned)cdiv64(nc, kChunksPerBlock * kMaskChunks)), dim3(kBlock), 0, st, mask,
                       n, chunk_counts, nc);
  int rc = exclusive_scan_u32(chunk_counts, nc, total, st);
  if (rc) return rc;
  if (step > n) step = n;                // the same answers, and j * step cannot wrap around
  if (cuts > 0)
    hipLaunchKernelGGL(k_mask_cuts, dim3((unsigned)cdiv64(cuts, kChunksPerBlock)), dim3(kBlock), 0, st, mask, n,
                       chunk_counts, step, cuts, total);
  return check_launch(who);
}

extern "C" int sga_mask_count(const uint8_t* mask, int64_t n, uint32_t* chunk_counts, int64_t* total, void* stream) {
  return mask_count("sga_mask_count", mask, n, chunk_counts, total, 0, 0, stream);
}

extern "C" int sga_mask_count_cuts(const uint8_t* mask, int64_t n, uint32_t* chunk_counts, int64_t step, int cuts,
                                   int64_t* totals, void* stream) {
  return mask_count("sga_mask_count_cuts", mask, n, chunk_counts, totals, step, cuts, stream);
}

extern "C" int sga_mask_fill(const uint8_t* mask, int64_t n,
                             const uint32_t* chunk_offsets, int32_t* idx_out,
                             int64_t idx_capacity, void* stream) {
  if (n == 0) return SGA_OK;
  if (!mask || !chunk_offsets || (!idx_out && idx_capacity > 0) || n < 0 ||
      n >= (1ll << 31)) {
    set_error("sga_mask_fill: bad argument");
    return SGA_ERR_ARG;
  }
  const int64_t nc = n_chunks_of(n);
  hipLaunchKernelGGL(k_mask_fill, dim3((unsigned)cdiv64(nc, kChunksPerBlock * kMaskChunks)), dim3(kBlock), 0,
                     (hipStream_t)stream, mask, n, chunk_offsets, idx_out, idx_capacity, nc);
  return check_launch("sga_mask_fill");
}

static inline int64_t n_groups_of(int64_t n) { return cdiv64(n_chunks_of(n), kGroupChunks); }
// Words of the scratch of sga_mask_totals / sga_mask_list: a count per chunk, an offset per group of 16.
extern "C" int64_t sga_mask_list_words(int64_t n) { return n_chunks_of(n) + n_groups_of(n); }

extern "C" int sga_mask_totals(const uint8_t* mask, int64_t n, uint32_t* scratch, int64_t step, int cuts, int64_t* totals,
                               void* stream) {
  if (!mask || !scratch || !totals || n < 1 || n >= (1ll << 31) || step < 0 || cuts < 0) {
    set_error("sga_mask_totals: bad argument (n=%lld, int32 indices need n < 2^31)", (long long)n);
    return SGA_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  const int64_t nc = n_chunks_of(n), ng = n_groups_of(n);
  if (step > n) step = n;                // the same answers, and j * step cannot wrap around
  hipLaunchKernelGGL(k_mask_groups, dim3((unsigned)ng), dim3(kBlock), 0, st, mask, n, scratch, scratch + nc, nc);
  const auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(1), dim3(kTotalsBlock), 0, st, mask, n, scratch, scratch + nc, ng, step, cuts, totals);
  };
  ng <= kTotalsBlock ? launch(k_mask_totals<1>) : launch(k_mask_totals<16>);
  return check_launch("sga_mask_totals");
}

extern "C" int sga_mask_list(const uint8_t* mask, int64_t n, const uint32_t* scratch, int32_t* idx_out, int64_t capacity,
                             const float* grad, float factor, float* const* values, const int64_t* counts, int n_parts,
                             void* stream) {
  const char* who = "sga_mask_list";
  if (!mask || !scratch || (!idx_out && capacity > 0) || n < 1 || n >= (1ll << 31) || capacity < 0) {
    set_error("%s: bad argument (n=%lld capacity=%lld)", who, (long long)n, (long long)capacity);
    return SGA_ERR_ARG;
  }
  Parts p = {};
  int64_t room = 0;
  if (grad) {
    if (!parts_of(who, values, counts, n_parts, &p, &room)) return SGA_ERR_ARG;
    if (capacity > room) {
      set_error("%s: the parts hold %lld values, the list %lld", who, (long long)room, (long long)capacity);
      return SGA_ERR_ARG;
    }
  }
  hipStream_t st = (hipStream_t)stream;
  const int64_t nc = n_chunks_of(n);
  const dim3 grid((unsigned)n_groups_of(n)), block(kBlock);
  const uint32_t* off = scratch + nc;
  if (!grad)
    hipLaunchKernelGGL((k_mask_list<false, false>), grid, block, 0, st, mask, n, scratch, off, idx_out, capacity, nc, grad,
                       factor, p);
  else if (factor != 1.0f)
    hipLaunchKernelGGL((k_mask_list<true, true>), grid, block, 0, st, mask, n, scratch, off, idx_out, capacity, nc, grad,
                       factor, p);
  else
    hipLaunchKernelGGL((k_mask_list<true, false>), grid, block, 0, st, mask, n, scratch, off, idx_out, capacity, nc, grad,
                       factor, p);
  return check_launch(who);
}
