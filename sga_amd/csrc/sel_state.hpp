// State of a select in its workspace, the hand-over of a sample's keys between the workgroups of one
// launch (sample_pick_body), and of the small buckets' counts to the finish.  No HIP in here: the host compiles it too.
#pragma once
#include <stddef.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define SGA_HOST_DEVICE __host__ __device__
#else
#define SGA_HOST_DEVICE
#endif

namespace sga {

struct SelState {
  uint32_t k;
  uint32_t prefix;
  uint32_t krem;
  uint32_t thresh_bits;
  uint32_t need;
  uint32_t n_gt;
  uint32_t n_eq;
  uint32_t nonfinite;
  uint32_t status;
  uint32_t total;
  uint32_t n_selected;
  uint32_t path;
  // sampled-bracket path
  uint32_t t_lo;        // candidates are keys in [t_lo, t_hi)
  uint32_t t_hi;
  uint32_t n_hi;        // keys >= t_hi
  uint32_t cand_count;  // keys in the bracket (may exceed capacity)
  uint32_t bracket_ok;  // 1: the sampled bracket holds the k-th key; radix passes skip
  uint32_t overflow;    // a candidate segment ran out of room
  uint32_t skip;        // 1: kernels driven by this state do nothing
  uint32_t done[3];     // per-level "workgroups finished" tickets (last one scans)
  uint32_t spec;        // 1: the single-sweep step committed on the sampled bracket (no way back)
  uint32_t negative;    // 1: an fp32 score array held a value below zero (magnitudes were ranked)
  uint32_t redone;      // 1: an out-of-place single-sweep step missed its bracket and was redone
  uint32_t in_sample;   // sample keys inside the bracket (~0: open below, nothing bounds them)
  uint32_t ticket;      // k_settle: workgroups that are done
  uint32_t edge_cnt;    // k_settle: entries of the edge list
  uint32_t edge_inv;    // k_settle: ~(smallest key of the edge list), and ...
  uint32_t edge_max;    // ... the largest, by atomic maxima (0: none)
  uint32_t ties_left;   // the settlement has left the ties to k_tail
  uint32_t tail_ticket; // k_tail: items handed out, and ...
  uint32_t tail_done;   // ... finished
  uint32_t finish_ticket; // k_small_finish: workgroups that have begun; the first one judges the bracket ...
  uint32_t verdict;     // ... 1: it holds the k-th key, 2: all of them go over the data again
  uint32_t redo_step;   // passes of that which are done
  uint32_t sampled[16]; // sample_pick_body: the launch that a workgroup of the sample has finished in
  uint32_t pad_[12];
};
static_assert(sizeof(SelState) == 256, "whole cache lines");

// The hand-over's memory holds anything before the launch: nobody clears a workspace.  Words there that happen
// to hold the launch's number let a workgroup pick from keys that have not arrived, or several workgroups from
// different ones.  So the pick is made for any words: what is read as a key is one (31 bits: it indexes a
// histogram in LDS), and the two ends of the bracket are written as one word, so that they are always one
// picking workgroup's own.  The select is exact for any bracket; a single-sweep step in place, which commits on
// it, reports a miss like any other (status 3).
SGA_HOST_DEVICE static inline uint32_t sampled_key(unsigned long long word, int half) {
  return (uint32_t)(word >> (32 * half)) & 0x7FFFFFFFu;
}
// Number of the count-th launch of the library that takes a sample: different for 2^31 launches, odd and so never
// zero as a cleared mark is, and spread over all 32 bits (consecutive small numbers are what index lists, counts
// and flags in recycled memory look like).  A recorded graph repeats its numbers: its marks are zero again at
// every start because the pick clears them and so does the kernel behind it (an early pick's clearing may come
// before the last mark); those of the small buckets' front are cleared by the kernel behind it alone.
SGA_HOST_DEVICE static inline uint32_t launch_number(uint32_t count) { return (2u * count + 1u) * 0x9E3779B1u; }
constexpr int kStateWords = sizeof(SelState) / 8;
constexpr int kBracketWord = offsetof(SelState, t_lo) / 8;
static_assert(offsetof(SelState, t_lo) % 8 == 0 && offsetof(SelState, t_hi) == offsetof(SelState, t_lo) + 4,
              "both ends of the bracket in one aligned word");
static_assert(offsetof(SelState, k) == 0, "word 0 is the rank");
// Word w of the state that the pick leaves: rank and bracket, everything else zero.
SGA_HOST_DEVICE static inline unsigned long long picked_word(int w, uint32_t k, uint32_t t_lo, uint32_t t_hi) {
  return w == 0 ? k : w == kBracketWord ? (unsigned long long)t_hi << 32 | t_lo : 0ull;
}

// What a chunk's two words carry from the sweep to the finish, numbers up to 1024 in halves whose sums over the eight
// chunks of a thread fit (an instruction per chunk is 0.07 us of the finish at 8 M coordinates):
//   a   keys above the bracket | ten bits of the bracket's tag | listed keys
//   b   keys equal to the lower end | a value was negative | no bracket, or no room | eight more of the tag |
//       non-finite keys
struct SmallChunk {
  static constexpr uint32_t kNumbers = 0x07FF07FFu, kNegative = 1u << 11, kLost = 1u << 12;
  uint32_t a, b;
  // the words of a chunk without a key in it, under the bracket [lo, hi)
  SGA_HOST_DEVICE static inline SmallChunk none(uint32_t lo, uint32_t hi) {
    uint32_t x = lo * 0x9E3779B1u ^ hi * 0x85EBCA6Bu;
    x = (x ^ (x >> 15)) * 0x2C1B3C6Du;
    return SmallChunk{(x & 0xF800F800u), ((x << 8) & 0xF8000000u) | ((x >> 3) & 0xE000u)};
  }
  SGA_HOST_DEVICE static inline SmallChunk of(uint32_t lo, uint32_t hi, uint32_t above, uint32_t listed, uint32_t equal,
                                              uint32_t nonfinite, bool negative, bool lost) {
    const SmallChunk z = none(lo, hi);
    return SmallChunk{z.a | above | listed << 16,
                      z.b | equal | nonfinite << 16 | (negative ? kNegative : 0u) | (lost ? kLost : 0u)};
  }
  // off_a, off_b: where words differ from none() of the state's bracket.  True: a chunk of another bracket, or a lost one.
  SGA_HOST_DEVICE static inline bool wrong(uint32_t off_a, uint32_t off_b) {
    return ((off_a | (off_b & ~kNegative)) & ~kNumbers) != 0u;
  }
};

}  // namespace sga
