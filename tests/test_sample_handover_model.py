"""Host-side models of how the workgroups of ``k_sample_pick`` and
``k_small_front`` (csrc/select_impl.hpp, csrc/small_select.hpp) hand their
sample keys and the bracket over inside one launch, and the pieces of it that
the host can compile (csrc/sel_state.hpp).

A workgroup stores its keys, then the launch's number as its mark, then looks
at all marks; whoever sees every mark reads all keys, picks a bracket and
writes the state, which also clears the marks.  The memory is the caller's and
holds anything before: marks that happen to equal the number let a workgroup
pick from keys that are not there yet.  The model runs every order of the
steps of three workgroups over every such memory and checks what the select
needs: a key indexes the pick's histogram in range, and the bracket left
behind is one picking workgroup's own.  The protocol that this one replaced
(keys as they come, the two ends as two stores) gives neither.

In the small buckets' front others wait for the bracket.  There the first
workgroup clears the state and the list's counters before its mark, a pick
writes the bracket and its copies alone, and the finish, a kernel behind it,
clears marks and copies.  The second model adds a sweeping workgroup and the
finish's judgement: whatever the memory held and in whatever order things
happen, a select that the finish accepts has counted all of its keys by the
state's own bracket, and everything else is done again over the data."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
GROUPS, NUMBER, BINS, SHIFT = 3, 7, 8192, 18
OWN = (0x10000000, 0x20000000, 0x30000000)             # what the workgroups store
STALE = 0xF0000005                                     # what the memory held, bit 31 set


def _runs(marks, masked, one_word):
    """All ends of one launch: ``(bracket, brackets picked, worst bin, marks left)``."""
    ends, seen = set(), set()
    # per workgroup: 0 store keys, 1 store mark, 2 look, 3 read and pick, 4 (and 5) write the state, None done
    start = ((0,) * GROUPS, (STALE,) * GROUPS, tuple(marks), (None, None), ((),) * GROUPS, -1)
    todo = [start]
    while todo:
        state = todo.pop()
        if state in seen:
            continue
        seen.add(state)
        pcs, words, marks_, bracket, picks, worst = state
        if all(pc is None for pc in pcs):
            ends.add((bracket, tuple(p for p in picks if p), worst, marks_))
            continue
        for g, pc in enumerate(pcs):
            if pc is None:
                continue
            w, m, b, p, bad, nxt = list(words), list(marks_), list(bracket), list(picks), worst, pc + 1
            if pc == 0:
                w[g] = OWN[g]
            elif pc == 1:
                m[g] = NUMBER
            elif pc == 2:
                nxt = 3 if all(x == NUMBER for x in m) else None
            elif pc == 3:
                keys = [x & 0x7FFFFFFF if masked else x for x in w]
                bad = max(bad, max(k >> SHIFT for k in keys))
                p[g] = (min(keys), max(keys) + 1)
            elif pc == 4:
                m = [0] * GROUPS
                b = list(p[g]) if one_word else [p[g][0], b[1]]
                nxt = None if one_word else 5
            else:
                b[1] = p[g][1]
                nxt = None
            todo.append((pcs[:g] + (nxt,) + pcs[g + 1:], tuple(w), tuple(m), tuple(b), tuple(p), bad))
    return ends


_MEMORIES = [[NUMBER * (bits >> g & 1) for g in range(GROUPS)] for bits in range(1 << GROUPS)]


@pytest.mark.parametrize("marks", _MEMORIES)
def test_any_memory_leaves_a_bracket_of_one_pick(marks):
    for bracket, picks, worst, left in _runs(marks, masked=True, one_word=True):
        assert picks and bracket in picks and bracket[0] < bracket[1]
        assert worst < BINS
        if not any(marks):                                # marks cleared before: the launch's own keys
            assert set(picks) == {(min(OWN), max(OWN) + 1)} and not any(left)


def test_the_replaced_protocol_does_neither():
    ends = [e for m in _MEMORIES for e in _runs(m, masked=False, one_word=False)]
    assert any(worst >= BINS for _, _, worst, _ in ends)
    assert any(bracket not in picks for bracket, picks, _, _ in ends)
    # on cleared marks it was sound
    assert all(b in p and w < BINS for b, p, w, _ in _runs([0] * GROUPS, masked=False, one_word=False))


def test_a_mark_can_come_after_the_clearing():
    """Which is why the next kernel clears the marks again: a recorded graph starts every
    replay with the same number."""
    assert any(any(left) for m in _MEMORIES for *_, left in _runs(m, masked=True, one_word=True))


# The front: two workgroups of the sample, two that sweep, and the finish.  A sweeping workgroup has two keys; one of
# them lies in either bracket that a pick can leave here, so that each reserves one entry of the list's counter.
PAIR = (0x10000000, 0x20000000)


def _front(marks, copy_held, counter_held, state_held, clears=True, tags=True):
    """All ends of one launch of the front: ``(accepted, brackets the sweeps used, bracket in the state, listed,
    counter)``."""
    ends, seen = set(), set()
    # sample: 0 clear (the first alone), 1 store keys, 2 store mark, 3 look, 4 read and pick, 5 copies, 6 state, None
    # sweep:  0 look for the bracket (or give up), 1 reserve and write the chunk's words, None
    start = ((0, 1), (0, 0), (STALE, STALE), tuple(marks), (None, None), copy_held, counter_held, state_held,
             (None, None), 0)
    todo = [start]
    while todo:
        at = todo.pop()
        if at in seen:
            continue
        seen.add(at)
        pcs, spcs, words, marks_, picks, copy, counter, bracket, used, listed = at
        if all(pc is None for pc in pcs + spcs):
            # the finish: of one bracket, the state's, nobody lost, and as many listed as the counter says
            ok = listed == counter and (not tags or all(u == bracket for u in used))
            ends.add((ok, used, bracket, listed, counter))
            continue
        for g, pc in enumerate(pcs):
            if pc is None:
                continue
            w, m, p, cp, cn, b, nxt = list(words), list(marks_), list(picks), copy, counter, bracket, pc + 1
            if pc == 0:
                if clears:
                    cn, b = 0, None
            elif pc == 1:
                w[g] = PAIR[g]
            elif pc == 2:
                m[g] = NUMBER
            elif pc == 3:
                nxt = 4 if all(x == NUMBER for x in m) else None
            elif pc == 4:
                keys = [x & 0x7FFFFFFF for x in w]
                p[g] = (min(keys), max(keys) + 1)
            elif pc == 5:
                cp = (NUMBER, p[g])
            else:
                b, nxt = p[g], None
            todo.append((pcs[:g] + (nxt,) + pcs[g + 1:], spcs, tuple(w), tuple(m), tuple(p), cp, cn, b, used, listed))
        for g, pc in enumerate(spcs):
            if pc is None:
                continue
            if pc == 0:
                looks = [None]                                     # gives up, without a bracket
                if copy[0] == NUMBER:
                    looks.append(copy[1])
                for got in looks:
                    todo.append((pcs, spcs[:g] + (1,) + spcs[g + 1:], words, marks_, picks, copy, counter, bracket,
                                 used[:g] + (got if got else "lost",) + used[g + 1:], listed))
            else:
                here = used[g] != "lost"
                todo.append((pcs, spcs[:g] + (None,) + spcs[g + 1:], words, marks_, picks, copy, counter + here, bracket,
                             used, listed + here))
    return ends


_OTHER = (0x30000000, 0x30000001)
_FRONTS = [(m, c, n, s) for m in ((0, 0), (NUMBER, 0), (0, NUMBER), (NUMBER, NUMBER))
           for c in ((0, None), (NUMBER, _OTHER)) for n in (0, 5, -1) for s in (None, _OTHER)]


@pytest.mark.parametrize("marks,copy,counter,state", _FRONTS)
def test_what_the_finish_accepts_is_one_bracket_and_all_keys(marks, copy, counter, state):
    ends = _front(marks, copy, counter, state)
    assert any(ok for ok, *_ in ends)
    for ok, used, bracket, listed, held in ends:
        if ok:
            assert used == (bracket, bracket) and listed == held == 2
    if not any(marks) and copy[0] != NUMBER:                       # cleared before: only a lost one is not accepted
        assert all(ok or "lost" in used for ok, used, *_ in ends)


def test_neither_the_clearing_nor_the_tags_can_be_left_out():
    """Stale counters alone: entries that the finish would read, and nobody wrote.  Another bracket alone: counts
    that add up, by two brackets."""
    assert all(not ok for ok, *_ in _front((0, 0), (0, None), 5, None, clears=False))
    assert any(ok and len(set(used)) == 2 for ok, used, *_ in _front((0, 0), (NUMBER, _OTHER), 0, None, tags=False))


def test_one_count_of_launches_in_the_library():
    lib = os.path.join(ROOT, "sga_amd", "libsga_hip.so")
    names = subprocess.run(["nm", "-C", lib], capture_output=True, text=True, check=True).stdout
    assert names.count("next_launch()::count") == 1


_PROGRAM = r"""
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include "sga_amd/csrc/sel_state.hpp"
using namespace sga;
int main() {
  int bad = 0;
  // any word is two keys of 31 bits
  for (unsigned long long w : {0ull, ~0ull, 0x80000000ull, 0xF000000580000000ull, 0x7FFFFFFF7FFFFFFFull, 0x0123456789ABCDEFull})
    for (int h = 0; h < 2; ++h) {
      const uint32_t k = sampled_key(w, h);
      bad += k >> 18 >= 8192u || k != ((uint32_t)(w >> (32 * h)) & 0x7FFFFFFFu);
    }
  // the words make up a state with the rank and the bracket alone
  unsigned long long words[kStateWords];
  for (int i = 0; i < kStateWords; ++i) words[i] = picked_word(i, 123456789u, 0x3F000001u, 0x80000000u);
  SelState got, want = {};
  std::memcpy(&got, words, sizeof(got));
  want.k = 123456789u; want.t_lo = 0x3F000001u; want.t_hi = 0x80000000u;
  bad += std::memcmp(&got, &want, sizeof(got)) != 0;
  // numbers of launches: never the cleared mark, none twice
  static unsigned char seen[1 << 29];
  for (uint32_t c = 0; c < 3000000u; ++c) {
    const uint32_t x = launch_number(c);
    bad += x == 0u || (seen[x >> 3] >> (x & 7) & 1);
    seen[x >> 3] |= (unsigned char)(1u << (x & 7));
  }
  // a chunk's words: numbers come back from the sums of eight chunks, a foreign bracket and a lost one do not pass
  const uint32_t nums[] = {0u, 1u, 511u, 1023u, 1024u};
  for (uint32_t lo : {0u, 1u, 0x3F000001u, 0x7F7FFFFFu, 0x7FFFFFFFu})
    for (uint32_t hi : {lo + 1u, lo + 0x1000u, 0x80000000u})
      for (uint32_t above : nums)
        for (uint32_t listed : nums)
          for (uint32_t equal : nums)
            for (int flags = 0; flags < 4; ++flags) {
              const uint32_t nf = (above * 7u + equal) % 1025u;
              const bool neg = flags & 1, lost = flags & 2;
              const SmallChunk c = SmallChunk::of(lo, hi, above, listed, equal, nf, neg, lost), z = SmallChunk::none(lo, hi);
              uint32_t sa = 0, sb = 0;
              for (int j = 0; j < 8; ++j) { sa += c.a & SmallChunk::kNumbers; sb += c.b & SmallChunk::kNumbers; }
              bad += (sa & 0xFFFFu) != 8u * above || sa >> 16 != 8u * listed || (sb & 0xFFFFu) != 8u * equal || sb >> 16 != 8u * nf;
              bad += (((c.b ^ z.b) & SmallChunk::kNegative) != 0u) != neg || SmallChunk::wrong(c.a ^ z.a, c.b ^ z.b) != lost;
            }
  // another bracket: 18 bits of a tag, so that a few in 2^18 pass
  uint32_t x = 1u;
  int missed = 0;
  for (int i = 0; i < 1 << 18; ++i) {
    x = x * 1664525u + 1013904223u;
    const uint32_t lo = x >> 1, lo2 = lo ^ (1u << (i % 31)), hi = lo + 1u + (x & 0xFFFFu);
    const SmallChunk c = SmallChunk::of(lo2, hi, 3u, 5u, 7u, 0u, false, false), z = SmallChunk::none(lo, hi);
    missed += !SmallChunk::wrong(c.a ^ z.a, c.b ^ z.b);
  }
  bad += missed > 16;
  std::printf("%d\n", bad);
  return bad != 0;
}
"""


def test_the_code_reads_and_writes_like_the_model(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(_PROGRAM)
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-I", ROOT, str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True).stdout == "0\n"
