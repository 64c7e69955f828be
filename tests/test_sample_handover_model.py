"""Host-side model of how the workgroups of ``k_sample_pick``
(csrc/select_impl.hpp) hand their sample keys over inside one launch, and the
pieces of it that the host can compile (csrc/sel_state.hpp).

A workgroup stores its keys, then the launch's number as its mark, then looks
at all marks; whoever sees every mark reads all keys, picks a bracket and
writes the state, which also clears the marks.  The memory is the caller's and
holds anything before: marks that happen to equal the number let a workgroup
pick from keys that are not there yet.  The model runs every order of the
steps of three workgroups over every such memory and checks what the select
needs: a key indexes the pick's histogram in range, and the bracket left
behind is one picking workgroup's own.  The protocol that this one replaced
(keys as they come, the two ends as two stores) gives neither."""
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
  std::printf("%d\n", bad);
  return bad != 0;
}
"""


def test_the_code_reads_and_writes_like_the_model(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(_PROGRAM)
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-I", ROOT, str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True).stdout == "0\n"
