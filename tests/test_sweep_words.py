"""The counters of the pressure-velocity iteration's team kernel
(pdac_words.hpp), compiled for the CPU: a block that starts while the team's
lead stores its last counters may read any mixture of old and new values, and
must not change a counter whatever it reads; behind the team the counters say
what the launches that go on expect."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pdac_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <map>
#include <utility>
#include <vector>
#include "pdac_words.hpp"

struct Lead {  // the team's lead: its stores in their order
  std::vector<std::pair<int, int32_t>> *log;
  int32_t load(int) const { return 0; }
  void store(int i, int32_t v) const { log->push_back({i, v}); }
};

struct Late {  // a late block 0: load k sees the value before or after the lead's stores, as bit k of 'seen' says
  const int32_t *before, *after;
  unsigned seen;
  int *loads, *stores;
  int32_t load(int i) const { return ((seen >> (*loads)++) & 1u) ? after[i] : before[i]; }
  void store(int, int32_t) const { ++*stores; }
};

int main() {
  int bad = 0;
  for (int maxout : {4, 9, 40})
    for (int s0 = 2; s0 <= 7 && s0 <= maxout; ++s0)
      for (int s = s0; s <= s0 + 4 && s <= maxout; ++s)
        for (int unc : {0, 17}) {
          // as k_visit leaves them before sweep s0: its predecessor unconverged,
          // the slot of s0 cleared, the third slot old
          int32_t before[C_N] = {}, after[C_N], T[TL_WORDS] = {};
          before[C_NIT] = s0;
          before[C_NIT1] = s0 - 1;
          before[C_WLP + 2 * ((s0 - 1) % 3)] = 5;
          before[C_WLP + 2 * ((s0 + 1) % 3) + 1] = 3;
          std::vector<std::pair<int, int32_t>> log;
          team_leave(Lead{&log}, s, unc, maxout);
          for (int i = 0; i < C_N; ++i) after[i] = before[i];
          for (auto &e : log) after[e.first] = e.second;
          // what the host and the next launches read
          const bool ended = unc == 0 || s >= maxout;
          if (after[C_DONE] != (unc == 0 ? 1 : ended ? 2 : 0)) ++bad;
          if (ended && after[C_NITF] != (unc == 0 ? s : maxout + 1)) ++bad;
          if (after[C_NIT] != s + 1 || after[C_WLP + 2 * (s % 3)] + after[C_WLP + 2 * (s % 3) + 1] != unc) ++bad;
          if (after[C_WLP + 2 * ((s + 1) % 3)] || after[C_WLP + 2 * ((s + 1) % 3) + 1]) ++bad;
          for (unsigned seen = 0; seen < 64; ++seen) {
            int loads = 0, tl = 0, stores = 0, st = 0, n = 0;
            (void)team_enter(Late{before, after, seen, &loads, &stores}, Late{T, T, 0, &tl, &stores}, maxout, 1000, st, n);
            if (loads > 6) { std::puts("more loads than orders tried"); return 2; }
            if (stores) {
              std::printf("late block wrote: team from sweep %d to %d, %d unconverged, maxout %d, order %u\n", s0, s, unc,
                          maxout, seen);
              ++bad;
            }
          }
        }
  std::printf("%d\n", bad);
  return bad ? 1 : 0;
}
"""


def test_late_block_of_a_team_writes_no_counter(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")
    src = tmp_path / "words.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "words"
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout
