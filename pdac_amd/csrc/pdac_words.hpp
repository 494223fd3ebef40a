// pdac_words.hpp -- the device counters of the pressure-velocity iteration
// and what its list kernels decide from them, apart from the kernels so that
// it can be compiled for the CPU too (tests/test_sweep_words.py).
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define PDAC_WORDS_FN __device__ __forceinline__
#else
#define PDAC_WORDS_FN inline
#endif

// device counters: sweep state of iter (done flag, sweep numbers of the two
// colour launches, the sweep that converged), EOS failures, three pairs of
// unconverged-cell counts per sweep (C_WLP), whether a team found no XCD
// (C_ALONE), and for the persistent iteration kernels an arrival counter for
// grid barriers and an error flag
enum Ctr { C_DONE = 0, C_NIT1 = 1, C_NIT = 2, C_ALONE = 3, C_EOS = 4, C_NITF = 5, C_WLP = 8, C_BAR = 14,
           C_ERR = 15, C_N = 16 };

// Words of the sweeps from lists (Fields::team, cleared by k_predict): the
// lengths of k_visit's lists, and those of one team launch, cleared again
// before the next: the lengths of its four lists, the blocks of each XCD that
// have started, the XCD chosen (+ 1; TL_NONE: none), the unconverged cells of
// three sweeps, and a barrier word per block.
constexpr int kTeamBlocks = 32;  // blocks of a team: one per compute unit of an XCD
enum TeamWord { TL_CNT = 0, TL_VIS = 8, TL_TEAM = 64, TL_REG = 64, TL_STATE = 80, TL_UNC = 84, TL_BAR = 96,
                TL_TEAM_END = 128, TL_WORDS = 128, TL_NONE = 99 };

// Whether a block of k_team goes on to the election of a team, and the sweep
// s0 and list length n that the team then starts with.  A block may start
// after a team has finished: the counters it reads are then being changed by
// the team's lead (team_leave), one by one and in no order.  So nothing is
// written here whatever they read: such a block returns, or goes on to an
// election that is over.  (That the last sweep had converged before this
// launch, k_lists has seen just before and set C_DONE.)
template <typename W>
PDAC_WORDS_FN bool team_enter(const W &ctr, const W &T, int maxout, int limit, int &s0, int &n) {
  if (ctr.load(C_DONE)) return false;
  s0 = ctr.load(C_NIT);
  n = T.load(TL_CNT);
  return s0 <= maxout && n <= limit && T.load(TL_CNT + 1) <= limit;
}

// The counters at a team's end, after sweep s with unc cells unconverged, by
// the team's lead alone: as k_visit leaves them, so that launches can go on.
template <typename W>
PDAC_WORDS_FN void team_leave(const W &ctr, int s, int unc, int maxout) {
  if (unc == 0 || s >= maxout) {
    ctr.store(C_NITF, unc == 0 ? s : maxout + 1);
    ctr.store(C_DONE, unc == 0 ? 1 : 2);
  }
  ctr.store(C_NIT, s + 1);
  const int prev = C_WLP + 2 * (s % 3), next = C_WLP + 2 * ((s + 1) % 3);
  ctr.store(prev, unc);
  ctr.store(prev + 1, 0);
  ctr.store(next, 0);
  ctr.store(next + 1, 0);
}
