// Three-launch turns (phx_engine.h) as the engine's launch sequences use them.
#pragma once

#include "phx_engine.h"

namespace phx_en {

struct AheadPass {
  void (*launch)(const EngineArgs &, hipStream_t);
  int nsub;
};

inline size_t ahead_lds_bytes(const phx_engine &e, int nsub) {
  return (ahead_hist_doubles(e.n_slices) + ahead_kick_doubles(e.n_slices, e.kick_shape) +
          (size_t)nsub * (e.record_stats ? ahead_red_doubles<true>() : ahead_red_doubles<false>())) *
         sizeof(double);
}

// Whether the low limbs of a slice's sums hold what one of the pass's blocks
// adds to it at most (2^(FX_LB - 1) a particle, below 2^63 together).  Blocks
// of up to 2^24 particles are every grid's for bunches up to that size, and
// those of 64 blocks and more for any bunch.
inline bool ahead_limbs_hold(int64_t n, int grid, int nsub, int hblk) {
  const int64_t rounds = (grid + (int64_t)hblk * nsub - 1) / ((int64_t)hblk * nsub);
  const int64_t groups = (phx_n_groups(n) + grid - 1) / grid;
  return rounds * nsub * groups * PHX_CHUNK <= (1LL << (63 - FX_LB + 1)) - 1;
}

// Whether the engine's turns can be three launches when e.ahead is set.
bool ahead_fits(const phx_engine &e);
// Groups of threads per block of its pass.
int ahead_max_nsub(const phx_engine &e);
// Ahead of the first of them; the pass, the merge.
int ahead_enqueue_start(const EngineArgs &a, hipStream_t s);
int ahead_enqueue_pass(const EngineArgs &a, hipStream_t s);
int ahead_enqueue_merge(const EngineArgs &a, hipStream_t s);

}  // namespace phx_en
