// Device side of the fused one-turn map (the engine): workspace layout,
// launch arguments and the bodies of the per-turn stages, shared by the
// single-engine kernels (phx_engine.hip) and the batch kernels, which run
// one stage of many engines in one launch (phx_batch.hip).
#pragma once

#include "phx_device.h"
#include "phx_sc.h"
#include "phx_slicing.h"
#include "phx_wake.h"

#define EN_STAT_NV 33
#define EN_NV (ZB_NV + EN_STAT_NV)
// the slice histogram: at most EN_HIST_BLOCKS blocks (partial histograms)
// of EN_HIST_THREADS threads, EN_HIST_PPT particles per thread and chunk
#ifndef EN_HIST_BLOCKS
#define EN_HIST_BLOCKS 256
#endif
#ifndef EN_HIST_THREADS
#define EN_HIST_THREADS 1024
#endif
#ifndef EN_HIST_PPT
#define EN_HIST_PPT PHX_PPT
#endif

namespace phx_en {


inline size_t round256(size_t b) { return (b + 255) / 256 * 256; }

// What a pass that slices its own turn (ahead_body) needs before it starts,
// formed by the merge of the turn before it: the turn's cuts, the bounds of
// x and y that scale its fixed-point sums (those of the state before it),
// the shift of its z sums (particle 0's z one turn on), the wake ring's
// slot and filling after the turn, and the turn.  The merge writes `next` and
// the convolution copies it to `cur`, which the merge of that turn reads while
// it writes `next` again: both addresses are known at launch, where a lookup
// by the turn counter is one more dependent load in kernels of 4 to 8 us.
// The program is looked up by the turn: a sequence's first turns may have
// others whose parameters differ in the last bit.  (The copy is not the pass's: a store ahead
// of its loop turns its scalar loads into vector loads.)
struct AheadState {
  double tail, head, width, mean_z, sigma_z, absx, absy, zshift;
  int nh, nf, turn, pad;
};

struct EngineWs {
  double *partials;   // [EN_NV][pass grid] (slot-major)
  double *p0;         // particle 0 before the pass: the shifts of its sums
  AheadState *next, *cur;  // in the rest of p0's 256 bytes
  AccParts acc;       // H partial histograms, T = 2 (x, y)
  double *conv_part;  // [n_kicks][conv_rows(S, T)][S]
};

__host__ __device__ inline int hist_blocks(int64_t n) {
  const int64_t nc = (n + PHX_CHUNK - 1) / PHX_CHUNK;
  return (int)(nc < EN_HIST_BLOCKS ? nc : EN_HIST_BLOCKS);
}

// The partials region holds the largest pass grid, so the layout does not
// depend on the grid chosen.
__host__ __device__ inline EngineWs engine_ws(void *ws, int64_t n, int S) {
  EngineWs w;
  char *p = reinterpret_cast<char *>(ws);
  const int64_t nc = phx_grid_for(n, PHX_MAX_GRID);
  const int Se = S > 0 ? S : 1;
  w.partials = reinterpret_cast<double *>(p);
  p += ((size_t)nc * EN_NV * 8 + 255) / 256 * 256;
  w.p0 = reinterpret_cast<double *>(p);
  w.next = reinterpret_cast<AheadState *>(p + 64);
  w.cur = w.next + 1;
  static_assert(64 + 2 * sizeof(AheadState) <= 256, "p0 region");
  p += 256;
  const int H = hist_blocks(n);
  w.acc = acc_parts_layout(p, H, Se, 2);
  p += acc_parts_bytes(H, Se, 2);
  w.conv_part = reinterpret_cast<double *>(p);
  return w;
}

// Whether the engine's convolution may have resistive-wall kicks in the
// dot-product form (conv_kinds 0: every kind).
__host__ __device__ inline bool engine_has_rw(const phx_engine &e) {
  return e.conv_kinds == 0 || (e.conv_kinds & (PHX_CONV_RW_DOT | PHX_CONV_RW_MFMA));
}

// The resistive-wall kick description (rw_desc_build), after the partial
// sums of the convolution.
__host__ __device__ inline RwKick *engine_rw_desc(const EngineWs &w, int n_kicks, int S, int T) {
  const int Se = S > 0 ? S : 1;
  return reinterpret_cast<RwKick *>(w.conv_part +
                                    (size_t)(n_kicks > 0 ? n_kicks : 1) * conv_rows(Se, T) * Se);
}

inline size_t engine_ws_bytes(int64_t n, int S, int n_kicks, int T) {
  const int64_t nc = phx_grid_for(n, PHX_MAX_GRID);
  const int Se = S > 0 ? S : 1;
  size_t b = round256((size_t)nc * EN_NV * 8) + 256 + acc_parts_bytes(hist_blocks(n), Se, 2);
  b += (size_t)(n_kicks > 0 ? n_kicks : 1) * conv_rows(Se, T) * Se * 8;
  b += rw_desc_bytes(T);
  return round256(b);
}

struct EngineArgs {
  phx_engine e;
  int n_kicks;
  int T;
  int grid;  // blocks of the particle pass (its partials: [slot][grid])
  int gmax;  // kicks one convolution block serves (LDS permitting)
  int nsub;  // three-launch turns: groups of PHX_BLOCK threads per pass block
             // (0: they do not apply)
  int hblk;  // and the pass's blocks, each storing one partial histogram
};

// ---------------------------------------------------------------------------
// Space-charge stages.  Their workspace (sc_ws): the Faddeeva coefficients,
// the cuts of the last space-charge slicing, the field parameters of every
// slice (one 64-byte row each) and the partial histograms of counts and
// sums of x, y, x^2, y^2 (laid out for the slicing's own slice count).
// ---------------------------------------------------------------------------
#define SC_TERMS 4

struct ScSlice {
  double mx, my, nl, pad;
  ScField f;
};

struct ScWs {
  WofzCoeffs *wc;
  phx_slice_state *state;
  ScSlice *slices;
  char *acc;  // acc_parts_layout(acc, hist_blocks(n), S, SC_TERMS)
};

__host__ __device__ inline size_t sc_r256(size_t b) { return (b + 255) / 256 * 256; }

__host__ __device__ inline ScWs sc_ws(void *base, int S) {
  ScWs w;
  char *p = reinterpret_cast<char *>(base);
  w.wc = reinterpret_cast<WofzCoeffs *>(p);
  p += sc_r256(sizeof(WofzCoeffs));
  w.state = reinterpret_cast<phx_slice_state *>(p);
  p += sc_r256(sizeof(phx_slice_state));
  w.slices = reinterpret_cast<ScSlice *>(p);
  p += sc_r256((size_t)(S > 0 ? S : 1) * sizeof(ScSlice));
  w.acc = p;
  return w;
}

inline size_t sc_ws_bytes(int64_t n, int S) {
  const int Se = S > 0 ? S : 1;
  return sc_r256(sizeof(WofzCoeffs)) + sc_r256(sizeof(phx_slice_state)) +
         sc_r256((size_t)Se * sizeof(ScSlice)) + sc_r256(acc_parts_bytes(hist_blocks(n), Se, SC_TERMS));
}

// What a space-charge kick of a pass reads: the cuts of the slicing after
// the previous stage, its slices' field parameters, the coefficients.
struct ScCtx {
  const ScSlice *sl;
  const WofzCoeffs *wc;
  SliceBins bins;
};

template <int N>
__device__ __forceinline__ void sc_kick_n(P6 (&p)[N], const ScCtx &c, const phx_spacecharge &sp) {
  double dx[N], dy[N], nl[N], ex[N], ey[N];
  ScField f[N];
  bool in[N];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const int s = c.bins.index(p[k].z);
    in[k] = s >= 0;
    const ScSlice &q = c.sl[in[k] ? s : 0];
    dx[k] = p[k].x - q.mx;
    dy[k] = p[k].y - q.my;
    nl[k] = q.nl;
    f[k] = q.f;
  }
  sc_field_n<N>(*c.wc, sp, dx, dy, f, ex, ey);
#pragma unroll
  for (int k = 0; k < N; ++k) {
    if (in[k]) {
      p[k].xp = p[k].xp + (ex[k] * nl[k]) * sp.prefactor;
      p[k].yp = p[k].yp + (ey[k] * nl[k]) * sp.prefactor;
    }
  }
}

__device__ __forceinline__ P6 load_p(const phx_engine &e, int64_t j) {
  P6 p;
  p.x = e.coords[0][j];
  p.xp = e.coords[1][j];
  p.y = e.coords[2][j];
  p.yp = e.coords[3][j];
  p.z = e.coords[4][j];
  p.dp = e.coords[5][j];
  return p;
}

__device__ __forceinline__ void store_p(const phx_engine &e, int64_t j, const P6 &p) {
  e.coords[0][j] = p.x;
  e.coords[1][j] = p.xp;
  e.coords[2][j] = p.y;
  e.coords[3][j] = p.yp;
  e.coords[4][j] = p.z;
  e.coords[5][j] = p.dp;
}

// nk = min(program kicks, engine kicks): the kick table holds the latter.
template <int KS>
__device__ __forceinline__ void kick_pending(P6 &p, const phx_turn_program &g, int nk,
                                             const SliceBins &bins, int S, const double *kicks) {
  const int s = bins.index(p.z);
  if (s >= 0) apply_kick_set<KS>(p, s, S, g.kick, nk, kicks);
}

// The pending kick's table values for the PHX_PPT particles of a group,
// read one group ahead of their use (the loads are otherwise a dependent
// gather in the middle of each group's arithmetic).  For the kick sets
// with straight-line code: DXDY (dipole x, y: 2 values per particle) and
// PLATES (dipole and quadrupole x, y: 4).  The kicks do not move z, so the
// slice index from the group's loaded z is the one kick_pending takes, and
// apply() adds in apply_kick_set's order: the same arithmetic.
template <int KS>
struct KickAhead {
  static constexpr int NV = KS == PHX_KICKS_DXDY ? 2 : (KS == PHX_KICKS_PLATES ? 4 : 0);
  static constexpr bool ON = NV > 0;
  double k[PHX_PPT][NV > 0 ? NV : 1];
  bool in[PHX_PPT];
  __device__ __forceinline__ void fetch(const P6 (&q)[PHX_PPT], const SliceBins &bins, int S,
                                        const double *kicks) {
#pragma unroll
    for (int j = 0; j < PHX_PPT; ++j) {
      const int b = bins.index(q[j].z);
      in[j] = b >= 0;
      const int s = in[j] ? b : 0;  // slot 0 is read and not used outside
#pragma unroll
      for (int i = 0; i < NV; ++i) k[j][i] = kicks[(size_t)i * S + s];
    }
  }
  __device__ __forceinline__ void apply(P6 (&q)[PHX_PPT]) const {
#pragma unroll
    for (int j = 0; j < PHX_PPT; ++j) {
      if (!in[j]) continue;
      if constexpr (KS == PHX_KICKS_DXDY) {
        q[j].xp = q[j].xp + k[j][0];
        q[j].yp = q[j].yp + k[j][1];
      } else if constexpr (KS == PHX_KICKS_PLATES) {
        q[j].xp = q[j].xp + k[j][0];
        q[j].xp = q[j].xp + k[j][1] * q[j].x;
        q[j].yp = q[j].yp + k[j][2];
        q[j].yp = q[j].yp + k[j][3] * q[j].y;
      }
    }
  }
};

// The six coordinate arrays of a pass.
struct GroupPtr {
  double *c[6];
};

// PHX_PASS_NT: the momenta xp, yp, dp (which the slice histogram after the
// pass does not read) are loaded and stored non-temporally, so that they do
// not push x, y and z out of the last-level cache before the histogram;
// with PHX_PASS_NT_ALL every coordinate's (old) value is loaded so.
#ifndef PHX_PASS_NT
#define PHX_PASS_NT 1
#endif
#ifndef PHX_PASS_NT_ALL
#define PHX_PASS_NT_ALL 0
#endif
__device__ __forceinline__ double ld_mom(const double *p) {
#if PHX_PASS_NT
  return __builtin_nontemporal_load(p);
#else
  return *p;
#endif
}
__device__ __forceinline__ double ld_pos(const double *p) {
#if PHX_PASS_NT_ALL
  return __builtin_nontemporal_load(p);
#else
  return *p;
#endif
}
__device__ __forceinline__ void st_mom(double *p, double v) {
#if PHX_PASS_NT
  __builtin_nontemporal_store(v, p);
#else
  *p = v;
#endif
}

// Coordinates addressed as the array's base (the kernel arguments, kept in
// scalar registers) plus one 32-bit byte offset per particle, shared by the
// six arrays: per-group pointers to six arrays, current and next group,
// would take 24 scalar registers across the particle loop (bunches up to
// PHX_ENGINE_MAX_N keep every offset below 2^32).
__device__ __forceinline__ const double *at_off(const double *b, uint32_t off) {
  return reinterpret_cast<const double *>(reinterpret_cast<const char *>(b) + off);
}
__device__ __forceinline__ double *at_off(double *b, uint32_t off) {
  return reinterpret_cast<double *>(reinterpret_cast<char *>(b) + off);
}

// The PHX_PPT particles of thread tid in the group starting at byte offset
// goff; lim: the group's particle count if it is the partial last group,
// else PHX_CHUNK (no guard needed).
__device__ __forceinline__ void group_load(const GroupPtr &gb, uint32_t goff, int lim, int tid,
                                           P6 (&p)[PHX_PPT]) {
#pragma unroll
  for (int k = 0; k < PHX_PPT; ++k) {
    const int o = tid + k * PHX_BLOCK;
    const uint32_t off = goff + (uint32_t)o * 8u;
    if (lim == PHX_CHUNK || o < lim)
      p[k] = P6{ld_pos(at_off(gb.c[0], off)), ld_mom(at_off(gb.c[1], off)),
                ld_pos(at_off(gb.c[2], off)), ld_mom(at_off(gb.c[3], off)),
                ld_pos(at_off(gb.c[4], off)), ld_mom(at_off(gb.c[5], off))};
    else
      p[k] = P6{0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  }
}

// Byte offset and particle count of group gg (uniform).
__device__ __forceinline__ int group_at(int64_t gg, int64_t n, uint32_t &off) {
  const int64_t b = gg * PHX_CHUNK;
  off = (uint32_t)b * 8u;
  const int64_t rest = n - b;
  return rest >= PHX_CHUNK ? PHX_CHUNK : (int)rest;
}

__device__ __forceinline__ void group_store(const GroupPtr &gb, uint32_t goff, int lim, int tid,
                                            const P6 (&p)[PHX_PPT]) {
#pragma unroll
  for (int k = 0; k < PHX_PPT; ++k) {
    const int o = tid + k * PHX_BLOCK;
    const uint32_t off = goff + (uint32_t)o * 8u;
    if (lim == PHX_CHUNK || o < lim) {
      *at_off(gb.c[0], off) = p[k].x; st_mom(at_off(gb.c[1], off), p[k].xp);
      *at_off(gb.c[2], off) = p[k].y; st_mom(at_off(gb.c[3], off), p[k].yp);
      *at_off(gb.c[4], off) = p[k].z; st_mom(at_off(gb.c[5], off), p[k].dp);
    }
  }
}

// stats slots: [0..6) sum u, [6..12) sum (u-u0), [12..33) sum (u-u0)(v-v0)
__device__ __forceinline__ void stats_accumulate(double *v, const P6 &p, const double *sh) {
  const double u[6] = {p.x, p.xp, p.y, p.yp, p.z, p.dp};
  double d[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    d[i] = u[i] - sh[i];
    v[i] = v[i] + u[i];
    v[6 + i] = v[6 + i] + d[i];
  }
  int q = 12;
#pragma unroll
  for (int i = 0; i < 6; ++i)
#pragma unroll
    for (int j = i; j < 6; ++j) {
      v[q] = v[q] + d[i] * d[j];
      ++q;
    }
}

template <bool REC, bool WAKE>
struct PassLayout {
  static constexpr int NV = (WAKE ? ZB_NV : 0) + (REC ? EN_STAT_NV : 0) + ((!WAKE && !REC) ? 1 : 0);
  static constexpr unsigned long long MINM = WAKE ? ZB_MINM : 0ULL;
  static constexpr unsigned long long MAXM = WAKE ? ZB_MAXM : 0ULL;
  static constexpr int SOFF = WAKE ? ZB_NV : 0;
};

// MODE 0: a turn; MODE 1: flush (pending kick + final statistics only).
// Persistent grid (a.grid blocks): each block walks its particle
// groups with the next group's coordinates loaded while the current one is
// computed, so the particle traffic overlaps the FP64 work.
// No workgroup barrier or fence precedes the last read of the turn program
// and the coordinate arrays are declared non-aliasing (__restrict__
// arguments): otherwise the compiler must assume the program may have been
// written and reloads it with vector loads that wait on the particle loads.
// So particle 0 is computed by every lane, and the kick table is read from
// global memory (it stays in the caches).  Dynamic LDS: the block reduction.
#ifndef PHX_PASS_MIN_BLOCKS
#define PHX_PASS_MIN_BLOCKS 1
#endif
#ifndef PHX_PASS_LAUNDER
#define PHX_PASS_LAUNDER 0
#endif
// Space-charge engines (sc_stages > 0) run this pass for stage 0 of a
// turn (stage: the offset of the stage's program from the turn's first;
// the later stages run sc_pass_body).  The pending wake kick and the
// statistics belong to stage 0.
// AHEAD: one of ahead_body's groups of threads (tid: the thread's index in
// it, lds its reduction area): the turn's cuts are known, the moved particles
// are added to the block's slice histogram `acc`, and the z sums are those of
// the next turn (aheadz: the cuts and scales of ahead_body; bid >= nblk: a
// group without particles).
enum { AHEAD_NONE = 0, AHEAD_TABLE, AHEAD_OWN };  // AHEAD_OWN: programs is the turn's program
struct AheadCtx {
  AccLds acc;
  const double *kicks;  // the pending kick table in LDS
  SliceBins bins;
  FxScale fx, fy;
};

// The dipole or plates kick of one particle of slice s (>= 0) from the table
// in LDS, with apply_kick_set's operations.
template <int KS>
__device__ __forceinline__ void kick_from_lds(P6 &p, int s, int S, const double *kicks) {
  p.xp = p.xp + kicks[s];
  if constexpr (KS == PHX_KICKS_DXDY) {
    p.yp = p.yp + kicks[S + s];
  } else {
    p.xp = p.xp + kicks[S + s] * p.x;
    p.yp = p.yp + kicks[2 * S + s];
    p.yp = p.yp + kicks[3 * S + s] * p.y;
  }
}

template <int MODE, bool REC, bool WAKE, int SHAPE, int KS, int DS, int AHEAD>
__device__ __forceinline__ void pass_body(
    const EngineArgs &a, double *__restrict__ x, double *__restrict__ xp,
    double *__restrict__ y, double *__restrict__ yp, double *__restrict__ z,
    double *__restrict__ dp, const phx_turn_program *__restrict__ programs,
    const double *__restrict__ kicks, int bid, int nblk, int stage, int tid, double *lds,
    const AheadCtx *ctx) {
  using L = PassLayout<REC, WAKE>;
  static_assert(!AHEAD || (MODE == 0 && WAKE && KS != PHX_KICKS_GENERIC), "ahead pass");
  const phx_engine &e = a.e;
  EngineWs w = engine_ws(e.ws, e.n, e.n_slices);
  const int64_t n = e.n;
  int prog;
  if constexpr (AHEAD) {
    prog = AHEAD == AHEAD_OWN ? 0 : e.turn_program[w.next->turn];
  } else {
    const int turn = *e.turn_counter;
    prog = e.turn_program[MODE == 0 ? turn : (turn > 0 ? turn - 1 : 0)] + stage;
  }
  const phx_turn_program &g = programs[prog];
  const int pend = stage == 0 ? *e.pending : 0;
  const int S = e.n_slices;
  const SliceBins bins(e.state->tail, e.state->width, S);
  // the cuts after this pass: a space-charge slicing's, or the wake's
  const bool minmax = (g.has_sc ? g.sc_slicer : g.slicer).cuts_mode == PHX_CUTS_MINMAX;
  const int nk = g.n_kicks < a.n_kicks ? g.n_kicks : a.n_kicks;
  const int64_t ng = AHEAD && bid >= nblk ? 0 : phx_n_groups(n);
  // the group's base pointers and particle count (uniform)
  const GroupPtr gb{{x, xp, y, yp, z, dp}};
  int64_t gi = bid;
  uint32_t gc = 0, gnx = 0;
  int lc = 0;
  if (!AHEAD || gi < ng) lc = group_at(gi, n, gc);
  P6 cur[PHX_PPT], nxt[PHX_PPT];
  group_load(gb, gc, lc, tid, cur);
  // Particle 0 sets the shifts of the shifted sums (stats.pyx:cov): its
  // state after the pending kick (statistics), and its z after this turn's
  // elements (cuts), which needs the kick only where a kick changes dp and
  // only the longitudinal elements.  Every lane computes it (uniform values;
  // once per block) from the snapshot taken before this pass: block 0
  // rewrites particle 0 while later blocks may still be starting.  (AHEAD:
  // the merge of the turn before left the z shift in the workspace.)
  double src[7];
  if constexpr (!AHEAD || REC) {
    const double *p0 = w.p0;
    P6 q = P6{p0[0], p0[1], p0[2], p0[3], p0[4], p0[5]};
    bool kick_dp = false;
    if constexpr (KS == PHX_KICKS_GENERIC) {
      for (int k = 0; k < nk; ++k) kick_dp = kick_dp || g.kick[k].plane == PHX_PLANE_DP;
    }
    if constexpr (AHEAD) {
      const int b = bins.index(q.z);
      if (pend && b >= 0) kick_from_lds<KS>(q, b, S, ctx->kicks);
    } else {
      if (pend && (REC || kick_dp)) kick_pending<KS>(q, g, nk, bins, S, kicks);
    }
    src[0] = q.x; src[1] = q.xp; src[2] = q.y; src[3] = q.yp; src[4] = q.z; src[5] = q.dp;
    if (MODE == 0 && !AHEAD) apply_shape_longitudinal<SHAPE>(q, g);
    src[6] = q.z;
  }
  if constexpr (AHEAD) src[6] = w.next->zshift;
  double v[L::NV];
#pragma unroll
  for (int i = 0; i < L::NV; ++i) v[i] = red_ident<L::MINM, L::MAXM>(i);
  double shs[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) shs[i] = AHEAD && !REC ? 0.0 : src[i];
  const double zshift = src[6];
  // four-launch pass: the kick's table values are read one group ahead
  constexpr bool KA = KickAhead<KS>::ON && !AHEAD;
  KickAhead<KS> ka;
  if (KA && pend) ka.fetch(cur, bins, S, kicks);
  for (; gi < ng; gi += nblk) {
    const int64_t gn = gi + nblk;
    int ln = 0;
    if (gn < ng) {
      ln = group_at(gn, n, gnx);
      group_load(gb, gnx, ln, tid, nxt);
    }
    if (pend) {
      if constexpr (AHEAD) {
#pragma unroll
        for (int k = 0; k < PHX_PPT; ++k) {
          const int b = bins.index(cur[k].z);
          if (b >= 0) kick_from_lds<KS>(cur[k], b, S, ctx->kicks);
        }
      } else if constexpr (KA) {
        ka.apply(cur);
      } else {
#pragma unroll
        for (int k = 0; k < PHX_PPT; ++k)
          kick_pending<KS>(cur[k], g, nk, bins, S, kicks);
      }
    }
    const bool full = lc == PHX_CHUNK;
    if (REC) {
#pragma unroll
      for (int k = 0; k < PHX_PPT; ++k)
        if (full || tid + k * PHX_BLOCK < lc)
          stats_accumulate(&v[L::SOFF], cur[k], shs);
    }
    if (MODE == 0) {
      // PHX_PASS_LAUNDER: read the element parameters from the program in
      // every group (a pointer the compiler cannot follow across
      // iterations) instead of holding them in scalar registers over the
      // loop; measured slower (more vector registers, 2 waves per SIMD)
      const phx_turn_program *gl = &g;
#if PHX_PASS_LAUNDER
      asm volatile("" : "+s"(gl));
#endif
      apply_shape_n<SHAPE, PHX_PPT, DS>(cur, *gl);
    }
    if (MODE == 0 || pend) group_store(gb, gc, lc, tid, cur);
    if constexpr (AHEAD) {
#pragma unroll
      for (int k = 0; k < PHX_PPT; ++k) {
        if (full || tid + k * PHX_BLOCK < lc) {
          const int s = ctx->bins.index(cur[k].z);
          if (s >= 0) {
            atomicAdd(&ctx->acc.counts[s], 1u);
            acc_add_value(ctx->acc, S, 0, s, cur[k].x, ctx->fx, w.acc.fallback);
            acc_add_value(ctx->acc, S, 1, s, cur[k].y, ctx->fy, w.acc.fallback);
          }
        }
      }
      apply_shape_longitudinal_n<SHAPE, PHX_PPT>(cur, g);  // z one turn on
    }
    if (WAKE) {
#pragma unroll
      for (int k = 0; k < PHX_PPT; ++k) {
        if (full || tid + k * PHX_BLOCK < lc) {
          double zb[ZB_NV];
#pragma unroll
          for (int i = 0; i < ZB_NV; ++i) zb[i] = v[i];
          // max |x|, |y| only scale the slices' fixed-point sums, which take
          // larger values too (acc_add_value): every PHX_PPT-th particle's do
          if (k == 0) zblock_accumulate<0x05u>(zb, cur[k], zshift, minmax);
          else zblock_accumulate<0u>(zb, cur[k], zshift, minmax);
#pragma unroll
          for (int i = 0; i < ZB_NV; ++i) v[i] = zb[i];
        }
      }
    }
#pragma unroll
    for (int k = 0; k < PHX_PPT; ++k) cur[k] = nxt[k];
    gc = gnx;
    lc = ln;
    // the next group's kick values, while this block's other waves compute
    if (KA && pend && gn < ng) ka.fetch(cur, bins, S, kicks);
  }
  if constexpr (AHEAD) {
    // the z sums and the maxima of |x| and |y| (the other slots are not kept)
    double c[ZA_NV];
#pragma unroll
    for (int i = 0; i < ZA_NV; ++i) c[i] = v[za_slot(i)];
    const double r = block_reduce_slots_at<ZA_NV, ZA_MINM, ZA_MAXM>(c, lds, tid);
    if (bid < nblk && tid < ZA_NV) w.partials[(size_t)za_slot(tid) * nblk + bid] = r;
    if constexpr (REC) {
      double t[EN_STAT_NV];
#pragma unroll
      for (int i = 0; i < EN_STAT_NV; ++i) t[i] = v[L::SOFF + i];
      const double q = block_reduce_slots_at<EN_STAT_NV, 0ULL, 0ULL>(t, lds, tid);
      if (bid < nblk && tid < EN_STAT_NV) w.partials[(size_t)(L::SOFF + tid) * nblk + bid] = q;
    }
  } else {
    const double r = block_reduce_slots<L::NV, L::MINM, L::MAXM>(v, lds);
    if (threadIdx.x < L::NV) w.partials[(size_t)threadIdx.x * nblk + bid] = r;
  }
}

template <int MODE, bool REC, bool WAKE, int SHAPE, int KS, int DS>
__device__ __forceinline__ void pass_body(
    const EngineArgs &a, double *__restrict__ x, double *__restrict__ xp,
    double *__restrict__ y, double *__restrict__ yp, double *__restrict__ z,
    double *__restrict__ dp, const phx_turn_program *__restrict__ programs,
    const double *__restrict__ kicks, int bid, int nblk, int stage = 0) {
  extern __shared__ double pass_lds[];
  pass_body<MODE, REC, WAKE, SHAPE, KS, DS, AHEAD_NONE>(a, x, xp, y, yp, z, dp, programs, kicks, bid,
                                                   nblk, stage, threadIdx.x, pass_lds, nullptr);
}

// ---------------------------------------------------------------------------
// Three-launch turns (EngineArgs.nsub > 0): pass with slicing, merge,
// convolution.  The cuts of a turn depend on z after its elements, which the
// longitudinal motion alone fixes (no kick on dp), so the pass of turn t can
// also sum z of turn t + 1 (the same program every turn) from the particles
// it holds: the merge folds those sums into the cuts of turn t + 1, and the
// pass of turn t + 1 slices each particle as it moves it.  The slice
// histogram's own launch and its 24 B per macroparticle go (11.2 of 45.4 us
// at 1e6 macroparticles, 42.6 of 231 us at 1e7), for a second evaluation of
// the longitudinal motion (nothing for a linear map, a sine for an RF kick).
// One pass block is nsub groups of PHX_BLOCK threads, each a block of the
// four-launch pass (the same particles in the same order, hence the same z
// sums and cuts bit for bit), sharing one histogram: a CU then stores one
// partial histogram, as many as the histogram kernel stored.  The slices' sums
// are the four-launch turn's too unless the bounds of |x| and |y|, which are
// those of the state before the turn, give them another scale (fx_scale).
// ---------------------------------------------------------------------------
__host__ __device__ inline size_t ahead_hist_doubles(int S) {
  return (acc_lds_bytes(S, 2) + 7) / 8;
}
// and the pending kick's table, which every particle reads at its slice: from
// global memory, 2 or 4 gathers per particle of a table that the streamed
// coordinates push out of the L1 (26.6 us against 20 us for a linear-map pass
// with a 1000-slice plates kick)
__host__ __device__ inline size_t ahead_kick_doubles(int S, int kick_shape) {
  return (size_t)(kick_shape == PHX_KICKS_PLATES ? 4 : 2) * S;
}
// LDS doubles of one group's reduction
template <bool REC>
__host__ __device__ constexpr int ahead_red_doubles() {
  return REC ? BR_LDS(EN_STAT_NV) : BR_LDS(ZA_NV);
}
// Groups of threads per block: three of the specialised passes' groups fill a
// CU (at most 168 vector registers), two of the others'.  Two-harmonic RF with
// amplitude detuning takes two: in 168 registers it spills 4 to 22 of them (40
// turns of 3e5, of 1e6 and 10 turns of 5e6 macroparticles, three and two
// groups: 1152 and 967, 1864 and 1572, 1485 and 1207 us); with chromaticity
// alone it spills 4 to 13 and keeps three (1015 and 945, 1532 and 1531, 1143
// and 1167 us).  The generic order with statistics spills at two as well; one
// group is the better up to 3e5 macroparticles (40 turns 2002 against 2204 us),
// two above (1e6: 3677 against 3589, 10 turns of 5e6: 3517 against 3079).
template <bool REC, int SHAPE, int DS>
constexpr int ahead_nsub() {
  constexpr bool RF2 = SHAPE == PHX_SHAPE_RF2_T || SHAPE == PHX_SHAPE_T_RF2;
  constexpr bool AMP = (DS & ~PHX_DETS_SMOOTH) == PHX_DETS_C1_AMP;
  return REC || SHAPE == PHX_SHAPE_GENERIC || (RF2 && AMP) ? 2 : 3;
}

// The partial histograms of a three-launch turn: hblk of them, the fallback
// sums where the four-launch turn has them.
__device__ __forceinline__ AccParts ahead_parts(const EngineWs &w, int S, int hblk) {
  AccParts P = acc_parts_layout(w.acc.cnt, hblk, S, 2);
  P.fallback = w.acc.fallback;
  return P;
}

// Pass block kb of nkb.
template <bool REC, int SHAPE, int KS, int DS, int AHEAD = AHEAD_TABLE>
__device__ __forceinline__ void ahead_body(
    const EngineArgs &a, double *__restrict__ x, double *__restrict__ xp,
    double *__restrict__ y, double *__restrict__ yp, double *__restrict__ z,
    double *__restrict__ dp, const phx_turn_program *__restrict__ programs,
    const double *__restrict__ kicks, int kb, int nkb, int nsub) {
  extern __shared__ double pass_lds[];
  const phx_engine &e = a.e;
  const int S = e.n_slices;
  const int sub = __builtin_amdgcn_readfirstlane(threadIdx.x / PHX_BLOCK);
  const int tid = threadIdx.x % PHX_BLOCK;
  double *kt = pass_lds + ahead_hist_doubles(S);
  double *red = kt + ahead_kick_doubles(S, KS) + sub * ahead_red_doubles<REC>();
  EngineWs w = engine_ws(e.ws, e.n, S);
  AheadCtx c;
  c.kicks = kt;
  c.acc = acc_lds_layout(reinterpret_cast<unsigned long long *>(pass_lds), S, 2);
  const AheadState &h = *w.next;
  for (int i = threadIdx.x; i < (int)ahead_kick_doubles(S, KS); i += blockDim.x) kt[i] = kicks[i];
  acc_lds_zero(c.acc, S, 2);  // ends with a barrier; the particle loads follow it
  c.bins = SliceBins(h.tail, h.width, S);
  c.fx = fx_scale(h.absx, e.n);
  c.fy = fx_scale(h.absy, e.n);
  for (int b0 = 0; b0 < a.grid; b0 += nkb * nsub)
    pass_body<0, REC, true, SHAPE, KS, DS, AHEAD>(a, x, xp, y, yp, z, dp, programs, kicks,
                                                 b0 + sub * nkb + kb, a.grid, 0, tid, red, &c);
  acc_lds_store(c.acc, S, 2, ahead_parts(w, S, a.hblk), kb);
}

// The cuts of a three-launch turn from folded z sums, the bounds of |x| and
// |y| and the ring's state after that turn, into its AheadState (one thread).
__device__ __forceinline__ void ahead_set(AheadState &h, const phx_slicer &cfg, int64_t n,
                                          const double *res, int nh, int nf, int turn) {
  phx_slice_state st;
  compute_cuts(cfg, n, res[0], res[1], res[2], res[3], res[4], st);
  h.tail = st.tail;
  h.head = st.head;
  h.width = st.width;
  h.mean_z = st.mean_z;
  h.sigma_z = st.sigma_z;
  h.absx = res[5];
  h.absy = res[7];
  h.nh = nh;
  h.nf = nf;
  h.turn = turn;
  h.pad = 0;
}

// Particle 0's z after two turns' longitudinal motion from c: the shift of
// the z sums that the next pass forms.
__device__ __forceinline__ double ahead_shift(double *const *c, const phx_turn_program &g) {
  P6 q = P6{0.0, 0.0, 0.0, 0.0, c[4][0], c[5][0]};
  apply_shape_longitudinal<PHX_SHAPE_GENERIC>(q, g);
  apply_shape_longitudinal<PHX_SHAPE_GENERIC>(q, g);
  return q.z;
}

__device__ __forceinline__ void ahead_fold(const double *partials, int grid, double *res) {
  fold_partials<ZB_MINM, ZB_MAXM, ZA_NV>(partials, grid, 0, ZA_NV, res);
}

// Before the first three-launch turn of a sequence: block bid of grid sums
// the z that the next turn's longitudinal motion gives the current state, in
// the pass's order, and the maxima of |x| and |y|; ahead_start_fold (one
// block) then sets the turn's AheadState.
__device__ __forceinline__ void ahead_start_body(const EngineArgs &a, int bid) {
  const phx_engine &e = a.e;
  extern __shared__ double pass_lds[];
  EngineWs w = engine_ws(e.ws, e.n, e.n_slices);
  const int turn = *e.turn_counter;
  const phx_turn_program &g = e.programs[e.turn_program[turn]];
  double *const *c = e.coords;
  const bool minmax = g.slicer.cuts_mode == PHX_CUTS_MINMAX;
  double zshift;
  {
    P6 q = P6{0.0, 0.0, 0.0, 0.0, c[4][0], c[5][0]};
    apply_shape_longitudinal<PHX_SHAPE_GENERIC>(q, g);
    zshift = q.z;
  }
  double v[ZB_NV];
#pragma unroll
  for (int i = 0; i < ZB_NV; ++i) v[i] = red_ident<ZB_MINM, ZB_MAXM>(i);
  const int64_t ng = phx_n_groups(e.n);
  for (int64_t gi = bid; gi < ng; gi += a.grid) {
    P6 p[PHX_PPT];
#pragma unroll
    for (int k = 0; k < PHX_PPT; ++k) {
      const int64_t j = gi * PHX_CHUNK + threadIdx.x + k * PHX_BLOCK;
      p[k] = P6{0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
      if (j < e.n) {
        p[k].x = c[0][j];
        p[k].y = c[2][j];
        p[k].z = c[4][j];
        p[k].dp = c[5][j];
      }
    }
    apply_shape_longitudinal_n<PHX_SHAPE_GENERIC, PHX_PPT>(p, g);
#pragma unroll
    for (int k = 0; k < PHX_PPT; ++k)
      if (gi * PHX_CHUNK + threadIdx.x + k * PHX_BLOCK < e.n) {
        if (k == 0) zblock_accumulate<0x05u>(v, p[k], zshift, minmax);
        else zblock_accumulate<0u>(v, p[k], zshift, minmax);
      }
  }
  double r[ZA_NV];
#pragma unroll
  for (int i = 0; i < ZA_NV; ++i) r[i] = v[za_slot(i)];
  const double t = block_reduce_slots<ZA_NV, ZA_MINM, ZA_MAXM>(r, pass_lds);
  if (threadIdx.x < ZA_NV) w.partials[(size_t)za_slot(threadIdx.x) * a.grid + bid] = t;
}

__device__ __forceinline__ void ahead_start_fold(const EngineArgs &a) {
  const phx_engine &e = a.e;
  __shared__ double res[ZB_NV];
  EngineWs w = engine_ws(e.ws, e.n, e.n_slices);
  const int turn = *e.turn_counter;
  const phx_turn_program &g = e.programs[e.turn_program[turn]];
  AheadState &h = *w.next;
  if (threadIdx.x < 6) w.p0[threadIdx.x] = e.coords[threadIdx.x][0];
  ahead_fold(w.partials, a.grid, res);
  if (threadIdx.x == 0) {
    const int cap = e.hist->capacity, nf = e.hist->n_filled;
    const int nh = (e.hist->head + 1) % cap, nf1 = nf + 1 < cap ? nf + 1 : cap;
    ahead_set(h, g.slicer, e.n, res, nh, nf1, turn);
    ahead_set(*w.cur, g.slicer, e.n, res, nh, nf1, turn);
  } else if (threadIdx.x == PHX_WAVE) {
    h.zshift = ahead_shift(e.coords, g);
  }
}

// The pass of space-charge stage `stage` > 0: the space-charge kick that
// ended the previous stage (the slicing after it is in the space-charge
// workspace), then the stage's elements, the coordinates written back and
// the z block of the result (11 partials per block, as pass_body without
// statistics).  The field evaluation needs many registers, so a thread
// holds one particle at a time, taking the particles of pass_body's groups
// in pass_body's order: the z-block sums, and so the cuts, are those
// pass_body would give.
template <int SHAPE, int DS>
__device__ __forceinline__ void sc_pass_body(
    const EngineArgs &a, double *__restrict__ x, double *__restrict__ xp,
    double *__restrict__ y, double *__restrict__ yp, double *__restrict__ z,
    double *__restrict__ dp, const phx_turn_program *__restrict__ programs, int bid, int nblk,
    int stage) {
  const phx_engine &e = a.e;
  extern __shared__ double pass_lds[];
  EngineWs w = engine_ws(e.ws, e.n, e.n_slices);
  const int64_t n = e.n;
  const int turn = *e.turn_counter;
  const int first = e.turn_program[turn];
  const phx_turn_program &g = programs[first + stage];
  const phx_spacecharge &sp = programs[first + stage - 1].sc;
  const ScWs sw = sc_ws(e.sc_ws, e.sc_slices);
  ScCtx scc;
  scc.sl = sw.slices;
  scc.wc = sw.wc;
  scc.bins = SliceBins(sw.state->tail, sw.state->width, sw.state->n_slices);
  // the cuts after this stage: its space-charge slicing's, or the wake's
  const bool minmax = (g.has_sc ? g.sc_slicer : g.slicer).cuts_mode == PHX_CUTS_MINMAX;
  // particle 0's z after this stage's elements: the shift of the z sums
  double zshift;
  {
    P6 q = P6{w.p0[0], w.p0[1], w.p0[2], w.p0[3], w.p0[4], w.p0[5]};
    apply_shape_longitudinal<SHAPE>(q, g);
    zshift = q.z;
  }
  // transverse-only stages leave z and dp as they are
  const bool store_long = SHAPE == PHX_SHAPE_T || SHAPE == PHX_SHAPE_NONE
                              ? false
                              : (SHAPE != PHX_SHAPE_GENERIC || g.n_long > 0 || g.n_lin > 0);
  double v[ZB_NV];
#pragma unroll
  for (int i = 0; i < ZB_NV; ++i) v[i] = red_ident<ZB_MINM, ZB_MAXM>(i);
  const int64_t ng = phx_n_groups(n);
  for (int64_t gi = bid; gi < ng; gi += nblk) {
    const int64_t b = gi * PHX_CHUNK;
    const int64_t rest = n - b;
    const int lim = rest >= PHX_CHUNK ? PHX_CHUNK : (int)rest;
#pragma unroll 1
    for (int k = 0; k < PHX_PPT; ++k) {
      const int o = (int)threadIdx.x + k * PHX_BLOCK;
      if (o < lim) {
        const int64_t j = b + o;
        P6 p[1];
        p[0] = P6{ld_pos(x + j), ld_mom(xp + j), ld_pos(y + j), ld_mom(yp + j), ld_pos(z + j),
                  ld_mom(dp + j)};
        sc_kick_n<1>(p, scc, sp);
        apply_shape_n<SHAPE, 1, DS>(p, g);
        x[j] = p[0].x;
        st_mom(xp + j, p[0].xp);
        y[j] = p[0].y;
        st_mom(yp + j, p[0].yp);
        if (store_long) {
          z[j] = p[0].z;
          st_mom(dp + j, p[0].dp);
        }
        zblock_accumulate<0x05u>(v, p[0], zshift, minmax);
      }
    }
  }
  const double r = block_reduce_slots<ZB_NV, ZB_MINM, ZB_MAXM>(v, pass_lds);
  if (threadIdx.x < ZB_NV) w.partials[(size_t)threadIdx.x * nblk + bid] = r;
}

// The cuts of this turn from the pass partials (one block): fold the z
// block (and the statistics slots) in a fixed order, the slicing state, the
// statistics row, particle 0 for the next pass, and the wake-history
// bookkeeping (WakeField.track: ages += C/(beta c), then the new entry at
// age 0, impedances/wakes.py:134-142).  FOLD_ALL: this block does every
// part (the batch's cuts stage, block 0 of the standalone histogram);
// otherwise only the fold into res and the shared cut values (the other
// histogram blocks).  Returns the state through *stp (thread 0).
template <bool REC, bool FOLD_ALL>
__device__ __forceinline__ void cuts_body(const EngineArgs &a, double *res,
                                          phx_slice_state *stp) {
  using L = PassLayout<REC, true>;
  const phx_engine &e = a.e;
  EngineWs w = engine_ws(e.ws, e.n, e.n_slices);
  const int turn = *e.turn_counter;
  const phx_turn_program &g = e.programs[e.turn_program[turn]];
  if (FOLD_ALL && threadIdx.x < 6) w.p0[threadIdx.x] = e.coords[threadIdx.x][0];
  fold_partials<L::MINM, L::MAXM>(w.partials, a.grid, 0, ZB_NV, res);
  if constexpr (REC && FOLD_ALL) fold_partials<L::MINM, L::MAXM>(w.partials, a.grid, ZB_NV, L::NV, res);
  // the wake history: every stored entry ages by the turn's increment, one
  // thread per entry (a serial loop made the block wait on one round trip
  // per entry); the slot the new entry takes when the ring is full is
  // skipped, since thread 0 then sets it to age 0
  phx_wake_hist *h = e.hist;
  int cap = 1, nf = 0, nh = 0;
  if (FOLD_ALL) {
    const int head = h->head;
    cap = h->capacity;
    nf = h->n_filled;
    nh = (head + 1) % cap;
    for (int i = threadIdx.x; i < nf; i += blockDim.x) {
      const int sl = ring_slot(head, i, cap);
      if (sl != nh) h->age[sl] = h->age[sl] + g.age_increment;
    }
    lds_sync();  // every thread has read the ring's state before thread 0 moves it
  }
  if (threadIdx.x == 0) {
    phx_slice_state st;
    compute_cuts(g.slicer, e.n, res[0], res[1], res[2], res[3], res[4], st);
    for (int i = 0; i < 6; ++i) st.absmax[i] = res[5 + i];
    st.turn = turn;
    st.pad = 0;
    *stp = st;
    if (FOLD_ALL) {
      *e.state = st;
      h->head = nh;
      h->n_filled = nf + 1 < cap ? nf + 1 : cap;
      h->age[nh] = 0.0;
      h->beta[nh] = g.beta;
    }
  }
  if (REC && FOLD_ALL && threadIdx.x < EN_STAT_NV)
    e.stats[(size_t)turn * EN_STAT_NV + threadIdx.x] = res[L::SOFF + threadIdx.x];
}

// Slice histogram of the new state: counts, sum x and sum y per slice in an
// LDS histogram, stored as partial bid of nblk.  FOLD: the block first folds
// the pass partials into the cuts itself (every block, identical results;
// block 0 also publishes them and does the turn's bookkeeping); otherwise
// the cuts stage did that and the block reads the state.
template <bool REC, bool FOLD>
__device__ __forceinline__ void hist_body(const EngineArgs &a, int bid, int nblk) {
  using L = PassLayout<REC, true>;
  extern __shared__ unsigned long long acc_lds[];
  __shared__ double res[L::NV];
  __shared__ phx_slice_state sh_st;
  const phx_engine &e = a.e;
  EngineWs w = engine_ws(e.ws, e.n, e.n_slices);
  const int S = e.n_slices;
  constexpr int CH = EN_HIST_THREADS * EN_HIST_PPT;
  const int64_t nc = (e.n + CH - 1) / CH;
  const int64_t n = e.n;
  // Each chunk loads the next one before it is binned.  No particle load is
  // in flight across a barrier: with the first chunk's loads issued ahead
  // of the fold of the cuts, some blocks' folds came out wrong on MI355X
  // (about 1 in 25 block folds on a new engine's first turns; none with
  // the loads issued after the last barrier).
  double zz[EN_HIST_PPT], xx[EN_HIST_PPT], yy[EN_HIST_PPT];
  double zn[EN_HIST_PPT], xn[EN_HIST_PPT], yn[EN_HIST_PPT];
  auto load_chunk = [&](int64_t c, double (&z)[EN_HIST_PPT], double (&x)[EN_HIST_PPT],
                        double (&y)[EN_HIST_PPT]) {
#pragma unroll
    for (int k = 0; k < EN_HIST_PPT; ++k) {
      const int64_t j = c * CH + threadIdx.x + (int64_t)k * EN_HIST_THREADS;
      if (c < nc && j < n) {
        z[k] = e.coords[4][j];
        x[k] = e.coords[0][j];
        y[k] = e.coords[2][j];
      } else {
        z[k] = 0.0;
        x[k] = 0.0;
        y[k] = 0.0;
      }
    }
  };
  if constexpr (FOLD) {
    if (bid == 0) cuts_body<REC, true>(a, res, &sh_st);
    else cuts_body<REC, false>(a, res, &sh_st);
  } else {
    if (threadIdx.x == 0) sh_st = *e.state;
  }
  AccLds A = acc_lds_layout(acc_lds, S, 2);
  acc_lds_zero(A, S, 2);  // ends with a barrier: the shared cuts are visible
  const SliceBins bins(sh_st.tail, sh_st.width, S);
  const FxScale fx = fx_scale(sh_st.absmax[0], n), fy = fx_scale(sh_st.absmax[2], n);
  load_chunk(bid, zz, xx, yy);
  for (int64_t c = bid; c < nc; c += nblk) {
    load_chunk(c + nblk, zn, xn, yn);
    const int64_t base = c * CH + threadIdx.x;
#pragma unroll
    for (int k = 0; k < EN_HIST_PPT; ++k) {
      const int64_t j = base + (int64_t)k * EN_HIST_THREADS;
      if (j < n) {
        const int s = bins.index(zz[k]);
        if (s >= 0) {
          atomicAdd(&A.counts[s], 1u);
          acc_add_value(A, S, 0, s, xx[k], fx, w.acc.fallback);
          acc_add_value(A, S, 1, s, yy[k], fy, w.acc.fallback);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < EN_HIST_PPT; ++k) {
      zz[k] = zn[k];
      xx[k] = xn[k];
      yy[k] = yn[k];
    }
  }
  acc_lds_store(A, S, 2, w.acc, bid);
}

// Merge the partial histograms; means and the new history entry:
// times = z_centers / (beta c) (particles/slicing.py:124-126, 303-307),
// moments n, n*mean_x, n*mean_y (impedances/wake_kicks.py:217, 235).
// Block (S + SL - 1) / SL, launched when the engine has resistive-wall kicks
// in the dot-product form, describes the turn's kicks for the convolution
// (rw_desc_build) while the others merge.
// Three-launch turns (ahead): the blocks after those fold the pass's z sums
// into the next turn's cuts and do the bookkeeping that the histogram's block
// 0 does in the four-launch turn (the merge blocks read the ring's new slot
// from the turn's AheadState, so that nothing they read is written here).
enum { MA_CUTS = 0, MA_SHIFT, MA_RING, MA_STATS, MA_STATS_BLOCKS = 4 };
#define MA_THREADS 512
__host__ __device__ inline int merge_blocks(int S, int SL, bool desc, bool ahead, bool rec) {
  return (S + SL - 1) / SL + (desc ? 1 : 0) +
         (ahead ? MA_STATS + (rec ? MA_STATS_BLOCKS : 0) : 0);
}

// What merge_slice reads besides the totals, loaded before their reduction.
struct MergeIn {
  double beta_c, over_x, over_y;
  double *times, *mom;  // the new history entry
};

template <int SL>
__device__ __forceinline__ MergeIn merge_in(const phx_engine &e, const EngineWs &w, int prog,
                                            int nh, int s) {
  const int S = e.n_slices;
  MergeIn in;
  in.beta_c = e.programs[prog].beta_c;
  in.times = e.hist->times + (size_t)nh * S;
  in.mom = e.hist->mom + (size_t)nh * 3 * S;
  const bool mine = threadIdx.x < SL && s < S;
  in.over_x = mine ? w.acc.fallback[s] : 0.0;
  in.over_y = mine ? w.acc.fallback[S + s] : 0.0;
  return in;
}

__device__ __forceinline__ void merge_slice(const phx_engine &e, const EngineWs &w, int s,
                                            const SliceTotals &tot, const MergeIn &in,
                                            double tail, double width, double absx, double absy) {
  const int S = e.n_slices;
  // bin edges as np.arange(tail, head + 1e-7*width, width)
  e.z_bins[s] = arange_value(tail, width, s);
  if (s == S - 1) e.z_bins[S] = arange_value(tail, width, S);
  const FxScale fx = fx_scale(absx, e.n), fy = fx_scale(absy, e.n);
  const double cnt = (double)tot.count;
  const double sx = fx_value(tot.hi[0], tot.lo[0], in.over_x, fx);
  const double sy = fx_value(tot.hi[1], tot.lo[1], in.over_y, fy);
  w.acc.fallback[s] = 0.0;
  w.acc.fallback[S + s] = 0.0;
  const double mx = tot.count ? sx / cnt : 0.0;
  const double my = tot.count ? sy / cnt : 0.0;
  e.counts[s] = (int32_t)tot.count;
  e.slice_means[s] = mx;
  e.slice_means[S + s] = my;
  const double zl = arange_value(tail, width, s), zr = arange_value(tail, width, s + 1);
  const double zc = zl + 0.5 * (zr - zl);
  in.times[s] = zc / in.beta_c;
  in.mom[s] = cnt;
  in.mom[S + s] = cnt * mx;
  in.mom[2 * S + s] = cnt * my;
}

template <int SL>
__device__ __forceinline__ void merge_body(const EngineArgs &a, int bid) {
  const phx_engine &e = a.e;
  EngineWs w = engine_ws(e.ws, e.n, e.n_slices);
  const int S = e.n_slices;
  SliceTotals tot;
  const int turn = e.state->turn;
  if (bid == (S + SL - 1) / SL) {
    if (a.n_kicks < 1 || !e.hist) return;
    const phx_turn_program &g = e.programs[e.turn_program[turn]];
    const phx_wake_hist *h = e.hist;
    rw_desc_build(h, *reinterpret_cast<const WakeKicks *>(g.kick), a.n_kicks, a.T,
                  engine_rw_desc(w, a.n_kicks, S, a.T), h->n_filled, h->head, h->beta[h->head]);
    return;
  }
  if (bid == 0 && threadIdx.x == 0) *e.turn_counter = turn + 1;
  const int s = bid * SL + threadIdx.x % SL;
  const MergeIn in = merge_in<SL>(e, w, e.turn_program[turn], e.hist->head, s);
  const double tail = e.state->tail, width = e.state->width;
  const double absx = e.state->absmax[0], absy = e.state->absmax[2];
  if (!acc_merge<2, SL>(w.acc, S, tot, bid)) return;
  merge_slice(e, w, s, tot, in, tail, width, absx, absy);
}

// The cuts of the next turn and this turn's published state.
__device__ __forceinline__ void ahead_cuts_block(const EngineArgs &a, const EngineWs &w,
                                                 const AheadState &h) {
  const phx_engine &e = a.e;
  __shared__ double res[ZB_NV];
  const phx_turn_program &g = e.programs[e.turn_program[h.turn]];
  const phx_slicer cfg = g.slicer;
  const int cap = e.hist->capacity;
  ahead_fold(w.partials, a.grid, res);
  if (threadIdx.x == 0) {
    phx_slice_state st;
    st.tail = h.tail;
    st.head = h.head;
    st.width = h.width;
    st.mean_z = h.mean_z;
    st.sigma_z = h.sigma_z;
    for (int i = 0; i < 6; ++i) st.absmax[i] = -INFINITY;
    st.absmax[0] = res[5];
    st.absmax[2] = res[7];
    st.n = e.n;
    st.n_slices = cfg.n_slices;
    st.turn = h.turn;
    st.valid = 1;
    st.pad = 0;
    *e.state = st;
    ahead_set(*w.next, cfg, e.n, res, (h.nh + 1) % cap, h.nf + 1 < cap ? h.nf + 1 : cap,
              h.turn + 1);
    *e.turn_counter = h.turn + 1;
  }
}

template <int SL>
__device__ __forceinline__ void ahead_merge_body(const EngineArgs &a, int bid) {
  const phx_engine &e = a.e;
  EngineWs w = engine_ws(e.ws, e.n, e.n_slices);
  const int S = e.n_slices;
  const AheadState h = *w.cur;
  const int nm = (S + SL - 1) / SL;
  if (bid >= nm) {
    const phx_turn_program &g = e.programs[e.turn_program[h.turn]];
    const int k = bid - nm;
    if (k == MA_CUTS) {
      ahead_cuts_block(a, w, h);
    } else if (k == MA_SHIFT) {
      if (threadIdx.x < 6) w.p0[threadIdx.x] = e.coords[threadIdx.x][0];
      if (threadIdx.x == PHX_WAVE) w.next->zshift = ahead_shift(e.coords, g);
    } else if (k == MA_RING) {
      // the stored entries age by the turn's increment; the new one (slot
      // h.nh) has age 0 (WakeField.track, impedances/wakes.py:134-142)
      phx_wake_hist *r = e.hist;
      for (int i = threadIdx.x; i < h.nf; i += blockDim.x) {
        const int sl = ring_slot(h.nh, i, r->capacity);
        r->age[sl] = i == 0 ? 0.0 : r->age[sl] + g.age_increment;
      }
      if (threadIdx.x == 0) {
        r->head = h.nh;
        r->n_filled = h.nf;
        r->beta[h.nh] = g.beta;
      }
    } else if (e.record_stats && k < MA_STATS + MA_STATS_BLOCKS) {
      __shared__ double st[EN_NV];
      constexpr int per = (EN_STAT_NV + MA_STATS_BLOCKS - 1) / MA_STATS_BLOCKS;
      const int i0 = ZB_NV + (k - MA_STATS) * per;
      const int i1 = i0 + per < EN_NV ? i0 + per : EN_NV;
      fold_partials<0ULL, 0ULL>(w.partials, a.grid, i0, i1, st);
      if (threadIdx.x < i1 - i0)
        e.stats[(size_t)h.turn * EN_STAT_NV + (i0 - ZB_NV) + threadIdx.x] = st[i0 + threadIdx.x];
    } else {
      rw_desc_build(e.hist, *reinterpret_cast<const WakeKicks *>(g.kick), a.n_kicks, a.T,
                    engine_rw_desc(w, a.n_kicks, S, a.T), h.nf, h.nh, g.beta);
    }
    return;
  }
  SliceTotals tot;
  const int s = bid * SL + threadIdx.x % SL;
  const MergeIn in = merge_in<SL>(e, w, e.turn_program[h.turn], h.nh, s);
  if (!acc_merge<2, SL, MA_THREADS>(ahead_parts(w, S, a.hblk), S, tot, bid)) return;
  merge_slice(e, w, s, tot, in, h.tail, h.width, h.absx, h.absy);
}

// Space-charge slicing of the state after stage `stage` (the slicing that
// TransverseGaussianSpaceCharge.track asks for with mean_x, mean_y, sigma_x,
// sigma_y, spacecharge/spacecharge.py:207-208): every block folds the
// stage pass's z block into the cuts of the stage program's sc_slicer
// (block 0 publishes them and records particle 0 for the next pass), then
// keeps an LDS histogram of counts and fixed-point sums of x, y, x^2 and
// y^2, stored as its partial.  The scales come from max |x| and max |y| of
// the same state, so every term fits.
__device__ __forceinline__ void sc_hist_body(const EngineArgs &a, int stage, int bid, int nblk) {
  extern __shared__ unsigned long long acc_lds[];
  __shared__ double res[ZB_NV];
  __shared__ phx_slice_state sh_st;
  const phx_engine &e = a.e;
  EngineWs w = engine_ws(e.ws, e.n, e.n_slices);
  const ScWs sw = sc_ws(e.sc_ws, e.sc_slices);
  const int turn = *e.turn_counter;
  const phx_turn_program &g = e.programs[e.turn_program[turn] + stage];
  const int S = g.sc_slicer.n_slices;
  const int64_t n = e.n;
  const AccParts P = acc_parts_layout(sw.acc, hist_blocks(n), S, SC_TERMS);
  fold_partials<ZB_MINM, ZB_MAXM>(w.partials, a.grid, 0, ZB_NV, res);
  if (threadIdx.x == 0) {
    phx_slice_state st;
    compute_cuts(g.sc_slicer, n, res[0], res[1], res[2], res[3], res[4], st);
    for (int i = 0; i < 6; ++i) st.absmax[i] = res[5 + i];
    st.turn = turn;
    st.pad = 0;
    sh_st = st;
    if (bid == 0) *sw.state = st;
  }
  if (bid == 0 && threadIdx.x < 6) w.p0[threadIdx.x] = e.coords[threadIdx.x][0];
  AccLds A = acc_lds_layout(acc_lds, S, SC_TERMS);
  acc_lds_zero(A, S, SC_TERMS);  // ends with a barrier: the shared cuts are visible
  const SliceBins bins(sh_st.tail, sh_st.width, S);
  const double bx = sh_st.absmax[0], by = sh_st.absmax[2];
  const FxScale fx = fx_scale(bx, n), fy = fx_scale(by, n);
  const FxScale fxx = fx_scale(bx * bx, n), fyy = fx_scale(by * by, n);
  constexpr int CH = EN_HIST_THREADS * EN_HIST_PPT;
  const int64_t nc = (n + CH - 1) / CH;
  double zz[EN_HIST_PPT], xx[EN_HIST_PPT], yy[EN_HIST_PPT];
  double zn[EN_HIST_PPT], xn[EN_HIST_PPT], yn[EN_HIST_PPT];
  auto load_chunk = [&](int64_t c, double (&zv)[EN_HIST_PPT], double (&xv)[EN_HIST_PPT],
                        double (&yv)[EN_HIST_PPT]) {
#pragma unroll
    for (int k = 0; k < EN_HIST_PPT; ++k) {
      const int64_t j = c * CH + threadIdx.x + (int64_t)k * EN_HIST_THREADS;
      if (c < nc && j < n) {
        zv[k] = e.coords[4][j];
        xv[k] = e.coords[0][j];
        yv[k] = e.coords[2][j];
      } else {
        zv[k] = 0.0;
        xv[k] = 0.0;
        yv[k] = 0.0;
      }
    }
  };
  load_chunk(bid, zz, xx, yy);
  for (int64_t c = bid; c < nc; c += nblk) {
    load_chunk(c + nblk, zn, xn, yn);
    const int64_t base = c * CH + threadIdx.x;
#pragma unroll
    for (int k = 0; k < EN_HIST_PPT; ++k) {
      const int64_t j = base + (int64_t)k * EN_HIST_THREADS;
      if (j < n) {
        const int s = bins.index(zz[k]);
        if (s >= 0) {
          atomicAdd(&A.counts[s], 1u);
          acc_add_value(A, S, 0, s, xx[k], fx, P.fallback);
          acc_add_value(A, S, 1, s, yy[k], fy, P.fallback);
          acc_add_value(A, S, 2, s, xx[k] * xx[k], fxx, P.fallback);
          acc_add_value(A, S, 3, s, yy[k] * yy[k], fyy, P.fallback);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < EN_HIST_PPT; ++k) {
      zz[k] = zn[k];
      xx[k] = xn[k];
      yy[k] = yn[k];
    }
  }
  acc_lds_store(A, S, SC_TERMS, P, bid);
}

// A fixed-point total as an unevaluated double-double hi + lo: fx_value
// before its last rounding, the out-of-range parts (if any) in lo.
__device__ __forceinline__ void fx_value_dd(unsigned long long hi_sum, unsigned long long lo_sum,
                                            double over, const FxScale &f, double &hi,
                                            double &lo) {
  const long long h = (long long)hi_sum + ((long long)lo_sum >> FX_LB);
  const double a = (double)h;
  const long long r = h - (long long)a;
  const double b = (double)(r * (1LL << FX_LB) + (long long)(lo_sum & ((1ULL << FX_LB) - 1ULL))) *
                   (1.0 / (double)(1LL << FX_LB));
  const double s = a + b;
  const double bb = s - a;
  const double t = (a - (s - bb)) + (b - bb);
  hi = s * f.unit;
  lo = t * f.unit + over;
}

// (q - x^2/n) / (n - 1) from double-double totals x = sum u, q = sum u^2:
// the variance with the single rounding of each u^2 and of the result.
__device__ __forceinline__ double var_from_sums(double xh, double xl, double qh, double ql,
                                                double n) {
  // x^2 as double-double
  const double ph = xh * xh;
  const double pl = fma(xh, xh, -ph) + 2.0 * xh * xl;
  // (ph + pl) / n
  const double q1 = ph / n;
  const double r = fma(-q1, n, ph);
  const double q2 = (r + pl) / n;
  // (qh + ql) - (q1 + q2)
  const double s = qh - q1;
  const double bb = s - qh;
  const double err = (qh - (s - bb)) + (-q1 - bb);
  const double d = s + ((err + ql) - q2);
  const double v = d / (n - 1.0);
  return v > 0.0 ? v : 0.0;
}

// Merge of the space-charge partial histograms: per slice the count, means
// (mean_per_slice: sum / n, 0 for empty slices), standard deviations
// (std_per_slice: 0 for n <= 1) and the line density, into the field rows
// the next stage's kick reads.
template <int SL>
__device__ __forceinline__ void sc_merge_body(const EngineArgs &a, int stage, int bid) {
  const phx_engine &e = a.e;
  const ScWs sw = sc_ws(e.sc_ws, e.sc_slices);
  const int turn = *e.turn_counter;
  const phx_turn_program &g = e.programs[e.turn_program[turn] + stage];
  const int S = g.sc_slicer.n_slices;
  const AccParts P = acc_parts_layout(sw.acc, hist_blocks(e.n), S, SC_TERMS);
  SliceTotals tot;
  if (!acc_merge<SC_TERMS, SL>(P, S, tot, bid)) return;
  const int s = bid * SL + threadIdx.x % SL;
  const phx_slice_state &st = *sw.state;
  const double tail = st.tail, width = st.width;
  const double bx = st.absmax[0], by = st.absmax[2];
  const FxScale sfx = fx_scale(bx, e.n), sfy = fx_scale(by, e.n);
  const FxScale sfxx = fx_scale(bx * bx, e.n), sfyy = fx_scale(by * by, e.n);
  const double cnt = (double)tot.count;
  const double fx = P.fallback[s], fy = P.fallback[S + s];
  const double fxx = P.fallback[2 * S + s], fyy = P.fallback[3 * S + s];
  P.fallback[s] = 0.0;
  P.fallback[S + s] = 0.0;
  P.fallback[2 * S + s] = 0.0;
  P.fallback[3 * S + s] = 0.0;
  const double sx = fx_value(tot.hi[0], tot.lo[0], fx, sfx);
  const double sy = fx_value(tot.hi[1], tot.lo[1], fy, sfy);
  ScSlice row;
  row.mx = tot.count ? sx / cnt : 0.0;
  row.my = tot.count ? sy / cnt : 0.0;
  double sgx = 0.0, sgy = 0.0;
  if (tot.count > 1) {
    double xh, xl, yh, yl, qxh, qxl, qyh, qyl;
    fx_value_dd(tot.hi[0], tot.lo[0], fx, sfx, xh, xl);
    fx_value_dd(tot.hi[1], tot.lo[1], fy, sfy, yh, yl);
    fx_value_dd(tot.hi[2], tot.lo[2], fxx, sfxx, qxh, qxl);
    fx_value_dd(tot.hi[3], tot.lo[3], fyy, sfyy, qyh, qyl);
    sgx = sqrt(var_from_sums(xh, xl, qxh, qxl, cnt));
    sgy = sqrt(var_from_sums(yh, yl, qyh, qyl, cnt));
  }
  row.nl = sc_line_density((int32_t)tot.count, g.sc.charge_per_mp, arange_value(tail, width, s),
                           arange_value(tail, width, s + 1));
  row.pad = 0.0;
  row.f = sc_field_params(sgx, sgy, g.sc);
  sw.slices[s] = row;
}

// Slices per merge block: 4 up to 512 slices, 8 above (5.2 / 6.3 us at 500
// slices, 7.2 / 6.3 us at 1000); integer sums, the same results.
__host__ __device__ inline int merge_sl(int S) { return S <= 512 ? 4 : 8; }

// The first block of a turn's convolution: its kicks are pending, and the next
// turn's AheadState, complete by now, becomes `cur` (a word per thread, loaded
// ahead of the block's own work and stored after it).
struct ConvPublish {
  static constexpr int NW = sizeof(AheadState) / 8;
  double v;
  bool mine;
  __device__ __forceinline__ void begin(const EngineWs &w, bool first_block) {
    mine = first_block && threadIdx.x < NW;
    v = mine ? reinterpret_cast<const double *>(w.next)[threadIdx.x] : 0.0;
  }
  __device__ __forceinline__ void end(const phx_engine &e, const EngineWs &w) const {
    if (!mine) return;
    reinterpret_cast<double *>(w.cur)[threadIdx.x] = v;
    if (threadIdx.x == 0) *e.pending = 1;
  }
};
static_assert(sizeof(AheadState) % 8 == 0, "AheadState is copied in words");

// Wake convolution block (tile, ki, t) of the general kernel.
__device__ __forceinline__ void conv_body(const EngineArgs &a, int tile, int ki, int t) {
  const phx_engine &e = a.e;
  EngineWs w = engine_ws(e.ws, e.n, e.n_slices);
  const phx_turn_program &g = e.programs[e.turn_program[e.state->turn]];
  const WakeKicks &kk = *reinterpret_cast<const WakeKicks *>(g.kick);
  ConvPublish pub;
  pub.begin(w, tile == 0 && ki == 0 && t == 0);
  wake_conv_block(e.hist, kk, e.n_slices, w.conv_part, a.T, e.kicks, a.gmax, tile, ki, t,
                  a.n_kicks);
  pub.end(e, w);
}

template <int KM>
__device__ __forceinline__ void conv_rw_body(const EngineArgs &a, int bid) {
  const phx_engine &e = a.e;
  EngineWs w = engine_ws(e.ws, e.n, e.n_slices);
  ConvPublish pub;
  pub.begin(w, bid == 0);
  wake_rw_block<KM>(e.hist, engine_rw_desc(w, a.n_kicks, e.n_slices, a.T), a.n_kicks,
                    e.n_slices, w.conv_part, a.T, e.kicks, bid);
  pub.end(e, w);
}

__device__ __forceinline__ void conv_reduce_body(const EngineArgs &a, int bid) {
  const phx_engine &e = a.e;
  EngineWs w = engine_ws(e.ws, e.n, e.n_slices);
  const phx_turn_program &g = e.programs[e.turn_program[e.state->turn]];
  const WakeKicks &kk = *reinterpret_cast<const WakeKicks *>(g.kick);
  wake_conv_reduce(e.hist, kk, a.n_kicks, e.n_slices, w.conv_part, a.T, e.kicks, bid);
}

// Launch arguments of engine e (checked): the record, its kick count and
// memory depth, the pass grid and the convolution blocks (phx_engine.hip).
int engine_args_for(const phx_engine *e, EngineArgs *out);

}  // namespace phx_en
