// Device-side building blocks shared by the standalone element kernels and
// the fused turn engine.  Everything here is FP64 and is compiled with
// -ffp-contract=off so that each arithmetic operation is one IEEE-754
// rounding.  Slicing, the linear map and the transverse map without detuning
// are the operations of the reference's NumPy expressions in their order.
// Where a sine or cosine enters (RF kicks, detuned phases), which no two
// libraries round alike, the expressions are arranged for fewer operations:
// phases in turns, constant quotients folded once, sums of products as FMAs,
// with fewer roundings than the reference's order.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/phx.h"
#include "phx_math.h"

#define PHX_BLOCK 256
#define PHX_WAVE 64
#ifndef PHX_PPT
#define PHX_PPT 2
#endif
#define PHX_CHUNK (PHX_BLOCK * PHX_PPT)
// Reducing particle passes run a persistent grid of G blocks: block b
// handles the particle groups b, b + G, b + 2G, ... of PHX_CHUNK particles
// (thread t: particles g*PHX_CHUNK + k*PHX_BLOCK + t, k < PHX_PPT), so block
// b's partial covers a fixed set of particles in a fixed order for a given G.
// The standalone reductions use G = PHX_STANDALONE_GRID (three blocks on
// each of MI355X's 256 CUs); the engine's pass uses the grid that stays
// resident for its kernel, at most PHX_MAX_GRID.

__host__ __device__ inline int64_t phx_n_groups(int64_t n) {
  return n <= 0 ? 0 : (n + PHX_CHUNK - 1) / PHX_CHUNK;
}
__host__ __device__ inline int phx_grid_for(int64_t n, int64_t grid) {
  const int64_t g = phx_n_groups(n);
  return (int)(g < grid ? g : grid);
}
__host__ __device__ inline int phx_pass_grid(int64_t n) {
  return phx_grid_for(n, PHX_STANDALONE_GRID);
}
// NumPy's 2.*np.pi as a double
#define PHX_TWO_PI 6.283185307179586
#define PHX_PI 3.141592653589793

struct P6 {
  double x, xp, y, yp, z, dp;
};

// Workgroup barrier for data exchanged through LDS only.  __syncthreads()
// also waits for every outstanding global load and store of the wave (its
// release fence covers global memory); this one waits for LDS operations
// only, so particle stores stay in flight across it.  Every barrier of this
// library protects LDS data only.  No kernel here leaves a global load in
// flight across it: the slice histogram's fold of the cuts, with the first
// particle loads issued ahead of it, gave wrong maxima in some blocks on
// MI355X.
__device__ __forceinline__ void lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ double p6_get(const P6 &p, int c) {
  switch (c) {
    case 0: return p.x;
    case 1: return p.xp;
    case 2: return p.y;
    case 3: return p.yp;
    case 4: return p.z;
    default: return p.dp;
  }
}

// ---------------------------------------------------------------------------
// Slice index: int32(floor((z - tail) / width)); particles/slicing.py:609-611.
// Returns the floor as a double; "inside" means 0 <= f < n_slices, which is
// false for NaN exactly as the int32 conversion of NaN (INT32_MIN on x86) is
// outside [0, n_slices).
// ---------------------------------------------------------------------------
__device__ __forceinline__ double slice_floor(double z, double tail, double width) {
  return floor((z - tail) / width);
}

// a / b, given r = 1.0 / b (correctly rounded): q0 = a r, the residual
// a - b q0 (exact, one FMA) and q0 + (a - b q0) r rounded once, which is the
// correctly rounded quotient when nothing overflows or underflows
// (Markstein's theorem on division by a correctly rounded reciprocal) --
// the same bits as the division, in three operations instead of the
// division's scaled Newton sequence.  Quotients outside [2^-900, 2^900]
// (zero, infinity, NaN, extreme magnitudes) are recomputed by the
// division itself.
__device__ __forceinline__ double div_rcp(double a, double b, double r) {
  const double q0 = a * r;
  const double e = fma(-q0, b, a);
  const double q = fma(e, r, q0);
  const double m = fabs(q);
  if (__builtin_expect(!(m >= 0x1p-900 && m <= 0x1p900), 0)) return a / b;
  return q;
}

// slice_floor with inv_width = 1.0 / width (the same value).
__device__ __forceinline__ double slice_floor_r(double z, double tail, double width,
                                                double inv_width) {
  return floor(div_rcp(z - tail, width, inv_width));
}

// The slices of one state for many particles: index(z) is the slice of z in
// [0, S), or a negative number outside the cuts; int32(floor((z - tail) /
// width)) exactly.  For widths in [2^-400, 2^400] the quotient is div_rcp's
// without its range check: a quotient of extreme magnitude only has to keep
// its sign and its place beyond S, and a non-finite one becomes NaN, which is
// outside either way.  Other widths (uniform) divide.
struct SliceBins {
  double tail, width, inv, S;
  bool plain;
  __device__ __forceinline__ SliceBins() {}
  __device__ __forceinline__ SliceBins(double t, double w, int n)
      : tail(t), width(w), inv(1.0 / w), S((double)n), plain(w >= 0x1p-400 && w <= 0x1p400) {}
  __device__ __forceinline__ int index(double z) const {
    const double a = z - tail;
    const double q0 = a * inv;
    double q = fma(fma(-q0, width, a), inv, q0);
    if (__builtin_expect(!plain, 0)) q = a / width;
    return q >= 0.0 && q < S ? (int)q : -1;
  }
};

__device__ __forceinline__ int32_t x86_cvt_i32(double f) {
  // cvttsd2si semantics: NaN and out-of-range values give INT32_MIN
  if (!(f >= -2147483648.0 && f < 2147483648.0)) return INT32_MIN;
  return (int32_t)f;
}

// ---------------------------------------------------------------------------
// Transverse segment map (trackers/transverse_tracking.py:138-196) with the
// detuners (trackers/detuners.py:64-98 chromaticity, :128-151 amplitude).
// ---------------------------------------------------------------------------
// A tune shift added to the phases (in turns) of N particles.
//   chromaticity: Horner form of (c0 + (c1 + c2 dp) dp) dp;
//   amplitude: dQ_x = (dapp_x Jx + dapp_xy Jy) / p0 with
//   Jx = ((1 + a^2)/b x^2 + 2 a x xp + b xp^2) / 2; the strengths come with
//   1 / (2 p0) folded in.
// SMOOTH: segments (PHX_DETS_SMOOTH) with alpha = 0, for which the host
// checked ax2 = ay2 = 0 and gx, gy > 0: then (ax2 x) xp is a zero added to
// bx xp^2 >= +0, which leaves it unchanged, and the term is dropped (the same
// bits for finite coordinates).
template <int N, bool SMOOTH = false>
__device__ __forceinline__ void detune_amplitude_n(const phx_detuner &d, const P6 (&p)[N],
                                                   double (&ux)[N], double (&uy)[N]) {
  const double f = 0.5 * d.inv_p0;
  const double axx = d.dapp_x * f, axy = d.dapp_xy * f, ayy = d.dapp_y * f, ayx = d.dapp_yx * f;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    double jx = (d.bx * p[k].xp) * p[k].xp, jy = (d.by * p[k].yp) * p[k].yp;
    if constexpr (!SMOOTH) {
      jx = fma(d.ax2 * p[k].x, p[k].xp, jx);
      jy = fma(d.ay2 * p[k].y, p[k].yp, jy);
    }
    jx = fma(d.gx * p[k].x, p[k].x, jx);
    jy = fma(d.gy * p[k].y, p[k].y, jy);
    ux[k] = ux[k] + fma(axx, jx, axy * jy);
    uy[k] = uy[k] + fma(ayy, jy, ayx * jx);
  }
}

template <int N>
__device__ __forceinline__ void detune_n(const phx_detuner &d, const P6 (&p)[N], double (&ux)[N],
                                         double (&uy)[N]) {
  if (d.type == PHX_DET_CHROMA) {
    double ax[N], ay[N];
#pragma unroll
    for (int k = 0; k < N; ++k) {
      ax[k] = d.cx[d.order - 1];
      ay[k] = d.cy[d.order - 1];
    }
    for (int i = d.order - 2; i >= 0; --i)
#pragma unroll
      for (int k = 0; k < N; ++k) {
        ax[k] = fma(ax[k], p[k].dp, d.cx[i]);
        ay[k] = fma(ay[k], p[k].dp, d.cy[i]);
      }
#pragma unroll
    for (int k = 0; k < N; ++k) {
      ux[k] = fma(ax[k], p[k].dp, ux[k]);
      uy[k] = fma(ay[k], p[k].dp, uy[k]);
    }
  } else {
    detune_amplitude_n<N>(d, p, ux, uy);
  }
}

// The detuner sets with straight-line code (PHX_DETS_*): first-order
// chromaticity (order-1 Horner: c0 * dp), then amplitude detuning; the
// arithmetic of detune_n for those sets.
template <int N, int DS>
__device__ __forceinline__ void detune_set_n(const phx_tseg &t, const P6 (&p)[N],
                                             double (&ux)[N], double (&uy)[N]) {
  const phx_detuner &c = t.det[0];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    ux[k] = fma(c.cx[0], p[k].dp, ux[k]);
    uy[k] = fma(c.cy[0], p[k].dp, uy[k]);
  }
  if constexpr ((DS & ~PHX_DETS_SMOOTH) == PHX_DETS_C1_AMP)
    detune_amplitude_n<N, (DS & PHX_DETS_SMOOTH) != 0>(t.det[1], p, ux, uy);
}

// The element functions act on N particles at once: the element's constants
// are read once and the N independent particles interleave (instruction-level
// parallelism for the long FP64 chains).  The arithmetic of each particle is
// the same for every N.
template <int N, int DS = PHX_DETS_GENERIC>
__device__ __forceinline__ void apply_tseg_n(P6 (&p)[N], const phx_tseg &t) {
  double M00[N], M01[N], M10[N], M11[N], M22[N], M23[N], M32[N], M33[N];
  constexpr bool SMOOTH = (DS & PHX_DETS_SMOOTH) != 0 && (DS & ~PHX_DETS_SMOOTH) >= PHX_DETS_C1;
  const int nd = DS == PHX_DETS_GENERIC ? t.n_detuners : (DS == PHX_DETS_NONE ? 0 : 1);
  if (nd == 0) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      M00[k] = t.M00; M01[k] = t.M01; M10[k] = t.M10; M11[k] = t.M11;
      M22[k] = t.M22; M23[k] = t.M23; M32[k] = t.M32; M33[k] = t.M33;
    }
  } else {
    // phases in turns, each detuner's shift added in order as the reference
    // adds it
    double u[2 * N], ux[N], uy[N], sn[2 * N], cs[2 * N];
#pragma unroll
    for (int k = 0; k < N; ++k) {
      ux[k] = t.dQ_x;
      uy[k] = t.dQ_y;
    }
    if constexpr (DS == PHX_DETS_GENERIC) {
      for (int i = 0; i < nd; ++i) detune_n<N>(t.det[i], p, ux, uy);
    } else {
      detune_set_n<N, DS>(t, p, ux, uy);
    }
    const double I00 = t.I00, I01 = t.I01, I10 = t.I10, I11 = t.I11;
    const double I22 = t.I22, I23 = t.I23, I32 = t.I32, I33 = t.I33;
    const double J00 = t.J00, J01 = t.J01, J10 = t.J10, J11 = t.J11;
    const double J22 = t.J22, J23 = t.J23, J32 = t.J32, J33 = t.J33;
#pragma unroll
    for (int k = 0; k < N; ++k) {
      u[k] = ux[k];
      u[N + k] = uy[k];
    }
    phx_sincos_turns_n<2 * N>(u, sn, cs);
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const double sx = sn[k], cx = cs[k], sy = sn[N + k], cy = cs[N + k];
      if constexpr (SMOOTH) {
        // 1 * cos + 0 * sin and 0 * cos + J * sin, each rounded once: the
        // same values
        M00[k] = cx;
        M01[k] = J01 * sx;
        M10[k] = J10 * sx;
        M11[k] = cx;
        M22[k] = cy;
        M23[k] = J23 * sy;
        M32[k] = J32 * sy;
        M33[k] = cy;
        continue;
      }
      M00[k] = fma(I00, cx, J00 * sx);
      M01[k] = fma(J01, sx, I01 * cx);
      M10[k] = fma(J10, sx, I10 * cx);
      M11[k] = fma(I11, cx, J11 * sx);
      M22[k] = fma(I22, cy, J22 * sy);
      M23[k] = fma(J23, sy, I23 * cy);
      M32[k] = fma(J32, sy, I32 * cy);
      M33[k] = fma(I33, cy, J33 * sy);
    }
  }
  const bool disp = !SMOOTH && t.with_dispersion != 0;
  const double dx0 = t.D_x_s0, dy0 = t.D_y_s0, dx1 = t.D_x_s1, dy1 = t.D_y_s1;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    P6 &q = p[k];
    if (disp) {
      q.x = q.x - dx0 * q.dp;
      q.y = q.y - dy0 * q.dp;
    }
    const double x = q.x, xp = q.xp, y = q.y, yp = q.yp;
    if (nd == 0) {  // the reference's operations, bit for bit
      q.x = M00[k] * x + M01[k] * xp;
      q.xp = M10[k] * x + M11[k] * xp;
      q.y = M22[k] * y + M23[k] * yp;
      q.yp = M32[k] * y + M33[k] * yp;
    } else {
      q.x = fma(M00[k], x, M01[k] * xp);
      q.xp = fma(M10[k], x, M11[k] * xp);
      q.y = fma(M22[k], y, M23[k] * yp);
      q.yp = fma(M32[k], y, M33[k] * yp);
    }
    if (disp) {
      q.x = q.x + dx1 * q.dp;
      q.y = q.y + dy1 * q.dp;
    }
  }
}

// ---------------------------------------------------------------------------
// Longitudinal maps (trackers/longitudinal_tracking.py).
// ---------------------------------------------------------------------------
// STAT: a stationary RF sequence (PHX_SHAPE_STATIONARY): beta_ratio = 1,
// phi_offset = phi_lock = p_increment = +0 and no dispersion, checked by the
// host, so that 1 * z = z, a phase offset of +0 and fma(dp, r, -0) = dp r drop
// those terms with the same bits.
template <int N, bool STAT = false>
__device__ __forceinline__ void drift_n(P6 (&p)[N], const phx_long_op &o) {
  // Drift.track: z = beta_ratio*z - eta(dp)*dp*length   (:107-111)
  const double e = -(o.eta0 * o.length);
  if constexpr (STAT) {
#pragma unroll
    for (int k = 0; k < N; ++k) p[k].z = fma(e, p[k].dp, p[k].z);
  } else {
    const double br = o.beta_ratio;
#pragma unroll
    for (int k = 0; k < N; ++k) p[k].z = fma(e, p[k].dp, br * p[k].z);
  }
}

template <int N, bool STAT = false>
__device__ __forceinline__ void rf_kick_n(P6 (&p)[N], const phx_long_op &o) {
  // Kick.track_with_dispersion / track_without_dispersion (:185-203):
  //   phi = h (2 pi z / C) + phi_offset + phi_lock
  //   dp = (dp p0_before + amplitude sin(phi) - p_increment) / p0_after
  // with phi in turns and the quotients by C and p0_after folded into the
  // kick's constants
  const double hz = o.harmonic * o.inv_circumference, amp = o.amplitude * o.inv_p0_after;
  const double ratio = o.p0_before == o.p0_after ? 1.0 : o.p0_before / o.p0_after;
  double u[N], sn[N];
  if constexpr (STAT) {
#pragma unroll
    for (int k = 0; k < N; ++k) u[k] = fma(p[k].z, hz, 0.0);
    phx_sin_turns_n<N>(u, sn);
#pragma unroll
    for (int k = 0; k < N; ++k) p[k].dp = fma(amp, sn[k], p[k].dp * ratio);
    return;
  }
  const bool disp = o.with_dispersion != 0;
  const double Dx = o.D_x, Dy = o.D_y;
  const double off = (o.phi_offset + o.phi_lock) * (1.0 / phx_math::TWO_PI);
  const double pinc = -(o.p_increment * o.inv_p0_after);
#pragma unroll
  for (int k = 0; k < N; ++k) {
    if (disp) {
      p[k].x = p[k].x - Dx * p[k].dp;
      p[k].y = p[k].y - Dy * p[k].dp;
    }
    u[k] = fma(p[k].z, hz, off);
  }
  phx_sin_turns_n<N>(u, sn);
#pragma unroll
  for (int k = 0; k < N; ++k) {
    p[k].dp = fma(amp, sn[k], fma(p[k].dp, ratio, pinc));
    if (disp) {
      p[k].x = p[k].x + Dx * p[k].dp;
      p[k].y = p[k].y + Dy * p[k].dp;
    }
  }
}

// A sequence is RFSystems' [drift, kicks..., drift] (:362-369) or a single
// Drift or Kick; the leading and trailing drifts are applied outside the
// loop over the inner operations, which keeps the kick's registers apart
// from the drift's.
template <int N>
__device__ __forceinline__ void shrink_n(P6 (&p)[N], const phx_long_seq &s) {
  // RFSystems._shrink_transverse_emittance (:556-565)
  if (s.shrink) {
    const double f = s.shrink_factor;
#pragma unroll
    for (int k = 0; k < N; ++k) {
      p[k].x = p[k].x * f;
      p[k].xp = p[k].xp * f;
      p[k].y = p[k].y * f;
      p[k].yp = p[k].yp * f;
    }
  }
}

template <int N>
__device__ __forceinline__ void apply_long_seq_n(P6 (&p)[N], const phx_long_seq &s) {
  const int n_ops = s.n_ops;
  const bool lead = n_ops > 0 && s.op[0].type == PHX_LONG_DRIFT;
  const bool trail = n_ops > 1 && s.op[n_ops - 1].type == PHX_LONG_DRIFT;
  if (lead) drift_n<N>(p, s.op[0]);
  const int i1 = trail ? n_ops - 1 : n_ops;
  for (int i = lead ? 1 : 0; i < i1; ++i) {
    if (s.op[i].type == PHX_LONG_DRIFT) drift_n<N>(p, s.op[i]);
    else rf_kick_n<N>(p, s.op[i]);
  }
  if (trail) drift_n<N>(p, s.op[n_ops - 1]);
  shrink_n<N>(p, s);
}

// RFSystems' sequence with NH harmonics: op[0] drift, op[1..NH] kicks,
// op[NH+1] drift.
template <int NH, int N, bool STAT = false>
__device__ __forceinline__ void apply_rf_seq_n(P6 (&p)[N], const phx_long_seq &s) {
  drift_n<N, STAT>(p, s.op[0]);
#pragma unroll
  for (int i = 1; i <= NH; ++i) rf_kick_n<N, STAT>(p, s.op[i]);
  drift_n<N, STAT>(p, s.op[NH + 1]);
  shrink_n<N>(p, s);
}

template <int N>
__device__ __forceinline__ void apply_linmap_n(P6 (&p)[N], const phx_linmap &m) {
  // LinearMap.track_with_dispersion -> track_without_dispersion (:731-759)
  const double Dx = m.D_x, Dy = m.D_y, cq = m.cosQ, sq = m.sinQ, lf = m.longfac;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    P6 &q = p[k];
    q.x = q.x - Dx * q.dp;
    q.y = q.y - Dy * q.dp;
    const double z0 = q.z, dp0 = q.dp;
    q.z = z0 * cq - (lf * dp0) * sq;
    q.dp = dp0 * cq + (z0 / lf) * sq;
    q.x = q.x + Dx * q.dp;
    q.y = q.y + Dy * q.dp;
  }
}

template <int N>
__device__ __forceinline__ void apply_program_n(P6 (&p)[N], const phx_turn_program &g) {
  for (int e = 0; e < g.n_el; ++e) {
    const int k = g.el_index[e];
    switch (g.el_type[e]) {
      case PHX_EL_TSEG: apply_tseg_n<N>(p, g.tseg[k]); break;
      case PHX_EL_LONG: apply_long_seq_n<N>(p, g.lseq[k]); break;
      default: apply_linmap_n<N>(p, g.lin[k]); break;
    }
  }
}

// A program of a known element order (PHX_SHAPE_*): the elements are
// applied in straight-line code, which the compiler schedules and allocates
// registers for far better than the interpreter's loop over element kinds.
template <int SHAPE, int N, int DS = PHX_DETS_GENERIC>
__device__ __forceinline__ void apply_shape_n(P6 (&p)[N], const phx_turn_program &g) {
  constexpr int SH = SHAPE & ~PHX_SHAPE_STATIONARY;
  constexpr bool ST = SH != SHAPE;
  if constexpr (SH == PHX_SHAPE_RF1_T) {
    apply_rf_seq_n<1, N, ST>(p, g.lseq[0]);
    apply_tseg_n<N, DS>(p, g.tseg[0]);
  } else if constexpr (SH == PHX_SHAPE_RF2_T) {
    apply_rf_seq_n<2, N, ST>(p, g.lseq[0]);
    apply_tseg_n<N, DS>(p, g.tseg[0]);
  } else if constexpr (SH == PHX_SHAPE_T_RF1) {
    apply_tseg_n<N, DS>(p, g.tseg[0]);
    apply_rf_seq_n<1, N, ST>(p, g.lseq[0]);
  } else if constexpr (SH == PHX_SHAPE_T_RF2) {
    apply_tseg_n<N, DS>(p, g.tseg[0]);
    apply_rf_seq_n<2, N, ST>(p, g.lseq[0]);
  } else if constexpr (SH == PHX_SHAPE_LIN_T) {
    apply_linmap_n<N>(p, g.lin[0]);
    apply_tseg_n<N, DS>(p, g.tseg[0]);
  } else if constexpr (SH == PHX_SHAPE_T_LIN) {
    apply_tseg_n<N, DS>(p, g.tseg[0]);
    apply_linmap_n<N>(p, g.lin[0]);
  } else if constexpr (SH == PHX_SHAPE_T) {
    apply_tseg_n<N, DS>(p, g.tseg[0]);
  } else if constexpr (SH == PHX_SHAPE_NONE) {
  } else {
    apply_program_n<N>(p, g);
  }
}

// z and dp after a program: only the longitudinal elements change them
// (transverse segments act on x, xp, y, yp), so applying those alone gives
// the same z and dp bit for bit.
template <int SHAPE, int N>
__device__ __forceinline__ void apply_shape_longitudinal_n(P6 (&p)[N], const phx_turn_program &g) {
  constexpr int SH = SHAPE & ~PHX_SHAPE_STATIONARY;
  constexpr bool ST = SH != SHAPE;
  if constexpr (SH == PHX_SHAPE_RF1_T || SH == PHX_SHAPE_T_RF1) {
    apply_rf_seq_n<1, N, ST>(p, g.lseq[0]);
  } else if constexpr (SH == PHX_SHAPE_RF2_T || SH == PHX_SHAPE_T_RF2) {
    apply_rf_seq_n<2, N, ST>(p, g.lseq[0]);
  } else if constexpr (SH == PHX_SHAPE_LIN_T || SH == PHX_SHAPE_T_LIN) {
    apply_linmap_n<N>(p, g.lin[0]);
  } else if constexpr (SH == PHX_SHAPE_GENERIC) {
    for (int e = 0; e < g.n_el; ++e) {
      const int k = g.el_index[e];
      if (g.el_type[e] == PHX_EL_LONG) apply_long_seq_n<N>(p, g.lseq[k]);
      else if (g.el_type[e] == PHX_EL_LINMAP) apply_linmap_n<N>(p, g.lin[k]);
    }
  }
}

template <int SHAPE>
__device__ __forceinline__ void apply_shape_longitudinal(P6 &q, const phx_turn_program &g) {
  apply_shape_longitudinal_n<SHAPE, 1>(*reinterpret_cast<P6(*)[1]>(&q), g);
}

__device__ __forceinline__ P6 (&one(P6 &p))[1] { return *reinterpret_cast<P6(*)[1]>(&p); }
__device__ __forceinline__ void apply_tseg(P6 &p, const phx_tseg &t) { apply_tseg_n<1>(one(p), t); }
__device__ __forceinline__ void apply_long_seq(P6 &p, const phx_long_seq &s) {
  apply_long_seq_n<1>(one(p), s);
}
__device__ __forceinline__ void apply_linmap(P6 &p, const phx_linmap &m) {
  apply_linmap_n<1>(one(p), m);
}
__device__ __forceinline__ void apply_program(P6 &p, const phx_turn_program &g) {
  apply_program_n<1>(one(p), g);
}

// ---------------------------------------------------------------------------
// Wake kick application (impedances/wake_kicks.py:160-361), kicks in order.
// ---------------------------------------------------------------------------
// Kick k of slice idx is kicks[k * n_slices + idx] (the [kick][slice]
// layout of the C ABI); the table is small and stays in the caches.
__device__ __forceinline__ void apply_wake_kicks(P6 &p, int32_t idx, int n_slices,
                                                 const phx_wake_kick *kd, int n_kicks,
                                                 const double *__restrict__ kicks) {
  if (idx < 0 || idx >= n_slices) return;
  for (int k = 0; k < n_kicks; ++k) {
    const phx_wake_kick &d = kd[k];
    double v = kicks[(size_t)k * n_slices + idx];
    if (d.multiply == 0) v = v * p.x;
    else if (d.multiply == 2) v = v * p.y;
    if (d.plane == PHX_PLANE_XP) p.xp = p.xp + v;
    else if (d.plane == PHX_PLANE_YP) p.yp = p.yp + v;
    else p.dp = p.dp + v;
  }
}

// The kick step for a known kick set (PHX_KICKS_*).
template <int KS>
__device__ __forceinline__ void apply_kick_set(P6 &p, int32_t idx, int n_slices,
                                               const phx_wake_kick *kd, int n_kicks,
                                               const double *__restrict__ kicks) {
  if constexpr (KS == PHX_KICKS_DXDY) {
    if (idx < 0 || idx >= n_slices) return;
    p.xp = p.xp + kicks[idx];
    p.yp = p.yp + kicks[(size_t)n_slices + idx];
  } else if constexpr (KS == PHX_KICKS_PLATES) {
    if (idx < 0 || idx >= n_slices) return;
    p.xp = p.xp + kicks[idx];
    p.xp = p.xp + kicks[(size_t)n_slices + idx] * p.x;
    p.yp = p.yp + kicks[(size_t)2 * n_slices + idx];
    p.yp = p.yp + kicks[(size_t)3 * n_slices + idx] * p.y;
  } else {
    apply_wake_kicks(p, idx, n_slices, kd, n_kicks, kicks);
  }
}

// ---------------------------------------------------------------------------
// Deterministic reductions.  Within a block: each wave combines its 64 lanes
// by data-parallel-primitive moves (row shifts by 1, 2, 4, 8, then the rows),
// 18 vector instructions per slot and no barrier, and one thread per slot
// then combines the waves in order.  (Through LDS, each slot's 256 values
// read by 16 threads, took three barriers: 2.2 us of the 22 us pass at 1e6
// macroparticles.)  Across chunks: each thread folds a fixed stride of chunks
// in increasing order, then the same block reduction.  For a given particle
// count the association order is fixed, so results are bit-reproducible, and
// a slot's result does not depend on which other slots are reduced with it.
// The operation of slot i is min if bit i of MINM is set, max if bit i of
// MAXM is set, else sum.
// ---------------------------------------------------------------------------
template <unsigned long long MINM, unsigned long long MAXM>
__device__ __forceinline__ double red_slot(int i, double a, double b) {
  if ((MINM >> i) & 1ULL) return fmin(a, b);
  if ((MAXM >> i) & 1ULL) return fmax(a, b);
  return a + b;
}

template <unsigned long long MINM, unsigned long long MAXM>
__device__ __forceinline__ double red_ident(int i) {
  if ((MINM >> i) & 1ULL) return INFINITY;
  if ((MAXM >> i) & 1ULL) return -INFINITY;
  return 0.0;
}

// The value of v in the lane that the DPP control names, `old` where there is
// none (a row's first lanes; rows outside ROWS).
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_move(double old, double v) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(v), CTRL, ROWS,
                                             0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(v), CTRL, ROWS,
                                             0xf, false);
  return __hiloint2double(hi, lo);
}

// Slot i's values of the wave's 64 lanes combined, in lane 63.
template <unsigned long long MINM, unsigned long long MAXM>
__device__ __forceinline__ double wave_reduce(int i, double v) {
  const double id = red_ident<MINM, MAXM>(i);
  v = red_slot<MINM, MAXM>(i, v, dpp_move<0x111, 0xf>(id, v));  // row_shr:1
  v = red_slot<MINM, MAXM>(i, v, dpp_move<0x112, 0xf>(id, v));  // row_shr:2
  v = red_slot<MINM, MAXM>(i, v, dpp_move<0x114, 0xf>(id, v));  // row_shr:4
  v = red_slot<MINM, MAXM>(i, v, dpp_move<0x118, 0xf>(id, v));  // row_shr:8
  v = red_slot<MINM, MAXM>(i, v, dpp_move<0x142, 0xa>(id, v));  // row_bcast:15
  v = red_slot<MINM, MAXM>(i, v, dpp_move<0x143, 0xc>(id, v));  // row_bcast:31
  return v;
}

// LDS doubles needed by block_reduce_slots for NV slots.
#define BR_LDS(NV) ((NV) * (PHX_BLOCK / PHX_WAVE))

// Block-reduce NV slots held by PHX_BLOCK threads of the block, t their index
// among them (a block of several such groups reduces each in lds of its own;
// every thread of the block calls it).  Thread t < NV gets the result of slot
// t as the return value (other threads: 0).  Slot t's operation is that of bit
// OFF + t of the masks.  lds: __shared__ double[BR_LDS(NV)].
template <int NV, unsigned long long MINM, unsigned long long MAXM, int OFF = 0>
__device__ __forceinline__ double block_reduce_slots_at(const double (&v)[NV], double *lds,
                                                        const int t) {
  constexpr int NW = PHX_BLOCK / PHX_WAVE;
  static_assert(NV <= PHX_BLOCK, "one thread per slot");
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const double r = wave_reduce<MINM, MAXM>(OFF + i, v[i]);
    if (t % PHX_WAVE == PHX_WAVE - 1) lds[(t / PHX_WAVE) * NV + i] = r;
  }
  lds_sync();
  double out = 0.0;
  if (t < NV) {
    out = lds[t];
#pragma unroll
    for (int w = 1; w < NW; ++w) out = red_slot<MINM, MAXM>(OFF + t, out, lds[w * NV + t]);
  }
  lds_sync();
  return out;
}

template <int NV, unsigned long long MINM, unsigned long long MAXM, int OFF = 0>
__device__ __forceinline__ double block_reduce_slots(const double (&v)[NV], double *lds) {
  return block_reduce_slots_at<NV, MINM, MAXM, OFF>(v, lds, threadIdx.x);
}

// Reduce per-chunk partials part[c*NV + i] over c < n_chunks into res[i]
// (__shared__, valid on all threads after return).  Called by one block.
// Fold of the per-block partials of a reducing pass, stored slot-major:
// slot i of block c is part[i * nc + c].  One wave folds one slot: lane l
// combines the partials l, l + 64, l + 128, ... in increasing order, then
// the 64 lane values combine in a fixed butterfly (exchange distance 32,
// 16, ..., 1; the operations are commutative, so every lane ends with the
// same value).  The order depends on nc only, not on the block size, so
// every fold of the same partials gives the same bits.  The waves of the
// block take slots i0 + w, i0 + w + W, ...; res[i] receives slot i.  Ends
// with a barrier.  SKIP >= 0: slot SKIP - 1 is left out (the next slot takes
// its place, so i1 - i0 slots are folded).
template <unsigned long long MINM, unsigned long long MAXM, int SKIP = -1>
__device__ __forceinline__ void fold_partials(const double *part, int64_t nc, int i0, int i1,
                                              double *res) {
  const int lane = threadIdx.x % PHX_WAVE, wv = threadIdx.x / PHX_WAVE;
  const int nw = blockDim.x / PHX_WAVE;
  for (int q = i0 + wv; q < i1; q += nw) {
    const int i = SKIP >= 0 && q >= SKIP - 1 ? q + 1 : q;
    const double *row = part + (size_t)i * nc;
    const double id = red_ident<MINM, MAXM>(i);
    double acc = id;
    // loads in batches, so that they are in flight together; padding with
    // the identity leaves the combination order unchanged
    constexpr int B = 8;
    for (int64_t c0 = lane; c0 < nc; c0 += (int64_t)B * PHX_WAVE) {
      double v[B];
#pragma unroll
      for (int k = 0; k < B; ++k) {
        const int64_t c = c0 + (int64_t)k * PHX_WAVE;
        v[k] = c < nc ? row[c] : id;
      }
#pragma unroll
      for (int k = 0; k < B; ++k) acc = red_slot<MINM, MAXM>(i, acc, v[k]);
    }
#pragma unroll
    for (int off = PHX_WAVE / 2; off > 0; off >>= 1)
      acc = red_slot<MINM, MAXM>(i, acc, __shfl_xor(acc, off));
    if (lane == 0) res[i] = acc;
  }
  lds_sync();
}

// ---------------------------------------------------------------------------
// Fixed-point accumulation of per-slice sums, in two 64-bit limbs.
// With |u| <= lim = 2^P and s = 2^(FX_HB - P): u s = h + r, h = rint(u s)
// (|h| <= 2^FX_HB), and l = rint(r 2^FX_LB), so u is kept to an absolute
// 2^(P - FX_HB - FX_LB) (2^-64 lim or finer for any bound the scale was taken
// from) and its sums are integer sums, independent of the order.
// Both limbs come from one FMA with the constant FX_MAGIC = 1.5 * 2^52, whose
// unit in the last place is 1: t = fma(u, s, FX_MAGIC) rounds u s to an
// integer that stands in t's low mantissa bits, so the 64-bit patterns of t
// are summed as they are (modulo 2^64) and bits(FX_MAGIC) times the number of
// terms is subtracted once per slice (acc_lds_store).  A value costs four
// FP64 operations (fma, subtract, fma, fma) where ldexp, llrint and 64-bit
// shifts and masks took about twenty instructions.
// The scale's P is rounded up to a multiple of 8 above twice the bound: the
// scale of a state and that of the turn before it (the fused engine's) agree
// unless the bound crosses such a power of two.
// ---------------------------------------------------------------------------
#define FX_LB 40
#define FX_HB 33
#define FX_MAGIC 6755399441055744.0  // 1.5 * 2^52
#define FX_MAGIC_BITS 0x4338000000000000ULL
#define FX_HUGE 0x1p1000  // beyond (and NaN): summed in FP64 as it is

struct FxScale {
  double s, lim, unit;  // 2^(hb - P), 2^P, and the value of h = 1: 2^(P - hb)
};

// 2^k, |k| <= 1022
__device__ __forceinline__ double fx_pow2(int k) {
  return __longlong_as_double((long long)(1023 + k) << 52);
}

// n: the largest number of terms of a sum; its h limb stays below 2^62 (FX_HB
// bits for up to 2^29 terms).
__device__ __forceinline__ FxScale fx_scale(double bound, int64_t n) {
  int P = 0;
  if (bound > 0.0 && bound < FX_HUGE) {
    // frexp's exponent is ilogb + 1; rounded up to a multiple of 8
    P = (__builtin_amdgcn_frexp_exp(bound) + 1 + 7) & ~7;
    P = P < -944 ? -944 : P;
  }
  int hb = FX_HB;
  if (n >> 29) hb -= 64 - __clzll((unsigned long long)(n >> 29));
  return FxScale{fx_pow2(hb - P), fx_pow2(P), fx_pow2(P - hb)};
}

// Sum of the limbs and of the out-of-range parts `over` (fallback sums:
// multiples of lim, exact in FP64, unless a term was not finite), as a
// correctly rounded double.
__device__ __forceinline__ double fx_value(unsigned long long hi_sum, unsigned long long lo_sum,
                                           double over, const FxScale &f) {
  long long h = (long long)hi_sum + ((long long)lo_sum >> FX_LB);
  const double oh = over * f.s;  // in units of h
  const bool in = fabs(oh) < 0x1p61;
  if (in) h += (long long)oh;
  const double a = (double)h;  // |h| may exceed 53 bits: keep the remainder
  const long long r = h - (long long)a;
  const double b = (double)(r * (1LL << FX_LB) + (long long)(lo_sum & ((1ULL << FX_LB) - 1ULL)));
  const double v = fma(b, 1.0 / (double)(1LL << FX_LB), a) * f.unit;
  return in ? v : v + over;
}

// The scale of the slice statistics (phx_slice_moments): every value is kept
// to the fixed quantum 2^(ilogb(bound) - 60), the integer h 2^FX_LB + l.  The
// covariance of a slice of two or three macroparticles is singular, its
// emittance the root of what the sums round to (a small number, or NaN), so
// the quantum is part of the result.  Terms up to 2^(ilogb(bound) + 2) stay
// in the limbs; h is below 2^22, its sums below 2^53 for up to 2^31 terms.
// No scale can be taken from a bound of zero, below 2^-1000 or beyond FX_HUGE
// (an infinity among the values): fx_scale's then, as its sums.
__device__ __forceinline__ bool fx_has_quantum(double bound) {
  return bound >= 0x1p-1000 && bound < FX_HUGE;
}

__device__ __forceinline__ FxScale fx_scale_quantum(double bound, int64_t n) {
  if (!fx_has_quantum(bound)) return fx_scale(bound, n);
  const int il = __builtin_amdgcn_frexp_exp(bound) - 1;
  return FxScale{fx_pow2(60 - FX_LB - il), fx_pow2(il + 2), fx_pow2(il + FX_LB - 60)};
}

// The sum of fx_scale_quantum's limbs: the integer, its upper part (from 2^32
// on) and its lower 32 bits each as a double, added and scaled.
__device__ __forceinline__ double fx_value_quantum(unsigned long long hi_sum,
                                                   unsigned long long lo_sum, double over,
                                                   double bound, const FxScale &f) {
  if (!fx_has_quantum(bound)) return fx_value(hi_sum, lo_sum, over, f);
  const long long h = (long long)hi_sum + (long long)(lo_sum >> FX_LB);
  const unsigned long long l = lo_sum & ((1ULL << FX_LB) - 1ULL);
  const long long top = h * (1LL << (FX_LB - 32)) + (long long)(l >> 32);
  const double s = (double)top * 0x1p32 + (double)(l & 0xffffffffULL);
  return (s * (1.0 / (double)(1LL << FX_LB))) * f.unit + over;
}

// ---------------------------------------------------------------------------
// Cuts of UniformBinSlicer (particles/slicing.py:395-413, 599-615) from the
// reduced z sums, and z_bins as np.arange(tail, head + 1e-7*width, width):
// buffer[0] = start, buffer[1] = start + step, delta = buffer[1] - start,
// buffer[i] = start + i*delta (NumPy's arange fill for float64).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void compute_cuts(const phx_slicer &cfg, int64_t n, double sum_z,
                                             double sum_dz, double sum_dz2, double zmin,
                                             double zmax, phx_slice_state &st) {
  double tail, head, mean_z = 0.0, sigma_z = 0.0;
  if (cfg.cuts_mode == PHX_CUTS_FIXED) {
    tail = cfg.z_cut_tail;
    head = cfg.z_cut_head;
  } else if (cfg.cuts_mode == PHX_CUTS_NSIGMA) {
    mean_z = sum_z / (double)n;
    double cov = 0.0;
    if (n >= 2) cov = (sum_dz2 - sum_dz * sum_dz / (double)n) / (double)(n - 1);
    sigma_z = sqrt(cov);
    tail = mean_z - cfg.n_sigma_z * sigma_z;
    head = mean_z + cfg.n_sigma_z * sigma_z;
  } else {
    tail = zmin;
    head = zmax;
    head = head + fabs(head) * 1e-15;
  }
  st.tail = tail;
  st.head = head;
  st.width = (head - tail) / (double)cfg.n_slices;
  st.mean_z = mean_z;
  st.sigma_z = sigma_z;
  st.n = n;
  st.n_slices = cfg.n_slices;
  st.valid = 1;
}

__device__ __forceinline__ double arange_value(double start, double step, int i) {
  if (i == 0) return start;
  const double second = start + step;
  if (i == 1) return second;
  const double delta = second - start;
  return start + (double)i * delta;
}
