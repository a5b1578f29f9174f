// The pass of three-launch turns (ahead_body in phx_engine.h), compiled for
// the element orders, kick sets and detuner sets of the four-launch pass.
#include "phx_ahead.h"
#include "phx_host.h"

using namespace phx_en;

namespace {

template <bool REC, int SHAPE, int KS, int DS>
__global__ void __launch_bounds__((ahead_nsub<REC, SHAPE, DS>() * PHX_BLOCK))
    k_engine_ahead(EngineArgs a, double *__restrict__ x, double *__restrict__ xp,
                   double *__restrict__ y, double *__restrict__ yp, double *__restrict__ z,
                   double *__restrict__ dp, const phx_turn_program *__restrict__ programs,
                   const double *__restrict__ kicks) {
  ahead_body<REC, SHAPE, KS, DS>(a, x, xp, y, yp, z, dp, programs, kicks, blockIdx.x, gridDim.x,
                                 a.nsub);
}

__global__ void __launch_bounds__(PHX_BLOCK) k_engine_ahead_start(EngineArgs a) {
  ahead_start_body(a, blockIdx.x);
}

__global__ void __launch_bounds__(PHX_BLOCK) k_engine_ahead_fold(EngineArgs a) {
  ahead_start_fold(a);
}

template <int SL>
__global__ void __launch_bounds__(MA_THREADS) k_engine_ahead_merge(EngineArgs a) {
  ahead_merge_body<SL>(a, blockIdx.x);
}

template <bool REC, int SHAPE, int KS, int DS>
void launch(const EngineArgs &a, hipStream_t s) {
  const phx_engine &e = a.e;
  double *const *c = e.coords;
  k_engine_ahead<REC, SHAPE, KS, DS>
      <<<dim3((unsigned)a.hblk), a.nsub * PHX_BLOCK, ahead_lds_bytes(e, a.nsub), s>>>(
          a, c[0], c[1], c[2], c[3], c[4], c[5], e.programs, e.kicks);
}

template <bool REC, int SHAPE, int KS, int DS>
AheadPass compiled() {
  return {launch<REC, SHAPE, KS, DS>, ahead_nsub<REC, SHAPE, DS>()};
}

template <bool REC, int SHAPE, int KS>
AheadPass pick_dets(int ds) {
  if constexpr (!REC && SHAPE != PHX_SHAPE_GENERIC) {
    switch (ds) {
      case PHX_DETS_NONE: return compiled<REC, SHAPE, KS, PHX_DETS_NONE>();
      case PHX_DETS_C1: return compiled<REC, SHAPE, KS, PHX_DETS_C1>();
      case PHX_DETS_C1_AMP: return compiled<REC, SHAPE, KS, PHX_DETS_C1_AMP>();
      case PHX_DETS_C1 | PHX_DETS_SMOOTH:
        return compiled<REC, SHAPE, KS, PHX_DETS_C1 | PHX_DETS_SMOOTH>();
      case PHX_DETS_C1_AMP | PHX_DETS_SMOOTH:
        return compiled<REC, SHAPE, KS, PHX_DETS_C1_AMP | PHX_DETS_SMOOTH>();
      default: break;
    }
  }
  return compiled<REC, SHAPE, KS, PHX_DETS_GENERIC>();
}

template <bool REC, int KS>
AheadPass pick_shape(int shape, int ds) {
  switch (shape) {
    case PHX_SHAPE_RF1_T | PHX_SHAPE_STATIONARY:
      if constexpr (!REC) return pick_dets<REC, PHX_SHAPE_RF1_T | PHX_SHAPE_STATIONARY, KS>(ds);
      return pick_dets<REC, PHX_SHAPE_RF1_T, KS>(ds);
    case PHX_SHAPE_RF1_T: return pick_dets<REC, PHX_SHAPE_RF1_T, KS>(ds);
    case PHX_SHAPE_RF2_T: return pick_dets<REC, PHX_SHAPE_RF2_T, KS>(ds);
    case PHX_SHAPE_T_RF1: return pick_dets<REC, PHX_SHAPE_T_RF1, KS>(ds);
    case PHX_SHAPE_T_RF2: return pick_dets<REC, PHX_SHAPE_T_RF2, KS>(ds);
    case PHX_SHAPE_LIN_T: return pick_dets<REC, PHX_SHAPE_LIN_T, KS>(ds);
    case PHX_SHAPE_T_LIN: return pick_dets<REC, PHX_SHAPE_T_LIN, KS>(ds);
    case PHX_SHAPE_T: return pick_dets<REC, PHX_SHAPE_T, KS>(ds);
    default: return pick_dets<REC, PHX_SHAPE_GENERIC, KS>(ds);
  }
}

AheadPass pick(const phx_engine &e) {
  const bool plates = e.kick_shape == PHX_KICKS_PLATES;
  if (e.record_stats)
    return plates ? pick_shape<true, PHX_KICKS_PLATES>(e.program_shape, e.det_shape)
                  : pick_shape<true, PHX_KICKS_DXDY>(e.program_shape, e.det_shape);
  return plates ? pick_shape<false, PHX_KICKS_PLATES>(e.program_shape, e.det_shape)
                : pick_shape<false, PHX_KICKS_DXDY>(e.program_shape, e.det_shape);
}

}  // namespace

bool phx_en::ahead_fits(const phx_engine &e) {
  return e.n_slices > 0 && e.n_kicks > 0 && e.sc_stages == 0 &&
         (e.kick_shape == PHX_KICKS_DXDY || e.kick_shape == PHX_KICKS_PLATES) &&
         ahead_lds_bytes(e, pick(e).nsub) <= phx_max_lds_bytes();
}

int phx_en::ahead_max_nsub(const phx_engine &e) { return pick(e).nsub; }

int phx_en::ahead_enqueue_start(const EngineArgs &a, hipStream_t s) {
  k_engine_ahead_start<<<dim3((unsigned)a.grid), PHX_BLOCK, BR_LDS(ZA_NV) * sizeof(double), s>>>(a);
  PHX_CHECK_LAUNCH("phx_engine: first turn's z sums");
  k_engine_ahead_fold<<<1, PHX_BLOCK, 0, s>>>(a);
  PHX_CHECK_LAUNCH("phx_engine: first turn's cuts");
  return PHX_OK;
}

int phx_en::ahead_enqueue_pass(const EngineArgs &a, hipStream_t s) {
  pick(a.e).launch(a, s);
  PHX_CHECK_LAUNCH("phx_engine: pass with slicing");
  return PHX_OK;
}

int phx_en::ahead_enqueue_merge(const EngineArgs &a, hipStream_t s) {
  const int S = a.e.n_slices, sl = merge_sl(S);
  const dim3 grid((unsigned)merge_blocks(S, sl, engine_has_rw(a.e), true, a.e.record_stats != 0));
  if (sl == 4) k_engine_ahead_merge<4><<<grid, MA_THREADS, 0, s>>>(a);
  else k_engine_ahead_merge<8><<<grid, MA_THREADS, 0, s>>>(a);
  PHX_CHECK_LAUNCH("phx_engine: merge");
  return PHX_OK;
}
