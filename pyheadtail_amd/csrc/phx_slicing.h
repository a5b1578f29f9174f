// Slicing building blocks shared by the standalone slicing calls and the
// fused engine: the z-moment block that fixes the cuts, and the per-slice
// fixed-point accumulators.
#pragma once

#include "phx_device.h"

size_t phx_max_lds_bytes();
int phx_num_cus();

struct Coords6 {
  const double *c[6];
};

// ---------------------------------------------------------------------------
// z block: [0] sum z  [1] sum (z - z0)  [2] sum (z - z0)^2  [3] min z
//          [4] max z  [5..10] max |u| over finite values of x,xp,y,yp,z,dp
// ---------------------------------------------------------------------------
#define ZB_NV 11
#define ZB_MINM (1ULL << 3)
#define ZB_MAXM (0x7FULL << 4)

// The slots that the fused engine's turns use (max |u| of x and y only), and
// their place among those above.
#define ZA_NV 7
#define ZA_MINM (1ULL << 3)
#define ZA_MAXM (0x7ULL << 4)
__host__ __device__ constexpr int za_slot(int i) { return i < 6 ? i : 7; }

// Bit i of AMASK: keep max |u_i| (the others stay -inf).  Comparisons
// instead of fmin/fmax: the same results here (a NaN z or u never replaces
// the running value, which is never NaN) without the NaN quieting of the
// fmin/fmax instructions.  minmax (uniform): whether the cuts need min and
// max z (PHX_CUTS_MINMAX).
template <unsigned AMASK = 0x3Fu>
__device__ __forceinline__ void zblock_accumulate(double (&v)[ZB_NV], const P6 &p, double shift,
                                                  bool minmax) {
  const double dz = p.z - shift;
  v[0] = v[0] + p.z;
  v[1] = v[1] + dz;
  v[2] = fma(dz, dz, v[2]);
  if (minmax) {
    v[3] = p.z < v[3] ? p.z : v[3];
    v[4] = p.z > v[4] ? p.z : v[4];
  }
  const double a[6] = {fabs(p.x), fabs(p.xp), fabs(p.y), fabs(p.yp), fabs(p.z), fabs(p.dp)};
#pragma unroll
  for (int i = 0; i < 6; ++i)
    if (((AMASK >> i) & 1u) && a[i] < INFINITY && a[i] > v[5 + i]) v[5 + i] = a[i];
}

// Called by one block with the reduced z block in res (shared): writes the
// cuts into *state and the n_slices+1 bin edges into z_bins.
__device__ __forceinline__ void zblock_finalize(const double *res, const phx_slicer &cfg,
                                                int64_t n, phx_slice_state *state,
                                                double *z_bins, int turn) {
  __shared__ double sh_tail, sh_width;
  if (threadIdx.x == 0) {
    phx_slice_state st;
    compute_cuts(cfg, n, res[0], res[1], res[2], res[3], res[4], st);
    for (int i = 0; i < 6; ++i) st.absmax[i] = res[5 + i];
    st.turn = turn;
    st.pad = 0;
    *state = st;
    sh_tail = st.tail;
    sh_width = st.width;
  }
  lds_sync();
  for (int i = threadIdx.x; i <= cfg.n_slices; i += blockDim.x)
    z_bins[i] = arange_value(sh_tail, sh_width, i);
  lds_sync();
}

// ---------------------------------------------------------------------------
// Per-slice accumulation terms and fixed-point accumulators.
// ---------------------------------------------------------------------------
struct AccTerms {
  int n;
  int a[PHX_MAX_TERMS], b[PHX_MAX_TERMS];
  const double *ca[PHX_MAX_TERMS];
  const double *cb[PHX_MAX_TERMS];
};

// Per-block partial histograms (no cross-block atomics: device-scope atomics
// to one address from many blocks serialise, so each block stores its own
// histogram and a slice-parallel kernel merges them).  Stored in tiles of
// ACC_TW consecutive slices, every tile holding all H partials, so that a
// merge block (one or two tiles) reads only whole cache lines of its own:
//   cnt[tile][h][ACC_TW] (u32), hl[tile][h][t][ACC_TW] = {hi, lo} (u64
//   pairs; one 128-byte line per tile and partial for t = 2),
//   fallback[t][s] (f64, only for non-finite or out-of-scale values, added
//   with FP64 atomics).
#define ACC_TW 4

__host__ __device__ inline size_t acc_cnt_index(int H, int h, int s) {
  return ((size_t)(s / ACC_TW) * H + h) * ACC_TW + s % ACC_TW;
}
__host__ __device__ inline size_t acc_hl_index(int H, int T, int h, int i, int s) {
  return (((size_t)(s / ACC_TW) * H + h) * T + i) * ACC_TW + s % ACC_TW;
}
__host__ __device__ inline size_t acc_tiled(int S) {  // S rounded up to whole tiles
  return ((size_t)S + ACC_TW - 1) / ACC_TW * ACC_TW;
}

struct AccParts {
  unsigned int *cnt;
  ulonglong2 *hl;
  double *fallback;
  int H;  // number of partial histograms (blocks)
};

struct AccLds {
  unsigned long long *hi;
  unsigned long long *lo;
  unsigned int *counts;
};

// Standalone workspace: [256 B reserved][chunk partials][partial histograms]
inline size_t acc_partials_bytes(int64_t n) {
  return ((size_t)phx_pass_grid(n) * 64 * sizeof(double) + 255) / 256 * 256;
}

__host__ __device__ inline size_t acc_parts_bytes(int H, int S, int T) {
  const size_t St = acc_tiled(S);
  return ((size_t)H * St * 4 + 255) / 256 * 256 + (size_t)H * T * St * 16 + (size_t)T * S * 8;
}

__host__ __device__ inline AccParts acc_parts_layout(void *base, int H, int S, int T) {
  const size_t St = acc_tiled(S);
  char *p = reinterpret_cast<char *>(base);
  AccParts a;
  a.H = H;
  a.cnt = reinterpret_cast<unsigned int *>(p);
  p += ((size_t)H * St * 4 + 255) / 256 * 256;
  a.hl = reinterpret_cast<ulonglong2 *>(p);
  p += (size_t)H * T * St * 16;
  a.fallback = reinterpret_cast<double *>(p);
  return a;
}

__host__ __device__ inline size_t acc_lds_bytes(int S, int T) { return (size_t)T * S * 16 + (size_t)S * 4; }

__device__ __forceinline__ AccLds acc_lds_layout(unsigned long long *base, int S, int T) {
  AccLds L;
  L.hi = base;
  L.lo = base + (size_t)T * S;
  L.counts = reinterpret_cast<unsigned int *>(base + (size_t)2 * T * S);
  return L;
}

__device__ __forceinline__ void acc_lds_zero(const AccLds &L, int S, int T) {
  for (int i = threadIdx.x; i < T * S; i += blockDim.x) {
    L.hi[i] = 0ULL;
    L.lo[i] = 0ULL;
  }
  for (int i = threadIdx.x; i < S; i += blockDim.x) L.counts[i] = 0u;
  lds_sync();
}

// Bound of |term| from max|u| (centres are per-slice means, |c| <= max|u|).
__device__ __forceinline__ double term_bound(const AccTerms &t, int i, const double *absmax) {
  double ba = absmax[t.a[i]] * (t.ca[i] ? 2.0 : 1.0);
  double bound = ba;
  if (t.b[i] >= 0) bound = ba * (absmax[t.b[i]] * (t.cb[i] ? 2.0 : 1.0));
  return bound;
}

// Adds u to sum i of slice s (every call adds one FX_MAGIC to both limbs).  A
// value beyond the scale's range leaves its nearest multiple of lim in the
// FP64 fallback (sums of such multiples are exact, so their order does not
// matter either) and the rest in the limbs; a non-finite one goes to the
// fallback as it is.
__device__ __forceinline__ void acc_add_value(const AccLds &L, int S, int i, int s, double u,
                                              const FxScale &f, double *fallback) {
  if (__builtin_expect(!(fabs(u) <= f.lim), 0)) {
    double c = u;
    if (fabs(u) < FX_HUGE) c = rint(u / f.lim) * f.lim;
    atomicAdd(&fallback[(size_t)i * S + s], c);
    u = fabs(u) < FX_HUGE ? u - c : 0.0;
  }
  const double t = fma(u, f.s, FX_MAGIC);
  const double r = fma(u, f.s, FX_MAGIC - t);  // u s - h, exact
  const double l = fma(r, (double)(1LL << FX_LB), FX_MAGIC);
  atomicAdd(&L.hi[(size_t)i * S + s], (unsigned long long)__double_as_longlong(t));
  atomicAdd(&L.lo[(size_t)i * S + s], (unsigned long long)__double_as_longlong(l));
}

// Store this block's LDS histogram as partial number h (every entry, zeros
// included, so the merge needs no prior clearing; the slots of a last,
// partly used tile are never read): the limbs without their FX_MAGICs, the
// low one reduced to FX_LB bits with its carry added to the high one.
__device__ __forceinline__ void acc_lds_store(const AccLds &L, int S, int T, const AccParts &P,
                                              int h) {
  lds_sync();
  for (int s = threadIdx.x; s < S; s += blockDim.x) P.cnt[acc_cnt_index(P.H, h, s)] = L.counts[s];
  // consecutive threads fill one tile's record [t][ACC_TW] after the other
  const int rec = T * ACC_TW;
  const int nq = (int)(acc_tiled(S) / ACC_TW) * rec;
  for (int q = threadIdx.x; q < nq; q += blockDim.x) {
    const int r = q % rec, i = r / ACC_TW;
    const int s = (q / rec) * ACC_TW + r % ACC_TW;
    if (s < S) {
      const unsigned long long m = (unsigned long long)L.counts[s] * FX_MAGIC_BITS;
      const long long lo = (long long)(L.lo[(size_t)i * S + s] - m);
      ulonglong2 v;
      v.x = L.hi[(size_t)i * S + s] - m + (unsigned long long)(lo >> FX_LB);
      v.y = (unsigned long long)lo & ((1ULL << FX_LB) - 1ULL);
      P.hl[acc_hl_index(P.H, T, h, i, s)] = v;
    }
  }
}

// Merge of the H partial histograms for a tile of SL slices (RD_SL unless
// the caller picks another), one block of PHX_BLOCK threads: thread t takes
// slice t % SL and the partials h = t / SL, t / SL + G, ... (G = PHX_BLOCK /
// SL); the G groups of a slice are then combined by lane exchanges within
// each wave and across the waves in LDS.  The sums are integers, so the
// order of the additions does not matter.  With the tiled layout and SL a
// multiple of ACC_TW, the lanes of a wave read whole lines that no other
// block reads.  Threads 0 .. SL-1 receive the totals of their slice.
#define RD_SL 4
#define RD_G (PHX_BLOCK / RD_SL)

struct SliceTotals {
  unsigned int count;
  unsigned long long hi[PHX_MAX_TERMS], lo[PHX_MAX_TERMS];
};

// bid: the tile of SL slices (blockIdx.x of the standalone launch); NT: the
// block's threads
template <int T, int SL = RD_SL, int NT = PHX_BLOCK>
__device__ __forceinline__ bool acc_merge(const AccParts &P, int S, SliceTotals &out, int bid) {
  constexpr int NVAL = 2 * T + 1;
  constexpr int NW = NT / PHX_WAVE;
  __shared__ unsigned long long wsum[NW][NVAL][SL];
  const int sl = threadIdx.x % SL, g = threadIdx.x / SL;
  const int s = bid * SL + sl;
  // v[0] = count, v[1 + 2i] = hi of term i, v[2 + 2i] = lo of term i
  unsigned long long v[NVAL];
#pragma unroll
  for (int i = 0; i < NVAL; ++i) v[i] = 0ULL;
  if (s < S) {
    for (int h = g; h < P.H; h += (NT / SL)) {
      v[0] += P.cnt[acc_cnt_index(P.H, h, s)];
#pragma unroll
      for (int i = 0; i < T; ++i) {
        const ulonglong2 q = P.hl[acc_hl_index(P.H, T, h, i, s)];
        v[1 + 2 * i] += q.x;
        v[2 + 2 * i] += q.y;
      }
    }
  }
  // lanes of one slice differ in the bits above log2(SL)
#pragma unroll
  for (int off = SL; off < PHX_WAVE; off <<= 1)
#pragma unroll
    for (int i = 0; i < NVAL; ++i) v[i] += __shfl_xor(v[i], off);
  const int lane = threadIdx.x % PHX_WAVE, wv = threadIdx.x / PHX_WAVE;
  if (lane < SL) {
#pragma unroll
    for (int i = 0; i < NVAL; ++i) wsum[wv][i][lane] = v[i];
  }
  lds_sync();
  if (threadIdx.x >= SL || s >= S) return false;
  unsigned long long tot[NVAL];
#pragma unroll
  for (int i = 0; i < NVAL; ++i) {
    tot[i] = 0ULL;
#pragma unroll
    for (int q = 0; q < NW; ++q) tot[i] += wsum[q][i][sl];
  }
  out.count = (unsigned int)tot[0];
#pragma unroll
  for (int i = 0; i < T; ++i) {
    out.hi[i] = tot[1 + 2 * i];
    out.lo[i] = tot[2 + 2 * i];
  }
  return true;
}
