// Bunch and per-slice statistics, and uniform-bin slicing.
//
// Reference behaviour restated here:
//   np.mean (general/pmath.py:183), cobra_functions/stats.pyx:cov (:17-45)
//   Slicer.get_long_cuts (particles/slicing.py:395-413)
//   UniformBinSlicer.compute_sliceset_kwargs (particles/slicing.py:599-615)
//   count_macroparticles_per_slice / mean_per_slice / std_per_slice /
//   cov_per_slice / emittance_per_slice (cobra_functions/stats.pyx:192-425)
#include "phx_device.h"
#include "phx_host.h"
#include "phx_slicing.h"

// ---------------------------------------------------------------------------
// Bunch sums of K arrays: slots [sum a (K)] [sum a-a0 (K)] [pairs (P)]
// [min (K)] [max (K)] [max|a| finite (K)].
// ---------------------------------------------------------------------------
struct Arrays6 {
  const double *a[6];
};

template <int K>
struct BunchLayout {
  static constexpr int P = K * (K + 1) / 2;
  static constexpr int NV = 5 * K + P;
  static constexpr int MIN0 = 2 * K + P;
  static constexpr unsigned long long MINM = ((1ULL << K) - 1ULL) << MIN0;
  static constexpr unsigned long long MAXM = ((1ULL << (2 * K)) - 1ULL) << (MIN0 + K);
};

template <int K>
__global__ void __launch_bounds__(PHX_BLOCK)
    k_bunch_sums(Arrays6 arr, int64_t n, double *partials) {
  using L = BunchLayout<K>;
  __shared__ double lds[BR_LDS(L::NV)];
  double shift[K];
#pragma unroll
  for (int i = 0; i < K; ++i) shift[i] = arr.a[i][0];
  double v[L::NV];
#pragma unroll
  for (int i = 0; i < L::NV; ++i) v[i] = red_ident<L::MINM, L::MAXM>(i);
  const int64_t ng = phx_n_groups(n);
  for (int64_t gi = blockIdx.x; gi < ng; gi += gridDim.x) {
  const int64_t base = gi * PHX_CHUNK;
#pragma unroll
  for (int k = 0; k < PHX_PPT; ++k) {
    const int64_t j = base + (int64_t)k * PHX_BLOCK + threadIdx.x;
    if (j < n) {
      double u[K];
#pragma unroll
      for (int i = 0; i < K; ++i) u[i] = arr.a[i][j];
      int p = 0;
#pragma unroll
      for (int i = 0; i < K; ++i) {
        v[i] = v[i] + u[i];
        const double di = u[i] - shift[i];
        v[K + i] = v[K + i] + di;
#pragma unroll
        for (int jj = i; jj < K; ++jj) {
          v[2 * K + p] = v[2 * K + p] + di * (u[jj] - shift[jj]);
          ++p;
        }
        v[L::MIN0 + i] = fmin(v[L::MIN0 + i], u[i]);
        v[L::MIN0 + K + i] = fmax(v[L::MIN0 + K + i], u[i]);
        const double au = fabs(u[i]);
        if (isfinite(au)) v[L::MIN0 + 2 * K + i] = fmax(v[L::MIN0 + 2 * K + i], au);
      }
    }
  }
  }
  const double r = block_reduce_slots<L::NV, L::MINM, L::MAXM>(v, lds);
  if (threadIdx.x < L::NV) partials[(int64_t)threadIdx.x * gridDim.x + blockIdx.x] = r;
}

// One block folds the chunk partials in a fixed order: a wave per slot, whose
// loads are a chain of a few round trips, so a wave for each of the slots
// (as far as one block has them) rather than four that take turns (1e6
// macroparticles: 1, 2 and 3 arrays 5.1, 8.4 and 13.0 us before, 3.4, 3.8 and
// 5.3 us now; the cuts 8.1 and 4.4 us).
#define FIN_THREADS 1024
template <int K>
__global__ void __launch_bounds__(FIN_THREADS)
    k_bunch_sums_fin(const double *partials, int64_t n_chunks, double *out) {
  using L = BunchLayout<K>;
  __shared__ double res[L::NV];
  fold_partials<L::MINM, L::MAXM>(partials, n_chunks, 0, L::NV, res);
  if (threadIdx.x < L::NV) out[threadIdx.x] = res[threadIdx.x];
}

extern "C" int64_t phx_bunch_sums_len(int32_t k) {
  if (k < 1 || k > 6) return -1;
  return 5 * k + k * (k + 1) / 2;
}

extern "C" int phx_bunch_sums(const double *const *arrays, int32_t k, int64_t n, double *out,
                              void *ws, phx_stream_t stream) {
  if (k < 1 || k > 6) return phx::fail(PHX_E_INVALID, "phx_bunch_sums: k=%d not in 1..6", k);
  if (n < 1) return phx::fail(PHX_E_INVALID, "phx_bunch_sums: n=%lld < 1", (long long)n);
  if (!arrays || !out || !ws) return phx::fail(PHX_E_INVALID, "phx_bunch_sums: null pointer");
  Arrays6 a{};
  for (int i = 0; i < k; ++i) {
    if (!arrays[i]) return phx::fail(PHX_E_INVALID, "phx_bunch_sums: array %d is null", i);
    a.a[i] = arrays[i];
  }
  double *partials = reinterpret_cast<double *>(reinterpret_cast<char *>(ws) + phx::WsLayout::kTicketBytes);
  const int64_t nc = phx_pass_grid(n);
  const dim3 grid((unsigned)nc);
  hipStream_t s = phx::as_stream(stream);
#define PHX_BS(KK)                                                              \
  case KK:                                                                      \
    k_bunch_sums<KK><<<grid, PHX_BLOCK, 0, s>>>(a, n, partials);                \
    k_bunch_sums_fin<KK><<<1, FIN_THREADS, 0, s>>>(partials, nc, out);            \
    break;
  switch (k) {
    PHX_BS(1)
    PHX_BS(2)
    PHX_BS(3)
    PHX_BS(4)
    PHX_BS(5)
    default:
      k_bunch_sums<6><<<grid, PHX_BLOCK, 0, s>>>(a, n, partials);
      k_bunch_sums_fin<6><<<1, FIN_THREADS, 0, s>>>(partials, nc, out);
      break;
  }
#undef PHX_BS
  PHX_CHECK_LAUNCH("phx_bunch_sums");
  return PHX_OK;
}

// ---------------------------------------------------------------------------
// Slicing cuts: z sums of the current coordinates and max|u| of all six.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(PHX_BLOCK)
    k_slice_cuts(Coords6 co, int64_t n, double *partials, bool minmax) {
  __shared__ double lds[BR_LDS(ZB_NV)];
  const double shift = co.c[4][0];
  double v[ZB_NV];
#pragma unroll
  for (int i = 0; i < ZB_NV; ++i) v[i] = red_ident<ZB_MINM, ZB_MAXM>(i);
  const int64_t ng = phx_n_groups(n);
  for (int64_t gi = blockIdx.x; gi < ng; gi += gridDim.x) {
  const int64_t base = gi * PHX_CHUNK;
#pragma unroll
  for (int k = 0; k < PHX_PPT; ++k) {
    const int64_t j = base + (int64_t)k * PHX_BLOCK + threadIdx.x;
    if (j < n) {
      P6 p;
      p.x = co.c[0] ? co.c[0][j] : 0.0;
      p.xp = co.c[1] ? co.c[1][j] : 0.0;
      p.y = co.c[2] ? co.c[2][j] : 0.0;
      p.yp = co.c[3] ? co.c[3][j] : 0.0;
      p.z = co.c[4][j];
      p.dp = co.c[5] ? co.c[5][j] : 0.0;
      zblock_accumulate(v, p, shift, minmax);
    }
  }
  }
  const double r = block_reduce_slots<ZB_NV, ZB_MINM, ZB_MAXM>(v, lds);
  if (threadIdx.x < ZB_NV) partials[(int64_t)threadIdx.x * gridDim.x + blockIdx.x] = r;
}

__global__ void __launch_bounds__(FIN_THREADS)
    k_slice_cuts_fin(const double *partials, int64_t n_chunks, phx_slicer cfg, int64_t n,
                     phx_slice_state *state, double *z_bins) {
  __shared__ double res[ZB_NV];
  fold_partials<ZB_MINM, ZB_MAXM>(partials, n_chunks, 0, ZB_NV, res);
  zblock_finalize(res, cfg, n, state, z_bins, -1);
}

extern "C" int phx_slice_cuts(const double *const coords[6], int64_t n, const phx_slicer *cfg,
                              phx_slice_state *state, double *z_bins, void *ws,
                              phx_stream_t stream) {
  if (!coords || !coords[4] || !cfg || !state || !z_bins || !ws)
    return phx::fail(PHX_E_INVALID, "phx_slice_cuts: null pointer");
  if (n < 1) return phx::fail(PHX_E_INVALID, "phx_slice_cuts: n=%lld < 1", (long long)n);
  if (cfg->n_slices < 1)
    return phx::fail(PHX_E_INVALID, "phx_slice_cuts: n_slices=%d < 1", cfg->n_slices);
  if (cfg->cuts_mode < PHX_CUTS_FIXED || cfg->cuts_mode > PHX_CUTS_MINMAX)
    return phx::fail(PHX_E_INVALID, "phx_slice_cuts: bad cuts_mode %d", cfg->cuts_mode);
  Coords6 co{};
  for (int i = 0; i < 6; ++i) co.c[i] = coords[i];
  double *partials = reinterpret_cast<double *>(reinterpret_cast<char *>(ws) + phx::WsLayout::kTicketBytes);
  const int64_t nc = phx_pass_grid(n);
  hipStream_t s = phx::as_stream(stream);
  k_slice_cuts<<<dim3((unsigned)nc), PHX_BLOCK, 0, s>>>(co, n, partials,
                                                         cfg->cuts_mode == PHX_CUTS_MINMAX);
  k_slice_cuts_fin<<<1, FIN_THREADS, 0, s>>>(partials, nc, *cfg, n, state, z_bins);
  PHX_CHECK_LAUNCH("phx_slice_cuts");
  return PHX_OK;
}

// ---------------------------------------------------------------------------
// Per-slice fixed-point accumulation.
// ---------------------------------------------------------------------------
__global__ void k_fill_zero(unsigned long long *p, size_t words) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < words;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = 0ULL;
}

#define ACC_BLOCKS 256
#define ACC_THREADS 1024

// The distinct centre arrays of the terms (at most two per term), staged in
// LDS: a centred term otherwise gathers its slices' centres from global
// memory, up to two gathers of 64 lanes per term and wave.  ia, ib: the
// staged array of each term's centre_a, centre_b (-1: none).  n = 0: not
// staged, the centres do not fit beside the sums.
struct AccCentres {
  int n;
  int ia[PHX_MAX_TERMS], ib[PHX_MAX_TERMS];
  const double *c[2 * PHX_MAX_TERMS];
};

struct AccItem {
  int s;
  P6 p;
};

// used: bit i, coordinate i is loaded.
__device__ __forceinline__ AccItem acc_item(const Coords6 &co, unsigned used, int64_t j,
                                            const int32_t *idx_in, double tail, double width) {
  AccItem it;
  it.p.x = used & 1u ? co.c[0][j] : 0.0;
  it.p.xp = used & 2u ? co.c[1][j] : 0.0;
  it.p.y = used & 4u ? co.c[2][j] : 0.0;
  it.p.yp = used & 8u ? co.c[3][j] : 0.0;
  it.p.z = used & 16u ? co.c[4][j] : 0.0;
  it.p.dp = used & 32u ? co.c[5][j] : 0.0;
  it.s = idx_in ? idx_in[j] : x86_cvt_i32(slice_floor(it.p.z, tail, width));
  return it;
}

// Bound by the LDS atomics (two 64-bit adds per term and particle) where
// enough waves hide the loads, so one block fills a CU: NT threads, a particle
// each and the next one's loads in flight (the sums take most of the LDS, so
// more blocks would not fit beside it).  T is compiled in: the terms' records
// stay in scalar registers and the atomics of a particle are independent.
// FULL: the sums alone fill the LDS (8192 slices with one term, 1241 with
// eight), which leaves no room for the terms' scales (three doubles a term, too
// many for registers): they are formed where they are used.
template <int T, int NT, bool FULL>
__global__ void __launch_bounds__(NT)
    k_slice_accumulate(Coords6 co, unsigned used, int64_t n, const phx_slice_state *state, int S,
                       AccTerms terms, AccCentres cen, bool quantum, const int32_t *idx_in,
                       int32_t *idx_out, AccParts P) {
  extern __shared__ unsigned long long acc_lds[];
  const double tail = state->tail, width = state->width;
  auto scale = [&](int i) {
    const double bound = term_bound(terms, i, state->absmax);
    return quantum ? fx_scale_quantum(bound, n) : fx_scale(bound, n);
  };
  constexpr bool STAGED = T > 0 && !FULL;
  FxScale *f = nullptr;
  if constexpr (STAGED) {
    __shared__ FxScale staged[T];
    f = staged;
    if (threadIdx.x < T) f[threadIdx.x] = scale(threadIdx.x);
  }
  AccLds L = acc_lds_layout(acc_lds, S, T);
  double *ct = reinterpret_cast<double *>(acc_lds + (acc_lds_bytes(S, T) + 7) / 8);
  for (int k = 0; k < cen.n; ++k)
    for (int i = threadIdx.x; i < S; i += NT) ct[(size_t)k * S + i] = cen.c[k][i];
  acc_lds_zero(L, S, T);
  const int64_t step = (int64_t)gridDim.x * NT;
  int64_t j = (int64_t)blockIdx.x * NT + threadIdx.x;
  AccItem cur = {0, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0}}, nxt = cur;
  if (j < n) cur = acc_item(co, used, j, idx_in, tail, width);
  for (; j < n; j += step) {
    if (j + step < n) nxt = acc_item(co, used, j + step, idx_in, tail, width);
    const int s = cur.s;
    if (idx_out) idx_out[j] = s;
    if (s >= 0 && s < S) {
      atomicAdd(&L.counts[s], 1u);
#pragma unroll
      for (int i = 0; i < T; ++i) {
        double u = p6_get(cur.p, terms.a[i]);
        if (terms.ca[i]) u = u - (cen.n ? ct[(size_t)cen.ia[i] * S + s] : terms.ca[i][s]);
        if (terms.b[i] >= 0) {
          double w = p6_get(cur.p, terms.b[i]);
          if (terms.cb[i]) w = w - (cen.n ? ct[(size_t)cen.ib[i] * S + s] : terms.cb[i][s]);
          u = u * w;
        }
        if constexpr (STAGED) acc_add_value(L, S, i, s, u, f[i], P.fallback);
        else acc_add_value(L, S, i, s, u, scale(i), P.fallback);
      }
    }
    cur = nxt;
  }
  acc_lds_store(L, S, T, P, blockIdx.x);
}

// Merge the partial histograms: counts, sums and means per slice (quantum: of
// fx_scale_quantum's integers); re-zero the FP64 fallback entries.
template <int T>
__global__ void __launch_bounds__(RD_SL * RD_G)
    k_slice_acc_merge(AccParts P, int S, AccTerms terms, const phx_slice_state *state, int64_t n,
                      bool quantum, int32_t *counts, double *sums, double *means) {
  SliceTotals tot;
  if (!acc_merge<T>(P, S, tot, blockIdx.x)) return;
  const int s = blockIdx.x * RD_SL + threadIdx.x % RD_SL;
  if (counts) counts[s] = (int32_t)tot.count;
#pragma unroll
  for (int i = 0; i < T; ++i) {
    const size_t k = (size_t)i * S + s;
    const double bound = term_bound(terms, i, state->absmax);
    const double v = quantum ? fx_value_quantum(tot.hi[i], tot.lo[i], P.fallback[k], bound,
                                                fx_scale_quantum(bound, n))
                             : fx_value(tot.hi[i], tot.lo[i], P.fallback[k], fx_scale(bound, n));
    P.fallback[k] = 0.0;
    if (sums) sums[k] = v;
    if (means) means[k] = tot.count ? v / (double)tot.count : 0.0;
  }
}

static int slice_accumulate(const char *who, bool quantum, const double *const coords[6],
                            int64_t n, const phx_slice_state *state, int32_t n_slices,
                            const phx_term *terms, int32_t n_terms, const int32_t *idx_in,
                            int32_t *idx_out, int32_t *counts, double *sums, double *means,
                            void *ws, phx_stream_t stream) {
  if (!coords || (!coords[4] && !idx_in) || !state || !counts || !ws)
    return phx::fail(PHX_E_INVALID, "%s: null pointer", who);
  if (n < 1) return phx::fail(PHX_E_INVALID, "%s: n=%lld < 1", who, (long long)n);
  if (n_slices < 1) return phx::fail(PHX_E_INVALID, "%s: n_slices < 1", who);
  if (n_terms < 0 || n_terms > PHX_MAX_TERMS)
    return phx::fail(PHX_E_LIMIT, "%s: n_terms=%d not in 0..%d", who, n_terms, PHX_MAX_TERMS);
  if (n_terms > 0 && (!terms || !sums))
    return phx::fail(PHX_E_INVALID, "%s: terms/sums null", who);
  const size_t lds_bytes = acc_lds_bytes(n_slices, n_terms);
  if (lds_bytes > phx_max_lds_bytes())
    return phx::fail(PHX_E_LIMIT,
                     "%s: %d slices x %d terms need %zu B of LDS (max %zu)", who, n_slices,
                     n_terms, lds_bytes, phx_max_lds_bytes());
  AccTerms t{};
  t.n = n_terms;
  for (int i = 0; i < n_terms; ++i) {
    if (terms[i].a < 0 || terms[i].a > 5 || terms[i].b > 5)
      return phx::fail(PHX_E_INVALID, "%s: bad coordinate index in term %d", who, i);
    if (!coords[terms[i].a] || (terms[i].b >= 0 && !coords[terms[i].b]))
      return phx::fail(PHX_E_INVALID, "%s: term %d uses a null coordinate", who, i);
    t.a[i] = terms[i].a;
    t.b[i] = terms[i].b;
    t.ca[i] = terms[i].center_a;
    t.cb[i] = terms[i].center_b;
  }
  Coords6 co{};
  for (int i = 0; i < 6; ++i) co.c[i] = coords[i];
  // the coordinates that the terms read, and z where it gives the index
  unsigned used = idx_in ? 0u : 1u << 4;
  AccCentres cen{};
  auto staged = [&](const double *c) {
    int k = 0;
    while (k < cen.n && cen.c[k] != c) ++k;
    if (k == cen.n) cen.c[cen.n++] = c;
    return k;
  };
  for (int i = 0; i < n_terms; ++i) {
    used |= 1u << t.a[i] | (t.b[i] >= 0 ? 1u << t.b[i] : 0u);
    cen.ia[i] = t.ca[i] ? staged(t.ca[i]) : -1;
    cen.ib[i] = t.b[i] >= 0 && t.cb[i] ? staged(t.cb[i]) : -1;
  }
  const int32_t S = n_slices;
  size_t lds = (lds_bytes + 7) / 8 * 8 + (size_t)cen.n * S * 8;
  const size_t scales = (size_t)n_terms * sizeof(FxScale);
  if (lds + scales > phx_max_lds_bytes()) {
    cen.n = 0;
    lds = lds_bytes;
  }
  const bool full = lds + scales > phx_max_lds_bytes();
  const int64_t nc = phx::n_chunks(n);
  const int H = (int)(nc < ACC_BLOCKS ? nc : ACC_BLOCKS);
  char *base = reinterpret_cast<char *>(ws) + phx::WsLayout::kTicketBytes + acc_partials_bytes(n);
  AccParts P = acc_parts_layout(base, H, S, n_terms);
  hipStream_t s = phx::as_stream(stream);
  // the FP64 fallback region may hold data of earlier calls with other
  // sizes: clear it (the merge leaves it zero again)
  const size_t fw = (size_t)n_terms * S;
  if (fw) {
    k_fill_zero<<<dim3((unsigned)((fw + 255) / 256 < 1024 ? (fw + 255) / 256 : 1024)), 256, 0,
                  s>>>(reinterpret_cast<unsigned long long *>(P.fallback), fw);
    PHX_CHECK_LAUNCH("phx_slice_accumulate: clear");
  }
  // at most a chunk per block: small blocks spread the particles over more CUs
  const bool small = nc <= ACC_BLOCKS;
  const dim3 mg((S + RD_SL - 1) / RD_SL);
  switch (n_terms) {
#define PHX_ACC(TT)                                                                         \
  if (full)                                                                                 \
    k_slice_accumulate<TT, ACC_THREADS, true><<<dim3(H), ACC_THREADS, lds, s>>>(            \
        co, used, n, state, S, t, cen, quantum, idx_in, idx_out, P);                        \
  else if (small)                                                                           \
    k_slice_accumulate<TT, PHX_BLOCK, false><<<dim3(H), PHX_BLOCK, lds, s>>>(               \
        co, used, n, state, S, t, cen, quantum, idx_in, idx_out, P);                        \
  else                                                                                      \
    k_slice_accumulate<TT, ACC_THREADS, false><<<dim3(H), ACC_THREADS, lds, s>>>(           \
        co, used, n, state, S, t, cen, quantum, idx_in, idx_out, P);                        \
  PHX_CHECK_LAUNCH("phx_slice_accumulate");                                                 \
  k_slice_acc_merge<TT><<<mg, RD_SL * RD_G, 0, s>>>(P, S, t, state, n, quantum, counts,     \
                                                    sums, means);                           \
  break;
    case 0: PHX_ACC(0)
    case 1: PHX_ACC(1)
    case 2: PHX_ACC(2)
    case 3: PHX_ACC(3)
    case 4: PHX_ACC(4)
    case 5: PHX_ACC(5)
    case 6: PHX_ACC(6)
    case 7: PHX_ACC(7)
    default: PHX_ACC(8)
#undef PHX_ACC
  }
  PHX_CHECK_LAUNCH("phx_slice_accumulate: merge");
  return PHX_OK;
}

extern "C" int phx_slice_accumulate(const double *const coords[6], int64_t n,
                                    const phx_slice_state *state, int32_t n_slices,
                                    const phx_term *terms, int32_t n_terms,
                                    const int32_t *idx_in, int32_t *idx_out, int32_t *counts,
                                    double *sums, double *means, void *ws,
                                    phx_stream_t stream) {
  return slice_accumulate("phx_slice_accumulate", false, coords, n, state, n_slices, terms,
                          n_terms, idx_in, idx_out, counts, sums, means, ws, stream);
}

extern "C" int phx_slice_moments(const double *const coords[6], int64_t n,
                                 const phx_slice_state *state, int32_t n_slices,
                                 const phx_term *terms, int32_t n_terms, const int32_t *idx_in,
                                 int32_t *idx_out, int32_t *counts, double *sums, double *means,
                                 void *ws, phx_stream_t stream) {
  return slice_accumulate("phx_slice_moments", true, coords, n, state, n_slices, terms, n_terms,
                          idx_in, idx_out, counts, sums, means, ws, stream);
}

// ---------------------------------------------------------------------------
// Per-slice std / cov / emittance (cobra_functions/stats.pyx:258-425).
// ---------------------------------------------------------------------------
__global__ void k_slice_finalize(int kind, int S, const int32_t *counts, const double *sums,
                                 int n_sums, double f_pre, double f_mul, double f_div,
                                 double *out) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= S) return;
  const int32_t nm = counts[s];
  double r;
  if (kind == 0 || kind == 1) {
    double v = sums[s];
    if (nm > 1) v = v / (double)(nm - 1);
    r = kind == 0 ? sqrt(v) : v;
  } else {
    // emittance_per_slice: covariances are each divided by (n-1) when n > 1
    auto cov = [&](int i) {
      double v = sums[(size_t)i * S + s];
      if (nm > 1) v = v / (double)(nm - 1);
      return v;
    };
    if (nm > 1) {
      double s11 = cov(0), s12 = cov(1), s22 = cov(2);
      if (n_sums == 6) {
        const double cdp2 = cov(5);
        if (cdp2 != 0.0) {
          const double cudp = cov(3), cupdp = cov(4);
          s11 = s11 - cudp * cudp / cdp2;
          s12 = s12 - cudp * cupdp / cdp2;
          s22 = s22 - cupdp * cupdp / cdp2;
        }
      }
      r = sqrt(s11 * s22 - s12 * s12);
    } else {
      r = 0.0;
    }
  }
  out[s] = ((f_pre * r) * f_mul) / f_div;
}

extern "C" int phx_slice_finalize(int32_t kind, int32_t n_slices, const int32_t *counts,
                                  const double *sums, int32_t n_sums, double f_pre,
                                  double f_mul, double f_div, double *out,
                                  phx_stream_t stream) {
  if (!counts || !sums || !out) return phx::fail(PHX_E_INVALID, "phx_slice_finalize: null pointer");
  if (n_slices < 1) return phx::fail(PHX_E_INVALID, "phx_slice_finalize: n_slices < 1");
  if (kind < 0 || kind > 2) return phx::fail(PHX_E_INVALID, "phx_slice_finalize: bad kind %d", kind);
  if (kind == 2 && n_sums != 3 && n_sums != 6)
    return phx::fail(PHX_E_INVALID, "phx_slice_finalize: emittance needs 3 or 6 sums");
  const int threads = 256;
  k_slice_finalize<<<dim3((n_slices + threads - 1) / threads), threads, 0,
                     phx::as_stream(stream)>>>(kind, n_slices, counts, sums, n_sums, f_pre,
                                               f_mul, f_div, out);
  PHX_CHECK_LAUNCH("phx_slice_finalize");
  return PHX_OK;
}

__global__ void k_slice_times(const double *zb, int S, double beta_c, double *zc, double *t) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= S) return;
  const double c = zb[s] + 0.5 * (zb[s + 1] - zb[s]);
  if (zc) zc[s] = c;
  if (t) t[s] = c / beta_c;
}

extern "C" int phx_slice_times(const double *z_bins, int32_t n_slices, double beta_c,
                               double *z_centers, double *times, phx_stream_t stream) {
  if (!z_bins || n_slices < 1) return phx::fail(PHX_E_INVALID, "phx_slice_times: bad arguments");
  k_slice_times<<<dim3((n_slices + 255) / 256), 256, 0, phx::as_stream(stream)>>>(
      z_bins, n_slices, beta_c, z_centers, times);
  PHX_CHECK_LAUNCH("phx_slice_times");
  return PHX_OK;
}
