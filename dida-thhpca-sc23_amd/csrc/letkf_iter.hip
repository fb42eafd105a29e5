// The FP64 analysis, one wavefront each (k <= 64), with W = sqrt(k-1) M^(-1/2)
// by polynomial iteration on FP64 MFMA (letkf_isqrt.h) instead of an
// eigensolve:
//
//   Gram      C = Yhat Yhat^T and b = Yhat (sqrt(R^-1 rloc) dep) on FP64 MFMA
//             16x16x4 over 64-obs blocks, the rows of the next half block in
//             flight while one computes; the tiles on and below the diagonal
//             only (10 of 16 at KP = 64).
//   solve     W = sqrt(k-1) M^(-1/2), M = C + (k-1)/rho I, and wbar = M^-1 b =
//             W (W b) / (k-1) (letkf_core.F90:94-210).  An analysis whose
//             condition bound is above kIsqrtMaxKappa, or that is not finite,
//             takes the register Jacobi from M's Cholesky factor L: at these
//             condition numbers a third to a half fewer sweeps than from M
//             (2 degrees, every analysis above the limit, k = 48: 10.23 and 6.98
//             ms a sweep, k = 64: 12.15 and 8.42), the same error up to kappa
//             1e7 (that of C and b, not the solver's).  Callers that set the
//             Jacobi's own parameters take it from M (k_letkf_plain,
//             k_letkf_wave).
//   out       the transform to HBM, or the ensemble update of the analysis's
//             column, or of its cube's rows (vertical localisation), fused.
//
// No state passes between analyses, so there are no chains: the grid has one
// wavefront per analysis, dispatched by tiles of columns largest candidate
// count first (the order the selection passes use), with the columns of a
// tile on one XCD, so that the obs rows they share are read into one L2.
//
// KP = k rounded up to 16: the work goes with KP^2 (Gram) and KP^3 (solve).
#include <cstring>

#include "letkf_device.h"
#include "letkf_isqrt.h"
#include "letkf_kernels.h"
#include "letkf_wave.h"

using namespace dida;

namespace {

// LDS of one analysis.  The obs staging (Gram), the tiles below the diagonal of
// three matrices (iteration) and the Jacobi's eigenvectors are not live
// together.
template <int KP>
struct ISmem {
  static constexpr int KPJ = KP <= 32 ? 32 : 64;  // the Jacobi's padded size
  static constexpr int LDV = KPJ + 1;
  static constexpr int kZ = Sym<KP / 16>::kOff * 256;
  union {
    struct {
      double V[16 * LDV];
      int32_t ogi[2][64];
      double orr[2][64], ow[2][64];
      double ct[272];
    };
    double z[3][kZ > 0 ? kZ : 1];
  };
  double b[KPJ], f[KPJ], u[KPJ];
};

// The FP64 Gram of one analysis: M = C (zero past k) and sm.b.  DENSE: obs o of the analysis is row off + o of yb (k values), rinv and
// dep; otherwise row idx[off + o] of the binned arrays (rows of ldy values,
// zero past k).
template <int KP, bool VERT, bool DENSE, class SM>
__device__ __forceinline__ void gram_lower(const dk_batched_args& a, int64_t off, int p,
                                           double clnp, SM& sm,
                                           Sym<KP / 16>& M) {
  constexpr int NJ = KP / 16;
  const int lane = threadIdx.x, g = lane >> 4, c = lane & 15;
  const int k = a.k;
  double bacc[NJ];
#pragma unroll
  for (int I = 0; I < NJ; ++I) bacc[I] = 0.0;
  M.zero();
  const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<double*>(a.yb), (short)0, 0xFFFFFFFF, 0x00020000);
  const int row_shift = a.ldy == 64 ? 9 : 8;  // bytes of a binned row
  const double* ybd = DENSE ? a.yb + off * k : nullptr;
  auto load_rows = [&](int buf, int h, double (&raw)[8][NJ]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int gi = sm.ogi[buf][h * 32 + 4 * e + g];
#pragma unroll
      for (int I = 0; I < NJ; ++I) {
        if constexpr (DENSE) {
          const int row = I * 16 + c;
          raw[e][I] = ybd[(int64_t)gi * k + (row < k ? row : k - 1)];
        } else {
          const uint32_t o = ((uint32_t)gi << row_shift) + (uint32_t)c * 8u;
          raw[e][I] = __longlong_as_double((long long)__builtin_amdgcn_raw_buffer_load_b64(
              rows, o + (uint32_t)(I * 16 * 8), 0, 0));
        }
      }
    }
  };
  auto half = [&](int buf, int h, const double (&raw)[8][NJ]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int ol = h * 32 + 4 * e + g;
      const double rr = sm.orr[buf][ol], w = sm.ow[buf][ol];
      double f[NJ];
#pragma unroll
      for (int I = 0; I < NJ; ++I) {
        f[I] = raw[e][I] * rr;
        bacc[I] = fma(raw[e][I], w, bacc[I]);
      }
#pragma unroll
      for (int I = 0; I < NJ; ++I)
#pragma unroll
        for (int J = 0; J <= I; ++J)
          M.t[Sym<NJ>::at(I, J)] = mfma_f64_16x16x4(f[I], f[J], M.t[Sym<NJ>::at(I, J)]);
    }
  };
  if (p > 0) {
    ObsMeta m;
    m.load_index<DENSE>(a, off, p, 0);
    m.load_obs<VERT, DENSE>(a, off);
    m.store_index(sm, 0);
    m.store_weights<VERT>(sm, 0, a, clnp);
    __syncthreads();
    double rawA[8][NJ], rawB[8][NJ];
    load_rows(0, 0, rawA);
    for (int base = 0; base < p; base += 64) {
      const int buf = (base >> 6) & 1;
      ObsMeta n;
      n.load_index<DENSE>(a, off, p, base + 64);
      load_rows(buf, 1, rawB);
      __builtin_amdgcn_sched_barrier(0);
      half(buf, 0, rawA);
      n.load_obs<VERT, DENSE>(a, off);
      n.store_index(sm, buf ^ 1);
      __syncthreads();
      load_rows(buf ^ 1, 0, rawA);
      __builtin_amdgcn_sched_barrier(0);
      if (base + 32 < p) half(buf, 1, rawB);
      n.store_weights<VERT>(sm, buf ^ 1, a, clnp);
      __syncthreads();
    }
  }
  if constexpr (DENSE) {
    // rows past k repeat row k - 1
    Sym<NJ>::each([&](int I, int J, int r) {
      if (!(I * 16 + 4 * r + g < k && J * 16 + c < k)) M.t[Sym<NJ>::at(I, J)][r] = 0.0;
    });
  }
#pragma unroll
  for (int I = 0; I < NJ; ++I) bacc[I] = sum_g(bacc[I]);
  __syncthreads();
  if (g == 0) {
#pragma unroll
    for (int I = 0; I < NJ; ++I) sm.b[I * 16 + c] = I * 16 + c < k ? bacc[I] : 0.0;
    if constexpr (ISmem<KP>::KPJ > KP)
      for (int i = KP + c; i < ISmem<KP>::KPJ; i += 16) sm.b[i] = 0.0;
  }
}

// y(J*16 + c) = sum_i W(i, J*16 + c) x(i) in every lane group, x from LDS.
template <int NJ>
__device__ __forceinline__ void sym_apply(const Sym<NJ>& W, const double* z, const double* x,
                                          double (&y)[NJ]) {
  const int g = (int)threadIdx.x >> 4;
#pragma unroll
  for (int J = 0; J < NJ; ++J) y[J] = 0.0;
#pragma unroll
  for (int I = 0; I < NJ; ++I)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const double xv = x[I * 16 + 4 * r + g];
#pragma unroll
      for (int J = 0; J < NJ; ++J) y[J] = fma(elem<NJ>(W, z, I, J, r), xv, y[J]);
    }
#pragma unroll
  for (int J = 0; J < NJ; ++J) y[J] = sum_g(y[J]);
}

// W (all tiles, zero past k) and wbar (sm.u, zero past k) of M and sm.b; info
// as the entry points report it.
template <int KP>
__device__ __forceinline__ int solve(const dk_batched_args& a, ISmem<KP>& sm, Sym<KP / 16>& M,
                                     double4_t (&W)[KP / 16][KP / 16]) {
  constexpr int NJ = KP / 16;
  constexpr int KPJ = ISmem<KP>::KPJ;
  constexpr int NJJ = KPJ / 16;
  const int lane = threadIdx.x, g = lane >> 4, c = lane & 15;
  const int k = a.k;
  const double km1 = (double)(k - 1);
  publish<NJ>(M, sm.z[0]);
  double inv;
  const int steps = sym_isqrt<NJ>(M, km1 / a.rho, &inv, sm.z[0], sm.z[1], sm.z[2]);
  if (steps > 0) {
    bool bad = false;
    double y[NJ];
    sym_apply<NJ>(M, sm.z[2], sm.b, y);
    if (g == 0)
#pragma unroll
      for (int J = 0; J < NJ; ++J) sm.f[J * 16 + c] = y[J];
    __syncthreads();
    sym_apply<NJ>(M, sm.z[2], sm.f, y);
    const double ws = sqrt(km1 * inv);
#pragma unroll
    for (int J = 0; J < NJ; ++J) {
      const double w = y[J] * inv;
      bad |= !__builtin_isfinite(sm.b[J * 16 + c]) || !__builtin_isfinite(w);
      if (g == 0) sm.u[J * 16 + c] = J * 16 + c < k ? w : 0.0;
    }
#pragma unroll
    for (int I = 0; I < NJ; ++I)
#pragma unroll
      for (int J = 0; J < NJ; ++J)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          W[I][J][r] = I * 16 + 4 * r + g < k && J * 16 + c < k
                           ? elem<NJ>(M, sm.z[2], I, J, r) * ws : 0.0;
    __syncthreads();
    return __any(bad) ? -2 : steps;
  }
  Wave<KPJ, DK_GRAM_FP64> w;
  w.patB = true;
  // from M's Cholesky factor, or from M where a pivot was not positive and finite
  // (one copy of the loads up to 32 members, where two spill: the core on 4096 analyses
  // of 16 members 66.8 us, 63.7 so; two above, where the loop spills: 1 degree, k = 64,
  // 10.05 ms, 10.00 so)
  bool root = true;
  constexpr int kCopies = NJ > 2 ? 2 : 1;
#pragma unroll kCopies
  for (;;) {
#pragma unroll
    for (int J = 0; J < NJJ; ++J)
#pragma unroll
      for (int I = 0; I < NJJ; ++I)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (I < NJ && J < NJ) w.X[J][I * 4 + r] = elem<NJ>(M, sm.z[0], I, J, r);
          else w.X[J][I * 4 + r] = 0.0;
        }
    if (!root) break;
    root = w.cholesky(k, sm.f, sm.u);
    if (root) break;
  }
  __syncthreads();  // z is read before the eigenvectors overwrite it
  bool conv;
  const int sweeps = w.jacobi(a.tol, a.max_sweeps, a.predict != 0, &conv);
  double4_t T[NJJ][NJJ], wb[NJJ];
  const bool bad = eig_transform<KPJ, DK_GRAM_FP64, false>(w, sm, km1, T, wb, root);
#pragma unroll
  for (int I = 0; I < NJ; ++I)
#pragma unroll
    for (int J = 0; J < NJ; ++J) W[I][J] = T[I][J];
  if (c == 0)
#pragma unroll
    for (int I = 0; I < NJJ; ++I)
#pragma unroll
      for (int r = 0; r < 4; ++r) sm.u[I * 16 + 4 * r + g] = wb[I][r];
  __syncthreads();
  return bad ? -2 : (conv ? sweeps : -1);
}

template <int KP, int MODE, bool DENSE>
__device__ __forceinline__ void iter_analysis(const dk_batched_args& a, int64_t col, int cube,
                                              ISmem<KP>& sm) {
  constexpr int NJ = KP / 16;
  constexpr bool VERT = MODE == kModeVertical;
  const int lane = threadIdx.x, g = lane >> 4, c = lane & 15;
  const int k = a.k;
  PhaseClock clk(a.phase_clk);
  const int64_t off = a.offset ? a.offset[col] - a.base : col * (int64_t)a.max_p;
  int p = a.nobsl[col];
  p = p < 0 ? 0 : (p > a.max_p ? a.max_p : p);
  if (off < 0 || off + p > a.capacity) p = 0;
  const int64_t aid = VERT ? col * a.ncube + cube : col;
  const double clnp = VERT ? a.cube_lnp[aid] : 0.0;
  int lo = 0, hi = p;
  if (VERT && a.sel_key) vertical_range(a, off, p, clnp, lo, hi);

  Sym<NJ> M;
  gram_lower<KP, VERT, DENSE>(a, off + lo, hi - lo, clnp, sm, M);
  const double a0 = (double)(k - 1) / a.rho;
#pragma unroll
  for (int J = 0; J < NJ; ++J)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (4 * r + g == c && J * 16 + c < k) M.t[Sym<NJ>::at(J, J)][r] += a0;
  clk.mark(DK_PHASE_GRAM);
  double4_t W[NJ][NJ];
  const int info = solve<KP>(a, sm, M, W);
  clk.mark(DK_PHASE_JACOBI);
  const bool bad = info == -2;
  const double nan = __builtin_nan("");
  if (a.info && lane == 0) a.info[aid] = info;
  if (a.wbar_out && g == 0)
#pragma unroll
    for (int J = 0; J < NJ; ++J) {
      const int i = J * 16 + c;
      if (i < k) a.wbar_out[(aid - a.trans_aid0) * k + i] = bad ? nan : sm.u[i];
    }
  if constexpr (MODE == kModeTransOut) {
    // W is symmetric: element (i, e) of trans from the lane that holds W(e, i),
    // so that 16 lanes write 16 consecutive values
    double* tr = a.trans_out + (aid - a.trans_aid0) * k * k;
    double wc[NJ];
#pragma unroll
    for (int J = 0; J < NJ; ++J) wc[J] = sm.u[J * 16 + c];
#pragma unroll
    for (int I = 0; I < NJ; ++I)
#pragma unroll
      for (int J = 0; J < NJ; ++J)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int e = I * 16 + 4 * r + g, i = J * 16 + c;
          if (i < k && e < k) tr[i + (int64_t)e * k] = bad ? nan : W[I][J][r] + wc[J];
        }
    clk.mark(DK_PHASE_TRANSFORM);
    return;
  } else {
    // T(i, e) = W + wbar 1^T on the first k rows and columns
#pragma unroll
    for (int I = 0; I < NJ; ++I)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double wb = sm.u[I * 16 + 4 * r + g];
#pragma unroll
        for (int J = 0; J < NJ; ++J) W[I][J][r] = bad ? nan : W[I][J][r] + wb;
      }
    clk.mark(DK_PHASE_TRANSFORM);
    const int32_t* rmap = VERT ? a.cube_rows + a.cube_row_off[cube] : nullptr;
    const int nr = VERT ? a.cube_row_off[cube + 1] - a.cube_row_off[cube] : a.nrow;
    if (VERT && a.cube_n > 1) {
      // horizontal cube of columns: every column takes the cube's transform
      const int aj = (int)(col % a.nlat), ai = (int)(col / a.nlat);
      const int sj = aj * a.cube_n, si = ai * a.cube_n;
      const int ej = min(sj + a.cube_n - 1, a.grid_nlat - 1);
      const int ei = min(si + a.cube_n - 1, a.grid_nlon - 1);
      for (int ilon = si; ilon <= ei; ++ilon)
        for (int ilat = sj; ilat <= ej; ++ilat)
          update_rows<KP, VERT>(k, a.nrow, a.xb, a.axb, a.xa, a.axa, a.rtps != 0, a.rtps_alpha,
                                (int64_t)ilat + (int64_t)a.grid_nlat * ilon, W, rmap, nr);
    } else {
      update_rows<KP, VERT>(k, a.nrow, a.xb, a.axb, a.xa, a.axa, a.rtps != 0, a.rtps_alpha, col,
                            W, rmap, nr);
    }
    clk.mark(DK_PHASE_UPDATE);
  }
}

// Wavefronts a SIMD the registers are bounded for: one at KP = 64 and 48 (three
// matrices and more, 128 or 72 registers each), two at 32, four at 16.
constexpr int iter_waves(int kp) { return kp >= 48 ? 1 : kp == 32 ? 2 : 4; }

// Work items: groups of S = gcols * max(ncube, 1) analyses, the columns of a
// selection tile (order: tiles TJ x TI, largest first) or gcols consecutive
// analyses from aid0.  Blocks go to the XCDs round-robin, so group q takes
// blocks with the same block % 8: (q / 8) * 8 S + s * 8 + q % 8.
template <int KP, int MODE, bool DENSE>
__global__ __launch_bounds__(64, iter_waves(KP)) void k_letkf_iter(dk_batched_args a,
                                                                   dk_iter_grid gr) {
  __shared__ ISmem<KP> sm;
  const int nq = MODE == kModeVertical ? a.ncube : 1;
  const int S = gr.gcols * nq;
  const int64_t b = blockIdx.x;
  const int64_t q = gr.group0 + b / (8 * S) * 8 + b % 8;
  const int s = (int)(b / 8 % S);
  if (q >= gr.ngroups) return;
  int64_t col;
  if (gr.order) {
    const int tile = gr.order[q];
    const int ntj = (a.nlat + gr.tj - 1) / gr.tj;
    const int u = s / nq;
    const int ilat = tile % ntj * gr.tj + u % gr.tj, ilon = tile / ntj * gr.ti + u / gr.tj;
    if (ilat >= a.nlat || ilon >= a.nlon) return;
    col = (int64_t)ilat + (int64_t)a.nlat * ilon;
  } else {
    const int64_t i = q * gr.gcols + s / nq;
    if (i >= gr.nanal) return;
    col = gr.aid0 + i;
  }
  iter_analysis<KP, MODE, DENSE>(a, col, s % nq, sm);
}

template <int KP>
int launch(const dk_batched_args* a, const dk_iter_grid* g, int64_t nblocks, hipStream_t s) {
  const unsigned nb = (unsigned)nblocks;
  if (!a->idx) k_letkf_iter<KP, kModeTransOut, true><<<nb, 64, 0, s>>>(*a, *g);
  else if (a->ncube > 0) k_letkf_iter<KP, kModeVertical, false><<<nb, 64, 0, s>>>(*a, *g);
  else if (a->trans_out) k_letkf_iter<KP, kModeTransOut, false><<<nb, 64, 0, s>>>(*a, *g);
  else k_letkf_iter<KP, kModeColumn, false><<<nb, 64, 0, s>>>(*a, *g);
  return (int)hipGetLastError();
}

}  // namespace

extern "C" int dk_letkf_iter(const dk_batched_args* a, const dk_iter_grid* grid, void* stream) {
  dk_iter_grid g = *grid;
  if (g.nanal <= 0) return 0;
  if (a->k < 2 || a->k > 64 || a->gram != DK_GRAM_FP64) return (int)hipErrorInvalidValue;
  if (a->idx ? (a->ldy != 32 && a->ldy != 64) || a->ldy < a->k : !a->trans_out)
    return (int)hipErrorInvalidValue;
  if (g.order) {
    g.gcols = g.tj * g.ti;
    g.ngroups = (int64_t)((a->nlat + g.tj - 1) / g.tj) * ((a->nlon + g.ti - 1) / g.ti);
  } else {
    g.gcols = 8;
    g.ngroups = (g.nanal + 7) / 8;
  }
  const int64_t S = (int64_t)g.gcols * (a->ncube > 0 && !a->trans_out ? a->ncube : 1);
  hipStream_t s = (hipStream_t)stream;
  // at most 2^25 blocks of 64 threads a launch (a grid holds 2^32 threads)
  const int64_t span = (((int64_t)1 << 25) / (8 * S) > 0 ? ((int64_t)1 << 25) / (8 * S) : 1) * 8;
  int e = 0;
  for (g.group0 = 0; g.group0 < g.ngroups && !e; g.group0 += span) {
    const int64_t n = g.ngroups - g.group0 < span ? g.ngroups - g.group0 : span;
    const int64_t nblocks = (n + 7) / 8 * 8 * S;
    e = a->k <= 16 ? launch<16>(a, &g, nblocks, s) : a->k <= 32 ? launch<32>(a, &g, nblocks, s)
        : a->k <= 48 ? launch<48>(a, &g, nblocks, s) : launch<64>(a, &g, nblocks, s);
  }
  return e;
}

extern "C" int dk_letkf_core_iter(const dk_core_args* c, void* stream) {
  if (c->nanal <= 0) return 0;
  if (c->list) return (int)hipErrorInvalidValue;
  if (c->k > 64) return dk_letkf_iter128(c, stream);
  dk_batched_args a;
  memset(&a, 0, sizeof a);
  a.k = c->k;
  a.ldy = c->k <= 32 ? 32 : 64;
  a.idx = c->idx;
  a.gram = c->gram;
  a.max_sweeps = c->max_sweeps;
  a.max_p = c->max_p;
  a.predict = c->predict;
  a.rho = c->rho;
  a.tol = c->tol;
  a.capacity = c->capacity;
  a.offset = c->offset;
  a.nobsl = c->nobsl;
  a.rloc = c->rloc;
  a.yb = c->yb;
  a.rinv = c->rinv;
  a.dep = c->dep;
  a.info = c->info;
  a.base = c->base;
  a.trans_out = c->trans;
  a.trans_aid0 = c->aid0;
  a.wbar_out = c->wbar;
  a.phase_clk = c->phase_clk;
  dk_iter_grid g;
  memset(&g, 0, sizeof g);
  g.aid0 = c->aid0;
  g.nanal = c->nanal;
  return dk_letkf_iter(&a, &g, stream);
}
