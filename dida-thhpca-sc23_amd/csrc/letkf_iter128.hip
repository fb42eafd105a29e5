// The FP64 analysis of 65 to 128 members, one workgroup (4 wavefronts) each,
// with W = sqrt(k-1) M^(-1/2) by the polynomial iteration of letkf_isqrt.h:
//
//   Gram      C = Yhat Yhat^T and b = Yhat (sqrt(R^-1 rloc) dep) on FP64 MFMA
//             16x16x4, stages of 16 obs, the rows of the next stage in flight.
//   solve     every iterate is symmetric: its NT (NT + 1) / 2 tiles on and below
//             the diagonal (NT = k / 16 rounded up) are dealt to the wavefronts in
//             equal runs of the row-major order, which hold them in registers.
//             A product reads both factors from LDS (two matrices of tiles, 147
//             KB at NT = 8), an element above the diagonal from the transposed
//             tile: a wavefront reads at most 10 operands for 9 MFMAs of 64
//             cycles, 160 of 576 LDS cycles, so the matrix units are the bound
//             (288 MFMAs a wavefront and product at NT = 8).  T, T^2, P and Z and the
//             operands of two steps fit 512 registers up to NT = 7; at NT = 8 323
//             spill (batched sweep of 80 x 160 columns, k = 112 and 113: 7.0 and 10.0
//             ms, 1.43 times for 1.47 times the MFMAs).
//   out       W and wbar = M^-1 b = W (W b) / (k-1) to HBM (letkf_core.F90:94-210).
//
// An analysis whose condition bound is above kIsqrtMaxKappa, or that is not
// finite, is marked for the register Jacobi of a second, persistent launch, from M's
// Cholesky factor (k_letkf_core_marked; in this kernel its registers and LDS would be
// everyone's).
#include <cstring>

#include "letkf_device.h"
#include "letkf_isqrt.h"
#include "letkf_kernels.h"

using namespace dida;

namespace {

// Tiles (row r[t], column c[t]) and the first tile of each wavefront.
template <int NT>
struct Deal {
  static constexpr int kTiles = NT * (NT + 1) / 2;
  int r[kTiles], c[kTiles];
  constexpr Deal() : r(), c() {
    int t = 0;
    for (int i = 0; i < NT; ++i)
      for (int j = 0; j <= i; ++j, ++t) {
        r[t] = i;
        c[t] = j;
      }
  }
  static constexpr int first(int w) {
    return w * (kTiles / 4) + (w < kTiles % 4 ? w : kTiles % 4);
  }
  constexpr bool row_of(int w, int x) const {
    for (int t = first(w); t < first(w + 1); ++t)
      if (r[t] == x) return true;
    return false;
  }
  constexpr bool col_of(int w, int x) const {
    for (int t = first(w); t < first(w + 1); ++t)
      if (c[t] == x) return true;
    return false;
  }
};

template <int NT>
struct Smem {
  static constexpr int kTiles = Deal<NT>::kTiles;
  double z[2][kTiles * 256];
  double b[128], x[128], part[256], red[4];
};

constexpr int tile_of(int i, int j) { return i * (i + 1) / 2 + j; }

// Element (i, j) of the matrix whose tiles are at z.
__device__ __forceinline__ double z_elem(const double* z, int i, int j) {
  const int I = i >> 4, J = j >> 4;
  return I >= J ? z[tile_of(I, J) * 256 + tile_at(i & 15, j & 15)]
                : z[tile_of(J, I) * 256 + tile_at(j & 15, i & 15)];
}

// The part of an analysis that wavefront W runs on its tiles.
template <int NT, int W>
struct Part {
  static constexpr Deal<NT> kDeal{};
  static constexpr int kFirst = Deal<NT>::first(W);
  static constexpr int kCount = Deal<NT>::first(W + 1) - kFirst;
  typedef double4_t Tiles[kCount];

  static constexpr unsigned mask(bool row) {
    unsigned m = 0;
    for (int x = 0; x < NT; ++x)
      if (row ? kDeal.row_of(W, x) : kDeal.col_of(W, x)) m |= 1u << x;
    return m;
  }
  static constexpr unsigned kRows = mask(true), kCols = mask(false);
  // tile rows of Yhat read by the Gram; b of tile rows T % 4 == W
  static constexpr unsigned kNeed = kRows | kCols | (0x11u << W & ((1u << NT) - 1));

  static __device__ __forceinline__ int tr(int t) { return kDeal.r[kFirst + t]; }
  static __device__ __forceinline__ int tc(int t) { return kDeal.c[kFirst + t]; }

  static __device__ __forceinline__ void zero(Tiles& D) {
#pragma unroll
    for (int t = 0; t < kCount; ++t) D[t] = double4_t{0.0, 0.0, 0.0, 0.0};
  }

  // D += A B, the factors' tiles at za and zb (SAME: the same matrix).  The
  // operands of a step of 4 are read while the step before multiplies, no
  // earlier: left to itself the compiler reads a dozen steps ahead and spills.
  template <bool SAME>
  static __device__ __forceinline__ void product(Tiles& D, const double* za, const double* zb) {
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    // (opaque, or the addresses of all tiles are formed once and kept: 600 spills)
    int dir[4], tra[4], o0 = 0;
    asm volatile("" : "+v"(o0));
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      dir[r] = o0 + tile_at(4 * r + g, c);
      tra[r] = o0 + tile_at(c, 4 * r + g);
    }
    double av[2][NT], bv[2][NT];
    auto load = [&](int s, double (&x)[NT], double (&y)[NT]) {
      const int K = s >> 2, r = s & 3;
#pragma unroll
      for (int X = 0; X < NT; ++X) {
        const int o = K >= X ? tile_of(K, X) * 256 + dir[r] : tile_of(X, K) * 256 + tra[r];
        if (kRows >> X & 1) x[X] = za[o];
        if (kCols >> X & 1) y[X] = SAME && (kRows >> X & 1) ? x[X] : zb[o];
      }
    };
    load(0, av[0], bv[0]);
#pragma unroll
    for (int s = 0; s < 4 * NT; ++s) {
      const int u = s & 1;
      if (s + 1 < 4 * NT) load(s + 1, av[u ^ 1], bv[u ^ 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < kCount; ++t)
        D[t] = mfma_f64_16x16x4(av[u][tr(t)], bv[u][tc(t)], D[t]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }

  static __device__ __forceinline__ void put(const Tiles& X, double* z) {
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
#pragma unroll
    for (int t = 0; t < kCount; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) z[(kFirst + t) * 256 + tile_at(4 * r + g, c)] = X[t][r];
  }
  // X (and Y) to z (and y), once every wavefront has read what was there
  static __device__ __forceinline__ void publish(const Tiles& X, double* z) {
    __syncthreads();
    put(X, z);
    __syncthreads();
  }
  static __device__ __forceinline__ void publish(const Tiles& X, double* z, const Tiles& Y,
                                                 double* y) {
    __syncthreads();
    put(X, z);
    put(Y, y);
    __syncthreads();
  }

  static __device__ __forceinline__ void gram(const dk_core_args& a, int64_t off, int p,
                                              Smem<NT>& sm, Tiles& M) {
    constexpr int U = 4;
    const int lane = threadIdx.x & 63, r16 = lane & 15, q4 = lane >> 4;
    const int k = a.k;
    zero(M);
    double bacc[NT];
#pragma unroll
    for (int T = 0; T < NT; ++T) bacc[T] = 0.0;
    const int nst = (p + 4 * U - 1) / (4 * U);
    int gn[U];
    auto load_idx = [&](int st) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int o = st * 4 * U + 4 * u + q4;
        const int oc = o < p ? o : 0;
        gn[u] = a.idx ? a.idx[off + oc] : (int)(off + oc);
      }
    };
    // rows T*16 + r16 (clamped to k - 1, masked later) and R^-1 rloc, d
    auto load_rows = [&](int st, double (&f)[U][NT], double (&rr)[U], double (&sd)[U]) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int o = st * 4 * U + 4 * u + q4;
        const bool ok = o < p;
        const int64_t gi = gn[u];
        const double* y = a.yb + gi * k;
#pragma unroll
        for (int T = 0; T < NT; ++T)
          if (kNeed >> T & 1) {
            const int row = T * 16 + r16;
            f[u][T] = y[T < NT - 1 || row < k ? row : k - 1];
          }
        rr[u] = ok ? (double)a.rinv[gi] * a.rloc[off + (ok ? o : 0)] : 0.0;
        sd[u] = a.dep[gi];
      }
    };
    auto compute = [&](double (&f)[U][NT], const double (&rr)[U], const double (&sd)[U]) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const double r = sqrt(rr[u]), d = r * sd[u];
#pragma unroll
        for (int T = 0; T < NT; ++T)
          if (kNeed >> T & 1)
            f[u][T] = T < NT - 1 || T * 16 + r16 < k ? f[u][T] * r : 0.0;
#pragma unroll
        for (int t = 0; t < kCount; ++t)
          M[t] = mfma_f64_16x16x4(f[u][tr(t)], f[u][tc(t)], M[t]);
#pragma unroll
        for (int T = W; T < NT; T += 4) bacc[T] = fma(f[u][T], d, bacc[T]);
      }
    };
    if (nst > 0) {
      double fA[U][NT], fB[U][NT], rA[U], rB[U], sA[U], sB[U];
      load_idx(0);
      load_rows(0, fA, rA, sA);
      if (nst > 1) load_idx(1);
      for (int st = 0; st < nst; st += 2) {
        if (st + 1 < nst) load_rows(st + 1, fB, rB, sB);
        if (st + 2 < nst) load_idx(st + 2);
        __builtin_amdgcn_sched_barrier(0);
        compute(fA, rA, sA);
        if (st + 1 >= nst) break;
        if (st + 2 < nst) load_rows(st + 2, fA, rA, sA);
        if (st + 3 < nst) load_idx(st + 3);
        __builtin_amdgcn_sched_barrier(0);
        compute(fB, rB, sB);
      }
    }
#pragma unroll
    for (int T = W; T < NT; T += 4) {
      bacc[T] += shfl_xor_d(bacc[T], 16);
      bacc[T] += shfl_xor_d(bacc[T], 32);
      if (q4 == 0) sm.b[T * 16 + r16] = bacc[T];
    }
  }

  // Bound of M's condition number from M^2 (T2, at z; a0 the smallest eigenvalue
  // of M at least), the same in every thread; NaN where M holds one.
  static __device__ __forceinline__ double kappa(const Tiles& T2, const double* z, double a0,
                                                 Smem<NT>& sm) {
    const int tid = threadIdx.x, lane = tid & 63, j = tid & 127;
    double s = 0.0;
    if (j < NT * 16)
      for (int i = (tid >> 7) * (NT * 8), e = i + NT * 8; i < e; ++i) s += fabs(z_elem(z, i, j));
    sm.part[tid] = s;
    double f = 0.0;
#pragma unroll
    for (int t = 0; t < kCount; ++t) {
      const double q = (T2[t][0] * T2[t][0] + T2[t][1] * T2[t][1]) +
                       (T2[t][2] * T2[t][2] + T2[t][3] * T2[t][3]);
      f += tr(t) == tc(t) ? q : 2.0 * q;
    }
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) f += shfl_xor_d(f, m);
    if (lane == 0) sm.red[W] = f;
    __syncthreads();
    const double u = sm.part[lane] + sm.part[lane + 128];
    const double v = sm.part[lane + 64] + sm.part[lane + 192];
    double m = v > u || v != v ? v : u;
#pragma unroll
    for (int x = 1; x < 64; x <<= 1) {
      const double o = shfl_xor_d(m, x);
      m = o > m || o != o ? o : m;
    }
    const double n1 = sqrt(m);
    const double n4 = sqrt(sqrt((sm.red[0] + sm.red[1]) + (sm.red[2] + sm.red[3])));
    // (below 1e-70 the trace of M^4 could underflow)
    return (n4 < n1 && a0 > 1e-70 ? n4 : n1) / a0 * (1.0 + 1e-12);
  }

  // Gram and iteration: Z at sm.z[0] with M^(-1/2) = sqrt(*inv) Z, and the steps
  // taken; or 0, for the Jacobi.
  static __device__ __forceinline__ int run(const dk_core_args& a, int64_t off, int p,
                                            Smem<NT>& sm, double* inv, PhaseClock& clk) {
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
    const int k = a.k;
    const double a0 = (double)(k - 1) / a.rho;
    Tiles T;
    gram(a, off, p, sm, T);
#pragma unroll
    for (int t = 0; t < kCount; ++t)
      if (tr(t) == tc(t))
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (4 * r + g == c && tc(t) * 16 + c < k) T[t][r] += a0;
    clk.mark(DK_PHASE_GRAM);
    double* z0 = sm.z[0];
    double* z1 = sm.z[1];
    Tiles T2;
    publish(T, z0);
    zero(T2);
    product<true>(T2, z0, z0);
    publish(T2, z1);
    const double kap = kappa(T2, z1, a0, sm);
    // (a0 outside this range could lose M^2 to underflow)
    // (the same in every thread, and scalar: barriers follow)
    const bool steps_ok = kap <= kIsqrtMaxKappa && a0 > 1e-100 && a0 < 1e100;
    if (!__builtin_amdgcn_readfirstlane(steps_ok)) return 0;
    int cls = 0;
#pragma unroll
    for (int i = 0; i < kIsqrtPlans - 1; ++i) cls += kap > kIsqrtPlan[i].kappa;
    const IsqrtPlan& plan = kIsqrtPlan[__builtin_amdgcn_readfirstlane(cls)];
    const double sc = 1.0 / (a0 * kap);
    *inv = sc;
#pragma unroll
    for (int t = 0; t < kCount; ++t) {
      T[t] *= sc;
      T2[t] *= sc * sc;
    }
    const int n = plan.nstep;
    Tiles Z;
    for (int s = 0;; ++s) {
      const int nc = plan.step[s].nc;
      const double c0 = plan.step[s].c[0], c1 = plan.step[s].c[1], c2 = plan.step[s].c[2],
                   c3 = plan.step[s].c[3], c4 = plan.step[s].c[4];
      auto diag = [&](int t, int r, double v) {
        return tr(t) == tc(t) && 4 * r + g == c ? v : 0.0;
      };
      Tiles P;
      if (nc == 5) {
        // T^2 and c2 I + c3 T + c4 T^2
        __syncthreads();
        put(T2, z1);
#pragma unroll
        for (int t = 0; t < kCount; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            z0[(kFirst + t) * 256 + tile_at(4 * r + g, c)] =
                fma(c4, T2[t][r], fma(c3, T[t][r], diag(t, r, c2)));
        __syncthreads();
#pragma unroll
        for (int t = 0; t < kCount; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) P[t][r] = fma(c1, T[t][r], diag(t, r, c0));
        product<false>(P, z1, z0);
      } else {
        const double c2m = nc == 3 ? c2 : 0.0;
#pragma unroll
        for (int t = 0; t < kCount; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            P[t][r] = fma(c2m, nc == 3 ? T2[t][r] : 0.0, fma(c1, T[t][r], diag(t, r, c0)));
      }
      const bool last = s + 1 == n;
      // Z <- Z P (Z = P after the first step), T <- P (T P)
      if (last) {
        publish(P, z1, Z, z0);
        zero(Z);
        product<false>(Z, z0, z1);
        break;
      }
      publish(P, z1, T, z0);
      zero(T);
      product<false>(T, z0, z1);
      if (s == 0) {
#pragma unroll
        for (int t = 0; t < kCount; ++t) Z[t] = P[t];
      } else {
        publish(Z, z0);
        zero(Z);
        product<false>(Z, z0, z1);
      }
      publish(T, z0);
      zero(T);
      product<false>(T, z1, z0);
      if (plan.step[s + 1].nc > 2) {
        publish(T, z0);
        zero(T2);
        product<true>(T2, z0, z0);
      }
    }
    publish(Z, z0);
    return n;
  }
};

template <int NT>
__global__ __launch_bounds__(256) void k_letkf_iter128(dk_core_args a) {
  __shared__ Smem<NT> sm;
  // groups of 8 consecutive analyses on one XCD (blocks go to the XCDs round
  // robin), so that the obs rows they share are read into one L2
  const int b = blockIdx.x;
  const int o = b / 64 * 64 + b % 8 * 8 + b / 8 % 8;
  if (o >= a.nanal) return;
  const int aid = a.aid0 + o;
  // (scalar: the barriers of the wavefronts' parts stand in branches that it decides)
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int k = a.k;
  PhaseClock clk(a.phase_clk);
  const int64_t off = a.offset ? a.offset[aid] - a.base : aid * (int64_t)a.max_p;
  int p = a.nobsl[aid];
  p = p < 0 ? 0 : (p > a.max_p ? a.max_p : p);
  if (off < 0 || off + p > a.capacity) p = 0;
  int steps;
  double inv = 0.0;
  switch (wave) {
    case 0: steps = Part<NT, 0>::run(a, off, p, sm, &inv, clk); break;
    case 1: steps = Part<NT, 1>::run(a, off, p, sm, &inv, clk); break;
    case 2: steps = Part<NT, 2>::run(a, off, p, sm, &inv, clk); break;
    default: steps = Part<NT, 3>::run(a, off, p, sm, &inv, clk); break;
  }
  __syncthreads();
  const int64_t slot = (int64_t)aid - a.aid0;
  double* trans = a.trans + slot * k * k;
  if (steps == 0) {
    if (tid == 0) trans[0] = __longlong_as_double(kMarkBits);
    return;
  }
  clk.mark(DK_PHASE_JACOBI);
  // wbar = inv Z (Z b), half the sum of a column in each half of the workgroup
  const double* z = sm.z[0];
  const int j = tid & 127, i0 = (tid >> 7) * (NT * 8);
  const double km1 = (double)(k - 1);
  int nonfinite = 0;
  for (int pass = 0; pass < 2; ++pass) {
    const double* x = pass ? sm.x : sm.b;
    double s = 0.0;
    if (j < NT * 16)
      for (int i = i0; i < i0 + NT * 8; ++i) s = fma(z_elem(z, i, j), x[i], s);
    sm.part[tid] = s;
    __syncthreads();
    if (tid < NT * 16) {
      const double y = (sm.part[tid] + sm.part[tid + 128]) * (pass ? inv : 1.0);
      nonfinite |= !__builtin_isfinite(y) || !__builtin_isfinite(sm.b[tid]);
      sm.x[tid] = y;
    }
    __syncthreads();
  }
  const bool bad = __syncthreads_or(nonfinite) != 0;
  const double nan = __builtin_nan("");
  const double ws = sqrt(km1 * inv);
  // trans(i, e) = W(i, e) + wbar(i): from tile (I, J) its elements as (e, i) and,
  // off the diagonal, transposed as (i, e), 16 lanes along i
  for (int t = wave, I = 0, J = 0; t < Smem<NT>::kTiles; t += 4) {
    while (tile_of(I + 1, 0) <= t) ++I;
    J = t - tile_of(I, 0);
    const double wj = sm.x[J * 16 + c], wi = sm.x[I * 16 + c];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int e = I * 16 + 4 * r + g, i = J * 16 + c;
      if (e < k && i < k)
        trans[i + (int64_t)e * k] =
            bad ? nan : fma(ws, z[t * 256 + tile_at(4 * r + g, c)], wj);
      if (I != J) {
        const int e2 = J * 16 + 4 * r + g, i2 = I * 16 + c;
        if (e2 < k && i2 < k)
          trans[i2 + (int64_t)e2 * k] =
              bad ? nan : fma(ws, z[t * 256 + tile_at(c, 4 * r + g)], wi);
      }
    }
  }
  if (a.wbar)
    for (int i = tid; i < k; i += 256) a.wbar[slot * k + i] = bad ? nan : sm.x[i];
  if (a.info && tid == 0) a.info[aid] = bad ? -2 : steps;
  clk.mark(DK_PHASE_TRANSFORM);
}

}  // namespace

extern "C" int dk_letkf_iter128(const dk_core_args* a, void* stream) {
  if (a->nanal <= 0) return 0;
  if (a->k <= 64 || a->k > 128 || a->gram != DK_GRAM_FP64 || a->list)
    return (int)hipErrorInvalidValue;
  hipStream_t s = (hipStream_t)stream;
  const unsigned nb = (unsigned)(((int64_t)a->nanal + 63) / 64 * 64);
  switch ((a->k + 15) / 16) {
    case 5: k_letkf_iter128<5><<<nb, 256, 0, s>>>(*a); break;
    case 6: k_letkf_iter128<6><<<nb, 256, 0, s>>>(*a); break;
    case 7: k_letkf_iter128<7><<<nb, 256, 0, s>>>(*a); break;
    default: k_letkf_iter128<8><<<nb, 256, 0, s>>>(*a); break;
  }
  const int e = (int)hipGetLastError();
  return e ? e : dk_letkf_core_marked(a, stream);
}
