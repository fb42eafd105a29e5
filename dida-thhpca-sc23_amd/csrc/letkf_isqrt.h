// M^(-1/2) of a symmetric positive definite matrix by polynomial iteration,
// one wavefront, every product on FP64 MFMA.
//
// With T = M / s, its eigenvalues t in [1/kappa, 1] and Z = I, a step takes a
// polynomial p with t p(t)^2 closer to 1 over the whole interval,
//   P = p(T),  Z <- Z P,  T <- P (T P),
// until T = I and Z = T_0^(-1/2).  p is the minimax one: x p(x^2), an odd
// polynomial of degree 3, 5 or 9, differs from 1 by at most e over
// [sqrt(t_min), sqrt(t_max)], which leaves t in [(1 - e)^2, (1 + e)^2] for the
// next step (a composition of best polynomials, the polynomial counterpart of
// the iterations of Nakatsukasa and Freund, SIAM Review 58, 2016).  Degree 9
// costs two products for P (T^2, and T^2 (c2 + c3 T + c4 T^2)), degree 5 one,
// degree 3 none; kIsqrtPlan holds, per bound on kappa, the sequence with the
// fewest products that ends with e below 2^-56.
//
// kappa: the smallest eigenvalue of M = C + a0 I is at least a0 (C has no
// negative one), the largest at most sqrt(|| M^2 ||_1) and (trace M^4)^(1/4),
// from one product that the first step needs anyway.  The iteration's own error
// grows with kappa (relative error in the 2-norm against 40-digit arithmetic, 64 x 64: 7e-16 at
// kappa 10, 3e-15 at 100, 3e-14 at 1300, 6e-14 at 3200; Jacobi with tolerance
// 1e-13: 2e-13 throughout) and would pass the Jacobi's at some 10 000; above
// kIsqrtMaxKappa an analysis takes the Jacobi (4096 analyses of 64 members, 512 obs:
// 0.67 ms below the limit, in the classes of most products, and 2.65 ms above it;
// 1024 of 128 members: 1.35 and 8.9 ms), so the line lies as high as the error allows.
// T <- P (T P) has the smallest
// error of the forms tried; (T P) P has three times its error, and the
// coupled form (T = Z Y, Y <- Y P) is unstable (1e-12 at 1000, 1e-10 at
// 10 000).
//
// Why not the Jacobi: a cold start takes 9 to 12 sweeps, each a chain of KP - 1
// rounds of dot product, angle and rotation, some 200 instructions a round
// at one wavefront a SIMD.  The matrices here have kappa 3 to 100 (local obs
// with a spectrum far from graded), where the iteration takes 10 to 14
// products of 160 MFMA (KP = 64) with no dependence between lanes at all.
//
// Layout: the 16 x 16 tiles on and below the diagonal in registers, element r
// of lane (g = l / 16, c = l % 16) of tile (I, J) = M(I*16 + 4r + g, J*16 + c),
// the result of mfma_f64_16x16x4.  Read as operands, tile (K, J) gives
// B(K*16 + 4r + g, J*16 + c) and, M being symmetric, tile (K, I) gives
// A(I*16 + c, K*16 + 4r + g): the lane that holds a result holds the operand.
// Where K is above, the operand is an element of the transposed tile below,
// read from LDS: every product writes its off-diagonal tiles there too (all
// iterates are polynomials in M, so every product is symmetric).  At KP = 64
// that is 80 registers a matrix instead of 128: with whole matrices in
// registers (and Z in LDS) the kernel spilled 416, each product waited on
// reloads, and a 1 degree sweep took 15.3 ms; 11.6 so, with MFMA results in VGPRs.
#pragma once

#include "letkf_device.h"

namespace dida {

struct IsqrtStep {
  int32_t nc;    // coefficients of p in powers of t: 2, 3 or 5
  double c[5];
};
struct IsqrtPlan {
  double kappa;  // bound on the condition number
  int32_t nstep;
  IsqrtStep step[4];
};
constexpr int kIsqrtPlans = 12;
constexpr double kIsqrtMaxKappa = 4096.0;
__constant__ const IsqrtPlan kIsqrtPlan[kIsqrtPlans] = {
    // kappa <= 2: 7 products
    {2.0, 2, {{5, {2.930243553402779, -5.476315927922004, 6.804957176308923, -4.408645111356129,
        1.149834324208462}},
       {5, {2.4609375, -3.28125, 2.953125, -1.40625, 0.2734375}}}},
    // kappa <= 4: 10 products
    {4.0, 3, {{5, {3.498030277570191, -8.984586211108892, 14.657674201979308, -11.973430739086151,
        3.8044301893726997}},
       {5, {2.460943478204899, -3.2812683944906493, 2.9531443142033673, -1.4062573577791324,
        0.2734379598615149}},
       {2, {1.5, -0.5, 0.0, 0.0, 0.0}}}},
    // kappa <= 8: 10 products
    {8.0, 3, {{5, {4.186885651453691, -14.403991138470987, 29.20247913077536, -28.065115912997534,
        10.093213411888534}},
       {5, {2.4611794380486876, -3.2819944477489744, 2.953906650783294, -1.4065477510512985,
        0.2734561099633896}},
       {2, {1.5, -0.5, 0.0, 0.0, 0.0}}}},
    // kappa <= 16: 11 products
    {16.0, 3, {{5, {5.021278584375493, -22.334752491456964, 53.22490909906152, -56.92392236178504,
        22.057560798676928}},
       {5, {2.46365005957486, -3.289599219932958, 2.9618892440360587, -1.4095861665820961,
        0.27364607602599444}},
       {3, {1.875, -1.25, 0.375, 0.0, 0.0}}}},
    // kappa <= 32: 12 products
    {32.0, 3, {{5, {6.015076279588356, -33.09563391458941, 88.27924312280776, -101.006001056639,
        40.912117592522165}},
       {5, {2.475707515493199, -3.3267807450883806, 3.000859458149964, -1.4243585306496422,
        0.2745712157530482}},
       {5, {2.4609375, -3.28125, 2.953125, -1.40625, 0.2734375}}}},
    // kappa <= 64: 12 products
    {64.0, 3, {{5, {7.151790066051095, -46.43556232103322, 133.54643437912654, -159.3414779246455,
        66.27153647233456}},
       {5, {2.511956657451227, -3.439207267458501, 3.1180931604483186, -1.4682175916521,
        0.27733308399620415}},
       {5, {2.4609375, -3.28125, 2.953125, -1.40625, 0.2734375}}}},
    // kappa <= 128: 14 products
    {128.0, 4, {{5, {8.37511028188687, -61.47602915983481, 185.73521630848944, -227.4782443041714,
        96.14514355278928}},
       {5, {2.5913300179202787, -3.6883481904048834, 3.3746016079858916, -1.5614741773297336,
        0.28328054202673564}},
       {3, {1.87500168727525, -1.2500018747489998, 0.37500018747494945, 0.0, 0.0}},
       {2, {1.5, -0.5, 0.0, 0.0, 0.0}}}},
    // kappa <= 256: 15 products
    {256.0, 4, {{5, {9.601856390902624, -76.96229825255085, 240.13326229681704,
        -299.0023258629703, 127.64795113005505}},
       {5, {2.7326221624027687, -4.139235353524874, 3.827479034556605, -1.7187867838742936,
        0.29354150356959796}},
       {5, {2.4609989207683256, -3.2814389884610042, 2.953323436636903, -1.4063255935765278,
        0.27344222463222323}},
       {2, {1.5, -0.5, 0.0, 0.0, 0.0}}}},
    // kappa <= 512: 16 products
    {512.0, 4, {{5, {10.748950692241019, -91.66446129686902, 292.13536569581737,
        -367.647117903867, 157.96008486597194}},
       {5, {2.952178411889042, -4.849297107505271, 4.513961407076106, -1.944252415633257,
        0.3087304741806296}},
       {5, {2.4617007305619, -3.2835986303531906, 2.9555908692025024, -1.4071891730828199,
        0.2734962035178481}},
       {3, {1.875, -1.25, 0.375, 0.0, 0.0}}}},
    // kappa <= 1024: 16 products
    {1024.0, 4, {{5, {11.75640461876193, -104.69325186978253, 338.4056696071483,
        -428.8668120287819, 185.0337869400125}},
       {5, {3.2619198699928456, -5.852379027747174, 5.438929825691906, -2.231552163065048,
        0.3288418860291944}},
       {5, {2.466032640690303, -3.2969375052669636, 2.9695882688262447, -1.4125125928905813,
        0.27382914325543883}},
       {3, {1.875, -1.25, 0.375, 0.0, 0.0}}}},
    // kappa <= 2048: 17 products
    {2048.0, 4, {{5, {12.595923695465602, -115.60998888072238, 377.27085210615115,
        -480.36095185040944, 207.82707710726876}},
       {5, {3.663993086286645, -7.1380544676944995, 6.568289074846145, -2.566096183114514,
        0.35317298014064447}},
       {5, {2.4824392788256873, -3.3475873896118817, 3.022624279384485, -1.4325657976617303,
        0.2750863180215699}},
       {5, {2.4609375, -3.28125, 2.953125, -1.40625, 0.2734375}}}},
    // kappa <= 4096: 17 products
    {4096.0, 4, {{5, {13.266700710926264, -124.36276224325611, 408.480355006326,
        -521.7481877564505, 226.15707610982685}},
       {5, {4.143963385643623, -8.640099133627986, 7.831865158861571, -2.9271122480198697,
        0.3803010077249447}},
       {5, {2.525825589508507, -3.4824623635655225, 3.1629535909918207, -1.484783166603468,
        0.2783821226481133}},
       {5, {2.4609375, -3.28125, 2.953125, -1.40625, 0.2734375}}}},
};

// The tiles on and below the diagonal of a symmetric matrix of NJ x NJ tiles.
template <int NJ>
struct Sym {
  static constexpr int kTiles = NJ * (NJ + 1) / 2;
  static constexpr int kOff = NJ * (NJ - 1) / 2;  // tiles below the diagonal
  double4_t t[kTiles];
  static __device__ constexpr int at(int I, int J) { return I * (I + 1) / 2 + J; }
  static __device__ constexpr int off(int I, int J) { return I * (I - 1) / 2 + J; }
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int i = 0; i < kTiles; ++i) t[i] = double4_t{0.0, 0.0, 0.0, 0.0};
  }
  // f(I, J, r) for the elements held
  template <class F>
  __device__ __forceinline__ static void each(F f) {
#pragma unroll
    for (int I = 0; I < NJ; ++I)
#pragma unroll
      for (int J = 0; J <= I; ++J)
#pragma unroll
        for (int r = 0; r < 4; ++r) f(I, J, r);
  }
};

// Place of element (row, col) of a 16 x 16 tile in LDS: the columns of a row
// are permuted so that both a tile's own rows (written) and its transpose
// (read) touch every bank once.
__device__ __forceinline__ int tile_at(int row, int col) { return row * 16 + (col ^ (row & 14)); }

// The tiles below the diagonal to LDS (z: 256 doubles a tile).
template <int NJ>
__device__ __forceinline__ void publish(const Sym<NJ>& M, double* z) {
  const int lane = threadIdx.x, g = lane >> 4, c = lane & 15;
  __syncthreads();  // what z held has been read
#pragma unroll
  for (int I = 1; I < NJ; ++I)
#pragma unroll
    for (int J = 0; J < I; ++J)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        z[Sym<NJ>::off(I, J) * 256 + tile_at(4 * r + g, c)] = M.t[Sym<NJ>::at(I, J)][r];
  __syncthreads();
}

// Element (K*16 + 4r + g, J*16 + c) of M, its tiles below the diagonal in z.
template <int NJ>
__device__ __forceinline__ double elem(const Sym<NJ>& M, const double* z, int K, int J, int r) {
  const int lane = threadIdx.x, g = lane >> 4, c = lane & 15;
  if (K >= J) return M.t[Sym<NJ>::at(K, J)][r];
  return z[Sym<NJ>::off(J, K) * 256 + tile_at(c, 4 * r + g)];
}

// D += A B for symmetric commuting A (its tiles below the diagonal in za) and B
// (b(K, J, r, o) = its elements, o an offset of 0 to add to LDS pointers).  o is
// opaque to the compiler: it would otherwise keep the elements that one
// product read for the next (48 of 512 registers, and spills).
template <int NJ, class FB>
__device__ __forceinline__ void sym_product(Sym<NJ>& D, const Sym<NJ>& A, const double* za,
                                            FB b) {
  int o = 0;
  asm volatile("" : "+v"(o));
#pragma unroll
  for (int K = 0; K < NJ; ++K)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      double av[NJ], bv[NJ];
#pragma unroll
      for (int I = 0; I < NJ; ++I) av[I] = elem<NJ>(A, za + o, K, I, r);
#pragma unroll
      for (int J = 0; J < NJ; ++J) bv[J] = b(K, J, r, o);
#pragma unroll
      for (int I = 0; I < NJ; ++I)
#pragma unroll
        for (int J = 0; J <= I; ++J)
          D.t[Sym<NJ>::at(I, J)] = mfma_f64_16x16x4(av[I], bv[J], D.t[Sym<NJ>::at(I, J)]);
    }
}

// Largest column sum of |M|, in every lane; NaN where there is one.
template <int NJ>
__device__ __forceinline__ double norm1(const Sym<NJ>& M, const double* z) {
  double m = 0.0;
#pragma unroll
  for (int J = 0; J < NJ; ++J) {
    double s = 0.0;
#pragma unroll
    for (int K = 0; K < NJ; ++K)
#pragma unroll
      for (int r = 0; r < 4; ++r) s += fabs(elem<NJ>(M, z, K, J, r));
    s += shfl_xor_d(s, 16);
    s += shfl_xor_d(s, 32);
    m = s > m || s != s ? s : m;  // (fmax would drop a NaN)
  }
#pragma unroll
  for (int x = 1; x < 16; x <<= 1) {
    const double o = shfl_xor_d(m, x);
    m = o > m || o != o ? o : m;
  }
  return m;
}

// || M ||_F^2 (trace M^2) in every lane.
template <int NJ>
__device__ __forceinline__ double frob2(const Sym<NJ>& M) {
  double d = 0.0, f = 0.0;
  Sym<NJ>::each([&](int I, int J, int r) {
    const double v = M.t[Sym<NJ>::at(I, J)][r];
    if (I == J) d = fma(v, v, d);
    else f = fma(v, v, f);
  });
  d = fma(2.0, f, d);
#pragma unroll
  for (int x = 1; x < 64; x <<= 1) d += shfl_xor_d(d, x);
  return d;
}

// T (in: M = C + a0 I, C positive semidefinite, published in z0; out: Z,
// published in z2) such that M^(-1/2) = sqrt(*inv) Z.  z0, z1, z2: LDS for the
// tiles below the diagonal of one matrix each.  Returns the steps taken, or 0
// with T and z0 unchanged where M is not finite or its condition bound is
// above kIsqrtMaxKappa.
template <int NJ>
__device__ __forceinline__ int sym_isqrt(Sym<NJ>& T, double a0, double* inv, double* z0,
                                         double* z1, double* z2) {
  typedef Sym<NJ> S;
  const int lane = threadIdx.x, g = lane >> 4, c = lane & 15;
  auto opT = [&](int K, int J, int r, int o) { return elem<NJ>(T, z0 + o, K, J, r); };
  S T2;
  T2.zero();
  sym_product<NJ>(T2, T, z0, opT);
  publish<NJ>(T2, z1);
  double top = sqrt(norm1<NJ>(T2, z1));
  if constexpr (NJ > 2) {
    // the tighter bound saves up to two products (1 degree, k = 64: 11.43 -> 11.33
    // ms a sweep); up to 32 members its reduction costs what it saves (vertical
    // localisation, k = 32: 3.90 and 3.94 ms)
    // (below 1e-70 the trace of M^4 could underflow)
    const double n4 = sqrt(sqrt(frob2<NJ>(T2)));
    top = n4 < top && a0 > 1e-70 ? n4 : top;
  }
  const double kap = top / a0 * (1.0 + 1e-12);
  // (a0 outside this range could lose M^2 to underflow)
  if (!(kap <= kIsqrtMaxKappa && a0 > 1e-100 && a0 < 1e100)) return 0;
  int cls = 0;
#pragma unroll
  for (int i = 0; i < kIsqrtPlans - 1; ++i) cls += kap > kIsqrtPlan[i].kappa;
  cls = __builtin_amdgcn_readfirstlane(cls);
  const IsqrtPlan& plan = kIsqrtPlan[cls];
  const double sc = 1.0 / (a0 * kap);
  *inv = sc;
#pragma unroll
  for (int i = 0; i < S::kTiles; ++i) {
    T.t[i] *= sc;
    T2.t[i] *= sc * sc;
  }
  publish<NJ>(T, z0);
  publish<NJ>(T2, z1);
  S Z;
  const int n = plan.nstep;
  for (int i = 0;; ++i) {
    const int nc = plan.step[i].nc;
    const double c0 = plan.step[i].c[0], c1 = plan.step[i].c[1], c2 = plan.step[i].c[2],
                 c3 = plan.step[i].c[3], c4 = plan.step[i].c[4];
    auto diag = [&](int K, int J, int r, double v) {
      return K == J && 4 * r + g == c ? v : 0.0;
    };
    S P;
    S::each([&](int I, int J, int r) {
      P.t[S::at(I, J)][r] = fma(c1, T.t[S::at(I, J)][r], diag(I, J, r, c0));
    });
    if (nc == 5) {
      sym_product<NJ>(P, T2, z1, [&](int K, int J, int r, int o) {
        return fma(c4, elem<NJ>(T2, z1 + o, K, J, r),
                   fma(c3, elem<NJ>(T, z0 + o, K, J, r), diag(K, J, r, c2)));
      });
    } else if (nc == 3) {
#pragma unroll
      for (int j = 0; j < S::kTiles; ++j) P.t[j] += c2 * T2.t[j];
    }
    publish<NJ>(P, z1);
    auto opP = [&](int K, int J, int r, int o) { return elem<NJ>(P, z1 + o, K, J, r); };
    const bool last = i + 1 == n;
    if (!last) {
      S U;
      U.zero();
      sym_product<NJ>(U, T, z0, opP);
      publish<NJ>(U, z0);
      T.zero();
      sym_product<NJ>(T, P, z1, [&](int K, int J, int r, int o) {
        return elem<NJ>(U, z0 + o, K, J, r);
      });
      publish<NJ>(T, z0);
    }
    // Z <- Z P (Z = P after the first step)
    if (i == 0) {
      Z = P;
    } else {
      S Y;
      Y.zero();
      sym_product<NJ>(Y, Z, z2, opP);
      Z = Y;
    }
    publish<NJ>(Z, z2);
    if (last) break;
    if (plan.step[i + 1].nc > 2) {
      T2.zero();
      sym_product<NJ>(T2, T, z0, opT);
      publish<NJ>(T2, z1);
    }
  }
  T = Z;
  return n;
}

}  // namespace dida
