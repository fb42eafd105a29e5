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
// negative one), the largest at most sqrt(|| M^2 ||_1), one product that the
// first step needs anyway.  The iteration's own error grows with kappa
// (relative error in the 2-norm against 40-digit arithmetic, 64 x 64: 7e-16 at
// kappa 10, 3e-15 at 100, 3e-14 at 1300, 6e-14 at 3200; Jacobi with tolerance
// 1e-13: 2e-13 throughout) and would pass the Jacobi's at some 10 000; above
// kIsqrtMaxKappa an analysis takes the Jacobi.  T <- P (T P) has the smallest
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
// Layout: double4_t M[I][J], element r of lane (g = l / 16, c = l % 16) =
// M(I*16 + 4r + g, J*16 + c), the result of mfma_f64_16x16x4.  Read as an
// operand, M[K][J][r] is B(K*16 + 4r + g, J*16 + c), and, M being symmetric,
// M[K][I][r] is A(I*16 + c, K*16 + 4r + g): a product needs no data movement.
// All iterates are polynomials in M, so every product is symmetric.
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

// The tiles above the diagonal from the ones below, through LDS (tile (I, J)
// written as element (4r + g, c), read as (c, 4r + g)), two at a time.
template <int NJ>
__device__ __forceinline__ void mirror_lower(double4_t (&D)[NJ][NJ], double* ct) {
  const int lane = threadIdx.x, g = lane >> 4, c = lane & 15;
  constexpr int NT = NJ * (NJ - 1) / 2;
  constexpr int kI[6] = {1, 2, 2, 3, 3, 3}, kJ[6] = {0, 0, 1, 0, 1, 2};
  static_assert(NT <= 6, "up to 4 x 4 tiles");
#pragma unroll
  for (int t = 0; t < NT; t += 2) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (t + u < NT)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          ct[u * 272 + (4 * r + g) * 17 + c] = D[kI[t + u]][kJ[t + u]][r];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (t + u < NT)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          D[kJ[t + u]][kI[t + u]][r] = ct[u * 272 + c * 17 + 4 * r + g];
    __syncthreads();  // read before the next tiles overwrite them
  }
}

// D += A B for symmetric commuting A, B given by their operands a(K, I, r) and
// b(K, J, r).  From 3 x 3 tiles on, the tiles on and below the diagonal only
// (mirrored after), which saves more MFMA than the mirror costs; at 2 x 2 it
// would save one tile of four.
template <int NJ, class FA, class FB>
__device__ __forceinline__ void sym_product(double4_t (&D)[NJ][NJ], FA a, FB b, double* ct) {
  constexpr bool kLower = NJ >= 3;
#pragma unroll
  for (int K = 0; K < NJ; ++K)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      double av[NJ];
#pragma unroll
      for (int I = 0; I < NJ; ++I) av[I] = a(K, I, r);
#pragma unroll
      for (int J = 0; J < NJ; ++J) {
        const double bv = b(K, J, r);
#pragma unroll
        for (int I = kLower ? J : 0; I < NJ; ++I) D[I][J] = mfma_f64_16x16x4(av[I], bv, D[I][J]);
      }
      // operands formed ahead of their MFMA would not fit the registers
      if constexpr (NJ >= 4) __builtin_amdgcn_sched_barrier(0);
    }
  if constexpr (kLower) mirror_lower<NJ>(D, ct);
}

template <int NJ>
__device__ __forceinline__ void zero(double4_t (&D)[NJ][NJ]) {
#pragma unroll
  for (int I = 0; I < NJ; ++I)
#pragma unroll
    for (int J = 0; J < NJ; ++J) D[I][J] = double4_t{0.0, 0.0, 0.0, 0.0};
}

// f(I, J, r) for every element of a matrix.
template <int NJ, class F>
__device__ __forceinline__ void each(F f) {
#pragma unroll
  for (int I = 0; I < NJ; ++I)
#pragma unroll
    for (int J = 0; J < NJ; ++J)
#pragma unroll
      for (int r = 0; r < 4; ++r) f(I, J, r);
}

// Largest column sum of |D|, in every lane; NaN where there is one.
template <int NJ>
__device__ __forceinline__ double norm1(const double4_t (&D)[NJ][NJ]) {
  double m = 0.0;
#pragma unroll
  for (int J = 0; J < NJ; ++J) {
    double s = 0.0;
#pragma unroll
    for (int I = 0; I < NJ; ++I)
#pragma unroll
      for (int r = 0; r < 4; ++r) s += fabs(D[I][J][r]);
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

// T (in: M = C + a0 I, C positive semidefinite; out: Z) such that
// M^(-1/2) = sqrt(*inv) Z.  z: KP x KP doubles of LDS for Z where three
// matrices and Z do not fit the registers (KP = 64), else unused.  Returns the
// steps taken, or 0 with T unchanged where M is not finite or its condition
// bound is above kIsqrtMaxKappa.
template <int KP>
__device__ __forceinline__ int sym_isqrt(double4_t (&T)[KP / 16][KP / 16], double a0, double* inv,
                                         double* ct, double* z) {
  constexpr int NJ = KP / 16;
  constexpr bool kZlds = KP >= 64;
  const int lane = threadIdx.x, g = lane >> 4, c = lane & 15;
  typedef double4_t Mat[NJ][NJ];
  auto opT = [&](int K, int I, int r) { return T[K][I][r]; };
  Mat T2;
  zero<NJ>(T2);
  sym_product<NJ>(T2, opT, opT, ct);
  const double kap = sqrt(norm1<NJ>(T2)) / a0 * (1.0 + 1e-12);
  // (a0 outside this range could lose M^2 to underflow)
  if (!(kap <= kIsqrtMaxKappa && a0 > 1e-100 && a0 < 1e100)) return 0;
  int cls = 0;
#pragma unroll
  for (int i = 0; i < kIsqrtPlans - 1; ++i) cls += kap > kIsqrtPlan[i].kappa;
  cls = __builtin_amdgcn_readfirstlane(cls);
  const IsqrtPlan& plan = kIsqrtPlan[cls];
  const double sc = 1.0 / (a0 * kap);
  *inv = sc;
  each<NJ>([&](int I, int J, int r) {
    T[I][J][r] *= sc;
    T2[I][J][r] *= sc * sc;
  });
  Mat Z;
  const int n = plan.nstep;
  for (int i = 0;; ++i) {
    const int nc = plan.step[i].nc;
    const double c0 = plan.step[i].c[0], c1 = plan.step[i].c[1], c2 = plan.step[i].c[2],
                 c3 = plan.step[i].c[3], c4 = plan.step[i].c[4];
    Mat P;
    each<NJ>([&](int I, int J, int r) {
      P[I][J][r] = fma(c1, T[I][J][r], I == J && 4 * r + g == c ? c0 : 0.0);
    });
    if (nc == 5) {
      sym_product<NJ>(
          P, [&](int K, int I, int r) { return T2[K][I][r]; },
          [&](int K, int J, int r) {
            return fma(c4, T2[K][J][r], fma(c3, T[K][J][r], K == J && 4 * r + g == c ? c2 : 0.0));
          },
          ct);
    } else if (nc == 3) {
      each<NJ>([&](int I, int J, int r) { P[I][J][r] = fma(c2, T2[I][J][r], P[I][J][r]); });
    }
    auto opP = [&](int K, int J, int r) { return P[K][J][r]; };
    const bool last = i + 1 == n;
    if (!last) {
      Mat U;
      zero<NJ>(U);
      sym_product<NJ>(U, opT, opP, ct);
      zero<NJ>(T);
      sym_product<NJ>(T, opP, [&](int K, int J, int r) { return U[K][J][r]; }, ct);
    }
    // Z <- Z P (Z = P after the first step)
    auto z_at = [&](int I, int J, int r) { return ((I * NJ + J) * 4 + r) * 64 + lane; };
    if (i == 0) {
      each<NJ>([&](int I, int J, int r) {
        if constexpr (kZlds) z[z_at(I, J, r)] = P[I][J][r];
        else Z[I][J][r] = P[I][J][r];
      });
    } else {
      Mat Y;
      zero<NJ>(Y);
      sym_product<NJ>(
          Y,
          [&](int K, int I, int r) {
            if constexpr (kZlds) return z[z_at(K, I, r)];
            else return Z[K][I][r];
          },
          opP, ct);
      if (last) {
        each<NJ>([&](int I, int J, int r) { T[I][J][r] = Y[I][J][r]; });
        return n;
      }
      each<NJ>([&](int I, int J, int r) {
        if constexpr (kZlds) z[z_at(I, J, r)] = Y[I][J][r];
        else Z[I][J][r] = Y[I][J][r];
      });
    }
    if (plan.step[i + 1].nc > 2) {
      zero<NJ>(T2);
      sym_product<NJ>(T2, opT, opT, ct);
    }
  }
}

}  // namespace dida
