// One-sided (Hestenes) Jacobi by a workgroup, for 64 < k <= 128.
//
// The 128 columns of A (LDS, column-major, leading dimension LDA; rows >= k
// and columns >= k are zero padding) are orthogonalised pairwise; a pair
// (p, q) is rotated while |a_p . a_q| > tol |a_p| |a_q|; column norms are
// recomputed at the start of each sweep and updated exactly in between
// (alpha' = alpha - t g, beta' = beta + t g).  A sweep without any rotation
// ends the iteration, or, with predict, a sweep in which no pair had
// g^2 > tol alpha beta (Jacobi converges quadratically, so the next sweep
// would rotate nothing).  flag[4] is LDS scratch.
// For a symmetric positive (semi)definite input the converged columns are
// lambda_j v_j (Hestenes 1958; Demmel & Veselic 1992).
#pragma once

#include "letkf_device.h"

namespace dida {

// ---------------------------------------------------------------------------
// The 128 x 128 block by 256 threads, with the columns in registers.
//
// Groups of eight threads (gp = tid / 8: 32 groups, 8 per wavefront) hold
// four column slots X[0..3] each (initially columns J * 32 + gp); thread sub
// of a group holds rows 8u + sub (u < 16) of its four columns.  Columns are
// kept as sc_j x_j with the scaled rotations of rotation_angle (two FMAs a
// row).  Each round rotates two independent pairs per group, (X0, X1) and
// (X2, X3) or (X0, X3) and (X2, X1), so renaming the slots changes partners
// for free.  Ordering (127 rounds a sweep; the fused kernel's order for two
// pairs per lane group, over 32 groups): for G = 64, 32, ..., 4, blocks of
// G rounds in steps of four, slots 1 and 3 moving once inside the step (from
// group gp ^ 1) and once between steps (from gp ^ lowbit(r + 4) / 2); then
// slots 1 and 3 of the first half of every block of G/4 groups swap with
// slots 0 and 2 of the partner group; three final rounds pair the four
// slots of each group.  Moves along group bits 0-2 stay in the wavefront
// (DPP and lane-swap VALU ops), the six a sweep along bits 3-4 go through
// LDS, which aliases A (the matrix is in registers meanwhile).  Every column returns to
// A at the index it came from, so zero padding columns stay at >= k.
struct JacobiXbuf {
  static constexpr int LD = 132;  // column stride (bank spread)
  double col[64 * LD];            // [2 gp + q][row]: two columns a group
  double nrm[64], sc[64], isc[64];
  int32_t id[64];
};

// sum over the eight lanes of a group (quad_perm [1,0,3,2], [2,3,0,1], then
// row_half_mirror); every lane of the group gets the same bits
__device__ __forceinline__ double oct_sum(double v) {
  v = v + dpp_d<0xB1>(v);
  v = v + dpp_d<0x4E>(v);
  return v + dpp_d<0x141>(v);
}

// v of lane l ^ V.  V = 8: DPP row_ror:8 inside each 16-lane row, one VALU
// instruction (1 degree, k = 128: 165.7 ms a sweep, against 171.6 by ds_swizzle).
// V = 16: ds_swizzle, one LDS instruction (172.2 by v_permlane16_swap, which takes
// a copy, the swap and a select).  V = 32: v_permlane32_swap of v with itself,
// whose first result holds the value of the lower lanes (l & ~V) and the second
// that of the upper ones (169.0 by ds_bpermute).
template <int V>
__device__ __forceinline__ unsigned lane_xor_u(unsigned v) {
  if constexpr (V == 8) {
    return (unsigned)dpp_u<0x128>((int)v);
  } else if constexpr (V == 16) {
    return (unsigned)__builtin_amdgcn_ds_swizzle((int)v, 0x1F | (16 << 10));
  } else {
    static_assert(V == 32, "lane xor of 8, 16 or 32");
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return (threadIdx.x & 32) ? r[0] : r[1];
  }
}
template <int V>
__device__ __forceinline__ double lane_xor(double v) {
  return __hiloint2double((int)lane_xor_u<V>((unsigned)__double2hiint(v)),
                          (int)lane_xor_u<V>((unsigned)__double2loint(v)));
}

struct Jacobi128 {
  static constexpr int NR = 16;  // rows per thread
  double X[4][NR];               // column slots of the group
  double nrm[4], sc[4], isc[4];  // squared norms, scales, inverse scales (between sweeps)
  int id[4];                     // column index in A
  // Within a sweep the state lives with the pair that is rotated: lanes 0-3
  // of a group hold the top tp and bottom bt of the round's first pair,
  // lanes 4-7 those of the second (row_half_mirror, lane i <-> 7 - i, trades
  // them between the halves).
  struct ColSt {
    double nrm, sc, isc;
  };
  ColSt tp, bt;
  __device__ __forceinline__ static ColSt pick(bool a, const ColSt& x, const ColSt& y) {
    return ColSt{a ? x.nrm : y.nrm, a ? x.sc : y.sc, a ? x.isc : y.isc};
  }

  template <int P, int Q>
  __device__ __forceinline__ double dot() const {
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
#pragma unroll
    for (int u = 0; u < NR; u += 4) {
      a0 = fma(X[P][u], X[Q][u], a0);
      a1 = fma(X[P][u + 1], X[Q][u + 1], a1);
      a2 = fma(X[P][u + 2], X[Q][u + 2], a2);
      a3 = fma(X[P][u + 3], X[Q][u + 3], a3);
    }
    return (a0 + a1) + (a2 + a3);
  }
  template <int P, int Q>
  __device__ __forceinline__ void apply(double t, double gm, double cs, double ic) {
    const double ta = t * (sc[Q] * isc[P]), tb = t * (sc[P] * isc[Q]);
#pragma unroll
    for (int u = 0; u < NR; ++u) {
      const double x = X[P][u], y = X[Q][u];
      X[P][u] = fma(-ta, y, x);
      X[Q][u] = fma(tb, x, y);
    }
    nrm[P] = fma(-t, gm, nrm[P]);
    nrm[Q] = fma(t, gm, nrm[Q]);
    sc[P] *= cs;
    sc[Q] *= cs;
    isc[P] *= ic;
    isc[Q] *= ic;
  }
  template <int P, int Q>
  __device__ __forceinline__ void rotate_x(double ta, double tb) {
#pragma unroll
    for (int u = 0; u < NR; ++u) {
      const double x = X[P][u], y = X[Q][u];
      X[P][u] = fma(-ta, y, x);
      X[Q][u] = fma(tb, x, y);
    }
  }
  // Lanes 0-3 of a group take the angle of the first pair, lanes 4-7 that
  // of the second: the quad sums of both dot products are exchanged across
  // the halves (row_half_mirror pairs lane i with 7 - i), each half finishes
  // its own pair's sum and angle from its state, updates that state, and the
  // two FMA factors of each pair come back the same way.
  template <int T0, int B0, int T1, int B1>
  __device__ __forceinline__ void round(double tol2, double tolp, bool& rotated, bool& big) {
    double x = dot<T0, B0>(), y = dot<T1, B1>();
    x = x + dpp_d<0xB1>(x);
    y = y + dpp_d<0xB1>(y);
    x = x + dpp_d<0x4E>(x);
    y = y + dpp_d<0x4E>(y);
    const bool second = (threadIdx.x & 4) != 0;
    const double gs = (second ? y : x) + dpp_d<0x141>(second ? x : y);
    double t, gm, cs, ic;
    rotation_angle(gs, tp.nrm, bt.nrm, tp.sc, bt.sc, tol2, tolp, rotated, big, t, gm, cs, ic);
    const double ta = t * (bt.sc * tp.isc), tb = t * (tp.sc * bt.isc);
    tp.nrm = fma(-t, gm, tp.nrm);
    bt.nrm = fma(t, gm, bt.nrm);
    tp.sc *= cs;
    bt.sc *= cs;
    tp.isc *= ic;
    bt.isc *= ic;
    const double tao = dpp_d<0x141>(ta), tbo = dpp_d<0x141>(tb);
    rotate_x<T0, B0>(second ? tao : ta, second ? tbo : tb);
    rotate_x<T1, B1>(second ? ta : tao, second ? tb : tbo);
  }
  // the bottoms' state trades halves (pairing (0, 1), (2, 3) <-> (0, 3), (2, 1))
  __device__ __forceinline__ void swap_bt() {
    bt.nrm = dpp_d<0x141>(bt.nrm);
    bt.sc = dpp_d<0x141>(bt.sc);
    bt.isc = dpp_d<0x141>(bt.isc);
  }
  // (0, 3), (2, 1) -> (0, 2), (3, 1): lanes 0-3 keep their top (column 0) and
  // take the top of lanes 4-7 (column 2) as bottom; lanes 4-7 take the bottom
  // of lanes 0-3 (column 3) as top and keep their bottom (column 1)
  __device__ __forceinline__ void cross_tb() {
    const bool second = (threadIdx.x & 4) != 0;
    const ColSt mt{dpp_d<0x141>(tp.nrm), dpp_d<0x141>(tp.sc), dpp_d<0x141>(tp.isc)};
    const ColSt mb{dpp_d<0x141>(bt.nrm), dpp_d<0x141>(bt.sc), dpp_d<0x141>(bt.isc)};
    tp = pick(second, mb, tp);
    bt = pick(second, bt, mt);
  }
  // the pair state at a sweep's start (lanes 0-3: slots 0, 1; 4-7: 2, 3)
  __device__ __forceinline__ void state_start() {
    const bool second = (threadIdx.x & 4) != 0;
    tp = ColSt{second ? nrm[2] : nrm[0], 1.0, 1.0};
    bt = ColSt{second ? nrm[3] : nrm[1], 1.0, 1.0};
  }
  // the scales of all four slots at a sweep's end (lanes 0-3 hold columns
  // 0 and 2, lanes 4-7 columns 3 and 1)
  __device__ __forceinline__ void state_end() {
    const bool second = (threadIdx.x & 4) != 0;
    const double mt = dpp_d<0x141>(tp.sc), mb = dpp_d<0x141>(bt.sc);
    sc[0] = second ? mt : tp.sc;
    sc[1] = second ? bt.sc : mb;
    sc[2] = second ? mb : bt.sc;
    sc[3] = second ? tp.sc : mt;
  }
  // slot J takes slot J of the group V / 8 groups away (lanes l ^ V)
  template <int J, int V>
  __device__ __forceinline__ void move_lane() {
#pragma unroll
    for (int u = 0; u < NR; ++u) X[J][u] = lane_xor<V>(X[J][u]);
    id[J] = (int)lane_xor_u<V>((unsigned)id[J]);
  }
  template <int V>
  __device__ __forceinline__ void move_bt_lane() {
    bt.nrm = lane_xor<V>(bt.nrm);
    bt.sc = lane_xor<V>(bt.sc);
    bt.isc = lane_xor<V>(bt.isc);
  }
  // the column of slot J (q: 0 or 1 of the group's two exchange places) to
  // the exchange area, and back from group src
  template <int J>
  __device__ __forceinline__ void put(JacobiXbuf& xb, int gp, int sub, int q) const {
#pragma unroll
    for (int u = 0; u < NR; ++u) xb.col[(2 * gp + q) * JacobiXbuf::LD + 8 * u + sub] = X[J][u];
    if (sub == 0) xb.id[2 * gp + q] = id[J];
  }
  template <int J>
  __device__ __forceinline__ void get(const JacobiXbuf& xb, int src, int sub, int q) {
#pragma unroll
    for (int u = 0; u < NR; ++u) X[J][u] = xb.col[(2 * src + q) * JacobiXbuf::LD + 8 * u + sub];
    id[J] = xb.id[2 * src + q];
  }
  // a half's state c to exchange place q of the group (lanes 0 and 4 write)
  __device__ __forceinline__ static void put_st(JacobiXbuf& xb, int gp, int sub, int q,
                                                const ColSt& c) {
    if ((sub & 3) == 0) {
      xb.nrm[2 * gp + q] = c.nrm;
      xb.sc[2 * gp + q] = c.sc;
      xb.isc[2 * gp + q] = c.isc;
    }
  }
  __device__ __forceinline__ static void get_st(const JacobiXbuf& xb, int src, int q, ColSt& c) {
    c.nrm = xb.nrm[2 * src + q];
    c.sc = xb.sc[2 * src + q];
    c.isc = xb.isc[2 * src + q];
  }
  // slots 1 and 3 from group gp ^ v with their state (v >= 8, through LDS:
  // in the pairing (0, 1), (2, 3), where the bottom state of lanes 0-3 is
  // slot 1's and of lanes 4-7 slot 3's)
  __device__ __forceinline__ void move_bottoms(JacobiXbuf& xb, int gp, int sub, int v) {
    if (v == 1) {
      move_lane<1, 8>();
      move_lane<3, 8>();
      move_bt_lane<8>();
    } else if (v == 2) {
      move_lane<1, 16>();
      move_lane<3, 16>();
      move_bt_lane<16>();
    } else if (v == 4) {
      move_lane<1, 32>();
      move_lane<3, 32>();
      move_bt_lane<32>();
    } else {
      const int qh = sub >> 2;  // the half's exchange place: slot 1 or 3
      put<1>(xb, gp, sub, 0);
      put<3>(xb, gp, sub, 1);
      put_st(xb, gp, sub, qh, bt);
      __syncthreads();
      get<1>(xb, gp ^ v, sub, 0);
      get<3>(xb, gp ^ v, sub, 1);
      get_st(xb, gp ^ v, qh, bt);
      __syncthreads();
    }
  }
  // first: slot B takes the partner's slot T; otherwise slot T takes the
  // partner's slot B (partner: lanes l ^ V); the pair's state alike
  template <int T, int B, int V>
  __device__ __forceinline__ void xswap_lane(bool first) {
#pragma unroll
    for (int u = 0; u < NR; ++u) {
      const double w = lane_xor<V>(first ? X[B][u] : X[T][u]);
      X[B][u] = first ? w : X[B][u];
      X[T][u] = first ? X[T][u] : w;
    }
    const int wi = (int)lane_xor_u<V>((unsigned)(first ? id[B] : id[T]));
    id[B] = first ? wi : id[B];
    id[T] = first ? id[T] : wi;
  }
  template <int V>
  __device__ __forceinline__ void xswap_st_lane(bool first) {
    double w = lane_xor<V>(first ? bt.nrm : tp.nrm);
    bt.nrm = first ? w : bt.nrm;
    tp.nrm = first ? tp.nrm : w;
    w = lane_xor<V>(first ? bt.sc : tp.sc);
    bt.sc = first ? w : bt.sc;
    tp.sc = first ? tp.sc : w;
    w = lane_xor<V>(first ? bt.isc : tp.isc);
    bt.isc = first ? w : bt.isc;
    tp.isc = first ? tp.isc : w;
  }
  // (0, 1) and (2, 3) swapped with group gp ^ d, in the pairing (0, 1), (2, 3)
  __device__ __forceinline__ void xswap(JacobiXbuf& xb, int gp, int sub, int d) {
    const bool first = (gp & d) == 0;
    if (d == 1) {
      xswap_lane<0, 1, 8>(first);
      xswap_lane<2, 3, 8>(first);
      xswap_st_lane<8>(first);
    } else if (d == 2) {
      xswap_lane<0, 1, 16>(first);
      xswap_lane<2, 3, 16>(first);
      xswap_st_lane<16>(first);
    } else if (d == 4) {
      xswap_lane<0, 1, 32>(first);
      xswap_lane<2, 3, 32>(first);
      xswap_st_lane<32>(first);
    } else {
      const int qh = sub >> 2;  // the half's pair: (0, 1) or (2, 3)
      // (the state by value: a choice between bt and tp in memory would keep
      // both there, two scratch loads in the chain of every round)
      const ColSt out = pick(first, bt, tp);
      if (first) {
        put<1>(xb, gp, sub, 0);
        put<3>(xb, gp, sub, 1);
      } else {
        put<0>(xb, gp, sub, 0);
        put<2>(xb, gp, sub, 1);
      }
      put_st(xb, gp, sub, qh, out);
      __syncthreads();
      if (first) {
        get<1>(xb, gp ^ d, sub, 0);
        get<3>(xb, gp ^ d, sub, 1);
      } else {
        get<0>(xb, gp ^ d, sub, 0);
        get<2>(xb, gp ^ d, sub, 1);
      }
      ColSt in;
      get_st(xb, gp ^ d, qh, in);
      bt = pick(first, in, bt);
      tp = pick(first, tp, in);
      __syncthreads();
    }
  }
  // X (columns J * 32 + gp, rows 8u + sub), a symmetric positive definite matrix M
  // of order k, zero past k, becomes its lower Cholesky factor: right-looking, a
  // column a step through LDS (col0, col1 in turn), one barrier each.  Returns whether
  // every pivot was positive and finite; otherwise X is undefined.
  __device__ __forceinline__ bool cholesky(int k, int gp, int sub, double* col0, double* col1) {
    bool ok = true;
#pragma unroll
    for (int J = 0; J < 4; ++J)
      for (int cg = 0; cg < 32; ++cg) {
        const int n = J * 32 + cg;
        if (n >= k) break;
        double* v = cg & 1 ? col1 : col0;
        if (gp == cg)
#pragma unroll
          for (int u = 4 * J; u < NR; ++u) v[8 * u + sub] = X[J][u];
        __syncthreads();
        const double d = v[n];
        ok &= d > 0.0 && d < __builtin_inf();
        const double rs = 1.0 / sqrt(d);
        double lc[4];
#pragma unroll
        for (int J2 = J; J2 < 4; ++J2)
          lc[J2] = J2 * 32 + gp > n ? v[J2 * 32 + gp] * rs : 0.0;
#pragma unroll
        for (int u = 4 * J; u < NR; ++u) {
          const double lr = 8 * u + sub >= n ? v[8 * u + sub] * rs : 0.0;
#pragma unroll
          for (int J2 = J; J2 < 4; ++J2)
            X[J2][u] = J2 == J && gp == cg ? lr : fma(-lr, lc[J2], X[J2][u]);
        }
      }
    // above the diagonal, in rows that no step of their own columns has cleared
#pragma unroll
    for (int J = 1; J < 4; ++J)
#pragma unroll
      for (int u = 0; u < 4 * J; ++u) X[J][u] = 0.0;
    return ok;
  }
  __device__ __forceinline__ void fold() {
#pragma unroll
    for (int J = 0; J < 4; ++J) {
#pragma unroll
      for (int u = 0; u < NR; ++u) X[J][u] *= sc[J];
      sc[J] = 1.0;
      isc[J] = 1.0;
    }
  }
};

// CHOL: A is a symmetric positive definite matrix of order k; the sweeps start
// from its Cholesky factor, and *root tells so (false: a pivot was not positive and
// finite, and they started from A).  col0, col1: LDS for a column each.
template <int LDA, int NTHREADS, bool CHOL = false>
__device__ int jacobi_regs128(double* A, int* flag, double tol, int max_sweeps, bool predict,
                              bool* converged, int k = 0, double* col0 = nullptr,
                              double* col1 = nullptr, bool* root = nullptr) {
  static_assert(NTHREADS == 256, "32 groups of eight threads");
  static_assert(sizeof(JacobiXbuf) <= sizeof(double) * 128 * LDA, "exchange area fits in A");
  constexpr int NR = Jacobi128::NR;
  const int tid = threadIdx.x, lane = tid & 63, sub = tid & 7, gp = tid >> 3;
  JacobiXbuf& xb = *reinterpret_cast<JacobiXbuf*>(A);
  Jacobi128 j;
#pragma unroll
  for (int J = 0; J < 4; ++J) {
    j.id[J] = J * 32 + gp;
#pragma unroll
    for (int u = 0; u < NR; ++u) j.X[J][u] = A[8 * u + sub + j.id[J] * LDA];
    j.sc[J] = 1.0;
    j.isc[J] = 1.0;
  }
  if (tid == 0) {
    flag[0] = 0;
    flag[2] = 0;
  }
  if constexpr (CHOL) {
    *root = j.cholesky(k, gp, sub, col0, col1);
    if (!*root)
#pragma unroll
      for (int J = 0; J < 4; ++J)
#pragma unroll
        for (int u = 0; u < NR; ++u) j.X[J][u] = A[8 * u + sub + j.id[J] * LDA];
  }
  __syncthreads();  // A is read before the exchange area is written
  const double tol2 = tol * tol;
  const double tolp = predict ? tol : __builtin_inf();
  int sweep = 0;
  *converged = false;
  for (; sweep < max_sweeps; ++sweep) {
    j.fold();
#pragma unroll
    for (int J = 0; J < 4; ++J) {
      double a0 = 0.0, a1 = 0.0;
#pragma unroll
      for (int u = 0; u < NR; u += 2) {
        a0 = fma(j.X[J][u], j.X[J][u], a0);
        a1 = fma(j.X[J][u + 1], j.X[J][u + 1], a1);
      }
      j.nrm[J] = oct_sum(a0 + a1);
    }
    j.state_start();
    bool rotated = false, big = false;
    for (int G = 64; G >= 4; G >>= 1) {
      for (int r = 0; r < G; r += 4) {
        j.round<0, 1, 2, 3>(tol2, tolp, rotated, big);
        j.swap_bt();
        j.round<0, 3, 2, 1>(tol2, tolp, rotated, big);
        j.move_bottoms(xb, gp, sub, 1);  // lanes l ^ 8: the bottom state moves along
        j.round<0, 3, 2, 1>(tol2, tolp, rotated, big);
        j.swap_bt();
        j.round<0, 1, 2, 3>(tol2, tolp, rotated, big);
        if (r + 4 < G) j.move_bottoms(xb, gp, sub, ((r + 4) & -(r + 4)) >> 1);
      }
      j.xswap(xb, gp, sub, G >> 2);
    }
    j.round<0, 1, 2, 3>(tol2, tolp, rotated, big);
    j.swap_bt();
    j.round<0, 3, 2, 1>(tol2, tolp, rotated, big);
    j.cross_tb();
    j.round<0, 2, 3, 1>(tol2, tolp, rotated, big);
    j.state_end();
    const bool any_rot = __any(rotated), any_big = __any(big);
    if (lane == 0) {
      if (any_rot) flag[sweep & 1] = 1;
      if (any_big) flag[2 + (sweep & 1)] = 1;
    }
    __syncthreads();
    if (flag[sweep & 1] == 0 || (predict && flag[2 + (sweep & 1)] == 0)) {
      *converged = true;
      ++sweep;
      break;
    }
    if (tid == 0) {
      flag[(sweep + 1) & 1] = 0;
      flag[2 + ((sweep + 1) & 1)] = 0;
    }
  }
  j.fold();
  __syncthreads();  // the exchange area is no longer read
#pragma unroll
  for (int J = 0; J < 4; ++J)
#pragma unroll
    for (int u = 0; u < NR; ++u) A[8 * u + sub + j.id[J] * LDA] = j.X[J][u];
  __syncthreads();
  return sweep;
}

}  // namespace dida
