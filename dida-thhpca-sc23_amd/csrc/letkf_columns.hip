// Ensemble update (xb_2_xa, letkf_compute.F90:231-301) of columns from transforms
// in HBM, on FP64 MFMA: Xa = trans^T Xb' + xbar_b, mean, re-centre, and optionally
// RTPS (Xa' <- Xa' (alpha sigma_b / sigma_a + 1 - alpha)).
#include <cstring>

#include "letkf_device.h"
#include "letkf_kernels.h"
#include "letkf_wave.h"

using namespace dida;

namespace {

// Update of columns from stored transforms: a column's own (trans + (col - col0)
// k^2) or, with horizontal cubes, the mean of the covering cubes' transforms
// (summed in the reference's cube order: longitude starts outer, latitude
// inner; averaging transforms equals averaging the cubes' re-centred analyses,
// which are linear in trans).
//
// Bound by HBM (Xb' in, Xa' out); the transforms come from L2 and stay in
// registers.  Columns between two consecutive starts or ends of cubes share
// their covering cubes, so a wavefront takes a block of them (up to clat x clon
// of one latitude and one longitude segment): the mean is formed once a block
// instead of once a column, and the rows of neighbouring latitudes are
// contiguous, one list of tiles of 16 rows.  Members go to the MFMA steps in
// the order i = 16 I + 4g + r, e = 16 E + 4g + r, so that a lane's four values
// of a tile are adjacent in trans, Xb' and Xa' (16-byte accesses).  Measured at 1
// degree, k = 64, cubes of 4 with overlap 2: 3.27 ms with a column a wavefront
// and 8-byte accesses, 1.57 ms (4.1 TB/s) so; bounded to 256 registers, two
// wavefronts a SIMD, it spills 55 and takes 1.8 ms.
struct ColSeg {
  int start, len, a0, a1;  // columns [start, start + len), cubes a0 .. a1
};
// Segment q of an axis of n columns, cubes of cn columns every st.
__device__ __forceinline__ ColSeg col_segment(int q, int n, int cn, int st, int na) {
  const int r = cn % st;
  const int m = r ? q >> 1 : q;
  ColSeg s;
  s.start = m * st + (r && (q & 1) ? r : 0);
  s.len = min(r ? (q & 1 ? st - r : r) : st, n - s.start);
  s.a0 = s.start - cn + 1 > 0 ? (s.start - cn + st) / st : 0;
  s.a1 = min(s.start / st, na - 1);
  return s;
}


// The columns of block b: nlat x nlon of them from col on (latitudes adjacent,
// longitudes u.nlat apart), covered by cubes aj0 .. aj1 by ai0 .. ai1.
struct ColBlock {
  int64_t col;
  int nlat, nlon, aj0, aj1, ai0, ai1;
};
__device__ __forceinline__ ColBlock col_block(const dk_update_args& u, const dk_update_grid& gr,
                                              int b) {
  if (u.cube_n <= 1) return ColBlock{(int64_t)u.col0 + b, 1, 1, 0, 0, 0, 0};
  const int pa = b % gr.plat;
  b /= gr.plat;
  const ColSeg sa = col_segment(b % gr.slat, u.nlat, u.cube_n, u.step, u.nalat);
  b /= gr.slat;
  const int po = b % gr.plon;
  const ColSeg so = col_segment(b / gr.plon, u.nlon, u.cube_n, u.step, u.nalon);
  const int ilat = sa.start + pa * gr.clat, ilon = so.start + po * gr.clon;
  return ColBlock{(int64_t)ilat + (int64_t)u.nlat * ilon,
                  min(gr.clat, sa.start + sa.len - ilat),
                  min(gr.clon, so.start + so.len - ilon),
                  sa.a0, sa.a1, so.a0, so.a1};
}

// Four consecutive values from p on; LAST (the tile that k ends in): those from n
// on zero.
template <bool LAST>
__device__ __forceinline__ double4_t load4(const double* p, int n) {
  double4_t v;
  if (!LAST || n >= 4) {
    const d2u_t a = *reinterpret_cast<const d2u_t*>(p);
    const d2u_t b = *reinterpret_cast<const d2u_t*>(p + 2);
    v = double4_t{a[0], a[1], b[0], b[1]};
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = r < n ? p[r] : 0.0;
  }
  return v;
}
template <bool LAST>
__device__ __forceinline__ f32x4_t load4(const float* p, int n) {
  f32x4_t v;
  if (!LAST || n >= 4) {
    v = *reinterpret_cast<const f4u_t*>(p);
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = r < n ? p[r] : 0.0f;
  }
  return v;
}
// Four consecutive values to p on, those from n on not.
__device__ __forceinline__ void store4(double* p, const double4_t& v, int n) {
  if (n >= 4) {
    *reinterpret_cast<d2u_t*>(p) = d2u_t{v[0], v[1]};
    *reinterpret_cast<d2u_t*>(p + 2) = d2u_t{v[2], v[3]};
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (r < n) p[r] = v[r];
  }
}
__device__ __forceinline__ void store4(float* p, const double4_t& v, int n) {
  if (n >= 4) {
    *reinterpret_cast<f4u_t*>(p) = f4u_t{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (r < n) p[r] = (float)v[r];
  }
}

// What is taken from the members' deviations: their mean; a row whose xbar_b is not
// finite has no finite member, as where xbar_b is added before the mean is taken.
__device__ __forceinline__ double centre_of(double mean, double xbar) {
  return __builtin_isfinite(xbar) ? mean : __builtin_nan("");
}

template <int KP>
__global__ __launch_bounds__(64, KP <= 32 ? 4 : KP == 48 ? 2 : 1) void k_update_cols(dk_update_args u,
                                                                      dk_update_grid gr) {
  constexpr int NJ = KP / 16;
  const int lane = threadIdx.x, g = lane >> 4, c = lane & 15;
  const int k = u.k;
  const int em = 4 * (c & 3) + (c >> 2);  // the member of a tile that lane c feeds
  const int i_last = (NJ - 1) * 16 + 4 * g;  // the lane's first member in the last tile
  const double4_t zero = double4_t{0.0, 0.0, 0.0, 0.0};
  double4_t T[NJ][NJ];
#pragma unroll
  for (int I = 0; I < NJ; ++I)
#pragma unroll
    for (int E = 0; E < NJ; ++E) T[I][E] = zero;
  auto add_trans = [&](const double* tr) {
#pragma unroll
    for (int E = 0; E < NJ; ++E) {
      const int e = E * 16 + em;
      const bool in = E < NJ - 1 || e < k;
      const double* col = tr + (int64_t)(in ? e : 0) * k;
#pragma unroll
      for (int I = 0; I < NJ - 1; ++I) {
        const double4_t v = load4<false>(col + I * 16 + 4 * g, 4);
        T[I][E] += in ? v : zero;
      }
      const double4_t v = load4<true>(col + i_last, k - i_last);
      T[NJ - 1][E] += in ? v : zero;
    }
  };
  const ColBlock cb = col_block(u, gr, blockIdx.x);
  if (cb.nlat <= 0 || cb.nlon <= 0) return;
  const int nlat = cb.nlat, nlon = cb.nlon;
  if (u.cube_n > 1) {
    for (int ai = cb.ai0; ai <= cb.ai1; ++ai)
      for (int aj = cb.aj0; aj <= cb.aj1; ++aj)
        add_trans(u.trans + ((int64_t)aj + (int64_t)u.nalat * ai) * k * k);
    const double cnt = (double)((cb.aj1 - cb.aj0 + 1) * (cb.ai1 - cb.ai0 + 1));
#pragma unroll
    for (int I = 0; I < NJ; ++I)
#pragma unroll
      for (int E = 0; E < NJ; ++E)
#pragma unroll
        for (int r = 0; r < 4; ++r) T[I][E][r] /= cnt;
  } else {
    add_trans(u.trans + (int64_t)blockIdx.x * k * k);
  }
  const int nr = nlat * u.nrow;
  for (int x = 0; x < nlon; ++x) {
    const int64_t col = cb.col + (int64_t)u.nlat * x;
    const double* xb = u.xb + col * u.nrow * k;
    const double* axb = u.axb + col * u.nrow;
    double* xa = u.xa + col * u.nrow * k;
    double* axa = u.axa + col * u.nrow;
    // Xb' and xbar of rows R0 + c, the next tile's in flight while one computes
    auto load_rows = [&](int R0, double4_t (&v)[NJ], double& xbar) {
      const int row = R0 + c < nr ? R0 + c : nr - 1;
      xbar = axb[row];
#pragma unroll
      for (int I = 0; I < NJ - 1; ++I)
        v[I] = load4<false>(xb + (int64_t)row * k + I * 16 + 4 * g, 4);
      v[NJ - 1] = load4<true>(xb + (int64_t)row * k + i_last, k - i_last);
    };
    double4_t xl[NJ];
    double xbar;
    load_rows(0, xl, xbar);
    for (int R0 = 0; R0 < nr; R0 += 16) {
      const int row = R0 + c;
      const bool rok = row < nr;
      double4_t xn[NJ], D[NJ];
      double xbarn;
      load_rows(R0 + 16, xn, xbarn);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int E = 0; E < NJ; ++E) D[E] = zero;
      double ssb = 0.0;
#pragma unroll
      for (int I = 0; I < NJ; ++I)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const double xv = xl[I][r];
          if (u.rtps) ssb = fma(xv, xv, ssb);
#pragma unroll
          for (int E = 0; E < NJ; ++E) D[E] = mfma_f64_16x16x4(T[I][E][r], xv, D[E]);
        }
      // D[E][r]: member 16 E + 4g + r of the lane's row without xbar (members
      // past k are zero, as their trans columns), so that the mean of the
      // deviations does not carry xbar's rounding
      double4_t s4 = D[0];
#pragma unroll
      for (int E = 1; E < NJ; ++E) s4 += D[E];
      const double mean = sum_g((s4[0] + s4[1]) + (s4[2] + s4[3])) / (double)k;
      const double centre = centre_of(mean, xbar);
#pragma unroll
      for (int E = 0; E < NJ; ++E) D[E] -= centre;
      double fac = 1.0;
      if (u.rtps) {
        double4_t q4 = zero;
#pragma unroll
        for (int E = 0; E < NJ - 1; ++E) q4 += D[E] * D[E];
        double ssa = (q4[0] + q4[1]) + (q4[2] + q4[3]);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          ssa += i_last + r < k ? D[NJ - 1][r] * D[NJ - 1][r] : 0.0;
        ssb = sum_g(ssb);
        ssa = sum_g(ssa);
        if (ssa > 0.0) fac = u.rtps_alpha * sqrt(ssb) / sqrt(ssa) + 1.0 - u.rtps_alpha;
#pragma unroll
        for (int E = 0; E < NJ; ++E) D[E] *= fac;
      }
      if (rok) {
        double* q = xa + (int64_t)row * k;
#pragma unroll
        for (int E = 0; E < NJ; ++E) {
          const int e = E * 16 + 4 * g;
          store4(q + e, D[E], E < NJ - 1 ? 4 : k - e);
        }
        if (g == 0) axa[row] = xbar + mean;
      }
#pragma unroll
      for (int I = 0; I < NJ; ++I) xl[I] = xn[I];
      xbar = xbarn;
    }
  }
}

// The same for 65 to 128 members (NT tiles of 16), a workgroup of four wavefronts a
// block of columns: wavefront w forms the members of tiles w and w + 4 (their
// trans columns in registers, 128 at NT = 8).  Every wavefront reads the rows
// itself, two tiles of members at a time with the next two in flight (they come
// from L1 after the first wavefront); only the row sums meet, through LDS, one
// barrier a tile of rows.  256 registers a lane, two workgroups a CU, so that
// one's transform loads run beside the other's products.  S: type that Xb' and
// Xa' are stored in; all arithmetic is FP64.  Measured
// at 1 degree, k = 128, FP32 state, 97 rows (15 GB, 0.2 TFLOP): 9.9 ms with rows
// staged in LDS a tile at a time, nothing in flight behind, 8.1 ms with whole rows
// in flight, 5.6 ms so (at NT = 8 the bound of 256 spills 39 registers, 44 with FP64
// state; at 7, 3); a tile a wavefront, eight wavefronts: 6.7 ms (168 registers, one
// workgroup a CU) and 11.5 ms (128, spilling more).
template <int NT, typename S>
__global__ __launch_bounds__(256, 2) void k_update_cols128(dk_update_args u,
                                                               dk_update_grid gr) {
  typedef decltype(load4<false>((const S*)nullptr, 4)) Raw;
  constexpr int NC = (NT + 1) / 2;
  __shared__ double sv[2][4][16], sq[2][4][16];
  const int w = (int)threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int k = u.k;
  const bool two = w + 4 < NT;                     // whether the wavefront has a second tile
  const int em = w * 16 + 4 * (c & 3) + (c >> 2);  // the member that lane c feeds (and + 64)
  const int e0 = w * 16 + 4 * g;                   // the lane's first member of D
  const int i_last = (NT - 1) * 16 + 4 * g;        // and of the last tile of a row
  const double4_t zero = double4_t{0.0, 0.0, 0.0, 0.0};
  const ColBlock cb = col_block(u, gr, blockIdx.x);
  if (cb.nlat <= 0 || cb.nlon <= 0) return;
  const bool in1 = em + 64 < k;  // (em < 64 < k)
  const uint32_t t0 = (uint32_t)em * (uint32_t)k + 4 * g;
  const uint32_t t1 = (uint32_t)(in1 ? em + 64 : 0) * (uint32_t)k + 4 * g;
  auto trans4 = [&](const double* tr, int x, int I) {
    const double* q = tr + ((x ? t1 : t0) + I * 16);
    return I < NT - 1 ? load4<false>(q, 4) : load4<true>(q, k - i_last);
  };
  double4_t T[2][NT];
  if (u.cube_n > 1) {
#pragma unroll
    for (int I = 0; I < NT; ++I) T[0][I] = T[1][I] = zero;
    for (int ai = cb.ai0; ai <= cb.ai1; ++ai)
      for (int aj = cb.aj0; aj <= cb.aj1; ++aj) {
        const double* tr = u.trans + ((int64_t)aj + (int64_t)u.nalat * ai) * k * k;
#pragma unroll
        for (int I = 0; I < NT; ++I) {
          T[0][I] += trans4(tr, 0, I);
          T[1][I] += trans4(tr, 1, I);
          if (I & 1) __builtin_amdgcn_sched_barrier(0);  // few in flight: registers
        }
      }
    const double cnt = (double)((cb.aj1 - cb.aj0 + 1) * (cb.ai1 - cb.ai0 + 1));
#pragma unroll
    for (int I = 0; I < NT; ++I)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        T[0][I][r] /= cnt;
        T[1][I][r] /= cnt;
      }
  } else {
    const double* tr = u.trans + (int64_t)blockIdx.x * k * k;
#pragma unroll
    for (int I = 0; I < NT; ++I) {
      T[0][I] = trans4(tr, 0, I);
      T[1][I] = trans4(tr, 1, I);
    }
  }
  if (!in1)
#pragma unroll
    for (int I = 0; I < NT; ++I) T[1][I] = zero;
  const S* xbs;
  S* xas;
  if constexpr (sizeof(S) == sizeof(float)) {
    xbs = u.xb32;
    xas = u.xa32;
  } else {
    xbs = u.xb;
    xas = u.xa;
  }
  const int nr = cb.nlat * u.nrow;
  int buf = 0;
  for (int y = 0; y < cb.nlon; ++y) {
    const int64_t row0 = (cb.col + (int64_t)u.nlat * y) * u.nrow;
    const S* xb = xbs + row0 * k;
    S* xa = xas + row0 * k;
    // the lane's members of tiles 2h and 2h + 1 of row R0 + c (clamped, in bounds)
    auto load_x = [&](int R0, int h, Raw (&v)[2]) {
      const uint32_t o = (uint32_t)(R0 + c < nr ? R0 + c : nr - 1) * (uint32_t)k + 4 * g;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int I = 2 * h + j;
        if (I < NT - 1) v[j] = load4<false>(xb + (o + I * 16), 4);
        if (I == NT - 1) v[j] = load4<true>(xb + (o + I * 16), k - i_last);
      }
    };
    Raw cur[2], nxt[2];
    load_x(0, 0, cur);
    for (int R0 = 0; R0 < nr; R0 += 16, buf ^= 1) {
      const int row = R0 + c;
      const double xbar = u.axb[row0 + (row < nr ? row : nr - 1)];
      double4_t D[2] = {zero, zero};
      double ssb = 0.0;
#pragma unroll
      for (int h = 0; h < NC; ++h) {
        if (h + 1 < NC) load_x(R0, h + 1, nxt);
        else load_x(R0 + 16, 0, nxt);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 2; ++j)
          if (2 * h + j < NT)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const double xv = (double)cur[j][r];
              if (u.rtps) ssb = fma(xv, xv, ssb);
              D[0] = mfma_f64_16x16x4(T[0][2 * h + j][r], xv, D[0]);
              if (two) D[1] = mfma_f64_16x16x4(T[1][2 * h + j][r], xv, D[1]);
            }
        cur[0] = nxt[0];
        cur[1] = nxt[1];
      }
      // D[x][r]: member e0 + 64 x + r of the lane's row without xbar
      const double4_t s4 = D[0] + D[1];
      const double s = sum_g((s4[0] + s4[1]) + (s4[2] + s4[3]));
      if (g == 0) sv[buf][w][c] = s;
      __syncthreads();
      const double mean =
          ((sv[buf][0][c] + sv[buf][1][c]) + (sv[buf][2][c] + sv[buf][3][c])) / (double)k;
      const double centre = centre_of(mean, xbar);
      D[0] -= centre;
      D[1] -= centre;
      if (u.rtps) {
        double q = 0.0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          q = fma(D[0][r], D[0][r], q);
          q += e0 + 64 + r < k ? D[1][r] * D[1][r] : 0.0;
        }
        q = sum_g(q);
        if (g == 0) sq[buf][w][c] = q;
        __syncthreads();
        ssb = sum_g(ssb);
        const double ssa =
            (sq[buf][0][c] + sq[buf][1][c]) + (sq[buf][2][c] + sq[buf][3][c]);
        const double fac =
            ssa > 0.0 ? u.rtps_alpha * sqrt(ssb) / sqrt(ssa) + 1.0 - u.rtps_alpha : 1.0;
        D[0] *= fac;
        D[1] *= fac;
      }
      if (row < nr) {
        const uint32_t o = (uint32_t)row * (uint32_t)k + e0;
        store4(xa + o, D[0], 4);
        store4(xa + (o + 64), D[1], k - e0 - 64);
        if (w == 0 && g == 0) u.axa[row0 + row] = xbar + mean;
      }
    }
  }
}

// How the columns are dealt: horizontal cubes to blocks (see ColBlock), the largest
// that still leave `least` of them (rows of a column are a chain of tiles, so a
// small grid is better split than shared).  Returns the number of blocks.
int64_t deal_columns(const dk_update_args* u, int64_t least, dk_update_grid* gr) {
  memset(gr, 0, sizeof *gr);
  if (u->cube_n <= 1) return u->ncol;
  const int st = u->step, per = u->cube_n % st ? 2 : 1;
  gr->slat = (u->nlat + st - 1) / st * per;
  const int slon = (u->nlon + st - 1) / st * per;
  gr->clat = gr->clon = st;
  auto blocks = [&] {
    gr->plat = (st + gr->clat - 1) / gr->clat;
    gr->plon = (st + gr->clon - 1) / gr->clon;
    return (int64_t)gr->slat * gr->plat * slon * gr->plon;
  };
  while (blocks() < least && gr->clat * gr->clon > 1) {
    if (gr->clon >= gr->clat) gr->clon = (gr->clon + 1) / 2;
    else gr->clat = (gr->clat + 1) / 2;
  }
  return blocks();
}

template <int NT>
int launch128(const dk_update_args* u, const dk_update_grid* gr, unsigned n, hipStream_t s) {
  if (u->xa32) k_update_cols128<NT, float><<<n, 256, 0, s>>>(*u, *gr);
  else k_update_cols128<NT, double><<<n, 256, 0, s>>>(*u, *gr);
  return (int)hipGetLastError();
}

}  // namespace

extern "C" int dk_update_cols(const dk_update_args* u, void* stream) {
  if (u->ncol <= 0) return 0;
  if (u->k < 2 || u->k > 128 || (u->k <= 64 && u->xa32)) return (int)hipErrorInvalidValue;
  hipStream_t s = (hipStream_t)stream;
  dk_update_grid gr;
  // 4 wavefronts a SIMD, or 8 workgroups a CU
  const unsigned n = (unsigned)deal_columns(u, u->k <= 64 ? 4096 : 2048, &gr);
  switch ((u->k + 15) / 16) {
    case 1: k_update_cols<16><<<n, 64, 0, s>>>(*u, gr); break;
    case 2: k_update_cols<32><<<n, 64, 0, s>>>(*u, gr); break;
    case 3: k_update_cols<48><<<n, 64, 0, s>>>(*u, gr); break;
    case 4: k_update_cols<64><<<n, 64, 0, s>>>(*u, gr); break;
    case 5: return launch128<5>(u, &gr, n, s);
    case 6: return launch128<6>(u, &gr, n, s);
    case 7: return launch128<7>(u, &gr, n, s);
    default: return launch128<8>(u, &gr, n, s);
  }
  return (int)hipGetLastError();
}
