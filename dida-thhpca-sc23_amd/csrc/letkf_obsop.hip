// Observation operator H(Xb) and centring on the GPU (the reference's
// letkf_obs.F90:120-178 with find_obs_grid :187-243, obs_interpolation_3d_2
// and ps2ph_3d_interp, obs_make.F90:233-381, and the half-level pressures of
// vert_coord_mod.F90:547-563).
//
// One wavefront per observation record, lanes over ensemble members (k <=
// 128, two members a lane past 64).  Per member: bilinear surface pressure,
// the level search over full-level pressures computed on the fly (carried
// over the record's levels in order, as the reference's loop does), log-p
// weights between the bracketing levels (the nearest level outside them),
// bilinear horizontal interpolation of member = mean + perturbation.  State
// loads are member-contiguous (coalesced across lanes); the ensemble mean of
// each scalar obs is a wave reduction.  Outputs are the scalar obs of the
// analysis in (record, level, variable) order.
//
// Bound by VALU issue, then by the gathers' latency (the state rows of 4
// corners, 512 bytes each at k = 64), so what is the same for the whole
// record or level is formed once: the record index is a scalar, which makes
// its columns scalar base addresses and a row an offset of one 32-bit multiply
// and add; the grid brackets come from 64 probes at a time (two rounds up to
// 4096 grid points, against 8 or 9 dependent loads); the level search walks
// all members' levels together on scalar coefficients, one half level a
// step; the level weight (two logarithms a member, one of the obs pressure
// and a division) serves every variable.  100 000 single-level records of
// u, v, T at 1 degree, 32 levels, k = 64: 808 -> 491 us; what is left is the
// gather of random 512-byte rows (1.6 GB fetched, 3.3 TB/s; 908 VALU
// instructions a record).
#include "letkf_device.h"
#include "letkf_kernels.h"

using namespace dida;

namespace {

// First index i of ascending g[0..n) with g[i] >= x (n if none), by a whole
// wavefront (x the same in every lane): 64 points split the range that holds
// it.
__device__ __forceinline__ int first_ge(const float* g, int n, double x) {
  const int lane = threadIdx.x & 63;
  int lo = 0, hi = n;  // every point below lo is < x, every point from hi on >= x
  while (lo < hi) {
    const int step = (hi - lo + 63) >> 6;
    const int i = lo + lane * step;
    const bool below = i < hi && (double)g[i < hi ? i : hi - 1] < x;
    const int cnt = __popcll(__builtin_amdgcn_ballot_w64(below));
    if (cnt == 0) {
      hi = lo;
    } else {
      const int last = lo + (cnt - 1) * step;  // the last probe below x
      const int next = last + step;
      hi = next < hi ? next : hi;
      lo = last + 1;
    }
  }
  return lo;
}

// find_obs_grid for one axis: the bracketing indices and the weight of the
// first (REAL(4) grid differences formed in single precision).
__device__ __forceinline__ double bracket(const float* g, int n, bool periodic, double x,
                                          int* i0, int* i1) {
#pragma clang fp contract(off)
  const int j = first_ge(g, n, x);
  if (j == 0) {
    *i0 = *i1 = 0;
    return 0.0;
  }
  if (j == n) {
    if (!periodic) {
      *i0 = *i1 = n - 1;
      return 1.0;
    }
    const float gw = g[0] + 360.0f;
    if (!((double)gw >= x)) {
      *i0 = *i1 = 0;
      return 0.0;
    }
    const double d = (double)(float)(gw - g[n - 1]);
    *i0 = n - 1;
    *i1 = 0;
    return (d - x + (double)g[n - 1]) / d;
  }
  const double d = (double)(float)(g[j] - g[j - 1]);
  *i0 = j - 1;
  *i1 = j;
  return (d - x + (double)g[j - 1]) / d;
}

// half-level pressure j (0-based, top first) over surface pressure ps
// (vert_coord_mod.F90:547-563); A holds vtype, c1, c2, ptop, p0
template <class A>
__device__ __forceinline__ double ph_half(const A& a, int j, double ps) {
#pragma clang fp contract(off)
  if (a.vtype == 0) return a.c1[j] * (ps - a.ptop) + a.ptop;
  return a.c1[j] * (a.p0 - a.ptop) + a.c2[j] * (ps - a.ptop) + a.ptop;
}

// full-level pressure j (0-based) of a member with surface pressure ps
template <class A>
__device__ __forceinline__ double ph_full(const A& a, int j, double ps) {
#pragma clang fp contract(off)
  return 0.5 * (ph_half(a, j, ps) + ph_half(a, j + 1, ps));
}

// M members a lane; OFF: unsigned type of a byte offset inside a column of the
// state (32 bits wherever nrow * k values fit).
template <int M, typename OFF>
__global__ __launch_bounds__(256) void k_obs_operator(dk_obsop_args a) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 +
                    __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (r >= a.nrec) return;
  const int k = a.k, nrow = a.nrow, nlat = a.nlat, nz = a.nz, onz = a.onz, onv = a.onv;
  const double rlat = a.rec_lat[r], rlon = a.rec_lon[r];
  int a0, a1, b0, b1;
  const double t1 = bracket(a.grid_lat, nlat, false, rlat, &a0, &a1);
  const double t2 = bracket(a.grid_lon, a.nlon, a.periodic != 0, rlon, &b0, &b1);
  // the corners' columns of the state: (a0, b0), (a1, b0), (a0, b1), (a1, b1)
  const char* xb[4];
  const double* xm[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int ja = __builtin_amdgcn_readfirstlane(q & 1 ? a1 : a0);
    const int jb = __builtin_amdgcn_readfirstlane(q & 2 ? b1 : b0);
    const int64_t col = (int64_t)ja + (int64_t)nlat * jb;
    xb[q] = reinterpret_cast<const char*>(a.xb + col * nrow * k);
    xm[q] = a.axb + col * nrow;
  }
  const int64_t s0 = r * onz * onv;
  for (int q = lane; q < onz * onv; q += 64) {
    a.lat[s0 + q] = rlat;
    a.lon[s0 + q] = rlon;
    if (a.ph) a.ph[s0 + q] = a.rec_ph[r * onz + q / onv];
  }
  // member e of row `row` at the corners, and the bilinear value
  auto horiz = [&](int row, int e) {
    const OFF o = ((OFF)row * (OFF)k + (OFF)e) * 8u;
    double x[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      x[q] = *reinterpret_cast<const double*>(xb[q] + o) + xm[q][row];
    const double r1 = x[0] * t1 + x[1] * (1 - t1);
    const double r2 = x[2] * t1 + x[3] * (1 - t1);
    return r1 * t2 + r2 * (1 - t2);
  };
  double ps[M];
  int jpos[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const int e = lane + 64 * m;
    ps[m] = e < k ? horiz(a.ps_row, e) : 0.0;
    jpos[m] = 0;
  }
  int j0 = 0;  // no member's level is below j0
  for (int l = 0; l < onz; ++l) {
    const double po = a.rec_ph[r * onz + l];
    // jpos: the first level at or below the member's last whose pressure is
    // not below po; the members at level j move on together
    {
      double h0[M];
#pragma unroll
      for (int m = 0; m < M; ++m) h0[m] = ph_half(a, j0 < nz ? j0 : 0, ps[m]);
      for (int j = j0; j < nz; ++j) {
        bool on = false;   // a member beyond level j
        bool stay = false; // a member that level j holds
#pragma unroll
        for (int m = 0; m < M; ++m) {
          const double h1 = ph_half(a, j + 1, ps[m]);
          const double full = 0.5 * (h0[m] + h1);
          h0[m] = h1;
          const bool mine = lane + 64 * m < k;
          if (jpos[m] == j && po > full) jpos[m] = j + 1;
          on |= mine && jpos[m] > j;
          stay |= mine && jpos[m] == j;
        }
        if (j == j0 && !__builtin_amdgcn_ballot_w64(stay)) j0 = j + 1;
        if (!__builtin_amdgcn_ballot_w64(on)) break;
      }
    }
    // weight of the level above between the bracketing levels, and their rows
    // relative to a variable's first
    const double lpo = log(po);
    double t3[M];
    int up[M], dn[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int p = jpos[m];
      const bool inside = p >= 1 && p < nz;
      up[m] = inside ? p - 1 : (p == 0 ? 0 : nz - 1);
      dn[m] = inside ? p : up[m];
      t3[m] = 0.0;
      if (inside && lane + 64 * m < k) {
        const double pu = ph_full(a, p - 1, ps[m]), pl = ph_full(a, p, ps[m]);
        const double lpl = log(pl);
        t3[m] = (lpl - lpo) / (lpl - log(pu));
      }
    }
    for (int v = 0; v < onv; ++v) {
      const int var = a.vid[v];
      const int vs = a.vstart[var];
      double h[M];
      double sum = 0.0;
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const int e = lane + 64 * m;
        h[m] = 0.0;
        if (e >= k) continue;
        if (a.vlev[var] > 1) {
          // (both rows requested at once; outside the column they are the same)
          const double hu = horiz(vs + up[m], e), hd = horiz(vs + dn[m], e);
          h[m] = dn[m] != up[m] ? hu * t3[m] + hd * (1 - t3[m]) : hu;
        } else {
          h[m] = horiz(vs, e);
        }
        sum += h[m];
      }
      for (int sh = 32; sh >= 1; sh >>= 1) sum += shfl_xor_d(sum, sh);
      const double mean = sum / k;
      const int64_t s = s0 + (int64_t)l * onv + v;
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const int e = lane + 64 * m;
        if (e < k) a.yb[s * k + e] = h[m] - mean;
      }
      if (lane == 0) a.dep[s] = a.yo[s] - mean;
    }
  }
}

// ps2alnp (obs_make.F90:418-437) at the centre level of every cube: one
// thread per (column, cube).  The reference reads the bottom half level
// ph_lev(nz + 1) without setting it; here it is the surface pressure of the
// coordinate table, as for every other half level.
__global__ void k_cube_lnp(dk_cube_lnp_args a) {
#pragma clang fp contract(off)
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= a.ncol * a.ncube) return;
  const int64_t an = t / a.ncube;
  const int q = (int)(t - an * a.ncube);
  const int sk = q * a.cube_nz;
  const int ek = min(sk + a.cube_nz - 1, a.nz - 1);
  const int ck = (sk + 1 + ek + 1) / 2 - 1;
  int64_t col = an;
  if (a.cube_n > 1) {
    const int aj = (int)(an % a.nalat), ai = (int)(an / a.nalat);
    const int sj = aj * a.cube_n, si = ai * a.cube_n;
    const int ej = min(sj + a.cube_n - 1, a.grid_nlat - 1);
    const int ei = min(si + a.cube_n - 1, a.grid_nlon - 1);
    col = (int64_t)((sj + ej) / 2) + (int64_t)a.grid_nlat * ((si + ei) / 2);
  }
  const double ps = a.axb[col * a.nrow + a.ps_row];
  a.cube_lnp[t] = log(ph_full(a, ck, ps));
}

__global__ void k_obs_lnp(int32_t nobs, const int32_t* __restrict__ perm,
                          const double* __restrict__ ph, double* __restrict__ lnp) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nobs) lnp[i] = log(ph[perm[i]]);
}

}  // namespace

extern "C" int dk_cube_lnp(const dk_cube_lnp_args* a, void* stream) {
  const int64_t n = a->ncol * a->ncube;
  if (n <= 0) return 0;
  k_cube_lnp<<<(unsigned)((n + 255) / 256), 256, 0, (hipStream_t)stream>>>(*a);
  return (int)hipGetLastError();
}

extern "C" int dk_obs_lnp(int32_t nobs, const int32_t* perm, const double* ph, double* lnp,
                          void* stream) {
  if (nobs <= 0) return 0;
  k_obs_lnp<<<(nobs + 255) / 256, 256, 0, (hipStream_t)stream>>>(nobs, perm, ph, lnp);
  return (int)hipGetLastError();
}

extern "C" int dk_obs_operator(const dk_obsop_args* a, void* stream) {
  if (a->nrec <= 0) return 0;
  if (a->k < 1 || a->k > 128) return (int)hipErrorInvalidValue;
  const unsigned nb = (unsigned)((a->nrec + 3) / 4);
  hipStream_t s = (hipStream_t)stream;
  const bool narrow = (uint64_t)a->nrow * (uint64_t)a->k * 8u <= 0xFFFFFFFFull;
  if (a->k <= 64) {
    if (narrow) k_obs_operator<1, uint32_t><<<nb, 256, 0, s>>>(*a);
    else k_obs_operator<1, uint64_t><<<nb, 256, 0, s>>>(*a);
  } else {
    if (narrow) k_obs_operator<2, uint32_t><<<nb, 256, 0, s>>>(*a);
    else k_obs_operator<2, uint64_t><<<nb, 256, 0, s>>>(*a);
  }
  return (int)hipGetLastError();
}
