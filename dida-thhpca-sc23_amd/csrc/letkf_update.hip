// Ensemble update (xb_2_xa, letkf_compute.F90:231-301) and the post-analysis
// blend of run_da_parallel (module_da_parallel.F90:216-259).
//
// Update with up to 64 members and the state in FP32 (the other updates:
// letkf_columns.hip), one workgroup per column: trans is staged in LDS as T[i][e] (member
// e contiguous, conflict-free), the column's Xb' rows stream through LDS a few
// rows at a time (ensemble-fastest, so every row is one coalesced load), and
// each lane forms Xa(e) = sum_i trans(i, e) Xb'(i) + xbar_b, the row mean, and
// the re-centred perturbation.  Optional RTPS (Whitaker & Hamill 2012; not in
// the reference): Xa' <- Xa' (alpha sigma_b / sigma_a + 1 - alpha).
#include "letkf_device.h"
#include "letkf_kernels.h"

using namespace dida;

namespace {

constexpr int kThreads = 256;

// Sum of v over the KP lanes of this thread's row slot.
template <int KP>
__device__ __forceinline__ double slot_sum(double v) {
#pragma unroll
  for (int s = 1; s < KP; s <<= 1) v += shfl_xor_d(v, s);
  return v;
}

// Up to 64 members with Xb' and Xa' stored in FP32 (xb32, xa32); the arithmetic is
// FP64.
template <int KP>
__global__ __launch_bounds__(kThreads) void k_update_f64(dk_update_args u) {
  constexpr int RP = kThreads / KP;
  constexpr int LDT = KP + 1;
  __shared__ double sT[KP * LDT];
  __shared__ double sX[RP * KP];
  const int c = blockIdx.x;
  const int64_t col = (int64_t)u.col0 + c;
  const int k = u.k, nrow = u.nrow;
  if (u.cube_n > 1) {
    // mean transform of the cubes covering the column, summed in the
    // reference's cube order (longitude starts outer, latitude inner);
    // averaging the transforms equals averaging the cubes' re-centred
    // analyses (xb_add2_xa / cube_count), which are linear in trans
    const int ilat = (int)(col % u.nlat), ilon = (int)(col / u.nlat);
    const int st = u.step, cn = u.cube_n;
    const int aj0 = ilat - cn + 1 > 0 ? (ilat - cn + 1 + st - 1) / st : 0;
    const int aj1 = min(ilat / st, u.nalat - 1);
    const int ai0 = ilon - cn + 1 > 0 ? (ilon - cn + 1 + st - 1) / st : 0;
    const int ai1 = min(ilon / st, u.nalon - 1);
    const double cnt = (double)((aj1 - aj0 + 1) * (ai1 - ai0 + 1));
    for (int t = threadIdx.x; t < k * k; t += kThreads) {
      double sum = 0.0;
      for (int ai = ai0; ai <= ai1; ++ai)
        for (int aj = aj0; aj <= aj1; ++aj)
          sum += u.trans[((int64_t)aj + (int64_t)u.nalat * ai) * k * k + t];
      const int i = t % k, e = t / k;
      sT[i * LDT + e] = sum / cnt;
    }
  } else {
    const double* T = u.trans + (int64_t)c * k * k;
    for (int t = threadIdx.x; t < k * k; t += kThreads) {
      const int i = t % k, e = t / k;
      sT[i * LDT + e] = T[t];
    }
  }
  const float* xbs = u.xb32;
  float* xas = u.xa32;
  const int e = threadIdx.x % KP, slot = threadIdx.x / KP;
  const double rk = 1.0 / (double)k;
  for (int row0 = 0; row0 < nrow; row0 += RP) {
    const int row = row0 + slot;
    const bool rowok = row < nrow;
    const bool ok = rowok && e < k;
    const int64_t cr = col * nrow + row;
    const double xv = ok ? (double)xbs[cr * k + e] : 0.0;
    __syncthreads();
    sX[slot * KP + e] = xv;
    __syncthreads();
    double acc = 0.0;
    if (rowok)
      for (int i = 0; i < k; ++i) acc += sT[i * LDT + e] * sX[slot * KP + i];
    const double xbar = rowok ? u.axb[cr] : 0.0;
    const double v = ok ? acc + xbar : 0.0;
    const double mean = slot_sum<KP>(v) / (double)k;
    double xa = ok ? v - mean : 0.0;
    if (u.rtps) {
      const double sb2 = slot_sum<KP>(xv * xv) * rk;
      const double sa2 = slot_sum<KP>(xa * xa) * rk;
      if (sa2 > 0.0) xa *= u.rtps_alpha * sqrt(sb2) / sqrt(sa2) + 1.0 - u.rtps_alpha;
    }
    if (ok) xas[cr * k + e] = (float)xa;
    if (rowok && e == 0) u.axa[cr] = mean;
  }
}

__global__ void k_cube_centres(int32_t nlat, int32_t nlon, int32_t cube_n, int32_t step,
                               const float* grid_lat, const float* grid_lon, float* ca_lat,
                               float* ca_lon) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int nalat = (nlat + step - 1) / step, nalon = (nlon + step - 1) / step;
  if (t < nalat) {
    const int s = t * step, e = min(s + cube_n - 1, nlat - 1);
    ca_lat[t] = grid_lat[(s + e) / 2];
  } else if (t < nalat + nalon) {
    const int s = (t - nalat) * step, e = min(s + cube_n - 1, nlon - 1);
    ca_lon[t - nalat] = grid_lon[(s + e) / 2];
  }
}

// Post-analysis blend and spreads: every value of Xb' and Xa' is read once and
// xa_out written once, so the kernel is bound by HBM.  L lanes take a row (a
// row's k members are contiguous), V = 2 members a lane and access where k and
// the arrays' alignment allow 16-byte accesses, and kPostRows rows are in
// flight a thread.  One thread a row, as before, made every access a gather of
// 64 rows: 1 degree, k = 32, 97 rows (4.9 GB): 12.1 ms; now 0.84 ms
// (5.7 TB/s).
constexpr int kPostRows = 4;

template <int V>
struct VecOf {
  typedef double type;
};
template <>
struct VecOf<2> {
  typedef double type __attribute__((ext_vector_type(2)));
};

template <int L, int V>
__global__ __launch_bounds__(kThreads) void k_post(dk_post_args a) {
  typedef typename VecOf<V>::type vec;
  constexpr int kR = kThreads / L;  // rows of the block at a time
  const int64_t ncr = (int64_t)a.nlat * a.nlon * a.nrow;
  const int64_t row0 = (int64_t)blockIdx.x * (kR * kPostRows) + threadIdx.x / L;
  const int l = threadIdx.x % L, k = a.k, nv = k / V;
  double axb[kPostRows], axa[kPostRows], sb[kPostRows], sa[kPostRows];
  bool in[kPostRows];
#pragma unroll
  for (int u = 0; u < kPostRows; ++u) {
    const int64_t t = row0 + u * kR;
    const int64_t tc = t < ncr ? t : ncr - 1;
    axb[u] = a.axb[tc];
    axa[u] = a.axa[tc];
    const int64_t col = tc / a.nrow;
    in[u] = fabs((double)a.grid_lat[(int)(col % a.nlat)]) <= a.polar_lat;
    sb[u] = sa[u] = 0.0;
  }
  for (int e = l; e < nv; e += L) {
    vec b[kPostRows], x[kPostRows];
#pragma unroll
    for (int u = 0; u < kPostRows; ++u) {
      const int64_t t = row0 + u * kR;
      const int64_t tc = t < ncr ? t : ncr - 1;
      b[u] = __builtin_nontemporal_load(reinterpret_cast<const vec*>(a.xb + tc * k) + e);
      x[u] = __builtin_nontemporal_load(reinterpret_cast<const vec*>(a.xa + tc * k) + e);
    }
#pragma unroll
    for (int u = 0; u < kPostRows; ++u) {
      const int64_t t = row0 + u * kR;
      vec o;
#pragma unroll
      for (int i = 0; i < V; ++i) {
        double bv, xv;
        if constexpr (V == 1) {
          bv = b[u];
          xv = x[u];
        } else {
          bv = b[u][i];
          xv = x[u][i];
        }
        const double v = in[u] ? a.gamma1 * (axb[u] + bv) + a.gamma2 * (axa[u] + xv)
                               : bv + axb[u];
        sb[u] = fma(bv, bv, sb[u]);
        sa[u] = fma(v - axa[u], v - axa[u], sa[u]);
        if constexpr (V == 1) o = v;
        else o[i] = v;
      }
      if (t < ncr)
        __builtin_nontemporal_store(o, reinterpret_cast<vec*>(a.xa_out + t * k) + e);
    }
  }
#pragma unroll
  for (int u = 0; u < kPostRows; ++u) {
#pragma unroll
    for (int m = 1; m < L; m <<= 1) {
      sb[u] += shfl_xor_d(sb[u], m);
      sa[u] += shfl_xor_d(sa[u], m);
    }
    const int64_t t = row0 + u * kR;
    if (l == 0 && t < ncr) {
      a.spread_b[t] = sqrt(sb[u] / k);
      a.spread_a[t] = sqrt((in[u] ? sa[u] : sb[u]) / k);
    }
  }
}

template <int V>
int post_launch(const dk_post_args* a, int64_t ncr, hipStream_t s) {
  const int n = a->k / V;  // accesses a row
#define DK_POST(L)                                                                       \
  k_post<L, V><<<(unsigned)((ncr + kThreads / L * kPostRows - 1) / (kThreads / L * kPostRows)), \
                 kThreads, 0, s>>>(*a)
  // lanes a row: the power of two that holds the row in one access a lane
  if (n <= 4) DK_POST(4);
  else if (n <= 8) DK_POST(8);
  else if (n <= 16) DK_POST(16);
  else if (n <= 32) DK_POST(32);
  else DK_POST(64);
#undef DK_POST
  return (int)hipGetLastError();
}

// Coupler block xb_atm[((nn nx + i) ny + j) ens + e] <-> state
// xb[((j nx + i) n_max + n0 + nn) ens_max + e0 + e].  A copy, bound by HBM: a
// block takes kThreads * kStructVecs accesses of one (level, latitude) plane in
// coupler order, so the coupler's side is fully coalesced and the state's
// contiguous over the members of a (row, column).  V = 2: 16-byte accesses
// (even member counts and starts, aligned arrays).  The plane's indices come
// from scalar divisions and one 32-bit division an access remains; three
// 64-bit divisions a value and 8-byte accesses ran at 4.2 TB/s (one 3-D
// variable of 1 degree, 32 levels, 32 members, 1.06 GB: 250 us in, 279 out; now
// 207 and 200).
constexpr int kStructVecs = 4;

template <bool TO_STATE, int V>
__global__ __launch_bounds__(kThreads) void k_struct_ens(int32_t ens, int32_t nx, int32_t ny,
                                                         int32_t ens_max, int32_t n_max,
                                                         int32_t e0, int32_t n0, uint32_t chunks,
                                                         const double* __restrict__ src,
                                                         double* __restrict__ dst) {
  typedef typename VecOf<V>::type vec;
  const uint32_t plane = blockIdx.x / chunks, chunk = blockIdx.x - plane * chunks;
  const uint32_t nn = plane / (uint32_t)nx, i = plane - nn * (uint32_t)nx;
  const uint32_t ev = (uint32_t)(ens / V);
  const int64_t pv = (int64_t)ny * ev;  // accesses of the plane
  const int64_t t0 = (int64_t)chunk * (kThreads * kStructVecs) + threadIdx.x;
  int64_t at[kStructVecs], st[kStructVecs];
  vec v[kStructVecs];
#pragma unroll
  for (int u = 0; u < kStructVecs; ++u) {
    int64_t t = t0 + u * kThreads;
    t = t < pv ? t : pv - 1;
    const uint64_t j = pv <= 0xFFFFFFFFll ? (uint32_t)t / ev : (uint64_t)t / ev;
    const uint32_t e = (uint32_t)(t - (int64_t)(j * ev)) * V;
    at[u] = ((int64_t)plane * ny + (int64_t)j) * ens + e;
    st[u] = (((int64_t)j * nx + i) * n_max + n0 + nn) * ens_max + e0 + e;
    v[u] = __builtin_nontemporal_load(
        reinterpret_cast<const vec*>(src + (TO_STATE ? at[u] : st[u])));
  }
#pragma unroll
  for (int u = 0; u < kStructVecs; ++u)
    if (t0 + u * kThreads < pv)
      __builtin_nontemporal_store(v[u], reinterpret_cast<vec*>(dst + (TO_STATE ? st[u] : at[u])));
}

template <bool TO_STATE, int V>
int struct_ens_launch(int32_t ens, int32_t n, int32_t nx, int32_t ny, int32_t ens_max,
                      int32_t n_max, int32_t e0, int32_t n0, const double* src, double* dst,
                      hipStream_t s) {
  constexpr int64_t kPer = kThreads * kStructVecs;
  const int64_t chunks = ((int64_t)ny * (ens / V) + kPer - 1) / kPer;
  // levels a launch: at most 2^24 blocks (a grid holds 2^32 threads)
  const int64_t lev = chunks * nx <= (1 << 24) ? (1 << 24) / (chunks * nx) : 1;
  for (int64_t k = 0; k < n; k += lev) {
    const int64_t m = n - k < lev ? n - k : lev;
    const int64_t skip = k * nx * ny * (int64_t)ens;  // coupler values of the levels before
    k_struct_ens<TO_STATE, V><<<(unsigned)(chunks * nx * m), kThreads, 0, s>>>(
        ens, nx, ny, ens_max, n_max, e0, n0 + (int32_t)k, (uint32_t)chunks,
        TO_STATE ? src + skip : src, TO_STATE ? dst : dst + skip);
    const int e = (int)hipGetLastError();
    if (e) return e;
  }
  return 0;
}

// Means: axb_atm[(nn nx + i) ny + j] <-> axb[(j nx + i) n_max + n0 + nn], a
// transpose of (nn, j) per latitude i through a 32 x 33 LDS tile so that
// both sides are read and written along their contiguous index.
template <bool TO_STATE>
__global__ __launch_bounds__(256) void k_struct_mean(int32_t n, int32_t nx, int32_t ny,
                                                     int32_t n_max, int32_t n0,
                                                     const double* __restrict__ src,
                                                     double* __restrict__ dst) {
  __shared__ double tile[32][33];
  const int j0 = blockIdx.x * 32, nn0 = blockIdx.y * 32, i = blockIdx.z;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  auto atm = [&](int nn, int j) { return ((int64_t)nn * nx + i) * ny + j; };
  auto st = [&](int nn, int j) { return ((int64_t)j * nx + i) * n_max + n0 + nn; };
  if (TO_STATE) {
    for (int y = ty; y < 32; y += 8) {
      const int nn = nn0 + y, j = j0 + tx;
      if (nn < n && j < ny) tile[y][tx] = src[atm(nn, j)];
    }
    __syncthreads();
    for (int y = ty; y < 32; y += 8) {
      const int j = j0 + y, nn = nn0 + tx;
      if (nn < n && j < ny) dst[st(nn, j)] = tile[tx][y];
    }
  } else {
    for (int y = ty; y < 32; y += 8) {
      const int j = j0 + y, nn = nn0 + tx;
      if (nn < n && j < ny) tile[tx][y] = src[st(nn, j)];
    }
    __syncthreads();
    for (int y = ty; y < 32; y += 8) {
      const int nn = nn0 + y, j = j0 + tx;
      if (nn < n && j < ny) dst[atm(nn, j)] = tile[y][tx];
    }
  }
}

}  // namespace

extern "C" int dk_struct_ens(int to_state, int32_t ens, int32_t n, int32_t nx, int32_t ny,
                             int32_t ens_max, int32_t n_max, int32_t e0, int32_t n0,
                             const double* src, double* dst, void* stream) {
  if ((int64_t)ens * n * nx * ny <= 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const bool wide = ens % 2 == 0 && ens_max % 2 == 0 && e0 % 2 == 0 &&
                    ((uintptr_t)src | (uintptr_t)dst) % 16 == 0;
#define DK_STRUCT(T, V) \
  struct_ens_launch<T, V>(ens, n, nx, ny, ens_max, n_max, e0, n0, src, dst, s)
  if (to_state) return wide ? DK_STRUCT(true, 2) : DK_STRUCT(true, 1);
  return wide ? DK_STRUCT(false, 2) : DK_STRUCT(false, 1);
#undef DK_STRUCT
}

extern "C" int dk_struct_mean(int to_state, int32_t n, int32_t nx, int32_t ny, int32_t n_max,
                              int32_t n0, const double* src, double* dst, void* stream) {
  if ((int64_t)n * nx * ny <= 0) return 0;
  if (nx > 65535) return (int)hipErrorInvalidValue;
  const dim3 grid((unsigned)((ny + 31) / 32), (unsigned)((n + 31) / 32), (unsigned)nx);
  hipStream_t s = (hipStream_t)stream;
  if (to_state) k_struct_mean<true><<<grid, 256, 0, s>>>(n, nx, ny, n_max, n0, src, dst);
  else k_struct_mean<false><<<grid, 256, 0, s>>>(n, nx, ny, n_max, n0, src, dst);
  return (int)hipGetLastError();
}

extern "C" int dk_update_f64(const dk_update_args* u, void* stream) {
  if (u->ncol <= 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const int k = u->k;
  if (k < 2 || k > 64 || !u->xa32) return (int)hipErrorInvalidValue;
  if (k <= 16) k_update_f64<16><<<u->ncol, kThreads, 0, s>>>(*u);
  else if (k <= 32) k_update_f64<32><<<u->ncol, kThreads, 0, s>>>(*u);
  else k_update_f64<64><<<u->ncol, kThreads, 0, s>>>(*u);
  return (int)hipGetLastError();
}

extern "C" int dk_cube_centres(int32_t nlat, int32_t nlon, int32_t cube_n, int32_t step,
                               const float* grid_lat, const float* grid_lon, float* ca_lat,
                               float* ca_lon, void* stream) {
  if (nlat < 1 || nlon < 1 || cube_n < 1 || step < 1) return (int)hipErrorInvalidValue;
  const int n = (nlat + step - 1) / step + (nlon + step - 1) / step;
  k_cube_centres<<<(n + 255) / 256, 256, 0, (hipStream_t)stream>>>(nlat, nlon, cube_n, step,
                                                                   grid_lat, grid_lon, ca_lat,
                                                                   ca_lon);
  return (int)hipGetLastError();
}

extern "C" int dk_post(const dk_post_args* a, void* stream) {
  const int64_t ncr = (int64_t)a->nlat * a->nlon * a->nrow;
  if (ncr <= 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const uintptr_t at = (uintptr_t)a->xb | (uintptr_t)a->xa | (uintptr_t)a->xa_out;
  return a->k % 2 == 0 && at % 16 == 0 ? post_launch<2>(a, ncr, s) : post_launch<1>(a, ncr, s);
}
