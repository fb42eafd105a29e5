// Batched LETKF form, one wavefront per local analysis.
//
// A persistent grid of one-wave workgroups drains a queue of column chains
// (sorted by local obs count).  Each wave runs the whole analysis of every
// column of its chain with the KP x KP working matrix held in registers in
// the MFMA result layout: lane (g = l/16, c = l%16) owns, for each column
// slot j = J*16 + c (J < KP/16), the rows row(I, r, g) (I < KP/16, r < 4),
// where row() is I*16 + 4g + r after a 16x16x32 half-precision Gram and
// I*16 + 4r + g after an FP64 16x16x4 product.  Because M = C + (k-1)/rho I
// is symmetric, these registers are also the A operand of M V, and the tiles
// of W come out in the A-operand layout of the update, so the only LDS state
// is the eigenvector basis V (the warm start of the next column).
//
//   Gram      C = Yhat Yhat^T, Yhat = Yb sqrt(R^-1 rloc): FP16/BF16 MFMA with
//             FP32 accumulation and the split hi + lo (x3), FP16 scaled per
//             analysis by a power of two; or FP64 MFMA.  b = Yhat^T
//             (sqrt(R^-1 rloc) dep) in FP64 (letkf_core.F90:58-79, 146-195).
//   warm      A0 = M V_prev on FP64 MFMA for all but the first column of a
//             chain; M is positive definite, so V stays a full basis.
//   Jacobi    one-sided, FP64, pairs (columns J = 2P, 2P+1 of a lane group)
//             rotated in parallel; the round ordering pairs the two halves of
//             every block of positions, recursively (KP - 1 rounds a sweep),
//             with only the bottom columns moving between rounds.
//   W, wbar   W = V diag(sqrt((k-1)/lambda)) V^T, wbar = V diag(1/lambda) V^T b
//             on FP64 MFMA; trans = W + wbar 1^T (letkf_core.F90:129-225).
//   update    Xa = trans^T Xb' + xbar_b, mean, re-centre, RTPS (xb_2_xa,
//             letkf_compute.F90:261-299) on FP64 MFMA.
#include <cstring>

#include "letkf_device.h"
#include "letkf_kernels.h"
#include "letkf_wave.h"

using namespace dida;

namespace {

// MODE: kModeColumn (one analysis per column, fused update), kModeVertical
// (one per column and level cube, fused update of the cube's rows) or
// kModeTransOut (one per horizontal cube, transform written to HBM)
// Returns whether the analysis's eigenvectors may warm-start the next one:
// not when it was not finite (its transform is NaN) or its eigensolve hit the
// sweep cap (its basis is not orthonormal, and A = M V_prev would then not
// carry the eigenvectors of M).
template <int KP, int GRAM, int MODE, bool FULLV>
__device__ bool wave_column(const dk_batched_args& a, int64_t col, int cube, bool warm,
                            WSmem<KP, FULLV>& sm, Wave<KP, GRAM>& w) {
  constexpr int NJ = Wave<KP, GRAM>::NJ;
  constexpr int NQ = Wave<KP, GRAM>::NQ;
  constexpr bool VERT = MODE == kModeVertical;
  const int lane = threadIdx.x, g = lane >> 4, c = lane & 15;
  const int k = a.k;
  PhaseClock clk(a.phase_clk);
  const int64_t off = a.offset[col] - a.base;
  int p = a.nobsl[col];
  p = p < 0 ? 0 : (p > a.max_p ? a.max_p : p);
  if (off < 0 || off + p > a.capacity) p = 0;
  // analysis id; the cube's centre ln p with vertical localisation
  const int64_t aid = VERT ? col * a.ncube + cube : col;
  const double clnp = VERT ? a.cube_lnp[aid] : 0.0;
  int lo = 0, hi = p;
  if (VERT && a.sel_key) vertical_range(a, off, p, clnp, lo, hi);

  w.template gram<VERT>(a, off + lo, hi - lo, clnp, sm);
  const double km1 = (double)(k - 1);
  w.shift(k, km1 / a.rho);
  clk.mark(DK_PHASE_GRAM);
  if (FULLV && warm) w.warm(sm);
  clk.mark(DK_PHASE_WARM);
  bool conv;
  const int sweeps = w.jacobi(a.tol, a.max_sweeps, a.predict != 0, &conv);
  clk.mark(DK_PHASE_JACOBI);

  double4_t T[NJ][NJ], wb[NJ];
  const bool bad = eig_transform<KP, GRAM, FULLV>(w, sm, km1, T, wb);
  const double nan = __builtin_nan("");
#pragma unroll
  for (int I = 0; I < NJ; ++I)
#pragma unroll
    for (int I2 = 0; I2 < NJ; ++I2)
#pragma unroll
      for (int r = 0; r < 4; ++r) T[I][I2][r] = bad ? nan : T[I][I2][r] + wb[I][r];
  if (a.info && lane == 0) a.info[aid] = bad ? -2 : (conv ? sweeps : -1);
  if (a.wbar_out && c == 0)
#pragma unroll
    for (int I = 0; I < NJ; ++I)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = rowB(I, r, g);
        if (i < k) a.wbar_out[(aid - a.trans_aid0) * k + i] = wb[I][r];
      }
  clk.mark(DK_PHASE_TRANSFORM);
  if constexpr (MODE == kModeTransOut) {
    // horizontal cubes: the transform goes to HBM; a per-column kernel
    // applies the mean of the covering cubes' transforms
    double* tr = a.trans_out + (aid - a.trans_aid0) * k * k;
#pragma unroll
    for (int I = 0; I < NJ; ++I)
#pragma unroll
      for (int I2 = 0; I2 < NJ; ++I2)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = rowB(I, r, g), e = I2 * 16 + c;
          if (i < k && e < k) tr[i + (int64_t)e * k] = T[I][I2][r];
        }
    return conv && !bad;
  }

  // update: all nrow rows of the column, or with vertical localisation the
  // cube's list of rows
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
                              (int64_t)ilat + (int64_t)a.grid_nlat * ilon, T, rmap, nr);
  } else {
    update_rows<KP, VERT>(k, a.nrow, a.xb, a.axb, a.xa, a.axa, a.rtps != 0, a.rtps_alpha, col,
                          T, rmap, nr);
  }
  clk.mark(DK_PHASE_UPDATE);
  (void)NQ;
  return conv && !bad;
}

// The plain form: one wavefront per analysis of [aid0, aid0 + gridDim.x) in
// grid order, every eigensolve cold (no chains), transform to HBM.  Two
// wavefronts a SIMD (256 registers each: the few spills cost less than the
// latency a second wavefront hides; config 2: 210 -> 198 ms a sweep).
template <int KP>
__global__ __launch_bounds__(64, 2) void k_letkf_plain(dk_batched_args a, int32_t aid0) {
  __shared__ WSmem<KP, false> sm;
  Wave<KP, DK_GRAM_FP64> w;
  wave_column<KP, DK_GRAM_FP64, kModeTransOut, false>(a, (int64_t)aid0 + blockIdx.x, 0, false,
                                                       sm, w);
}

// First longitude of stripe g of n groups (groups of whole longitudes).
__device__ __forceinline__ int stripe_lo(int g, int n, int nlon) {
  return (int)(((int64_t)g * nlon) / n);
}

// One wavefront per SIMD: the fused analysis needs about 490 registers
// (at 256, two waves a SIMD, it spills 300-700 of them and runs slower).  Up to
// 32 members two fit (204 to 238 registers, where unbounded instances took 257
// and ran one: vertical localisation, k = 28, 14.1 -> 10.8 ms); bounded to
// three they spill up to 70 (1 degree, k = 32, 4.57 -> 4.89 ms).
template <int KP, int GRAM, int MODE>
__global__ __launch_bounds__(64, KP == 32 ? 2 : 1) void k_letkf_wave(dk_batched_args a) {
  __shared__ WSmem<KP, true> sm;
  Wave<KP, GRAM> w;
  const int lane = threadIdx.x;
  // one queue (ngroup 0) or ngroup group queues, own group first
  const int ng = a.ngroup > 0 ? a.ngroup : 1;
  const int g0 = a.ngroup > 0 ? (int)(blockIdx.x % (unsigned)ng) : 0;
  int s = 0, gq = g0, beg = 0;
  int cnt = a.bucketed ? (int)*a.nchain_dev : a.nchain;
  if (a.ngroup > 0) {
    beg = stripe_lo(gq, ng, a.nlon) * a.chains_per_lon;
    cnt = stripe_lo(gq + 1, ng, a.nlon) * a.chains_per_lon - beg;
  }
  for (;;) {
    int item = 0;
    if (lane == 0) item = atomicAdd(a.queue_head + gq, 1);
    item = __shfl(item, 0, kWave);
    if (item >= cnt) {
      if (++s >= ng) break;
      gq = (g0 + s) % ng;
      beg = stripe_lo(gq, ng, a.nlon) * a.chains_per_lon;
      cnt = stripe_lo(gq + 1, ng, a.nlon) * a.chains_per_lon - beg;
      continue;
    }
    const int chain = a.queue ? a.queue[beg + item] : beg + item;
    int ilon, lat0, lat1;
    if (a.bucketed) {
      const int c0 = a.chain_col0[chain];
      ilon = c0 / a.nlat;
      lat0 = c0 - ilon * a.nlat;
      lat1 = lat0 + a.chain_ncol[chain];
    } else {
      ilon = chain / a.chains_per_lon;
      lat0 = (chain % a.chains_per_lon) * a.chain_len;
      lat1 = min(lat0 + a.chain_len, a.nlat);
    }
    // an analysis warm-starts from the previous one of its chain unless that
    // one was not finite or did not converge
    bool prev_ok = false;
    for (int ilat = lat0; ilat < lat1; ++ilat) {
      const int64_t col = (int64_t)ilon * a.nlat + ilat;
      if constexpr (MODE == kModeVertical) {
        // the cubes of a column in alternating order, so that every analysis
        // warm-starts from the adjacent cube of its column or the same cube
        // of the previous column
        const bool down = ((ilat - lat0) & 1) != 0;
        for (int t = 0; t < a.ncube; ++t)
          prev_ok = wave_column<KP, GRAM, MODE, true>(a, col, down ? a.ncube - 1 - t : t,
                                                      a.warm_start && prev_ok, sm, w);
      } else {
        prev_ok = wave_column<KP, GRAM, MODE, true>(a, col, 0, a.warm_start && prev_ok, sm, w);
      }
    }
  }
}

// Sort key of chain c: 2^32 - 1 - cost, so that an ascending radix sort puts
// the most expensive chains first.  Cost of a column ~ its local obs count
// (Gram) + 10 k (eigensolve, transform and update), times the number of
// vertical cubes.
__global__ void k_chain_keys(dk_batched_args a, uint32_t* key, int32_t* id) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= a.nchain) return;
  int ilon, lat0, lat1;
  if (a.bucketed) {
    // a.nchain entries are sorted; those past the built chains go last
    if (c >= (int)*a.nchain_dev) {
      key[c] = 0xFFFFFFFFu;
      id[c] = c;
      return;
    }
    const int c0 = a.chain_col0[c];
    ilon = c0 / a.nlat;
    lat0 = c0 - ilon * a.nlat;
    lat1 = lat0 + a.chain_ncol[c];
  } else {
    ilon = c / a.chains_per_lon;
    lat0 = (c % a.chains_per_lon) * a.chain_len;
    lat1 = min(lat0 + a.chain_len, a.nlat);
  }
  double cost = 0.0;
  for (int ilat = lat0; ilat < lat1; ++ilat)
    cost += (double)a.nobsl[(int64_t)ilon * a.nlat + ilat] + 10.0 * a.k;
  if (a.ncube > 0) cost *= a.ncube;
  key[c] = 0xFFFFFFFFu - (uint32_t)fmin(cost, 4.0e9);
  id[c] = c;
}

__device__ __forceinline__ int bucket_of(int p, const dk_chain_build_args& a) {
  int b = 0;
  while (b + 1 < a.nbucket && p >= a.lo[b + 1]) ++b;
  return b;
}

// One wavefront per longitude: the chains of its latitudes, counted (kWrite
// false) or written.  A chain is a piece of a run of columns of one bucket:
// the run is cut every len[bucket] columns from its start.  Lane t holds
// latitudes [t per, (t + 1) per): the run start entering each lane comes
// from a max-scan of the lanes' last run starts, a chain starts where the
// offset from its run start is a multiple of the length, and a chain ends at
// the next chain start (a suffix min-scan of the lanes' first ones).
template <bool kWrite>
__global__ __launch_bounds__(256) void k_chain_build(dk_chain_build_args a) {
  const int lane = threadIdx.x & 63;
  const int ilon = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
  if (ilon >= a.nlon) return;
  const int n = a.nlat;
  const int32_t* p = a.nobsl + (int64_t)ilon * n;
  const int per = (n + kWave - 1) / kWave;
  const int i0 = min(lane * per, n), i1 = min(i0 + per, n);
  const int prevb = i0 > 0 && i0 < n ? bucket_of(p[i0 - 1], a) : -1;
  // the lane's last run start (or -1), then the one entering the lane
  int last = -1;
  int b = prevb;
  for (int i = i0; i < i1; ++i) {
    const int bi = bucket_of(p[i], a);
    if (bi != b) last = i;
    b = bi;
  }
  int inc = last;
  for (int o = 1; o < kWave; o <<= 1) {
    const int t = __shfl_up(inc, o, kWave);
    if (lane >= o) inc = max(inc, t);
  }
  int rs = __shfl_up(inc, 1, kWave);
  if (lane == 0) rs = -1;
  // chain starts of the lane: count and first
  int cnt = 0, first = n;
  {
    int r = rs;
    b = prevb;
    for (int i = i0; i < i1; ++i) {
      const int bi = bucket_of(p[i], a);
      if (bi != b) r = i;
      b = bi;
      const int len = a.len[bi] > 0 ? a.len[bi] : 1;
      if ((i - r) % len == 0) {
        first = min(first, i);
        ++cnt;
      }
    }
  }
  int before = cnt;  // inclusive scan of the counts
  for (int o = 1; o < kWave; o <<= 1) {
    const int t = __shfl_up(before, o, kWave);
    if (lane >= o) before += t;
  }
  const int total = __shfl(before, kWave - 1, kWave);
  before -= cnt;
  if (!kWrite) {
    if (lane == 0) a.line_cnt[ilon] = total;
    return;
  }
  // the first chain start above the lane (n if none)
  int nx = first;
  for (int o = 1; o < kWave; o <<= 1) {
    const int t = __shfl_down(nx, o, kWave);
    if (lane + o < kWave) nx = min(nx, t);
  }
  nx = __shfl_down(nx, 1, kWave);
  if (lane == kWave - 1) nx = n;
  const int64_t out = a.line_off[ilon] + before;
  int r = rs, prev = -1, k = 0;
  b = prevb;
  for (int i = i0; i < i1; ++i) {
    const int bi = bucket_of(p[i], a);
    if (bi != b) r = i;
    b = bi;
    const int len = a.len[bi] > 0 ? a.len[bi] : 1;
    if ((i - r) % len == 0) {
      if (prev >= 0) a.chain_ncol[out + k - 1] = i - prev;
      a.chain_col0[out + k] = ilon * n + i;
      prev = i;
      ++k;
    }
  }
  if (prev >= 0) a.chain_ncol[out + k - 1] = nx - prev;
}

// Grouped queue: chain (ilon, latchain) of stripe g goes to position
// stripe_lo(g) cpl + latchain * width(g) + (ilon - stripe_lo(g)).
__global__ void k_chain_groups(dk_batched_args a, int32_t* order) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= a.nchain) return;
  const int cpl = a.chains_per_lon, ng = a.ngroup;
  const int ilon = c / cpl, lc = c % cpl;
  int g = 0;
  while (g + 1 < ng && stripe_lo(g + 1, ng, a.nlon) <= ilon) ++g;
  const int l0 = stripe_lo(g, ng, a.nlon), wdt = stripe_lo(g + 1, ng, a.nlon) - l0;
  order[l0 * cpl + lc * wdt + (ilon - l0)] = c;
}

template <int KP, int GRAM>
int wlaunch(const dk_batched_args* a, int nblocks, hipStream_t s) {
  if (a->ncube > 0) k_letkf_wave<KP, GRAM, kModeVertical><<<nblocks, 64, 0, s>>>(*a);
  else if (a->trans_out) k_letkf_wave<KP, GRAM, kModeTransOut><<<nblocks, 64, 0, s>>>(*a);
  else k_letkf_wave<KP, GRAM, kModeColumn><<<nblocks, 64, 0, s>>>(*a);
  return (int)hipGetLastError();
}

template <int KP, int GRAM>
int wocc() {
  int nb = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_letkf_wave<KP, GRAM, kModeColumn>, 64,
                                                   0))
    return 1;
  return nb > 0 ? nb : 1;
}

template <int KP>
int wdispatch(const dk_batched_args* a, int nblocks, hipStream_t s) {
  switch (a->gram) {
    case DK_GRAM_FP64: return wlaunch<KP, DK_GRAM_FP64>(a, nblocks, s);
    case DK_GRAM_BF16X3: return wlaunch<KP, DK_GRAM_BF16X3>(a, nblocks, s);
    case DK_GRAM_FP16X3: return wlaunch<KP, DK_GRAM_FP16X3>(a, nblocks, s);
    case DK_GRAM_BF16: return wlaunch<KP, DK_GRAM_BF16>(a, nblocks, s);
  }
  return (int)hipErrorInvalidValue;
}

template <int KP>
int wocc_dispatch(int gram) {
  switch (gram) {
    case DK_GRAM_FP64: return wocc<KP, DK_GRAM_FP64>();
    case DK_GRAM_BF16X3: return wocc<KP, DK_GRAM_BF16X3>();
    case DK_GRAM_FP16X3: return wocc<KP, DK_GRAM_FP16X3>();
    case DK_GRAM_BF16: return wocc<KP, DK_GRAM_BF16>();
  }
  return 1;
}

}  // namespace

extern "C" int dk_wave_blocks_per_cu(int k, int gram) {
  if (k <= 32) return wocc_dispatch<32>(gram);
  return wocc_dispatch<64>(gram);
}

extern "C" int dk_letkf_plain_wave(const dk_core_args* c, void* stream) {
  if (c->nanal <= 0) return 0;
  if (c->k < 2 || c->k > 64 || c->gram != DK_GRAM_FP64 || !c->idx) return (int)hipErrorInvalidValue;
  dk_batched_args a;
  memset(&a, 0, sizeof a);
  a.k = c->k;
  a.ldy = c->k <= 32 ? 32 : 64;
  a.max_sweeps = c->max_sweeps;
  a.max_p = c->max_p;
  a.predict = c->predict;
  a.rho = c->rho;
  a.tol = c->tol;
  a.capacity = c->capacity;
  a.offset = c->offset;
  a.nobsl = c->nobsl;
  a.idx = c->idx;
  a.rloc = c->rloc;
  a.yb = c->yb;
  a.rinv = c->rinv;
  a.dep = c->dep;
  a.info = c->info;
  a.base = c->base;
  a.trans_out = c->trans;
  a.trans_aid0 = c->aid0;
  a.wbar_out = c->wbar;
  hipStream_t s = (hipStream_t)stream;
  if (c->k <= 32) k_letkf_plain<32><<<c->nanal, 64, 0, s>>>(a, c->aid0);
  else k_letkf_plain<64><<<c->nanal, 64, 0, s>>>(a, c->aid0);
  return (int)hipGetLastError();
}

extern "C" int dk_chain_groups(const dk_batched_args* a, int32_t* order, void* stream) {
  if (a->nchain <= 0 || a->ngroup <= 0) return 0;
  k_chain_groups<<<(a->nchain + 255) / 256, 256, 0, (hipStream_t)stream>>>(*a, order);
  return (int)hipGetLastError();
}

extern "C" int dk_chain_build(const dk_chain_build_args* a, int write, void* stream) {
  if (a->nlon <= 0) return 0;
  if (a->nbucket < 1 || a->nbucket > DK_NBUCKET) return (int)hipErrorInvalidValue;
  const unsigned nb = (unsigned)((a->nlon + 3) / 4);
  if (write) k_chain_build<true><<<nb, 256, 0, (hipStream_t)stream>>>(*a);
  else k_chain_build<false><<<nb, 256, 0, (hipStream_t)stream>>>(*a);
  return (int)hipGetLastError();
}

extern "C" int dk_chain_keys(const dk_batched_args* a, uint32_t* key, int32_t* id, void* stream) {
  if (a->nchain <= 0) return 0;
  k_chain_keys<<<(a->nchain + 255) / 256, 256, 0, (hipStream_t)stream>>>(*a, key, id);
  return (int)hipGetLastError();
}

extern "C" int dk_letkf_wave(const dk_batched_args* a, int nblocks, void* stream) {
  if (a->nchain <= 0) return 0;
  if (a->k < 2 || a->k > 64) return (int)hipErrorInvalidValue;
  if (a->ldy != (a->k <= 32 ? 32 : 64)) return (int)hipErrorInvalidValue;
  if (a->gram == DK_GRAM_FP64 ? !a->yb : !a->yb32) return (int)hipErrorInvalidValue;
  hipStream_t s = (hipStream_t)stream;
  if (a->k <= 32) return wdispatch<32>(a, nblocks, s);
  return wdispatch<64>(a, nblocks, s);
}
