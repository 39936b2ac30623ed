// All-pairs Coulomb sums for point-charge solutes.
//   potential  phi(j) = sum_i q_i / |r_j - r_i|            (mkrhs.f90:102-114)
//   field      E(j)   = sum_i q_i (r_j - r_i) / |r_j - r_i|^3  (efld.f90:98-114)
// Each lane owns one target; sources stream through LDS.  Work comes as a
// table of tiles (targets tb..te-1, at most 64, and sources sb..se-1): for a
// batch of molecules every tile stays inside one molecule, so each sums only
// its own molecule's charges.
// The potential kernel can return the field of the same sources as well
// (the solute field at the cavity points that the forces contract with
// zeta), which costs one all-pairs pass less than a separate field kernel.
// 1/r comes from the hardware reciprocal square root refined by one
// third-order step (relative error a few ulp), which replaces an IEEE sqrt
// and divide per pair.
// When there are few targets (the field of the cavity charges at the nuclei)
// the sources of a target tile are split into chunks, one tile each, and
// the partial fields are summed afterwards in chunk order, so results are
// deterministic.
#include "ddx_device.hpp"
#include "ddx_kernels.hpp"

#include <algorithm>
#include <mutex>

namespace ddx {
namespace {

constexpr int kCT = 256;          // threads per workgroup, sources per LDS tile
constexpr int kTW = 2 * kCT;      // targets per tile of the uniform tiling: two per thread
constexpr int kFW = kWave;        // targets per tile of the table-driven kernels: one per lane

// 1/sqrt(x) for x > 0: v_rsq_f64 (relative error below 2^-24 on gfx950)
// and one third-order correction: with e = 1 - x y^2, y (1 + e/2 + 3e^2/8)
// leaves a relative error of order e^3 plus rounding (about 1 ulp)
__device__ __forceinline__ double rsqrt_nr(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y, e * fma(0.375, e, 0.5), y);
}

// phi(j) and, with FIELD, the field ef(:, j) of the same sources, from one
// evaluation of 1/r per pair; one wave per tile (tb, te, sb, se) of at most
// kFW targets, one per lane, the sources through LDS kFW at a time and added
// in order.
//   Bound by FP64 issue: 18 operations and one v_rsq_f64 a pair, four pairs in
// flight (a bound of 6 or 8 waves per SIMD costs the unrolled loop its
// registers: 610 and 698 us against 601 at 2000 atoms).  One-wave workgroups of
// 64 targets spread over the chip whatever their number; with 512 targets to a
// workgroup of four waves (two per thread) 642 atoms made 61 workgroups.  That
// form -> this one, in us (lmax, grid): 60 atoms (6, 302) 9.5 -> 5.9; 259 (6,
// 110) 30 -> 17; 642 (6, 110) 71 -> 39; 200 (10, 1202) 27.5 -> 24.0; 1000 (8,
// 590) 202 -> 195; 2000 (8, 590) 614 -> 601.  From there on either form may win
// by what its last workgroups leave idle: with the field 2000 -> 1850 us at 3500
// atoms, 4970 -> 4740 at 6000, 5010 -> 5110 at 6400, 9600 -> 9160 at 12 000 (302
// points); without 1434 -> 1345, 3676 -> 3610, 3855 -> 3950, 7050 -> 6925.  Two
// targets per lane in one wave: 70 us at 642 atoms, 755 at 2000, 5000 at 6400.
template <bool FIELD>
__global__ __launch_bounds__(kFW) void k_potential(const int4 *__restrict__ tiles,
                                                   const double *__restrict__ q,
                                                   const double4 *__restrict__ src,
                                                   const double *__restrict__ trg,
                                                   double *__restrict__ phi,
                                                   double *__restrict__ ef) {
  __shared__ double4 tile[kFW];
  const int4 tl = tiles[blockIdx.x];
  const int j = tl.x + (int)threadIdx.x, jc = min(j, tl.y - 1);
  const double ax = trg[3 * (size_t)jc], ay = trg[3 * (size_t)jc + 1],
               az = trg[3 * (size_t)jc + 2];
  double va = 0.0, e0 = 0.0, e1 = 0.0, e2 = 0.0;
  int i = min(tl.z + (int)threadIdx.x, tl.w - 1);
  double4 s = make_double4(0.0, 0.0, 0.0, 0.0);
  double qi = 0.0;
  if (tl.z < tl.w) {
    s = src[i];
    qi = q[i];
  }
  for (int i0 = tl.z; i0 < tl.w; i0 += kFW) {
    wave_lds_sync();   // the previous sources are read
    tile[threadIdx.x] = make_double4(s.x, s.y, s.z, qi);
    wave_lds_sync();
    i = min(i + kFW, tl.w - 1);   // the next sources, loaded under this block's sums
    s = src[i];
    qi = q[i];
    const int cnt = min(kFW, tl.w - i0);
#pragma unroll 4
    for (int k = 0; k < cnt; ++k) {
      const double4 sk = tile[k];
      const double dx = ax - sk.x, dy = ay - sk.y, dz = az - sk.z;
      const double y = rsqrt_nr(dx * dx + dy * dy + dz * dz);
      const double qy = sk.w * y;
      va = va + qy;
      if (FIELD) {
        const double f = qy * (y * y);
        e0 = e0 + f * dx;
        e1 = e1 + f * dy;
        e2 = e2 + f * dz;
      }
    }
  }
  if (j < tl.y) {
    phi[j] = va;
    if (FIELD) {
      ef[3 * (size_t)j] = e0;
      ef[3 * (size_t)j + 1] = e1;
      ef[3 * (size_t)j + 2] = e2;
    }
  }
}

// fields of the sources sb..se-1 of tile tl at its targets tb..te-1 (two per
// thread, targets tb + t and tb + t + kCT); the sums of thread t come back in
// e[0..2] (first target) and e[3..5] (second), zero for targets past te
__device__ __forceinline__ void field_tile(const int4 tl, const double *__restrict__ q,
                                           const double *__restrict__ src,
                                           const double *__restrict__ trg, double4 *tile,
                                           double e[6]) {
  const int j0 = tl.x + threadIdx.x, j1 = j0 + kCT;
  double ax = 0.0, ay = 0.0, az = 0.0, bx = 0.0, by = 0.0, bz = 0.0;
  if (j0 < tl.y) {
    ax = trg[3 * (size_t)j0];
    ay = trg[3 * (size_t)j0 + 1];
    az = trg[3 * (size_t)j0 + 2];
  }
  if (j1 < tl.y) {
    bx = trg[3 * (size_t)j1];
    by = trg[3 * (size_t)j1 + 1];
    bz = trg[3 * (size_t)j1 + 2];
  }
  double ea0 = 0.0, ea1 = 0.0, ea2 = 0.0, eb0 = 0.0, eb1 = 0.0, eb2 = 0.0;
  for (int i0 = tl.z; i0 < tl.w; i0 += kCT) {
    int i = i0 + threadIdx.x;
    if (i < tl.w)
      tile[threadIdx.x] = make_double4(src[3 * (size_t)i], src[3 * (size_t)i + 1],
                                       src[3 * (size_t)i + 2], q[i]);
    __syncthreads();
    int cnt = min(kCT, tl.w - i0);
    for (int k = 0; k < cnt; ++k) {
      const double4 s = tile[k];
      {
        const double dx = ax - s.x, dy = ay - s.y, dz = az - s.z;
        const double y = rsqrt_nr(dx * dx + dy * dy + dz * dz);
        const double f = s.w * (y * y * y);
        ea0 = ea0 + f * dx;
        ea1 = ea1 + f * dy;
        ea2 = ea2 + f * dz;
      }
      {
        const double dx = bx - s.x, dy = by - s.y, dz = bz - s.z;
        const double y = rsqrt_nr(dx * dx + dy * dy + dz * dz);
        const double f = s.w * (y * y * y);
        eb0 = eb0 + f * dx;
        eb1 = eb1 + f * dy;
        eb2 = eb2 + f * dz;
      }
    }
    __syncthreads();
  }
  if (j0 >= tl.y) ea0 = ea1 = ea2 = 0.0;
  if (j1 >= tl.y) eb0 = eb1 = eb2 = 0.0;
  e[0] = ea0;
  e[1] = ea1;
  e[2] = ea2;
  e[3] = eb0;
  e[4] = eb1;
  e[5] = eb2;
}

// ef of the targets of a target tile = sum of the partials of its chunk
// tiles b0 .. b1-1 (kTW targets each), in a fixed order: each
// target's chunks are split over kRq threads (chunk c to thread c mod kRq),
// whose sums meet in LDS in thread order.  blockIdx.y picks the slice of
// kCT / kRq targets.
constexpr int kRq = 8;
__device__ __forceinline__ void field_reduce(int b0, int b1, int tb, int te,
                                             const double *__restrict__ part,
                                             double *__restrict__ ef, double (*red)[3]) {
  const int r = threadIdx.x % kRq;
  const int t = blockIdx.y * (kCT / kRq) + threadIdx.x / kRq;
  double e0 = 0.0, e1 = 0.0, e2 = 0.0;
  for (int b = b0 + r; b < b1; b += kRq) {
    const size_t o = ((size_t)b * kTW + t) * 3;
    e0 += part[o];
    e1 += part[o + 1];
    e2 += part[o + 2];
  }
  red[threadIdx.x][0] = e0;
  red[threadIdx.x][1] = e1;
  red[threadIdx.x][2] = e2;
  __syncthreads();
  const int j = tb + t;
  if (r == 0 && j < te) {
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
    for (int k = 0; k < kRq; ++k) {
      s0 += red[threadIdx.x + k][0];
      s1 += red[threadIdx.x + k][1];
      s2 += red[threadIdx.x + k][2];
    }
    ef[3 * (size_t)j] = s0;
    ef[3 * (size_t)j + 1] = s1;
    ef[3 * (size_t)j + 2] = s2;
  }
}

// The tiled field (few targets per molecule: the nuclei): one wave per tile
// of at most kFW targets, one per lane, the tile's sources through LDS kFW at
// a time; part[(b kFW + t) 3] holds tile b's partial field at target t.
__global__ __launch_bounds__(kFW) void k_field_w(const int4 *__restrict__ tiles,
                                                 const double *__restrict__ q,
                                                 const double *__restrict__ src,
                                                 const double *__restrict__ trg,
                                                 double *__restrict__ part) {
  __shared__ double4 tile[kFW];
  const int4 tl = tiles[blockIdx.x];
  const int j = tl.x + (int)threadIdx.x;
  double ax = 0.0, ay = 0.0, az = 0.0;
  if (j < tl.y) {
    ax = trg[3 * (size_t)j];
    ay = trg[3 * (size_t)j + 1];
    az = trg[3 * (size_t)j + 2];
  }
  double e0 = 0.0, e1 = 0.0, e2 = 0.0;
  for (int i0 = tl.z; i0 < tl.w; i0 += kFW) {
    const int i = i0 + (int)threadIdx.x;
    __syncthreads();   // the previous sources are read
    if (i < tl.w)
      tile[threadIdx.x] = make_double4(src[3 * (size_t)i], src[3 * (size_t)i + 1],
                                       src[3 * (size_t)i + 2], q[i]);
    __syncthreads();
    const int cnt = min(kFW, tl.w - i0);
    for (int k = 0; k < cnt; ++k) {
      const double4 sk = tile[k];
      const double dx = ax - sk.x, dy = ay - sk.y, dz = az - sk.z;
      const double y = rsqrt_nr(dx * dx + dy * dy + dz * dz);
      const double f = sk.w * (y * y * y);
      e0 = e0 + f * dx;
      e1 = e1 + f * dy;
      e2 = e2 + f * dz;
    }
  }
  if (j >= tl.y) e0 = e1 = e2 = 0.0;
  const size_t o = ((size_t)blockIdx.x * kFW + threadIdx.x) * 3;
  part[o] = e0;
  part[o + 1] = e1;
  part[o + 2] = e2;
}

// ef of the targets of group g = the partials of its tiles grp[g] ..
// grp[g+1]-1 (the source chunks of one target tile) in a fixed order: the
// chunks are split over kRw waves (chunk c to wave c mod kRw), lane t of each
// adding target t's, eight tiles loaded before they are added, and the waves'
// sums meet in LDS in wave order.  A tile's partials are one contiguous run of
// a wave's loads (with the lanes across the chunks they were 64 lines): 128 -> 44
// us at 2000 atoms (lmax 8, 590 points), 65 -> 27 at 1000.
constexpr int kRw = 4;
__global__ __launch_bounds__(kFW * kRw) void k_field_reduce_w(const int *__restrict__ grp,
                                                              const int4 *__restrict__ tiles,
                                                              const double *__restrict__ part,
                                                              double *__restrict__ ef) {
  __shared__ double red[kRw][3][kFW];
  const int b0 = grp[blockIdx.x], b1 = grp[blockIdx.x + 1];
  const int4 tl = tiles[b0];
  const int t = threadIdx.x % kFW, r = threadIdx.x / kFW;
  double e0 = 0.0, e1 = 0.0, e2 = 0.0;
  for (int b = b0 + r; b < b1; b += 8 * kRw) {
    double v[8][3];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const size_t o = ((size_t)min(b + u * kRw, b1 - 1) * kFW + t) * 3;
      v[u][0] = part[o];
      v[u][1] = part[o + 1];
      v[u][2] = part[o + 2];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (b + u * kRw < b1) {
        e0 += v[u][0];
        e1 += v[u][1];
        e2 += v[u][2];
      }
    }
  }
  red[r][0][t] = e0;
  red[r][1][t] = e1;
  red[r][2][t] = e2;
  __syncthreads();
  const int j = tl.x + t;
  if (r < 3 && j < tl.y) {   // wave r: component r
    double sum = 0.0;
#pragma unroll
    for (int k = 0; k < kRw; ++k) sum += red[k][r][t];
    ef[3 * (size_t)j + r] = sum;
  }
}

// The same field on a uniform tiling that needs no table: tile b covers
// target tile b / nchunk (kTW targets) and source chunk b % nchunk (`chunk`
// sources).  With one chunk the sums go straight to ef; with more, to
// part[(b kTW + t) 3], which k_field_reduce_uniform sums in chunk order.
__device__ __forceinline__ int4 uniform_tile(int b, int nchunk, int chunk, int ntrg, int nsrc) {
  const int tt = b / nchunk, c = b - tt * nchunk;
  const int tb = tt * kTW, sb = (int)min((long long)c * chunk, (long long)nsrc);
  return make_int4(tb, min(tb + kTW, ntrg), sb, (int)min((long long)sb + chunk, (long long)nsrc));
}

__global__ __launch_bounds__(kCT) void k_field_uniform(int ntrg, int nsrc, int nchunk, int chunk,
                                                       const double *__restrict__ q,
                                                       const double *__restrict__ src,
                                                       const double *__restrict__ trg,
                                                       double *__restrict__ part,
                                                       double *__restrict__ ef) {
  __shared__ double4 tile[kCT];
  double e[6];
  const int4 tl = uniform_tile(blockIdx.x, nchunk, chunk, ntrg, nsrc);
  field_tile(tl, q, src, trg, tile, e);
  if (nchunk == 1) {
    const int j0 = tl.x + threadIdx.x, j1 = j0 + kCT;
    if (j0 < tl.y) {
      ef[3 * (size_t)j0] = e[0];
      ef[3 * (size_t)j0 + 1] = e[1];
      ef[3 * (size_t)j0 + 2] = e[2];
    }
    if (j1 < tl.y) {
      ef[3 * (size_t)j1] = e[3];
      ef[3 * (size_t)j1 + 1] = e[4];
      ef[3 * (size_t)j1 + 2] = e[5];
    }
    return;
  }
  const size_t o = ((size_t)blockIdx.x * kTW + threadIdx.x) * 3, o1 = o + 3 * (size_t)kCT;
  part[o] = e[0];
  part[o + 1] = e[1];
  part[o + 2] = e[2];
  part[o1] = e[3];
  part[o1 + 1] = e[4];
  part[o1 + 2] = e[5];
}

__global__ __launch_bounds__(kCT) void k_field_reduce_uniform(int ntrg, int nchunk,
                                                              const double *__restrict__ part,
                                                              double *__restrict__ ef) {
  __shared__ double red[kCT][3];
  const int tb = blockIdx.x * kTW;
  field_reduce(blockIdx.x * nchunk, (blockIdx.x + 1) * nchunk, tb, min(tb + kTW, ntrg), part,
               ef, red);
}

__global__ void k_psi(int n, int nylm, double fac, const double *__restrict__ q,
                      double *__restrict__ psi) {
  size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= (size_t)n * nylm) return;
  psi[k] = (k % nylm == 0) ? fac * q[k / nylm] : 0.0;
}

// A tile table: tiles of kFW targets, per instance; `info` holds each
// instance's first target, first source, first tile and first target tile
// (and the ends after the last instance; for one instance the two rows come
// with the launch).  With a chunk length the sources of each target tile are
// cut into chunks, one tile each, and grp receives the first tile of each
// target tile.
struct TileRows {
  int4 a, b;
};
__global__ void k_make_tiles(int ninst, int ntile, long long chunk, TileRows one,
                             const int4 *__restrict__ info, int4 *__restrict__ tiles,
                             int *__restrict__ grp) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b > ntile) return;
  if (b == ntile) {
    if (grp) grp[ninst > 1 ? info[ninst].w : one.b.w] = ntile;
    return;
  }
  int4 lo = one.a, hi = one.b;
  if (ninst > 1) {
    int l = 0, h = ninst;   // info[l].z <= b < info[h].z
    while (h - l > 1) {
      const int m = (l + h) >> 1;
      if (info[m].z <= b) l = m;
      else h = m;
    }
    lo = info[l];
    hi = info[l + 1];
  }
  const int ntt = hi.w - lo.w, nch = (hi.z - lo.z) / ntt;
  const int tt = (b - lo.z) / nch, c = (b - lo.z) - tt * nch;
  const int tb = lo.x + tt * kFW;
  const long long sb = lo.y + c * chunk;
  tiles[b] = make_int4(tb, min(tb + kFW, hi.x), (int)sb, (int)min(sb + chunk, (long long)hi.y));
  if (grp && c == 0) grp[lo.w + tt] = b;
}

// sources per field tile: about 32768 one-wave tiles (several rounds of the
// resident waves, so that the uneven last chunks of each target tile do not
// leave CUs idle), whole multiples of kFW and at least 4 kFW; work = target
// tiles x sources
constexpr long long kFieldTiles = 32768;
long long field_chunk(long long work) {
  long long chunk = (work + kFieldTiles - 1) / kFieldTiles;
  chunk = ((chunk + kFW - 1) / kFW) * kFW;
  return std::max<long long>(chunk, 4 * kFW);
}

// targets toff[q] .. toff[q+1]-1 and sources soff[q] .. soff[q+1]-1 of ninst
// instances; split: the sources in chunks, with the groups.  The rows of
// several instances stay in t's host vector until its next use.
int make_tiles(ddx_handle *h, TileTable &t, int ninst, const int *toff, const int *soff,
               bool split) {
  long long work = 0;   // target tiles x sources
  for (int q = 0; q < ninst; ++q)
    work += (long long)((toff[q + 1] - toff[q] + kFW - 1) / kFW) * (soff[q + 1] - soff[q]);
  const long long chunk = split ? field_chunk(work) : 0x7fffffff;
  t.rows.resize(ninst + 1);
  long long nt = 0, ng = 0;
  for (int q = 0; q <= ninst; ++q) {
    t.rows[q] = make_int4(toff[q], soff[q], (int)nt, (int)ng);
    if (q == ninst) break;
    const long long ntt = (toff[q + 1] - toff[q] + kFW - 1) / kFW;
    const long long nch = std::max<long long>(1, (soff[q + 1] - soff[q] + chunk - 1) / chunk);
    nt += ntt * nch;
    ng += ntt;
  }
  if (nt > 0x7ffffffell) {
    set_error("%lld Coulomb tiles exceed the 32-bit index", nt);
    return DDX_ERR_CAPACITY;
  }
  t.ntile = (int)nt;
  t.ngrp = (int)ng;
  DDX_TRY(t.tiles.reserve((size_t)nt + 1));
  if (split) DDX_TRY(t.grp.reserve((size_t)ng + 1));
  if (ninst > 1) {
    DDX_TRY(t.info.reserve(ninst + 1));
    DDX_HIP(hipMemcpyAsync(t.info.p, t.rows.data(), (ninst + 1) * sizeof(int4),
                           hipMemcpyHostToDevice, h->stream));
  }
  hipLaunchKernelGGL(k_make_tiles, dim3((unsigned)(nt / 256 + 1)), dim3(256), 0, h->stream, ninst,
                     (int)nt, chunk, TileRows{t.rows[0], t.rows[ninst > 1 ? 1 : ninst]}, t.info.p,
                     t.tiles.p, split ? t.grp.p : nullptr);
  DDX_HIP(hipGetLastError());
  return DDX_OK;
}

}  // namespace

int potential_tiles(ddx_handle *h, TileTable &t, int nsrc, int ntrg) {
  const int toff[2] = {0, ntrg}, soff[2] = {0, nsrc};
  return make_tiles(h, t, 1, toff, soff, false);
}

int build_coulomb_tiles(ddx_handle *h) {
  // potential (and solute field) at the cavity points from the spheres, and
  // the field of the cavity charges at the nuclei
  DDX_TRY(make_tiles(h, h->ctile, h->ninst, h->h_cavoff.data(), h->h_soff.data(), false));
  return make_tiles(h, h->ftile, h->ninst, h->h_soff.data(), h->h_cavoff.data(), true);
}

int coulomb_potential(ddx_handle *h, const TileTable &t, const double *q, const double4 *src,
                      const double *trg3, double *phi, double *ef) {
  const int ntile = t.ntile;
  if (ntile <= 0) return DDX_OK;
  TimedLaunch tl(h, DDX_K_POTENTIAL, h->stream);
  if (ef)
    hipExtLaunchKernelGGL(k_potential<true>, dim3(ntile), dim3(kFW), 0, h->stream, tl.b, tl.e, 0,
                          t.tiles.p, q, src, trg3, phi, ef);
  else
    hipExtLaunchKernelGGL(k_potential<false>, dim3(ntile), dim3(kFW), 0, h->stream, tl.b, tl.e,
                          0, t.tiles.p, q, src, trg3, phi, nullptr);
  DDX_HIP(hipGetLastError());
  return DDX_OK;
}

int coulomb_field(ddx_handle *h, const TileTable &t, const double *q, const double *src3,
                  const double *trg3, double *ef) {
  const int ntile = t.ntile, ngrp = t.ngrp;
  const int4 *tiles = t.tiles.p;
  const int *grp = t.grp.p;
  if (ntile <= 0 || ngrp <= 0) return DDX_OK;
  DDX_TRY(h->fpart.reserve((size_t)ntile * kFW * 3));
  {
    TimedLaunch tl(h, DDX_K_FIELD, h->stream);
    hipExtLaunchKernelGGL(k_field_w, dim3(ntile), dim3(kFW), 0, h->stream, tl.b, tl.e, 0, tiles,
                          q, src3, trg3, h->fpart.p);
  }
  DDX_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_field_reduce_w, dim3(ngrp), dim3(kFW * kRw), 0, h->stream, grp, tiles,
                     h->fpart.p, ef);
  DDX_HIP(hipGetLastError());
  return DDX_OK;
}

// the field of nsrc arbitrary charges at ntrg arbitrary points (efld.f90:87-116)
int coulomb_field_points(ddx_handle *h, int nsrc, const double *q, const double *src3, int ntrg,
                         const double *trg3, double *ef) {
  if (ntrg <= 0) return DDX_OK;
  const int toff[2] = {0, ntrg}, soff[2] = {0, nsrc};
  DDX_TRY(make_tiles(h, h->xtile, 1, toff, soff, true));
  return coulomb_field(h, h->xtile, q, src3, trg3, ef);
}

int make_psi_n(ddx_handle *h, int n, int nylm, const double *charge, double *psi) {
  size_t nn = (size_t)n * nylm;
  double fac = sqrt(4.0 * (4.0 * atan(1.0)));
  hipLaunchKernelGGL(k_psi, dim3((nn + 255) / 256), dim3(256), 0, h->stream, n, nylm, fac,
                     charge, psi);
  DDX_HIP(hipGetLastError());
  return DDX_OK;
}

int make_psi(ddx_handle *h, const double *charge, double *psi) {
  return make_psi_n(h, h->n, h->nylm, charge, psi);
}

// ---------------------------------------------------------------------------
// The field without allocation.  Its partial sums live in `scratch`, a
// file-scope device array of kScratchBytes on every GPU the library runs on
// (held until the process ends).  In host code the array's name is only a
// stand-in: its device address on the current GPU comes from
// hipGetSymbolAddress, once per device, and only that address is used.
constexpr size_t kScratchBytes = size_t(32) << 20;
constexpr int kMaxDevices = 64;
static __device__ __align__(256) double scratch[kScratchBytes / sizeof(double)];
static double *g_scratch[kMaxDevices];

int noalloc_setup(double **out) {
  int dev = 0;
  DDX_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) {
    set_error("device %d beyond the %d devices the scratch table covers", dev, kMaxDevices);
    return DDX_ERR_ARG;
  }
  static std::mutex mu;
  std::lock_guard<std::mutex> lock(mu);
  if (!g_scratch[dev]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      set_error("hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
      return DDX_ERR_HIP;
    }
    g_scratch[dev] = static_cast<double *>(p);
  }
  if (out) *out = g_scratch[dev];
  return DDX_OK;
}

}  // namespace ddx

extern "C" int ddx_efld_noalloc(int nsrc, const double *src, const double *csrc, int ntrg,
                                const double *ctrg, double *ef, void *stream) {
  using namespace ddx;
  if (nsrc < 0 || ntrg < 0 || (nsrc && (!src || !csrc)) || (ntrg && (!ctrg || !ef))) {
    set_error("ddx_efld_noalloc: invalid arguments");
    return DDX_ERR_ARG;
  }
  double *part = nullptr;
  DDX_TRY(noalloc_setup(&part));
  if (ntrg == 0) return DDX_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // chunks as the table-driven path cuts them (about 8192 tiles, at least
  // 4 kCT sources each), then fewer where the partials would not fit
  const long long ntt = (ntrg + kTW - 1) / kTW;
  const long long max_tiles = (long long)(kScratchBytes / (sizeof(double) * 3 * kTW));
  long long chunk = (ntt * nsrc + 8191) / 8192;
  chunk = std::max<long long>(4 * kCT, ((chunk + kCT - 1) / kCT) * kCT);
  long long nchunk = std::max<long long>(1, (nsrc + chunk - 1) / chunk);
  if (ntt * nchunk > max_tiles) {
    nchunk = std::max<long long>(1, max_tiles / ntt);
    chunk = std::max<long long>(1, (nsrc + nchunk - 1) / nchunk);
    chunk = ((chunk + kCT - 1) / kCT) * kCT;
    nchunk = std::max<long long>(1, (nsrc + chunk - 1) / chunk);
  }
  const size_t need = nchunk > 1 ? (size_t)(ntt * nchunk) * kTW * 3 * sizeof(double) : 0;
  if (need > kScratchBytes || ntt * nchunk > 0x7fffffffll) {
    set_error("ddx_efld_noalloc: %lld partial tiles exceed the %zu-byte scratch",
              ntt * nchunk, kScratchBytes);
    return DDX_ERR_CAPACITY;
  }
  hipLaunchKernelGGL(k_field_uniform, dim3((unsigned)(ntt * nchunk)), dim3(kCT), 0, s, ntrg,
                     nsrc, (int)nchunk, (int)chunk, src, csrc, ctrg, part, ef);
  DDX_HIP(hipGetLastError());
  if (nchunk > 1) {
    hipLaunchKernelGGL(k_field_reduce_uniform, dim3((unsigned)ntt, kTW / (kCT / kRq)), dim3(kCT),
                       0, s, ntrg, (int)nchunk, part, ef);
    DDX_HIP(hipGetLastError());
  }
  return DDX_OK;
}
