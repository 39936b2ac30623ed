// Device setup of one ddCOSMO system (the per-geometry part of ddinit,
// ddcosmo.f90:308-468), plus the triple lists the sweeps run on.
//
//   neighbours  CSR, increasing j, |c_i - c_j| <= r_i + r_j (ddcosmo.f90:308-324):
//               by the O(n^2) scan where no instance has more than 4096
//               spheres, else through a spatial hash in O(n)
//   per point   fi = sum_j chi(t_n^ij), ui = max(0, 1 - fi) when fi <= 1,
//               zi in the switch region (ddcosmo.f90:359-411), plus a 64-bit
//               mask of the neighbours j with t_n^ij < 1
//   cavity      exposed points ui > 0, sphere-major (ddcosmo.f90:422-468)
//   triples     every (owner sphere o, point n, container c) with t < 1,
//               grouped by container c (owners ascending, then points, the
//               loop order of adjrhs, ddcosmo.f90:1316-1381), with the
//               geometry the sweeps need: cos/sin theta, cos/sin phi of
//               s = v/|v| (ylmbas, ddcosmo.f90:846-866), t and the weight
//               W = chi(t)/max(fi, 1) (ddcosmo.f90:1722-1730, 1340-1348).
//               pttri lists the triples of each point in neighbour order
//               (the loop order of calcv, ddcosmo.f90:1701-1739); tslot is
//               its inverse, the slot of each triple in its point's list.
//
// A small system's setup is bound by its launches and host round trips, not
// by their work, so the counts that later kernels need are made where the data
// is at hand: k_points also counts the triples of every (container, owner) and
// leaves the offsets within a sphere's points, the sums over spheres are one
// scan launch, and the host waits once, for the five totals that size the
// triple arrays.  60 atoms: 290 us with 45 launches and copies and three waits,
// now 77 us with 13 launches and one wait; 2000 atoms 490 -> 181 us.  (On a
// geometry no larger than an earlier one of the handle: one with more triples or
// exposed points than all before also frees and allocates their arrays, 0.3 to
// 0.6 ms at 300 to 1000 atoms.)
#include "ddx_device.hpp"
#include "ddx_kernels.hpp"

#include <algorithm>
#include <cmath>

namespace ddx {
namespace {

constexpr int kSetupThreads = 256;

// Neighbour search on a spatial hash.  Cubes of edge h >= 2 max r: two
// spheres that overlap lie in the same or in adjacent cubes.  Cube (ix, iy,
// iz) of instance k goes to bucket hash(k, ix, iy, iz) mod T; a bucket may
// hold several cubes, and the exact overlap test sorts them out.
__device__ __forceinline__ unsigned cell_bucket(long long ix, long long iy, long long iz,
                                                int inst, unsigned mask) {
  unsigned long long v = (unsigned long long)ix * 0x9E3779B97F4A7C15ull;
  v ^= (unsigned long long)iy * 0xC2B2AE3D27D4EB4Full;
  v ^= (unsigned long long)iz * 0x165667B19E3779F9ull;
  v ^= (unsigned long long)(unsigned)inst * 0xD6E8FEB86659FD93ull;
  v ^= v >> 31;
  return (unsigned)v & mask;
}

__device__ __forceinline__ long long cube_of(double x, double inv_h) {
  return (long long)floor(x * inv_h);
}

__device__ __forceinline__ unsigned sphere_bucket(const double4 &s, int inst, double inv_h,
                                                  unsigned mask, int d) {
  return cell_bucket(cube_of(s.x, inv_h) + d % 3 - 1, cube_of(s.y, inv_h) + (d / 3) % 3 - 1,
                     cube_of(s.z, inv_h) + d / 9 - 1, inst, mask);
}

// bucket of each sphere's own cube (d = 13: offsets 0, 0, 0) and the bucket sizes
__global__ void k_cell_count(const double4 *__restrict__ sph, const int *__restrict__ inst,
                             int n, double inv_h, unsigned mask, int *__restrict__ key,
                             int *__restrict__ bcnt) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const unsigned b = sphere_bucket(sph[i], inst ? inst[i] : 0, inv_h, mask, 13);
  key[i] = (int)b;
  atomicAdd(&bcnt[b], 1);
}

// spheres bucket by bucket (order inside a bucket is free; bcnt ends at 0)
__global__ void k_cell_fill(int n, const int *__restrict__ key, const int *__restrict__ boff,
                            int *__restrict__ bcnt, int *__restrict__ bsph) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int b = key[i];
  bsph[boff[b] + atomicSub(&bcnt[b], 1) - 1] = i;
}

// The same search without the hash, for instances of at most kDirectSearch
// spheres: one wave per sphere i tests every sphere of its instance, in
// increasing j, 64 at a time.  cand and deg as k_nbr_find leaves them.
// Up to there one launch of n / 64 tests a wave beats the hash's five
// (2000 atoms: 35 -> 14 us; 512 molecules of up to 795: 371 us for the find
// alone -> 67 us; 20 000 atoms: 72 us by the hash, n / 64 tests would take 250).
constexpr int kDirectSearch = 4096;

__global__ __launch_bounds__(kSetupThreads) void k_nbr_direct(
    const double4 *__restrict__ sph, const int *__restrict__ inst, const int *__restrict__ soff,
    int n, int *__restrict__ deg, int *__restrict__ cand) {
  const int i = __builtin_amdgcn_readfirstlane(
      (int)(blockIdx.x * (kSetupThreads / kWave) + threadIdx.x / kWave));
  if (i >= n) return;
  const int lane = lane_id();
  const int sb = inst ? soff[inst[i]] : 0, se = inst ? soff[inst[i] + 1] : n;
  const double4 si = sph[i];
  int cnt = 0;
#pragma unroll 4
  for (int j0 = sb; j0 < se; j0 += kWave) {
    const int j = j0 + lane;
    const double4 sj = sph[min(j, se - 1)];
    const bool hit = j < se && j != i && spheres_overlap(si, sj);
    const unsigned long long bal = __ballot(hit);
    const int pos = cnt + ballot_prefix(bal);
    if (hit && pos < kMaxDegree) cand[(size_t)i * kMaxDegree + pos] = j;
    cnt += __popcll(bal);
  }
  if (lane == 0) deg[i] = cnt;
}

// One wave per sphere i: the spheres j != i of its instance that overlap it,
// from the buckets of the 27 cubes around it, in increasing j, into
// cand(kMaxDegree, i); deg[i] = their number (also when above kMaxDegree,
// which the host turns into an error).
__global__ __launch_bounds__(kSetupThreads) void k_nbr_find(
    const double4 *__restrict__ sph, const int *__restrict__ inst, int n, double inv_h,
    unsigned mask, const int *__restrict__ boff, const int *__restrict__ bsph,
    int *__restrict__ deg, int *__restrict__ cand) {
  constexpr int W = kSetupThreads / kWave;
  __shared__ int list[W][kMaxDegree];
  const int wv = threadIdx.x / kWave, lane = lane_id();
  const int i = blockIdx.x * W + wv;
  int cnt = 0;
  if (i < n) {
    const double4 si = sph[i];
    const int ki = inst ? inst[i] : 0;
    // lane d < 27 takes cube d; a bucket that an earlier cube maps to is
    // left out
    const unsigned myb = lane < 27 ? sphere_bucket(si, ki, inv_h, mask, lane) : 0xffffffffu;
    bool dup = false;
    for (int e = 0; e < 27; ++e) {
      const unsigned be = (unsigned)__shfl((int)myb, e, kWave);
      dup = dup || (e < lane && be == myb);
    }
    unsigned long long todo = __ballot(lane < 27 && !dup);
    while (todo) {
      const int d = __ffsll(todo) - 1;
      todo &= todo - 1;
      const unsigned b = (unsigned)__shfl((int)myb, d, kWave);
      const int beg = boff[b], end = boff[b + 1];
      for (int k0 = beg; k0 < end; k0 += kWave) {
        const int k = k0 + lane;
        bool hit = false;
        int j = 0;
        if (k < end) {
          j = bsph[k];
          hit = j != i && (!inst || inst[j] == ki) && spheres_overlap(si, sph[j]);
        }
        const unsigned long long bal = __ballot(hit);
        const int pos = cnt + ballot_prefix(bal);
        if (hit && pos < kMaxDegree) list[wv][pos] = j;
        cnt += __popcll(bal);
      }
    }
  }
  __syncthreads();
  if (i < n) {
    if (lane == 0) deg[i] = cnt;
    cnt = min(cnt, kMaxDegree);   // (more is an error, found after this kernel)
    if (lane < cnt) {
      const int j = list[wv][lane];
      int rank = 0;
      for (int m = 0; m < cnt; ++m) rank += list[wv][m] < j ? 1 : 0;
      cand[(size_t)i * kMaxDegree + rank] = j;
    }
  }
}

// One wave per sphere i: its CSR list from the sorted candidates, and
// rev[q] = position of sphere i in the neighbour list of nl[q] (the number of
// smaller candidates there).
__global__ __launch_bounds__(kSetupThreads) void k_nbr_csr(int n, const int *__restrict__ deg,
                                                           const int *__restrict__ cand,
                                                           const int *__restrict__ inl,
                                                           int *__restrict__ nl,
                                                           int *__restrict__ rev) {
  const int i = __builtin_amdgcn_readfirstlane(
      (int)(blockIdx.x * (kSetupThreads / kWave) + threadIdx.x / kWave));
  if (i >= n) return;
  const int lane = lane_id();
  const int d = min(deg[i], kMaxDegree), b = inl[i];
  const int j = lane < d ? cand[(size_t)i * kMaxDegree + lane] : 0;
  const int dj = lane < d ? min(deg[j], kMaxDegree) : 0;
  int r = 0;
#pragma unroll 4
  for (int k = 0; k < d; ++k) {
    const int jk = __builtin_amdgcn_readlane(j, k), dk = __builtin_amdgcn_readlane(dj, k);
    const int c = cand[(size_t)jk * kMaxDegree + min(lane, max(dk - 1, 0))];
    const int rank = __popcll(__ballot(lane < dk && c < i));
    r = lane == k ? rank : r;
  }
  if (lane < d) {
    nl[b + lane] = j;
    rev[b + lane] = r;
  }
}

// OR of a 64-bit value over the wave (every lane receives it)
__device__ __forceinline__ unsigned long long wave_or64(unsigned long long v) {
  unsigned lo = (unsigned)v, hi = (unsigned)(v >> 32);
  lo |= partner_u32<0>(lo); hi |= partner_u32<0>(hi);
  lo |= partner_u32<1>(lo); hi |= partner_u32<1>(hi);
  lo |= partner_u32<2>(lo); hi |= partner_u32<2>(hi);
  lo |= partner_u32<3>(lo); hi |= partner_u32<3>(hi);
  lo |= partner_u32<4>(lo); hi |= partner_u32<4>(hi);
  lo |= partner_u32<5>(lo); hi |= partner_u32<5>(hi);
  return ((unsigned long long)hi << 32) | lo;
}

// The pair (container nl[inl[o] + kr], owner o) of owner o's neighbour kr,
// as an index of the container-major pair list: the owner's rank in the
// container's list is rev of the mirrored pair.
__device__ __forceinline__ int pair_of(const int *__restrict__ inl, const int *__restrict__ nl,
                                       const int *__restrict__ rev, int o, int kr) {
  const int q = inl[o] + kr;
  return inl[nl[q]] + rev[q];
}

// A sphere's points are cut into `runs` (1 or kRuns) runs of whole 64-point
// groups, one wave each: four where the spheres alone would leave most of the
// chip's 1024 SIMDs idle.  Run r of sphere i is number i runs + r.
//   Whole setup with one run -> four, us (points): 60 atoms 109 -> 69 (302), 642
// 92 -> 74 (110), 1000 189 -> 123 (590), 2000 220 -> 174 (590), 4000 139 -> 140
// (110) and 337 -> 283 (590).  Four is the faster beyond the line as well, on
// large grids (6000 494 -> 411 at 590 points, 20 000 765 -> 714 at 302; 12 000 at
// 110 points 292 -> 289): the line only bounds the arrays that hold 64 counts to
// a run.
constexpr int kRuns = 4;
constexpr int kRunSpheres = 4096;   // fewer spheres than this: kRuns

__device__ __forceinline__ int run_begin(int ngrid, int runs, int r) {
  return min(ngrid, (ngrid + kWave - 1) / kWave * r / runs * kWave);
}

// fi, ui, zi of every point (ddcosmo.f90:441-498) and the mask of the
// neighbours that contain it.  One wave per run of sphere i: the sphere's
// neighbours' centres and radii are staged in LDS (lane k loads neighbour k;
// the degree is at most 64), then the lanes take the run's points 64 at a
// time, each adding its terms over the neighbours in list order.  The exact
// terms (square root, divisions) are evaluated only for the neighbours that
// may contain the point, |v|^2 at most r^2 (1 + 1e-12): every t < 1 passes
// that test by far more than any rounding.  Beside them, while the masks are
// in registers: the number of the run's triples and exposed points before
// each point (ptoff, cavidx, within the run) and in all (runcnt, cavcnt), and
// its triples with each neighbour (paircnt, by the pair's place in the
// container's list and r).
__global__ __launch_bounds__(kSetupThreads) void k_points(
    const double4 *__restrict__ sph, const double4 *__restrict__ grid, int ngrid, int runs,
    const int *__restrict__ inl, const int *__restrict__ nl, const int *__restrict__ rev,
    double eta, int igrad, double *__restrict__ fi, double *__restrict__ ui,
    double *__restrict__ zi, unsigned long long *__restrict__ tmask, int *__restrict__ ptoff,
    int *__restrict__ cavidx, int *__restrict__ runcnt, int *__restrict__ cavcnt,
    int *__restrict__ paircnt, int n) {
  constexpr int kW = kSetupThreads / kWave;
  __shared__ double4 nb[kW][kWave];
  const int wave = threadIdx.x / kWave, lane = lane_id();
  const int run = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * kW + wave));
  const int i = run / runs, r = run - i * runs;
  if (i >= n) return;
  const int beg = inl[i], deg = min(inl[i + 1] - beg, kMaxDegree);
  const int jn = lane < deg ? nl[beg + lane] : 0;
  if (lane < deg) nb[wave][lane] = sph[jn];
  wave_lds_sync();
  const double4 si = sph[i];
  const int p0 = run_begin(ngrid, runs, r), p1 = run_begin(ngrid, runs, r + 1);
  int pairs = 0, before = 0, cav = 0;
  for (int n0 = p0; n0 < p1; n0 += kWave) {
    const int pn = n0 + lane;
    const bool in = pn < p1;
    const size_t p = (size_t)i * ngrid + pn;
    const double4 g = grid[in ? pn : p1 - 1];
    double f = 0.0, z0 = 0.0, z1 = 0.0, z2 = 0.0;
    unsigned long long mask = 0, cand = 0;
    // the neighbours that may contain the point (the cheap test), then the
    // exact terms of those only, in neighbour order: the lanes of a wave
    // would otherwise all wait through the square root and divisions of
    // every neighbour that contains any one of them
    for (int k = 0; k < deg; ++k) {
      const double4 sj = nb[wave][k];
      double v[3];
      point_vec(si, g, sj, v);
      const double d2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
      if (d2 <= sj.w * sj.w * (1.0 + 1e-12)) cand |= 1ull << k;
    }
    if (!in) cand = 0;
    for (; cand; cand &= cand - 1) {
      const int k = __ffsll((long long)cand) - 1;
      const double4 sj = nb[wave][k];
      double v[3];
      point_vec(si, g, sj, v);
      double vv = norm3(v);
      double t = vv / sj.w;
      if (t < 1.0) {
        f += fsw(t, eta);
        mask |= 1ull << k;
        if (igrad && t > 1.0 - eta) {
          double fac = dfsw(t, eta) / sj.w;
          z0 += fac * v[0] / vv;
          z1 += fac * v[1] / vv;
          z2 += fac * v[2] / vv;
        }
      }
    }
    const double u = (f <= 1.0) ? 1.0 - f : 0.0;
    const unsigned long long open = __ballot(in && u > 0.0);
    // triples before this lane's point, neighbour by neighbour, and the
    // neighbours' counts in the lanes that keep them
    int pre = before, all = 0;
    unsigned long long w = wave_or64(mask);
    while (w) {
      const int kr = __ffsll((long long)w) - 1;
      w &= w - 1;
      const unsigned long long hit = __ballot((mask >> kr) & 1ull);
      const int c = __popcll(hit);
      pre += ballot_prefix(hit);
      all += c;
      if (lane == kr) pairs += c;
    }
    if (in) {
      fi[p] = f;
      ui[p] = u;
      if (igrad) {
        zi[3 * p + 0] = z0;
        zi[3 * p + 1] = z1;
        zi[3 * p + 2] = z2;
      }
      tmask[p] = mask;
      ptoff[p] = pre;
      cavidx[p] = cav + ballot_prefix(open);
    }
    before += all;
    cav += __popcll(open);
  }
  if (lane == 0) {
    runcnt[run] = before;
    cavcnt[run] = cav;
  }
  if (lane < deg) paircnt[(size_t)(inl[jn] + rev[beg + lane]) * runs + r] = pairs;
}

// One wave per container c: the triples before each of its (owner, run)
// (pairloc), their number (tcnt) and the sweep units they make (ucnt).
__global__ __launch_bounds__(kSetupThreads) void k_pair_scan(int n, int runs,
                                                             const int *__restrict__ inl,
                                                             const int *__restrict__ paircnt,
                                                             int *__restrict__ pairloc,
                                                             int *__restrict__ tcnt,
                                                             int *__restrict__ ucnt) {
  const int c = __builtin_amdgcn_readfirstlane(
      (int)(blockIdx.x * (kSetupThreads / kWave) + threadIdx.x / kWave));
  if (c >= n) return;
  const int lane = lane_id();
  const int beg = inl[c], deg = inl[c + 1] - beg;
  const size_t q = ((size_t)beg + lane) * runs;
  int v[kRuns], sum = 0;
#pragma unroll
  for (int r = 0; r < kRuns; ++r) v[r] = (lane < deg && r < runs) ? paircnt[q + r] : 0;
#pragma unroll
  for (int r = 0; r < kRuns; ++r) sum += v[r];
  int incl = sum;
  for (int off = 1; off < kWave; off <<= 1) {
    const int t = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += t;
  }
  int at = incl - sum;
#pragma unroll
  for (int r = 0; r < kRuns; ++r) {
    if (lane < deg && r < runs) pairloc[q + r] = at;
    at += v[r];
  }
  if (lane == kWave - 1) {
    tcnt[c] = incl;
    ucnt[c] = (incl + kWave - 1) / kWave;
  }
}

// One wave per run of owner sphere o, in one pass over its masks: the final
// ptoff and cavidx of its points and the exposed points' coordinates, and for
// each point and each neighbour c containing it the triple's place in c's run
// of owner o (points ascending), its point index (tp) and its slot in the
// point's list (pttri, tslot).  Lane kr keeps the next place of neighbour
// kr's run.
__global__ __launch_bounds__(kSetupThreads) void k_sphere_lists(
    int n, int ngrid, int runs, const double4 *__restrict__ sph,
    const double4 *__restrict__ grid, const int *__restrict__ inl, const int *__restrict__ nl,
    const int *__restrict__ rev, const unsigned long long *__restrict__ tmask,
    const double *__restrict__ ui, const int *__restrict__ toff, const int *__restrict__ pairloc,
    const int *__restrict__ runoff, const int *__restrict__ cavrun, int *__restrict__ ptoff,
    int *__restrict__ cavidx, double *__restrict__ ccav, int *__restrict__ tp,
    int *__restrict__ pttri, int *__restrict__ tslot) {
  const int run = __builtin_amdgcn_readfirstlane(
      (int)(blockIdx.x * (kSetupThreads / kWave) + threadIdx.x / kWave));
  const int o = run / runs, r = run - o * runs;
  if (o >= n) return;
  const int lane = lane_id();
  const int deg = inl[o + 1] - inl[o];
  const int tb = runoff[run], cb = cavrun[run];
  int next = 0;
  if (lane < deg) {
    const int c = nl[inl[o] + lane];
    next = toff[c] + pairloc[(size_t)pair_of(inl, nl, rev, o, lane) * runs + r];
  }
  const double4 so = sph[o];
  const int p0 = run_begin(ngrid, runs, r), p1 = run_begin(ngrid, runs, r + 1);
  for (int n0 = p0; n0 < p1; n0 += kWave) {
    const int pn = n0 + lane;
    const bool in = pn < p1;
    const size_t p = (size_t)o * ngrid + min(pn, p1 - 1);
    const unsigned long long m = in ? tmask[p] : 0ull;
    const double u = ui[p];
    const int first = tb + ptoff[p], ic = cb + cavidx[p];
    if (in) {
      ptoff[p] = first;
      cavidx[p] = ic;
      if (u > 0.0) {
        const double4 g = grid[pn];
        ccav[3 * (size_t)ic + 0] = so.x + so.w * g.x;
        ccav[3 * (size_t)ic + 1] = so.y + so.w * g.y;
        ccav[3 * (size_t)ic + 2] = so.z + so.w * g.z;
      }
    }
    unsigned long long w = wave_or64(m);
    while (w) {
      const int kr = __ffsll((long long)w) - 1;
      w &= w - 1;
      const bool hit = (m >> kr) & 1ull;
      const unsigned long long b = __ballot(hit);
      const int base = __builtin_amdgcn_readlane(next, kr);
      if (hit) {
        const int idx = base + ballot_prefix(b);
        const int slot = first + __popcll(m & ((1ull << kr) - 1ull));
        tp[idx] = (int)p;
        pttri[slot] = idx;
        tslot[idx] = slot;
      }
      if (lane == kr) next += __popcll(b);
    }
  }
  if (run == n * runs - 1 && lane == 0) {
    const size_t np = (size_t)n * ngrid;
    ptoff[np] = runoff[run + 1];
    cavidx[np] = cavrun[run + 1];
  }
}

// The record of triple (owner point p = o ngrid + n, container c), as calcv
// and adjrhs evaluate it (ddcosmo.f90:1707-1727, 1325-1345; the angles as
// ylmbas takes them, ddcosmo.f90:845-857, with cos phi = 1 on the axis).
__device__ __forceinline__ void triple_record(const double4 &so, const double4 &g,
                                              const double4 &sc, double f, double eta,
                                              double4 &geo, double2 &tw) {
  double v[3];
  point_vec(so, g, sc, v);
  const double vv = norm3(v);
  const double t = vv / sc.w;
  const double s0 = v[0] / vv, s1 = v[1] / vv, s2 = v[2] / vv;
  const double cthe = s2;
  const double sthe = sqrt(1.0 - cthe * cthe);
  double cphi = 1.0, sphi = 0.0;
  if (sthe != 0.0) {
    cphi = s0 / sthe;
    sphi = s1 / sthe;
  }
  const double chi = fsw(t, eta);
  const double w = (f > 1.0) ? chi / f : chi;
  geo = make_double4(cthe, sthe, cphi, sphi);
  tw = make_double2(t, w);
}

// `wpc` waves (1 or 4) per container c: the records of its triples, all lanes
// busy, and with g32 / w32 the FP32 sweeps' records of them (geo32_of, and W).
__global__ __launch_bounds__(kSetupThreads) void k_triple_geo(
    int n, int ngrid, int wpc, double eta, const double4 *__restrict__ sph,
    const double4 *__restrict__ grid, const int *__restrict__ toff, const int *__restrict__ tp,
    const double *__restrict__ fi, double4 *__restrict__ tgeo, double2 *__restrict__ ttw,
    float4 *__restrict__ g32, float *__restrict__ w32) {
  const int w = __builtin_amdgcn_readfirstlane(
      (int)(blockIdx.x * (kSetupThreads / kWave) + threadIdx.x / kWave));
  const int c = w / wpc;
  if (c >= n) return;
  const double4 sc = sph[c];
  const int end = toff[c + 1];
  for (int k = toff[c] + (w - c * wpc) * kWave + lane_id(); k < end; k += wpc * kWave) {
    const unsigned p = (unsigned)tp[k];
    const unsigned o = p / (unsigned)ngrid, pn = p - o * (unsigned)ngrid;
    double4 a;
    double2 b;
    triple_record(sph[o], grid[pn], sc, fi[p], eta, a, b);
    tgeo[k] = a;
    ttw[k] = b;
    if (g32) {
      g32[k] = geo32_of(a, b);
      w32[k] = (float)b.y;
    }
  }
}

// Work units of the sweeps: runs of kWave triples of one container.
// A launch of the sweep hands contiguous ranges of units to a fixed number
// of workers; a segment is the part of one worker's range inside one
// container, and each segment leaves one partial L* S vector.
// Where each sweep worker starts: (container, unit, segment, triple) of its
// first unit, worker w's being floor(w U / G), and the end of the last one's
// range (G + 1 entries).  Made once per setup: found by every worker of every
// sweep, the container was a binary search of dependent loads (11 of them at
// 2000 spheres, 17 in the 512-molecule batch) ahead of the first triple.
__global__ void k_worker_start(int n, const int *__restrict__ uoff, const int *__restrict__ segoff,
                               const int *__restrict__ toff, long long U, long long G,
                               int4 *__restrict__ wstart) {
  const long long w = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (w > G) return;
  const int u0 = (int)(w * U / G);
  if (w == G) {
    wstart[w] = make_int4(n, u0, 0, 0);
    return;
  }
  int lo = 0, hi = n;   // uoff[lo] <= u0 < uoff[hi]: the last c with uoff[c] <= u0
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (uoff[mid] <= u0) lo = mid;
    else hi = mid;
  }
  const int b = uoff[lo];
  int seg = segoff[lo];
  if (u0 > b) seg += 1 + (int)(w - (((long long)b + 1) * G + U - 1) / U);
  wstart[w] = make_int4(lo, u0, seg, toff[lo] + (u0 - b) * kWave);
}

// segments per container: its first unit starts one, and so does every
// worker whose range begins inside the container (worker w starts at unit
// floor(w U / G))
__global__ void k_seg_count(int n, const int *__restrict__ uoff, long long U, long long G,
                            int *__restrict__ segcnt) {
  int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  const long long a = uoff[c], b = uoff[c + 1];
  int cnt = 0;
  if (b > a) {
    const long long hi = (b * G + U - 1) / U, lo = ((a + 1) * G + U - 1) / U;
    cnt = 1 + (int)(hi > lo ? hi - lo : 0);
  }
  segcnt[c] = cnt;
}

// cavity offset of each instance: the exposed points before its first sphere
__global__ void k_cav_offsets(int ninst, int runs, const int *__restrict__ soff,
                              const int *__restrict__ cavrun, int *__restrict__ out) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q <= ninst) out[q] = cavrun[(size_t)soff[q] * runs];
}

}  // namespace

int lists_ready(const ddx_handle *h, const char *what) {
  if (h->have_lists) return DDX_OK;
  set_error("%s: the setup of the handle's geometry failed; upload another one and run it", what);
  return DDX_ERR_STATE;
}

int run_setup(ddx_handle *h) {
  hipStream_t s = h->stream;
  h->have_setup = h->have_lists = false;
  int n = h->n, ng = h->ngrid;
  size_t np = (size_t)n * ng;
  h->np = np;
  drop_round_graphs(h);   // captured solver rounds hold the old buffers
  if (np > 0x7fffffffull) {
    // point indices are 32-bit in the per-point kernels
    set_error("nsph * ngrid = %zu points exceed the 32-bit point index", np);
    return DDX_ERR_CAPACITY;
  }

  const int *inst = h->inst.p;
  const int W = kSetupThreads / kWave;
  const dim3 per_sphere((n + W - 1) / W);
  if (h->maps_n != n) {
    DDX_TRY(h->soff.reserve(h->ninst + 1));
    DDX_HIP(hipMemcpyAsync(h->soff.p, h->h_soff.data(), (h->ninst + 1) * sizeof(int),
                           hipMemcpyHostToDevice, s));
    h->most = 0;
    for (int q = 0; q < h->ninst; ++q) h->most = std::max(h->most, h->h_soff[q + 1] - h->h_soff[q]);
  }

  // neighbour lists; the arrays are sized by the degree cap, so that nothing
  // here waits for a count
  DDX_TRY(h->degcnt.reserve(n + 1));
  DDX_TRY(h->inl.reserve(n + 1));
  DDX_TRY(h->cand.reserve((size_t)n * kMaxDegree));
  if (h->most <= kDirectSearch) {
    hipLaunchKernelGGL(k_nbr_direct, per_sphere, dim3(kSetupThreads), 0, s, h->sph.p, inst,
                       h->soff.p, n, h->degcnt.p, h->cand.p);
    DDX_HIP(hipGetLastError());
  } else {
    unsigned T = 64;
    while (T < 2u * (unsigned)n) T <<= 1;
    const double inv_h = 1.0 / (2.0 * h->rmax * (1.0 + 1e-12));
    DDX_TRY(h->ckey.reserve(n));
    DDX_TRY(h->bcnt.reserve(T + 1));
    DDX_TRY(h->boff.reserve(T + 1));
    DDX_TRY(h->bsph.reserve(n));
    DDX_HIP(hipMemsetAsync(h->bcnt.p, 0, (T + 1) * sizeof(int), s));
    hipLaunchKernelGGL(k_cell_count, dim3((n + 255) / 256), dim3(256), 0, s, h->sph.p, inst, n,
                       inv_h, T - 1, h->ckey.p, h->bcnt.p);
    DDX_HIP(hipGetLastError());
    DDX_TRY(scan_exclusive(h->bcnt.p, h->boff.p, T, h->scan_tmp, s));
    hipLaunchKernelGGL(k_cell_fill, dim3((n + 255) / 256), dim3(256), 0, s, n, h->ckey.p,
                       h->boff.p, h->bcnt.p, h->bsph.p);
    DDX_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_nbr_find, per_sphere, dim3(kSetupThreads), 0, s, h->sph.p, inst, n,
                       inv_h, T - 1, h->boff.p, h->bsph.p, h->degcnt.p, h->cand.p);
    DDX_HIP(hipGetLastError());
  }
  {
    const Scan deg = {h->degcnt.p, h->inl.p, (size_t)n, kMaxDegree, h->d_counts + kCntPairs,
                      h->d_counts + kCntDegree};
    DDX_TRY(scan_arrays(&deg, 1, h->scan_tmp, s));
  }
  const size_t cap = (size_t)n * kMaxDegree + 1;
  const int runs = n < kRunSpheres ? kRuns : 1;
  DDX_TRY(h->nl.reserve(cap));
  DDX_TRY(h->rev.reserve(cap));
  DDX_TRY(h->paircnt.reserve(cap * runs));
  DDX_TRY(h->pairloc.reserve(cap * runs));
  hipLaunchKernelGGL(k_nbr_csr, per_sphere, dim3(kSetupThreads), 0, s, n, h->degcnt.p, h->cand.p,
                     h->inl.p, h->nl.p, h->rev.p);
  DDX_HIP(hipGetLastError());

  // per-point quantities, and the counts of the triples
  const size_t nrun = (size_t)n * runs;
  DDX_TRY(h->fi.reserve(np));
  DDX_TRY(h->ui.reserve(np));
  if (h->igrad) DDX_TRY(h->zi.reserve(3 * np));
  DDX_TRY(h->tmask.reserve(np));
  DDX_TRY(h->ptoff.reserve(np + 1));
  DDX_TRY(h->cavidx.reserve(np + 1));
  DDX_TRY(h->runcnt.reserve(nrun));
  DDX_TRY(h->runoff.reserve(nrun + 1));
  DDX_TRY(h->cavcnt.reserve(nrun));
  DDX_TRY(h->cavrun.reserve(nrun + 1));
  DDX_TRY(h->tcnt.reserve(n));
  DDX_TRY(h->toff.reserve(n + 1));
  DDX_TRY(h->ucnt.reserve(n));
  DDX_TRY(h->uoff.reserve(n + 1));
  const dim3 per_run((unsigned)((nrun + W - 1) / W));
  hipLaunchKernelGGL(k_points, per_run, dim3(kSetupThreads), 0, s, h->sph.p, h->grid.p, ng, runs,
                     h->inl.p, h->nl.p, h->rev.p, h->eta, h->igrad, h->fi.p, h->ui.p,
                     h->igrad ? h->zi.p : nullptr, h->tmask.p, h->ptoff.p, h->cavidx.p,
                     h->runcnt.p, h->cavcnt.p, h->paircnt.p, n);
  DDX_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_pair_scan, per_sphere, dim3(kSetupThreads), 0, s, n, runs, h->inl.p,
                     h->paircnt.p, h->pairloc.p, h->tcnt.p, h->ucnt.p);
  DDX_HIP(hipGetLastError());
  {
    constexpr int all = 0x7fffffff;
    const Scan sums[4] = {
        {h->runcnt.p, h->runoff.p, nrun, all, h->d_counts + kCntTriples, nullptr},
        {h->cavcnt.p, h->cavrun.p, nrun, all, h->d_counts + kCntCav, nullptr},
        {h->tcnt.p, h->toff.p, (size_t)n, all, nullptr, nullptr},
        {h->ucnt.p, h->uoff.p, (size_t)n, all, h->d_counts + kCntUnits, nullptr}};
    DDX_TRY(scan_arrays(sums, 4, h->scan_tmp, s));
  }
  // the cavity offset of each instance, read back with the counts
  std::vector<int> cavoff;
  if (h->ninst > 1) {
    DDX_TRY(h->cavoff.reserve((size_t)h->ninst + 1));
    hipLaunchKernelGGL(k_cav_offsets, dim3((h->ninst + 256) / 256), dim3(256), 0, s, h->ninst,
                       runs, h->soff.p, h->cavrun.p, h->cavoff.p);
    DDX_HIP(hipGetLastError());
    cavoff.resize(h->ninst + 1);
    DDX_HIP(hipMemcpyAsync(cavoff.data(), h->cavoff.p, (h->ninst + 1) * sizeof(int),
                           hipMemcpyDeviceToHost, s));
  }
  DDX_HIP(hipStreamSynchronize(s));
  const int nnl = h->h_counts[kCntPairs], maxdeg = h->h_counts[kCntDegree];
  const int ntri = h->h_counts[kCntTriples], ncav = h->h_counts[kCntCav];
  const int nunit = h->h_counts[kCntUnits];
  h->nnl = nnl;
  h->maxdeg = maxdeg;
  if (maxdeg > kMaxDegree) {
    set_error("a sphere overlaps %d others; at most %d are supported", maxdeg, kMaxDegree);
    return DDX_ERR_CAPACITY;
  }
  h->ntri = ntri;
  h->ncav = ncav;
  h->nunit = nunit;
  if (h->ninst > 1) h->h_cavoff.swap(cavoff);
  // workers: whole multiples of the R = 8 per CU one-wave workgroups that
  // the FP64 sweeps keep resident (two waves per SIMD; the lmax 6 FP32 sweep
  // holds four), as many as give about
  // kUnitsPerWorker units each (or as many per compute unit as ddx_autotune
  // chose).  Short ranges keep waves queued behind the resident ones, which
  // hides the memory latency of their triples; a partial last round of
  // workgroups would leave most CUs idle at the end.
  long long G = (long long)h->workers_per_cu * h->ncu;
  if (!h->workers_fixed) {
    const double rounds = (double)nunit / ((double)kUnitsPerWorker * (double)G);
    G *= std::max(1LL, std::llround(rounds));
  }
  if (G > nunit) G = nunit;
  h->nworker = (int)G;
  DDX_TRY(h->segcnt.reserve(n + 1));
  DDX_TRY(h->segoff.reserve(n + 1));
  // (a container with units implies U > 0 and G > 0)
  hipLaunchKernelGGL(k_seg_count, dim3((n + 255) / 256), dim3(256), 0, s, n, h->uoff.p,
                     (long long)nunit, G, h->segcnt.p);
  DDX_HIP(hipGetLastError());
  DDX_TRY(scan_exclusive(h->segcnt.p, h->segoff.p, n, h->scan_tmp, s));
  h->nseg_cap = (int)G + n;   // segments: at most one per container plus one per worker
  DDX_TRY(h->wstart.reserve((size_t)G + 1));
  if (G > 0) {
    hipLaunchKernelGGL(k_worker_start, dim3((unsigned)((G + 256) / 256)), dim3(256), 0, s, n,
                       h->uoff.p, h->segoff.p, h->toff.p, (long long)nunit, G, h->wstart.p);
    DDX_HIP(hipGetLastError());
  }

  h->have_geo32 = false;   // the float copies are remade on their next use
  h->fmm.lists_ok = false;  // as are the near lists of the far-field sums
  DDX_TRY(h->tgeo.reserve(ntri + 1));
  DDX_TRY(h->ttw.reserve(ntri + 1));
  DDX_TRY(h->tp.reserve(ntri + 1));
  DDX_TRY(h->pttri.reserve(ntri + 1));
  DDX_TRY(h->tslot.reserve(ntri + 1));
  DDX_TRY(h->ccav.reserve(3 * (size_t)ncav + 3));
  hipLaunchKernelGGL(k_sphere_lists, per_run, dim3(kSetupThreads), 0, s, n, ng, runs, h->sph.p,
                     h->grid.p, h->inl.p, h->nl.p, h->rev.p, h->tmask.p, h->ui.p, h->toff.p,
                     h->pairloc.p, h->runoff.p, h->cavrun.p, h->ptoff.p, h->cavidx.p, h->ccav.p,
                     h->tp.p, h->pttri.p, h->tslot.p);
  DDX_HIP(hipGetLastError());
  if (ntri > 0) {
    // the float copies come with the records when the handle runs the mixed
    // precision, else on the first FP32 sweep
    const bool f32 = h->prec == DDX_PREC_MIXED;
    if (f32) {
      DDX_TRY(h->tgeo32.reserve(ntri + 1));
      DDX_TRY(h->ttw32.reserve(ntri + 1));
    }
    hipLaunchKernelGGL(k_triple_geo, per_run, dim3(kSetupThreads), 0, s, n, ng, runs, h->eta,
                       h->sph.p, h->grid.p, h->toff.p, h->tp.p, h->fi.p, h->tgeo.p, h->ttw.p,
                       f32 ? h->tgeo32.p : nullptr, f32 ? h->ttw32.p : nullptr);
    DDX_HIP(hipGetLastError());
    h->have_geo32 = f32;
  }
  // the solver's block maps (once per handle: they depend on the sphere
  // counts only),
  // Coulomb tiles
  if (h->maps_n != n) {
    DDX_TRY(build_solver_maps(h));
    h->maps_n = n;
  }
  if (h->ninst == 1) h->h_cavoff.assign({0, ncav});
  DDX_TRY(build_coulomb_tiles(h));
  h->have_setup = h->have_lists = true;
  h->stats.ntriples = ntri;
  h->stats.nnl = nnl;
  h->stats.ncav = ncav;
  h->stats.max_degree = maxdeg;
  return DDX_OK;
}

}  // namespace ddx
