// Jacobi iteration with Pulay DIIS, on the device (jacobi_diis.f90:43-438).
//
// One iteration is
//   y      = O x                              (matvec callback: lx or lstarx)
//   x_new  = D^-1 (rhs - y)                   (ldm1x, matvec.f90:246-269)
//   DIIS   store x_new, e = x_new - x; B row of dot products; bordered
//          system by Gauss-Jordan with full pivoting; x_new = sum c_i x_i
//          (diis/makeb/gjinv, jacobi_diis.f90:198-400, drop-10 rule included)
//   norm   hnorm(x_new - x) (matvec.f90:281-323); converged when < tol
// as three kernels: k_jacobi (update + Gram-row partial sums, fused),
// k_diis_small (the previous norm's test, B update, Gauss-Jordan by one wave,
// coefficients) and k_extrap (extrapolation, increment norm partials,
// x <- x_new); without DIIS k_norm takes the second one's place.  Single
// systems take forms arranged for latency: k_jacobi_two and k_extrap_one up to
// 512 elements a workgroup, and up to one workgroup of both solves to a compute
// unit k_diis_extrap, the last two kernels in one launch.  The bookkeeping
// lives in a device DiisState; once it says done every later kernel returns
// at once, so the host can enqueue iterations ahead.  The kernel that ends a
// solve writes its results to a record in pinned memory, which the host polls.
//
// A handle may hold a batch of independent instances (molecules): each has
// its own DiisState and converges on its own, exactly as if solved alone.
// Every workgroup of k_jacobi and k_extrap works inside one instance (the
// block maps jblk, eblk), so that its partial sums belong to that instance;
// k_diis_small runs one workgroup per instance.  A plain handle is a batch
// of one.
#include "ddx_device.hpp"
#include "ddx_kernels.hpp"

#include <algorithm>
#include <cstddef>
#include <cstring>
#include <iterator>

namespace ddx {
namespace {

constexpr int kJThreads = 256;
constexpr int kPartStride = kDiisMax + 1;   // 25 dots + self dot per block
// mixed precision: every kRefresh-th round applies the FP64 operator to the
// iterate itself (the FP64 image of the iterate restarts exactly there)
constexpr int kRefresh = 8;
// rounds per captured graph group (a multiple of kRefresh, so that every
// group of a mixed-precision solve starts at the same phase and one graph
// serves them all)
constexpr int kGraphRounds = 32;

// Pointers of one system's Jacobi/DIIS iteration; the kernels below take
// one or two systems (the paired direct and adjoint solves), selected by
// blockIdx.y (blockIdx.x for the single-workgroup kernels).
struct SysArgs {
  const double *rhs, *y;     // y: ny partial arrays of nylm nsph, summed here,
  int ny;                    // or with yp the per-segment sums of L* S:
  const double *yp;          //   y(lm, c) = sum of yp(lm, s), s in segoff[c] ..
  const int *segoff;
  double *x, *xs;            // xs = cf x, kept for the L X sweep (null for L*)
  double *xd, *ed, *xnew;    // DIIS history (ed: float in mixed precision) and the Jacobi step
  double *part, *part_e;     // Gram-row (26 rows of nbj) and increment-norm partial sums
  int *newslot;              // per instance
  DiisState *st;             // per instance, then the summary of a batch
  // mixed precision: the operator's image of the iterate carried in FP64
  double *yacc;              // L x (L* x): y adds to it (acc = 1) or replaces it
  int acc;                   //   (acc = 0, a round with the FP64 operator on x)
  double *inc;               // the last increment x_new - x (null: not kept)
  int xs_inc;                // xs = cf inc instead of cf x (the next round applies
                             //   the FP32 operator to the increment)
  DiisState *rec;            // the host's record of the solve (pinned host memory)
};
struct Systems {
  SysArgs s[2];
};

//
// a history value as double, converted where it is used: the empty asm keeps
// the compiler from moving the conversion (and the wait for its load) into
// the branch that loaded it, ahead of the element's other loads
__device__ __forceinline__ double widen_late(double v) { return v; }
__device__ __forceinline__ double widen_late(float v) {
  asm volatile("" : "+v"(v));
  return (double)v;
}

// x_new = D^-1 (rhs - y) and the residual x_new - x of that rounded x_new (no
// fused multiply-subtract: both kernels that call it give the same bits)
__device__ __forceinline__ void jacobi_step(double facl, double rhs, double y, double x,
                                            double &xn, double &dx) {
#pragma clang fp contract(off)
  xn = facl * (rhs - y);
  dx = xn - x;
}

// E is the storage type of the residual history: double, or float in mixed
// precision, where the history only steers the extrapolation coefficients.
// Each residual is rounded to E once and that rounded value enters every dot
// product it is part of (its self dot included), so that B stays the Gram
// matrix of the stored vectors.
template <typename E>
__global__ __launch_bounds__(kJThreads) void k_jacobi(size_t nn, int nylm, int diis_max,
                                                      const int4 *__restrict__ jblk, int nbj,
                                                      const double *__restrict__ facl,
                                                      Systems sys) {
  const SysArgs &q0 = sys.s[blockIdx.y];
  const int4 blk = jblk[blockIdx.x];   // instance, elements blk.y .. blk.z - 1
  const DiisState *__restrict__ st = q0.st + blk.x;
  if (st->done) return;
  const double *__restrict__ rhs = q0.rhs;
  const double *__restrict__ y = q0.y;
  const int ny = q0.ny;
  const double *__restrict__ yp = q0.yp;
  const int *__restrict__ segoff = q0.segoff;
  const double *__restrict__ x = q0.x;
  double *__restrict__ xd = q0.xd;
  E *__restrict__ ed = reinterpret_cast<E *>(q0.ed);
  double *__restrict__ xnew = q0.xnew;
  double *__restrict__ part = q0.part;
  __shared__ double wpart[kJThreads / kWave][kPartStride];
  const int nmat = st->nmat;
  const int off = (diis_max > 0 && nmat >= diis_max) ? 10 : 0;
  const int ndot = diis_max > 0 ? nmat - off - 1 : 0;
  double *xo = diis_max > 0 ? xd + (size_t)st->slot[nmat - 1] * nn : xnew;
  E *eo = diis_max > 0 ? ed + (size_t)st->slot[nmat - 1] * nn : nullptr;
  const E *eh[kDiisMax];
#pragma unroll
  for (int q = 0; q < kDiisMax; ++q)
    eh[q] = (q < ndot) ? ed + (size_t)st->slot[off + q] * nn : nullptr;
  if constexpr (sizeof(E) == 4) {
    // FP32 history: slots past ndot read the first slot's element again (a
    // cache hit, its value unused), so that every load is unconditional and
    // none waits at a branch for the one before it
    const E *fill = ndot > 0 ? eh[0] : (eo ? eo : reinterpret_cast<const E *>(x));
#pragma unroll
    for (int q = 0; q < kDiisMax; ++q)
      if (q >= ndot) eh[q] = fill;
  }
  double acc[kDiisMax];
#pragma unroll
  for (int q = 0; q < kDiisMax; ++q) acc[q] = 0.0;
  double self = 0.0;
  for (size_t k = (size_t)blk.y + threadIdx.x; k < (size_t)blk.z; k += kJThreads) {
    // element indices fit in 32 bits (build_solver_maps checks nylm nsph)
    const unsigned c = (unsigned)k / (unsigned)nylm;
    const unsigned lm = (unsigned)k - c * (unsigned)nylm;
    // the history residuals are read first, with the element's other
    // operands, so that all of them are in flight together (kept as E until
    // the dot products, so that no conversion waits for its load early)
    E ev[kDiisMax];
#pragma unroll
    for (int q = 0; q < kDiisMax; ++q) {
      if constexpr (sizeof(E) == 4)
        ev[q] = eh[q][k];
      else
        ev[q] = (q < ndot) ? eh[q][k] : E(0);
    }
    double yk;
    if (yp) {
      yk = 0.0;
      for (int j = segoff[c]; j < segoff[c + 1]; ++j) yk += yp[(size_t)j * nylm + lm];
    } else {
      yk = y[k];
      for (int j = 1; j < ny; ++j) yk += y[(size_t)j * nn + k];
    }
    if (q0.yacc) {
      if (q0.acc) yk += q0.yacc[k];
      q0.yacc[k] = yk;
    }
    double xn, dx;
    jacobi_step(facl[lm], rhs[k], yk, x[k], xn, dx);
    const E er = (E)dx;
    const double e = (double)er;
    xo[k] = xn;
    if (eo) {
      eo[k] = er;
#pragma unroll
      for (int q = 0; q < kDiisMax; ++q)
        if (q < ndot) acc[q] += widen_late(ev[q]) * e;
      self += e * e;
    }
  }
  if (diis_max == 0) return;
  // all 26 partial dots of the block: butterflies per wave, one barrier
  const int wave = threadIdx.x / kWave;
#pragma unroll
  for (int q = 0; q < kDiisMax; ++q) {
    if (q < ndot) {
      double v = wave_sum(acc[q]);
      if (lane_id() == 0) wpart[wave][q] = v;
    }
  }
  self = wave_sum(self);
  if (lane_id() == 0) wpart[wave][kDiisMax] = self;
  __syncthreads();
  const int q = threadIdx.x;
  if (q < ndot || q == kDiisMax)
    part[(size_t)q * nbj + blockIdx.x] =
        (wpart[0][q] + wpart[1][q]) + (wpart[2][q] + wpart[3][q]);
}

// element at a 32-bit byte offset of a wave-uniform base
template <typename T>
__device__ __forceinline__ T load_at(const void *base, unsigned bytes) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + bytes);
}

// the largest number of Gram dots of an iteration: nmat stays below diis_max
// or drops by ten
constexpr int kMaxDots = kDiisMax - 2;

// One thread's two elements of k_jacobi_two: history residuals (H of them,
// those past ndot re-read slot 0 and meet only unread sums), operator image,
// Jacobi step, stores, and its shares of the Gram dots, self dot last.
template <typename E, int H>
__device__ __forceinline__ void jacobi_two_elements(
    const SysArgs &a, unsigned nn, unsigned nylm, const unsigned (&k)[2], const bool (&live)[2],
    const unsigned (&lm)[2], const int (&s0)[2], const int (&s1)[2], const double (&rhs)[2],
    const double (&x)[2], const double (&f)[2], const unsigned (&slot)[kMaxDots], unsigned cur,
    double (&acc)[kMaxDots + 1]) {
  E ev[2][H];
#pragma unroll
  for (int q = 0; q < H; ++q)
#pragma unroll
    for (int i = 0; i < 2; ++i)
      ev[i][q] = load_at<E>(a.ed, (slot[q] * nn + k[i]) * (unsigned)sizeof(E));
  double y[2] = {0.0, 0.0}, ya[2] = {0.0, 0.0};
  const bool add = a.yacc && a.acc;
  if (add) {
#pragma unroll
    for (int i = 0; i < 2; ++i) ya[i] = a.yacc[k[i]];
  }
  if (a.yp) {
    // sums over the segments in order, the loads of eight segments of both
    // elements in flight together (past the last one: read again, not added)
    const int n0 = s1[0] - s0[0], n1 = s1[1] - s0[1];
    for (int j = 0; j < max(n0, n1); j += 8) {
      double v[2][8];
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        v[0][t] = a.yp[(size_t)(s0[0] + max(min(j + t, n0 - 1), 0)) * nylm + lm[0]];
        v[1][t] = a.yp[(size_t)(s0[1] + max(min(j + t, n1 - 1), 0)) * nylm + lm[1]];
      }
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        if (j + t < n0) y[0] += v[0][t];
        if (j + t < n1) y[1] += v[1][t];
      }
    }
  } else {
    double v[2][kProjSplit];
#pragma unroll
    for (int j = 0; j < kProjSplit; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i) v[i][j] = a.y[(size_t)min(j, a.ny - 1) * nn + k[i]];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      y[i] = v[i][0];
#pragma unroll
      for (int j = 1; j < kProjSplit; ++j)
        if (j < a.ny) y[i] += v[i][j];
    }
  }
  E *__restrict__ eo = reinterpret_cast<E *>(a.ed) + (size_t)cur * nn;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if (!live[i]) continue;
    if (add) y[i] += ya[i];
    double xn, dx;
    jacobi_step(f[i], rhs[i], y[i], x[i], xn, dx);
    const E er = (E)dx;
    const double e = (double)er;
    if (a.yacc) a.yacc[k[i]] = y[i];
    a.xd[(size_t)cur * nn + k[i]] = xn;
    eo[k[i]] = er;
#pragma unroll
    for (int q = 0; q < H; ++q) acc[q] += (double)ev[i][q] * e;
    acc[kMaxDots] += e * e;
  }
}

// The state as the round found it, for k_diis_extrap: into the next state by
// one workgroup, all loads ahead of the stores.
__device__ __forceinline__ void copy_state(DiisState *st) {
  constexpr int kWords = (int)(offsetof(DiisState, hist) / sizeof(double));
  constexpr int kEach = (kWords + kJThreads - 1) / kJThreads;
  const double *from = reinterpret_cast<const double *>(st);
  double *to = reinterpret_cast<double *>(st + 1);
  double v[kEach];
#pragma unroll
  for (int i = 0; i < kEach; ++i) v[i] = from[min((int)threadIdx.x + i * kJThreads, kWords - 1)];
#pragma unroll
  for (int i = 0; i < kEach; ++i)
    if ((int)threadIdx.x + i * kJThreads < kWords) to[threadIdx.x + i * kJThreads] = v[i];
}

// k_jacobi for one system of at most 512 elements per workgroup, two per
// thread: the same sums, arranged for latency.  Such a launch (under 700
// workgroups at 2000 atoms) is a chain of memory round trips of 0.7 us and
// more, not of bytes:
//  * the workgroup's range comes from its index (the block map's formula) and
//    the next vector's slot from the state, instead of a map's load each;
//  * all pointers are read from the argument block at once;
//  * what does not depend on the DIIS state (segment ranges, right-hand side,
//    iterate) loads while the state does, then both elements' history and
//    segment shares together, without a branch between their loads;
//  * the 24 wave sums meet in one reduce-scatter (the lane pairs of wave_sum,
//    the same bits) instead of one six-stage sum each.
// Average launch of k_jacobi -> this kernel: 12.5 -> 5.8 us at 60 atoms, 18.9 ->
// 7.7 us at 200 atoms and lmax 10, 12.1 -> 7.7 us at 1000, 14.8 -> 12.5 us at
// 2000, 31.2 -> 26.9 us at 4096, 40.5 -> 37.4 us at 6400 atoms (lmax 8, the last
// size that it takes; FP32 history 35.9 -> 28.6); 36.0 in both at 20 000 atoms
// and lmax 4.
template <typename E>
__global__ __launch_bounds__(kJThreads) void k_jacobi_two(unsigned nn, unsigned nylm,
                                                          int diis_max, unsigned nbj,
                                                          const double *__restrict__ facl,
                                                          Systems sys) {
  const SysArgs a = sys.s[blockIdx.y];
  if (blockIdx.x == nbj) {   // (launched where k_diis_extrap follows)
    copy_state(a.st);
    return;
  }
  asm volatile("" ::"s"(a.rhs), "s"(a.y), "s"(a.yp), "s"(a.segoff), "s"(a.x), "s"(a.ed),
               "s"(a.st), "s"(a.yacc), "s"(a.part), "s"(facl));
  const DiisState *__restrict__ st = a.st;
  __shared__ double wpart[kJThreads / kWave][kMaxDots + 1];
  const bool done = st->done != 0;
  const int nmat = st->nmat;
  const unsigned cur = (unsigned)st->cur;
  int all[kDiisMax];
#pragma unroll
  for (int q = 0; q < kDiisMax; ++q) all[q] = st->slot[q];
  const unsigned end = nn * (blockIdx.x + 1) / nbj;
  unsigned k[2], lm[2];
  bool live[2];
  double rhs[2], x[2], f[2];
  int s0[2], s1[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    k[i] = nn * blockIdx.x / nbj + threadIdx.x + i * kJThreads;
    live[i] = k[i] < end;
    if (!live[i]) k[i] = end - 1;   // a duplicate whose results are dropped
    const unsigned c = k[i] / nylm;
    lm[i] = k[i] - c * nylm;
    rhs[i] = a.rhs[k[i]];
    x[i] = a.x[k[i]];
    f[i] = facl[lm[i]];
    s0[i] = a.segoff[c];
    s1[i] = a.segoff[c + 1];
  }
  const int off = nmat >= diis_max ? 10 : 0, ndot = nmat - off - 1;
  unsigned slot[kMaxDots];
#pragma unroll
  for (int q = 0; q < kMaxDots; ++q) {
    const int s = off ? all[q + 10 < kDiisMax ? q + 10 : 0] : all[q];
    slot[q] = (unsigned)(q < ndot ? s : all[0]);
  }
  // (keeps the loads above ahead of the test)
  asm volatile("" ::"v"(rhs[0]), "v"(rhs[1]), "v"(x[0]), "v"(x[1]), "v"(f[0]), "v"(f[1]),
               "v"(s0[0]), "v"(s0[1]), "v"(s1[0]), "v"(s1[1]));
  if (done) return;
  double acc[kMaxDots + 1];
#pragma unroll
  for (int q = 0; q <= kMaxDots; ++q) acc[q] = 0.0;
  // the loads of a thread follow the history's depth
  if (ndot <= 8)
    jacobi_two_elements<E, 8>(a, nn, nylm, k, live, lm, s0, s1, rhs, x, f, slot, cur, acc);
  else if (ndot <= 16)
    jacobi_two_elements<E, 16>(a, nn, nylm, k, live, lm, s0, s1, rhs, x, f, slot, cur, acc);
  else
    jacobi_two_elements<E, kMaxDots>(a, nn, nylm, k, live, lm, s0, s1, rhs, x, f, slot, cur, acc);
  const int wave = threadIdx.x / kWave;
  int base = 0, len = kMaxDots + 1;
  wave_reduce_split<0, kMaxDots + 1, double>(acc, base, len);
  static_assert(reduced_len(kMaxDots + 1, 6) == 1, "one value per lane");
  if (len > 0) wpart[wave][base] = acc[0];
  __syncthreads();
  const int q = threadIdx.x;
  if (q < ndot || q == kMaxDots)
    a.part[(size_t)(q == kMaxDots ? kDiisMax : q) * nbj + blockIdx.x] =
        (wpart[0][q] + wpart[1][q]) + (wpart[2][q] + wpart[3][q]);
}

// The DIIS bookkeeping of one iteration on one wave, on the bordered Gram matrix
// B (0-based here; the reference's b(r+1, c+1)) of n1 = nmat + 1 <= 25 rows,
// staged in LDS.
//
//   drop-10 rule   when nmat reached diis_max the 10 oldest vectors go: rows
//                  and columns 11.. move to 1.. (jacobi_diis.f90:216-227)
//   makeb          new row/column of dot products (jacobi_diis.f90:258-297)
//   gjinv          Gauss-Jordan with full pivoting, right-hand side e_1
//                  (jacobi_diis.f90:299-400).  Pivot: the largest |a(j,k)|
//                  over rows j and columns k not yet pivoted (piv(j) != 1,
//                  piv(k) == 0), first in row-major order on ties, as the
//                  reference's nested loops pick it; the inverse's column
//                  unscrambling does not touch the solution and is skipped.
constexpr int kB = kDiisMax;      // register columns per row (n1 <= 25)

// value of v in lane `src`; src must be wave-uniform (it is moved to an SGPR)
__device__ __forceinline__ double lane_value(double v, int src) {
  const int s = __builtin_amdgcn_readfirstlane(src);
  const long long bits = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(bits & 0xffffffffll), s);
  const int hi = __builtin_amdgcn_readlane((int)(bits >> 32), s);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

constexpr int kSmallThreads = 256;

// Tells the host, which polls the record, that the solve has ended.  Once per
// solve: a copy of the state's header after every second round cost two
// copy kernels (2.3 us each at 60 atoms, 4 us at 2000) in the round's chain.
__device__ __forceinline__ void post_done(DiisState *rec) {
  __threadfence_system();
  __hip_atomic_store(&rec->done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// An instance has ended with iteration it0, by one whole wave.  A batch's is
// folded into the summary, which is done when the last instance is; a single
// system's results go to the host's record.
__device__ __forceinline__ void instance_done(DiisState *sum, const DiisState *st, DiisState *rec,
                                              int it0, double norm, int ok) {
  if (sum) {
    if (lane_id() != 0) return;
    atomicMax(&sum->it, it0 + 1);
    atomicAnd(&sum->ok, ok);
    if (atomicSub(&sum->remaining, 1) == 1) {
      sum->done = 1;
      post_done(rec);
    }
    return;
  }
  for (int q = lane_id(); q <= min(it0, kMaxIter); q += kWave)
    rec->hist[q] = q == it0 ? norm : st->hist[q];
  if (lane_id() == 0) {
    rec->it = it0 + 1;
    rec->ok = ok;
  }
  __threadfence_system();   // the whole wave's stores before lane 0's flag
  if (lane_id() == 0) post_done(rec);
}

// lanes per summed value in the Gram-row reduction of k_diis_small
constexpr int kTPQ = 8;

// partials r, r + kTPQ, ... of one value, added in that order; K loads per
// lane are in flight together (indices past nb re-read the last partial and
// are not added, so that no load is conditional)
template <int K>
__device__ __forceinline__ double sum_partials(const double *__restrict__ src, int nb, int r) {
  double s = 0.0;
  for (int b0 = r; b0 < nb; b0 += kTPQ * K) {
    double v[K];
#pragma unroll
    for (int i = 0; i < K; ++i) v[i] = src[min(b0 + kTPQ * i, nb - 1)];
#pragma unroll
    for (int i = 0; i < K; ++i)
      if (b0 + kTPQ * i < nb) s += v[i];
  }
  return s;
}

// largest 32-bit value over the wave (the DPP combines of wave_sum)
__device__ __forceinline__ unsigned wave_max_u32(unsigned v) {
  v = max(v, partner_u32<5>(v));
  v = max(v, partner_u32<4>(v));
  v = max(v, partner_u32<3>(v));
  v = max(v, partner_u32<2>(v));
  v = max(v, partner_u32<1>(v));
  v = max(v, partner_u32<0>(v));
  return (unsigned)__builtin_amdgcn_readfirstlane((int)v);
}

// max(|a|, |b|) (fmax would first quieten each operand)
__device__ __forceinline__ double max_abs(double a, double b) {
  double m;
  asm("v_max_f64 %0, |%1|, |%2|" : "=v"(m) : "v"(a), "v"(b));
  return m;
}

constexpr int kGramSums = kPartStride + 2;
// the staged B: kB rows of kBs doubles (an odd stride: a column's rows fall into
// different banks), and room for the new row after the oldest have gone
constexpr int kBs = kB + 2, kStage = (kB + 1) * kBs;

// The Gram-row dot products and the increment norms of the previous iteration
// into red: value q < 26 is the sum of nblk workgroup partials part[q nbj ..],
// values 26 and 27 those of nblk_e partials part_e0 and part_e1.  Eight
// consecutive lanes share a value, each sums every eighth partial, so that all
// loads are in flight together, and the eight partial sums meet in three
// lane-pair stages within the group.
__device__ __forceinline__ void gram_sums(int tid, int nblk, int nblk_e,
                                          const double *__restrict__ part, int nbj,
                                          const double *__restrict__ part_e0,
                                          const double *__restrict__ part_e1, double *red) {
#pragma clang fp contract(off)
  const int q = tid / kTPQ, r = tid % kTPQ;
  const bool norm_row = q >= kPartStride;
  const double *src = q > kPartStride ? part_e1 : norm_row ? part_e0 : part + (size_t)q * nbj;
  const int nb = norm_row ? nblk_e : nblk;
  // (a wave's eight values need as many loads as the longest of them)
  const bool last = __builtin_amdgcn_readfirstlane(tid / kWave) == kPartStride * kTPQ / kWave;
  const int most = last ? max(nblk, nblk_e) : nblk;
  double s;
  if (most <= kTPQ * 8)
    s = sum_partials<8>(src, nb, r);
  else if (most <= kTPQ * 16)
    s = sum_partials<16>(src, nb, r);
  else
    s = sum_partials<24>(src, nb, r);
  s += partner<3>(s);
  s += partner<4>(s);
  s += partner<5>(s);
  if (r == 0 && q < kGramSums) red[q] = s;
}

// `per` >= 192 threads take the words of the state's B through registers
// (load_b) to LDS (stage_b).
constexpr int kBWords = (kB * kB + 191) / 192;
__device__ __forceinline__ void load_b(const DiisState *st, int t, int per,
                                       double (&v)[kBWords]) {
#pragma unroll
  for (int i = 0; i < kBWords; ++i) v[i] = st->b[min(t + i * per, kB * kB - 1)];
}
__device__ __forceinline__ void stage_b(double *bs, int t, int per, const double (&v)[kBWords]) {
#pragma unroll
  for (int i = 0; i < kBWords; ++i) {
    const int q = t + i * per;
    if (q < kB * kB) bs[q / kB * kBs + q % kB] = v[i];
  }
}

// Row and column nmat + off of the staged B for the new vector, by one wave:
// the border's 1, the dots, the self dot.
__device__ __forceinline__ void add_row(double *bs, const double *red, int off, int nmat) {
  const int c = min(lane_id(), nmat);
  const double dot = red[c == nmat ? kDiisMax : max(c - 1, 0)], v = c == 0 ? 1.0 : dot;
  bs[(nmat + off) * kBs + c + off] = v;
  bs[(c + off) * kBs + nmat + off] = v;
  wave_lds_sync();
}

// Entry (r, c) of the bordered matrix: row and column 0 are (0, 1, 1, ..), the
// others are the staged B's, `off` rows and columns further on (0, or 10 when
// the oldest vectors go).
__device__ __forceinline__ double border(const double *bs, int off, int r, int c) {
  const double v = bs[(r + off) * kBs + c + off];
  const double edge = r == c ? 0.0 : 1.0;
  return r == 0 || c == 0 ? edge : v;
}

// Gauss-Jordan with full pivoting on the bordered system of k_diis_small,
// n1 = nmat + 1 <= 2 J rows, by one wave without barriers.  Lane L works on row
// r = L & 31 and on the columns 2 j + (L >> 5), j < J.  A row exchange of the
// reference is an exchange of two `pos` values (a lane's current row index);
// the right-hand side e_1 is bv.
//   Pivot: the largest |a(j, k)| over the rows and columns not yet pivoted,
// first in row-major order of the current indices on ties, as the reference's
// nested loops pick it.  Each lane takes the maximum of its own columns and
// the first column that has it; then the high words meet in six 32-bit
// lane-pair stages, and only where several lanes share the largest high word
// do the low words and the row-major codes (pos * 32 + column) follow.  A
// pivoted column holds the in-place inverse, which neither later pivots nor
// the solution read: it becomes zero, which is never a pivot, and stays zero,
// the pivot rows' entries being zero there too.
//   NaN is never a pivot (it compares with nothing in the reference's search; the
// largest of a lane's values leaves it out, and a lane that has nothing else
// takes no part), and once nothing else is left the system is singular: the
// iteration keeps the Jacobi step and DIIS starts again.
//   The pivot row reaches the other lanes through LDS (in issue order within
// the wave, no barrier).  The update a - pc * dum keeps the reference's two
// roundings: `keep` is 1, and 0 with dum = -1 on the pivot row, whose result
// is pc itself.
//   Bound by the issue of one wave, about 250 instructions a step at J = 13.
// One wave rather than four: with four (four columns to a lane) every step
// held a workgroup barrier, an exchange of candidates through LDS and two
// six-stage reductions of 64-bit values.  Average launch of k_diis_small, four
// waves -> one wave and its loads unchained: 15.5 -> 9.8 us at 60 atoms (up
// to 22 rows), 20.9 -> 13.7 us at 2000 atoms (up to 25), 19.2 -> 12.6 us on a
// batch of 64 molecules.  B staged in LDS by the whole workgroup instead of row
// by row in registers, the candidates' inverses ahead of the search's end and
// the dots of few partials not padded to the norm's number: 13.7 -> 12.9 us at
// 2000 atoms.
template <int J>
__device__ __forceinline__ bool eliminate(const double *bs, int off, int nmat, double *rowbuf,
                                          double &bv, int &pos) {
#pragma clang fp contract(off)
  constexpr int JP = J <= 4 ? 4 : J <= 8 ? 8 : 16;
  typedef double Row __attribute__((ext_vector_type(JP)));
  const int lane = lane_id(), r = lane & 31, half = lane >> 5;
  const int n1 = nmat + 1;
  Row g;
#pragma unroll
  for (int j = 0; j < JP; ++j) g[j] = 0.0;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int c = 2 * j + half;
    double v = border(bs, off, min(r, nmat), min(c, nmat));
    asm volatile("" : "+v"(v));   // (unconditional: all loads in flight together)
    g[j] = (r < n1 && c < n1) ? v : 0.0;
  }
  bv = (r == 0) ? 1.0 : 0.0;
  pos = r;
  bool rowlive = r < n1;
  for (int it = 0; it < n1; ++it) {
    // the lane's largest value and its first column
    double m[J];
#pragma unroll
    for (int j = 0; j < J; j += 2) m[j] = max_abs(g[j], j + 1 < J ? g[j + 1] : g[j]);
#pragma unroll
    for (int w = 2; w < J; w *= 2)
#pragma unroll
      for (int j = 0; j + w < J; j += 2 * w) m[j] = max_abs(m[j], m[j + w]);
    const double big = rowlive && m[0] > 0.0 ? m[0] : 0.0;   // (NaN: no candidate)
    int jc = 0;
#pragma unroll
    for (int j = J - 1; j >= 0; --j) jc = (fabs(g[j]) == big) ? j : jc;
    const int code = pos * 32 + 2 * jc + half;
    // every lane inverts its own candidate while the search goes on
    double rec = 1.0 / big;
    const unsigned long long bits = (unsigned long long)__double_as_longlong(big);
    const unsigned hi = (unsigned)(bits >> 32), lo = (unsigned)bits;
    const unsigned mhi = wave_max_u32(hi);
    asm volatile("" : "+v"(rec));   // (not after the search: it fills the search's waits)
    unsigned long long cand = __ballot(hi == mhi);
    if (__popcll(cand) > 1) {
      const unsigned mlo = wave_max_u32(hi == mhi ? lo : 0u);
      const bool tie = (hi == mhi) & (lo == mlo);
      if (mhi == 0u && mlo == 0u) return false;   // nothing left above zero
      cand = __ballot(tie);
      if (__popcll(cand) > 1) {
        const unsigned first = wave_max_u32(tie ? ~(unsigned)code : 0u);
        cand = __ballot(tie && ~(unsigned)code == first);
      }
    }
    const int src = __builtin_amdgcn_readfirstlane(__ffsll(cand) - 1);
    const int best = __builtin_amdgcn_readlane(code, src);
    const int lr = src & 31, hc = src >> 5;
    const int irow = best >> 5, icol = best & 31, jj = icol >> 1;
    // the pivot column: the multipliers a(j, icol) of all rows, in both halves
    const double col = g[jj];
    const double d = lane_value(col, src);
    if (d == 0.0) return false;
    g[jj] = (half == hc) ? 0.0 : col;
    const bool prow = r == lr;
    if (prow) {
#pragma unroll
      for (int j = 0; j < J; ++j) rowbuf[half * 16 + j] = g[j];
    }
    wave_lds_sync();
    const unsigned long long cb = (unsigned long long)__double_as_longlong(col);
    const auto sl = __builtin_amdgcn_permlane32_swap((unsigned)cb, (unsigned)cb, false, false);
    const auto sh = __builtin_amdgcn_permlane32_swap((unsigned)(cb >> 32), (unsigned)(cb >> 32),
                                                     false, false);
    // (the swap of a register with itself leaves the lower half's values in
    // the first result and the upper half's in the second, in all lanes)
    const unsigned long long db = ((unsigned long long)(hc ? sh[1] : sh[0]) << 32) |
                                  (hc ? sl[1] : sl[0]);
    const double dum = prow ? -1.0 : __longlong_as_double((long long)db);
    const double keep = prow ? 0.0 : 1.0;
    const double pinv = __builtin_copysign(lane_value(rec, src), d);
    double pr[J];
#pragma unroll
    for (int j = 0; j < J; ++j) pr[j] = rowbuf[half * 16 + j];
    wave_lds_sync();
    pos = prow ? icol : (pos == icol ? irow : pos);
    rowlive = rowlive & !prow;
    const double bp = lane_value(bv, lr) * pinv;
    bv = __builtin_fma(bv, keep, -(bp * dum));
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const double pc = pr[j] * pinv;
      g[j] = __builtin_fma(g[j], keep, -(pc * dum));
    }
  }
  return true;
}

// eliminate with the register count of a lane that the system's size needs
__device__ __forceinline__ bool eliminate_any(const double *bs, int off, int nmat,
                                              double *rowbuf, double &bv, int &pos) {
  bool ok;
  if (nmat < 8) ok = eliminate<4>(bs, off, nmat, rowbuf, bv, pos);
  else if (nmat < 14) ok = eliminate<7>(bs, off, nmat, rowbuf, bv, pos);
  else if (nmat < 20) ok = eliminate<10>(bs, off, nmat, rowbuf, bv, pos);
  else ok = eliminate<13>(bs, off, nmat, rowbuf, bv, pos);
  return ok;
}

// The new B into the state, by one wave: the new row and column, or all of it
// where the oldest vectors went.
__device__ __forceinline__ void store_b(const double *bs, int off, int nmat, DiisState *st) {
  const int lane = lane_id();
  if (off) {
    for (int q = lane; q < kB * kB; q += kWave) {
      const int r = q / kB, c = q % kB;
      if (r <= nmat && c <= nmat) st->b[q] = border(bs, off, r, c);
    }
  } else if (lane <= nmat) {
    const double v = border(bs, 0, nmat, lane);
    st->b[nmat * kB + lane] = v;
    st->b[lane * kB + nmat] = v;
  }
}

// logical slots once the oldest have been recycled: j <- j + 10 for j < nmat,
// the recycled ones after
__device__ __forceinline__ int recycle(int myslot, int off, int nmat, int diis_max) {
  const int lane = lane_id();
  const int src = lane < nmat ? lane + 10 : lane - nmat;
  const int moved = __shfl(myslot, src < diis_max ? src : 0, kWave);
  return off ? moved : myslot;
}

__global__ __launch_bounds__(kSmallThreads) void k_diis_small(
    int diis_max, int nbj, int nbe, int nsph_all, const int *__restrict__ jboff,
    const int *__restrict__ eboff, const int *__restrict__ soff, int ninst, int maxit,
    Systems sys) {
#pragma clang fp contract(off)
  const SysArgs &q0 = sys.s[blockIdx.y];
  const int inst = blockIdx.x;
  DiisState *__restrict__ st = q0.st + inst;
  const int tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
  // Every state word, the rows of B and the workgroup partials are loaded at
  // once, none behind a test of another (a launch is a chain of memory round
  // trips of about 0.7 us each): the block ranges of a single system come
  // with the launch, and the partials of Gram dots that do not exist yet are
  // read and not used.
  const int done = st->done;
  const double tol = st->tol;
  int nmat = st->nmat;
  const int it0 = st->it;
  const bool pending = st->pending_norm != 0;
  int jb = 0, eb = 0, nblk = nbj, nblk_e = nbe, nsph = nsph_all;
  if (ninst > 1) {
    jb = jboff[inst];
    eb = eboff[inst];
    nblk = jboff[inst + 1] - jb;
    nblk_e = eboff[inst + 1] - eb;
    nsph = soff[inst + 1] - soff[inst];
  }
  DiisState *sum = ninst > 1 ? q0.st + ninst : nullptr;
  int myslot = st->slot[min(lane, kDiisMax - 1)];
  __shared__ double bs[kStage];
  __shared__ double red[kGramSums];
  double old[kBWords];
  load_b(st, tid, kSmallThreads, old);
  gram_sums(tid, nblk, nblk_e, q0.part + jb, nbj, q0.part_e + eb, q0.part_e + eb, red);
  stage_b(bs, tid, kSmallThreads, old);
  __syncthreads();
  if (done) return;
  const int off = (nmat >= diis_max) ? 10 : 0;
  const int lastslot = __builtin_amdgcn_readlane(myslot, __builtin_amdgcn_readfirstlane(nmat - 1));
  if (pending) {
    // rms of the per-sphere norms and the convergence test of the previous
    // iteration (rmsvec, jacobi_diis.f90:405-438; jacobi_diis.f90:153-156),
    // evaluated alike by every thread
    const double norm = sqrt(red[kPartStride] / (double)nsph);
    const bool stop = norm < tol || it0 + 1 >= maxit;
    if (tid == 0) {
      if (it0 <= kMaxIter) st->hist[it0] = norm;
      st->it = it0 + 1;
      st->norm = norm;
      st->ok = norm < tol;
      st->pending_norm = 0;
      if (stop) st->done = 1;
    }
    if (stop && wave == 0) instance_done(sum, st, q0.rec, it0, norm, norm < tol);
    if (stop) return;
  }
  // the bordered system is one wave's work from here on
  if (wave != 0) return;
  nmat -= off;
  myslot = recycle(myslot, off, nmat, diis_max);
  add_row(bs, red, off, nmat);
  // persist B and the slot map; k_extrap leaves this iteration's norm
  store_b(bs, off, nmat, st);
  if (lane < diis_max) st->slot[lane] = myslot;
  if (lane == 0) {
    st->pending_norm = 1;
    q0.newslot[inst] = lastslot;
  }

  __shared__ __align__(16) double rowbuf[32];
  double bv;
  int pos;
  const bool ok = eliminate_any(bs, off, nmat, rowbuf, bv, pos);
  if (ok) {
    if (lane <= nmat && pos >= 1) st->coef[pos - 1] = bv;
  }
  const int cur = __builtin_amdgcn_readlane(myslot, ok ? __builtin_amdgcn_readfirstlane(nmat) : 0);
  if (lane == 0) {
    st->cur = cur;
    if (!ok) {
      st->nmat = 1;
      st->ncoef = 0;
      st->singular += 1;
    } else {
      st->ncoef = nmat;
      st->nmat = nmat + 1;
    }
  }
}

// x_new = sum_i c_i x_i (or the plain Jacobi step), increment norm partials
// per sphere (hsnorm, ddcosmo.f90:1233-1271), x <- x_new, and xs = cf x_new
// where the system keeps it.  The workgroup streams its spheres' elements
// with all 256 threads (consecutive threads, consecutive elements) and
// leaves each element's norm term in LDS; then one thread per sphere adds
// its terms in lm order, as hsnorm does.  Spheres beyond the LDS stage are
// taken in chunks.
constexpr int kExtrapTerms = 2048;   // staged norm terms per workgroup (nylm <= 289)

__global__ __launch_bounds__(kJThreads) void k_extrap(int nylm, size_t nn, int diis_max,
                                                      const int4 *__restrict__ eblk,
                                                      const double *__restrict__ invl1,
                                                      const double *__restrict__ cf,
                                                      Systems sys) {
  const SysArgs &q0 = sys.s[blockIdx.y];
  const int4 blk = eblk[blockIdx.x];   // instance, spheres blk.y .. blk.z - 1
  const DiisState *__restrict__ st = q0.st + blk.x;
  if (st->done) return;
  const double *__restrict__ xd = q0.xd;
  const double *__restrict__ xnew = q0.xnew;
  const int *__restrict__ newslot = q0.newslot + blk.x;
  double *__restrict__ x = q0.x;
  double *__restrict__ xsc = q0.xs;
  double *__restrict__ incw = q0.inc;
  const bool xs_inc = q0.xs_inc != 0;
  double *__restrict__ part = q0.part_e;
  __shared__ double lds[kJThreads / kWave];
  __shared__ double terms[kExtrapTerms];
  const int ncoef = diis_max > 0 ? st->ncoef : 0;
  const double *xs[kDiisMax];
  double cs[kDiisMax];
#pragma unroll
  for (int q = 0; q < kDiisMax; ++q) {
    xs[q] = (q < ncoef) ? xd + (size_t)st->slot[q] * nn : nullptr;
    cs[q] = (q < ncoef) ? st->coef[q] : 0.0;
  }
  const double *xj = diis_max > 0 ? xd + (size_t)(*newslot) * nn : xnew;
  const int chunk = kExtrapTerms / nylm;   // spheres per pass, at least 7
  const int step = kJThreads % nylm;       // lm advance per thread stride
  double usq = 0.0;
  for (int c0 = blk.y; c0 < blk.z; c0 += chunk) {
    const int c1 = min(blk.z, c0 + chunk);
    const unsigned ne = (unsigned)(c1 - c0) * (unsigned)nylm;
    const size_t e0 = (size_t)c0 * nylm;
    int lm = (int)(threadIdx.x % (unsigned)nylm);
    // two elements per step (j and j + 256), all their loads issued before
    // either one's stores
    for (unsigned j = threadIdx.x; j < ne; j += 2 * kJThreads) {
      const bool two = j + kJThreads < ne;
      int lm2 = lm + step;
      if (lm2 >= nylm) lm2 -= nylm;
      const size_t k = e0 + j, k2 = two ? k + kJThreads : k;
      double xn = 0.0, xn2 = 0.0;
      if (ncoef > 0) {
        double a[kDiisMax], b[kDiisMax];
#pragma unroll
        for (int q = 0; q < kDiisMax; ++q) {
          a[q] = (q < ncoef) ? xs[q][k] : 0.0;
          b[q] = (q < ncoef) ? xs[q][k2] : 0.0;
        }
#pragma unroll
        for (int q = 0; q < kDiisMax; ++q) {
          if (q < ncoef) {
            xn = xn + cs[q] * a[q];
            xn2 = xn2 + cs[q] * b[q];
          }
        }
      } else {
        xn = xj[k];
        xn2 = xj[k2];
      }
      const double x1 = x[k], x2 = x[k2];
      const double inc = xn - x1, inc2 = xn2 - x2;
      x[k] = xn;
      if (xsc) xsc[k] = cf[lm] * (xs_inc ? inc : xn);
      if (incw) incw[k] = inc;
      terms[j] = invl1[lm] * inc * inc;
      if (two) {
        x[k2] = xn2;
        if (xsc) xsc[k2] = cf[lm2] * (xs_inc ? inc2 : xn2);
        if (incw) incw[k2] = inc2;
        terms[j + kJThreads] = invl1[lm2] * inc2 * inc2;
      }
      lm = lm2 + step;
      if (lm >= nylm) lm -= nylm;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < c1 - c0; i += kJThreads) {
      const double *t = terms + (size_t)i * nylm;
      double sq = 0.0;
      for (int l = 0; l < nylm; ++l) sq += t[l];
      const double u = sqrt(sq);
      usq += u * u;
    }
    __syncthreads();
  }
  const double tot = block_sum_256(usq, lds);
  if (threadIdx.x == 0) part[blockIdx.x] = tot;
}

// Sum of the squared norms of `count` <= 64 spheres by one wave, a sphere to a
// lane: its nylm terms from LDS in order, eight loaded ahead of the additions.
__device__ __forceinline__ double sphere_norms(const double *terms, unsigned count,
                                               unsigned nylm) {
  double usq = 0.0;
  const unsigned lane = (unsigned)lane_id();
  if (lane < count) {
    const double *t = terms + lane * nylm;
    const int last = (int)nylm - 1;
    double sq = 0.0, ahead[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) ahead[i] = t[min(i, last)];
    for (int l = 0; l <= last; l += 8) {
      double v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[i] = ahead[i];
        ahead[i] = t[min(l + 8 + i, last)];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (l + i <= last) sq += v[i];
    }
    const double u = sqrt(sq);
    usq += u * u;
  }
  return wave_sum(usq);
}

// one element of the C newest history vectors, all loads in flight together
template <int C>
__device__ __forceinline__ void load_history_c(const double *__restrict__ xd, unsigned nn,
                                               unsigned k, const unsigned (&slot)[kB - 1],
                                               double (&v)[kB - 1]) {
#pragma unroll
  for (int q = 0; q < C; ++q)
    v[q] = load_at<double>(xd, (slot[q] * nn + k) * (unsigned)sizeof(double));
#pragma unroll
  for (int q = C; q < kB - 1; ++q) v[q] = 0.0;
}

// ... at least `depth` of them
__device__ __forceinline__ void load_history(const double *__restrict__ xd, unsigned nn,
                                             unsigned k, const unsigned (&slot)[kB - 1], int depth,
                                             double (&v)[kB - 1]) {
  if (depth <= 8) load_history_c<8>(xd, nn, k, slot, v);
  else if (depth <= 16) load_history_c<16>(xd, nn, k, slot, v);
  else load_history_c<kB - 1>(xd, nn, k, slot, v);
}

// x_new = sum_i c_i x_i of one element: the history values of the C >= ncoef
// newest slots are loaded together (those past ncoef re-read slot 0 and are
// not added).
template <int C>
__device__ __forceinline__ double extrapolate(const double *__restrict__ xd, unsigned nn,
                                              unsigned k, const unsigned (&slot)[kDiisMax],
                                              const double (&coef)[kDiisMax], int ncoef) {
  double v[C];
#pragma unroll
  for (int q = 0; q < C; ++q)
    v[q] = load_at<double>(xd, (slot[q] * nn + k) * (unsigned)sizeof(double));
  double xn = 0.0;
#pragma unroll
  for (int q = 0; q < C; ++q)
    if (q < ncoef) xn = xn + coef[q] * v[q];
  return xn;
}

// k_extrap for one system whose workgroups stage all their spheres at once
// (at most kExtrapTerms elements, 64 spheres), one element per thread of 512:
// the same sums, arranged for latency as k_jacobi_two is.  The workgroup's
// spheres come from its index, the slots and coefficients load with the state
// and beside the iterate, the history without a branch between its loads, and
// the serial sum of a sphere's norm terms reads LDS eight terms ahead of its
// additions.  512 threads for the usual 200..480 elements: two elements to
// each of 256 threads took 198 registers and two rounds of workgroups at 2000
// atoms.  Average launch of k_extrap -> this kernel: 9.2 -> 4.6 us at 60 atoms,
// 12.1 -> 6.9 us at 200 atoms and lmax 10, 13.2 -> 9.0 us at 1000, 15.7 -> 14.2
// us at 2000 atoms (lmax 8; near its bytes there), 43.2 -> 37.5 us at 6400.
constexpr int kExtrapThreads = 512;

__global__ __launch_bounds__(kExtrapThreads) void k_extrap_one(
    unsigned n, unsigned nylm, unsigned nn, unsigned nbe, const double *__restrict__ invl1,
    const double *__restrict__ cf, Systems sys) {
  const SysArgs a = sys.s[blockIdx.y];
  asm volatile("" ::"s"(a.x), "s"(a.xs), "s"(a.xd), "s"(a.st), "s"(a.inc), "s"(a.newslot),
               "s"(a.part_e), "s"(invl1), "s"(cf));
  const DiisState *__restrict__ st = a.st;
  __shared__ double terms[kExtrapTerms];
  const bool done = st->done != 0;
  const int ncoef = st->ncoef;
  const unsigned newest = (unsigned)*a.newslot;
  unsigned slot[kDiisMax];
  double coef[kDiisMax];
#pragma unroll
  for (int q = 0; q < kDiisMax; ++q) {
    slot[q] = (unsigned)st->slot[q];
    coef[q] = st->coef[q];
  }
  // (the slots past ncoef need not exist: a shorter history has fewer of them)
#pragma unroll
  for (int q = 0; q < kDiisMax; ++q)
    slot[q] = __builtin_amdgcn_readfirstlane((int)(q < ncoef ? slot[q] : slot[0]));
  if (done) return;
  const unsigned c0 = n * blockIdx.x / nbe, c1 = n * (blockIdx.x + 1) / nbe;
  const unsigned ne = (c1 - c0) * nylm, e0 = c0 * nylm;
  const bool xs_inc = a.xs_inc != 0;
  for (unsigned j = threadIdx.x; j < ne; j += kExtrapThreads) {
    const unsigned k = e0 + j, lm = k % nylm;
    const double x = a.x[k], il = invl1[lm], cl = cf[lm];
    double xn;
    if (ncoef == 0)   // the plain Jacobi step
      xn = a.xd[(size_t)newest * nn + k];
    else if (ncoef <= 8)
      xn = extrapolate<8>(a.xd, nn, k, slot, coef, ncoef);
    else if (ncoef <= 16)
      xn = extrapolate<16>(a.xd, nn, k, slot, coef, ncoef);
    else
      xn = extrapolate<kDiisMax - 1>(a.xd, nn, k, slot, coef, ncoef);
    const double inc = xn - x;
    a.x[k] = xn;
    if (a.xs) a.xs[k] = cl * (xs_inc ? inc : xn);
    if (a.inc) a.inc[k] = inc;
    terms[j] = il * inc * inc;
  }
  __syncthreads();
  if (threadIdx.x >= kWave) return;
  const double usq = sphere_norms(terms, c1 - c0, nylm);
  if (threadIdx.x == 0) a.part_e[blockIdx.x] = usq;
}

// k_diis_small and k_extrap_one in one launch, for one system whose workgroups
// have a compute unit each: every workgroup solves the bordered system for itself (its
// wave 0; the same operations, so the same weights in all of them), while its
// other waves, one element to a thread, have the iterate and the history in
// flight; then they extrapolate as k_extrap_one does.
//   They read the copy of the state that k_jacobi_two left behind it, and the
// first of them writes the state.  A workgroup may leave its norm partial
// while another still sums the previous iteration's, so the two iterations'
// partials alternate between two arrays, by the iteration's parity.
//   Bound by the elimination (one wave's serial chain, 0.6 us a row).  Launches
// of 7.2 to 21 us and 4.6 us become one of 8.3 to 21.4 us at 60 atoms; a whole
// step, two launches -> one: 60 atoms 1203 -> 1165 us, 259 atoms 1510 -> 1469,
// 400 atoms 1538 -> 1484 (lmax 6).
__global__ __launch_bounds__(kExtrapThreads, 4) void k_diis_extrap(
    unsigned n, unsigned nylm, unsigned nn, unsigned nbe, int nbj, int diis_max, int maxit,
    const double *__restrict__ invl1, const double *__restrict__ cf, Systems sys) {
  const SysArgs s = sys.s[blockIdx.y];
  asm volatile("" ::"s"(s.x), "s"(s.xs), "s"(s.xd), "s"(s.st), "s"(s.inc), "s"(s.part),
               "s"(s.part_e), "s"(invl1), "s"(cf));
  const DiisState *__restrict__ old = s.st + 1;
  const int tid = threadIdx.x, lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const unsigned nelem = blockDim.x - kWave;   // one element to a thread
  __shared__ double terms[kExtrapTerms];
  __shared__ double bs[kStage];
  __shared__ double red[kGramSums];
  __shared__ double weight[kB];
  __shared__ __align__(16) double rowbuf[32];
  __shared__ int solved;
  const bool done = old->done != 0, pending = old->pending_norm != 0;
  const double tol = old->tol;
  const int nmat0 = old->nmat, it0 = old->it;
  const int off = nmat0 >= diis_max ? 10 : 0, nmat = nmat0 - off;   // nmat: the weights' number
  const unsigned c0 = n * blockIdx.x / nbe, c1 = n * (blockIdx.x + 1) / nbe;
  const unsigned ne = (c1 - c0) * nylm, e0 = c0 * nylm;
  // the previous iteration's norm and convergence test, as in k_diis_small
  const auto test = [&](double &norm) {
    norm = sqrt(red[kPartStride + (it0 & 1)] / (double)(int)n);
    return pending && (norm < tol || it0 + 1 >= maxit);
  };
  double norm;
  // (two paths with the same barriers, so that no register of one is kept in
  // the other)
  if (wave == 0) {
    const int slots = old->slot[min(lane, kDiisMax - 1)];
    gram_sums(tid, nbj, (int)nbe, s.part, nbj, s.part_e, s.part_e + nbe, red);
    __syncthreads();
    if (done) return;
    const bool stop = test(norm);
    double bv;
    int pos;
    bool ok = false;
    if (!stop) {
      add_row(bs, red, off, nmat);
      ok = eliminate_any(bs, off, nmat, rowbuf, bv, pos);
      if (ok && lane <= nmat && pos >= 1) weight[pos - 1] = bv;
      if (lane == 0) solved = ok;
    }
    __syncthreads();
    if (blockIdx.x == 0) {
      DiisState *st = s.st;
      if (pending && lane == 0) {
        if (it0 <= kMaxIter) st->hist[it0] = norm;
        st->it = it0 + 1;
        st->norm = norm;
        st->ok = norm < tol;
      }
      if (stop) {
        instance_done(nullptr, st, s.rec, it0, norm, norm < tol);
        if (lane == 0) st->done = 1;
      } else {
        store_b(bs, off, nmat, st);
        const int myslot = recycle(slots, off, nmat, diis_max);
        if (lane < diis_max) st->slot[lane] = myslot;
        const int cur = __builtin_amdgcn_readlane(
            myslot, __builtin_amdgcn_readfirstlane(ok ? nmat : 0));
        if (lane == 0) {
          st->cur = cur;
          st->nmat = ok ? nmat + 1 : 1;
          st->pending_norm = 1;
          if (!ok) st->singular += 1;
        }
      }
    }
    if (!stop) __syncthreads();
    return;
  }
  // the old B into LDS, and beside it what the elements need
  double b[kBWords];
  load_b(old, tid - kWave, nelem, b);
  unsigned slot[kB - 1];
  {
    int all[kDiisMax];
#pragma unroll
    for (int q = 0; q < kDiisMax; ++q) all[q] = old->slot[q];
#pragma unroll
    for (int q = 0; q < kB - 1; ++q) {   // (past nmat: slot 0, read and not added)
      const int s = off ? all[q + 10 < kDiisMax ? q + 10 : 0] : all[q];
      slot[q] = (unsigned)__builtin_amdgcn_readfirstlane(q < nmat ? s : all[0]);
    }
  }
  unsigned k = e0 + min((unsigned)tid - kWave, ne - 1);
  double x = s.x[k], il = invl1[k % nylm], cl = cf[k % nylm], v[kB - 1];
  if (tid < kGramSums * kTPQ)
    gram_sums(tid, nbj, (int)nbe, s.part, nbj, s.part_e, s.part_e + nbe, red);
  stage_b(bs, tid - kWave, nelem, b);
  load_history(s.xd, nn, k, slot, nmat, v);
  __syncthreads();
  if (done) return;
  const bool stop = test(norm);
  __syncthreads();
  if (stop) return;
  const bool ok = solved != 0;
  for (unsigned j = (unsigned)tid - kWave; j < ne; j += nelem) {
    if (j >= nelem) {
      k = e0 + j;
      x = s.x[k];
      il = invl1[k % nylm];
      cl = cf[k % nylm];
      load_history(s.xd, nn, k, slot, nmat, v);
    }
    double xn = 0.0;
    if (ok) {
#pragma unroll
      for (int q = 0; q < kB - 1; ++q)
        if (q < nmat) xn = xn + weight[q] * v[q];
    } else {   // the plain Jacobi step: the newest vector
#pragma unroll
      for (int q = 0; q < kB - 1; ++q)
        if (q == nmat - 1) xn = v[q];
    }
    const double inc = xn - x;
    s.x[k] = xn;
    if (s.xs) s.xs[k] = cl * (s.xs_inc ? inc : xn);
    if (s.inc) s.inc[k] = inc;
    terms[j] = il * inc * inc;
  }
  __syncthreads();
  if (wave != 1) return;
  const double usq = sphere_norms(terms, c1 - c0, nylm);
  const int it = pending ? it0 + 1 : it0;   // this iteration
  if (lane == 0) s.part_e[(it & 1) * nbe + blockIdx.x] = usq;
}

// rms of the per-sphere norms and the convergence test (rmsvec,
// jacobi_diis.f90:405-438; jacobi_diis.f90:153-156)
__global__ __launch_bounds__(kWave) void k_norm(const int *__restrict__ eboff,
                                                const int *__restrict__ soff, int ninst,
                                                int maxit, Systems sys) {
  const int inst = blockIdx.x;
  DiisState *__restrict__ st = sys.s[blockIdx.y].st + inst;
  if (st->done) return;
  const double tol = st->tol;
  const double *__restrict__ part = sys.s[blockIdx.y].part_e;
  double s = 0.0;
  for (int b = eboff[inst] + threadIdx.x; b < eboff[inst + 1]; b += kWave) s += part[b];
  s = wave_sum(s);
  const double norm = sqrt(s / (double)(soff[inst + 1] - soff[inst]));
  const int it = st->it;
  const bool stop = norm < tol || it + 1 >= maxit;
  if (threadIdx.x == 0) {
    if (it <= kMaxIter) st->hist[it] = norm;
    st->it = it + 1;
    st->norm = norm;
    st->ok = norm < tol;
    st->done = stop;
  }
  if (stop)
    instance_done(ninst > 1 ? sys.s[blockIdx.y].st + ninst : nullptr, st, sys.s[blockIdx.y].rec,
                  it, norm, norm < tol);
}

// fresh states for the ninst instances and the summary of a batch
__global__ void k_diis_init(int ninst, double tol, DiisState *__restrict__ st) {
  const int q = blockIdx.x;
  DiisState *d = st + q;
  const int t = threadIdx.x;
  if (t < kDiisMax) d->slot[t] = t;
  if (t == 0) {
    d->nmat = 1;
    d->cur = 0;
    d->it = 0;
    d->done = 0;
    d->ok = q < ninst ? 0 : 1;
    d->singular = 0;
    d->pending_norm = 0;
    d->ncoef = 0;
    d->remaining = q < ninst ? 0 : ninst;
    d->norm = 0.0;
    d->tol = tol;
  }
}

// per instance: iterations as the reference reports them and the ok flag
__global__ void k_diis_results(int ninst, int maxit, const DiisState *__restrict__ st,
                               int *__restrict__ res) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= ninst) return;
  res[2 * q] = st[q].ok ? st[q].it : maxit + 1;
  res[2 * q + 1] = st[q].ok;
}

__global__ void k_ldm1x(size_t nn, int nylm, const double *__restrict__ facl,
                        const double *__restrict__ x, double *__restrict__ y) {
  size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < nn) y[k] = facl[k % nylm] * x[k];
}

__global__ __launch_bounds__(kJThreads) void k_hnorm_part(int nsph, int nylm,
                                                          const double *__restrict__ invl1,
                                                          const double *__restrict__ x,
                                                          double *__restrict__ part) {
  __shared__ double lds[kJThreads / kWave];
  const int wave = threadIdx.x / kWave, lane = lane_id(), wpb = kJThreads / kWave;
  double usq = 0.0;
  for (int i = blockIdx.x * wpb + wave; i < nsph; i += gridDim.x * wpb) {
    double s = 0.0;
    for (int lm = lane; lm < nylm; lm += kWave) {
      double v = x[(size_t)i * nylm + lm];
      s += invl1[lm] * v * v;
    }
    s = wave_sum(s);
    double u = sqrt(s);
    usq += u * u;
  }
  if (lane != 0) usq = 0.0;
  double tot = block_sum_256(usq, lds);
  if (threadIdx.x == 0) part[blockIdx.x] = tot;
}

__global__ __launch_bounds__(kWave) void k_sum_parts(int nblk, double scale,
                                                     const double *__restrict__ part,
                                                     double *__restrict__ out) {
  double s = 0.0;
  for (int b = threadIdx.x; b < nblk; b += kWave) s += part[b];
  s = wave_sum(s);
  if (threadIdx.x == 0) *out = scale * s;
}

// g(n,i) = -ui phi(ic) for exposed points (wghpot, ddcosmo.f90:1187-1224)
__global__ void k_wghpot(size_t np, const double *__restrict__ ui, const int *__restrict__ cavidx,
                         const double *__restrict__ phi, double *__restrict__ g) {
  size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  double u = ui[p];
  g[p] = (u != 0.0) ? -u * phi[cavidx[p]] : 0.0;
}

// partial dot products over the elements of each k_jacobi block
__global__ __launch_bounds__(kJThreads) void k_dot_part(const int4 *__restrict__ jblk,
                                                        const double *__restrict__ a,
                                                        const double *__restrict__ b,
                                                        double *__restrict__ part) {
  __shared__ double lds[kJThreads / kWave];
  const int4 blk = jblk[blockIdx.x];
  double s = 0.0;
  for (size_t k = (size_t)blk.y + threadIdx.x; k < (size_t)blk.z; k += kJThreads)
    s += a[k] * b[k];
  double tot = block_sum_256(s, lds);
  if (threadIdx.x == 0) part[blockIdx.x] = tot;
}

// out[q] = scale * sum of the partials of instance q's blocks, one wave each
__global__ __launch_bounds__(kWave) void k_inst_sum(const int *__restrict__ boff, double scale,
                                                    const double *__restrict__ part,
                                                    double *__restrict__ out) {
  const int q = blockIdx.x;
  double s = 0.0;
  for (int b = boff[q] + threadIdx.x; b < boff[q + 1]; b += kWave) s += part[b];
  s = wave_sum(s);
  if (threadIdx.x == 0) out[q] = scale * s;
}

int grid_blocks(size_t work, int per_block, int cap) {
  size_t b = (work + per_block - 1) / per_block;
  if (b < 1) b = 1;
  if (b > (size_t)cap) b = cap;
  return (int)b;
}

}  // namespace

int device_ldm1x(ddx_handle *h, hipStream_t s, const double *x, double *y) {
  size_t nn = (size_t)h->nylm * h->n;
  hipLaunchKernelGGL(k_ldm1x, dim3((nn + 255) / 256), dim3(256), 0, s, nn, h->nylm,
                     h->facl.p, x, y);
  DDX_HIP(hipGetLastError());
  return DDX_OK;
}

int device_hnorm(ddx_handle *h, const double *x, double *norm_host) {
  int nb = grid_blocks(h->n, kJThreads / kWave, 1024);
  DDX_TRY(h->part.reserve(1024 + 1));
  hipLaunchKernelGGL(k_hnorm_part, dim3(nb), dim3(kJThreads), 0, h->stream, h->n, h->nylm,
                     h->cf.p + h->nylm, x, h->part.p);
  DDX_HIP(hipGetLastError());
  DDX_TRY(h->energy.reserve(h->ninst + 4));
  double *out = h->energy.p + h->ninst + 1;
  hipLaunchKernelGGL(k_sum_parts, dim3(1), dim3(kWave), 0, h->stream, nb, 1.0, h->part.p, out);
  DDX_HIP(hipGetLastError());
  double s = 0.0;
  DDX_HIP(hipMemcpyAsync(&s, out, sizeof(double), hipMemcpyDeviceToHost, h->stream));
  DDX_HIP(hipStreamSynchronize(h->stream));
  *norm_host = sqrt(s / (double)h->n);
  return DDX_OK;
}

int build_rhs(ddx_handle *h, const double *d_phi, double *d_rhs) {
  Lane &ln = h->lane[0];   // lane 0 runs on the handle's stream
  DDX_TRY(ln.P.reserve(h->np));
  hipLaunchKernelGGL(k_wghpot, dim3((h->np + 255) / 256), dim3(256), 0, h->stream, h->np,
                     h->ui.p, h->cavidx.p, d_phi, ln.P.p);
  DDX_HIP(hipGetLastError());
  // rhs(lm, i) = sum_n Y(lm, n) w_n g(n, i)   (intrhs per sphere, cosmo.f90:114-116)
  return project(h, h->stream, 1.0, ln.P.p, d_rhs, nullptr, 1);
}

int energy_dot(ddx_handle *h, const double *a, const double *b, double scale, double *d_out) {
  DDX_TRY(h->part.reserve((size_t)h->nbj + 1));
  hipLaunchKernelGGL(k_dot_part, dim3(h->nbj), dim3(kJThreads), 0, h->stream, h->jblk.p, a, b,
                     h->part.p);
  DDX_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_inst_sum, dim3(h->ninst), dim3(kWave), 0, h->stream, h->jboff.p, scale,
                     h->part.p, d_out);
  DDX_HIP(hipGetLastError());
  return DDX_OK;
}

// Block maps of the solver kernels, from the instances' sphere ranges: each
// instance's elements (spheres) are split evenly over
// ceil(elements / 512) (ceil(spheres / sp)) workgroups, at most 1024 each.
// sp, the spheres per k_extrap workgroup, is 4 up to
// about 8000 spheres in all and grows to 32 for larger systems and batches,
// where the per-workgroup reads of the DIIS state would dominate.
int build_solver_maps(ddx_handle *h) {
  std::vector<int4> jb, eb;
  std::vector<int> jo(h->ninst + 1), eo(h->ninst + 1);
  const long long ny = h->nylm;
  const int sp = std::max(4, std::min(32, h->n / 2048 / 4 * 4));
  for (int q = 0; q < h->ninst; ++q) {
    const int s0 = h->h_soff[q], s1 = h->h_soff[q + 1];
    const long long e0 = s0 * ny, e1 = s1 * ny;
    jo[q] = (int)jb.size();
    const int nj = grid_blocks((size_t)(e1 - e0), kJThreads * 2, 1024);
    for (int j = 0; j < nj; ++j)
      jb.push_back(make_int4(q, (int)(e0 + (e1 - e0) * j / nj), (int)(e0 + (e1 - e0) * (j + 1) / nj), 0));
    eo[q] = (int)eb.size();
    const int ne = grid_blocks((size_t)(s1 - s0), sp, 1024);
    for (int j = 0; j < ne; ++j)
      eb.push_back(make_int4(q, s0 + (int)((long long)(s1 - s0) * j / ne),
                             s0 + (int)((long long)(s1 - s0) * (j + 1) / ne), 0));
  }
  jo[h->ninst] = (int)jb.size();
  eo[h->ninst] = (int)eb.size();
  if ((long long)h->n * ny > 0x7fffffffll) {
    set_error("nylm * nsph = %lld exceeds the 32-bit element index", (long long)h->n * ny);
    return DDX_ERR_CAPACITY;
  }
  h->nbj = (int)jb.size();
  h->nbe = (int)eb.size();
  const int nblk = (h->n + 15) / 16;   // workgroups of one projection pass
  h->ysplit = nblk >= 1024 ? 1 : std::min(kProjSplit, (1024 + nblk - 1) / nblk);
  DDX_TRY(h->jblk.reserve(jb.size()));
  DDX_TRY(h->eblk.reserve(eb.size()));
  DDX_TRY(h->jboff.reserve(jo.size()));
  DDX_TRY(h->eboff.reserve(eo.size()));
  hipStream_t s = h->stream;
  DDX_HIP(hipMemcpyAsync(h->jblk.p, jb.data(), jb.size() * sizeof(int4), hipMemcpyHostToDevice, s));
  DDX_HIP(hipMemcpyAsync(h->eblk.p, eb.data(), eb.size() * sizeof(int4), hipMemcpyHostToDevice, s));
  DDX_HIP(hipMemcpyAsync(h->jboff.p, jo.data(), jo.size() * sizeof(int), hipMemcpyHostToDevice, s));
  DDX_HIP(hipMemcpyAsync(h->eboff.p, eo.data(), eo.size() * sizeof(int), hipMemcpyHostToDevice, s));
  DDX_HIP(hipStreamSynchronize(s));   // (built once per handle)
  return DDX_OK;
}

namespace {
SysArgs sys_args(const ddx_handle *h, Lane &ln) {
  SysArgs a;
  a.rhs = ln.rhs;
  a.y = ln.y.p;
  a.ny = ln.star ? 1 : h->ysplit;
  a.yp = ln.star ? ln.yp.p : nullptr;
  a.segoff = h->segoff.p;
  a.x = ln.x;
  a.xs = ln.star ? nullptr : ln.xs.p;
  a.xd = ln.xd.p;
  a.ed = ln.ed.p;
  a.xnew = ln.xnew.p;
  a.part = ln.part.p;
  a.part_e = ln.part.p + (size_t)h->nbj * kPartStride;
  a.newslot = ln.misc.p;
  a.st = ln.diis.p;
  a.yacc = ln.incr ? ln.yacc.p : nullptr;
  a.acc = 0;
  // the increment is read by the FP32 L* operator only: the L X sweep of
  // an increment round reads xs = cf inc, which k_extrap writes as well
  a.inc = (ln.incr && ln.star) ? ln.inc.p : nullptr;
  a.xs_inc = 0;
  a.rec = ln.d_rec;
  return a;
}

// drops the timer records of one kernel class for rounds >= keep of a group
void drop_rounds(ddx_handle *h, int cls, int serial, int keep) {
  KernelTimer &t = h->ktimer[cls];
  size_t n = 0;
  for (size_t k = 0; k < t.recs.size(); ++k) {
    const KernelTimer::Rec &r = t.recs[k];
    if (r.solve == serial && r.round >= keep) {
      t.pool.push_back(r.b);
      t.pool.push_back(r.e);
    } else {
      t.recs[n++] = r;
    }
  }
  t.recs.resize(n);
}
}  // namespace

int solve_begin(ddx_handle *h, Lane &ln, int star, int diis_max, double tol, const double *d_rhs,
                double *d_x, int max_iter) {
  if (!(diis_max == 0 || (diis_max > 10 && diis_max <= kDiisMax))) {
    set_error("diis_max must be 0 or in 11..%d", kDiisMax);
    return DDX_ERR_ARG;
  }
  if (max_iter < 1 || max_iter > kMaxIter) {
    set_error("n_iter must be in 1..%d", kMaxIter);
    return DDX_ERR_ARG;
  }
  size_t nn = (size_t)h->nylm * h->n;
  DDX_TRY(ln.y.reserve(nn * kProjSplit));
  DDX_TRY(ln.xnew.reserve(nn));
  DDX_TRY(ln.xs.reserve(nn + 1));
  if (diis_max > 0) {
    DDX_TRY(ln.xd.reserve(nn * diis_max));
    DDX_TRY(ln.ed.reserve(nn * diis_max));
  }
  DDX_TRY(ln.part.reserve((size_t)h->nbj * kPartStride + 2 * (size_t)h->nbe + 1));
  // the L* sweep leaves per-segment sums that k_jacobi reads: its buffer must
  // not move once the solve has started
  if (star) DDX_TRY(ln.yp.reserve((size_t)h->nseg_cap * h->nylm + 1));
  DDX_TRY(ln.diis.reserve(h->ninst + 1));   // and the summary, or k_diis_extrap's copy
  DDX_TRY(ln.misc.reserve(h->ninst + 1));
  DDX_TRY(ln.res.reserve(2 * (size_t)h->ninst + 2));
  ln.star = star;
  ln.diis_max = diis_max;
  ln.max_iter = max_iter;
  ln.tol = tol;
  ln.rhs = d_rhs;
  ln.x = d_x;
  // with DIIS the norm of iteration k is evaluated by the DIIS kernel of
  // iteration k + 1, so up to max_iter + 1 rounds are enqueued
  ln.rounds = diis_max > 0 ? max_iter + 1 : max_iter;
  ln.enqueued = 0;
  ln.group = 3;
  ln.active = true;
  ln.h_diis->done = 0;   // (no kernel of an earlier solve writes it any more)

  const int nst = h->ninst > 1 ? h->ninst + 1 : 1;
  hipLaunchKernelGGL(k_diis_init, dim3(nst), dim3(kWave), 0, ln.stream, h->ninst, tol,
                     ln.diis.p);
  DDX_HIP(hipGetLastError());
  // the L X sweep reads cf x: from here on k_extrap keeps it
  if (!star) DDX_TRY(cf_scale(h, ln.stream, d_x, ln.xs.p));
  return DDX_OK;
}

namespace {
// Whether k_jacobi_two takes a system: one instance, DIIS on, block ranges of
// at most 512 elements whose bounds and history offsets fit 32 bits (up to
// 524 288 elements: 6400 atoms at lmax 8).  Past that a workgroup's threads
// take more than two elements and the launch is bound by its bytes; a batch's
// blocks need their map.
bool jacobi_two_fits(const ddx_handle *h, size_t nn, int diis_max) {
  return h->ninst == 1 && diis_max > 0 && nn <= 2 * (size_t)kJThreads * h->nbj &&
         nn * (h->nbj + 1) < (1ull << 32) && nn * kDiisMax * sizeof(double) < (1ull << 32);
}

// Whether k_extrap_one takes a system: as k_jacobi_two, with every workgroup's
// spheres staged at once.
bool extrap_one_fits(const ddx_handle *h, size_t nn, int diis_max) {
  const int most = (h->n + h->nbe - 1) / h->nbe;   // spheres of a workgroup
  return jacobi_two_fits(h, nn, diis_max) && most <= kWave && most * h->nylm <= kExtrapTerms;
}

// Whether k_diis_extrap takes a system: as k_extrap_one, and a compute unit for
// every workgroup of both solves.  With two workgroups to a unit, each loading
// the state and the dots for itself, there is nothing left to gain: a step of
// 642 atoms takes 1583 us with it and 1588 without, 1000 atoms (lmax 8) 3363
// and 3331.
bool diis_extrap_fits(const ddx_handle *h, size_t nn, int diis_max) {
  return extrap_one_fits(h, nn, diis_max) && 2 * h->nbe <= h->ncu;
}

// `nr` rounds of one solve, or of a direct and an adjoint solve in lockstep
int enqueue_rounds(ddx_handle *h, Lane *const *lanes, int count, int nr) {
  Lane &l0 = *lanes[0];
  const bool pair = count == 2;
  hipStream_t s = l0.stream;
  size_t nn = (size_t)h->nylm * h->n;
  const int nbj = h->nbj, nbe = h->nbe, ninst = h->ninst;
  const double *invl1 = h->cf.p + h->nylm;   // 1/(l+1) table stored after cf
  const int diis_max = l0.diis_max;
  const bool fused = diis_extrap_fits(h, nn, diis_max);
  Systems sys{};
  for (int k = 0; k < count; ++k) sys.s[k] = sys_args(h, *lanes[k]);
  for (int g = 0; g < nr; ++g, ++l0.enqueued) {
    h->tag_round = l0.enqueued;
    // mixed precision: rounds 0, kRefresh, 2 kRefresh, ... apply the FP64
    // operator to the iterate itself; the others the FP32 operator to the
    // last increment, added to the FP64 image
    const bool incr = l0.incr;
    const bool exact = !incr || l0.enqueued % kRefresh == 0;
    const bool next_exact = !incr || (l0.enqueued + 1) % kRefresh == 0;
    for (int k = 0; k < count; ++k) {
      lanes[k]->f32 = !exact;
      sys.s[k].acc = exact ? 0 : 1;
      sys.s[k].xs_inc = next_exact ? 0 : 1;
    }
    const double *xa = pair ? (exact ? lanes[1]->x : lanes[1]->inc.p) : nullptr;
    const double *x1 = exact ? l0.x : l0.inc.p;
    int rc;
    if (pair) {
      rc = apply_pair(h, l0, l0.y.p, *lanes[1], xa, h->ysplit);
    } else if (l0.star) {
      rc = apply_lstarx(h, l0, x1, l0.y.p, solve_gate(h, l0), false);
    } else {
      rc = apply_lx(h, l0, x1, l0.y.p, solve_gate(h, l0), true, h->ysplit);
    }
    for (int k = 0; k < count; ++k) lanes[k]->f32 = false;
    DDX_TRY(rc);
    {
      TimedLaunch tl(h, DDX_K_JACOBI, s);
      // mixed precision keeps the residual history in FP32
      const auto launch = [&](auto two, auto one) {
        if (jacobi_two_fits(h, nn, diis_max))
          hipExtLaunchKernelGGL(two, dim3(nbj + (fused ? 1 : 0), count), dim3(kJThreads), 0, s, tl.b, tl.e, 0,
                                (unsigned)nn, (unsigned)h->nylm, diis_max, (unsigned)nbj,
                                h->facl.p, sys);
        else
          hipExtLaunchKernelGGL(one, dim3(nbj, count), dim3(kJThreads), 0, s, tl.b, tl.e, 0, nn,
                                h->nylm, diis_max, h->jblk.p, nbj, h->facl.p, sys);
      };
      if (l0.incr) launch(k_jacobi_two<float>, k_jacobi<float>);
      else launch(k_jacobi_two<double>, k_jacobi<double>);
    }
    DDX_HIP(hipGetLastError());
    if (fused) {
      TimedLaunch tl(h, DDX_K_DIIS, s);
      const int most = (h->n + nbe - 1) / nbe * h->nylm;   // elements of a workgroup
      const int nt = std::max(kSmallThreads,
                              std::min(kExtrapThreads, kWave + (most + kWave - 1) / kWave * kWave));
      hipExtLaunchKernelGGL(k_diis_extrap, dim3(nbe, count), dim3(nt), 0, s, tl.b, tl.e, 0, (unsigned)h->n, (unsigned)h->nylm, (unsigned)nn,
                            (unsigned)nbe, nbj, diis_max, l0.max_iter, invl1, h->cf.p, sys);
      DDX_HIP(hipGetLastError());
      continue;
    }
    if (diis_max > 0) {
      TimedLaunch tl(h, DDX_K_DIIS, s);
      hipExtLaunchKernelGGL(k_diis_small, dim3(ninst, count), dim3(kSmallThreads), 0, s, tl.b,
                            tl.e, 0, diis_max, nbj, nbe, h->n, h->jboff.p, h->eboff.p, h->soff.p,
                            ninst, l0.max_iter, sys);
      DDX_HIP(hipGetLastError());
    }
    {
      TimedLaunch tl(h, DDX_K_EXTRAP, s);
      if (extrap_one_fits(h, nn, diis_max))
        hipExtLaunchKernelGGL(k_extrap_one, dim3(nbe, count), dim3(kExtrapThreads), 0, s, tl.b, tl.e, 0,
                              (unsigned)h->n, (unsigned)h->nylm, (unsigned)nn, (unsigned)nbe,
                              invl1, h->cf.p, sys);
      else
        hipExtLaunchKernelGGL(k_extrap, dim3(nbe, count), dim3(kJThreads), 0, s, tl.b, tl.e, 0,
                              h->nylm, nn, diis_max, h->eblk.p, invl1, h->cf.p, sys);
    }
    DDX_HIP(hipGetLastError());
    if (diis_max == 0) {
      hipLaunchKernelGGL(k_norm, dim3(ninst, count), dim3(kWave), 0, s, h->eboff.p, h->soff.p,
                         ninst, l0.max_iter, sys);
      DDX_HIP(hipGetLastError());
    }
  }
  return DDX_OK;
}

// what a captured group of rounds depends on: every pointer and setting the
// launches take
std::vector<uintptr_t> round_key(const ddx_handle *h, Lane *const *lanes, int count, int nr) {
  std::vector<uintptr_t> k = {(uintptr_t)count, (uintptr_t)nr, (uintptr_t)h->ysplit,
                              (uintptr_t)h->nbj, (uintptr_t)h->nbe, (uintptr_t)h->nworker};
  for (int c = 0; c < count; ++c) {
    const Lane &l = *lanes[c];
    const uintptr_t v[] = {(uintptr_t)l.star, (uintptr_t)l.incr,
                           (uintptr_t)(l.incr ? lanes[0]->enqueued % kRefresh : 0),
                           (uintptr_t)l.yacc.p, (uintptr_t)l.inc.p, (uintptr_t)l.diis_max,
                           (uintptr_t)l.max_iter,
                           (uintptr_t)l.rhs, (uintptr_t)l.x, (uintptr_t)l.y.p, (uintptr_t)l.xnew.p,
                           (uintptr_t)l.xs.p, (uintptr_t)l.P.p, (uintptr_t)l.xiw.p,
                           (uintptr_t)l.rw.p, (uintptr_t)l.yp.p, (uintptr_t)l.xd.p,
                           (uintptr_t)l.ed.p, (uintptr_t)l.part.p, (uintptr_t)l.diis.p,
                           (uintptr_t)l.misc.p, (uintptr_t)l.stream};
    k.insert(k.end(), std::begin(v), std::end(v));
    uint64_t tb;
    std::memcpy(&tb, &l.tol, 8);
    k.push_back((uintptr_t)tb);
  }
  return k;
}

bool timers_on(const ddx_handle *h) {
  for (const auto &t : h->ktimer)
    if (t.on) return true;
  return false;
}

// the group of nr rounds as a HIP graph: captured on first use with these
// lanes, replayed afterwards (every round's state lives in device memory)
int launch_round_graph(ddx_handle *h, Lane *const *lanes, int count, int nr) {
  Lane &l0 = *lanes[0];
  const std::vector<uintptr_t> key = round_key(h, lanes, count, nr);
  hipGraphExec_t exec = nullptr;
  for (auto &g : h->round_graphs)
    if (g.key == key) exec = g.exec;
  if (!exec) {
    hipGraph_t graph = nullptr;
    const int first = l0.enqueued;
    DDX_HIP(hipStreamBeginCapture(l0.stream, hipStreamCaptureModeRelaxed));
    const int rc = enqueue_rounds(h, lanes, count, nr);
    const hipError_t ec = hipStreamEndCapture(l0.stream, &graph);
    l0.enqueued = first;
    if (rc != DDX_OK) {
      if (graph) (void)hipGraphDestroy(graph);
      return rc;
    }
    DDX_HIP(ec);
    const hipError_t ei = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    DDX_HIP(ei);
    // keyed on the buffers as they stand after the capture
    h->round_graphs.push_back({round_key(h, lanes, count, nr), exec});
  }
  DDX_HIP(hipGraphLaunch(exec, l0.stream));
  l0.enqueued += nr;
  return DDX_OK;
}
}  // namespace

void drop_round_graphs(ddx_handle *h) {
  for (auto &g : h->round_graphs)
    if (g.exec) (void)hipGraphExecDestroy(g.exec);
  h->round_graphs.clear();
}

// Enqueues the next group of rounds, its end marked by h->gev[slot].  The
// first group of a solve (3 rounds) runs eagerly and makes every buffer the
// rounds use; eager groups after it are single rounds.
// With graphs on (and no kernel timer) each later group is one launch of a
// captured graph of kGraphRounds rounds, which covers the rest of a typical
// solve; the rounds after convergence return at once.
int solve_enqueue(ddx_handle *h, Lane *const *lanes, int count, int slot) {
  Lane &l0 = *lanes[0];
  const bool pair = count == 2;
  if (pair && (l0.star != 0 || lanes[1]->star != 1 || lanes[1]->stream != l0.stream ||
               lanes[1]->diis_max != l0.diis_max || lanes[1]->rounds != l0.rounds)) {
    set_error("paired solves need a direct and an adjoint solve with equal settings");
    return DDX_ERR_ARG;
  }
  hipStream_t s = l0.stream;
  h->tag_solve = l0.serial;
  const bool graph = h->use_graphs && l0.enqueued > 0 && !timers_on(h);
  const int nr = std::min(graph ? kGraphRounds : l0.group, l0.rounds - l0.enqueued);
  if (graph)
    DDX_TRY(launch_round_graph(h, lanes, count, nr));
  else
    DDX_TRY(enqueue_rounds(h, lanes, count, nr));
  h->tag_solve = -1;
  h->tag_round = 0;
  l0.group = 1;
  DDX_HIP(hipEventRecord(h->gev[slot], s));
  return DDX_OK;
}

int solve_end(ddx_handle *h, Lane &ln, int *n_iter, int *ok, std::vector<double> *hist) {
  const DiisState *hs = ln.h_diis;
  ln.active = false;
  // a batch: the summary's ok and largest count; per instance in h_res
  *n_iter = hs->ok ? hs->it : ln.max_iter + 1;
  *ok = hs->ok;
  if (hist) {
    if (h->ninst == 1) hist->assign(hs->hist, hs->hist + (hs->it < kMaxIter ? hs->it : kMaxIter));
    else hist->clear();
  }
  return DDX_OK;
}

namespace {
// (an acquire, against the device's fence ahead of its store: the record's
// other values are read after it)
bool lanes_done(Lane *const *lanes, int count) {
  for (int k = 0; k < count; ++k)
    if (!__atomic_load_n(&lanes[k]->h_diis->done, __ATOMIC_ACQUIRE)) return false;
  return true;
}

// Enqueues groups of rounds until the lanes' records say done or all rounds
// have run.  Two groups are in flight: while one runs, the next is already
// queued behind it, so the device does not wait for the host, and the host
// sees the end of a solve within the group that brought it (the one queued
// after it returns at once).  Of the graph groups only the first runs ahead
// (behind the eager first group): a later one would mostly repeat finished
// rounds.
int run_groups(ddx_handle *h, Lane *const *lanes, int count) {
  int head = 0, queued = 0, groups = 0;
  while (!lanes_done(lanes, count)) {
    const bool more = lanes[0]->enqueued < lanes[0]->rounds;
    if (more && (queued == 0 || (queued == 1 && (!h->use_graphs || groups == 1)))) {
      DDX_TRY(solve_enqueue(h, lanes, count, (head + queued) & 1));
      ++queued;
      ++groups;
      continue;
    }
    if (queued == 0) break;
    // poll the record beside the group's event for about a millisecond (the
    // calling thread is busy for that long), then sleep on the event
    hipError_t e = hipErrorNotReady;
    for (int spin = 0; spin < 1000 && e == hipErrorNotReady; ++spin) {
      if (lanes_done(lanes, count)) return DDX_OK;
      e = hipEventQuery(h->gev[head]);
    }
    if (e == hipErrorNotReady) e = hipEventSynchronize(h->gev[head]);
    DDX_HIP(e);
    head ^= 1;
    --queued;
  }
  return DDX_OK;
}
}  // namespace

int solve_run(ddx_handle *h, Lane *const *lanes, int count) {
  const int serial = h->solve_serial++;
  for (int k = 0; k < count; ++k) lanes[k]->serial = serial;
  const int rc = run_groups(h, lanes, count);
  if (rc != DDX_OK) {
    // no kernel of this solve may write its record once another one starts
    (void)hipStreamSynchronize(lanes[0]->stream);
    return rc;
  }
  // a single system's record is complete; a batch's states are copied
  if (h->ninst > 1 || !lanes_done(lanes, count)) {
    for (int k = 0; k < count; ++k) {
      Lane &ln = *lanes[k];
      DDX_HIP(hipMemcpyAsync(ln.h_diis, solve_gate(h, ln), sizeof(DiisState),
                             hipMemcpyDeviceToHost, ln.stream));
      if (h->ninst > 1) {
        hipLaunchKernelGGL(k_diis_results, dim3((h->ninst + 255) / 256), dim3(256), 0, ln.stream,
                           h->ninst, ln.max_iter, ln.diis.p, ln.res.p);
        DDX_HIP(hipGetLastError());
        ln.h_res.resize(2 * (size_t)h->ninst);
        DDX_HIP(hipMemcpyAsync(ln.h_res.data(), ln.res.p, 2 * sizeof(int) * h->ninst,
                               hipMemcpyDeviceToHost, ln.stream));
      }
    }
    DDX_HIP(hipStreamSynchronize(lanes[0]->stream));
  }
  // launches of rounds after a solve's last iteration returned at once:
  // drop them from the timers
  int it[2] = {0, 0}, itmax = 0;
  for (int k = 0; k < count; ++k) {
    it[k] = lanes[k]->h_diis->it;
    if (it[k] > itmax) itmax = it[k];
  }
  const int shared[3] = {DDX_K_JACOBI, DDX_K_DIIS, DDX_K_EXTRAP};
  for (int c : shared) drop_rounds(h, c, serial, itmax);
  if (count == 2) {
    drop_rounds(h, DDX_K_SWEEP_PAIR, serial, itmax);
    drop_rounds(h, DDX_K_PROJECT, serial, it[0]);
    drop_rounds(h, DDX_K_EXPAND, serial, it[1]);
  } else {
    const bool star = lanes[0]->star;
    drop_rounds(h, star ? DDX_K_SWEEP_LSTAR : DDX_K_SWEEP_L, serial, it[0]);
    drop_rounds(h, star ? DDX_K_EXPAND : DDX_K_PROJECT, serial, it[0]);
  }
  return DDX_OK;
}

// Mixed precision: one Jacobi/DIIS iteration whose operator image L x
// (L* x) is carried in FP64 and refreshed exactly.  Round 0 and every
// kRefresh-th round apply the FP64 operator to the iterate; the rounds in
// between apply the FP32 sweeps and products to the last increment
// x_new - x and add the result to the FP64 image.  The Jacobi update, the
// residual rhs - L x, the iterate history and extrapolation, the norms and
// the convergence test are the FP64 path's (jacobi_diis.f90:102-183): the
// FP32 rounding enters only through increments, which shrink with the
// iteration, so the error carried in the image stays near 1e-7 of the
// increments since the last refresh and the iteration counts stay those of
// FP64 to within one or two.  The residual history, which only sets the
// extrapolation coefficients (its Gram matrix, accumulated in FP64, and the
// bordered solve), is stored in FP32: half the bytes of the Gram-row pass.
int solve_run_mixed(ddx_handle *h, Lane *const *lanes, int count) {
  DDX_TRY(make_tables32(h));
  const size_t nn = (size_t)h->nylm * h->n;
  for (int k = 0; k < count; ++k) {
    DDX_TRY(lanes[k]->yacc.reserve(nn + 1));
    DDX_TRY(lanes[k]->inc.reserve(nn + 1));
    lanes[k]->incr = true;
  }
  const int rc = solve_run(h, lanes, count);
  for (int k = 0; k < count; ++k) lanes[k]->incr = false;
  return rc;
}

int solve_lanes(ddx_handle *h, Lane *const *lanes, int count) {
  return h->prec == DDX_PREC_MIXED ? solve_run_mixed(h, lanes, count)
                                   : solve_run(h, lanes, count);
}

int solve_jacobi_diis(ddx_handle *h, Lane &ln, int star, int diis_max, double tol,
                      const double *d_rhs, double *d_x, int max_iter, int *n_iter, int *ok,
                      std::vector<double> *hist) {
  DDX_TRY(solve_begin(h, ln, star, diis_max, tol, d_rhs, d_x, max_iter));
  Lane *lp = &ln;
  DDX_TRY(solve_run(h, &lp, 1));
  return solve_end(h, ln, n_iter, ok, hist);
}

}  // namespace ddx
