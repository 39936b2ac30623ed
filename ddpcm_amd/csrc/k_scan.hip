// Exclusive prefix sums of int arrays, up to four arrays in one launch.
//
// Each workgroup scans a tile of its array and leaves the tile's total; where
// an array has more than one tile, a second launch adds to every tile the sum
// of the totals before it (each workgroup sums them itself: at most a few
// thousand).  One launch for arrays of one tile, two otherwise, whatever the
// number of arrays: a launch costs about 3 us, and the setup of a 60-atom
// system had 18 of them in its scans.
#include "ddx_device.hpp"
#include "ddx_kernels.hpp"

namespace ddx {
namespace {

constexpr int kScanThreads = 1024;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;

// exclusive prefix of v over the workgroup; *total = the sum
__device__ __forceinline__ int block_prefix(int v, int *wsum, int *total) {
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  int incl = v;
  for (int off = 1; off < kWave; off <<= 1) {
    const int t = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += t;
  }
  if (lane == kWave - 1) wsum[wave] = incl;
  __syncthreads();
  // (every wave sums the sixteen totals alike)
  int base = 0, sum = 0;
#pragma unroll
  for (int w = 0; w < kScanThreads / kWave; ++w) {
    const int s = wsum[w];
    if (w < wave) base += s;
    sum += s;
  }
  *total = sum;
  return base + incl - v;
}

__global__ __launch_bounds__(kScanThreads) void k_scan_tile(Scans sc, int nb, int *__restrict__ tot) {
  __shared__ int wsum[kScanThreads / kWave];
  __shared__ int wmax[kScanThreads / kWave];
  const Scan a = sc.s[blockIdx.y];
  const size_t base = (size_t)blockIdx.x * kScanTile;
  if (base >= a.n && !(blockIdx.x == 0)) return;
  const size_t mine = base + (size_t)threadIdx.x * kScanItems;
  int vals[kScanItems], run = 0, big = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) vals[k] = mine + k < a.n ? a.in[mine + k] : 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    big = max(big, vals[k]);
    const int v = min(vals[k], a.cap);
    vals[k] = run;
    run += v;
  }
  int total;
  const int excl = block_prefix(run, wsum, &total);
#pragma unroll
  for (int k = 0; k < kScanItems; ++k)
    if (mine + k < a.n) a.out[mine + k] = excl + vals[k];
  if (a.max) {   // the largest value (capped or not) beside the sum
    big = wave_max_int(big);
    if (lane_id() == 0) wmax[threadIdx.x / kWave] = big;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < kScanThreads / kWave; ++w) big = max(big, wmax[w]);
      tot[(size_t)kMaxScans * nb + blockIdx.x] = big;
    }
  }
  if (threadIdx.x == 0) {
    tot[(size_t)blockIdx.y * nb + blockIdx.x] = total;
    if (a.n <= (size_t)kScanTile) {   // the only tile: the result is complete
      a.out[a.n] = total;
      if (a.rec) *a.rec = total;
      if (a.max) *a.max = big;
    }
  }
}

__global__ __launch_bounds__(kScanThreads) void k_scan_add(Scans sc, int nb,
                                                           const int *__restrict__ tot) {
  __shared__ int wsum[kScanThreads / kWave];
  const Scan a = sc.s[blockIdx.y];
  const size_t base = (size_t)blockIdx.x * kScanTile;
  if (a.n <= (size_t)kScanTile || base >= a.n) return;
  const int *t = tot + (size_t)blockIdx.y * nb;
  int before = 0;
  for (int b = threadIdx.x; b < (int)blockIdx.x; b += kScanThreads) before += t[b];
  int off;
  (void)block_prefix(before, wsum, &off);
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const size_t g = base + (size_t)k * kScanThreads + threadIdx.x;
    if (g < a.n) a.out[g] += off;
  }
  if (base + kScanTile >= a.n && threadIdx.x == 0) {   // the last tile
    const int sum = off + t[blockIdx.x];
    a.out[a.n] = sum;
    if (a.rec) *a.rec = sum;
    if (a.max) {
      int big = 0;
      for (int b = 0; b <= (int)blockIdx.x; ++b) big = max(big, tot[(size_t)kMaxScans * nb + b]);
      *a.max = big;
    }
  }
}

}  // namespace

int scan_arrays(const Scan *scans, int count, DevArray<int> &tmp, hipStream_t s) {
  Scans sc{};
  size_t most = 1;
  for (int k = 0; k < count; ++k) {
    sc.s[k] = scans[k];
    if (scans[k].n > most) most = scans[k].n;
  }
  const size_t nb = (most + kScanTile - 1) / kScanTile;
  DDX_TRY(tmp.reserve((kMaxScans + 1) * nb));
  hipLaunchKernelGGL(k_scan_tile, dim3((unsigned)nb, count), dim3(kScanThreads), 0, s, sc, (int)nb,
                     tmp.p);
  DDX_HIP(hipGetLastError());
  if (nb > 1) {
    hipLaunchKernelGGL(k_scan_add, dim3((unsigned)nb, count), dim3(kScanThreads), 0, s, sc,
                       (int)nb, tmp.p);
    DDX_HIP(hipGetLastError());
  }
  return DDX_OK;
}

int scan_exclusive(const int *in, int *out, size_t n, DevArray<int> &tmp, hipStream_t s) {
  const Scan a{in, out, n, 0x7fffffff, nullptr, nullptr};
  return scan_arrays(&a, 1, tmp, s);
}

}  // namespace ddx
