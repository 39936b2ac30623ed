// C-ABI of libddx: the reference module's procedures on device-resident state.
#include <chrono>
#include <cmath>
#include <cstdarg>
#include <cstring>
#include <vector>

#include "ddx_device.hpp"
#include "ddx_kernels.hpp"
#include "tables.hpp"

namespace ddx {

static thread_local char g_err[512] = "";

void set_error(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

namespace {

template <typename T>
int upload(DevArray<T> &d, const T *src, size_t n, hipStream_t s) {
  DDX_TRY(d.reserve(n));
  if (n) DDX_HIP(hipMemcpyAsync(d.p, src, n * sizeof(T), hipMemcpyHostToDevice, s));
  return DDX_OK;
}

int download(double *dst, const double *src, size_t n, hipStream_t s) {
  if (n) DDX_HIP(hipMemcpyAsync(dst, src, n * sizeof(double), hipMemcpyDeviceToHost, s));
  return DDX_OK;
}

int sync(ddx_handle *h) {
  DDX_HIP(hipStreamSynchronize(h->stream));
  h->stage_busy = false;
  return DDX_OK;
}

// (x, y, z, r) and charges of n spheres from the pinned stage (5 n values:
// x, y, z, r, q) to the device arrays; without q (only the first 4 n) or
// without sph (only the charges)
__global__ void k_unstage(int n, const double *__restrict__ in, double4 *__restrict__ sph,
                          double *__restrict__ q) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (sph) sph[i] = make_double4(in[i], in[n + i], in[2 * n + i], in[3 * n + i]);
  if (q) q[i] = in[4 * (size_t)n + i];
}

// the results of a run into pinned host memory
__global__ void k_export(int ne, const double *__restrict__ e, int nf,
                         const double *__restrict__ f, double *__restrict__ out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < ne) out[k] = e[k];
  else if (k - ne < nf) out[k] = f[k - ne];
}

// A call's inputs travel through pinned memory of the handle, read by one
// kernel on the stream, with no copy call and no wait (a pageable copy of a
// few hundred bytes holds the caller for about 15 us).
int stage_inputs(ddx_handle *h, const double *x, const double *y, const double *z,
                 const double *r, const double *charge) {
  const size_t n = h->n;
  if (h->stage_busy) DDX_TRY(sync(h));
  double *st = h->h_stage;
  if (x) {
    std::memcpy(st, x, n * sizeof(double));
    std::memcpy(st + n, y, n * sizeof(double));
    std::memcpy(st + 2 * n, z, n * sizeof(double));
    std::memcpy(st + 3 * n, r, n * sizeof(double));
    DDX_TRY(h->sph.reserve(n));
  }
  if (charge) {
    std::memcpy(st + 4 * n, charge, n * sizeof(double));
    DDX_TRY(h->charge.reserve(n));
  }
  hipLaunchKernelGGL(k_unstage, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, h->stream,
                     (int)n, h->d_stage, x ? h->sph.p : nullptr, charge ? h->charge.p : nullptr);
  DDX_HIP(hipGetLastError());
  h->stage_busy = true;
  return DDX_OK;
}

// the time of the last setup, once its events have passed
int read_setup_time(ddx_handle *h) {
  if (!h->setup_timed) return DDX_OK;
  DDX_HIP(hipEventSynchronize(h->ev[6]));
  float ms = 0.f;
  DDX_HIP(hipEventElapsedTime(&ms, h->ev[0], h->ev[6]));
  h->stats.ms_setup = ms;
  h->setup_timed = false;
  return DDX_OK;
}

double tol_of(int iconv) {
  double p = 1.0;
  for (int k = 0; k < iconv; ++k) p *= 10.0;
  return 1.0 / p;   // 10^-iconv (cosmo.f90:80)
}

int set_geometry(ddx_handle *h, const double *x, const double *y, const double *z,
                 const double *r, const double *charge) {
  for (int i = 0; i < h->n; ++i) {
    if (!(r[i] > 0.0)) {
      set_error("radius of sphere %d is not positive", i + 1);
      return DDX_ERR_ARG;
    }
    h->rmax = i == 0 || r[i] > h->rmax ? r[i] : h->rmax;
  }
  h->h_x.assign(x, x + h->n);
  h->h_y.assign(y, y + h->n);
  h->h_z.assign(z, z + h->n);
  h->h_r.assign(r, r + h->n);
  return stage_inputs(h, x, y, z, r, charge);
}

// Start of the direct solve L X = g (rhs in h->rhs, X in h->sigma) on a lane,
// from the guess D^-1 rhs (cosmo.f90:136-138).
// The guess of solve `star` for right-hand side v into x: D^-1 v as the
// reference (cosmo.f90:136-138,174-176), or the handle's previous solution,
// or the learned guess (ddx_set_guess).
int initial_guess(ddx_handle *h, int star, const double *v, double *x) {
  const bool prev = star ? h->have_s : h->have_sigma;
  if (h->guess_mode == DDX_GUESS_PREVIOUS && prev) return DDX_OK;
  if (h->guess_mode == DDX_GUESS_LEARNED) return learned_guess(h, star, v, x, false);
  if (h->guess_mode == DDX_GUESS_LEARNED_PREVIOUS) {
    if (!prev) DDX_TRY(device_ldm1x(h, h->stream, v, x));
    return learned_guess(h, star, v, x, prev);
  }
  return device_ldm1x(h, h->stream, v, x);
}

int begin_direct(ddx_handle *h, Lane &ln) {
  DDX_TRY(initial_guess(h, 0, h->rhs.p, h->sigma.p));
  return solve_begin(h, ln, 0, kDiisMax, tol_of(h->iconv), h->rhs.p, h->sigma.p, kMaxIter);
}

// Start of the adjoint solve L* S = psi (S in h->s) from D^-1 psi
// (cosmo.f90:174-176).
int begin_adjoint(ddx_handle *h, Lane &ln, const double *d_psi) {
  DDX_TRY(initial_guess(h, 1, d_psi, h->s.p));
  return solve_begin(h, ln, 1, kDiisMax, tol_of(h->iconv), d_psi, h->s.p, kMaxIter);
}

// per-instance iteration counts of the solve that just ended on a lane
void inst_iterations(const ddx_handle *h, const Lane &ln, int nit, std::vector<int> &out) {
  out.assign(h->ninst, nit);
  if (h->ninst > 1)
    for (int q = 0; q < h->ninst; ++q) out[q] = ln.h_res[2 * q];
}

// a call that only a plain handle takes
int single(const ddx_handle *h, const char *what) {
  if (h->ninst == 1) return DDX_OK;
  set_error("%s takes a handle of one system; this one holds a batch of %d", what, h->ninst);
  return DDX_ERR_STATE;
}

// End of the direct solve; the energies go to energy[0 .. ninst) on the
// handle's stream.
int end_direct(ddx_handle *h, Lane &ln, const double *d_psi, int *ok) {
  int nit = 0;
  DDX_TRY(solve_end(h, ln, &nit, ok, &h->hist_direct));
  h->stats.niter_direct = nit;
  inst_iterations(h, ln, nit, h->iters_direct);
  DDX_TRY(energy_dot(h, h->sigma.p, d_psi, 0.5 * ((h->eps - 1.0) / h->eps), h->energy.p));
  h->have_sigma = true;
  h->conv_sigma = *ok != 0;
  return DDX_OK;
}

int end_adjoint(ddx_handle *h, Lane &ln, int *ok) {
  int nit = 0;
  DDX_TRY(solve_end(h, ln, &nit, ok, &h->hist_adjoint));
  h->stats.niter_adjoint = nit;
  inst_iterations(h, ln, nit, h->iters_adjoint);
  h->have_s = true;
  h->conv_s = *ok != 0;
  return DDX_OK;
}

int noconv(bool star) {
  set_error(star ? "adjoint ddCOSMO did not converge" : "ddCOSMO did not converge");
  return DDX_ERR_NOCONV;
}

// Direct solve on lane 0; X in h->sigma, E in energy[0].
int run_direct(ddx_handle *h, const double *d_psi) {
  Lane *ln = &h->lane[0];
  int ok = 0;
  DDX_TRY(begin_direct(h, *ln));
  DDX_TRY(solve_lanes(h, &ln, 1));
  DDX_TRY(end_direct(h, *ln, d_psi, &ok));
  return ok ? DDX_OK : noconv(false);
}

int run_adjoint(ddx_handle *h, const double *d_psi) {
  Lane *ln = &h->lane[0];
  int ok = 0;
  DDX_TRY(begin_adjoint(h, *ln, d_psi));
  DDX_TRY(solve_lanes(h, &ln, 1));
  DDX_TRY(end_adjoint(h, *ln, &ok));
  return ok ? DDX_OK : noconv(true);
}

int reserve_vectors(ddx_handle *h) {
  size_t nn = (size_t)h->nylm * h->n;
  DDX_TRY(h->rhs.reserve(nn));
  DDX_TRY(h->sigma.reserve(nn));
  DDX_TRY(h->s.reserve(nn));
  DDX_TRY(h->psi.reserve(nn));
  DDX_TRY(h->x.reserve(nn));
  DDX_TRY(h->fx.reserve(3 * (size_t)h->n + 3));
  DDX_TRY(h->energy.reserve(h->ninst + 4));
  return DDX_OK;
}

// The whole E (+F) pipeline on device state: setup must be current and the
// charges uploaded.  main.f90:178-265.
int pipeline(ddx_handle *h) {
  hipStream_t s = h->stream;
  h->results_ok = false;
  DDX_TRY(reserve_vectors(h));
  DDX_TRY(h->phi.reserve((size_t)h->ncav + 1));
  DDX_TRY(h->zeta.reserve((size_t)h->ncav + 1));
  if (h->igrad) DDX_TRY(h->ef.reserve(field_buffer_size(h)));
  DDX_HIP(hipEventRecord(h->ev[1], s));
  // potential at the cavity points, with forces also the solute field there
  if (use_fmm(h))
    DDX_TRY(fmm_potential(h, h->charge.p, h->phi.p, h->igrad ? h->ef.p : nullptr));
  else
    DDX_TRY(coulomb_potential(h, h->ctile, h->charge.p, h->sph.p, h->ccav.p,
                              h->phi.p, h->igrad ? h->ef.p : nullptr));
  DDX_TRY(make_psi(h, h->charge.p, h->psi.p));
  DDX_TRY(build_rhs(h, h->phi.p, h->rhs.p));
  DDX_HIP(hipEventRecord(h->ev[2], s));
  int ok_d = 0, ok_a = 1;
  if (h->igrad) {
    // the direct and the adjoint solve in lockstep: neither depends on the
    // other (cosmo.f90:136-196), and each sweep builds the basis for both
    Lane *lanes[2] = {&h->lane[0], &h->lane[1]};
    DDX_TRY(begin_direct(h, h->lane[0]));
    DDX_TRY(begin_adjoint(h, h->lane[1], h->psi.p));
    DDX_TRY(solve_lanes(h, lanes, 2));
    DDX_TRY(end_direct(h, h->lane[0], h->psi.p, &ok_d));
    DDX_TRY(end_adjoint(h, h->lane[1], &ok_a));
  } else {
    Lane *ln = &h->lane[0];
    DDX_TRY(begin_direct(h, *ln));
    DDX_TRY(solve_lanes(h, &ln, 1));
    DDX_TRY(end_direct(h, *ln, h->psi.p, &ok_d));
  }
  DDX_HIP(hipEventRecord(h->ev[3], s));
  // a plain handle stops at a solve that did not converge (the reference
  // stops, cosmo.f90:154,192); a batch completes the others and reports it
  if (h->ninst == 1 && !ok_d) {
    DDX_TRY(sync(h));
    return noconv(false);
  }
  if (h->ninst == 1 && !ok_a) {
    DDX_TRY(sync(h));
    return noconv(true);
  }
  if (h->igrad) {
    // xi = basis^T S serves both branches that follow: zeta and its field
    // at the nuclei (compute-bound all-pairs sums) on the second stream,
    // beside the force kernels (memory-bound) on the first; joined before
    // the contractions add into fx
    DDX_TRY(h->xi.reserve(h->np));
    DDX_TRY(expand(h, s, h->s.p, h->xi.p, false, nullptr));
    DDX_HIP(hipEventRecord(h->fev[0], s));
    DDX_HIP(hipStreamWaitEvent(h->stream2, h->fev[0], 0));
    h->stream = h->stream2;
    int rc = make_zeta(h, h->s.p, h->zeta.p, true);
    if (rc == DDX_OK) rc = field_forces_fields(h, h->charge.p, h->zeta.p, true);
    h->stream = s;
    DDX_TRY(rc);
    DDX_HIP(hipEventRecord(h->fev[1], h->stream2));
    DDX_TRY(forces_dd(h, h->phi.p, h->sigma.p, h->s.p, h->fx.p, true));
    DDX_HIP(hipStreamWaitEvent(s, h->fev[1], 0));
    DDX_TRY(field_forces_contract(h, h->charge.p, h->zeta.p, h->fx.p));
    DDX_HIP(hipEventRecord(h->ev[5], s));
  }
  const int nf = h->igrad ? 3 * h->n : 0;
  hipLaunchKernelGGL(k_export, dim3((unsigned)((h->ninst + nf + 255) / 256)), dim3(256), 0, s,
                     h->ninst, h->energy.p, nf, h->fx.p, h->d_out);
  DDX_HIP(hipGetLastError());
  DDX_TRY(sync(h));
  h->results_ok = true;
  DDX_TRY(read_setup_time(h));
  // with forces the two solves run together: ms_direct covers both and
  // ms_adjoint is zero
  float ms = 0.f;
  DDX_HIP(hipEventElapsedTime(&ms, h->ev[1], h->ev[2]));
  h->stats.ms_rhs = ms;
  DDX_HIP(hipEventElapsedTime(&ms, h->ev[2], h->ev[3]));
  h->stats.ms_direct = ms;
  h->stats.ms_adjoint = 0.0;
  if (h->igrad) {
    DDX_HIP(hipEventElapsedTime(&ms, h->ev[3], h->ev[5]));
    h->stats.ms_forces = ms;
  }
  if (!ok_d || !ok_a) {
    int first = -1;
    const std::vector<int> &it = !ok_d ? h->iters_direct : h->iters_adjoint;
    for (int q = 0; q < h->ninst && first < 0; ++q)
      if (it[q] > kMaxIter) first = q;
    set_error("%s ddCOSMO did not converge for instance %d of the batch",
              !ok_d ? "direct" : "adjoint", first);
    return DDX_ERR_NOCONV;
  }
  return DDX_OK;
}

// (its time is read once the events have passed: here nothing waits)
int timed_setup(ddx_handle *h) {
  h->setup_timed = false;
  DDX_HIP(hipEventRecord(h->ev[0], h->stream));
  DDX_TRY(run_setup(h));
  DDX_HIP(hipEventRecord(h->ev[6], h->stream));
  h->stage_busy = false;   // run_setup has waited for its counts, past the inputs
  h->setup_timed = true;
  return DDX_OK;
}

}  // namespace
}  // namespace ddx

using namespace ddx;

extern "C" {

const char *ddx_last_error(void) { return g_err; }

}  // extern "C"

namespace ddx {
namespace {
// A handle of `count` instances with nsph[q] spheres each (count = 1, nsph
// = null: a plain handle of n spheres).
int create(ddx_handle **out, int n, int count, const int *nsph, const double *x,
           const double *y, const double *z, const double *rvdw, int iprint, int lmax,
           int ngrid, int iconv, int igrad, double eps, double eta) {
  if (!out || n < 1 || count < 1 || !x || !y || !z || !rvdw) {
    set_error("ddx_init: invalid arguments");
    return DDX_ERR_ARG;
  }
  if (lmax < 0 || lmax > kMaxLmax) {
    set_error("lmax %d not supported (0..%d)", lmax, kMaxLmax);
    return DDX_ERR_ARG;
  }
  if (!(eta > 0.0 && eta <= 1.0) || !(eps > 0.0) || iconv < 0 || iconv > 15) {
    set_error("ddx_init: eps, eta or iconv out of range");
    return DDX_ERR_ARG;
  }
  ddx_handle *h = new ddx_handle();
  h->n = n;
  h->ninst = count;
  h->h_soff.assign(1, 0);
  for (int q = 0; q < count; ++q) h->h_soff.push_back(h->h_soff.back() + (nsph ? nsph[q] : n));
  h->lmax = lmax;
  h->nylm = (lmax + 1) * (lmax + 1);
  h->ngrid = snap_ngrid(ngrid);
  h->iconv = iconv;
  h->igrad = igrad != 0;
  h->iprint = iprint;
  h->eps = eps;
  h->eta = eta;
  int rc = DDX_OK;
  auto fail = [&](int code) {
    ddx_free(h);
    return code;
  };
  if (hipStreamCreate(&h->stream) != hipSuccess || hipStreamCreate(&h->stream2) != hipSuccess) {
    set_error("hipStreamCreate failed");
    return fail(DDX_ERR_HIP);
  }
  for (auto &e : h->fev)
    if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
      set_error("hipEventCreate failed");
      return fail(DDX_ERR_HIP);
    }
  for (Lane &ln : h->lane) ln.stream = h->stream;
  {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&h->ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        h->ncu < 1) {
      set_error("cannot query the compute units of the device");
      return fail(DDX_ERR_HIP);
    }
  }
  // the scratch address of ddx_efld_noalloc on this device, looked up here
  // so that a later call under graph capture finds it ready
  if ((rc = noalloc_setup(nullptr)) != DDX_OK) return fail(rc);
  for (auto &e : h->ev)
    if (hipEventCreate(&e) != hipSuccess) {
      set_error("hipEventCreate failed");
      return fail(DDX_ERR_HIP);
    }
  // one pinned allocation (each is a call of tens of microseconds): the
  // lanes' records, the setup's counts, a call's inputs, the results
  {
    const size_t rec = (sizeof(DiisState) + 63) / 64 * 64, cnt = 64;
    static_assert(kSetupCounts * sizeof(int) <= 64, "the counts fit their line");
    const size_t in = 5 * (size_t)n * sizeof(double);
    const size_t res = (3 * (size_t)n + count) * sizeof(double);
    char *hp = nullptr, *dp = nullptr;
    // (coherent: the host polls the lanes' records while kernels run; mapped
    // and portable as by default)
    const unsigned kind = hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent;
    if (hipHostMalloc((void **)&hp, 2 * rec + cnt + in + res, kind) != hipSuccess) {
      set_error("hipHostMalloc failed");
      return fail(DDX_ERR_ALLOC);
    }
    h->h_pinned = hp;
    if (hipHostGetDevicePointer((void **)&dp, hp, 0) != hipSuccess) {
      set_error("hipHostGetDevicePointer failed");
      return fail(DDX_ERR_HIP);
    }
    for (int k = 0; k < 2; ++k) {
      h->lane[k].h_diis = (DiisState *)(hp + k * rec);
      h->lane[k].d_rec = (DiisState *)(dp + k * rec);
    }
    h->h_counts = (int *)(hp + 2 * rec);
    h->d_counts = (int *)(dp + 2 * rec);
    h->h_stage = (double *)(hp + 2 * rec + cnt);
    h->d_stage = (double *)(dp + 2 * rec + cnt);
    h->h_out = (double *)(hp + 2 * rec + cnt + in);
    h->d_out = (double *)(dp + 2 * rec + cnt + in);
  }
  for (auto &e : h->gev)
    if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
      set_error("hipEventCreate failed");
      return fail(DDX_ERR_HIP);
    }
  // one-time tables (ddcosmo.f90:225-267)
  if (lebedev_grid(h->ngrid, h->h_grid, h->h_w) != 0) {
    set_error("no Lebedev grid of %d points", h->ngrid);
    return fail(DDX_ERR_ARG);
  }
  harmonic_factors(lmax, h->h_facl, h->h_facs);
  int nylm = h->nylm, ng = h->ngrid;
  h->h_basis.assign((size_t)nylm * ng, 0.0);
  for (int i = 0; i < ng; ++i)
    real_harmonics(lmax, h->h_facs.data(), &h->h_grid[3 * i], &h->h_basis[(size_t)nylm * i]);
  std::vector<double> yw((size_t)nylm * ng);
  for (int i = 0; i < ng; ++i)
    for (int k = 0; k < nylm; ++k) yw[(size_t)nylm * i + k] = h->h_basis[(size_t)nylm * i + k] * h->h_w[i];
  std::vector<double4> g4(ng);
  for (int i = 0; i < ng; ++i)
    g4[i] = make_double4(h->h_grid[3 * i], h->h_grid[3 * i + 1], h->h_grid[3 * i + 2], h->h_w[i]);
  // cf = facs / facl, then 1/(l+1) (hsnorm), 1/facl = 4pi/(2l+1) (intmlp),
  // the scales K of the FP32 sweep's basis and cf K
  std::vector<double> cf(5 * (size_t)nylm);
  for (int l = 0; l <= lmax; ++l)
    for (int m = -l; m <= l; ++m) {
      int k = l * l + l + m;
      cf[k] = h->h_facs[k] / h->h_facl[k];
      cf[nylm + k] = 1.0 / (1.0 + (double)l);
      cf[2 * nylm + k] = 1.0 / h->h_facl[k];
      cf[3 * nylm + k] = ddx::sweep_basis_scale(l, m < 0 ? -m : m);
      cf[4 * nylm + k] = cf[k] * cf[3 * nylm + k];
    }
  hipStream_t s = h->stream;
  if ((rc = upload(h->grid, g4.data(), ng, s)) ||
      (rc = upload(h->Y, h->h_basis.data(), h->h_basis.size(), s)) ||
      (rc = upload(h->Yw, yw.data(), yw.size(), s)) ||
      (rc = upload(h->facl, h->h_facl.data(), nylm, s)) ||
      (rc = upload(h->facs, h->h_facs.data(), nylm, s)) ||
      (rc = upload(h->cf, cf.data(), cf.size(), s)) || (rc = make_ptables(h)) ||
      (rc = sync(h)))
    return fail(rc);
  if (count > 1) {
    std::vector<int> inst(n);
    for (int q = 0; q < count; ++q)
      for (int i = h->h_soff[q]; i < h->h_soff[q + 1]; ++i) inst[i] = q;
    if ((rc = h->inst.reserve(n)) ||
        (rc = hipMemcpy(h->inst.p, inst.data(), n * sizeof(int), hipMemcpyHostToDevice) ==
                      hipSuccess ? DDX_OK : DDX_ERR_HIP))
      return fail(rc);
  }
  if ((rc = set_geometry(h, x, y, z, rvdw, nullptr)) || (rc = timed_setup(h)) ||
      (rc = sync(h)) || (rc = read_setup_time(h)))
    return fail(rc);
  *out = h;
  return DDX_OK;
}
}  // namespace
}  // namespace ddx

extern "C" {

int ddx_init(ddx_handle **out, int n, const double *x, const double *y, const double *z,
             const double *rvdw, int iprint, int lmax, int ngrid, int iconv, int igrad,
             double eps, double eta) {
  return create(out, n, 1, nullptr, x, y, z, rvdw, iprint, lmax, ngrid, iconv, igrad, eps, eta);
}

int ddx_batch_init(ddx_handle **out, int count, const int *nsph, const double *x,
                   const double *y, const double *z, const double *rvdw, int lmax, int ngrid,
                   int iconv, int igrad, double eps, double eta) {
  if (!nsph || count < 1) {
    set_error("ddx_batch_init: invalid arguments");
    return DDX_ERR_ARG;
  }
  long long n = 0;
  for (int q = 0; q < count; ++q) {
    if (nsph[q] < 1) {
      set_error("ddx_batch_init: instance %d has no spheres", q);
      return DDX_ERR_ARG;
    }
    n += nsph[q];
  }
  if (n > 0x7fffffffll) {
    set_error("ddx_batch_init: too many spheres");
    return DDX_ERR_ARG;
  }
  return create(out, (int)n, count, nsph, x, y, z, rvdw, 0, lmax, ngrid, iconv, igrad, eps, eta);
}

int ddx_free(ddx_handle *h) {
  if (!h) return DDX_OK;
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  if (h->h_pinned) (void)hipHostFree(h->h_pinned);
  for (auto &e : h->gev)
    if (e) (void)hipEventDestroy(e);
  drop_round_graphs(h);
  for (auto &t : h->ktimer) {
    for (auto &r : t.recs) {
      (void)hipEventDestroy(r.b);
      (void)hipEventDestroy(r.e);
    }
    for (auto e : t.pool) (void)hipEventDestroy(e);
  }
  for (auto &e : h->ev)
    if (e) (void)hipEventDestroy(e);
  for (auto &e : h->fev)
    if (e) (void)hipEventDestroy(e);
  hipStream_t s = h->stream, s2 = h->stream2;
  delete h;   // device arrays release themselves
  if (s) (void)hipStreamDestroy(s);
  if (s2) (void)hipStreamDestroy(s2);
  return DDX_OK;
}

int ddx_get_sizes(const ddx_handle *h, int *nsph, int *ncav, int *nylm, int *ngrid, int *lmax) {
  if (!h) return DDX_ERR_ARG;
  if (nsph) *nsph = h->n;
  if (ncav) *ncav = h->ncav;
  if (nylm) *nylm = h->nylm;
  if (ngrid) *ngrid = h->ngrid;
  if (lmax) *lmax = h->lmax;
  return DDX_OK;
}

int ddx_get_array(const ddx_handle *hc, const char *name, double *dst) {
  ddx_handle *h = const_cast<ddx_handle *>(hc);
  if (!h || !name || !dst) return DDX_ERR_ARG;
  size_t np = h->np;
  auto cp = [&](const std::vector<double> &v) {
    std::memcpy(dst, v.data(), v.size() * sizeof(double));
    return DDX_OK;
  };
  if (!strcmp(name, "grid")) return cp(h->h_grid);
  if (!strcmp(name, "w")) return cp(h->h_w);
  if (!strcmp(name, "basis")) return cp(h->h_basis);
  if (!strcmp(name, "facl")) return cp(h->h_facl);
  if (!strcmp(name, "facs")) return cp(h->h_facs);
  if (!strcmp(name, "rsph")) return cp(h->h_r);
  if (!strcmp(name, "csph")) {
    for (int i = 0; i < h->n; ++i) {
      dst[3 * i] = h->h_x[i];
      dst[3 * i + 1] = h->h_y[i];
      dst[3 * i + 2] = h->h_z[i];
    }
    return DDX_OK;
  }
  const double *src = nullptr;
  size_t cnt = 0;
  if (!strcmp(name, "fi") || !strcmp(name, "ui") || !strcmp(name, "zi") || !strcmp(name, "ccav"))
    DDX_TRY(lists_ready(h, "ddx_get_array"));
  if (!strcmp(name, "fi")) { src = h->fi.p; cnt = np; }
  else if (!strcmp(name, "ui")) { src = h->ui.p; cnt = np; }
  else if (!strcmp(name, "zi")) {
    if (!h->igrad) { set_error("zi exists only with igrad = 1"); return DDX_ERR_STATE; }
    src = h->zi.p; cnt = 3 * np;
  } else if (!strcmp(name, "ccav")) { src = h->ccav.p; cnt = 3 * (size_t)h->ncav; }
  else if (!strcmp(name, "rhs") || !strcmp(name, "xi") || !strcmp(name, "sigma") ||
           !strcmp(name, "s")) {
    // the last RHS a direct solve used (cosmo.f90:102-128), the last
    // xi = basis^T S of the forces (forces_dd.f90:108-114), the last
    // solutions sigma (direct) and S (adjoint)
    const bool xi = !strcmp(name, "xi");
    src = xi ? h->xi.p : name[0] == 'r' ? h->rhs.p : name[1] == 'i' ? h->sigma.p : h->s.p;
    if (!strcmp(name, "sigma") && !h->have_sigma) src = nullptr;
    if (!strcmp(name, "s") && !h->have_s) src = nullptr;
    cnt = xi ? np : (size_t)h->nylm * h->n;
    if (!src) {
      set_error("'%s' is not available yet", name);
      return DDX_ERR_STATE;
    }
  } else {
    set_error("unknown array '%s'", name);
    return DDX_ERR_ARG;
  }
  DDX_TRY(download(dst, src, cnt, h->stream));
  return sync(h);
}

int ddx_get_neighbours(const ddx_handle *hc, int *inl, int *nl) {
  ddx_handle *h = const_cast<ddx_handle *>(hc);
  if (!h || !inl || !nl) return DDX_ERR_ARG;
  DDX_TRY(lists_ready(h, "ddx_get_neighbours"));
  DDX_HIP(hipMemcpyAsync(inl, h->inl.p, (h->n + 1) * sizeof(int), hipMemcpyDeviceToHost, h->stream));
  if (h->nnl)
    DDX_HIP(hipMemcpyAsync(nl, h->nl.p, h->nnl * sizeof(int), hipMemcpyDeviceToHost, h->stream));
  DDX_TRY(sync(h));
  for (int i = 0; i <= h->n; ++i) inl[i] += 1;
  for (int k = 0; k < h->nnl; ++k) nl[k] += 1;
  return DDX_OK;
}

int ddx_mkrhs(ddx_handle *h, const double *charge, double *phi, double *psi) {
  if (!h || !charge || !phi || !psi) return DDX_ERR_ARG;
  DDX_TRY(lists_ready(h, "ddx_mkrhs"));
  DDX_TRY(reserve_vectors(h));
  DDX_TRY(stage_inputs(h, nullptr, nullptr, nullptr, nullptr, charge));
  DDX_TRY(h->phi.reserve((size_t)h->ncav + 1));
  if (use_fmm(h))
    DDX_TRY(fmm_potential(h, h->charge.p, h->phi.p, nullptr));
  else
    DDX_TRY(coulomb_potential(h, h->ctile, h->charge.p, h->sph.p, h->ccav.p,
                              h->phi.p, nullptr));
  DDX_TRY(make_psi(h, h->charge.p, h->psi.p));
  DDX_TRY(download(phi, h->phi.p, h->ncav, h->stream));
  DDX_TRY(download(psi, h->psi.p, (size_t)h->nylm * h->n, h->stream));
  h->have_charge = true;
  return sync(h);
}

int ddx_mkrhs_at(ddx_handle *h, int n, const double *charge, const double *x, const double *y,
                 const double *z, int ncav, const double *ccav, double *phi, int nylm,
                 double *psi) {
  if (!h || n < 1 || ncav < 0 || nylm < 1 || !charge || !x || !y || !z ||
      (ncav && (!ccav || !phi)) || !psi) {
    set_error("ddx_mkrhs_at: invalid arguments");
    return DDX_ERR_ARG;
  }
  hipStream_t s = h->stream;
  std::vector<double4> src(n);
  for (int i = 0; i < n; ++i) src[i] = make_double4(x[i], y[i], z[i], 0.0);
  DevArray<double4> dsrc;
  DevArray<double> dq, dtrg, dphi, dpsi;
  TileTable dtile;
  DDX_TRY(potential_tiles(h, dtile, n, ncav));
  DDX_TRY(upload(dsrc, src.data(), n, s));
  DDX_TRY(upload(dq, charge, n, s));
  DDX_TRY(upload(dtrg, ccav, 3 * (size_t)ncav, s));
  DDX_TRY(dphi.reserve((size_t)ncav + 1));
  DDX_TRY(dpsi.reserve((size_t)nylm * n));
  DDX_TRY(coulomb_potential(h, dtile, dq.p, dsrc.p, dtrg.p, dphi.p, nullptr));
  DDX_TRY(make_psi_n(h, n, nylm, dq.p, dpsi.p));
  DDX_TRY(download(phi, dphi.p, ncav, s));
  DDX_TRY(download(psi, dpsi.p, (size_t)nylm * n, s));
  return sync(h);
}

int ddx_cosmo(ddx_handle *h, int star, int cart, const double *phi, const double *glm,
              const double *psi, double *sigma, double *esolv) {
  if (!h || !psi || !sigma) return DDX_ERR_ARG;
  DDX_TRY(single(h, "ddx_cosmo"));
  DDX_TRY(lists_ready(h, "ddx_cosmo"));
  h->results_ok = false;
  hipStream_t s = h->stream;
  size_t nn = (size_t)h->nylm * h->n;
  DDX_TRY(reserve_vectors(h));
  DDX_TRY(upload(h->psi, psi, nn, s));
  int rc;
  if (!star) {
    if (cart) {
      if (!phi) return DDX_ERR_ARG;
      DDX_TRY(upload(h->phi, phi, (size_t)h->ncav, s));
      DDX_TRY(build_rhs(h, h->phi.p, h->rhs.p));
    } else {
      if (!glm) return DDX_ERR_ARG;
      DDX_TRY(upload(h->rhs, glm, nn, s));
    }
    rc = run_direct(h, h->psi.p);
    if (rc != DDX_OK && rc != DDX_ERR_NOCONV) return rc;
    DDX_TRY(download(sigma, h->sigma.p, nn, s));
    if (esolv) DDX_TRY(download(esolv, h->energy.p, 1, s));
  } else {
    rc = run_adjoint(h, h->psi.p);
    if (rc != DDX_OK && rc != DDX_ERR_NOCONV) return rc;
    DDX_TRY(download(sigma, h->s.p, nn, s));
  }
  DDX_TRY(sync(h));
  return rc;
}

int ddx_forces_dd(ddx_handle *h, const double *phi, const double *sigma, const double *s_adj,
                  double *fx) {
  if (!h || !phi || !sigma || !s_adj || !fx) return DDX_ERR_ARG;
  DDX_TRY(lists_ready(h, "ddx_forces_dd"));
  h->results_ok = false;
  hipStream_t s = h->stream;
  size_t nn = (size_t)h->nylm * h->n;
  DDX_TRY(reserve_vectors(h));
  DDX_TRY(upload(h->phi, phi, (size_t)h->ncav, s));
  DDX_TRY(upload(h->sigma, sigma, nn, s));
  DDX_TRY(upload(h->s, s_adj, nn, s));
  DDX_TRY(forces_dd(h, h->phi.p, h->sigma.p, h->s.p, h->fx.p));
  DDX_TRY(download(fx, h->fx.p, 3 * (size_t)h->n, s));
  return sync(h);
}

int ddx_mkzeta(ddx_handle *h, const double *s_adj, double *zeta) {
  if (!h || !s_adj || !zeta) return DDX_ERR_ARG;
  DDX_TRY(lists_ready(h, "ddx_mkzeta"));
  hipStream_t s = h->stream;
  DDX_TRY(reserve_vectors(h));
  DDX_TRY(upload(h->s, s_adj, (size_t)h->nylm * h->n, s));
  DDX_TRY(h->zeta.reserve((size_t)h->ncav + 1));
  DDX_TRY(make_zeta(h, h->s.p, h->zeta.p));
  DDX_TRY(download(zeta, h->zeta.p, h->ncav, s));
  return sync(h);
}

int ddx_efld(ddx_handle *h, int nsrc, const double *src, const double *csrc, int ntrg,
             const double *ctrg, double *ef) {
  if (!h || nsrc < 0 || ntrg < 0 || (nsrc && (!src || !csrc)) || (ntrg && (!ctrg || !ef)))
    return DDX_ERR_ARG;
  hipStream_t s = h->stream;
  DevArray<double> dq, dsrc, dtrg, def;
  DDX_TRY(upload(dq, src, nsrc, s));
  DDX_TRY(upload(dsrc, csrc, 3 * (size_t)nsrc, s));
  DDX_TRY(upload(dtrg, ctrg, 3 * (size_t)ntrg, s));
  DDX_TRY(def.reserve(3 * (size_t)ntrg + 3));
  DDX_TRY(coulomb_field_points(h, nsrc, dq.p, dsrc.p, ntrg, dtrg.p, def.p));
  DDX_TRY(download(ef, def.p, 3 * (size_t)ntrg, s));
  return sync(h);
}

static int op_apply(ddx_handle *h, int which, const double *x, double *y) {
  if (!h || !x || !y) return DDX_ERR_ARG;
  if (which < 2) DDX_TRY(lists_ready(h, which ? "ddx_lstarx" : "ddx_lx"));
  hipStream_t s = h->stream;
  size_t nn = (size_t)h->nylm * h->n;
  DDX_TRY(reserve_vectors(h));
  DDX_TRY(h->y.reserve(nn));
  DDX_TRY(upload(h->x, x, nn, s));
  // in the handle's precision: the FP32 operators under mixed precision
  Lane &l0 = h->lane[0];
  if (which < 2 && h->prec == DDX_PREC_MIXED) {
    DDX_TRY(make_tables32(h));
    l0.f32 = true;
  }
  int rc = DDX_OK;
  if (which == 0) rc = apply_lx(h, l0, h->x.p, h->y.p, nullptr, false, 1);
  else if (which == 1) rc = apply_lstarx(h, l0, h->x.p, h->y.p, nullptr, true);
  else rc = device_ldm1x(h, s, h->x.p, h->y.p);
  l0.f32 = false;
  DDX_TRY(rc);
  DDX_TRY(download(y, h->y.p, nn, s));
  return sync(h);
}

int ddx_lx(ddx_handle *h, const double *x, double *y) { return op_apply(h, 0, x, y); }
int ddx_lstarx(ddx_handle *h, const double *x, double *y) { return op_apply(h, 1, x, y); }
int ddx_ldm1x(ddx_handle *h, const double *x, double *y) { return op_apply(h, 2, x, y); }

int ddx_hnorm(ddx_handle *h, const double *x, double *norm) {
  if (!h || !x || !norm) return DDX_ERR_ARG;
  size_t nn = (size_t)h->nylm * h->n;
  DDX_TRY(reserve_vectors(h));
  DDX_TRY(upload(h->x, x, nn, h->stream));
  return device_hnorm(h, h->x.p, norm);
}

int ddx_jacobi_diis(ddx_handle *h, int star, int diis_max, double tol, const double *rhs,
                    double *x, int *n_iter, int *ok) {
  if (!h || !rhs || !x || !n_iter || !ok) return DDX_ERR_ARG;
  DDX_TRY(single(h, "ddx_jacobi_diis"));
  DDX_TRY(lists_ready(h, "ddx_jacobi_diis"));
  hipStream_t s = h->stream;
  size_t nn = (size_t)h->nylm * h->n;
  DDX_TRY(reserve_vectors(h));
  DDX_TRY(upload(h->rhs, rhs, nn, s));
  DDX_TRY(upload(h->x, x, nn, s));
  DDX_TRY(solve_jacobi_diis(h, h->lane[0], star ? 1 : 0, diis_max, tol, h->rhs.p, h->x.p, *n_iter,
                            n_iter, ok, star ? &h->hist_adjoint : &h->hist_direct));
  DDX_TRY(download(x, h->x.p, nn, s));
  return sync(h);
}

int ddx_get_history(const ddx_handle *h, int star, int cap, double *norms, int *count) {
  if (!h || !count) return DDX_ERR_ARG;
  if (star < 0 || star > 2) return DDX_ERR_ARG;
  const std::vector<double> &v =
      star == 2 ? h->hist_ops : star ? h->hist_adjoint : h->hist_direct;
  int c = (int)v.size();
  *count = c;
  if (norms)
    for (int k = 0; k < c && k < cap; ++k) norms[k] = v[k];
  return DDX_OK;
}

int ddx_upload(ddx_handle *h, const double *x, const double *y, const double *z,
               const double *rvdw, const double *charge) {
  if (!h || !x || !y || !z || !rvdw || !charge) return DDX_ERR_ARG;
  DDX_TRY(set_geometry(h, x, y, z, rvdw, charge));
  h->have_charge = true;
  h->have_setup = false;
  return DDX_OK;
}

int ddx_run(ddx_handle *h) {
  if (!h) return DDX_ERR_ARG;
  if (!h->have_charge) {
    set_error("ddx_run needs ddx_upload first");
    return DDX_ERR_STATE;
  }
  DDX_TRY(timed_setup(h));
  return pipeline(h);
}

int ddx_result(ddx_handle *h, double *esolv, double *fx) {
  if (!h) return DDX_ERR_ARG;
  DDX_TRY(single(h, "ddx_result"));
  return ddx_batch_result(h, esolv, fx);
}

int ddx_batch_result(ddx_handle *h, double *esolv, double *fx) {
  if (!h) return DDX_ERR_ARG;
  if (h->results_ok) {   // the last pipeline left them in pinned memory
    if (esolv) std::memcpy(esolv, h->h_out, h->ninst * sizeof(double));
    if (fx && h->igrad) std::memcpy(fx, h->h_out + h->ninst, 3 * (size_t)h->n * sizeof(double));
    return DDX_OK;
  }
  if (esolv) DDX_TRY(download(esolv, h->energy.p, h->ninst, h->stream));
  if (fx && h->igrad) DDX_TRY(download(fx, h->fx.p, 3 * (size_t)h->n, h->stream));
  return sync(h);
}

int ddx_energy_forces(ddx_handle *h, const double *charge, double *esolv, double *fx) {
  if (!h || !charge || !esolv) return DDX_ERR_ARG;
  DDX_TRY(single(h, "ddx_energy_forces"));
  return ddx_batch_energy_forces(h, charge, esolv, fx);
}

int ddx_batch_energy_forces(ddx_handle *h, const double *charge, double *esolv, double *fx) {
  if (!h || !charge || !esolv) return DDX_ERR_ARG;
  DDX_TRY(stage_inputs(h, nullptr, nullptr, nullptr, nullptr, charge));
  h->have_charge = true;
  if (!h->have_setup) DDX_TRY(timed_setup(h));
  const int rc = pipeline(h);
  if (rc != DDX_OK && !(rc == DDX_ERR_NOCONV && h->ninst > 1)) return rc;
  DDX_TRY(ddx_batch_result(h, esolv, fx));
  return rc;
}

int ddx_batch_iterations(const ddx_handle *h, int *direct, int *adjoint) {
  if (!h) return DDX_ERR_ARG;
  for (int q = 0; q < h->ninst; ++q) {
    if (direct) direct[q] = q < (int)h->iters_direct.size() ? h->iters_direct[q] : 0;
    if (adjoint) adjoint[q] = q < (int)h->iters_adjoint.size() ? h->iters_adjoint[q] : 0;
  }
  return DDX_OK;
}

int ddx_batch_sizes(const ddx_handle *h, int *count, int *sph_off, int *cav_off) {
  if (!h) return DDX_ERR_ARG;
  if (count) *count = h->ninst;
  for (int q = 0; q <= h->ninst; ++q) {
    if (sph_off) sph_off[q] = h->h_soff[q];
    if (cav_off) cav_off[q] = q < (int)h->h_cavoff.size() ? h->h_cavoff[q] : 0;
  }
  return DDX_OK;
}

int ddx_set_precision(ddx_handle *h, int prec) {
  if (!h || (prec != DDX_PREC_FP64 && prec != DDX_PREC_MIXED)) return DDX_ERR_ARG;
  DDX_TRY(sync(h));
  h->prec = prec;
  return DDX_OK;
}

// The launch shapes of the solver, picked by timing the whole pipeline on
// the uploaded system: sweep workers per compute unit (4 .. 64), then the
// point split of the L X projection (1, 2, 4).  Each candidate runs twice,
// the second run timed; the last run uses the choice.
int ddx_autotune(ddx_handle *h, int *workers_per_cu, int *proj_split) {
  if (!h) return DDX_ERR_ARG;
  if (!h->have_charge) {
    set_error("ddx_autotune needs ddx_upload first");
    return DDX_ERR_STATE;
  }
  auto run_ms = [h](double *ms) -> int {
    DDX_TRY(timed_setup(h));
    DDX_TRY(pipeline(h));
    DDX_TRY(sync(h));
    const auto t0 = std::chrono::steady_clock::now();
    DDX_TRY(timed_setup(h));
    DDX_TRY(pipeline(h));
    DDX_TRY(sync(h));
    *ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return DDX_OK;
  };
  static const int kWorkers[] = {4, 8, 16, 32, 64};
  static const int kSplits[] = {1, 2, 4};
  double best = 1e300, t = 0.0;
  int bw = h->workers_per_cu, bs = 1;
  h->workers_fixed = true;
  for (int w : kWorkers) {
    h->workers_per_cu = w;
    DDX_TRY(run_ms(&t));
    if (t < best) best = t, bw = w;
  }
  h->workers_per_cu = bw;
  best = 1e300;
  for (int sp : kSplits) {
    h->ysplit = sp;   // the block maps exist after the runs above
    DDX_TRY(run_ms(&t));
    if (t < best) best = t, bs = sp;
  }
  h->ysplit = bs;
  DDX_TRY(timed_setup(h));
  DDX_TRY(pipeline(h));
  DDX_TRY(sync(h));
  if (workers_per_cu) *workers_per_cu = bw;
  if (proj_split) *proj_split = bs;
  return DDX_OK;
}

int ddx_set_coulomb(ddx_handle *h, int mode) {
  if (!h || mode < DDX_COULOMB_AUTO || mode > DDX_COULOMB_FMM) {
    set_error("ddx_set_coulomb: mode must be one of DDX_COULOMB_*");
    return DDX_ERR_ARG;
  }
  if (mode == DDX_COULOMB_FMM && h->ninst > 1) {
    set_error("ddx_set_coulomb: batch handles sum the Coulomb terms directly");
    return DDX_ERR_STATE;
  }
  DDX_TRY(sync(h));
  h->coulomb_mode = mode;
  return DDX_OK;
}

int ddx_set_graphs(ddx_handle *h, int enable) {
  if (!h) return DDX_ERR_ARG;
  DDX_TRY(sync(h));
  h->use_graphs = enable != 0;
  return DDX_OK;
}

int ddx_kernel_timer(ddx_handle *h, int kernel, int enable) {
  if (!h || kernel < 0 || kernel >= DDX_K_COUNT) return DDX_ERR_ARG;
  KernelTimer &t = h->ktimer[kernel];
  DDX_TRY(sync(h));
  for (auto &r : t.recs) {
    t.pool.push_back(r.b);
    t.pool.push_back(r.e);
  }
  t.recs.clear();
  t.on = enable != 0;
  return DDX_OK;
}

int ddx_kernel_timer_read(ddx_handle *h, int kernel, int *launches, double *total_ms) {
  if (!h || kernel < 0 || kernel >= DDX_K_COUNT || !launches || !total_ms) return DDX_ERR_ARG;
  KernelTimer &t = h->ktimer[kernel];
  DDX_TRY(sync(h));
  double tot = 0.0;
  for (auto &r : t.recs) {
    float ms = 0.f;
    DDX_HIP(hipEventElapsedTime(&ms, r.b, r.e));
    tot += ms;
    t.pool.push_back(r.b);
    t.pool.push_back(r.e);
  }
  *launches = (int)t.recs.size();
  *total_ms = tot;
  t.recs.clear();
  return DDX_OK;
}

int ddx_get_stats(const ddx_handle *h, ddx_stats *st) {
  if (!h || !st) return DDX_ERR_ARG;
  DDX_TRY(read_setup_time(const_cast<ddx_handle *>(h)));
  *st = h->stats;
  return DDX_OK;
}

}  // extern "C"
