// The off-diagonal ddCOSMO operators on the neighbour triples.
//
// For a triple t = (owner sphere o, grid point n, container sphere c) with
// t_n^oc < 1 define the vector
//     R_lm(t) = 4pi/(2l+1) * (t_n^oc)^l * Y_lm(s_n^oc)
// (the factors of intmlp, ddcosmo.f90:1140-1178, and of adjrhs,
// ddcosmo.f90:1359-1377).  Then
//     L X :  P(n,o)  = sum_{t at (o,n)} W_t R(t) . X_c        (calcv, ddcosmo.f90:1671-1746)
//            (LX)_o  = - sum_n w_n Y(:,n) P(n,o)              (intrhs + lx, matvec.f90:127-136)
//     L* S:  xi(n,o) = Y(:,n) . S_o                           (matvec.f90:196-204)
//            (L*S)_c = - sum_{t in c} w_n xi(n,o) W_t R(t)    (adjrhs, matvec.f90:213-223)
//
// One sweep kernel serves both operators, and both at once: the triples are
// grouped by container c, one wave per container.  The per-(l, m) constant
// cf = facs * 4pi/(2l+1) is applied outside the triple loop: L X contracts
// with X' = cf X (16 values to a vector register, read by row broadcast),
// L* S accumulates sum_t coef_t p~ trig in registers per lane and multiplies
// by cf after one register reduce-scatter per segment.  When the direct
// and the adjoint solve run in lockstep a single pass over the triples
// builds each basis once for both.
// The basis follows ylmbas (ddcosmo.f90:830-895) with t^l folded into the
// Legendre recurrence of polleg (m outer, l inner, ddcosmo.f90:1056-1094):
//     p~(m, m)   = t^m P_m^m,   p~(m+1, m) = (2m+1) (t cos) p~(m, m)
//     p~(l, m)   = [(2l-1) (t cos) p~(l-1, m) - (l+m-1) t^2 p~(l-2, m)] / (l-m)
// and cos/sin(m phi) by the Chebyshev recurrence of trgev
// (ddcosmo.f90:1103-1125).
#include "ddx_device.hpp"
#include "ddx_kernels.hpp"

#include <type_traits>

namespace ddx {
namespace {

__host__ __device__ constexpr int lmi(int l, int m) { return l * l + l + m; }

// The adjoint accumulators of a lane live in registers.  Where all nylm of
// them do not fit they are split into blocks of consecutive m, each built by
// its own pass over the chunk's triples: block b holds the entries (l, +-m)
// with mblock_begin(b) <= m < mblock_begin(b + 1).  The first pass of the
// paired sweep also evaluates L X and gets a smaller budget.  The budgets
// are the largest that the register allocator fits in 256 VGPRs without
// spilling (its resource report, at two waves per SIMD).
// FP32 accumulators (F) take one register each instead of two.
__host__ __device__ constexpr int acc_cap(int lmax, bool F) {
  return F ? 128 : ((lmax == 13 || lmax == 14) ? 64 : 72);
}
__host__ __device__ constexpr int acc_pair_less(bool F) { return F ? 32 : 16; }  // taken by L X
__host__ __device__ constexpr int acc_one(bool F) { return F ? 144 : 81; }  // one block up to here

// entries (l, +-m), l = m..lmax
__host__ __device__ constexpr int mcount(int lmax, int m) {
  return (m == 0 ? 1 : 2) * (lmax + 1 - m);
}
// accumulators of m0 <= m < m1
__host__ __device__ constexpr int mspan(int lmax, int m0, int m1) {
  int c = 0;
  for (int m = m0; m < m1; ++m) c += mcount(lmax, m);
  return c;
}
// first m of block b; lmax + 1 once the blocks are used up
__host__ __device__ constexpr int mblock_begin(int lmax, bool dir, int b, bool F) {
  if ((lmax + 1) * (lmax + 1) <= acc_one(F)) return b == 0 ? 0 : lmax + 1;
  int m = 0;
  for (int k = 0; k < b && m <= lmax; ++k) {
    const int cap = acc_cap(lmax, F) - ((k == 0 && dir) ? acc_pair_less(F) : 0);
    int cnt = 0;
    while (m <= lmax && cnt + mcount(lmax, m) <= cap) cnt += mcount(lmax, m++);
  }
  return m;
}
// position of entry (l, m) (neg: (l, -m)) among the accumulators of the
// block m0 <= m < m1: lm order when the block holds all entries, else m by
// m, and inside m: l, +m before -m
__host__ __device__ constexpr int aidx(int lmax, int m0, int m1, int l, int m, bool neg) {
  if (m0 == 0 && m1 == lmax + 1) return l * l + l + (neg ? -m : m);
  return mspan(lmax, m0, m) + (m == 0 ? l : 2 * (l - m) + (neg ? 1 : 0));
}

// X' of the container, 16 values to a register: lane i holds the values 16 j + i
// mod 16 in r[j], so that every row of 16 lanes holds them all and an FMA reads
// value e of its row by row_newbcast.
//   What it replaces: every lane read the values from the wave's LDS row, a
// broadcast of 16 bytes in 8 cycles to each pair of values, so that at lmax 8
// the eight waves of a compute unit took the LDS 2600 cycles a triple against
// 3400 of FP64 issue, and waited for each read a few instructions later.  With
// the values as scalars (8 or 16 to a load through the scalar cache, one load
// ahead) the paired FP64 sweep of 2000 atoms took as long, 56 and 51 us, waiting
// for those; without either 32.  Paired FP64 sweep, LDS -> registers, us: 60
// atoms (lmax 6) 5.6 -> 4.7; 642 (6) 9.0 -> 6.9; 1000 (8) 34.9 -> 26.4; 2000 (8)
// 57 -> 44.5; 1500 (10) 132 -> 108; 500 (12) 66 -> 59; 300 (16) 80 -> 70.  FP32:
// 642 (6) 6.8 -> 5.7; 2000 (8) 36.3 -> 36.2.  What bounds the FP64 sweep now is
// its issue (43 us at 2000 atoms with every load and store left out) and the
// scattered stores of the terms (13 us in part under it).
template <typename R, int NY>
struct XRow {
  static constexpr int NR = (NY + 15) / 16;
  R r[NR];
};
__device__ __forceinline__ double fma_r(double a, double b, double c) {
  return __builtin_fma(a, b, c);
}
__device__ __forceinline__ float fma_r(float a, float b, float c) { return fmaf(a, b, c); }

// The sums of one basis value p: ap += p qc and an += p qs (the adjoint's),
// a += x_NA p and b += x_NB p (L X), x_N the value that lane N of the row holds.
//   A DPP read of a register must follow its last write by a vector instruction
// by two more instructions, which the compiler does not see to inside an asm
// block: the adjoint's FMAs come first, or waits stand in their place.
template <int NA, int NB>
__device__ __forceinline__ void fma4(double &ap, double &an, double &a, double &b, double p, double qc, double qs,
                                     double xa, double xb) {
  asm("v_fmac_f64_e32 %0, %4, %5\n\t"
      "v_fmac_f64_e32 %1, %4, %6\n\t"
      "v_fmac_f64_dpp %2, %7, %4 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %3, %8, %4 row_newbcast:%10 row_mask:0xf bank_mask:0xf"
      : "+&v"(ap), "+&v"(an), "+&v"(a), "+&v"(b)
      : "v"(p), "v"(qc), "v"(qs), "v"(xa), "v"(xb), "n"(NA), "n"(NB));
}
template <int NA, int NB>
__device__ __forceinline__ void fma4(float &ap, float &an, float &a, float &b, float p, float qc, float qs,
                                     float xa, float xb) {
  asm("v_fmac_f32_e32 %0, %4, %5\n\t"
      "v_fmac_f32_e32 %1, %4, %6\n\t"
      "v_fmac_f32_dpp %2, %7, %4 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %3, %8, %4 row_newbcast:%10 row_mask:0xf bank_mask:0xf"
      : "+&v"(ap), "+&v"(an), "+&v"(a), "+&v"(b)
      : "v"(p), "v"(qc), "v"(qs), "v"(xa), "v"(xb), "n"(NA), "n"(NB));
}
template <int NA>
__device__ __forceinline__ void fma2(double &ap, double &a, double p, double qc, double xa) {
  asm("v_fmac_f64_e32 %0, %2, %3\n\t"
      "s_nop 0\n\t"
      "v_fmac_f64_dpp %1, %4, %2 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
      : "+&v"(ap), "+&v"(a)
      : "v"(p), "v"(qc), "v"(xa), "n"(NA));
}
template <int NA>
__device__ __forceinline__ void fma2(float &ap, float &a, float p, float qc, float xa) {
  asm("v_fmac_f32_e32 %0, %2, %3\n\t"
      "s_nop 0\n\t"
      "v_fmac_f32_dpp %1, %4, %2 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
      : "+&v"(ap), "+&v"(a)
      : "v"(p), "v"(qc), "v"(xa), "n"(NA));
}
template <int NA, int NB>
__device__ __forceinline__ void dot2(double &a, double &b, double p, double xa, double xb) {
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %3, %2 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %4, %2 row_newbcast:%6 row_mask:0xf bank_mask:0xf"
      : "+&v"(a), "+&v"(b)
      : "v"(p), "v"(xa), "v"(xb), "n"(NA), "n"(NB));
}
template <int NA, int NB>
__device__ __forceinline__ void dot2(float &a, float &b, float p, float xa, float xb) {
  asm("s_nop 1\n\t"
      "v_fmac_f32_dpp %0, %3, %2 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %1, %4, %2 row_newbcast:%6 row_mask:0xf bank_mask:0xf"
      : "+&v"(a), "+&v"(b)
      : "v"(p), "v"(xa), "v"(xb), "n"(NA), "n"(NB));
}
template <int NA>
__device__ __forceinline__ void dot1(double &a, double p, double xa) {
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %2, %1 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
      : "+&v"(a)
      : "v"(p), "v"(xa), "n"(NA));
}
template <int NA>
__device__ __forceinline__ void dot1(float &a, float p, float xa) {
  asm("s_nop 1\n\t"
      "v_fmac_f32_dpp %0, %2, %1 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
      : "+&v"(a)
      : "v"(p), "v"(xa), "n"(NA));
}

// f(B), f(B + 1), .., f(E - 1) with the index as a constant expression
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F &&f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}
#define DDX_INLINE __attribute__((always_inline))

// the sums of p = p~_lm for the two entries (l, +-m)
template <int LMAX, bool DIR, bool ACC, int AM0, int AM1, int L, int M, typename R, int NY>
__device__ __forceinline__ void visit(const XRow<R, NY> &X, R p, R qc, R qs, R &a, R &b, R *acc) {
  constexpr int ea = lmi(L, M), eb = lmi(L, -M);
  if constexpr (ACC) {
    R &ap = acc[aidx(LMAX, AM0, AM1, L, M, false)];
    if constexpr (M == 0) {
      if constexpr (DIR) fma2<ea % 16>(ap, a, p, qc, X.r[ea / 16]);
      else ap = fma_r(p, qc, ap);
    } else {
      R &an = acc[aidx(LMAX, AM0, AM1, L, M, true)];
      if constexpr (DIR) {
        fma4<ea % 16, eb % 16>(ap, an, a, b, p, qc, qs, X.r[ea / 16], X.r[eb / 16]);
      } else {
        ap = fma_r(p, qc, ap);
        an = fma_r(p, qs, an);
      }
    }
  } else if constexpr (DIR) {
    if constexpr (M == 0) dot1<ea % 16>(a, p, X.r[ea / 16]);
    else dot2<ea % 16, eb % 16>(a, b, p, X.r[ea / 16], X.r[eb / 16]);
  }
}

// One triple: returns sum_lm p~_lm trig_m Xc'_lm when DIR and adds
// coef p~_lm trig_m to the accumulators of AM0 <= |m| < AM1 (trig_m =
// cos(m phi) for m >= 0, sin(|m| phi) for m < 0).  Without DIR the
// recurrences in m only step up to AM0 before the l recurrence starts.
// ct = t cos theta, st = t sin theta, t2 = t^2; coef is x0 w0 rounded, and the
// entry (0, 0) adds the product itself.  All roundings are written out: the DIIS
// extrapolation makes 1e-9 of a sum contracted differently.
template <int LMAX, bool DIR, int AM0, int AM1>
__device__ __forceinline__ double sweep_triple(double ct, double st, double t2, double cphi,
                                               double sphi,
                                               const XRow<double, (LMAX + 1) * (LMAX + 1)> &X,
                                               double x0, double w0, double coef,
                                               double *acc) {
#pragma clang fp contract(off)
  typedef double R;
  constexpr bool ADJ = AM0 < AM1;
  constexpr int MB = DIR ? 0 : AM0;          // first m with the l recurrence
  constexpr int ME = DIR ? LMAX + 1 : AM1;   // one past the last m needed
  R s = 0.0;
  R pmm = 1.0;   // t^m P_m^m
  R cm = 1.0, sm = 0.0, cprev = 0.0, sprev = 0.0;
  static_for<0, ME>([&](auto mc) DDX_INLINE {
    constexpr int m = decltype(mc)::value;
    if constexpr (m >= MB) {
      constexpr bool acc_m = ADJ && m >= AM0 && m < AM1;
      R qc = 0.0, qs = 0.0;
      if (acc_m) {
        qc = (m == 0) ? coef : coef * cm;
        qs = (m == 0) ? R(0) : coef * sm;
      }
      R a = 0.0, b = 0.0;
      // one m after the other: what is live stays within the registers
      if (DIR && m > 0) asm volatile("" : "+v"(pmm) : "v"(s));
      R p0 = 0.0, p1 = pmm;   // p~(l - 1, m), p~(l, m)
      static_for<m, LMAX + 1>([&](auto lc) DDX_INLINE {
        constexpr int l = decltype(lc)::value;
        if constexpr (l == m + 1) {
          p0 = p1;
          p1 = ((R)(2 * m + 1) * ct) * p0;
        } else if constexpr (l > m + 1) {
          constexpr R one = 1;
          constexpr R ca = (R)(2 * l - 1) * (one / (R)(l - m));
          constexpr R cb = (R)(l + m - 1) * (one / (R)(l - m));
          const R p2 = __builtin_fma(ca, ct * p1, -(cb * (t2 * p0)));
          p0 = p1;
          p1 = p2;
        }
        if constexpr (l == 0) {
          if constexpr (acc_m) acc[0] = __builtin_fma(x0, w0, acc[0]);
          visit<LMAX, DIR, false, AM0, AM1, l, m>(X, p1, qc, qs, a, b, acc);
        } else {
          visit<LMAX, DIR, acc_m, AM0, AM1, l, m>(X, p1, qc, qs, a, b, acc);
        }
      });
      if (DIR) s = (m == 0) ? a : s + __builtin_fma(cm, a, sm * b);
    }
    if constexpr (m + 1 < ME) {
      pmm = (-(R)(2 * m + 1) * st) * pmm;
      R cn, sn;
      if (m == 0) { cn = cphi; sn = sphi; }
      else {
        cn = __builtin_fma(R(2) * cphi, cm, -cprev);
        sn = __builtin_fma(R(2) * cphi, sm, -sprev);
      }
      cprev = cm; sprev = sm; cm = cn; sm = sn;
    }
  });
  return s;
}

// Ratio K(l, m) / K(l - 1, m) of the scales of the FP32 basis (l > m), and
// the coefficient of t^2 q(l - 2, m) in its recurrence (l >= m + 2).
__host__ __device__ constexpr double basis_ratio(int l, int m) {
  return l == m + 1 ? 2.0 * m + 1.0 : (2.0 * l - 1.0) / (double)(l - m);
}
__host__ __device__ constexpr double basis_beta(int l, int m) {
  return ((double)(l + m - 1) / (double)(l - m)) / (basis_ratio(l, m) * basis_ratio(l - 1, m));
}

// sweep_triple in FP32 on the scaled basis q_lm = p~_lm / K_lm (ct = t cos
// theta, st = t sin theta, t^2 = ct^2 + st^2), where
//     K(m, m) = -(2m - 1) K(m - 1, m - 1),  K(m + 1, m) = (2m + 1) K(m, m),
//     K(l, m) = (2l - 1) / (l - m) K(l - 1, m),
// so that every recurrence step has one product less:
//     q(m, m) = st q(m - 1, m - 1),  q(m + 1, m) = ct q(m, m),
//     q(l, m) = ct q(l - 1, m) - beta(l, m) t^2 q(l - 2, m).
// Xc holds K X' and the caller multiplies the adjoint sums by K.
template <int LMAX, bool DIR, int AM0, int AM1>
__device__ __forceinline__ float sweep_triple32(float ct, float st, float cphi, float sphi,
                                                const XRow<float, (LMAX + 1) * (LMAX + 1)> &X,
                                                float coef, float *acc) {
  constexpr bool ADJ = AM0 < AM1;
  constexpr int MB = DIR ? 0 : AM0;          // first m with the l recurrence
  constexpr int ME = DIR ? LMAX + 1 : AM1;   // one past the last m needed
  const float t2 = fmaf(ct, ct, st * st), c2 = 2.0f * cphi;
  float s = 0.0f;
  float qmm = 1.0f;
  float cm = 1.0f, sm = 0.0f, cprev = 0.0f, sprev = 0.0f;
  static_for<0, ME>([&](auto mc) DDX_INLINE {
    constexpr int m = decltype(mc)::value;
    if constexpr (m >= MB) {
      constexpr bool acc_m = ADJ && m >= AM0 && m < AM1;
      float qc = 0.0f, qs = 0.0f;
      if (acc_m) {
        qc = (m == 0) ? coef : coef * cm;
        qs = (m == 0) ? 0.0f : coef * sm;
      }
      float a = 0.0f, b = 0.0f;
      if (DIR && m > 0) asm volatile("" : "+v"(qmm) : "v"(s));
      float q0 = 0.0f, q1 = qmm;   // q(l - 1, m), q(l, m)
      static_for<m, LMAX + 1>([&](auto lc) DDX_INLINE {
        constexpr int l = decltype(lc)::value;
        if constexpr (l == m + 1) {
          q0 = q1;
          q1 = ct * q0;
        } else if constexpr (l > m + 1) {
          const float q2 = fmaf(-(float)basis_beta(l, m), t2 * q0, ct * q1);
          q0 = q1;
          q1 = q2;
        }
        visit<LMAX, DIR, acc_m, AM0, AM1, l, m>(X, q1, qc, qs, a, b, acc);
      });
      if (DIR) {
        if (m == 0) {
          s = a;
        } else {
          s = fmaf(cm, a, s);
          s = fmaf(sm, b, s);
        }
      }
    }
    if constexpr (m + 1 < ME) {
      qmm = st * qmm;
      float cn, sn;
      if (m == 0) {
        cn = cphi;
        sn = sphi;
      } else {
        cn = fmaf(c2, cm, -cprev);
        sn = fmaf(c2, sm, -sprev);
      }
      cprev = cm; sprev = sm; cm = cn; sm = sn;
    }
  });
  return s;
}

// The per-triple records in the sweep's arithmetic: (cos theta, sin theta,
// cos phi, sin phi) and (t, W) as double4 / double2 for the FP64 sweep;
// (t cos theta, t sin theta, cos phi, sin phi) as float4 and W as float for
// the FP32 sweep (20 bytes: t enters only through those products and t^2).
template <typename R>
struct Geo {
  typedef double4 G4;
  typedef double2 G2;
};
template <>
struct Geo<float> {
  typedef float4 G4;   // (t cos theta, t sin theta, cos phi, sin phi)
  typedef float G2;    // W
};

// One pass over triples beg..end-1 (end > beg) of a container: rw[tslot] =
// W (R . X_c) when DIR, and when AM0 < AM1 the (l, +-m),
// AM0 <= m < AM1, entries of the chunk's share of (L*S)_c, -cf * sum_t w_n
// xi(n, o) W p~ trig, into the segment row yp.  The FP32 pass works on the
// scaled basis of sweep_triple32: X holds K X' and the sums are scaled by
// cf K (the table after cf, 1/(l+1), 1/facl and K in cf).
template <typename R, int LMAX, bool DIR, int AM0, int AM1>
__device__ __forceinline__ void sweep_pass(
    int beg, int end, const typename Geo<R>::G4 *__restrict__ tgeo,
    const typename Geo<R>::G2 *__restrict__ ttw,
    const int *__restrict__ tslot, const int *__restrict__ tp, const XRow<R, (LMAX + 1) * (LMAX + 1)> &X,
    R *__restrict__ rw, int spare, const R *__restrict__ xiw,
    const double *__restrict__ cf, double *__restrict__ yp) {
  constexpr bool F = sizeof(R) == 4;
  constexpr bool ADJ = AM0 < AM1;
  constexpr int NA = ADJ ? mspan(LMAX, AM0, AM1) : 1;
  R acc[NA];
#pragma unroll
  for (int k = 0; k < NA; ++k) acc[k] = R(0);
  typedef typename Geo<R>::G4 G4;
  typedef typename Geo<R>::G2 G2;
  int k = beg + lane_id();
  if constexpr (F) {
    // Software pipeline, two triples deep: geometry, slot and owner point of
    // triple k + 128 and xi of triple k + 64 load while triple k is evaluated.
    // Indices past the chunk read its last triple instead, so that no load
    // is conditional, and the loop is unrolled by three so that the three
    // stages rotate by name (a register copy of a load in flight waits for
    // it).  The rounds have no exit between their steps, which would let the
    // compiler sink the loads to their uses: a lane past the chunk's end
    // evaluates its clamped triple with weight 0 and stores into the spare
    // slot rw[spare].
    struct Stage {
      G4 g;
      G2 w;   // W
      int s, p;
      R x;
    };
    const int last = end - 1;
    auto fetch = [&](Stage &st, int j) {
      j = min(j, last);
      st.g = tgeo[j];
      st.w = ttw[j];
      if constexpr (DIR) st.s = tslot[j];
      if constexpr (ADJ) st.p = tp[j];
    };
    Stage A, B, C;
    fetch(A, k);
    if constexpr (ADJ) A.x = xiw[A.p];
    fetch(B, k + kWave);
    // triple k from cur; triple k + 128 into fut, xi of triple k + 64 into nxt
    auto step = [&](Stage &cur, Stage &nxt, Stage &fut) {
      fetch(fut, k + 2 * kWave);
      if constexpr (ADJ) nxt.x = xiw[nxt.p];
      const bool live = k < end;
      const R coef = ADJ ? (live ? cur.x * cur.w : R(0)) : R(0);
      const R v = sweep_triple32<LMAX, DIR, AM0, AM1>(cur.g.x, cur.g.y, cur.g.z, cur.g.w, X,
                                                      coef, acc);
      if constexpr (DIR) rw[live ? cur.s : spare] = cur.w * v;
      k += kWave;
    };
    const int nit = (end - beg + kWave - 1) / kWave;   // the same in all lanes
    int it = 0;
    for (; it + 3 <= nit; it += 3) {
      step(A, B, C);
      step(B, C, A);
      step(C, A, B);
    }
    if (it < nit) {
      step(A, B, C);
      if (it + 1 < nit) step(B, C, A);
    }
  } else {
    // Indices past the chunk as in FP32.  One stage of registers: the triple's
    // values leave the loaded registers first, then the loads of the next
    // triple go into these and are waited for a whole evaluation later.  (A loop
    // that copied stages down, with its loads under bounds tests, waited for
    // them in the iteration that issued them.)
    const int last = end - 1;
    const int k0 = min(k, last);
    G4 g = tgeo[k0];
    G2 w = ttw[k0];
    int slot = 0, pn = 0;
    R x = R(0);
    if constexpr (DIR) slot = tslot[k0];
    if constexpr (ADJ) {
      x = xiw[tp[k0]];
      pn = tp[min(k + kWave, last)];
    }
    for (int it = (end - beg + kWave - 1) / kWave; it > 0; --it) {
      const bool live = k < end;
      R ct = g.x * w.x, st = g.y * w.x, t2 = w.x * w.x;
      R cphi, sphi, wt, x0 = R(0);
      int at = 0;
      asm volatile("v_mov_b64_e32 %0, %1" : "=&v"(cphi) : "v"(g.z));
      asm volatile("v_mov_b64_e32 %0, %1" : "=&v"(sphi) : "v"(g.w));
      asm volatile("v_mov_b64_e32 %0, %1" : "=&v"(wt) : "v"(w.y));
      if constexpr (DIR) at = live ? slot : spare;
      if constexpr (ADJ) x0 = live ? x : R(0);
      R coef = x0 * wt;
      asm volatile("" : "+v"(ct), "+v"(st), "+v"(t2), "+v"(x0), "+v"(coef), "+v"(at));
      const int j = min(k + kWave, last);
      g = tgeo[j];
      w = ttw[j];
      if constexpr (DIR) slot = tslot[j];
      if constexpr (ADJ) {
        x = xiw[pn];
        pn = tp[min(k + 2 * kWave, last)];
      }
      __builtin_amdgcn_sched_barrier(0);
      const R v = sweep_triple<LMAX, DIR, AM0, AM1>(ct, st, t2, cphi, sphi, X, x0, wt, coef, acc);
      if constexpr (DIR) rw[at] = wt * v;
      k += kWave;
    }
  }
  if constexpr (ADJ) {
    // sum of acc over the 64 lanes, entry by entry, spread over the lanes
    int base = 0, len = NA;
    wave_reduce_split<0, NA, R>(acc, base, len);
    constexpr int NF = reduced_len(NA, 6);
    constexpr int NY = (LMAX + 1) * (LMAX + 1);
    const double *cs = F ? cf + 4 * NY : cf;   // cf K or cf
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      if (j < len) {
        // lm of block entry q
        const int q = base + j;
        int lm = q;
#pragma unroll
        for (int m = AM0; m < ((AM0 == 0 && AM1 == LMAX + 1) ? AM0 : AM1); ++m) {
          const int o = mspan(LMAX, AM0, m);
          if (q >= o && q < o + mcount(LMAX, m)) {
            const int r = q - o;
            const int l = m + (m == 0 ? r : (r >> 1));
            lm = lmi(l, (m > 0 && (r & 1)) ? -m : m);
          }
        }
        yp[lm] = -(cs[lm] * (double)acc[j]);
      }
    }
  }
}

// The adjoint passes of blocks B.. (the first also evaluates L X when DIR)
template <typename R, int LMAX, bool DIR, int B>
__device__ __forceinline__ void sweep_blocks(
    int beg, int end, const typename Geo<R>::G4 *__restrict__ tgeo,
    const typename Geo<R>::G2 *__restrict__ ttw,
    const int *__restrict__ tslot, const int *__restrict__ tp, const XRow<R, (LMAX + 1) * (LMAX + 1)> &X,
    R *__restrict__ rw, int spare, const R *__restrict__ xiw,
    const double *__restrict__ cf, double *__restrict__ yp) {
  constexpr bool F = sizeof(R) == 4;
  constexpr int M0 = mblock_begin(LMAX, DIR, B, F), M1 = mblock_begin(LMAX, DIR, B + 1, F);
  sweep_pass<R, LMAX, DIR && B == 0, M0, M1>(beg, end, tgeo, ttw, tslot, tp, X, rw, spare,
                                             xiw, cf, yp);
  if constexpr (M1 <= LMAX) sweep_blocks<R, LMAX, DIR, B + 1>(beg, end, tgeo, ttw, tslot, tp,
                                                             X, rw, spare, xiw, cf, yp);
}

// Triples beg..end-1 of container c: rw[tslot] = W (R . X_c) when DIR
// (rw[spare]: scratch), and when ADJ the chunk's share of (L*S)_c into the
// segment row yp.
template <typename R, int LMAX, bool DIR, bool ADJ>
__device__ __forceinline__ void sweep_chunk(
    int c, int beg, int end, const typename Geo<R>::G4 *__restrict__ tgeo,
    const typename Geo<R>::G2 *__restrict__ ttw,
    const int *__restrict__ tslot, const int *__restrict__ tp, const double *__restrict__ Xs,
    R *__restrict__ rw, int spare, const R *__restrict__ xiw, const double *__restrict__ cf,
    double *__restrict__ yp) {
  constexpr int NY = (LMAX + 1) * (LMAX + 1);
  // (rounded to R; K X' in FP32, for the scaled basis of sweep_triple32)
  XRow<R, NY> X;
  if constexpr (DIR) {
#pragma unroll
    for (int j = 0; j < XRow<R, NY>::NR; ++j) {
      const int k = min(16 * j + (lane_id() & 15), NY - 1);
      const double x = Xs[(size_t)c * NY + k];
      X.r[j] = sizeof(R) == 4 ? (R)(x * cf[3 * NY + k]) : (R)x;
    }
  }
  if constexpr (ADJ)
    sweep_blocks<R, LMAX, DIR, 0>(beg, end, tgeo, ttw, tslot, tp, X, rw, spare, xiw, cf, yp);
  else
    sweep_pass<R, LMAX, true, 0, 0>(beg, end, tgeo, ttw, tslot, tp, X, rw, spare, xiw, cf, yp);
}

// Workgroups go to the 8 XCDs in turn: the b-th of n, renumbered so that each
// XCD takes a contiguous range.  In a batch a molecule's point values and terms
// then stay in one XCD's L2: paired FP32 sweep of 512 molecules (lmax 6) 485 ->
// 445 us, FP64 of 64 molecules 45.8 -> 41.7.  A large single system, whose
// points do not fit there, is better off in turn: 1500 atoms (lmax 10) 110.6
// against 115.1 us, 6000 (lmax 8) 127 against 131.
__device__ __forceinline__ int xcd_block(int b, int n) {
  const int x = b & 7, per = n >> 3, rem = n & 7;
  return x * per + min(x, rem) + (b >> 3);
}

// One wave per worker w (kSweepWaves to a workgroup, w < G): units
// floor(w U / G) .. floor((w+1) U / G) - 1, container by container.  DIR:
// L X terms (rw, slot order); ADJ: one partial L* S per segment (yp).  A side whose solve
// has ended (gate done) is skipped; in a batch (inst: the instance of each
// sphere, gates: the summaries after ninst instance states) so is every
// container of an instance that has converged.
// (two waves per SIMD: the register budget that keeps a block of
// accumulators, X' and the loads ahead without spilling)
template <typename R, int LMAX, bool DIR, bool ADJ>
__global__ __launch_bounds__(kWave * kSweepWaves, 2) void k_sweep(
    int G, const int4 *__restrict__ wstart, const int *__restrict__ uoff,
    const int *__restrict__ segoff, const int *__restrict__ toff,
    const typename Geo<R>::G4 *__restrict__ tgeo,
    const typename Geo<R>::G2 *__restrict__ ttw,
    const int *__restrict__ tslot, const int *__restrict__ tp, const double *__restrict__ Xs,
    R *__restrict__ rw, int spare, const R *__restrict__ xiw, const double *__restrict__ cf,
    double *__restrict__ yp, const DiisState *__restrict__ gdir,
    const DiisState *__restrict__ gadj, const int *__restrict__ inst, int ninst) {
  constexpr int NY = (LMAX + 1) * (LMAX + 1);
  // (the wave index through readfirstlane: the compiler does not see that
  // threadIdx.x / 64 is uniform across a wave, and every quantity below
  // would otherwise live in vector registers and load per lane)
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  const int b = inst ? xcd_block((int)blockIdx.x, (int)gridDim.x) : (int)blockIdx.x;
  const int w = b * kSweepWaves + wave;
  if (w >= G) return;
  const int4 at = wstart[w];
  const int u1 = wstart[w + 1].y;
  const bool dir = DIR && !(gdir && gdir->done);
  const bool adj = ADJ && !(gadj && gadj->done);
  if (!dir && !adj) return;
  int c = at.x, seg = at.z, beg = at.w;
  for (int u = at.y; u < u1;) {
    int uc = uoff[c + 1];
    while (uc <= u) {   // on to the next container (some hold no triples)
      ++c;
      uc = uoff[c + 1];
      seg = segoff[c];
      beg = toff[c];
    }
    const int ue = min(u1, uc);
    const int end = min(toff[c + 1], beg + (ue - u) * kWave);
    double *ys = yp + (size_t)seg * NY;
    bool dc = dir, ac = adj;
    if (inst) {
      const int q = inst[c] - ninst;   // the instance's state, before the summary
      dc = dc && !(gdir && gdir[q].done);
      ac = ac && !(gadj && gadj[q].done);
    }
    if constexpr (DIR && ADJ) {
      if (dc && ac)
        sweep_chunk<R, LMAX, true, true>(c, beg, end, tgeo, ttw, tslot, tp, Xs, rw, spare, xiw, cf, ys);
      else if (dc)
        sweep_chunk<R, LMAX, true, false>(c, beg, end, tgeo, ttw, tslot, tp, Xs, rw, spare, xiw, cf, ys);
      else if (ac)
        sweep_chunk<R, LMAX, false, true>(c, beg, end, tgeo, ttw, tslot, tp, Xs, rw, spare, xiw, cf, ys);
    } else if constexpr (DIR) {
      if (dc)
        sweep_chunk<R, LMAX, true, false>(c, beg, end, tgeo, ttw, tslot, tp, Xs, rw, spare, xiw, cf, ys);
    } else {
      if (ac)
        sweep_chunk<R, LMAX, false, true>(c, beg, end, tgeo, ttw, tslot, tp, Xs, rw, spare, xiw, cf, ys);
    }
    u = ue;
  }
}

// P(n,o) = sum of the point's weighted terms, in neighbour order.  Points
// with ui = 1, which calcv skips (ddcosmo.f90:1698), are exactly the points
// without triples (ui < 1 iff some t < 1), so their P is zero here as well.
template <typename R>
__global__ __launch_bounds__(256) void k_gather_points(size_t np, int ngrid,
                                                       const int *__restrict__ ptoff,
                                                       const R *__restrict__ rw,
                                                       R *__restrict__ P,
                                                       const DiisState *__restrict__ gate,
                                                       const int *__restrict__ inst, int ninst) {
  // points of spheres whose molecules have all converged are not read again
  {
    const size_t p0 = (size_t)blockIdx.x * blockDim.x;
    const size_t p1 = min(np, p0 + blockDim.x);
    if (!spheres_active(gate, inst, ninst, (int)(p0 / ngrid), (int)((p1 - 1) / ngrid) + 1))
      return;
  }
  size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  const int b = ptoff[p], e = ptoff[p + 1];
  // the first four terms are loaded together (most points have at most
  // four), then added in order like the rest
  R v[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = (b + k < e) ? rw[b + k] : R(0);
  R s = R(0);
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (b + k < e) s += v[k];
  for (int k = b + 4; k < e; ++k) s += rw[k];
  P[p] = s;
}

// (L*S)_c = sum of its segments' shares, in segment order
__global__ void k_seg_sum(int n, int nylm, const int *__restrict__ segoff,
                          const double *__restrict__ yp, double *__restrict__ y,
                          const DiisState *__restrict__ gate) {
  if (gate && gate->done) return;
  size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= (size_t)n * nylm) return;
  const int c = (int)(k / nylm), lm = (int)(k % nylm);
  double r = 0.0;
  for (int j = segoff[c]; j < segoff[c + 1]; ++j) r += yp[(size_t)j * nylm + lm];
  y[k] = r;
}

// xs = cf * x, elementwise over (nylm, nsph)
__global__ void k_cf_scale(size_t nn, int nylm, const double *__restrict__ cf,
                           const double *__restrict__ x, double *__restrict__ xs) {
  size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < nn) xs[k] = cf[k % nylm] * x[k];
}

// ---------------------------------------------------------------------------
// Far-field expansions of the Coulomb sums (used by k_fmm.hip).  The local
// expansion at target sphere i of the point charges j far from it:
//   A_i,lm = cf_lm sum_{j: d_ij^2 >= rc_i^2} (q_j / d) t^l p~_l^m(cos) trig_m,
//   t = R_i / d,  rc_i = R_i / rho
// (addition theorem: 1/|R s - v| = sum_l 4pi/(2l+1) R^l / d^(l+1)
// Y_lm(s) Y_lm(v / d) for R < d), so that the far charges' potential at the
// point R_i s of sphere i is sum_lm A_lm Y_lm(s), with a truncation error
// below (q / (d - R)) rho^(P+1) per charge.  One wave per target sphere,
// lanes over the charges of its instance, one pass per block of
// accumulators (the sweep's m-blocks), each lane's sums reduce-scattered.
template <int P, int AM0, int AM1>
__device__ __forceinline__ void p2l_pass(int i, double4 si, double rc2, int sb, int se,
                                         const double4 *__restrict__ sph,
                                         const double *__restrict__ q,
                                         const double *__restrict__ cf, double *__restrict__ A) {
  constexpr int NA = mspan(P, AM0, AM1);
  constexpr int NY = (P + 1) * (P + 1);
  const XRow<double, NY> none{};
  double acc[NA];
#pragma unroll
  for (int k = 0; k < NA; ++k) acc[k] = 0.0;
  for (int j = sb + (int)threadIdx.x; j < se; j += kWave) {
    const double4 sj = sph[j];
    const double vx = sj.x - si.x, vy = sj.y - si.y, vz = sj.z - si.z;
    double d2;
    {
#pragma clang fp contract(off)
      const double ax = si.x - sj.x, ay = si.y - sj.y, az = si.z - sj.z;
      d2 = (ax * ax + ay * ay) + az * az;   // as the near lists classify the pair
    }
    double coef = 0.0, cthe = 1.0, sthe = 0.0, cphi = 1.0, sphi = 0.0, t = 0.0;
    if (d2 >= rc2 && j != i) {
      const double id = 1.0 / sqrt(d2);
      const double rxy = sqrt(vx * vx + vy * vy);
      coef = q[j] * id;
      t = si.w * id;
      cthe = vz * id;
      sthe = rxy * id;
      if (rxy > 0.0) {
        cphi = vx / rxy;
        sphi = vy / rxy;
      }
    }
    sweep_triple<P, false, AM0, AM1>(cthe * t, sthe * t, t * t, cphi, sphi, none, coef, 1.0, coef, acc);
  }
  int base = 0, len = NA;
  wave_reduce_split<0, NA, double>(acc, base, len);
  constexpr int NF = reduced_len(NA, 6);
#pragma unroll
  for (int j = 0; j < NF; ++j) {
    if (j < len) {
      const int qi = base + j;
      int lm = qi;
#pragma unroll
      for (int m = AM0; m < ((AM0 == 0 && AM1 == P + 1) ? AM0 : AM1); ++m) {
        const int o = mspan(P, AM0, m);
        if (qi >= o && qi < o + mcount(P, m)) {
          const int r = qi - o;
          const int l = m + (m == 0 ? r : (r >> 1));
          lm = lmi(l, (m > 0 && (r & 1)) ? -m : m);
        }
      }
      A[(size_t)i * NY + lm] = cf[lm] * acc[j];
    }
  }
}

template <int P, int B>
__device__ __forceinline__ void p2l_blocks(int i, double4 si, double rc2, int sb, int se,
                                           const double4 *__restrict__ sph,
                                           const double *__restrict__ q,
                                           const double *__restrict__ cf,
                                           double *__restrict__ A) {
  constexpr int M0 = mblock_begin(P, false, B, false), M1 = mblock_begin(P, false, B + 1, false);
  p2l_pass<P, M0, M1>(i, si, rc2, sb, se, sph, q, cf, A);
  if constexpr (M1 <= P) p2l_blocks<P, B + 1>(i, si, rc2, sb, se, sph, q, cf, A);
}

// sources of target sphere i: the spheres of its instance (soff, inst) or
// all n spheres
template <int P>
__global__ __launch_bounds__(kWave, 2) void k_p2l(int n, const double4 *__restrict__ sph,
                                                  const double *__restrict__ q,
                                                  const int *__restrict__ inst,
                                                  const int *__restrict__ soff, double rho,
                                                  const double *__restrict__ cf,
                                                  double *__restrict__ A) {
  const int i = blockIdx.x;
  if (i >= n) return;
  const double4 si = sph[i];
  const double rc = si.w / rho;
  int sb = 0, se = n;
  if (inst) {
    sb = soff[inst[i]];
    se = soff[inst[i] + 1];
  }
  p2l_blocks<P, 0>(i, si, rc * rc, sb, se, sph, q, cf, A);
}

// the FP32 sweeps' per-triple records (geo32_of, and W), made once per
// setup (on the first FP32 sweep after it)
__global__ void k_geo_to_f32(long long n, const double4 *__restrict__ g,
                             const double2 *__restrict__ w, float4 *__restrict__ g32,
                             float *__restrict__ w32) {
  const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const double4 a = g[k];
  const double2 b = w[k];
  g32[k] = geo32_of(a, b);
  w32[k] = (float)b.y;
}

int geometry32(ddx_handle *h, hipStream_t s) {
  if (h->have_geo32) return DDX_OK;
  DDX_TRY(h->tgeo32.reserve((size_t)h->ntri + 1));
  DDX_TRY(h->ttw32.reserve((size_t)h->ntri + 1));
  if (h->ntri > 0) {
    hipLaunchKernelGGL(k_geo_to_f32, dim3((unsigned)(((long long)h->ntri + 255) / 256)),
                       dim3(256), 0, s, (long long)h->ntri, h->tgeo.p, h->ttw.p, h->tgeo32.p,
                       h->ttw32.p);
    DDX_HIP(hipGetLastError());
  }
  h->have_geo32 = true;
  return DDX_OK;
}

template <typename R, int LMAX, bool DIR, bool ADJ>
int launch_sweep(ddx_handle *h, hipStream_t s, const double *Xs, R *rw, const R *xiw, double *yp,
                 const DiisState *gdir, const DiisState *gadj) {
  if (h->nworker == 0) return DDX_OK;
  const typename Geo<R>::G4 *tgeo;
  const typename Geo<R>::G2 *ttw;
  if constexpr (sizeof(R) == 4) {
    DDX_TRY(geometry32(h, s));
    tgeo = h->tgeo32.p;
    ttw = h->ttw32.p;
  } else {
    tgeo = h->tgeo.p;
    ttw = h->ttw.p;
  }
  TimedLaunch tl(h, (DIR && ADJ) ? DDX_K_SWEEP_PAIR : (DIR ? DDX_K_SWEEP_L : DDX_K_SWEEP_LSTAR), s);
  hipExtLaunchKernelGGL((k_sweep<R, LMAX, DIR, ADJ>),
                        dim3((h->nworker + kSweepWaves - 1) / kSweepWaves),
                        dim3(kWave * kSweepWaves), 0, s, tl.b,
                        tl.e, 0, h->nworker, h->wstart.p, h->uoff.p, h->segoff.p, h->toff.p, tgeo,
                        ttw, h->tslot.p, h->tp.p, Xs, rw, (int)h->ntri, xiw, h->cf.p, yp, gdir, gadj,
                        h->ninst > 1 ? h->inst.p : nullptr, h->ninst);
  DDX_HIP(hipGetLastError());
  return DDX_OK;
}

template <typename R, int LMAX>
int sweep_lmax(ddx_handle *h, hipStream_t s, int mode, const double *Xs, R *rw, const R *xiw,
               double *y, const DiisState *gdir, const DiisState *gadj) {
  if (mode == 3) return launch_sweep<R, LMAX, true, true>(h, s, Xs, rw, xiw, y, gdir, gadj);
  if (mode == 1) return launch_sweep<R, LMAX, true, false>(h, s, Xs, rw, xiw, y, gdir, gadj);
  return launch_sweep<R, LMAX, false, true>(h, s, Xs, rw, xiw, y, gdir, gadj);
}

// mode: 1 = L X terms, 2 = L* S shares per segment, 3 = both.  R: the
// arithmetic of the sweep (double, or float in the increment rounds of the
// mixed precision); X' and the L* S shares stay double.
template <typename R>
int sweep(ddx_handle *h, hipStream_t s, int mode, const double *Xs, R *rw, const R *xiw,
          double *y, const DiisState *gdir, const DiisState *gadj) {
  if (h->n == 0) return DDX_OK;
  switch (h->lmax) {
    case 0: return sweep_lmax<R, 0>(h, s, mode, Xs, rw, xiw, y, gdir, gadj);
    case 1: return sweep_lmax<R, 1>(h, s, mode, Xs, rw, xiw, y, gdir, gadj);
    case 2: return sweep_lmax<R, 2>(h, s, mode, Xs, rw, xiw, y, gdir, gadj);
    case 3: return sweep_lmax<R, 3>(h, s, mode, Xs, rw, xiw, y, gdir, gadj);
    case 4: return sweep_lmax<R, 4>(h, s, mode, Xs, rw, xiw, y, gdir, gadj);
    case 5: return sweep_lmax<R, 5>(h, s, mode, Xs, rw, xiw, y, gdir, gadj);
    case 6: return sweep_lmax<R, 6>(h, s, mode, Xs, rw, xiw, y, gdir, gadj);
    case 7: return sweep_lmax<R, 7>(h, s, mode, Xs, rw, xiw, y, gdir, gadj);
    case 8: return sweep_lmax<R, 8>(h, s, mode, Xs, rw, xiw, y, gdir, gadj);
    case 9: return sweep_lmax<R, 9>(h, s, mode, Xs, rw, xiw, y, gdir, gadj);
    case 10: return sweep_lmax<R, 10>(h, s, mode, Xs, rw, xiw, y, gdir, gadj);
    case 11: return sweep_lmax<R, 11>(h, s, mode, Xs, rw, xiw, y, gdir, gadj);
    case 12: return sweep_lmax<R, 12>(h, s, mode, Xs, rw, xiw, y, gdir, gadj);
    case 13: return sweep_lmax<R, 13>(h, s, mode, Xs, rw, xiw, y, gdir, gadj);
    case 14: return sweep_lmax<R, 14>(h, s, mode, Xs, rw, xiw, y, gdir, gadj);
    case 15: return sweep_lmax<R, 15>(h, s, mode, Xs, rw, xiw, y, gdir, gadj);
    case 16: return sweep_lmax<R, 16>(h, s, mode, Xs, rw, xiw, y, gdir, gadj);
    default: set_error("lmax %d not supported (0..16)", h->lmax); return DDX_ERR_ARG;
  }
}

// P = gathered L X terms of each point; y = - Yw^T-projection of P
template <typename R>
int finish_lx(ddx_handle *h, Lane &ln, double *y, const DiisState *gate, int ysplit) {
  hipStream_t s = ln.stream;
  R *rw = reinterpret_cast<R *>(ln.rw.p);
  R *P = reinterpret_cast<R *>(ln.P.p);
  if constexpr (sizeof(R) == 4) {
    bool done = false;
    DDX_TRY(project32_gathered(h, s, -1.0, rw, y, gate, ysplit, &done));
    if (done) return DDX_OK;
  }
  hipLaunchKernelGGL(k_gather_points<R>, dim3((h->np + 255) / 256), dim3(256), 0, s, h->np,
                     h->ngrid, h->ptoff.p, rw, P, gate, h->ninst > 1 ? h->inst.p : nullptr,
                     h->ninst);
  DDX_HIP(hipGetLastError());
  // y(lm, o) = - sum_n Yw(lm, n) P(n, o)
  if constexpr (sizeof(R) == 4) return project32(h, s, -1.0, P, y, gate, ysplit);
  else return project(h, s, -1.0, P, y, gate, ysplit);
}

// the lane's point values of the L* S sweep: w_n xi(n, o) in R
template <typename R>
int expand_xi(ddx_handle *h, Lane &ln, const double *x, const DiisState *gate) {
  R *xiw = reinterpret_cast<R *>(ln.xiw.p);
  if constexpr (sizeof(R) == 4) return expand32(h, ln.stream, x, xiw, true, gate);
  else return expand(h, ln.stream, x, xiw, true, gate);
}

template <typename R>
int lx_r(ddx_handle *h, Lane &ln, const double *x, double *y, const DiisState *gate,
         bool xs_ready, int ysplit) {
  if (!xs_ready) DDX_TRY(cf_scale(h, ln.stream, x, ln.xs.p));
  DDX_TRY(sweep<R>(h, ln.stream, 1, ln.xs.p, reinterpret_cast<R *>(ln.rw.p), nullptr, nullptr,
                   gate, nullptr));
  return finish_lx<R>(h, ln, y, gate, ysplit);
}

template <typename R>
int lstarx_r(ddx_handle *h, Lane &ln, const double *x, double *y, const DiisState *gate,
             bool want_y) {
  // w_n xi(n, o) = w_n sum_lm Y(lm, n) x(lm, o)
  DDX_TRY(expand_xi<R>(h, ln, x, gate));
  DDX_TRY(sweep<R>(h, ln.stream, 2, nullptr, nullptr, reinterpret_cast<const R *>(ln.xiw.p),
                   ln.yp.p, nullptr, gate));
  return want_y ? seg_sum(h, ln.stream, ln.yp.p, y, gate) : DDX_OK;
}

template <typename R>
int pair_r(ddx_handle *h, Lane &ld, double *yd, const DiisState *gd, Lane &la, const double *xa,
           const DiisState *ga, int ysplit) {
  DDX_TRY(expand_xi<R>(h, la, xa, ga));
  DDX_TRY(sweep<R>(h, ld.stream, 3, ld.xs.p, reinterpret_cast<R *>(ld.rw.p),
                   reinterpret_cast<const R *>(la.xiw.p), la.yp.p, gd, ga));
  return finish_lx<R>(h, ld, yd, gd, ysplit);
}

int reserve_lx(ddx_handle *h, Lane &ln) {
  DDX_TRY(ln.rw.reserve(h->ntri + 1));
  DDX_TRY(ln.P.reserve(h->np));
  return ln.xs.reserve((size_t)h->nylm * h->n + 1);
}

int reserve_lstarx(ddx_handle *h, Lane &ln) {
  DDX_TRY(ln.xiw.reserve(h->np));
  return ln.yp.reserve((size_t)h->nseg_cap * h->nylm + 1);
}

}  // namespace

double sweep_basis_scale(int l, int m) {
  double K = 1.0;
  for (int j = 1; j <= m; ++j) K *= -(2.0 * j - 1.0);
  for (int j = m + 1; j <= l; ++j) K *= basis_ratio(j, m);
  return K;
}

int cf_scale(ddx_handle *h, hipStream_t s, const double *x, double *xs) {
  size_t nn = (size_t)h->nylm * h->n;
  if (nn == 0) return DDX_OK;
  hipLaunchKernelGGL(k_cf_scale, dim3((nn + 255) / 256), dim3(256), 0, s, nn, h->nylm, h->cf.p, x,
                     xs);
  DDX_HIP(hipGetLastError());
  return DDX_OK;
}

int seg_sum(ddx_handle *h, hipStream_t s, const double *yp, double *y, const DiisState *gate) {
  size_t nn = (size_t)h->nylm * h->n;
  if (nn == 0) return DDX_OK;
  hipLaunchKernelGGL(k_seg_sum, dim3((nn + 255) / 256), dim3(256), 0, s, h->n, h->nylm,
                     h->segoff.p, yp, y, gate);
  DDX_HIP(hipGetLastError());
  return DDX_OK;
}

// The applies below run in the lane's precision: ln.f32 selects the FP32
// sweeps, gather and MFMA products of the mixed precision.
int apply_lx(ddx_handle *h, Lane &ln, const double *x, double *y, const DiisState *gate,
             bool xs_ready, int ysplit) {
  DDX_TRY(reserve_lx(h, ln));
  return ln.f32 ? lx_r<float>(h, ln, x, y, gate, xs_ready, ysplit)
                : lx_r<double>(h, ln, x, y, gate, xs_ready, ysplit);
}

int apply_lstarx(ddx_handle *h, Lane &ln, const double *x, double *y, const DiisState *gate,
                 bool want_y) {
  DDX_TRY(reserve_lstarx(h, ln));
  return ln.f32 ? lstarx_r<float>(h, ln, x, y, gate, want_y)
                : lstarx_r<double>(h, ln, x, y, gate, want_y);
}

int apply_pair(ddx_handle *h, Lane &ld, double *yd, Lane &la, const double *xa, int ysplit) {
  DDX_TRY(reserve_lx(h, ld));
  DDX_TRY(reserve_lstarx(h, la));
  const DiisState *gd = solve_gate(h, ld), *ga = solve_gate(h, la);
  return ld.f32 ? pair_r<float>(h, ld, yd, gd, la, xa, ga, ysplit)
                : pair_r<double>(h, ld, yd, gd, la, xa, ga, ysplit);
}

// A (n, (P+1)^2) of the far charges of every sphere (k_p2l); cfP: the cf
// factors to order P
int fmm_p2l(ddx_handle *h, int P, double rho, const double *q, const double *cfP, double *A) {
  if (h->n == 0) return DDX_OK;
  const int *inst = h->ninst > 1 ? h->inst.p : nullptr;
  const int *soff = h->ninst > 1 ? h->soff.p : nullptr;
  hipStream_t s = h->stream;
  switch (P) {
    case 8:
      hipLaunchKernelGGL(k_p2l<8>, dim3(h->n), dim3(kWave), 0, s, h->n, h->sph.p, q, inst, soff,
                         rho, cfP, A);
      break;
    case 12:
      hipLaunchKernelGGL(k_p2l<12>, dim3(h->n), dim3(kWave), 0, s, h->n, h->sph.p, q, inst,
                         soff, rho, cfP, A);
      break;
    case 16:
      hipLaunchKernelGGL(k_p2l<16>, dim3(h->n), dim3(kWave), 0, s, h->n, h->sph.p, q, inst,
                         soff, rho, cfP, A);
      break;
    default:
      set_error("far-field order %d not built (8, 12, 16)", P);
      return DDX_ERR_ARG;
  }
  DDX_HIP(hipGetLastError());
  return DDX_OK;
}

}  // namespace ddx
