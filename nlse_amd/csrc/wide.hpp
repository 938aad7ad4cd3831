// Complex128 fields: the split step with FP64 storage and FP64 arithmetic.
//
// The reference keeps the precision of E_in: a complex128 field is
// propagated in complex128 (nlse.py:531-534; _prepare_output_array
// allocates A with E_in's dtype, nlse.py:271-273), i.e. double-precision
// FFTs, complex128 elementwise kernels and a float64 |A|^2.  The tables it
// multiplies with keep their own precision: the 2-D propagator is complex64
// (nlse.py:194-197), the potential term k/2*V is computed in V's dtype
// (nlse.py:425; float32 for a float32 V), the drive product in complex64
// (ddgpe.py:155-156).  These kernels reproduce that: every table value is
// rounded the way the reference rounds it, everything else is FP64.
//
// Same structure as the complex64 engine: a Stockham transform of a line held
// as a natural set v[m] = x[t + m*T] in registers, FP64 butterflies
// (fft_line.hpp) with double2 storage and a double2 LDS exchange, fused
// into row sweeps (I_x, N, F_x) and column sweeps (F_y, P, I_y).  The
// nonlocal response is a direct FP64 "same" convolution of |A|^2 with the
// kernel, as oaconvolve computes it on float64 data (nlse.py:406-409).
#pragma once
#include "fft_line.hpp"
#include "step_ops.hpp"

namespace nlse {

// LDS line of N double2 with one double2 of padding every 8 entries.
constexpr int WPADSH = 3;
template <int N>
struct WLine {
  static constexpr int SIZE = LdsLine<N, WPADSH, 0>::SIZE;
};

// Forward or unnormalised inverse DFT of G lines: the factored FP64 butterflies
// of fft_line.hpp with FP64 exchanges.
template <int N, int P, int G, bool INV, int SYNC, bool KEEP>
__device__ __forceinline__ void wfft_line(double2 (&v)[G][P], int t, const Twid<N, P, KEEP>& W, const Buf& tw,
                                          double2* lds) {
  fft_line_io<N, P, G, INV, G, WPADSH, F64X, SYNC>(v, v, t, W, tw, lds, WLine<N>::SIZE);
}

// ------------------------------------------------------------ pointwise
// Device records of one nonlinear application (from nlse_nl1 / nlse_nl2):
// the dz-scaled coefficients as given, and for the potential term the step
// `dzv` and the multiplier `vmul` separately, so that V' = vmul*V can be
// rounded in V's own precision as the reference's k/2*V array is.  vmul = 0
// means V enters as given (dzv then carries the whole multiplier).
struct WNL1 {
  double adz, gdz, inv_isat, dzv;
  double adz_i, gdz_i, dzv_i;
  double vmul;
  int cplx;
  int pad_;
};
struct WNL2 {
  double adz, gs_dz, gc_dz, inv_is_s, inv_is_o, dzv;
  double adz_i, gs_dz_i, gc_dz_i, dzv_i;
  double vmul;
  int cplx;
  int pad_;
};
// Rabi rotation in FP64: c - 1 and s, complex for a complex dz.
struct WRabi {
  double cm1, sn, cm1_i, sn_i;
};

// V kinds of the complex128 engine: the complex64 engine's two plus float64
// and complex128 potentials.
enum : int { V_REAL64 = 3, V_CPLX128 = 4 };

// V' = vmul * V in V's precision (float32 V: fl32(fl32(vmul) * V), the value
// numpy/cupy give k/2*V for a float32 array; complex64 V: the same per part,
// which is exact complex64 scaling by a real), returned as FP64 (re, im).
__device__ __forceinline__ double2 wvprime(const void* V, int vkind, int64_t idx, double vmul) {
  if (vkind == V_CPLX) {
    const float2 w = reinterpret_cast<const float2*>(V)[idx];
    if (vmul == 0.0) return make_double2((double)w.x, (double)w.y);
    const float m = (float)vmul;
    return make_double2((double)(m * w.x), (double)(m * w.y));
  }
  if (vkind == V_REAL64) {
    const double x = reinterpret_cast<const double*>(V)[idx];
    return make_double2(vmul != 0.0 ? vmul * x : x, 0.0);
  }
  if (vkind == V_CPLX128) {
    const double2 w = reinterpret_cast<const double2*>(V)[idx];
    return vmul != 0.0 ? make_double2(vmul * w.x, vmul * w.y) : w;
  }
  return make_double2(0.0, 0.0);
}

// V' of the P points idx + m * step, the kind tested once; a float32 potential
// is given in vf (loaded beside the field).
template <int P>
__device__ __forceinline__ void wvprime_set(double (&vr)[P], double (&vi)[P], const float (&vf)[P], const void* V,
                                            int vkind, int64_t idx, int step, double vmul) {
#pragma unroll
  for (int m = 0; m < P; ++m) {
    vr[m] = vmul != 0.0 ? (double)((float)vmul * vf[m]) : (double)vf[m];
    vi[m] = 0.0;
  }
  auto each = [&](int kind) {
#pragma unroll
    for (int m = 0; m < P; ++m) {
      const double2 w = wvprime(V, kind, idx + m * step, vmul);
      vr[m] = w.x;
      vi[m] = w.y;
    }
  };
  if (vkind == V_CPLX) each(V_CPLX);
  else if (vkind == V_REAL64) each(V_REAL64);
  else if (vkind == V_CPLX128) each(V_CPLX128);
}

// A *= exp(-a + i th) for n points {Re A, Im A, a, th} in private memory as
// A + A (f - 1) with f - 1 = expm1(-a) cos(th) - 2 sin^2(th/2) + i e^{-a}
// sin(th), by the library functions: arguments outside the series' ranges.
typedef __attribute__((address_space(5))) double private_double;
__device__ __noinline__ inline void wphase_lib(private_double* p, int n) {
  for (int m = 0; m < n; ++m) {
    private_double* q = p + 4 * m;
    const double ax = q[0], ay = q[1];
    double s2, c2;
    sincos(0.5 * q[3], &s2, &c2);
    const double em = expm1(-q[2]);
    const double cosm1 = -2.0 * s2 * s2;
    const double dr = fma(em, 1.0 + cosm1, cosm1);
    const double di = (1.0 + em) * (2.0 * s2 * c2);
    q[0] = ax + fma(ax, dr, -ay * di);
    q[1] = ay + fma(ay, dr, ax * di);
  }
}

// e^x - 1 for |x| <= 1/8: Taylor series to x^12 (next term 3e-21 relative).
__device__ __forceinline__ double wexpm1_small(double x) {
  double p = 1.0 / 479001600.0;
  p = fma(x, p, 1.0 / 39916800.0);
  p = fma(x, p, 1.0 / 3628800.0);
  p = fma(x, p, 1.0 / 362880.0);
  p = fma(x, p, 1.0 / 40320.0);
  p = fma(x, p, 1.0 / 5040.0);
  p = fma(x, p, 1.0 / 720.0);
  p = fma(x, p, 1.0 / 120.0);
  p = fma(x, p, 1.0 / 24.0);
  p = fma(x, p, 1.0 / 6.0);
  p = fma(x, p, 0.5);
  return fma(x * x, p, x);
}

// sin and cos for |x| <= pi/4: Taylor series to x^17 and x^18 (next terms 1e-19
// and 3e-21 relative).
__device__ __forceinline__ void wsincos_small(double x, double& s, double& c) {
  const double z = x * x;
  double p = 1.0 / 355687428096000.0;
  p = fma(z, p, -1.0 / 1307674368000.0);
  p = fma(z, p, 1.0 / 6227020800.0);
  p = fma(z, p, -1.0 / 39916800.0);
  p = fma(z, p, 1.0 / 362880.0);
  p = fma(z, p, -1.0 / 5040.0);
  p = fma(z, p, 1.0 / 120.0);
  p = fma(z, p, -1.0 / 6.0);
  s = fma(x * z, p, x);
  double q = -1.0 / 6402373705728000.0;
  q = fma(z, q, 1.0 / 20922789888000.0);
  q = fma(z, q, -1.0 / 87178291200.0);
  q = fma(z, q, 1.0 / 479001600.0);
  q = fma(z, q, -1.0 / 3628800.0);
  q = fma(z, q, 1.0 / 40320.0);
  q = fma(z, q, -1.0 / 720.0);
  q = fma(z, q, 1.0 / 24.0);
  q = fma(z, q, -0.5);
  c = fma(z, q, 1.0);
}

// The same on P points with one choice of the evaluation for the wave: the
// series for phases up to 2^16 (reduced by multiples of pi where one of the wave
// passes pi/2) and losses up to 1/8: about 45 operations a point, 35 where one
// loss serves all points, against some 250 of the library functions.
template <int P>
__device__ __forceinline__ void wapply(double2 (&A)[P], const double (&a)[P], bool one_loss, const double (&th)[P]) {
  bool small = true, series = true;
#pragma unroll
  for (int m = 0; m < P; ++m) {
    small = small && fabs(th[m]) <= 1.5707963267948966;
    series = series && fabs(th[m]) <= 65536.0 && fabs(a[m]) <= 0.125;
  }
  if (wave_all(series)) {
    const bool reduce = !wave_all(small);
    double em = wexpm1_small(-a[0]);
#pragma unroll
    for (int m = 0; m < P; ++m) {
      if (m > 0 && !one_loss) em = wexpm1_small(-a[m]);
      // half phase h = n pi/2 + r: sin^2 h and sin h cos h are sin^2 r and
      // sin r cos r for even n, cos^2 r and -sin r cos r for odd n
      double h = 0.5 * th[m], s2, c2;
      bool odd = false;
      if (reduce) {
        const double n = rint(h * 0.63661977236758138);
        h = fma(-n, 6.123233995736766e-17, fma(-n, 1.5707963267948966, h));
        odd = ((int)n & 1) != 0;
      }
      wsincos_small(h, s2, c2);
      const double q = odd ? c2 : s2, r = odd ? -s2 : c2;
      const double cosm1 = -2.0 * q * q;
      const double dr = fma(em, 1.0 + cosm1, cosm1);
      const double di = (1.0 + em) * (2.0 * q * r);
      A[m] = make_double2(A[m].x + fma(A[m].x, dr, -A[m].y * di), A[m].y + fma(A[m].y, dr, A[m].x * di));
    }
  } else {
    double pts[4 * P];
#pragma unroll
    for (int m = 0; m < P; ++m) {
      pts[4 * m] = A[m].x;
      pts[4 * m + 1] = A[m].y;
      pts[4 * m + 2] = a[m];
      pts[4 * m + 3] = th[m];
    }
    wphase_lib((private_double*)pts, P);
#pragma unroll
    for (int m = 0; m < P; ++m) A[m] = make_double2(pts[4 * m], pts[4 * m + 1]);
  }
}

// nl_prop / nl_prop_without_V on P points of a complex128 field
// (kernels_gpu.py:4-65 / kernels_cpu.py:5-63 in complex128): intensity I
// (|A|^2, or the convolved intensity of a nonlocal response), V' of the points.
template <int P>
__device__ __forceinline__ void wnl1(double2 (&A)[P], const double (&I)[P], const WNL1& p, bool loss_sat,
                                     const double (&vr)[P], const double (&vi)[P], bool has_vi) {
  double a[P], th[P];
  const bool sats = wave_any(p.inv_isat != 0.0), cplx = wave_any(p.cplx != 0);
#pragma unroll
  for (int m = 0; m < P; ++m) {
    const double sat = sats ? 1.0 / fma(I[m], p.inv_isat, 1.0) : 1.0;
    const double s = loss_sat ? sat : 1.0;
    a[m] = fma(p.adz, s, fma(p.dzv, vi[m], 0.0));
    th[m] = fma(p.gdz * I[m], sat, p.dzv * vr[m]);
    if (cplx) {
      a[m] = fma(p.gdz_i * I[m], sat, fma(p.dzv_i, vr[m], a[m]));
      th[m] -= fma(p.dzv_i, vi[m], p.adz_i * s);
    }
  }
  wapply<P>(A, a, !(cplx || has_vi || (loss_sat && sats)), th);
}

// nl_prop_c for one component (kernels_cpu.py:66-141) from the shared
// intensity snapshot (Is: own component, Io: the other).
template <int P>
__device__ __forceinline__ void wnl2(double2 (&A)[P], const double (&Is)[P], const double (&Io)[P], const WNL2& p,
                                     const double (&vr)[P], const double (&vi)[P], bool has_vi) {
  double a[P], th[P];
  const bool sats = wave_any(p.inv_is_s != 0.0 || p.inv_is_o != 0.0), cplx = wave_any(p.cplx != 0);
#pragma unroll
  for (int m = 0; m < P; ++m) {
    const double sat = sats ? 1.0 / fma(Io[m], p.inv_is_o, fma(Is[m], p.inv_is_s, 1.0)) : 1.0;
    a[m] = fma(p.adz, sat, p.dzv * vi[m]);
    th[m] = fma(p.gs_dz * Is[m], sat, fma(p.gc_dz * Io[m], sat, p.dzv * vr[m]));
    if (cplx) {
      a[m] = fma(p.gs_dz_i * Is[m], sat, fma(p.gc_dz_i * Io[m], sat, fma(p.dzv_i, vr[m], a[m])));
      th[m] -= fma(p.dzv_i, vi[m], p.adz_i * sat);
    }
  }
  wapply<P>(A, a, !(cplx || has_vi || sats), th);
}

__device__ __forceinline__ void wrabi(double2& A1, double2& A2, const WRabi& r) {
  const double2 a1 = A1, a2 = A2;
  A1 = make_double2(a1.x + fma(r.cm1, a1.x, fma(-r.cm1_i, a1.y, fma(r.sn, a2.y, r.sn_i * a2.x))),
                    a1.y + fma(r.cm1, a1.y, fma(r.cm1_i, a1.x, fma(-r.sn, a2.x, r.sn_i * a2.y))));
  A2 = make_double2(a2.x + fma(r.cm1, a2.x, fma(-r.cm1_i, a2.y, fma(r.sn, a1.y, r.sn_i * a1.x))),
                    a2.y + fma(r.cm1, a2.y, fma(r.cm1_i, a2.x, fma(-r.sn, a1.x, r.sn_i * a1.y))));
}

// One drive term of ddgpe.py:155-156 for a complex128 field: the product
// F_r * F_t * dz * 1j is formed in complex64 (both profiles are complex64
// arrays, dz a Python float), each product rounded as numpy rounds it,
// then subtracted in FP64.
__device__ __forceinline__ double2 wdrive(double2 A, float2 fr, float2 ft, float dz) {
#pragma clang fp contract(off)
  const float qx = fr.x * ft.x - fr.y * ft.y;
  const float qy = fr.x * ft.y + fr.y * ft.x;
  const float sx = qx * dz, sy = qy * dz;
  // (sx + i sy) * 1j = -sy + i sx
  return make_double2(A.x + (double)sy, A.y - (double)sx);
}

// Propagator kinds (shared with the complex64 engine): the complex64 value
// P of the reference table, promoted to FP64 and scaled by `scale` (a power
// of two: exact), multiplies the FP64 field.
__device__ __forceinline__ double2 wcmul(double2 a, double2 b) {
  return make_double2(fma(a.x, b.x, -a.y * b.y), fma(a.x, b.y, a.y * b.x));
}

// ------------------------------------------------------------- row sweep
struct WRowArgs {
  double2* A;
  int64_t ngroups;        // rows (G=1) or row pairs (G=2)
  int64_t rows_per_item;  // rows per item and component
  const double2* tw;
  int inverse_first;
  int forward_last;
  int has_a;
  int has_rabi;
  int has_drive;
  int has_b;
  int loss_sat;
  int write_I;            // store the field and |A|^2 (FP64) after I_x, nothing else
  const void* nlp_a;      // WNL1[items] or WNL2[items*2]
  const void* nlp_b;
  const WRabi* rabi;      // [items]
  const void* V;
  int vkind;
  int64_t v_item_stride;
  double* I;              // |A|^2 written by write_I (layout of A)
  const double* Ic;       // intensity used by the nonlinear step (null: |A|^2)
  const float2* drv_r0;
  const float2* drv_r1;
  float2 drv_t0;
  float2 drv_t1;
  float drv_dz;
  double out_scale;
};

// Two waves per SIMD of 1024^2 points load, transform and store in step, so a
// sweep is the sum of its memory time (5 us), VALU (5 us) and exchanges (3 us)
// and launch, not their maximum: 18.8 us.  Series instead of library functions
// and the factored butterflies took a 2-D step from 43.3 to 37.6 us (2048^2: 118.7
// to 87.5, 256^2: 16.3 to 12.0); 4 points per lane (121 us at 2048^2) and kept
// twiddles at 1024 points did not help.
// Rows of length N (x rows of 2-D fields, t rows of 3-D fields): LPB line
// groups per block, G components per group.  Dynamic LDS: LPB*G lines.
template <int N, int P, int LPB, int G>
__global__ __launch_bounds__(LPB*(N / P)) void k_wrow(WRowArgs a) {
  extern __shared__ double2 wsm[];
  constexpr int T = N / P;
  constexpr int LINE = WLine<N>::SIZE;
  const int li = threadIdx.x / T;
  const int t = threadIdx.x % T;
  const int64_t gi = (int64_t)blockIdx.x * LPB + li;
  const bool active = gi < a.ngroups;
  const int64_t gsafe = active ? gi : 0;
  const int64_t item = gsafe / a.rows_per_item;
  const int64_t y = gsafe - item * a.rows_per_item;
  int64_t off[G];
  if constexpr (G == 1) {
    off[0] = gsafe * N;
  } else {
    off[0] = ((item * 2) * a.rows_per_item + y) * N;
    off[1] = off[0] + a.rows_per_item * N;
  }
  double2* lline = wsm + li * G * LINE;
  constexpr int SYNC = T <= 64 ? SYNC_WAVE : SYNC_BLOCK;
  constexpr bool KEEP = false;  // kept, they take 40 more VGPRs for 2 % at 256^2 and nothing beyond

  double2 v[G][P];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int m = 0; m < P; ++m) v[g][m] = active ? a.A[off[g] + t + m * T] : make_double2(0.0, 0.0);
  const Buf tw(a.tw);
  const Twid<N, P, KEEP> W = load_twiddles<N, P, KEEP>(tw, t);
  // a float32 potential is loaded beside the field
  const int64_t vbase = item * a.v_item_stride + y * N + t;
  const bool v_early = a.vkind == V_REAL && (a.has_a || a.has_b);
  float vf[P];
#pragma unroll
  for (int m = 0; m < P; ++m) vf[m] = v_early ? reinterpret_cast<const float*>(a.V)[vbase + m * T] : 0.f;

  auto put = [&]() __attribute__((always_inline)) {
    if (!active) return;
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int m = 0; m < P; ++m) a.A[off[g] + t + m * T] = v[g][m];
  };

  if (a.inverse_first) wfft_line<N, P, G, true, SYNC>(v, t, W, tw, lline);

  if (a.write_I) {
    put();
    if (active) {
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int m = 0; m < P; ++m) a.I[off[g] + t + m * T] = v[g][m].x * v[g][m].x + v[g][m].y * v[g][m].y;
    }
    return;
  }

  // nonlinear application with the records `nlp`: intensities from the
  // convolved buffer (nonlocal response) or |A|^2, V' rounded per record
  const bool has_vi = a.vkind == V_CPLX || a.vkind == V_CPLX128;
  auto nl_pass = [&](const void* nlp, bool use_ic) __attribute__((always_inline)) {
    double I[G][P], vr[P], vi[P];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int m = 0; m < P; ++m) I[g][m] = v[g][m].x * v[g][m].x + v[g][m].y * v[g][m].y;
    if (use_ic) {
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int m = 0; m < P; ++m) I[g][m] = a.Ic[off[g] + t + m * T];
    }
    if constexpr (G == 1) {
      const WNL1 p = reinterpret_cast<const WNL1*>(nlp)[item];
      wvprime_set<P>(vr, vi, vf, a.V, a.vkind, vbase, T, p.vmul);
      wnl1<P>(v[0], I[0], p, a.loss_sat != 0, vr, vi, has_vi);
    } else {
      const WNL2* pp = reinterpret_cast<const WNL2*>(nlp) + 2 * item;
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const WNL2 p = pp[g];
        wvprime_set<P>(vr, vi, vf, a.V, a.vkind, vbase, T, p.vmul);
        wnl2<P>(v[g], I[g], I[1 - g], p, vr, vi, has_vi);
      }
    }
  };
  if (a.has_a) {
    nl_pass(a.nlp_a, a.Ic != nullptr);
    if constexpr (G == 2) {
      if (a.has_rabi) {
        const WRabi rb = a.rabi[item];
#pragma unroll
        for (int m = 0; m < P; ++m) wrabi(v[0][m], v[1][m], rb);
      }
    }
  }
  if constexpr (G == 2) {
    if (a.has_drive) {
#pragma unroll
      for (int m = 0; m < P; ++m) {
        const int64_t ri = y * N + t + m * T;
        v[1][m] = wdrive(v[1][m], a.drv_r0[ri], a.drv_t0, a.drv_dz);
        v[1][m] = wdrive(v[1][m], a.drv_r1[ri], a.drv_t1, a.drv_dz);
      }
    }
  }
  // the second application (start of the next Strang step) always sees |A|^2
  if (a.has_b) nl_pass(a.nlp_b, false);

  if (a.forward_last) wfft_line<N, P, G, false, SYNC>(v, t, W, tw, lline);

  if (a.out_scale != 1.0) {
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int m = 0; m < P; ++m) v[g][m] = make_double2(v[g][m].x * a.out_scale, v[g][m].y * a.out_scale);
  }
  put();
}

// ---------------------------------------------------------- column sweep
struct WColArgs {
  double2* A;
  int64_t nslabs;
  int64_t NX;          // columns per slab (the row stride, in elements)
  int ncomp;           // propagator component = slab % ncomp
  const double2* tw;
  int do_fwd, do_prop, do_inv;
  int pkind;           // PROP_SEP64, PROP_C64, PROP_SEP3D or PROP_C128
  const double2* px;   // [ncomp][nx]
  const double2* py;   // [ncomp][ny]
  const float2* ptab;  // [ncomp][ny][nx]
  const double2* pt;   // [nt]
  const double2* ptab128;  // [ny][NX]
  int nt;
  double scale;
  double out_scale;
};

// Columns of length N: WT adjacent columns per block, one per thread column.
template <int N, int P, int WT>
__global__ __launch_bounds__(WT*(N / P)) void k_wcol(WColArgs a) {
  extern __shared__ double2 wsm[];
  constexpr int T = N / P;
  constexpr int LINE = ColLine<N, WT, double2>::SIZE;
  const int cw = threadIdx.x % WT;
  const int t = threadIdx.x / WT;
  const int64_t tiles = a.NX / WT;
  // XCD-aware order: blocks are dispatched to the 8 XCDs in turn, so block b
  // takes tile (b mod 8) * (nblocks / 8) + b / 8 and the neighbouring tiles
  // that share a 128-byte row segment run on one XCD (one L2 fill)
  const int64_t nblk = (int64_t)gridDim.x, bx = (int64_t)blockIdx.x;
  const int64_t tb = (nblk % 8 == 0) ? (bx % 8) * (nblk / 8) + bx / 8 : bx;
  const int64_t slab = tb / tiles;
  const int64_t c0 = (tb % tiles) * WT + cw;
  const int64_t base = slab * (int64_t)N * a.NX + c0;
  double2* lline = wsm + cw * LINE;

  double2 v[1][P];
#pragma unroll
  for (int m = 0; m < P; ++m) v[0][m] = a.A[base + (int64_t)(t + m * T) * a.NX];

  const Buf tw(a.tw);
  const Twid<N, P, false> W = load_twiddles<N, P, false>(tw, t);

  if (a.do_fwd) wfft_line<N, P, 1, false, SYNC_BLOCK>(v, t, W, tw, lline);
  if (a.do_prop) {
    const int comp = (int)(slab % a.ncomp);
    if (a.pkind == PROP_SEP64) {
      const double2 px = a.px[comp * a.NX + c0];
#pragma unroll
      for (int m = 0; m < P; ++m) {
        const double2 py = a.py[comp * N + t + m * T];
        // the complex64 value of the reference's table (nlse.py:194-197)
        const float pr = (float)fma(px.x, py.x, -px.y * py.y);
        const float pi = (float)fma(px.x, py.y, px.y * py.x);
        v[0][m] = wcmul(v[0][m], make_double2((double)pr * a.scale, (double)pi * a.scale));
      }
    } else if (a.pkind == PROP_C64) {
      const float2* pt = a.ptab + (int64_t)comp * N * a.NX + c0;
#pragma unroll
      for (int m = 0; m < P; ++m) {
        const float2 q = pt[(int64_t)(t + m * T) * a.NX];
        v[0][m] = wcmul(v[0][m], make_double2((double)q.x * a.scale, (double)q.y * a.scale));
      }
    } else if (a.pkind == PROP_SEP3D) {
      const double2 px = a.px[c0 / a.nt];
      const double2 ptt = a.pt[c0 % a.nt];
#pragma unroll
      for (int m = 0; m < P; ++m) {
        const double2 py = a.py[t + m * T];
        // complex64 2-D part times the complex128 temporal factor (nlse_3d.py:105-114)
        const double p2r = (double)(float)fma(px.x, py.x, -px.y * py.y);
        const double p2i = (double)(float)fma(px.x, py.y, px.y * py.x);
        const double2 pp = make_double2(fma(p2r, ptt.x, -p2i * ptt.y) * a.scale, fma(p2r, ptt.y, p2i * ptt.x) * a.scale);
        v[0][m] = wcmul(v[0][m], pp);
      }
    } else if (a.pkind == PROP_C128) {
#pragma unroll
      for (int m = 0; m < P; ++m) {
        const double2 q = a.ptab128[(int64_t)(t + m * T) * a.NX + c0];
        v[0][m] = wcmul(v[0][m], make_double2(q.x * a.scale, q.y * a.scale));
      }
    }
  }
  if (a.do_inv) wfft_line<N, P, 1, true, SYNC_BLOCK>(v, t, W, tw, lline);
  if (a.out_scale != 1.0) {
#pragma unroll
    for (int m = 0; m < P; ++m) v[0][m] = make_double2(v[0][m].x * a.out_scale, v[0][m].y * a.out_scale);
  }
#pragma unroll
  for (int m = 0; m < P; ++m) a.A[base + (int64_t)(t + m * T) * a.NX] = v[0][m];
}

// ------------------------------------------------- nonlocal response (2-D)
// Ic = oaconvolve(I, K, mode="same") per slab, zero padding, FP64:
//   Ic(y, x) = sum_{a,b} K[a][b] I(y + rh - a, x + rw - b),  kh = 2 rh + 1, kw = 2 rw + 1.
// Blocks of WCONV_TILE^2 outputs stage the tile and its halo in LDS when it
// fits (WConvArgs::lds); otherwise they read I through the caches.
constexpr int WCONV_TILE = 16;
struct WConvArgs {
  const double* I;
  double* Ic;
  int64_t nslabs;
  int ny, nx;
  const double* K;  // [kh][kw]
  int kh, kw;
  int lds;          // 1: halo tile in LDS
  // matrix-core form (k_wconv2d_mfma): the kernel flipped in both axes,
  // each row with 16 zeros in front, [kh][kpw]; null: the direct form
  const double* KP;
  int kpw;
  int pair;         // 1: K even in y (rows u and kh-1-u share one product)
};
// chunks of 4 staged columns of the matrix-core form for half-width rw
// (16 + 2 rw rounded up to an even number of chunks), and its largest
inline int wconv_mfma_chunks(int rw) { return (16 + 2 * rw + 7) / 8 * 2; }
constexpr int WCONV_MFMA_MAX_CHUNKS = 12;

// ------------------------------------------------------------------ 1-D
struct WLine1DArgs {
  double2* A;
  int64_t ngroups;
  const double2* tw;
  const double2* prop;    // [ncomp][N] complex128 propagator
  double scale;           // 1/N
  int64_t nsteps;
  int precision;
  int loss_sat;
  const void* nl_full;    // WNL1[items] / WNL2[items*2]
  const void* nl_pre;
  const void* nl_post;
  const WRabi* rabi;
  const void* V;
  int vkind;
  const double* nlk;      // nonlocal kernel [2*nlr+1] (null: local)
  int nlr;
};

// Whole 1-D runs (see k_line1d) on complex128 lines; dynamic LDS: LPB*G lines.
template <int N, int P, int LPB, int G>
__global__ __launch_bounds__(LPB*(N / P)) void k_wline1d(WLine1DArgs a) {
  extern __shared__ double2 wsm[];
  constexpr int T = N / P;
  constexpr int LINE = WLine<N>::SIZE;
  const int li = threadIdx.x / T;
  const int t = threadIdx.x % T;
  const int64_t gi = (int64_t)blockIdx.x * LPB + li;
  const bool active = gi < a.ngroups;
  const int64_t item = active ? gi : 0;
  int64_t off[G];
  off[0] = item * G * N;
  if constexpr (G == 2) off[1] = off[0] + N;
  double2* lline = wsm + li * G * LINE;

  double2 v[G][P];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int m = 0; m < P; ++m) v[g][m] = active ? a.A[off[g] + t + m * T] : make_double2(0.0, 0.0);
  double2 pr[G][P];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int m = 0; m < P; ++m) pr[g][m] = a.prop[g * N + t + m * T];

  constexpr int SYNC = T <= 64 ? SYNC_WAVE : SYNC_BLOCK;
  constexpr bool KEEP = G == 1 && twid_kept(N, P);  // two lines leave no registers for them
  const Buf tw(a.tw);
  const Twid<N, P, KEEP> W = load_twiddles<N, P, KEEP>(tw, t);
  const bool has_vi = a.vkind == V_CPLX || a.vkind == V_CPLX128;
  float vf[P];
#pragma unroll
  for (int m = 0; m < P; ++m) vf[m] = a.vkind == V_REAL ? reinterpret_cast<const float*>(a.V)[t + m * T] : 0.f;

  auto apply_nl = [&](const void* prm) __attribute__((always_inline)) {
    double I[G][P];
    if (a.nlk != nullptr) {
      // convolved intensities (nlse_1d.py:65-66 kernel), FP64
      double* ib = reinterpret_cast<double*>(lline);
      __syncthreads();
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int m = 0; m < P; ++m) ib[g * N + t + m * T] = v[g][m].x * v[g][m].x + v[g][m].y * v[g][m].y;
      __syncthreads();
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int m = 0; m < P; ++m) {
          const int x = t + m * T;
          const int j0 = x - a.nlr < 0 ? 0 : x - a.nlr;
          const int j1 = x + a.nlr > N - 1 ? N - 1 : x + a.nlr;
          double acc = 0.0;
          for (int j = j0; j <= j1; ++j) acc = fma(a.nlk[x - j + a.nlr], ib[g * N + j], acc);
          I[g][m] = acc;
        }
      __syncthreads();
    } else {
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int m = 0; m < P; ++m) I[g][m] = v[g][m].x * v[g][m].x + v[g][m].y * v[g][m].y;
    }
    double vr[P], vi[P];
    if constexpr (G == 1) {
      const WNL1 p = reinterpret_cast<const WNL1*>(prm)[item];
      wvprime_set<P>(vr, vi, vf, a.V, a.vkind, t, T, p.vmul);
      wnl1<P>(v[0], I[0], p, a.loss_sat != 0, vr, vi, has_vi);
    } else {
      const WNL2* pp = reinterpret_cast<const WNL2*>(prm) + 2 * item;
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const WNL2 p = pp[g];
        wvprime_set<P>(vr, vi, vf, a.V, a.vkind, t, T, p.vmul);
        wnl2<P>(v[g], I[g], I[1 - g], p, vr, vi, has_vi);
      }
    }
  };

  for (int64_t s = 0; s < a.nsteps; ++s) {
    if (a.precision == 1) apply_nl(a.nl_pre);
    wfft_line<N, P, G, false, SYNC>(v, t, W, tw, lline);
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int m = 0; m < P; ++m)
        v[g][m] = wcmul(v[g][m], make_double2(pr[g][m].x * a.scale, pr[g][m].y * a.scale));
    wfft_line<N, P, G, true, SYNC>(v, t, W, tw, lline);
    if (a.precision == 1) {
      apply_nl(a.nl_post);
    } else {
      apply_nl(a.nl_full);
      if constexpr (G == 2) {
        if (a.rabi != nullptr) {
          const WRabi rb = a.rabi[item];
#pragma unroll
          for (int m = 0; m < P; ++m) wrabi(v[0][m], v[1][m], rb);
        }
      }
    }
  }
  if (active) {
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int m = 0; m < P; ++m) a.A[off[g] + t + m * T] = v[g][m];
  }
}

// ---------------------------------------------- per-length dispatch table
struct WideOps {
  int (*twiddles)(const double2**);
  int (*row)(int G, const WRowArgs&, hipStream_t);
  int (*col)(const WColArgs&, hipStream_t);
  int (*line1d)(int G, const WLine1DArgs&, hipStream_t);
};

// Dispatch table of a line length (wide.hip), or null.
const WideOps* wide_ops(int64_t n);
int wide_conv2d(const WConvArgs& a, hipStream_t s);
// whether a kh x kw kernel takes the matrix-core form (chunks and LDS)
bool wide_conv2d_mfma_fits(int kh, int kw);

}  // namespace nlse
