// Pointwise operators of the split step (device side), shared by the fused
// line passes and the standalone operator kernels.
//
// Reference semantics: NLSE/kernels_cpu.py (numba, FP64 intermediates,
// one rounding at the store) and NLSE/kernels_gpu.py (saturated loss).
// The factor exp(dz*(-a + i theta)) is applied as A + A*(f - 1) with
//   f - 1 = expm1(-a)*cos(theta) - 2 sin^2(theta/2)
//         + i * exp(-a) * 2 sin(theta/2) cos(theta/2)
// so that f - 1 (small) carries full relative precision and the update
// rounds once at the magnitude of A.  A plain FP32 factor exp(-a) would
// carry a fixed rounding error (up to 3e-8) that a 1000-step run turns into
// a 3e-5 amplitude bias; the numba reference has no such bias.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_line.hpp"

namespace nlse {

// A complex step dz = dr + i di (imaginary-time evolution, nlse.py:505-508)
// turns exp(dz (-L + i Th)) into exp(-(dr L + di Th) + i (dr Th - di L)):
// the records hold every dz-scaled coefficient twice, scaled by dr and by
// di; `cplx` (wave-uniform) is nonzero only when di != 0, so real steps
// skip the second set.

// One nonlinear application, single component (nl_prop / nl_prop_without_V).
struct NLParams1 {
  float adz;       // dz * alpha'        (alpha' = alpha/2)
  float gdz;       // dz * g             (g = k/2 n2 c eps0)
  float inv_isat;  // 1 / Isat'          (Isat' = 2 I_sat/(eps0 c)); 0 for inf
  float vdz;       // dz, multiplier of V' (k/2 V)
  float adz_i = 0.f, gdz_i = 0.f, vdz_i = 0.f;  // the same scaled by Im(dz)
  int cplx = 0;
};

// One nonlinear application for one component of a two-component field
// (nl_prop_c / nl_prop_without_V_c, kernels_cpu.py:66-141).
struct NLParams2 {
  float adz;         // dz * alpha'
  float gs_dz;       // dz * g_self   (multiplies I_self * sat)
  float gc_dz;       // dz * g_cross  (multiplies I_other * sat)
  float inv_is_s;    // 1/Isat applied to I_self
  float inv_is_o;    // 1/Isat applied to I_other
  float vdz;         // dz * (multiplier of V for this component)
  float adz_i = 0.f, gs_dz_i = 0.f, gc_dz_i = 0.f, vdz_i = 0.f;  // scaled by Im(dz)
  int cplx = 0;
  int pad_ = 0;
};

// Rabi rotation A1' = c A1 - i s A2, A2' = c A2 - i s A1 with c - 1 and s
// precomputed in FP64 (kernels_cpu.py:144-161); complex for a complex dz.
struct RabiParams {
  float cm1;  // cos(omega dz) - 1
  float sn;   // sin(omega dz)
  float cm1_i = 0.f, sn_i = 0.f;  // imaginary parts
};

// sin and cos of h, |h| <= pi/4: polynomials of least largest error (6e-11 and
// 6e-12; each coefficient rounded to FP32 before the next ones were fitted, so
// that these make up for it).  With the Taylor coefficients the mean of |f|^2 - 1
// is -1.5e-9 at phases near pi/2, with these -1e-10.
__device__ __forceinline__ void sincos_small(float h, float& s, float& c) {
  const float x2 = h * h;
  float ps = fmaf(x2, 2.80394079e-6f, -1.98502734e-4f);
  ps = fmaf(x2, ps, 8.33337288e-3f);
  ps = fmaf(x2, ps, -1.66666672e-1f);
  s = fmaf(h * x2, ps, h);
  float pc = fmaf(x2, -2.89776466e-7f, 2.48229862e-5f);
  pc = fmaf(x2, pc, -1.38889824e-3f);
  pc = fmaf(x2, pc, 4.16666679e-2f);
  pc = fmaf(x2, pc, -0.5f);
  c = fmaf(x2, pc, 1.0f);
}

// q and r with sin^2 h = q^2 and sin h cos h = q r, |h| <= 2^15: h = n pi/2 + x
// in two FMAs (the first is exact), q = sin x and r = cos x for even n, q = cos x
// and r = -sin x for odd n.
__device__ __forceinline__ void sincos_reduced(float h, float& q, float& r) {
  const float n = rintf(h * 0.636619772f);
  const float x = fmaf(-n, -4.37113901e-8f, fmaf(-n, 1.57079637f, h));
  float s, c;
  sincos_small(x, s, c);
  const bool odd = ((int)n & 1) != 0;
  q = odd ? c : s;
  r = odd ? -s : c;
}

// expm1(x), |x| <= 1/8: Taylor series to x^7 (remainder 0.125^8/8! < 2e-12).
__device__ __forceinline__ float expm1_small(float x) {
  float p = fmaf(x, 1.98412698e-4f, 1.38888889e-3f);  // 1/7!, 1/6!
  p = fmaf(x, p, 8.33333333e-3f);                      // 1/5!
  p = fmaf(x, p, 4.16666667e-2f);                      // 1/4!
  p = fmaf(x, p, 1.66666667e-1f);                      // 1/3!
  p = fmaf(x, p, 0.5f);                                // 1/2!
  return fmaf(x * x, p, x);
}

// expm1(x), |x| <= 80: x = n ln 2 + y in two FMAs (the first is exact), 2^n
// (expm1(y) + 1) - 1 with the Taylor series of y to y^8 (remainder 0.35^9/9! =
// 2e-10).
__device__ __forceinline__ float expm1_reduced(float x) {
  const float n = rintf(x * 1.44269504f);
  const float y = fmaf(-n, -1.90465432e-9f, fmaf(-n, 0.693147182f, x));
  float p = fmaf(y, 2.48015873e-5f, 1.98412698e-4f);  // 1/8!, 1/7!
  p = fmaf(y, p, 1.38888889e-3f);
  p = fmaf(y, p, 8.33333333e-3f);
  p = fmaf(y, p, 4.16666667e-2f);
  p = fmaf(y, p, 1.66666667e-1f);
  p = fmaf(y, p, 0.5f);
  p = fmaf(y * y, p, y);
  const float e = ldexpf(1.0f, (int)n);
  return fmaf(e, p, e - 1.0f);
}

// Ranges of the reduced forms; beyond them (and for NaN) the library functions.
constexpr float PHASE_REDUCED = 65536.0f, LOSS_REDUCED = 80.0f;

// 1/d to ~1 ulp: hardware reciprocal and one Newton step; exact for d = 1.
__device__ __forceinline__ float recip(float d) {
  float r = __builtin_amdgcn_rcpf(d);
  return fmaf(r, fmaf(-d, r, 1.0f), r);
}

__device__ __forceinline__ bool wave_all(bool c) {
  return __builtin_amdgcn_read_exec() == __builtin_amdgcn_ballot_w64(c);
}
__device__ __forceinline__ bool wave_any(bool c) { return __builtin_amdgcn_ballot_w64(c) != 0; }

// A *= exp(-a + i th) for n points {Re A, Im A, a, th} in private memory with
// the library functions, for arguments outside the ranges of the forms above.
// Out of line and on a copy of the points: such phases of complex64 fields hold
// no digits, and a call amid the points would tie up the registers of the others.
typedef __attribute__((address_space(5))) float private_float;
__device__ __noinline__ void phase_loss_lib(private_float* p, int n) {
  for (int m = 0; m < n; ++m) {
    private_float* q = p + 4 * m;
    const float ax = q[0], ay = q[1];
    float s2, c2;
    const float em = expm1f(-q[2]);
    sincosf(0.5f * q[3], &s2, &c2);
    const float cm1 = -2.0f * s2 * s2;
    const float dr = fmaf(em, 1.0f + cm1, cm1);
    const float di = (1.0f + em) * (2.0f * s2 * c2);
    q[0] = ax + fmaf(ax, dr, -ay * di);
    q[1] = ay + fmaf(ay, dr, ax * di);
  }
}

// (a strided by `as`: 0 for one loss)
template <int P>
__device__ __forceinline__ void phase_loss_slow(float2* A, const float* a, int as, const float* th) {
  float pts[4 * P];
#pragma unroll
  for (int m = 0; m < P; ++m) {
    pts[4 * m] = A[m].x;
    pts[4 * m + 1] = A[m].y;
    pts[4 * m + 2] = a[m * as];
    pts[4 * m + 3] = th[m];
  }
  phase_loss_lib((private_float*)pts, P);
#pragma unroll
  for (int m = 0; m < P; ++m) A[m] = make_float2(pts[4 * m], pts[4 * m + 1]);
}

// A *= 1 + em + ..., the factor f = exp(-a + i theta) as A + A (f - 1), from em =
// expm1(-a) and q, r of the half phase.
__device__ __forceinline__ float2 apply_half_phase(float2 A, float em, float q, float r) {
  const float cosm1 = -2.0f * q * q;
  const float dr = fmaf(em, 1.0f + cosm1, cosm1);
  const float di = (1.0f + em) * (2.0f * q * r);
  const float cx = fmaf(A.x, dr, -A.y * di);
  const float cy = fmaf(A.y, dr, A.x * di);
  return make_float2(A.x + cx, A.y + cy);
}

// Apply exp(-a + i theta) to P points with one wave-uniform choice of the
// evaluation path for all of them.
template <int P>
__device__ __forceinline__ void apply_phase_loss_block(float2* A, const float* a, const float* theta) {
  bool small = true, reduced = true;
#pragma unroll
  for (int m = 0; m < P; ++m) {
    small = small && fabsf(0.5f * theta[m]) <= 0.78539816f && fabsf(a[m]) <= 0.125f;
    reduced = reduced && fabsf(theta[m]) <= PHASE_REDUCED && fabsf(a[m]) <= LOSS_REDUCED;
  }
  if (wave_all(small)) {
#pragma unroll
    for (int m = 0; m < P; ++m) {
      float s2, c2;
      sincos_small(0.5f * theta[m], s2, c2);
      A[m] = apply_half_phase(A[m], expm1_small(-a[m]), s2, c2);
    }
  } else if (wave_all(reduced)) {
#pragma unroll
    for (int m = 0; m < P; ++m) {
      float q, r;
      sincos_reduced(0.5f * theta[m], q, r);
      A[m] = apply_half_phase(A[m], expm1_reduced(-a[m]), q, r);
    }
  } else {
    phase_loss_slow<P>(A, a, 1, theta);
  }
}

__device__ __forceinline__ float2 apply_phase_loss(float2 A, float a, float theta) {
  apply_phase_loss_block<1>(&A, &a, &theta);
  return A;
}

// sin(x) and cos(x) - 1 for |x| <= 1/4: Taylor series to x^7 and x^8, 1/5! raised
// by 1e-7 and 1/6! by 2.3e-8: that cancels, over the range, the roundings of 1/3!
// and 1/4! to FP32 and the omitted x^9 and x^10 (remainders 1.1e-11 and 6e-13).
// The errors of the two enter |f|^2 - 1 with one sign at every step, so a run adds
// them up: at phases near 1/4 the mean of |f|^2 - 1 is 5e-12, as that of the
// half-angle form; -6.6e-10 with cosine terms to x^6 alone.
__device__ __forceinline__ void sincosm1_quarter(float x, float& s, float& cm1) {
  const float x2 = x * x;
  float ps = fmaf(x2, -1.98412698e-4f, 8.33343342e-3f);
  ps = fmaf(x2, ps, -1.66666667e-1f);
  s = fmaf(x * x2, ps, x);
  float pc = fmaf(x2, 2.48015873e-5f, -1.38891186e-3f);
  pc = fmaf(x2, pc, 4.16666667e-2f);
  pc = fmaf(x2, pc, -0.5f);
  cm1 = x2 * pc;
}

// A *= exp(-a + i th[m]) on P points with one loss `a` for all of them:
// e^{-a} - 1 is evaluated once, and steps of small phase (the wave's largest
// |th| <= 1/4) take the short series: about 18 operations per point against
// 38 of apply_phase_loss_block.  Phases past pi/2 and losses past 1/8 are reduced
// in registers.  By the library on a copy of the wave's points in private memory,
// 20 steps of 28 fields of 1024^2 with phases of 1.7 took 9.1 ms, and with the
// library inlined 7.8; now 5.4 (5.3 with small phases).  The power changed by up to
// 6e-8 a step, now 5e-11.
template <int P>
__device__ __forceinline__ void apply_phase_block(float2* A, float a, const float* th) {
  bool quarter = fabsf(a) <= 0.125f, half = quarter, reduced = fabsf(a) <= LOSS_REDUCED;
#pragma unroll
  for (int m = 0; m < P; ++m) {
    quarter = quarter && fabsf(th[m]) <= 0.25f;
    half = half && fabsf(th[m]) <= 1.5707963f;
    reduced = reduced && fabsf(th[m]) <= PHASE_REDUCED;
  }
  const float em = expm1_small(-a), e1 = 1.0f + em;
  if (wave_all(quarter)) {
#pragma unroll
    for (int m = 0; m < P; ++m) {
      float sn, cm1;
      sincosm1_quarter(th[m], sn, cm1);
      const float dr = fmaf(e1, cm1, em), di = e1 * sn;
      A[m] = make_float2(A[m].x + fmaf(A[m].x, dr, -A[m].y * di), A[m].y + fmaf(A[m].y, dr, A[m].x * di));
    }
  } else if (wave_all(half)) {
#pragma unroll
    for (int m = 0; m < P; ++m) {
      float s2, c2;
      sincos_small(0.5f * th[m], s2, c2);
      const float cm1 = -2.0f * s2 * s2;
      const float dr = fmaf(e1, cm1, em), di = e1 * (2.0f * s2 * c2);
      A[m] = make_float2(A[m].x + fmaf(A[m].x, dr, -A[m].y * di), A[m].y + fmaf(A[m].y, dr, A[m].x * di));
    }
  } else if (wave_all(reduced)) {
    const float emr = expm1_reduced(-a);
#pragma unroll
    for (int m = 0; m < P; ++m) {
      float q, r;
      sincos_reduced(0.5f * th[m], q, r);
      A[m] = apply_half_phase(A[m], emr, q, r);
    }
  } else {
    phase_loss_slow<P>(A, &a, 0, th);
  }
}

// nl_prop on P points with the intensity I given per point (|A|^2, or its
// convolution for the nonlocal response) and the potential vr + i vi (has_vi,
// uniform: a complex one).  GEN: instances that also take losses which vary
// from point to point (saturated loss, complex V, complex dz).
template <int P, bool GEN>
__device__ __forceinline__ void nl1_block_I(float2* A, const float* I, const struct NLParams1& p, bool loss_sat,
                                            bool has_vi, const float* vr, const float* vi) {
  float th[P];
  if (!GEN || !(loss_sat || has_vi || wave_any(p.cplx != 0))) {
#pragma unroll
    for (int m = 0; m < P; ++m) {
      const float sat = recip(fmaf(I[m], p.inv_isat, 1.0f));
      th[m] = fmaf(p.gdz * I[m], sat, p.vdz * vr[m]);
    }
    apply_phase_block<P>(A, p.adz, th);
  } else {
    float a[P];
#pragma unroll
    for (int m = 0; m < P; ++m) {
      const float sat = recip(fmaf(I[m], p.inv_isat, 1.0f));
      th[m] = fmaf(p.gdz * I[m], sat, p.vdz * vr[m]);
      a[m] = fmaf(p.vdz, vi[m], loss_sat ? p.adz * sat : p.adz);
      if (p.cplx) {
        a[m] = fmaf(p.gdz_i * I[m], sat, fmaf(p.vdz_i, vr[m], a[m]));
        th[m] -= fmaf(p.vdz_i, vi[m], loss_sat ? p.adz_i * sat : p.adz_i);
      }
    }
    apply_phase_loss_block<P>(A, a, th);
  }
}

// nl_prop on P points (see nl1), potential values given per point.
template <int P, bool GEN>
__device__ __forceinline__ void nl1_block(float2* A, const struct NLParams1& p, bool loss_sat, bool has_vi,
                                          const float* vr, const float* vi) {
  float I[P];
#pragma unroll
  for (int m = 0; m < P; ++m) I[m] = A[m].x * A[m].x + A[m].y * A[m].y;
  nl1_block_I<P, GEN>(A, I, p, loss_sat, has_vi, vr, vi);
}

// The imaginary-dz terms of one two-component application (see NLParams2).
__device__ __forceinline__ void nl2_imag(const NLParams2& p, float Is, float Io, float sat, float vr, float vi,
                                         float& a, float& th) {
  if (p.cplx) {
    a = fmaf(p.gs_dz_i * Is, sat, fmaf(p.gc_dz_i * Io, sat, fmaf(p.vdz_i, vr, a)));
    th -= fmaf(p.vdz_i, vi, p.adz_i * sat);
  }
}

// nl_prop_c for both components of P points from one intensity snapshot.
template <int P>
__device__ __forceinline__ void nl2_block(float2* A1, float2* A2, const struct NLParams2& p1,
                                          const struct NLParams2& p2, const float* vr, const float* vi) {
  float a1[P], t1[P], a2[P], t2[P];
#pragma unroll
  for (int m = 0; m < P; ++m) {
    const float I1 = A1[m].x * A1[m].x + A1[m].y * A1[m].y;
    const float I2 = A2[m].x * A2[m].x + A2[m].y * A2[m].y;
    const float s1 = recip(fmaf(I2, p1.inv_is_o, fmaf(I1, p1.inv_is_s, 1.0f)));
    const float s2 = recip(fmaf(I1, p2.inv_is_o, fmaf(I2, p2.inv_is_s, 1.0f)));
    t1[m] = fmaf(p1.gs_dz * I1, s1, fmaf(p1.gc_dz * I2, s1, p1.vdz * vr[m]));
    a1[m] = fmaf(p1.vdz, vi[m], p1.adz * s1);
    t2[m] = fmaf(p2.gs_dz * I2, s2, fmaf(p2.gc_dz * I1, s2, p2.vdz * vr[m]));
    a2[m] = fmaf(p2.vdz, vi[m], p2.adz * s2);
    nl2_imag(p1, I1, I2, s1, vr[m], vi[m], a1[m], t1[m]);
    nl2_imag(p2, I2, I1, s2, vr[m], vi[m], a2[m], t2[m]);
  }
  apply_phase_loss_block<P>(A1, a1, t1);
  apply_phase_loss_block<P>(A2, a2, t2);
}

template <int P>
__device__ __forceinline__ void nl2_block_I(float2* A1, float2* A2, const float* I1, const float* I2,
                                            const struct NLParams2& p1, const struct NLParams2& p2, const float* vr,
                                            const float* vi) {
  float a1[P], t1[P], a2[P], t2[P];
#pragma unroll
  for (int m = 0; m < P; ++m) {
    const float s1 = recip(fmaf(I2[m], p1.inv_is_o, fmaf(I1[m], p1.inv_is_s, 1.0f)));
    const float s2 = recip(fmaf(I1[m], p2.inv_is_o, fmaf(I2[m], p2.inv_is_s, 1.0f)));
    t1[m] = fmaf(p1.gs_dz * I1[m], s1, fmaf(p1.gc_dz * I2[m], s1, p1.vdz * vr[m]));
    a1[m] = fmaf(p1.vdz, vi[m], p1.adz * s1);
    t2[m] = fmaf(p2.gs_dz * I2[m], s2, fmaf(p2.gc_dz * I1[m], s2, p2.vdz * vr[m]));
    a2[m] = fmaf(p2.vdz, vi[m], p2.adz * s2);
    nl2_imag(p1, I1[m], I2[m], s1, vr[m], vi[m], a1[m], t1[m]);
    nl2_imag(p2, I2[m], I1[m], s2, vr[m], vi[m], a2[m], t2[m]);
  }
  apply_phase_loss_block<P>(A1, a1, t1);
  apply_phase_loss_block<P>(A2, a2, t2);
}

// V kinds
enum : int { V_NONE = 0, V_REAL = 1, V_CPLX = 2 };

__device__ __forceinline__ void load_v(const void* V, int vkind, int64_t idx, float& vr, float& vi) {
  vr = 0.f;
  vi = 0.f;
  if (vkind == V_REAL) {
    vr = reinterpret_cast<const float*>(V)[idx];
  } else if (vkind == V_CPLX) {
    float2 w = reinterpret_cast<const float2*>(V)[idx];
    vr = w.x;
    vi = w.y;
  }
}

// V at the P points base + d + m*T of a line (base uniform, d per lane; vr,
// vi zero without V).  The kind is tested once for the whole set: with a
// per-point test the compiler waits for each load at the branch join,
// serialising P load latencies.
template <int P, int T, bool CPLX = true>
__device__ __forceinline__ void load_v_set(const void* V, int vkind, int64_t base, uint32_t d, float* vr, float* vi) {
  if (vkind == V_REAL) {
    const Buf p(reinterpret_cast<const float*>(V) + base);
#pragma unroll
    for (int m = 0; m < P; ++m) {
      vr[m] = p.load<float>(4u * d, 4u * m * T);
      vi[m] = 0.f;
    }
  } else if (CPLX && vkind == V_CPLX) {
    const Buf p(reinterpret_cast<const float2*>(V) + base);
#pragma unroll
    for (int m = 0; m < P; ++m) {
      const float2 w = p.load<float2>(8u * d, 8u * m * T);
      vr[m] = w.x;
      vi[m] = w.y;
    }
  } else {
#pragma unroll
    for (int m = 0; m < P; ++m) {
      vr[m] = 0.f;
      vi[m] = 0.f;
    }
  }
}

// nl_prop: A *= exp(dz*(-alpha' [*sat] + i g I sat + i V'))
// A complex V' = vr + i vi contributes i*V' = -vi + i vr.
__device__ __forceinline__ float2 nl1(float2 A, const NLParams1& p, bool loss_sat, float vr, float vi) {
  const float I = A.x * A.x + A.y * A.y;
  const float sat = recip(fmaf(I, p.inv_isat, 1.0f));
  float theta = fmaf(p.gdz * I, sat, p.vdz * vr);
  float a = fmaf(p.vdz, vi, loss_sat ? p.adz * sat : p.adz);
  if (p.cplx) {
    a = fmaf(p.gdz_i * I, sat, fmaf(p.vdz_i, vr, a));
    theta -= fmaf(p.vdz_i, vi, loss_sat ? p.adz_i * sat : p.adz_i);
  }
  return apply_phase_loss(A, a, theta);
}

// nl_prop_c for one component from the shared intensity snapshot.
__device__ __forceinline__ float2 nl2(float2 A, float Is, float Io, const NLParams2& p, float vr, float vi) {
  const float sat = recip(fmaf(Io, p.inv_is_o, fmaf(Is, p.inv_is_s, 1.0f)));
  float theta = fmaf(p.gs_dz * Is, sat, fmaf(p.gc_dz * Io, sat, p.vdz * vr));
  float a = fmaf(p.vdz, vi, p.adz * sat);
  nl2_imag(p, Is, Io, sat, vr, vi, a, theta);
  return apply_phase_loss(A, a, theta);
}

__device__ __forceinline__ void rabi(float2& A1, float2& A2, const RabiParams& r) {
  // A1' = A1 + (c-1) A1 - i s A2 with complex c - 1 = cr + i ci and
  // s = sr + i si:  (c-1) A = (cr x - ci y) + i (cr y + ci x),
  // -i s B = (sr v + si u) - i (sr u - si v) for B = u + i v
  const float2 a1 = A1, a2 = A2;
  A1 = make_float2(a1.x + fmaf(r.cm1, a1.x, fmaf(-r.cm1_i, a1.y, fmaf(r.sn, a2.y, r.sn_i * a2.x))),
                   a1.y + fmaf(r.cm1, a1.y, fmaf(r.cm1_i, a1.x, fmaf(-r.sn, a2.x, r.sn_i * a2.y))));
  A2 = make_float2(a2.x + fmaf(r.cm1, a2.x, fmaf(-r.cm1_i, a2.y, fmaf(r.sn, a1.y, r.sn_i * a1.x))),
                   a2.y + fmaf(r.cm1, a2.y, fmaf(r.cm1_i, a2.x, fmaf(-r.sn, a1.x, r.sn_i * a1.y))));
}

// A_c64 * P where P is the complex64 rounding of the FP64 product px*py
// (the reference builds exp(-i(kx^2+ky^2) dz/2k) in FP64 and casts it to
// complex64, nlse.py:194-197); px carries the factor 1/N, an exact power of
// two.  The product is a complex64 one, as the reference's: its FP32 roundings
// are not free of bias (-2.8e-9 of the power per step in the speckle workload),
// and an FP64 product, nearer to the exact result, would leave the complex64
// reference by 5e-6 of the power over 2001 steps.
__device__ __forceinline__ float2 prop_sep_c64(float2 A, double2 px, double2 py) {
  const float pr = (float)fma(px.x, py.x, -px.y * py.y);
  const float pi = (float)fma(px.x, py.y, px.y * py.x);
  return make_float2(fmaf(A.x, pr, -A.y * pi), fmaf(A.x, pi, A.y * pr));
}

__device__ __forceinline__ float2 prop_c64(float2 A, float2 P, float scale) {
  P.x *= scale;
  P.y *= scale;
  return make_float2(fmaf(A.x, P.x, -A.y * P.y), fmaf(A.x, P.y, A.y * P.x));
}

// A times a complex128 propagator (numpy multiplies complex64 by complex128
// in complex128 and casts back, nlse_1d.py:104, nlse_3d.py:112).
__device__ __forceinline__ double2 prop_c128(double2 A, double2 P, double scale) {
  const double px = P.x * scale, py = P.y * scale;
  return make_double2(fma(A.x, px, -A.y * py), fma(A.x, py, A.y * px));
}

// 3-D propagator (nlse_3d.py:105-114): P = complex64(px*py) (the 2-D part,
// cast to complex64 by the reference) times the complex128 temporal factor
// pt (scaled by 1/N).
__device__ __forceinline__ double2 prop_sep3d(double2 A, double2 px, double2 py, double2 pt) {
  const double p2r = (double)(float)fma(px.x, py.x, -px.y * py.y);
  const double p2i = (double)(float)fma(px.x, py.y, px.y * py.x);
  const double pr = fma(p2r, pt.x, -p2i * pt.y);
  const double pi = fma(p2r, pt.y, p2i * pt.x);
  return make_double2(fma(A.x, pr, -A.y * pi), fma(A.x, pi, A.y * pr));
}

}  // namespace nlse
