/*
 * nlse_hip.h -- C ABI of the MI355X split-step engine (libnlse_hip.so).
 *
 * Drop-in boundary for the backend="GPU" side of Quantum-Optics-LKB/NLSE
 * v2.3.0.  The reference binds its GPU path in the `backend` property
 * setter (NLSE/nlse.py:162-186) to three things, each replaced here:
 *
 *   VkFFTApp(shape, dtype, ndim, stream, inplace=True, norm=1)
 *       nlse.py:207-218, executed at nlse.py:435-438
 *       -> nlse_fft_plan_create / nlse_fft_exec / nlse_fft_plan_destroy
 *   kernels_gpu.{square_mod, nl_prop, nl_prop_without_V, nl_prop_c,
 *       nl_prop_without_V_c, rabi_coupling}   NLSE/kernels_gpu.py:4-190
 *       -> nlse_square_mod, nlse_nl_prop, nlse_nl_prop_c, nlse_rabi_coupling,
 *          nlse_mul_propagator (the `A *= propagator` of nlse.py:437)
 *   the split_step / out_field loop            nlse.py:372-619
 *       -> nlse_plan_* + nlse_run: many fused split steps per call
 *   the power integrals of the normalisation and of callbacks.norm
 *       nlse.py:297-303, callbacks.py:54      -> nlse_sumsq (FP64)
 *
 * Conventions
 *   - Every entry point returns 0 on success and a negative code on error;
 *     nothing throws across the boundary.  nlse_last_error() returns the
 *     message of the last failure on the calling thread.
 *   - Pointers named `*_dev` are device pointers (hipMalloc'd or torch
 *     tensors' data_ptr()); everything else is host memory.
 *   - `stream` is a hipStream_t passed as void*; all work is asynchronous
 *     on that stream.  Objects are not thread-safe.
 *   - complex64 = interleaved float (re, im); complex128 = interleaved double.
 *   - Transform sizes must be powers of two, 8 <= n <= 4096.
 */
#ifndef NLSE_HIP_H
#define NLSE_HIP_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define NLSE_OK 0
#define NLSE_ERR_ARG (-1)     /* invalid argument / shape */
#define NLSE_ERR_HIP (-2)     /* HIP runtime error */
#define NLSE_ERR_STATE (-3)   /* object not ready (missing tables) */

int nlse_version(void);
const char* nlse_last_error(void);

/* ------------------------------------------------------------------ FFT
 * Batched in-place complex64 FFT over the last `ndim` (1..3) axes of a
 * C-contiguous array of `batch` * prod(dims) elements; dims are given
 * slowest first.  Forward is unnormalised (kernel e^{-i}); the inverse is
 * scaled by 1/prod(dims) (VkFFT norm=1, pyFFTW normalise_idft=True).
 * Replaces pyvkfft.cuda.VkFFTApp, NLSE/nlse.py:207-218,435-438. */
typedef struct nlse_fft_plan nlse_fft_plan;
int nlse_fft_plan_create(int ndim, const int64_t* dims, int64_t batch, nlse_fft_plan** out);
int nlse_fft_exec(nlse_fft_plan* plan, void* a_dev, int inverse, void* stream);
int nlse_fft_plan_destroy(nlse_fft_plan* plan);
/* The same plan for complex128 data (interleaved double): FP64 transforms
 * (VkFFTApp with a complex128 dtype, nlse.py:207-218).  Executed and
 * destroyed with nlse_fft_exec / nlse_fft_plan_destroy. */
int nlse_fft_plan_create_c128(int ndim, const int64_t* dims, int64_t batch, nlse_fft_plan** out);

/* ---------------------------------------------------- operator kernels
 * Elementwise operators with the semantics of NLSE/kernels_gpu.py and
 * NLSE/kernels_cpu.py.  The field holds n_items * item_size points; every
 * per-item parameter is a device array of doubles read at index
 * (item * stride), so stride 0 broadcasts one value (the reference's
 * (N_real, 1, 1) parameter broadcasting, README.md:147-159).
 * V_dev (item_size points, shared by all items) may be NULL; v_kind is
 * 1 for float32 V and 2 for complex64 V. */
typedef struct nlse_bparam {
  const double* v_dev;
  int64_t stride;
} nlse_bparam;

/* square_mod: A_sq = |A|^2 (kernels_gpu.py:179-190) */
int nlse_square_mod(const void* A_dev, void* A_sq_dev, int64_t n, void* stream);

/* nl_prop / nl_prop_without_V (kernels_gpu.py:4-65, kernels_cpu.py:5-63):
 * A *= exp(dz (-alpha [* sat] + i g A_sq sat + i V)), sat = 1/(1+A_sq/Isat).
 * loss_saturates = 0 gives the CPU semantics (loss not multiplied by sat),
 * 1 the GPU semantics. */
int nlse_nl_prop(void* A_dev, const float* A_sq_dev, int64_t n_items, int64_t item_size,
                 double dz, nlse_bparam alpha, const void* V_dev, int v_kind,
                 nlse_bparam g, nlse_bparam Isat, int loss_saturates, void* stream);

/* nl_prop_c / nl_prop_without_V_c (kernels_gpu.py:68-139):
 * A1 *= exp(dz (-alpha sat + i (g11 I1 sat + g12 I2 sat) + i V)),
 * sat = 1/(1 + I1/Isat1 + I2/Isat2).  A1, I1, I2 may be strided views:
 * item b, point p is at  base + b*item_stride + p. */
int nlse_nl_prop_c(void* A1_dev, const float* I1_dev, const float* I2_dev, int64_t n_items,
                   int64_t item_size, int64_t a_item_stride, int64_t i_item_stride,
                   double dz, nlse_bparam alpha, const void* V_dev, int v_kind,
                   nlse_bparam g11, nlse_bparam g12, nlse_bparam Isat1, nlse_bparam Isat2,
                   void* stream);

/* rabi_coupling (kernels_gpu.py:142-156): A1' = cos(w dz) A1 - i sin(w dz) A2,
 * A2' = cos(w dz) A2 - i sin(w dz) A1, computed from the old values. */
int nlse_rabi_coupling(void* A1_dev, void* A2_dev, int64_t n_items, int64_t item_size,
                       int64_t item_stride, double dz, nlse_bparam omega, void* stream);

/* A *= propagator (nlse.py:437): the propagator (prop_items * item_size
 * points) is broadcast over the leading items of A; prop_kind 1 =
 * complex64 (multiply in complex64), 2 = complex128 (multiply in
 * complex128, result rounded to complex64, nlse_1d.py:104). */
int nlse_mul_propagator(void* A_dev, const void* prop_dev, int prop_kind, int64_t n_items,
                        int64_t item_size, int64_t prop_items, void* stream);

/* A[item] *= (float)s[item]: the normalisation A = E_00 * E_in of
 * _prepare_output_array (nlse.py:304), E_00 rounded to float like numpy's
 * complex64 arithmetic.  A may be a strided component view (item_stride). */
int nlse_scale(void* A_dev, int64_t n_items, int64_t item_size, int64_t item_stride, nlse_bparam s,
               void* stream);

/* Cavity drive of DDGPE.laser_excitation (ddgpe.py:155-156), one term:
 * A -= F_r * F_t * dz * 1j in complex64 arithmetic, F_r (item_size points)
 * broadcast over items; A may be a strided component view. */
int nlse_cavity_drive(void* A_dev, int64_t n_items, int64_t item_size, int64_t item_stride,
                      const void* Fr_dev, float ft_re, float ft_im, double dz, void* stream);
/* The same on a complex128 field: the drive term is formed in complex64 as
 * the reference's complex64 profiles make it, then subtracted in FP64. */
int nlse_cavity_drive_c128(void* A_dev, int64_t n_items, int64_t item_size, int64_t item_stride,
                           const void* Fr_dev, float ft_re, float ft_im, double dz, void* stream);

/* Per-item FP64 sum of |A|^2 over item_size points -> out_dev[n_items]
 * (power integrals of nlse.py:297-303 and callbacks.py:54). */
int nlse_sumsq(const void* A_dev, int64_t n_items, int64_t item_size, double* out_dev, void* stream);
/* The same for a complex128 field. */
int nlse_sumsq_c128(const void* A_dev, int64_t n_items, int64_t item_size, double* out_dev, void* stream);
/* A[item] *= s[item] on a complex128 field, in FP64 (the normalisation of a
 * complex128 E_in, nlse.py:304). */
int nlse_scale_c128(void* A_dev, int64_t n_items, int64_t item_size, int64_t item_stride, nlse_bparam s,
                    void* stream);
/* nlse_sumsq without any allocation: no counterpart in the reference; for
 * callers that cannot allocate device memory (code under graph capture,
 * tight serving loops).  The block partials live in a fixed file-scope
 * device array of the library (65536 doubles, 512 KiB per GPU, held until
 * the process ends), so n_items * ceil(item_size / 4096) must not exceed
 * 65536 (larger requests return an error).  Results equal nlse_sumsq bit
 * for bit.  Every call on one GPU shares that array: calls that overlap on
 * one GPU (other streams, other threads) race. */
int nlse_sumsq_noalloc(const void* A_dev, int64_t n_items, int64_t item_size, double* out_dev, void* stream);

/* Per-item FP64 sum of |A - B|^2 (differences formed in FP64) -> out_dev[n_items].
 * No counterpart in the reference: the error measure and the drift test of
 * the learned corrector (relative L2 of two complex64 fields). */
int nlse_sumsq_diff(const void* A_dev, const void* B_dev, int64_t n_items, int64_t item_size, double* out_dev,
                    void* stream);

/* Hamiltonian terms of the single-component 2-D model (no counterpart in
 * the reference; the drift test of the learned corrector).  For
 *   dA/dz = (i/2k) lap A + i (g I/(1 + I/Is) + vscale V) A,  I = |A|^2,
 * H = dx dy sum[(1/2k)|grad A|^2 - G(I) - vscale Re(V) I] is conserved
 * without loss, G(I) = g Is (I - Is ln(1 + I/Is)) (g I^2/2 for Is = inf).
 * nlse_sumsq_weighted: per item sum of (wx[x] + wy[y]) |A[y][x]|^2 over an
 * (ny, nx) item, FP64 (wx = kx^2, wy = ky^2 on the transformed field gives
 * N sum |grad A|^2 by Parseval).  nlse_nl_energy: per item sum of
 * G(|A|^2) + vscale Re(V) |A|^2, FP64, inv_isat = 1/Is (0: Kerr); V as for
 * nlse_plan_set_potential (v_kind 0 none, 1 float32, 2 complex64; stride 0
 * shares one plane). */
int nlse_sumsq_weighted(const void* A_dev, int64_t n_items, int64_t ny, int64_t nx, const double* wx_dev,
                        const double* wy_dev, double* out_dev, void* stream);
int nlse_nl_energy(const void* A_dev, int64_t n_items, int64_t item_size, double g, double inv_isat,
                   const void* V_dev, int v_kind, int64_t v_item_stride, double vscale, double* out_dev,
                   void* stream);

/* Nonlinear index change of callbacks.evaluate_delta_n (callbacks.py:57-82)
 * and callbacks.adapt_delta_z (callbacks.py:85-112) in FP32, rounded op by
 * op in the reference's evaluation order:
 *   q = re*re + im*im                    (qc == 0, callbacks.py:80)
 *   q = re*re + ((im*im)*qc)*qe / 2      (qc = c, qe = eps0: the operator
 *                                         precedence of callbacks.py:109)
 *   delta_n = (coef[item] * q) / (1 + q / isat[item])
 * nlse_delta_n writes delta_n for every point to out_dev (float32, A's
 * shape); nlse_delta_n_max writes its maximum over all items and points
 * to out_dev[0] (the `delta_n.max()` of callbacks.py:111). */
int nlse_delta_n(const void* A_dev, int64_t n_items, int64_t item_size, float qc, float qe, nlse_bparam coef,
                 nlse_bparam isat, float* out_dev, void* stream);
int nlse_delta_n_max(const void* A_dev, int64_t n_items, int64_t item_size, float qc, float qe,
                     nlse_bparam coef, nlse_bparam isat, float* out_dev, void* stream);
/* The same on a complex128 field, in FP64 (out_dev: float64). */
int nlse_delta_n_c128(const void* A_dev, int64_t n_items, int64_t item_size, double qc, double qe,
                      nlse_bparam coef, nlse_bparam isat, double* out_dev, void* stream);
int nlse_delta_n_max_c128(const void* A_dev, int64_t n_items, int64_t item_size, double qc, double qe,
                          nlse_bparam coef, nlse_bparam isat, double* out_dev, void* stream);

/* ------------------------------------------- initial state and drive
 * Number kinds of nlse_vortex's arrays. */
#define NLSE_NUM_F32 0
#define NLSE_NUM_F64 1
#define NLSE_NUM_I32 2
#define NLSE_NUM_I64 3

/* Vortex phase imprint of kernels_gpu.vortex_cp (kernels_gpu.py:159-176):
 *   im[k] += angle(((ii[k] - i0) + 1j*(jj[k] - j0)) ** charge)
 * for k < n, evaluated as the principal value of charge*atan2 in (-pi, pi]
 * (FP64), added in im's precision.  im is float32 or float64; ii, jj (the
 * meshgrid coordinates) any NLSE_NUM_* kind.  The CPU kernel of the
 * reference (kernels_cpu.py:164-183) shadows i, j with its loop indices;
 * this follows the GPU kernel. */
int nlse_vortex(void* im_dev, int im_kind, int64_t n, double i0, double j0, const void* ii_dev,
                const void* jj_dev, int coord_kind, int charge, void* stream);

/* Dense propagator table of NLSE._build_propagator (nlse.py:188-197) for an
 * (ny, nx) grid, complex64:
 *   out[y*nx + x] = complex64(exp(-1j * 0.5 * (kx[x]^2 + ky[y]^2) / k * dz))
 * from the FP64 wavenumbers kx_dev[nx], ky_dev[ny] and inv_k = 1.0 / k,
 * evaluated in FP64 in numpy's operation order (theta = ((-0.5 s) * inv_k)
 * * dz, each operation rounded, then cos/sin) and rounded to complex64 —
 * equal to the reference's host table. */
int nlse_propagator_dense(void* out_dev, const double* kx_dev, const double* ky_dev, int64_t nx, int64_t ny,
                          double inv_k, double dz, void* stream);

/* Counter-based random numbers (no counterpart in the reference, which
 * draws from cupy.random / numpy.random): Philox4x64-10, the generator of
 * numpy.random.Philox.  Block b (b < nblocks) encrypts the counter
 * (counter + b + 1) with key[2] and writes its four words to out_dev[4b..];
 * with the same key and counter the words equal numpy.random.Philox(
 * counter=counter, key=key).random_raw(4 * nblocks). */
int nlse_philox4x64(uint64_t* out_dev, int64_t nblocks, const uint64_t counter[4], const uint64_t key[2],
                    void* stream);

/* DDGPE.add_noise (ddgpe.py:96-125) on a (n_items, 2, item_size) field:
 *   A[:, 0] += amp0 * dz * (z0 + 1j*z1),  A[:, 1] += amp1 * dz * (z2 + 1j*z3)
 * with amp_c = noise * sqrt(gamma_c / (4 dX dY)).  Point p takes Philox block
 * p of (counter, key) (as nlse_philox4x64) and turns words (0,1) and (2,3)
 * into standard normals by Box-Muller on 53-bit uniforms u:
 *   z0 = sqrt(-2 ln(1 - u0)) cos(2 pi u1), z1 = ... sin(2 pi u1).
 * The same draw is added to every item (the reference draws one (NY, NX)
 * array and broadcasts it).  Complex128 arithmetic, complex64 result.
 * Bitwise equality with cupy.random.normal is not attainable; successive
 * calls must advance the counter (e.g. counter[1] = call index). */
int nlse_add_noise(void* A_dev, int64_t n_items, int64_t item_size, const uint64_t counter[4],
                   const uint64_t key[2], double dz, double amp0, double amp1, void* stream);

/* ------------------------------------------------------ fused engine
 * A plan runs whole split-step loops (nlse.py:566-588) on one field shape.
 * Its tables are set once; nlse_run then performs `nsteps` steps from real
 * space to real space: 2-D fields take two HBM sweeps per step, 3-D fields
 * four, 1-D fields run all steps of a line in one launch. */
typedef struct nlse_plan nlse_plan;

typedef struct nlse_plan_desc {
  int ndim;          /* 1: (items, [2,] NX); 2: (items, [2,] NY, NX); 3: (items, NY, NX, NT) */
  int64_t ny, nx;    /* transform sizes (ny ignored for ndim 1) */
  int64_t nt;        /* third (fastest) axis of ndim 3 */
  int64_t items;     /* leading (broadcast) items; the kernels chosen depend on the points
                        (lines of ndim 1) of all items: the same field rounds differently, within
                        the parity bounds, in stacks of other sizes */
  int ncomp;         /* 1, or 2 for CNLSE / DDGPE layouts (..., 2, NY, NX) */
  int loss_saturates;
  int row_points;    /* points per thread of the x-row kernels (radix plan): 0 = default for
                        the field's size, else 8 or 16 (or the small fields' own size) */
  int col_width;     /* 0 = default; columns per block of the column pass */
  int field_c128;    /* 1: the field is complex128 and is propagated in FP64 (a complex128
                        E_in keeps its precision, nlse.py:531-534); 0: complex64 */
} nlse_plan_desc;

/* Single-component nonlinear parameters of one application (one per item):
 * adz = dz*alpha/2, gdz = dz*k/2*n2*c*eps0, inv_isat = (eps0 c)/(2 I_sat)
 * (0 for I_sat = inf), vdz = multiplier of the plan's V (dz*k/2 for NLSE,
 * whose real-space phase is dz*k/2*V, nlse.py:425). */
typedef struct nlse_nl1 {
  double adz, gdz, inv_isat, vdz;
  /* a complex delta_z (imaginary-time evolution, nlse.py:505-508) also
   * needs the dz-scaled coefficients scaled by Im(dz); the fields above
   * then hold the Re(dz)-scaled ones.  All zero for a real step. */
  double adz_i, gdz_i, vdz_i;
} nlse_nl1;
/* Two-component parameters for one component (two per item, component 0
 * then 1): see nl_prop_c; `vdz` multiplies the shared V; the _i fields are
 * the Im(dz)-scaled coefficients of a complex step (zero otherwise). */
typedef struct nlse_nl2 {
  double adz, gs_dz, gc_dz, inv_is_s, inv_is_o, vdz;
  double adz_i, gs_dz_i, gc_dz_i, vdz_i;
} nlse_nl2;

#define NLSE_SLOT_FULL 0      /* precision="single": N(dz)             */
#define NLSE_SLOT_HALF_PRE 1  /* precision="double": N before the FFTs */
#define NLSE_SLOT_HALF_POST 2 /* precision="double": N after the FFTs  */

int nlse_plan_create(const nlse_plan_desc* desc, nlse_plan** out);
int nlse_plan_destroy(nlse_plan* plan);
/* Separable propagator: px [ncomp][nx], py [ncomp][ny] complex128 with
 * P(ky,kx) = complex64(px*py), the product taken in FP64. */
int nlse_plan_set_propagator_sep(nlse_plan* plan, const double* px, const double* py);
/* 1-D plans: complex128 propagator [ncomp][nx] (host memory), multiplied in
 * FP64 like numpy's complex64*complex128 (nlse_1d.py:98-105). */
int nlse_plan_set_propagator_c128(nlse_plan* plan, const double* prop);
/* 3-D plans: the separable 2-D factors (nlse_plan_set_propagator_sep) plus
 * the complex128 temporal factor pt[nt] = exp(-i D0/2 omega^2)
 * (nlse_3d.py:105-114; no dz factor in the reference). */
int nlse_plan_set_propagator_t(nlse_plan* plan, const double* pt);
/* 3-D plans: a dense complex128 propagator [ny][nx][nt] in device memory
 * owned by the caller (e.g. a propagator assigned by the user). */
int nlse_plan_set_propagator_3d_c128(nlse_plan* plan, const void* prop_dev);
/* Dense complex64 propagator [ncomp][ny][nx] in device memory owned by the
 * caller (kept alive by the caller while the plan uses it). */
int nlse_plan_set_propagator_c64(nlse_plan* plan, const void* prop_dev);
int nlse_plan_set_nl1(nlse_plan* plan, int slot, const nlse_nl1* params);  /* [items] */
/* complex128 plans: the multiplier of V in each record of `slot`
 * ([items*ncomp]: k/2 for NLSE, nlse.py:425; k/2 and k2/2 for CNLSE; 1 for
 * the raw V of DDGPE), so that the potential term is evaluated as the
 * reference does: V' = vmul*V rounded in V's precision (float32 for a
 * float32 V), then multiplied by the step vdz/vmul in FP64.  NULL (or 0)
 * uses V as given with the record's vdz. */
int nlse_plan_set_vmul(nlse_plan* plan, int slot, const double* vmul);
int nlse_plan_set_nl2(nlse_plan* plan, int slot, const nlse_nl2* params);  /* [items*2] */
/* Rabi rotation of the single-precision step: cm1 = cos(w dz)-1, sn = sin(w dz)
 * per item (host arrays), or cm1 = sn = NULL to disable.  cm1_i and sn_i
 * are their imaginary parts for a complex dz (NULL: zero). */
int nlse_plan_set_rabi(nlse_plan* plan, const double* cm1, const double* sn, const double* cm1_i,
                       const double* sn_i);
/* Potential V as given by the user (device float32 or complex64, v_kind 1
 * or 2; complex128 plans also take float64 (3) and complex128 (4);
 * [ny][nx] or [items][ny][nx]); each application scales it by its vdz. */
int nlse_plan_set_potential(nlse_plan* plan, const void* V_dev, int v_kind, int64_t v_item_stride);
/* Cavity drive of DDGPE.laser_excitation (ddgpe.py:127-156), applied to
 * component 1 after every step s: A -= F_r0*F_t0[s]*dz*1j; A -= F_r1*F_t1[s]*dz*1j.
 * F_r* are device complex64 [ny][nx]; F_t* host complex64 arrays indexed by
 * the absolute step number; n_t their length.  NULL disables. */
int nlse_plan_set_drive(nlse_plan* plan, const void* Fr0_dev, const void* Fr1_dev,
                        const float* Ft0, const float* Ft1, int64_t n_t, double dz);
/* Nonlocal response (replaces the nl_profile convolution, nlse.py:143-153,
 * 406-409, 444-447; cnlse.py:243-249, 317-323; nlse_1d.py:65-66): every
 * nonlinear application uses the zero-padded linear "same" convolution of
 * |A|^2 with `kernel` (host float64, row-major kh x kw, both odd; 1-D plans
 * take kh = 1).  2-D kernels must be square and even in both axes (the K0
 * profile is).  NULL disables.  3-D plans reject it (the reference's
 * oaconvolve rejects a 2-D kernel on a 3-D field). */
int nlse_plan_set_nonlocal(nlse_plan* plan, const double* kernel, int64_t kh, int64_t kw);
/* Nonlocal response given in Fourier space (no counterpart in the
 * reference, whose response is the real-space K0 convolution above): every
 * nonlinear application uses the periodic convolution of |A|^2 whose
 * spectrum is the real, even function `quad` (host float64, the quadrant
 * [ky = 0..ny/2][kx = 0..nx/2], e.g. the Lorentzian 1/(1 + k^2 l^2)).
 * 2-D plans only; NULL disables. */
int nlse_plan_set_nonlocal_spectrum(nlse_plan* plan, const double* quad, int64_t qy, int64_t qx);
/* Run nsteps split steps on A (device, real space in and out).
 * precision: 0 "single" (Lie), 1 "double" (Strang).  step0 is the absolute
 * index of the first step (drive time index). */
int nlse_run(nlse_plan* plan, void* A_dev, int64_t nsteps, int precision, int64_t step0,
             void* stream);
/* nlse_run for a field that stays at the same address: the steady steps
 * are captured once into a hipGraph of `chunk` steps and replayed.  The
 * capture is kept while the field address, the table pointers and the
 * table kinds stay the same: setters that rewrite a table in place
 * (nonlinear records, Rabi, propagator factors, V contents) keep it, and
 * the replay reads the new values; the nonlocal and drive setters drop it.
 * Setters copy synchronously after waiting for the stream of the plan's
 * latest run, so steps queued before a setter read the old values; they
 * must not be called from another host thread during a run.  Results are
 * identical to nlse_run.  Plans with a drive profile and 1-D plans (one
 * launch per run) run as nlse_run. */
int nlse_run_graph(nlse_plan* plan, void* A_dev, int64_t nsteps, int precision, int64_t chunk, void* stream);
/* Capture, instantiate and upload the graph nlse_run_graph would replay for
 * (A_dev, precision, chunk), without running a step, so a later
 * nlse_run_graph call pays no capture cost (no reference counterpart: VkFFT
 * plans are built inside out_field, nlse.py:550).  No-op for plans that run
 * without a graph. */
int nlse_graph_prepare(nlse_plan* plan, void* A_dev, int precision, int64_t chunk, void* stream);
/* Launch one sweep type `count` times in place on A (device): pass 0 is a
 * steady-state row sweep (I_x, nonlinear step, F_x), pass 1 a column sweep
 * (F_y, propagator, I_y); with a nonlocal response, passes 2-6 are its
 * launches: 2 I_x + intensity transform, 3 band convolution, 4 intensity
 * column sweep, 5 nonlinear step + F_x, 6 passes 3 and 4 as a step runs
 * them (one shared launch where the tile allows).  The data is meaningless
 * afterwards; this exists to time each kernel of the step in isolation. */
int nlse_run_pass(nlse_plan* plan, void* A_dev, int pass, int64_t count, int precision, void* stream);
/* Kernel configuration actually used: points per thread of the x-row
 * kernels (their radix plan) and columns per block of the column sweep. */
int nlse_plan_config(const nlse_plan* plan, int* row_points, int* col_width);

/* ------------------------------------------------------------------
 * Uneven batches (no counterpart in the reference: its batching is the
 * leading-dimension broadcast of one grid, nlse.py:320-327).  Many 2-D
 * single-component NLSE fields of different grids and parameters advance
 * together: one launch per sweep and line length for the whole batch (or one
 * per sweep), steady steps replayed from a captured hipGraph.  Grids: powers
 * of two in [128, 2048] on both axes. */
typedef struct nlse_batch nlse_batch;
typedef struct {
  int64_t ny, nx;
  int64_t offset;     /* first complex64 element of this field in the batch buffer */
  const double* px;   /* host complex128 [nx]: exp(-i kx^2 dz / 2k) */
  const double* py;   /* host complex128 [ny] */
  nlse_nl1 nl[3];     /* slots NLSE_SLOT_FULL, _HALF_PRE, _HALF_POST */
  const void* V_dev;  /* device float32 / complex64 [ny][nx], or NULL */
  int v_kind;
} nlse_batch_item;
int nlse_batch_create(const nlse_batch_item* items, int64_t count, int loss_saturates, nlse_batch** out);
int nlse_batch_destroy(nlse_batch* batch);
/* Grids of the batch sweeps, row and column kernels.  By default the launch of
 * a line length has a block for every pass of its units (what one block of the
 * single-field kernels does), and the single launch of all lengths (below) 4 and
 * 1 blocks per CU that stride over the units.  set_grid: that many blocks per CU
 * stride over the units in both (1 to 64; where they cover the units of a
 * length, its launch is the default one).  default_grid: back to the default.
 * Results are identical; the autotuner times both. */
int nlse_batch_set_grid(nlse_batch* batch, int row_blocks_per_cu, int col_blocks_per_cu);
int nlse_batch_default_grid(nlse_batch* batch);
/* on != 0: every sweep of the batch is ONE persistent launch over the
 * units of all line lengths (each unit's length selects its code path);
 * 0 (default): one launch per line length present.  Results are
 * identical; the autotuner times both. */
int nlse_batch_set_single_launch(nlse_batch* batch, int on);
/* Work units of the row and column sweeps, and how many of them the blocks of a
 * sweep's launches take at a time (all of them by default). */
int nlse_batch_config(const nlse_batch* batch, int64_t* row_units, int64_t* col_units, int* row_grid,
                      int* col_grid);
/* nsteps split steps of every field of the batch buffer `base_dev` (real
 * space in and out); chunk > 0 replays chunks of steady steps from a
 * captured graph (results identical to chunk = 0). */
int nlse_batch_run(nlse_batch* batch, void* base_dev, int64_t nsteps, int precision, int64_t chunk,
                   void* stream);
/* Capture, instantiate and upload the graph of `chunk` steady steps that
 * nlse_batch_run replays, without running a step. */
int nlse_batch_graph_prepare(nlse_batch* batch, void* base_dev, int precision, int64_t chunk, void* stream);
/* Timing only: `count` row (pass 0) or column (pass 1) sweeps of the batch. */
int nlse_batch_run_pass(nlse_batch* batch, void* base_dev, int pass, int64_t count, void* stream);

/* ------------------------------------------------------------------
 * Learned corrector kernels (no counterpart in the reference).  A Fourier
 * neural operator maps a coarse split step to the fine-step result; its
 * products run on the BF16 matrix cores with FP32 accumulation.  All
 * pointers are device pointers, all calls asynchronous on `stream`. */
/* C(m,n) = alpha sum_k A(m,k) B(k,n) + beta C(m,n) [+ bias[n]], batched:
 * A(m,k) = A[b*sa + m*sam + k*sak], B(k,n) = B[b*sb + k*sbk + n*sbn],
 * C(m,n) = C[b*sc + m*scm + n*scn].  Operands FP32 in memory, rounded to
 * BF16 on load.  act != NULL also stores gelu(C) at the same offsets.
 * Products with few output tiles and a long K split K into slices whose
 * partial sums go to a library workspace (one per GPU, grown on demand,
 * kept until the process ends) and are summed in a fixed order: calls on
 * one stream are ordered, calls from concurrent streams of one GPU race. */
int nlse_fno_gemm(int M, int N, int K, int batch, const float* A, int64_t sam, int64_t sak, int64_t sa,
                  const float* B, int64_t sbk, int64_t sbn, int64_t sb, float* C, int64_t scm, int64_t scn,
                  int64_t sc, float alpha, float beta, const float* bias, float* act, void* stream);
/* Pointwise (1x1) channel mixing over hw pixels of channel-major planes:
 * Y[b][o][p] = sum_c X[b][c][p] W[c][o] + beta Y[b][o][p] [+ bias[o]],
 * act != NULL also stores gelu(Y) (act == Y: only gelu(Y), in place);
 * operands rounded to BF16, FP32
 * accumulation (the products of nlse_fno_gemm with M = hw, N = cout,
 * K = cin).  (cin, cout) in {(4,32), (32,32), (32,2), (4,16), (16,16),
 * (16,2), (4,8), (8,8), (8,2)}; other shapes return NLSE_ERR_ARG. */
int nlse_fno_pointwise(const float* X, const float* W, const float* bias, float* Y, float* act, int B, int cin,
                       int cout, int64_t hw, float beta, void* stream);
/* Per-mode complex channel mixing of a spectral layer (32 x 32 modes):
 * P1 [B*Cin][64][64] -> Q [B*Cout][64][64] with R [1024][Cout][Cin][2]. */
int nlse_fno_mix(const float* P1, float* Q, const float* R, int B, int Cin, int Cout, void* stream);
/* Adjoint of nlse_fno_mix: dP1 and dR (summed over the batch) from dQ. */
int nlse_fno_mix_bwd(const float* P1, const float* dQ, const float* R, float* dP1, float* dR, int B, int Cin,
                     int Cout, void* stream);
int nlse_fno_gelu_bwd(const float* z, const float* dy, float* dz, int64_t n, void* stream);
/* out[c] = sum_r x[r*sr + c*sc], r < rows, c < cols (FP64 partials). */
int nlse_fno_colsum(const float* x, int64_t rows, int64_t cols, int64_t sr, int64_t sc, float* out, void* stream);
/* out[i] = sum_p x[p*n + i] (split-K partial products). */
int nlse_fno_sum_parts(const float* x, int parts, int64_t n, float* out, void* stream);
/* Network input [B][4][hw] = [Re Y, Im Y, Re X, Im X] * inv_s[b] (Y, X complex64). */
int nlse_fno_pack(const void* Y, const void* X, const float* inv_s, float* out, int B, int64_t hw, void* stream);
/* Training target [B][2][hw] = (F - Y) * inv_s[b]. */
int nlse_fno_residual(const void* F, const void* Y, const float* inv_s, float* tgt, int B, int64_t hw,
                      void* stream);
/* A = Y + s[b] (out_re + i out_im), out [B][2][hw]. */
int nlse_fno_apply(const void* Y, const float* out, const float* s, void* A, int B, int64_t hw, void* stream);
/* d = 2 (out - tgt) / n and FP64 partial sums of (out - tgt)^2 in part[nparts]. */
int nlse_fno_mse(const float* out, const float* tgt, float* d, int64_t n, double* part, int nparts, void* stream);
/* One Adam step (bias-corrected, step t >= 1) on n parameters. */
int nlse_fno_adam(float* w, const float* g, float* m, float* v, int64_t n, float lr, float b1, float b2, float eps,
                  int64_t t, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* NLSE_HIP_H */
