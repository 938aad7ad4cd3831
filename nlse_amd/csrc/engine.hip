// libnlse_hip.so: host side of the MI355X split-step engine and its C ABI
// (declared in include/nlse_hip.h).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/nlse_hip.h"
#include "band.hpp"
#include "common.hpp"
#include "lines.hpp"
#include "wide.hpp"

using namespace nlse;

// ------------------------------------------------------------ errors
namespace nlse {

std::string& error_buffer() {
  static thread_local std::string buf;
  return buf;
}

int fail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  error_buffer() = buf;
  return code;
}

}  // namespace nlse

static const LineOps* line_ops(int64_t n) {
  static const LineOps ops[] = {make_ops_8(),   make_ops_16(),  make_ops_32(),  make_ops_64(),
                                make_ops_128(), make_ops_256(), make_ops_512(), make_ops_1024(),
                                make_ops_2048(), make_ops_4096()};
  if (!is_pow2(n) || n < 8 || n > 4096) return nullptr;
  int l = 0;
  while ((int64_t(1) << l) < n) ++l;
  return &ops[l - 3];
}

namespace nlse {
const LineOps* line_ops_public(int64_t n) { return line_ops(n); }
}  // namespace nlse

static RowArgs row_defaults() {
  RowArgs a;
  std::memset(&a, 0, sizeof a);
  a.out_scale = 1.f;
  return a;
}

static ColArgs col_defaults() {
  ColArgs a;
  std::memset(&a, 0, sizeof a);
  a.scale = 1.f;
  a.out_scale = 1.f;
  a.ncomp = 1;
  return a;
}

// ================================================================= C ABI
extern "C" {

int nlse_version(void) { return 100; }
const char* nlse_last_error(void) { return nlse::error_buffer().c_str(); }

// ---------------------------------------------------------------- FFT
struct nlse_fft_plan {
  int ndim;
  int64_t dims[3];
  int64_t batch;
  const LineOps* ops[3];
  const double2* tw[3];
  int colw[3];
  bool wide;               // complex128 data (FP64 transforms)
  const WideOps* wops[3];
};

// complex128 plan: the wide kernels' transforms (FP64 throughout)
int nlse_fft_plan_create_c128(int ndim, const int64_t* dims, int64_t batch, nlse_fft_plan** out) {
  if (!out) return fail(NLSE_ERR_ARG, "null output pointer");
  *out = nullptr;
  if (ndim < 1 || ndim > 3 || !dims || batch < 1) return fail(NLSE_ERR_ARG, "bad fft plan arguments");
  nlse_fft_plan p{};
  p.ndim = ndim;
  p.batch = batch;
  p.wide = true;
  for (int d = 0; d < ndim; ++d) {
    p.dims[d] = dims[d];
    p.wops[d] = wide_ops(dims[d]);
    if (!p.wops[d]) return fail(NLSE_ERR_ARG, "fft size %lld unsupported (power of two in [8, 4096])",
                                 (long long)dims[d]);
    int rc = p.wops[d]->twiddles(&p.tw[d]);
    if (rc) return rc;
  }
  *out = new nlse_fft_plan(p);
  return NLSE_OK;
}

static int fft_exec_wide(nlse_fft_plan* p, void* a_dev, int inverse, hipStream_t s) {
  int64_t total = 1;
  for (int d = 0; d < p->ndim; ++d) total *= p->dims[d];
  const double scale = inverse ? 1.0 / (double)total : 1.0;
  const int last = p->ndim - 1;
  WRowArgs a;
  std::memset(&a, 0, sizeof a);
  a.A = (double2*)a_dev;
  a.ngroups = p->batch * (total / p->dims[last]);
  a.rows_per_item = a.ngroups;
  a.tw = p->tw[last];
  a.inverse_first = inverse ? 1 : 0;
  a.forward_last = inverse ? 0 : 1;
  a.out_scale = (last == 0) ? scale : 1.0;
  int rc = p->wops[last]->row(1, a, s);
  if (rc) return rc;
  for (int d = last - 1; d >= 0; --d) {
    int64_t cols = 1, outer = p->batch;
    for (int e = d + 1; e < p->ndim; ++e) cols *= p->dims[e];
    for (int e = 0; e < d; ++e) outer *= p->dims[e];
    WColArgs c;
    std::memset(&c, 0, sizeof c);
    c.A = (double2*)a_dev;
    c.nslabs = outer;
    c.NX = cols;
    c.ncomp = 1;
    c.tw = p->tw[d];
    c.do_fwd = inverse ? 0 : 1;
    c.do_inv = inverse ? 1 : 0;
    c.scale = 1.0;
    c.out_scale = (d == 0) ? scale : 1.0;
    if ((rc = p->wops[d]->col(c, s))) return rc;
  }
  return NLSE_OK;
}

int nlse_fft_plan_create(int ndim, const int64_t* dims, int64_t batch, nlse_fft_plan** out) {
  if (!out) return fail(NLSE_ERR_ARG, "null output pointer");
  *out = nullptr;
  if (ndim < 1 || ndim > 3 || !dims || batch < 1) return fail(NLSE_ERR_ARG, "bad fft plan arguments");
  nlse_fft_plan p{};
  p.ndim = ndim;
  p.batch = batch;
  for (int d = 0; d < ndim; ++d) {
    p.dims[d] = dims[d];
    p.ops[d] = line_ops(dims[d]);
    if (!p.ops[d]) return fail(NLSE_ERR_ARG, "fft size %lld unsupported (power of two in [8, 4096])",
                                (long long)dims[d]);
    int rc = p.ops[d]->twiddles(&p.tw[d]);
    if (rc) return rc;
  }
  // axis d (not the last) is a strided transform with `cols` contiguous columns
  for (int d = 0; d + 1 < ndim; ++d) {
    int64_t cols = 1;
    for (int e = d + 1; e < ndim; ++e) cols *= dims[e];
    p.colw[d] = p.ops[d]->colw(cols, 0, false);
  }
  *out = new nlse_fft_plan(p);
  return NLSE_OK;
}

int nlse_fft_exec(nlse_fft_plan* p, void* a_dev, int inverse, void* stream) {
  if (!p || !a_dev) return fail(NLSE_ERR_ARG, "null argument");
  hipStream_t s = (hipStream_t)stream;
  if (p->wide) return fft_exec_wide(p, a_dev, inverse, s);
  int64_t total = 1;
  for (int d = 0; d < p->ndim; ++d) total *= p->dims[d];
  const float scale = inverse ? (float)(1.0 / (double)total) : 1.f;
  const int last = p->ndim - 1;
  // contiguous axis
  {
    RowArgs a = row_defaults();
    a.A = (float2*)a_dev;
    a.ngroups = p->batch * (total / p->dims[last]);
    a.rows_per_item = a.ngroups;
    a.tw = p->tw[last];
    a.inverse_first = inverse ? 1 : 0;
    a.forward_last = inverse ? 0 : 1;
    a.out_scale = (last == 0) ? scale : 1.f;
    int rc = p->ops[last]->row(p->ops[last]->p_row, 1, a, s);
    if (rc) return rc;
  }
  for (int d = last - 1; d >= 0; --d) {
    int64_t cols = 1, outer = p->batch;
    for (int e = d + 1; e < p->ndim; ++e) cols *= p->dims[e];
    for (int e = 0; e < d; ++e) outer *= p->dims[e];
    ColArgs a = col_defaults();
    a.A = (float2*)a_dev;
    a.nslabs = outer;
    a.NX = (int)cols;
    a.tw = p->tw[d];
    a.do_fwd = inverse ? 0 : 1;
    a.do_inv = inverse ? 1 : 0;
    a.out_scale = (d == 0) ? scale : 1.f;
    int rc = p->ops[d]->col(p->colw[d], false, a, s);
    if (rc) return rc;
  }
  return NLSE_OK;
}

int nlse_fft_plan_destroy(nlse_fft_plan* p) {
  delete p;
  return NLSE_OK;
}

}  // extern "C"

// ------------------------------------------------ operator kernels
namespace nlse {

// scratch for partial sums, grown on demand, one per device
static std::mutex g_scr_mu;
static std::map<int, std::pair<double*, size_t>> g_scratch;

int scratch_doubles(size_t n, double** out) {
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_scr_mu);
  auto& e = g_scratch[dev];
  if (e.second < n) {
    if (e.first) HIP_TRY(hipFree(e.first));
    e.first = nullptr;
    e.second = 0;
    HIP_TRY(hipMalloc(&e.first, n * sizeof(double)));
    e.second = n;
  }
  *out = e.first;
  return NLSE_OK;
}

}  // namespace nlse

namespace {

__device__ __forceinline__ double bp(const nlse_bparam& p, int64_t item) { return p.v_dev[item * p.stride]; }

__global__ void k_square_mod(const float2* __restrict__ A, float* __restrict__ S, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float2 a = A[i];
    S[i] = a.x * a.x + a.y * a.y;
  }
}

__global__ void k_nl_prop(float2* A, const float* I, int64_t items, int64_t isz, double dz, nlse_bparam alpha,
                          const void* V, int vkind, nlse_bparam g, nlse_bparam isat, int loss_sat) {
  const int64_t n = items * isz;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t item = i / isz, p = i - item * isz;
    NLParams1 prm;
    prm.adz = (float)(dz * bp(alpha, item));
    prm.gdz = (float)(dz * bp(g, item));
    const double is = bp(isat, item);
    prm.inv_isat = __builtin_isinf(is) ? 0.f : (float)(1.0 / is);
    prm.vdz = (float)dz;
    float vr, vi;
    load_v(V, vkind, p, vr, vi);
    // the standalone operator takes A_sq from the caller (it may hold a
    // convolved intensity): evaluate with the supplied I
    const float2 a = A[i];
    const float Ii = I[i];
    const float sat = 1.0f / (1.0f + Ii * prm.inv_isat);
    const float theta = fmaf(prm.gdz * Ii, sat, prm.vdz * vr);
    const float am = fmaf(prm.vdz, vi, loss_sat ? prm.adz * sat : prm.adz);
    A[i] = apply_phase_loss(a, am, theta);
  }
}

__global__ void k_nl_prop_c(float2* A1, const float* I1, const float* I2, int64_t items, int64_t isz,
                            int64_t astr, int64_t istr, double dz, nlse_bparam alpha, const void* V, int vkind,
                            nlse_bparam g11, nlse_bparam g12, nlse_bparam is1, nlse_bparam is2) {
  const int64_t n = items * isz;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t item = i / isz, p = i - item * isz;
    NLParams2 prm;
    prm.adz = (float)(dz * bp(alpha, item));
    prm.gs_dz = (float)(dz * bp(g11, item));
    prm.gc_dz = (float)(dz * bp(g12, item));
    const double a1 = bp(is1, item), a2 = bp(is2, item);
    prm.inv_is_s = __builtin_isinf(a1) ? 0.f : (float)(1.0 / a1);
    prm.inv_is_o = __builtin_isinf(a2) ? 0.f : (float)(1.0 / a2);
    prm.vdz = (float)dz;
    float vr, vi;
    load_v(V, vkind, p, vr, vi);
    const int64_t ia = item * astr + p, ii = item * istr + p;
    A1[ia] = nl2(A1[ia], I1[ii], I2[ii], prm, vr, vi);
  }
}

__global__ void k_rabi(float2* A1, float2* A2, int64_t items, int64_t isz, int64_t str, double dz,
                       nlse_bparam omega) {
  const int64_t n = items * isz;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t item = i / isz, p = i - item * isz;
    const double w = bp(omega, item) * dz;
    RabiParams r;
    const double sh = std::sin(0.5 * w);
    r.cm1 = (float)(-2.0 * sh * sh);
    r.sn = (float)std::sin(w);
    const int64_t k = item * str + p;
    float2 a1 = A1[k], a2 = A2[k];
    rabi(a1, a2, r);
    A1[k] = a1;
    A2[k] = a2;
  }
}

__global__ void k_mul_prop(float2* A, const void* P, int kind, int64_t items, int64_t isz, int64_t pitems) {
  const int64_t n = items * isz;
  const int64_t pn = pitems * isz;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t pi = i % pn;
    if (kind == 1)
      A[i] = prop_c64(A[i], reinterpret_cast<const float2*>(P)[pi], 1.f);
    else
      A[i] = to_f32(prop_c128(to_f64(A[i]), reinterpret_cast<const double2*>(P)[pi], 1.0));
  }
}

__global__ void k_scale(float2* A, int64_t items, int64_t isz, int64_t str, nlse_bparam sp) {
  const int64_t n = items * isz;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t item = i / isz, p = i - item * isz;
    const float s = (float)bp(sp, item);
    float2 a = A[item * str + p];
    A[item * str + p] = make_float2(a.x * s, a.y * s);
  }
}

__global__ void k_drive(float2* A, int64_t items, int64_t isz, int64_t str, const float2* Fr, float2 ft, float dz) {
  const int64_t n = items * isz;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t item = i / isz, p = i - item * isz;
    float2 q = cmul(Fr[p], ft);
    q = make_float2(q.x * dz, q.y * dz);
    float2 a = A[item * str + p];
    A[item * str + p] = make_float2(a.x + q.y, a.y - q.x);
  }
}

// Per-item FP64 sum of squares: block partials then a per-item pass, in a
// fixed order (deterministic).
constexpr int SUMSQ_THREADS = 256;
constexpr int SUMSQ_CHUNK = SUMSQ_THREADS * 16;

// DIFF: the sum of |A - B|^2 (the difference formed in FP64, exact for
// two float32 values of similar magnitude).
template <bool DIFF>
__global__ __launch_bounds__(SUMSQ_THREADS) void k_sumsq_part(const float2* A, const float2* B, int64_t isz,
                                                             int64_t nchunks, double* part) {
  const int64_t item = blockIdx.x / nchunks, ch = blockIdx.x % nchunks;
  const float2* a = A + item * isz;
  const float2* b = DIFF ? B + item * isz : nullptr;
  const int64_t beg = ch * SUMSQ_CHUNK, end = beg + SUMSQ_CHUNK < isz ? beg + SUMSQ_CHUNK : isz;
  double acc = 0.0;
  for (int64_t i = beg + threadIdx.x; i < end; i += SUMSQ_THREADS) {
    const float2 v = a[i];
    double x = v.x, y = v.y;
    if constexpr (DIFF) {
      const float2 w = b[i];
      x -= (double)w.x;
      y -= (double)w.y;
    }
    acc += x * x + y * y;
  }
  __shared__ double red[SUMSQ_THREADS];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = SUMSQ_THREADS / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(SUMSQ_THREADS) void k_sumsq_final(const double* part, int64_t nchunks, double* out) {
  const int64_t item = blockIdx.x;
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < nchunks; i += SUMSQ_THREADS) acc += part[item * nchunks + i];
  __shared__ double red[SUMSQ_THREADS];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = SUMSQ_THREADS / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[item] = red[0];
}

// Per-item FP64 sums of other point terms, same two passes and order.
// Weighted: (wx[x] + wy[y]) |A|^2 on an (ny, nx) item (the kinetic term of
// the Hamiltonian from a transformed field, wx = kx^2, wy = ky^2).
// Energy: G(|A|^2) + vscale Re(V) |A|^2 with G(I) = g Is (I - Is ln(1 + I/Is)),
// Is = 1/inv_isat (g I^2 / 2 when inv_isat = 0), the antiderivative of the
// saturable phase rate g I / (1 + I/Is).
struct TermWeighted {
  const float2* A;
  const double* wx;
  const double* wy;
  int64_t nx;
  __device__ double operator()(int64_t item, int64_t i, int64_t isz) const {
    const float2 v = A[item * isz + i];
    const int64_t y = i / nx;
    return (wx[i - y * nx] + wy[y]) * ((double)v.x * v.x + (double)v.y * v.y);
  }
};

struct TermEnergy {
  const float2* A;
  double g, inv_isat, vscale;
  const void* V;
  int vkind;
  int64_t v_item_stride;
  __device__ double operator()(int64_t item, int64_t i, int64_t isz) const {
    const float2 v = A[item * isz + i];
    const double I = (double)v.x * v.x + (double)v.y * v.y;
    double G;
    if (inv_isat == 0.0) {
      G = 0.5 * g * I * I;
    } else {
      const double x = I * inv_isat;
      // x - log1p(x), by its series where the difference cancels
      const double d = x < 1e-4 ? x * x * (0.5 - x * (1.0 / 3.0 - 0.25 * x)) : x - log1p(x);
      G = g * d / (inv_isat * inv_isat);
    }
    double pot = 0.0;
    if (vkind == V_REAL)
      pot = (double)static_cast<const float*>(V)[item * v_item_stride + i];
    else if (vkind == V_CPLX)
      pot = (double)static_cast<const float2*>(V)[item * v_item_stride + i].x;
    return G + vscale * pot * I;
  }
};

template <class Term>
__global__ __launch_bounds__(SUMSQ_THREADS) void k_sum_part(Term term, int64_t isz, int64_t nchunks, double* part) {
  const int64_t item = blockIdx.x / nchunks, ch = blockIdx.x % nchunks;
  const int64_t beg = ch * SUMSQ_CHUNK, end = beg + SUMSQ_CHUNK < isz ? beg + SUMSQ_CHUNK : isz;
  double acc = 0.0;
  for (int64_t i = beg + threadIdx.x; i < end; i += SUMSQ_THREADS) acc += term(item, i, isz);
  __shared__ double red[SUMSQ_THREADS];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = SUMSQ_THREADS / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

template <class Term>
static int sum_launch(const Term& term, int64_t items, int64_t isz, double* out, void* stream, const char* name) {
  const int64_t nchunks = (isz + SUMSQ_CHUNK - 1) / SUMSQ_CHUNK;
  double* part = nullptr;
  int rc = scratch_doubles((size_t)(items * nchunks), &part);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(k_sum_part<Term>, dim3((unsigned)(items * nchunks)), dim3(SUMSQ_THREADS), 0, s, term, isz,
                     nchunks, part);
  rc = launch_status(name);
  if (rc) return rc;
  hipLaunchKernelGGL(k_sumsq_final, dim3((unsigned)items), dim3(SUMSQ_THREADS), 0, s, part, nchunks, out);
  return launch_status("k_sumsq_final");
}


// Nonlinear index change of callbacks.py:57-112 in FP32, rounded op by op in
// the order the reference's array expressions evaluate:
//   q = re*re + im*im                       (evaluate_delta_n, callbacks.py:80)
//   q = re*re + ((im*im)*qc)*qe/2           (adapt_delta_z, callbacks.py:109,
//                                            qc = c, qe = eps0; qc = 0 selects
//                                            the first form)
//   delta_n = (coef*q) / (1 + q/I_sat)
// coef is c eps0/2 n2 (evaluate) or |n2| (adapt).
__device__ __forceinline__ float delta_n_point(float2 a, float qc, float qe, float coef, float isat) {
  // each product rounds before the sum, as numpy's array ops do (plain
  // operators here: the contract(off) pragma does not reach into the bodies
  // of __fmul_rn / __fadd_rn)
#pragma clang fp contract(off)
  const float yy = a.y * a.y;
  const float im = qc != 0.f ? ((yy * qc) * qe) * 0.5f : yy;
  const float q = a.x * a.x + im;
  return (coef * q) / (1.0f + q / isat);
}

__global__ void k_delta_n(const float2* A, int64_t items, int64_t isz, float qc, float qe, nlse_bparam coef,
                          nlse_bparam isat, float* out) {
  const int64_t n = items * isz;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t item = i / isz;
    out[i] = delta_n_point(A[i], qc, qe, (float)bp(coef, item), (float)bp(isat, item));
  }
}

// max over all points: block maxima (as doubles, exact) then one block
__global__ __launch_bounds__(SUMSQ_THREADS) void k_delta_n_max_part(const float2* A, int64_t isz, int64_t nchunks,
                                                                   float qc, float qe, nlse_bparam coef,
                                                                   nlse_bparam isat,
                                                                   double* part) {
  const int64_t item = blockIdx.x / nchunks, ch = blockIdx.x % nchunks;
  const float2* a = A + item * isz;
  const float cf = (float)bp(coef, item), is = (float)bp(isat, item);
  const int64_t beg = ch * SUMSQ_CHUNK, end = beg + SUMSQ_CHUNK < isz ? beg + SUMSQ_CHUNK : isz;
  float m = -__builtin_inff();
  for (int64_t i = beg + threadIdx.x; i < end; i += SUMSQ_THREADS) m = fmaxf(m, delta_n_point(a[i], qc, qe, cf, is));
  __shared__ float red[SUMSQ_THREADS];
  red[threadIdx.x] = m;
  __syncthreads();
  for (int w = SUMSQ_THREADS / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(SUMSQ_THREADS) void k_max_final(const double* part, int64_t n, float* out) {
  float m = -__builtin_inff();
  for (int64_t i = threadIdx.x; i < n; i += SUMSQ_THREADS) m = fmaxf(m, (float)part[i]);
  __shared__ float red[SUMSQ_THREADS];
  red[threadIdx.x] = m;
  __syncthreads();
  for (int w = SUMSQ_THREADS / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = red[0];
}

unsigned grid_for(int64_t n) {
  int64_t b = (n + 255) / 256;
  if (b > 65536) b = 65536;
  if (b < 1) b = 1;
  return (unsigned)b;
}

bool bparam_ok(const nlse_bparam& p) { return p.v_dev != nullptr && p.stride >= 0; }

}  // namespace

extern "C" {

int nlse_square_mod(const void* A, void* S, int64_t n, void* stream) {
  if (!A || !S || n < 0) return fail(NLSE_ERR_ARG, "bad square_mod arguments");
  if (n == 0) return NLSE_OK;
  hipLaunchKernelGGL(k_square_mod, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, (const float2*)A,
                     (float*)S, n);
  return launch_status("k_square_mod");
}

int nlse_nl_prop(void* A, const float* I, int64_t items, int64_t isz, double dz, nlse_bparam alpha,
                 const void* V, int vkind, nlse_bparam g, nlse_bparam isat, int loss_sat, void* stream) {
  if (!A || !I || items < 0 || isz < 0 || !bparam_ok(alpha) || !bparam_ok(g) || !bparam_ok(isat))
    return fail(NLSE_ERR_ARG, "bad nl_prop arguments");
  if (vkind != V_NONE && vkind != V_REAL && vkind != V_CPLX) return fail(NLSE_ERR_ARG, "bad v_kind %d", vkind);
  if (vkind != V_NONE && !V) return fail(NLSE_ERR_ARG, "null V with v_kind %d", vkind);
  const int64_t n = items * isz;
  if (n == 0) return NLSE_OK;
  hipLaunchKernelGGL(k_nl_prop, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, (float2*)A, I, items, isz,
                     dz, alpha, V, vkind, g, isat, loss_sat);
  return launch_status("k_nl_prop");
}

int nlse_nl_prop_c(void* A1, const float* I1, const float* I2, int64_t items, int64_t isz, int64_t astr,
                   int64_t istr, double dz, nlse_bparam alpha, const void* V, int vkind, nlse_bparam g11,
                   nlse_bparam g12, nlse_bparam is1, nlse_bparam is2, void* stream) {
  if (!A1 || !I1 || !I2 || items < 0 || isz < 0 || !bparam_ok(alpha) || !bparam_ok(g11) || !bparam_ok(g12) ||
      !bparam_ok(is1) || !bparam_ok(is2))
    return fail(NLSE_ERR_ARG, "bad nl_prop_c arguments");
  if (vkind != V_NONE && !V) return fail(NLSE_ERR_ARG, "null V with v_kind %d", vkind);
  const int64_t n = items * isz;
  if (n == 0) return NLSE_OK;
  hipLaunchKernelGGL(k_nl_prop_c, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, (float2*)A1, I1, I2, items,
                     isz, astr, istr, dz, alpha, V, vkind, g11, g12, is1, is2);
  return launch_status("k_nl_prop_c");
}

int nlse_rabi_coupling(void* A1, void* A2, int64_t items, int64_t isz, int64_t str, double dz, nlse_bparam omega,
                       void* stream) {
  if (!A1 || !A2 || items < 0 || isz < 0 || !bparam_ok(omega)) return fail(NLSE_ERR_ARG, "bad rabi arguments");
  const int64_t n = items * isz;
  if (n == 0) return NLSE_OK;
  hipLaunchKernelGGL(k_rabi, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, (float2*)A1, (float2*)A2, items,
                     isz, str, dz, omega);
  return launch_status("k_rabi");
}

int nlse_mul_propagator(void* A, const void* P, int kind, int64_t items, int64_t isz, int64_t pitems,
                        void* stream) {
  if (!A || !P || (kind != 1 && kind != 2) || items < 0 || isz < 0 || pitems < 1 || (items % pitems) != 0)
    return fail(NLSE_ERR_ARG, "bad mul_propagator arguments");
  const int64_t n = items * isz;
  if (n == 0) return NLSE_OK;
  hipLaunchKernelGGL(k_mul_prop, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, (float2*)A, P, kind, items,
                     isz, pitems);
  return launch_status("k_mul_prop");
}

int nlse_scale(void* A, int64_t items, int64_t isz, int64_t str, nlse_bparam sp, void* stream) {
  if (!A || items < 0 || isz < 0 || str < 0 || !bparam_ok(sp)) return fail(NLSE_ERR_ARG, "bad scale arguments");
  const int64_t n = items * isz;
  if (n == 0) return NLSE_OK;
  hipLaunchKernelGGL(k_scale, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, (float2*)A, items, isz, str, sp);
  return launch_status("k_scale");
}

int nlse_cavity_drive(void* A, int64_t items, int64_t isz, int64_t str, const void* Fr, float ft_re, float ft_im,
                      double dz, void* stream) {
  if (!A || !Fr || items < 0 || isz < 0 || str < 0) return fail(NLSE_ERR_ARG, "bad cavity_drive arguments");
  const int64_t n = items * isz;
  if (n == 0) return NLSE_OK;
  hipLaunchKernelGGL(k_drive, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, (float2*)A, items, isz, str,
                     (const float2*)Fr, make_float2(ft_re, ft_im), (float)dz);
  return launch_status("k_drive");
}

static int sumsq_launch(const void* A, const void* B, int64_t items, int64_t isz, double* out, void* stream) {
  const int64_t nchunks = (isz + SUMSQ_CHUNK - 1) / SUMSQ_CHUNK;
  double* part = nullptr;
  int rc = scratch_doubles((size_t)(items * nchunks), &part);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  if (B)
    hipLaunchKernelGGL(k_sumsq_part<true>, dim3((unsigned)(items * nchunks)), dim3(SUMSQ_THREADS), 0, s,
                       (const float2*)A, (const float2*)B, isz, nchunks, part);
  else
    hipLaunchKernelGGL(k_sumsq_part<false>, dim3((unsigned)(items * nchunks)), dim3(SUMSQ_THREADS), 0, s,
                       (const float2*)A, (const float2*)nullptr, isz, nchunks, part);
  rc = launch_status("k_sumsq_part");
  if (rc) return rc;
  hipLaunchKernelGGL(k_sumsq_final, dim3((unsigned)items), dim3(SUMSQ_THREADS), 0, s, part, nchunks, out);
  return launch_status("k_sumsq_final");
}

int nlse_sumsq(const void* A, int64_t items, int64_t isz, double* out, void* stream) {
  if (!A || !out || items < 1 || isz < 1) return fail(NLSE_ERR_ARG, "bad sumsq arguments");
  return sumsq_launch(A, nullptr, items, isz, out, stream);
}

// Fixed scratch of nlse_sumsq_noalloc: the block partial sums live in a
// file-scope device array (one copy per GPU, held until the process ends)
// instead of the grown-on-demand buffer of scratch_doubles, so the entry
// point never allocates.  Host code uses the address hipGetSymbolAddress
// returns for the current device, never the array's name.
constexpr int64_t NOALLOC_PARTIALS = 1 << 16;  // 512 KiB of FP64 partials
static __device__ __align__(256) double scratch[NOALLOC_PARTIALS];
static std::mutex g_noalloc_mu;
static std::map<int, double*> g_noalloc;  // device -> address of `scratch`

static int noalloc_scratch(double** out) {
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_noalloc_mu);
  auto it = g_noalloc.find(dev);
  if (it == g_noalloc.end()) {
    double* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      return fail(NLSE_ERR_HIP, "hipGetSymbolAddress(scratch) failed on device %d: %s", dev, hipGetErrorString(e));
    it = g_noalloc.emplace(dev, ptr).first;
  }
  *out = it->second;
  return NLSE_OK;
}

int nlse_sumsq_noalloc(const void* A, int64_t items, int64_t isz, double* out, void* stream) {
  if (!A || !out || items < 1 || isz < 1) return fail(NLSE_ERR_ARG, "bad sumsq arguments");
  const int64_t nchunks = (isz + SUMSQ_CHUNK - 1) / SUMSQ_CHUNK;
  if (nchunks > NOALLOC_PARTIALS / items)
    return fail(NLSE_ERR_ARG,
                "nlse_sumsq_noalloc: %lld items x %lld points need %lld partial sums, more than its fixed scratch "
                "of %lld (items * ceil(points / %d) must not exceed it)",
                (long long)items, (long long)isz, (long long)(items * nchunks), (long long)NOALLOC_PARTIALS,
                SUMSQ_CHUNK);
  double* part = nullptr;
  int rc = noalloc_scratch(&part);
  if (rc) return rc;
  // every partial is written by k_sumsq_part before k_sumsq_final reads it:
  // nothing to clear
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(k_sumsq_part<false>, dim3((unsigned)(items * nchunks)), dim3(SUMSQ_THREADS), 0, s,
                     (const float2*)A, (const float2*)nullptr, isz, nchunks, part);
  rc = launch_status("k_sumsq_part");
  if (rc) return rc;
  hipLaunchKernelGGL(k_sumsq_final, dim3((unsigned)items), dim3(SUMSQ_THREADS), 0, s, part, nchunks, out);
  return launch_status("k_sumsq_final");
}

int nlse_sumsq_diff(const void* A, const void* B, int64_t items, int64_t isz, double* out, void* stream) {
  if (!A || !B || !out || items < 1 || isz < 1) return fail(NLSE_ERR_ARG, "bad sumsq_diff arguments");
  return sumsq_launch(A, B, items, isz, out, stream);
}

int nlse_sumsq_weighted(const void* A, int64_t items, int64_t ny, int64_t nx, const double* wx, const double* wy,
                        double* out, void* stream) {
  if (!A || !wx || !wy || !out || items < 1 || ny < 1 || nx < 1) return fail(NLSE_ERR_ARG, "bad sumsq_weighted arguments");
  const TermWeighted t{(const float2*)A, wx, wy, nx};
  return sum_launch(t, items, ny * nx, out, stream, "k_sum_part(weighted)");
}

int nlse_nl_energy(const void* A, int64_t items, int64_t isz, double g, double inv_isat, const void* V, int vkind,
                   int64_t v_item_stride, double vscale, double* out, void* stream) {
  if (!A || !out || items < 1 || isz < 1 || inv_isat < 0 || (vkind != V_NONE && !V) ||
      (vkind != V_NONE && vkind != V_REAL && vkind != V_CPLX) || v_item_stride < 0)
    return fail(NLSE_ERR_ARG, "bad nl_energy arguments");
  const TermEnergy t{(const float2*)A, g, inv_isat, vscale, V, vkind, v_item_stride};
  return sum_launch(t, items, isz, out, stream, "k_sum_part(energy)");
}

int nlse_delta_n(const void* A, int64_t items, int64_t isz, float qc, float qe, nlse_bparam coef,
                 nlse_bparam isat, float* out, void* stream) {
  if (!A || !out || items < 0 || isz < 0 || !bparam_ok(coef) || !bparam_ok(isat))
    return fail(NLSE_ERR_ARG, "bad delta_n arguments");
  const int64_t n = items * isz;
  if (n == 0) return NLSE_OK;
  hipLaunchKernelGGL(k_delta_n, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, (const float2*)A, items, isz,
                     qc, qe, coef, isat, out);
  return launch_status("k_delta_n");
}

int nlse_delta_n_max(const void* A, int64_t items, int64_t isz, float qc, float qe, nlse_bparam coef,
                     nlse_bparam isat, float* out, void* stream) {
  if (!A || !out || items < 1 || isz < 1 || !bparam_ok(coef) || !bparam_ok(isat))
    return fail(NLSE_ERR_ARG, "bad delta_n_max arguments");
  const int64_t nchunks = (isz + SUMSQ_CHUNK - 1) / SUMSQ_CHUNK;
  double* part = nullptr;
  int rc = scratch_doubles((size_t)(items * nchunks), &part);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(k_delta_n_max_part, dim3((unsigned)(items * nchunks)), dim3(SUMSQ_THREADS), 0, s,
                     (const float2*)A, isz, nchunks, qc, qe, coef, isat, part);
  rc = launch_status("k_delta_n_max_part");
  if (rc) return rc;
  hipLaunchKernelGGL(k_max_final, dim3(1), dim3(SUMSQ_THREADS), 0, s, part, items * nchunks, out);
  return launch_status("k_max_final");
}

// ------------------------------------------------------- fused plan
struct nlse_plan {
  nlse_plan_desc d;
  const LineOps* rops = nullptr;  // rows (NX) / x columns in 3-D
  const LineOps* cops = nullptr;  // columns (NY)
  const LineOps* tops = nullptr;  // t rows (NT, 3-D)
  const double2* twx = nullptr;
  const double2* twy = nullptr;
  const double2* twt = nullptr;
  int row_points = 0;             // row kernels' set size (radix plan) if given, else chosen (row_p)
  bool small = false;             // small-field plans (SMALL_FIELD)
  bool large = false;             // a stack of LARGE_STACK points
  int through = 0;                // level of the field's stores (through_level; complex64)
  bool cplx = false;              // any nonlinear record of a complex dz
  bool cplx_slot[3] = {false, false, false};
  int colw = 1;                   // y-column tile
  int colw_x = 1;                 // x-column tile (3-D)
  double2* prop128 = nullptr;     // 1-D complex128 propagator [ncomp][nx]
  double2* pt = nullptr;          // 3-D temporal factor [nt]
  const double2* ptab128 = nullptr;  // 3-D dense complex128 table (caller-owned)
  // propagator
  int pkind = -1;
  double2* px = nullptr;
  double2* py = nullptr;
  const float2* ptab = nullptr;
  // nonlinear parameters per slot (device)
  void* nl[3] = {nullptr, nullptr, nullptr};
  RabiParams* rabi = nullptr;
  const void* V = nullptr;
  int vkind = V_NONE;
  int64_t v_item_stride = 0;
  // drive
  const float2* fr0 = nullptr;
  const float2* fr1 = nullptr;
  std::vector<float2> ft0, ft1;
  float drv_dz = 0.f;
  bool drive = false;
  // nonlocal response
  struct {
    bool on = false;
    int r = 0;                      // kernel half-width (after trimming)
    int64_t M = 0;                  // row pairing of the packed intensity (torus rows unless full)
    bool full = false;              // one component on the full NY-row torus (spectral response)
    bool unpack = false;            // spectral response of row-pair-packed spectra (k_colu)
    bool direct = false;            // every point convolved directly
    const LineOps* zops = nullptr;  // columns of length M
    const double2* twz = nullptr;
    int colw = 1;
    float2* Z = nullptr;            // [items][M][nx]
    float* kq = nullptr;            // [M/2+1][nx/2+1] spectrum / (M nx)
    double* K = nullptr;            // 1-D kernel [2r+1]
    float* KT = nullptr;            // 2-D kernel, transposed [2r+1][kr]
    int kr = 0, kc = 0;
    int pitch = 0;                  // LDS row pitch of k_nl_band (0: tile width)
    bool mfma = false;              // band tiles on the matrix cores (band_mfma_body)
    float* KP = nullptr;            // their kernel rows, zero-padded [2r+1][kpw]
    int kpw = 0;

    int* rowmap = nullptr;          // [ny]
    int nb = 0;
    BandTile* tiles = nullptr;
    int ntiles = 0;
    size_t lds = 0;
    float* rowband = nullptr;
    float* colband = nullptr;
  } nlc;
  // stream of the plan's latest run: setters wait for it before rewriting a
  // table in place, so steps already queued read the values they were
  // queued with
  hipStream_t last = nullptr;
  bool ran = false;
  // complex128 fields: the wide kernels (wide.hpp), FP64 records
  bool wide = false;
  const WideOps* wr = nullptr;  // rows (NX) / x columns in 3-D
  const WideOps* wc = nullptr;  // columns (NY)
  const WideOps* wt = nullptr;  // t rows (NT)
  const double2* wtwx = nullptr;
  const double2* wtwy = nullptr;
  const double2* wtwt = nullptr;
  std::vector<nlse_nl1> nl1_host[3];  // the records as given (wide: rebuilt when vmul changes)
  std::vector<nlse_nl2> nl2_host[3];
  std::vector<double> vmul[3];        // multiplier of V per record (0: V as given)
  struct {
    double* K = nullptr;  // 2-D kernel [kh][kw], FP64
    int kh = 0, kw = 0;
    double* KP = nullptr;  // flipped, zero-padded rows of the matrix-core form [kh][kpw]
    int kpw = 0;
    bool pair = false;     // K even in y
    double* I = nullptr;   // |A|^2 in real space, layout of A
    double* Ic = nullptr;  // its convolution
  } wn;
  // captured steady steps
  hipStream_t cap = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  std::vector<uint64_t> gkey;
};

static void graph_free(nlse_plan* p);

static void nlc_free(nlse_plan* p) {
  auto& n = p->nlc;
  (void)hipFree(n.Z);
  (void)hipFree(n.kq);
  (void)hipFree(n.K);
  (void)hipFree(n.KT);
  (void)hipFree(n.KP);

  (void)hipFree(n.rowmap);
  (void)hipFree(n.tiles);
  (void)hipFree(n.rowband);
  (void)hipFree(n.colband);
  n = {};
  (void)hipFree(p->wn.K);
  (void)hipFree(p->wn.KP);
  (void)hipFree(p->wn.I);
  (void)hipFree(p->wn.Ic);
  p->wn = {};
}

int nlse_plan_create(const nlse_plan_desc* d, nlse_plan** out) {
  if (!out || !d) return fail(NLSE_ERR_ARG, "null argument");
  *out = nullptr;
  if (d->ndim < 1 || d->ndim > 3) return fail(NLSE_ERR_ARG, "nlse_plan supports ndim 1, 2, 3 (got %d)", d->ndim);
  if (d->items < 1 || (d->ncomp != 1 && d->ncomp != 2))
    return fail(NLSE_ERR_ARG, "bad items/ncomp (%lld, %d)", (long long)d->items, d->ncomp);
  if (d->ndim == 3 && d->ncomp != 1) return fail(NLSE_ERR_ARG, "3-D plans have one component");
  if (d->field_c128 != 0 && d->field_c128 != 1) return fail(NLSE_ERR_ARG, "field_c128 must be 0 or 1");
  nlse_plan* p = new nlse_plan();
  p->d = *d;
  if (d->field_c128) {
    p->wide = true;
    p->wr = wide_ops(d->nx);
    p->wc = d->ndim >= 2 ? wide_ops(d->ny) : p->wr;
    p->wt = d->ndim == 3 ? wide_ops(d->nt) : p->wr;
    if (!p->wr || !p->wc || !p->wt) {
      delete p;
      return fail(NLSE_ERR_ARG, "grid (%lld, %lld, %lld) unsupported (powers of two in [8, 4096])", (long long)d->ny,
                  (long long)d->nx, (long long)d->nt);
    }
    int rc = p->wr->twiddles(&p->wtwx);
    if (!rc) rc = p->wc->twiddles(&p->wtwy);
    if (!rc) rc = p->wt->twiddles(&p->wtwt);
    if (rc) {
      delete p;
      return rc;
    }
    if (d->row_points != 0) {
      delete p;
      return fail(NLSE_ERR_ARG, "complex128 plans have one radix plan (row_points must be 0)");
    }
    *out = p;
    return NLSE_OK;
  }
  p->rops = line_ops(d->nx);
  p->cops = d->ndim >= 2 ? line_ops(d->ny) : p->rops;
  p->tops = d->ndim == 3 ? line_ops(d->nt) : p->rops;
  if (!p->rops || !p->cops || !p->tops) {
    delete p;
    return fail(NLSE_ERR_ARG, "grid (%lld, %lld, %lld) unsupported (powers of two in [8, 4096])", (long long)d->ny,
                (long long)d->nx, (long long)d->nt);
  }
  int rc = p->rops->twiddles(&p->twx);
  if (!rc) rc = p->cops->twiddles(&p->twy);
  if (!rc) rc = p->tops->twiddles(&p->twt);
  if (rc) {
    delete p;
    return rc;
  }
  const int64_t points = d->items * d->ncomp * (d->ndim >= 2 ? d->ny : 1) * d->nx * (d->ndim == 3 ? d->nt : 1);
  p->small = d->ndim == 2 && points <= SMALL_FIELD;
  p->large = d->ndim == 2 && d->ncomp == 1 && d->items > 1 && points >= LARGE_STACK;
  p->through = through_level(points * 8);
  if (d->row_points != 0) {
    const int pr = p->rops->p_row, pa = p->rops->p_row_alt, ps = p->rops->p_row_small;
    const bool ok = d->row_points == pr || (d->ndim != 1 && (d->row_points == pa || (p->small && d->row_points == ps)));
    if (!ok) {
      delete p;
      return fail(NLSE_ERR_ARG, "row_points %d unsupported for rows of %lld (0, %d or %d)", d->row_points,
                  (long long)d->nx, pr, pa);
    }
    p->row_points = d->row_points;
  }
  if (d->ndim == 2) {
    // default tile: the widest of 8, 4, 2, 1 columns that gives every CU a
    // block, or every second CU one of at most 256 threads (wider tiles read
    // longer row segments, see LineCfg::WDEF).  Local step at W = 8 / 4 / 2:
    // 1024^2 24.9 / 21.3 / - us, 512^2 - / 10.6 / 11.4 us, 256^2 10.6 / 8.3 /
    // 7.8 us.  Columns of 1024 points and more in fields that are not written
    // through take at most 4: the L2 joins the segments of neighbouring tiles
    // (same XCD) before they leave it, and smaller blocks overlap better.
    // Column sweep at W = 8 / 4: 8 x 1024^2 47.9 / 40.2 us, 28 x 1024^2 139 /
    // 123, 2 x 2048^2 54.0 / 48.3, 6 x 2048^2 139 / 131 us; written through
    // 4 x 1024^2 26.8 / 29.2, 2048^2 28.5 / 32.3 us
    int want = d->col_width;
    if (want == 0) {
      int dev = 0, cus = 256;
      if (hipGetDevice(&dev) != hipSuccess ||
          hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
        cus = 256;
      const int64_t t = d->ny / (p->small ? p->cops->p_col_small : p->cops->p_col);
      want = p->cops->colw(d->nx, 0, p->small);
      if (!p->through && d->ny >= 1024) want = std::min(want, 4);
      for (; want > 1; want >>= 1) {
        const int64_t blocks = d->items * d->ncomp * (d->nx / want);
        if (blocks >= cus || (2 * blocks >= cus && want * t <= 256)) break;
      }
    }
    p->colw = p->cops->colw(d->nx, want, p->small);
  }
  if (d->ndim == 3) {
    p->colw = p->cops->colw(d->nx * d->nt, d->col_width, false);
    p->colw_x = p->rops->colw(d->nt, d->col_width, false);
  }
  *out = p;
  return NLSE_OK;
}

int nlse_plan_destroy(nlse_plan* p) {
  if (!p) return NLSE_OK;
  (void)hipFree(p->px);
  (void)hipFree(p->py);
  for (void* q : p->nl) (void)hipFree(q);
  (void)hipFree(p->prop128);
  (void)hipFree(p->pt);
  (void)hipFree(p->rabi);
  nlc_free(p);
  graph_free(p);
  if (p->cap) (void)hipStreamDestroy(p->cap);
  delete p;
  return NLSE_OK;
}

// Points per thread of the x-row sweep.  With a nonlocal response only a
// run's first sweep is one: it keeps the default plan.
static int row_p(const nlse_plan* p) {
  if (p->wide) return 8;
  if (p->row_points) return p->row_points;
  if (p->nlc.on) return p->rops->p_row;
  return p->small ? p->rops->p_row_small : (p->large ? p->rops->p_row_large : p->rops->p_row);
}

int nlse_plan_config(const nlse_plan* p, int* row_points, int* col_width) {
  // 3-D plans report their y-column tile
  if (!p) return fail(NLSE_ERR_ARG, "null plan");
  if (p->wide) {
    if (row_points) *row_points = row_p(p);
    if (col_width) *col_width = 0;
    return NLSE_OK;
  }
  if (row_points) *row_points = row_p(p);
  if (col_width) *col_width = p->colw;
  return NLSE_OK;
}

// Copy a host table into the plan's device buffer (allocated on first use).
// A buffer that already exists may be read by steps still queued on the
// stream of the plan's latest run (or by a replay of its graph): the copy
// waits for that stream first.  hipMemcpy alone would not, since it is
// ordered on the null stream only and torch's streams do not block on it.
static int upload(nlse_plan* p, void** dst, const void* src, size_t bytes) {
  if (!*dst) {
    HIP_TRY(hipMalloc(dst, bytes));
  } else if (p->ran) {
    HIP_TRY(hipStreamSynchronize(p->last));
  }
  HIP_TRY(hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice));
  return NLSE_OK;
}

int nlse_plan_set_propagator_sep(nlse_plan* p, const double* px, const double* py) {
  if (!p || !px || !py) return fail(NLSE_ERR_ARG, "null argument");
  if (p->d.ndim == 1) return fail(NLSE_ERR_ARG, "1-D plans take nlse_plan_set_propagator_c128");
  const int nc = p->d.ncomp;
  int rc = upload(p, (void**)&p->px, px, sizeof(double2) * nc * p->d.nx);
  if (!rc) rc = upload(p, (void**)&p->py, py, sizeof(double2) * nc * p->d.ny);
  if (rc) return rc;
  p->pkind = p->d.ndim == 3 ? PROP_SEP3D : PROP_SEP64;
  return NLSE_OK;
}

int nlse_plan_set_propagator_c128(nlse_plan* p, const double* prop) {
  if (!p || !prop) return fail(NLSE_ERR_ARG, "null argument");
  if (p->d.ndim != 1) return fail(NLSE_ERR_ARG, "complex128 line propagator is for 1-D plans");
  int rc = upload(p, (void**)&p->prop128, prop, sizeof(double2) * p->d.ncomp * p->d.nx);
  if (rc) return rc;
  p->pkind = PROP_C64;  // any non-negative kind marks the plan ready
  return NLSE_OK;
}

int nlse_plan_set_propagator_t(nlse_plan* p, const double* pt) {
  if (!p || !pt) return fail(NLSE_ERR_ARG, "null argument");
  if (p->d.ndim != 3) return fail(NLSE_ERR_ARG, "temporal propagator factor is for 3-D plans");
  return upload(p, (void**)&p->pt, pt, sizeof(double2) * p->d.nt);
}

int nlse_plan_set_propagator_3d_c128(nlse_plan* p, const void* tab) {
  if (!p || !tab) return fail(NLSE_ERR_ARG, "null argument");
  if (p->d.ndim != 3) return fail(NLSE_ERR_ARG, "dense complex128 propagators are for 3-D plans");
  p->ptab128 = (const double2*)tab;
  p->pkind = PROP_C128;
  return NLSE_OK;
}

int nlse_plan_set_propagator_c64(nlse_plan* p, const void* tab) {
  if (!p || !tab) return fail(NLSE_ERR_ARG, "null argument");
  if (p->d.ndim != 2) return fail(NLSE_ERR_ARG, "dense complex64 propagators are for 2-D plans");
  p->ptab = (const float2*)tab;
  p->pkind = PROP_C64;
  return NLSE_OK;
}


// Device records of a complex128 plan's slot from the records as given and
// the slot's V multipliers: the V phase step dzv = vdz / vmul, so that the
// kernels form dzv * fl(vmul * V) with V' rounded in V's own precision.
static double vstep(double vdz, double vmul) { return vmul != 0.0 ? vdz / vmul : vdz; }

static int wide_upload_nl(nlse_plan* p, int slot) {
  const auto& vm = p->vmul[slot];
  if (p->d.ncomp == 1) {
    const auto& r = p->nl1_host[slot];
    if (r.empty()) return NLSE_OK;
    std::vector<WNL1> h(r.size());
    for (size_t i = 0; i < r.size(); ++i) {
      const double m = i < vm.size() ? vm[i] : 0.0;
      h[i] = WNL1{r[i].adz,   r[i].gdz,   r[i].inv_isat, vstep(r[i].vdz, m), r[i].adz_i, r[i].gdz_i,
                  vstep(r[i].vdz_i, m), m, (r[i].adz_i != 0.0 || r[i].gdz_i != 0.0 || r[i].vdz_i != 0.0) ? 1 : 0, 0};
    }
    return upload(p, &p->nl[slot], h.data(), h.size() * sizeof(WNL1));
  }
  const auto& r = p->nl2_host[slot];
  if (r.empty()) return NLSE_OK;
  std::vector<WNL2> h(r.size());
  for (size_t i = 0; i < r.size(); ++i) {
    const double m = i < vm.size() ? vm[i] : 0.0;
    const bool cx = r[i].adz_i != 0.0 || r[i].gs_dz_i != 0.0 || r[i].gc_dz_i != 0.0 || r[i].vdz_i != 0.0;
    h[i] = WNL2{r[i].adz,   r[i].gs_dz,   r[i].gc_dz,   r[i].inv_is_s,     r[i].inv_is_o, vstep(r[i].vdz, m),
                r[i].adz_i, r[i].gs_dz_i, r[i].gc_dz_i, vstep(r[i].vdz_i, m), m,           cx ? 1 : 0, 0};
  }
  return upload(p, &p->nl[slot], h.data(), h.size() * sizeof(WNL2));
}

int nlse_plan_set_vmul(nlse_plan* p, int slot, const double* vmul) {
  if (!p || slot < 0 || slot > 2) return fail(NLSE_ERR_ARG, "bad set_vmul arguments");
  if (!p->wide) return fail(NLSE_ERR_ARG, "set_vmul applies to complex128 plans");
  const int64_t n = p->d.items * p->d.ncomp;
  if (vmul) p->vmul[slot].assign(vmul, vmul + n);
  else p->vmul[slot].clear();
  return wide_upload_nl(p, slot);
}

int nlse_plan_set_nl1(nlse_plan* p, int slot, const nlse_nl1* prm) {
  if (!p || !prm || slot < 0 || slot > 2) return fail(NLSE_ERR_ARG, "bad set_nl1 arguments");
  if (p->d.ncomp != 1) return fail(NLSE_ERR_ARG, "set_nl1 on a two-component plan");
  if (p->wide) {
    p->nl1_host[slot].assign(prm, prm + p->d.items);
    return wide_upload_nl(p, slot);
  }
  std::vector<NLParams1> h(p->d.items);
  bool cx = false;
  for (int64_t i = 0; i < p->d.items; ++i) {
    h[i].adz = (float)prm[i].adz;
    h[i].gdz = (float)prm[i].gdz;
    h[i].inv_isat = (float)prm[i].inv_isat;
    h[i].vdz = (float)prm[i].vdz;
    h[i].adz_i = (float)prm[i].adz_i;
    h[i].gdz_i = (float)prm[i].gdz_i;
    h[i].vdz_i = (float)prm[i].vdz_i;
    h[i].cplx = prm[i].adz_i != 0.0 || prm[i].gdz_i != 0.0 || prm[i].vdz_i != 0.0;
    cx = cx || h[i].cplx;
  }
  p->cplx_slot[slot] = cx;
  p->cplx = p->cplx_slot[0] || p->cplx_slot[1] || p->cplx_slot[2];
  return upload(p, &p->nl[slot], h.data(), h.size() * sizeof(NLParams1));
}

int nlse_plan_set_nl2(nlse_plan* p, int slot, const nlse_nl2* prm) {
  if (!p || !prm || slot < 0 || slot > 2) return fail(NLSE_ERR_ARG, "bad set_nl2 arguments");
  if (p->d.ncomp != 2) return fail(NLSE_ERR_ARG, "set_nl2 on a one-component plan");
  if (p->wide) {
    p->nl2_host[slot].assign(prm, prm + p->d.items * 2);
    return wide_upload_nl(p, slot);
  }
  std::vector<NLParams2> h(p->d.items * 2);
  for (int64_t i = 0; i < p->d.items * 2; ++i) {
    h[i].adz = (float)prm[i].adz;
    h[i].gs_dz = (float)prm[i].gs_dz;
    h[i].gc_dz = (float)prm[i].gc_dz;
    h[i].inv_is_s = (float)prm[i].inv_is_s;
    h[i].inv_is_o = (float)prm[i].inv_is_o;
    h[i].vdz = (float)prm[i].vdz;
    h[i].adz_i = (float)prm[i].adz_i;
    h[i].gs_dz_i = (float)prm[i].gs_dz_i;
    h[i].gc_dz_i = (float)prm[i].gc_dz_i;
    h[i].vdz_i = (float)prm[i].vdz_i;
    h[i].cplx = prm[i].adz_i != 0.0 || prm[i].gs_dz_i != 0.0 || prm[i].gc_dz_i != 0.0 || prm[i].vdz_i != 0.0;
  }
  return upload(p, &p->nl[slot], h.data(), h.size() * sizeof(NLParams2));
}

int nlse_plan_set_rabi(nlse_plan* p, const double* cm1, const double* sn, const double* cm1_i, const double* sn_i) {
  if (!p) return fail(NLSE_ERR_ARG, "null plan");
  if (!cm1 || !sn) {
    (void)hipFree(p->rabi);
    p->rabi = nullptr;
    return NLSE_OK;
  }
  if (p->wide) {
    std::vector<WRabi> h(p->d.items);
    for (int64_t i = 0; i < p->d.items; ++i)
      h[i] = WRabi{cm1[i], sn[i], cm1_i ? cm1_i[i] : 0.0, sn_i ? sn_i[i] : 0.0};
    return upload(p, (void**)&p->rabi, h.data(), h.size() * sizeof(WRabi));
  }
  std::vector<RabiParams> h(p->d.items);
  for (int64_t i = 0; i < p->d.items; ++i) {
    h[i].cm1 = (float)cm1[i];
    h[i].sn = (float)sn[i];
    h[i].cm1_i = cm1_i ? (float)cm1_i[i] : 0.f;
    h[i].sn_i = sn_i ? (float)sn_i[i] : 0.f;
  }
  return upload(p, (void**)&p->rabi, h.data(), h.size() * sizeof(RabiParams));
}

int nlse_plan_set_potential(nlse_plan* p, const void* V, int vkind, int64_t vstride) {
  if (!p) return fail(NLSE_ERR_ARG, "null plan");
  const bool ok = vkind == V_NONE || vkind == V_REAL || vkind == V_CPLX ||
                  (p->wide && (vkind == V_REAL64 || vkind == V_CPLX128));
  if (!ok) return fail(NLSE_ERR_ARG, "bad v_kind %d", vkind);
  if (vkind != V_NONE && !V) return fail(NLSE_ERR_ARG, "null V");
  p->V = V;
  p->vkind = vkind;
  p->v_item_stride = vstride;
  return NLSE_OK;
}

int nlse_plan_set_drive(nlse_plan* p, const void* fr0, const void* fr1, const float* ft0, const float* ft1,
                        int64_t n_t, double dz) {
  if (!p) return fail(NLSE_ERR_ARG, "null plan");
  graph_free(p);  // captured launches bake in table pointers
  if (!fr0) {
    p->drive = false;
    return NLSE_OK;
  }
  if (p->d.ncomp != 2 || !fr1 || !ft0 || !ft1 || n_t < 0) return fail(NLSE_ERR_ARG, "bad drive arguments");
  p->fr0 = (const float2*)fr0;
  p->fr1 = (const float2*)fr1;
  p->ft0.assign((const float2*)ft0, (const float2*)ft0 + n_t);
  p->ft1.assign((const float2*)ft1, (const float2*)ft1 + n_t);
  p->drv_dz = (float)dz;
  p->drive = true;
  return NLSE_OK;
}

// LDS bytes of one k_nl_band block for tiles of `nc` columns.
static size_t band_lds(int nc, int r, int kc, int pitch) { return band_lds_floats(nc, r, kc, pitch) * sizeof(float); }

// Band geometry and kernel spectrum of a 2-D plan (see nonlocal.hpp).
static int nlc_setup_2d(nlse_plan* p, const double* kernel, int kw) {
  auto& n = p->nlc;
  const int64_t ny = p->d.ny, nx = p->d.nx, items = p->d.items, slabs = items * p->d.ncomp;
  const int r0 = kw / 2;
  for (int u = 0; u < kw; ++u)
    for (int v = 0; v < kw; ++v) {
      const double k = kernel[u * kw + v];
      if (k != kernel[(kw - 1 - u) * kw + v] || k != kernel[u * kw + (kw - 1 - v)])
        return fail(NLSE_ERR_ARG, "nonlocal kernel must be even in both axes");
    }
  // taps farther than the field extent only ever meet the zero padding
  const int r = (int)std::min<int64_t>(r0, std::max(ny, nx) - 1);
  const int w = 2 * r + 1;
  n.r = r;
  n.M = p->d.ncomp == 1 ? ny / 2 : ny;
  n.direct = n.M < 8 || 2 * r >= n.M || 2 * r >= nx;
  // band rows in increasing order
  std::vector<int> rowmap(ny, -1);
  int nb = 0;
  for (int64_t y = 0; y < ny; ++y) {
    const int64_t yp = y % n.M;
    if (n.direct || yp < r || yp >= n.M - r) rowmap[y] = nb++;
  }
  n.nb = nb;
  // band tiles on the matrix cores when a tile's staged intensities and the
  // kernel fit 64 KB of LDS (else the VALU form, which stages the kernel in
  // chunks of rows)
  size_t mfma_lds = 0;
  for (int tx = 1; tx <= 4; tx *= 2) mfma_lds = std::max(mfma_lds, band_mfma_lds_floats(tx, r) * sizeof(float));
  n.mfma = NLSE_BAND_MFMA && mfma_lds <= 64 * 1024 && band_mfma_chunks(r) <= BAND_MFMA_MAX_CHUNKS;
  // output tiles: band rows over the full width, side columns elsewhere
  std::vector<BandTile> tiles;
  auto strip = [&](int64_t ya, int64_t yb, int x0, int width) {
    for (int cx = 0; cx < width; cx += 64) {
      const int nc = std::min(64, width - cx);
      const int h = n.mfma ? 16 * (4 / band_mfma_tx(nc)) : (64 / nc) * RB_BAND;
      for (int64_t y0 = ya; y0 < yb; y0 += h)
        tiles.push_back(BandTile{(int)y0, x0 + cx, (int)std::min<int64_t>(h, yb - y0), nc});
    }
  };
  for (int64_t y = 0; y < ny;) {
    const bool band = rowmap[y] >= 0;
    int64_t e = y;
    while (e < ny && (rowmap[e] >= 0) == band) ++e;
    if (band) {
      for (int x0 = 0; x0 < nx; x0 += 64) strip(y, e, x0, (int)std::min<int64_t>(64, nx - x0));
    } else {
      strip(y, e, 0, r);
      strip(y, e, (int)nx - r, r);
    }
    y = e;
  }
  // kernel rows padded to a multiple of KU_BAND, staged in chunks of kc rows
  std::vector<int> widths;
  for (const BandTile& t : tiles)
    if (std::find(widths.begin(), widths.end(), t.ncols) == widths.end()) widths.push_back(t.ncols);
  // LDS row pitch: fixed 128 or 256 floats (immediate offsets) when the
  // widest staged tile fits, else the tile width
  int wmax = 0;
  for (int nc : widths) wmax = std::max(wmax, nc + 2 * r);
  n.pitch = wmax <= 128 ? 128 : (wmax <= 256 ? 256 : 0);
  auto lds_for = [&](int kc) {
    size_t m = 0;
    for (int nc : widths) m = std::max(m, band_lds(nc, r, kc, n.pitch));
    return m;
  };
  n.kr = (w + KU_BAND - 1) / KU_BAND * KU_BAND;
  n.kc = n.kr;
  while (n.kc > KU_BAND && lds_for(n.kc) > 64 * 1024) n.kc -= KU_BAND;
  n.lds = lds_for(n.kc);
  if (n.mfma) {
    n.lds = 0;
    for (int nc : widths) n.lds = std::max(n.lds, band_mfma_lds_floats(band_mfma_tx(nc), r) * sizeof(float));
  }
  if (n.lds > 150 * 1024) return fail(NLSE_ERR_ARG, "nonlocal kernel too wide (%d points)", kw);
  std::vector<double> kp((size_t)n.kr * w, 0.0);
  for (int u = 0; u < w; ++u)
    for (int v = 0; v < w; ++v) kp[(size_t)u * w + v] = kernel[(size_t)(u + r0 - r) * kw + (v + r0 - r)];
  std::vector<float> kt((size_t)w * n.kr, 0.f);
  for (int u = 0; u < w; ++u)
    for (int v = 0; v < w; ++v) kt[(size_t)v * n.kr + u] = (float)kp[(size_t)u * w + v];
  int rc = upload(p, (void**)&n.KT, kt.data(), kt.size() * sizeof(float));
  if (!rc && n.mfma) {
    n.kpw = band_mfma_kpw(r);
    std::vector<float> km((size_t)w * n.kpw, 0.f);
    for (int u = 0; u < w; ++u)
      for (int v = 0; v < w; ++v) km[(size_t)u * n.kpw + 16 + v] = (float)kp[(size_t)u * w + v];
    rc = upload(p, (void**)&n.KP, km.data(), km.size() * sizeof(float));
  }
  if (!rc) rc = upload(p, (void**)&n.rowmap, rowmap.data(), rowmap.size() * sizeof(int));
  if (!rc) rc = upload(p, (void**)&n.tiles, tiles.data(), tiles.size() * sizeof(BandTile));
  if (rc) return rc;
  n.ntiles = (int)tiles.size();
  HIP_TRY(hipMalloc((void**)&n.rowband, sizeof(float) * slabs * nb * nx));
  if (!n.direct) {
    HIP_TRY(hipMalloc((void**)&n.colband, sizeof(float) * slabs * ny * 2 * r));
    HIP_TRY(hipMalloc((void**)&n.Z, sizeof(float2) * items * n.M * nx));
    n.zops = line_ops(n.M);
    if (!n.zops) return fail(NLSE_ERR_ARG, "unsupported intensity column length %lld", (long long)n.M);
    if ((rc = n.zops->twiddles(&n.twz))) return rc;
    n.colw = n.zops->colw(nx, p->d.col_width, false);
    // spectrum of the kernel wrapped on the M x nx torus, centre at (0, 0):
    // real and even, K^(ky, kx) = sum_{u,v} K[u][v] cos(2pi ky (u-r)/M) cos(2pi kx (v-r)/nx)
    const int64_t hy = n.M / 2 + 1, hx = nx / 2 + 1;
    std::vector<double> cx(nx), cy(n.M);
    for (int64_t j = 0; j < nx; ++j) cx[j] = std::cos(2.0 * M_PI * (double)j / (double)nx);
    for (int64_t j = 0; j < n.M; ++j) cy[j] = std::cos(2.0 * M_PI * (double)j / (double)n.M);
    // x sums over kernel columns v in order, the phase index k (v - r) mod
    // nx stepped by (v - r) along k
    std::vector<double> row((size_t)w * hx, 0.0);
    for (int u = 0; u < w; ++u) {
      double* ru = row.data() + (size_t)u * hx;
      for (int v = 0; v < w; ++v) {
        const double kv = kp[(size_t)u * w + v];
        const int64_t step = ((int64_t)(v - r) % nx + nx) % nx;
        int64_t ph = 0;
        for (int64_t k = 0; k < hx; ++k) {
          ru[k] += kv * cx[ph];
          ph += step;
          if (ph >= nx) ph -= nx;
        }
      }
    }
    const double norm = 1.0 / ((double)n.M * (double)nx);
    // the y sums run over kernel rows u in order for every kx at once (the
    // innermost loop contiguous in kx; one cosine per (ky, u))
    std::vector<float> kq((size_t)hy * hx);
    std::vector<double> acc((size_t)hx);
    for (int64_t ky = 0; ky < hy; ++ky) {
      std::fill(acc.begin(), acc.end(), 0.0);
      for (int u = 0; u < w; ++u) {
        const double c = cy[((ky * (u - r)) % n.M + n.M) % n.M];
        const double* ru = row.data() + (size_t)u * hx;
        for (int64_t k = 0; k < hx; ++k) acc[k] += c * ru[k];
      }
      for (int64_t k = 0; k < hx; ++k) kq[(size_t)ky * hx + k] = (float)(acc[k] * norm);
    }
    if ((rc = upload(p, (void**)&n.kq, kq.data(), kq.size() * sizeof(float)))) return rc;
  }
  if (n.lds > 64 * 1024) {
    const void* fn = n.pitch == 128 ? (const void*)k_nl_band<128>
                                    : (n.pitch == 256 ? (const void*)k_nl_band<256> : (const void*)k_nl_band<0>);
    HIP_TRY(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)n.lds));
  }
  return NLSE_OK;
}

int nlse_plan_set_nonlocal_spectrum(nlse_plan* p, const double* quad, int64_t qy, int64_t qx) {
  if (!p) return fail(NLSE_ERR_ARG, "null plan");
  graph_free(p);  // captured launches bake in table pointers
  nlc_free(p);
  if (!quad) return NLSE_OK;
  if (p->d.ndim != 2) return fail(NLSE_ERR_ARG, "spectral nonlocal responses are for 2-D plans");
  if (p->wide) return fail(NLSE_ERR_ARG, "spectral nonlocal responses are for complex64 plans");
  const int64_t ny = p->d.ny, nx = p->d.nx, items = p->d.items;
  if (qy != ny / 2 + 1 || qx != nx / 2 + 1)
    return fail(NLSE_ERR_ARG, "spectrum quadrant must be (%lld, %lld)", (long long)(ny / 2 + 1),
                (long long)(nx / 2 + 1));
  auto& n = p->nlc;
  int rc = NLSE_OK;
  n.r = 0;
  n.direct = false;
  // one component: rows packed in pairs (y, y + NY/2) as for the kernel
  // convolution, the full-torus y convolution done on unpacked column
  // pairs (k_colu); two components: one complex line I1 + i I2 per row.
  // NLSE_SPECTRAL_FULL_ROWS selects the earlier form that transforms every
  // row's intensity on its own (twice the intensity work).
#ifndef NLSE_SPECTRAL_FULL_ROWS
#define NLSE_SPECTRAL_FULL_ROWS 0
#endif
  n.full = p->d.ncomp == 1 && NLSE_SPECTRAL_FULL_ROWS;
  n.unpack = p->d.ncomp == 1 && !NLSE_SPECTRAL_FULL_ROWS;
  n.M = p->d.ncomp == 1 ? ny / 2 : ny;
  n.nb = 0;
  std::vector<int> rowmap(ny, -1);
  std::vector<float> kq((size_t)qy * qx);
  const double norm = 1.0 / ((double)ny * (double)nx);
  for (size_t i = 0; i < kq.size(); ++i) kq[i] = (float)(quad[i] * norm);
  n.zops = line_ops(ny);
  if (!n.zops) rc = fail(NLSE_ERR_ARG, "unsupported column length %lld", (long long)ny);
  if (!rc) rc = n.zops->twiddles(&n.twz);
  if (!rc) rc = upload(p, (void**)&n.rowmap, rowmap.data(), rowmap.size() * sizeof(int));
  if (!rc) rc = upload(p, (void**)&n.kq, kq.data(), kq.size() * sizeof(float));
  const int64_t zrows = n.full ? ny : n.M;
  if (!rc && hipMalloc((void**)&n.Z, sizeof(float2) * items * zrows * nx) != hipSuccess)
    rc = fail(NLSE_ERR_HIP, "hipMalloc of the intensity buffer failed");
  if (rc) {
    nlc_free(p);
    return rc;
  }
  n.colw = n.zops->colw(nx, p->d.col_width, false);
  n.on = true;
  return NLSE_OK;
}

int nlse_plan_set_nonlocal(nlse_plan* p, const double* kernel, int64_t kh, int64_t kw) {
  if (!p) return fail(NLSE_ERR_ARG, "null plan");
  graph_free(p);  // captured launches bake in table pointers
  nlc_free(p);
  if (!kernel) return NLSE_OK;
  if (p->d.ndim == 3) return fail(NLSE_ERR_ARG, "in1 and in2 should have the same dimensionality");
  if (kw < 1 || kh < 1 || kw % 2 == 0 || kh % 2 == 0)
    return fail(NLSE_ERR_ARG, "nonlocal kernel sizes must be odd (got %lld x %lld)", (long long)kh, (long long)kw);
  int rc;
  if (p->d.ndim == 1) {
    if (kh != 1) return fail(NLSE_ERR_ARG, "1-D plans take a 1-D nonlocal kernel");
    const int r0 = (int)(kw / 2);
    const int r = (int)std::min<int64_t>(r0, p->d.nx - 1);
    rc = upload(p, (void**)&p->nlc.K, kernel + (r0 - r), sizeof(double) * (2 * r + 1));
    p->nlc.r = r;
  } else if (p->wide) {
    // direct FP64 convolution; taps farther than the field extent only ever
    // meet the zero padding and are dropped
    const int rh0 = (int)(kh / 2), rw0 = (int)(kw / 2);
    const int rh = (int)std::min<int64_t>(rh0, p->d.ny - 1), rw = (int)std::min<int64_t>(rw0, p->d.nx - 1);
    const int h = 2 * rh + 1, w = 2 * rw + 1;
    std::vector<double> k((size_t)h * w);
    for (int u = 0; u < h; ++u)
      for (int v = 0; v < w; ++v) k[(size_t)u * w + v] = kernel[(size_t)(u + rh0 - rh) * kw + (v + rw0 - rw)];
    const size_t pts = (size_t)(p->d.items * p->d.ncomp * p->d.ny * p->d.nx);
    rc = upload(p, (void**)&p->wn.K, k.data(), k.size() * sizeof(double));
    if (!rc && hipMalloc((void**)&p->wn.I, pts * sizeof(double)) != hipSuccess)
      rc = fail(NLSE_ERR_HIP, "hipMalloc of the intensity buffer failed");
    if (!rc && hipMalloc((void**)&p->wn.Ic, pts * sizeof(double)) != hipSuccess)
      rc = fail(NLSE_ERR_HIP, "hipMalloc of the convolved intensity buffer failed");
    p->wn.kh = h;
    p->wn.kw = w;
    if (!rc && wide_conv2d_mfma_fits(h, w)) {
      // matrix-core form: rows flipped in both axes, 16 zeros in front
      const int kpw = 4 * wconv_mfma_chunks(rw) + 16;
      std::vector<double> kpad((size_t)h * kpw, 0.0);
      for (int u = 0; u < h; ++u)
        for (int v = 0; v < w; ++v) kpad[(size_t)u * kpw + 16 + v] = k[(size_t)(h - 1 - u) * w + (w - 1 - v)];
      bool even = true;
      for (int u = 0; u < h && even; ++u)
        for (int v = 0; v < w; ++v)
          if (kpad[(size_t)u * kpw + 16 + v] != kpad[(size_t)(h - 1 - u) * kpw + 16 + v]) {
            even = false;
            break;
          }
      rc = upload(p, (void**)&p->wn.KP, kpad.data(), kpad.size() * sizeof(double));
      p->wn.kpw = kpw;
      p->wn.pair = even;
    }
  } else {
    if (kh != kw) return fail(NLSE_ERR_ARG, "2-D nonlocal kernels must be square");
    if (kw > 8191) return fail(NLSE_ERR_ARG, "nonlocal kernel too wide (%lld points)", (long long)kw);
    rc = nlc_setup_2d(p, kernel, (int)kw);
  }
  if (rc) {
    nlc_free(p);
    return rc;
  }
  p->nlc.on = true;
  return NLSE_OK;
}

static int check_ready(const nlse_plan* p, int precision) {
  if (p->pkind < 0) return fail(NLSE_ERR_STATE, "propagator not set");
  if (precision == 0 && !p->nl[NLSE_SLOT_FULL]) return fail(NLSE_ERR_STATE, "nonlinear parameters (single) not set");
  if (precision == 1 && (!p->nl[NLSE_SLOT_HALF_PRE] || !p->nl[NLSE_SLOT_HALF_POST]))
    return fail(NLSE_ERR_STATE, "nonlinear parameters (double) not set");
  return NLSE_OK;
}

// The loss of a nonlinear application varies from point to point.
static int nl_general(const nlse_plan* p) { return p->d.loss_saturates || p->vkind == V_CPLX || p->cplx; }

static RowArgs plan_row_args(const nlse_plan* p, void* A) {
  RowArgs r = row_defaults();
  r.A = (float2*)A;
  r.rows_per_item = p->d.ny;
  r.ngroups = p->d.items * p->d.ny;
  r.tw = p->twx;
  r.loss_sat = p->d.loss_saturates;
  r.V = p->V;
  r.vkind = p->vkind;
  r.v_item_stride = p->v_item_stride;
  r.rabi = p->rabi;
  r.drv_r0 = p->fr0;
  r.drv_r1 = p->fr1;
  r.drv_dz = p->drv_dz;
  r.general = nl_general(p);
  r.through = p->through;
  return r;
}

static ColArgs plan_col_args(const nlse_plan* p, void* A) {
  ColArgs c = col_defaults();
  c.A = (float2*)A;
  c.nslabs = p->d.items * p->d.ncomp;
  c.NX = (int)p->d.nx;
  c.ncomp = p->d.ncomp;
  c.tw = p->twy;
  c.do_fwd = c.do_prop = c.do_inv = 1;
  c.pkind = p->pkind;
  c.px = p->px;
  c.py = p->py;
  c.ptab = p->ptab;
  c.scale = (float)(1.0 / ((double)p->d.nx * (double)p->d.ny));
  c.through = p->through;
  return c;
}

// steady-state row sweep of step k (not the first or the last sweep of a run)
static RowArgs mid_row(const nlse_plan* p, const RowArgs& r, int precision, bool last) {
  RowArgs a = r;
  a.inverse_first = 1;
  a.forward_last = last ? 0 : 1;
  a.has_a = 1;
  a.nlp_a = precision == 1 ? p->nl[NLSE_SLOT_HALF_POST] : p->nl[NLSE_SLOT_FULL];
  a.has_rabi = (precision == 0 && p->rabi != nullptr && p->d.ncomp == 2) ? 1 : 0;
  a.has_b = (precision == 1 && !last) ? 1 : 0;
  a.nlp_b = p->nl[NLSE_SLOT_HALF_PRE];
  return a;
}

// ------------------------------------------- nonlocal response (2-D)
static NlcArgs plan_nlc_args(const nlse_plan* p, void* A) {
  NlcArgs a;
  std::memset(&a, 0, sizeof a);
  const auto& n = p->nlc;
  a.A = (float2*)A;
  a.Z = n.Z;
  a.M = n.M;
  a.ny = p->d.ny;
  a.ncomp = p->d.ncomp;
  a.ngroups = p->d.items * n.M;
  a.tw = p->twx;
  a.write_z = n.direct ? 0 : 1;
  a.loss_sat = p->d.loss_saturates;
  a.rabi = p->rabi;
  a.V = p->V;
  a.vkind = p->vkind;
  a.v_item_stride = p->v_item_stride;
  a.drv_r0 = p->fr0;
  a.drv_r1 = p->fr1;
  a.drv_dz = p->drv_dz;
  a.out_scale = 1.f;
  a.rowmap = n.rowmap;
  a.rowband = n.rowband;
  a.colband = n.colband;
  a.nb = n.nb;
  a.r = n.r;
  a.direct = n.direct ? 1 : 0;
  a.full = n.full ? 1 : 0;
  a.general = nl_general(p);
  a.through = p->through;
  return a;
}

static BandArgs band_args(const nlse_plan* p, const void* A);

static int band_launch(const nlse_plan* p, const void* A, hipStream_t s) {
  const auto& n = p->nlc;
  const int64_t slabs = p->d.items * p->d.ncomp;
  if (n.ntiles == 0) return NLSE_OK;
  if (slabs > 65535) return fail(NLSE_ERR_ARG, "too many fields for the nonlocal band pass (%lld)", (long long)slabs);
  const BandArgs b = band_args(p, A);
  const dim3 grid((unsigned)n.ntiles, (unsigned)slabs), block(64 * BAND_WAVES);
  if (n.pitch == 128)
    hipLaunchKernelGGL(k_nl_band<128>, grid, block, n.lds, s, b);
  else if (n.pitch == 256)
    hipLaunchKernelGGL(k_nl_band<256>, grid, block, n.lds, s, b);
  else
    hipLaunchKernelGGL(k_nl_band<0>, grid, block, n.lds, s, b);
  return launch_status("k_nl_band");
}

static BandArgs band_args(const nlse_plan* p, const void* A) {
  const auto& n = p->nlc;
  BandArgs b;
  b.A = (const float2*)A;
  b.ny = (int)p->d.ny;
  b.nx = (int)p->d.nx;
  b.r = n.r;
  b.KT = n.KT;
  b.kr = n.kr;
  b.kc = n.kc;
  b.tiles = n.tiles;
  b.ntiles = n.ntiles;
  b.rowmap = n.rowmap;
  b.nb = n.nb;
  b.rowband = n.rowband;
  b.colband = n.colband;
  b.KP = n.KP;
  b.kpw = n.kpw;
  b.mfma = n.mfma ? 1 : 0;
  return b;
}

static ColArgs nlc_col_args(const nlse_plan* p) {
  ColArgs c = col_defaults();
  c.A = p->nlc.Z;
  c.nslabs = p->d.items;
  c.NX = (int)p->d.nx;
  c.ncomp = 1;
  c.tw = p->nlc.twz;
  c.do_fwd = c.do_prop = c.do_inv = 1;
  c.pkind = PROP_KREAL;
  c.kq = p->nlc.kq;
  c.through = p->through;
  return c;
}

// One nonlinear application with the nonlocal response: [I_x,] the
// convolved intensity, N, [Rabi, drive, F_x].  drive_step < 0: no drive.
#ifndef NLSE_MERGE_BAND
#define NLSE_MERGE_BAND 1
#endif

// Band pass and intensity column sweep.  Both only read what the first
// nonlocal row pass wrote, so they share one launch where the column tile
// allows it (k_colz_band: the band tiles, on the matrix cores or the VALU,
// run beside the sweep); a second stream costs more in cross-queue waits
// than it overlaps.
static int band_and_z(nlse_plan* p, const void* A, hipStream_t s, const ColArgs* cz_override = nullptr) {
  auto& n = p->nlc;
  const int64_t slabs = p->d.items * p->d.ncomp;
  const ColArgs cz = cz_override ? *cz_override : nlc_col_args(p);
  if (n.unpack) return n.zops->colu(cz, s);  // spectral response: no band points
  int rc = NLSE_OK;
  if (NLSE_MERGE_BAND && !n.direct && n.ntiles > 0 && slabs <= 65535) {
    rc = n.zops->colz_band(n.colw, cz, band_args(p, A), n.pitch, n.lds, (int64_t)n.ntiles * slabs, s);
    if (rc <= 0) return rc;  // launched, or an error
  }
  if ((rc = band_launch(p, A, s))) return rc;
  if (!n.direct) rc = n.zops->col(n.colw, false, cz, s);
  return rc;
}

static int nlc_apply(nlse_plan* p, void* A, int inverse_first, int forward_last, const void* nlp, bool rabi,
                     int64_t drive_step, hipStream_t s) {
  NlcArgs a = plan_nlc_args(p, A);
  a.inverse_first = inverse_first;
  int rc = NLSE_OK;
  if (a.inverse_first || a.write_z) rc = p->rops->nlc(1, a, s);
  if (rc) return rc;
  if ((rc = band_and_z(p, A, s))) return rc;
  a.forward_last = forward_last;
  a.nlp = nlp;
  a.has_rabi = rabi ? 1 : 0;
  if (drive_step >= 0) {
    a.has_drive = 1;
    a.drv_t0 = p->ft0[drive_step];
    a.drv_t1 = p->ft1[drive_step];
  }
  return p->rops->nlc(2, a, s);
}

static int run1d(nlse_plan* p, void* A, int64_t nsteps, int precision, hipStream_t s) {
  Line1DArgs a;
  std::memset(&a, 0, sizeof a);
  a.A = (float2*)A;
  a.ngroups = p->d.items;
  a.tw = p->twx;
  a.prop = p->prop128;
  a.scale = 1.0 / (double)p->d.nx;
  a.nsteps = nsteps;
  a.precision = precision;
  a.loss_sat = p->d.loss_saturates;
  a.nl_full = p->nl[NLSE_SLOT_FULL];
  a.nl_pre = p->nl[NLSE_SLOT_HALF_PRE];
  a.nl_post = p->nl[NLSE_SLOT_HALF_POST];
  a.rabi = (precision == 0 && p->d.ncomp == 2) ? p->rabi : nullptr;
  a.V = p->V;
  a.vkind = p->vkind;
  a.nlk = p->nlc.on ? p->nlc.K : nullptr;
  a.nlr = p->nlc.r;
  a.general = nl_general(p);
  return p->rops->line1d(p->d.ncomp, a, s);
}

// ---------------------------------------------------------- step chains
// Every multi-sweep run is first(), then step(k) for k = 0..nsteps-1, where
// step(k) ends with the sweep that returns the field to real space when k
// is the last step.  Steps that are not the last are "steady": the same
// launches with the same arguments (drive aside), which is what a captured
// graph replays.
//
// 2-D (local): between sweeps the field is x-spectral, B = F_x(A).
//   first:  row pass F_x [after N(dz/2) in "double"]
//   step:   column pass (F_y, P/(NX NY), I_y), row pass (I_x, N, [Rabi,
//           drive,] [N(dz/2) of the next step,] F_x unless last)
// 2-D (nonlocal): the row pass becomes one or two nonlocal applications
//   (nlc_apply: intensity transform, band pass, intensity sweep, N).
// 3-D field (items, NY, NX, NT), t fastest.  Between sweeps the field is
// t- and x-spectral; a step is four sweeps:
//   y columns: F_y, P/(NX NY NT), I_y   x columns: I_x
//   t rows:    I_t, N, F_t               x columns: F_x (unless last)

static RowArgs row3d_args(const nlse_plan* p, void* A) {
  RowArgs r = row_defaults();
  r.A = (float2*)A;
  r.rows_per_item = p->d.ny * p->d.nx;
  r.ngroups = p->d.items * p->d.ny * p->d.nx;
  r.tw = p->twt;
  r.loss_sat = p->d.loss_saturates;
  r.V = p->V;
  r.vkind = p->vkind;
  r.v_item_stride = p->v_item_stride;
  r.general = nl_general(p);
  r.through = p->through;
  return r;
}

static ColArgs colx3d_args(const nlse_plan* p, void* A) {
  ColArgs cx = col_defaults();
  cx.A = (float2*)A;
  cx.nslabs = p->d.items * p->d.ny;
  cx.NX = (int)p->d.nt;
  cx.tw = p->twx;
  cx.through = p->through;
  return cx;
}

static ColArgs coly3d_args(const nlse_plan* p, void* A) {
  ColArgs cy = col_defaults();
  cy.A = (float2*)A;
  cy.nslabs = p->d.items;
  cy.NX = (int)(p->d.nx * p->d.nt);
  cy.tw = p->twy;
  cy.do_fwd = cy.do_prop = cy.do_inv = 1;
  cy.pkind = p->pkind;
  cy.ptab128 = p->ptab128;
  cy.px = p->px;
  cy.py = p->py;
  cy.pt = p->pt;
  cy.nt = (int)p->d.nt;
  cy.scale = (float)(1.0 / ((double)p->d.nx * (double)p->d.ny * (double)p->d.nt));
  cy.through = p->through;
  return cy;
}


// ------------------------------------------------- complex128 chains
// The same sweeps as the complex64 chains below, on the wide kernels; the
// nonlocal response is three launches: I_x with |A|^2 stored, the direct
// FP64 convolution, then the nonlinear step with the convolved intensity.
static WRowArgs wrow_args(const nlse_plan* p, void* A) {
  WRowArgs r;
  std::memset(&r, 0, sizeof r);
  r.A = (double2*)A;
  r.rows_per_item = p->d.ny;
  r.ngroups = p->d.items * p->d.ny;
  r.tw = p->wtwx;
  r.loss_sat = p->d.loss_saturates;
  r.V = p->V;
  r.vkind = p->vkind;
  r.v_item_stride = p->v_item_stride;
  r.rabi = (const WRabi*)p->rabi;
  r.drv_r0 = p->fr0;
  r.drv_r1 = p->fr1;
  r.drv_dz = p->drv_dz;
  r.out_scale = 1.0;
  return r;
}

static WColArgs wcol_args(const nlse_plan* p, void* A) {
  WColArgs c;
  std::memset(&c, 0, sizeof c);
  c.A = (double2*)A;
  c.nslabs = p->d.items * p->d.ncomp;
  c.NX = p->d.nx;
  c.ncomp = p->d.ncomp;
  c.tw = p->wtwy;
  c.do_fwd = c.do_prop = c.do_inv = 1;
  c.pkind = p->pkind;
  c.px = p->px;
  c.py = p->py;
  c.ptab = p->ptab;
  c.scale = 1.0 / ((double)p->d.nx * (double)p->d.ny);
  c.out_scale = 1.0;
  return c;
}

static WRowArgs wmid_row(const nlse_plan* p, const WRowArgs& r, int precision, bool last) {
  WRowArgs a = r;
  a.inverse_first = 1;
  a.forward_last = last ? 0 : 1;
  a.has_a = 1;
  a.nlp_a = precision == 1 ? p->nl[NLSE_SLOT_HALF_POST] : p->nl[NLSE_SLOT_FULL];
  a.has_rabi = (precision == 0 && p->rabi != nullptr && p->d.ncomp == 2) ? 1 : 0;
  a.has_b = (precision == 1 && !last) ? 1 : 0;
  a.nlp_b = p->nl[NLSE_SLOT_HALF_PRE];
  return a;
}

// One nonlinear application with the nonlocal response (2-D).
static int wnlc_apply(nlse_plan* p, void* A, int inverse_first, int forward_last, const void* nlp, bool rabi,
                      int64_t drive_step, hipStream_t s) {
  const int G = (int)p->d.ncomp;
  WRowArgs a = wrow_args(p, A);
  a.inverse_first = inverse_first;
  a.write_I = 1;
  a.I = p->wn.I;
  int rc = p->wr->row(G, a, s);
  if (rc) return rc;
  WConvArgs c;
  c.I = p->wn.I;
  c.Ic = p->wn.Ic;
  c.nslabs = p->d.items * p->d.ncomp;
  c.ny = (int)p->d.ny;
  c.nx = (int)p->d.nx;
  c.K = p->wn.K;
  c.kh = p->wn.kh;
  c.kw = p->wn.kw;
  c.lds = 0;
  c.KP = p->wn.KP;
  c.kpw = p->wn.kpw;
  c.pair = p->wn.pair ? 1 : 0;
  if ((rc = wide_conv2d(c, s))) return rc;
  WRowArgs b = wrow_args(p, A);
  b.has_a = 1;
  b.nlp_a = nlp;
  b.Ic = p->wn.Ic;
  b.has_rabi = rabi ? 1 : 0;
  b.forward_last = forward_last;
  if (drive_step >= 0) {
    b.has_drive = 1;
    b.drv_t0 = p->ft0[drive_step];
    b.drv_t1 = p->ft1[drive_step];
  }
  return p->wr->row(G, b, s);
}

static WRowArgs wrow3d_args(const nlse_plan* p, void* A) {
  WRowArgs r = wrow_args(p, A);
  r.rows_per_item = p->d.ny * p->d.nx;
  r.ngroups = p->d.items * p->d.ny * p->d.nx;
  r.tw = p->wtwt;
  r.rabi = nullptr;
  return r;
}

static WColArgs wcolx3d_args(const nlse_plan* p, void* A) {
  WColArgs c;
  std::memset(&c, 0, sizeof c);
  c.A = (double2*)A;
  c.nslabs = p->d.items * p->d.ny;
  c.NX = p->d.nt;
  c.ncomp = 1;
  c.tw = p->wtwx;
  c.scale = 1.0;
  c.out_scale = 1.0;
  return c;
}

static WColArgs wcoly3d_args(const nlse_plan* p, void* A) {
  WColArgs c = wcol_args(p, A);
  c.nslabs = p->d.items;
  c.NX = p->d.nx * p->d.nt;
  c.ncomp = 1;
  c.ptab128 = p->ptab128;
  c.pt = p->pt;
  c.nt = (int)p->d.nt;
  c.scale = 1.0 / ((double)p->d.nx * (double)p->d.ny * (double)p->d.nt);
  return c;
}

static int wchain_first(nlse_plan* p, void* A, int precision, hipStream_t s) {
  int rc;
  if (p->d.ndim == 3) {
    WRowArgs a = wrow3d_args(p, A);
    a.forward_last = 1;
    a.has_b = precision == 1;
    a.nlp_b = p->nl[NLSE_SLOT_HALF_PRE];
    if ((rc = p->wt->row(1, a, s))) return rc;
    WColArgs c = wcolx3d_args(p, A);
    c.do_fwd = 1;
    return p->wr->col(c, s);
  }
  if (p->nlc.on && precision == 1) return wnlc_apply(p, A, 0, 1, p->nl[NLSE_SLOT_HALF_PRE], false, -1, s);
  WRowArgs a = wrow_args(p, A);
  a.forward_last = 1;
  a.has_b = (!p->nlc.on && precision == 1) ? 1 : 0;
  a.nlp_b = p->nl[NLSE_SLOT_HALF_PRE];
  return p->wr->row(p->d.ncomp, a, s);
}

static int wchain_step(nlse_plan* p, void* A, int precision, bool last, int64_t abs_k, hipStream_t s) {
  int rc;
  if (p->d.ndim == 3) {
    if ((rc = p->wc->col(wcoly3d_args(p, A), s))) return rc;
    WColArgs ci = wcolx3d_args(p, A);
    ci.do_inv = 1;
    if ((rc = p->wr->col(ci, s))) return rc;
    WRowArgs a = wmid_row(p, wrow3d_args(p, A), precision, last);
    if ((rc = p->wt->row(1, a, s))) return rc;
    if (last) return NLSE_OK;
    WColArgs cf = wcolx3d_args(p, A);
    cf.do_fwd = 1;
    return p->wr->col(cf, s);
  }
  if ((rc = p->wc->col(wcol_args(p, A), s))) return rc;
  if (p->nlc.on) {
    const int64_t ds = p->drive ? abs_k : -1;
    if (precision == 0) {
      const bool rabi = p->rabi != nullptr && p->d.ncomp == 2;
      return wnlc_apply(p, A, 1, last ? 0 : 1, p->nl[NLSE_SLOT_FULL], rabi, ds, s);
    }
    if ((rc = wnlc_apply(p, A, 1, 0, p->nl[NLSE_SLOT_HALF_POST], false, ds, s))) return rc;
    return last ? NLSE_OK : wnlc_apply(p, A, 0, 1, p->nl[NLSE_SLOT_HALF_PRE], false, -1, s);
  }
  WRowArgs a = wmid_row(p, wrow_args(p, A), precision, last);
  a.has_drive = p->drive ? 1 : 0;
  if (p->drive) {
    a.drv_t0 = p->ft0[abs_k];
    a.drv_t1 = p->ft1[abs_k];
  }
  return p->wr->row(p->d.ncomp, a, s);
}

static int wrun1d(nlse_plan* p, void* A, int64_t nsteps, int precision, hipStream_t s) {
  WLine1DArgs a;
  std::memset(&a, 0, sizeof a);
  a.A = (double2*)A;
  a.ngroups = p->d.items;
  a.tw = p->wtwx;
  a.prop = p->prop128;
  a.scale = 1.0 / (double)p->d.nx;
  a.nsteps = nsteps;
  a.precision = precision;
  a.loss_sat = p->d.loss_saturates;
  a.nl_full = p->nl[NLSE_SLOT_FULL];
  a.nl_pre = p->nl[NLSE_SLOT_HALF_PRE];
  a.nl_post = p->nl[NLSE_SLOT_HALF_POST];
  a.rabi = (precision == 0 && p->d.ncomp == 2) ? (const WRabi*)p->rabi : nullptr;
  a.V = p->V;
  a.vkind = p->vkind;
  a.nlk = p->nlc.on ? p->nlc.K : nullptr;
  a.nlr = p->nlc.r;
  return p->wr->line1d(p->d.ncomp, a, s);
}

// x-row sweep with the plan's row kernel (default or alternative radix plan)
static int launch_rows(const nlse_plan* p, int G, const RowArgs& a, hipStream_t s) {
  return p->rops->row(row_p(p), G, a, s);
}

static int chain_first(nlse_plan* p, void* A, int precision, hipStream_t s) {
  if (p->wide) return wchain_first(p, A, precision, s);
  int rc;
  if (p->d.ndim == 3) {
    RowArgs a = row3d_args(p, A);
    a.forward_last = 1;
    a.has_b = precision == 1;
    a.nlp_b = p->nl[NLSE_SLOT_HALF_PRE];
    if ((rc = p->tops->row(p->tops->p_row, 1, a, s))) return rc;
    ColArgs c = colx3d_args(p, A);
    c.do_fwd = 1;
    return p->rops->col(p->colw_x, false, c, s);
  }
  if (p->nlc.on && precision == 1) return nlc_apply(p, A, 0, 1, p->nl[NLSE_SLOT_HALF_PRE], false, -1, s);
  RowArgs a = plan_row_args(p, A);
  a.forward_last = 1;
  a.has_b = (!p->nlc.on && precision == 1) ? 1 : 0;
  a.nlp_b = p->nl[NLSE_SLOT_HALF_PRE];
  return launch_rows(p, p->d.ncomp, a, s);
}

// Step k of a run (absolute step index `abs_k` for the drive profile).
static int chain_step(nlse_plan* p, void* A, int precision, bool last, int64_t abs_k, hipStream_t s) {
  if (p->wide) return wchain_step(p, A, precision, last, abs_k, s);
  int rc;
  if (p->d.ndim == 3) {
    if ((rc = p->cops->col(p->colw, false, coly3d_args(p, A), s))) return rc;
    ColArgs ci = colx3d_args(p, A);
    ci.do_inv = 1;
    if ((rc = p->rops->col(p->colw_x, false, ci, s))) return rc;
    RowArgs a = mid_row(p, row3d_args(p, A), precision, last);
    if ((rc = p->tops->row(p->tops->p_row, 1, a, s))) return rc;
    if (last) return NLSE_OK;
    ColArgs cf = colx3d_args(p, A);
    cf.do_fwd = 1;
    return p->rops->col(p->colw_x, false, cf, s);
  }
  if ((rc = p->cops->col(p->colw, p->small, plan_col_args(p, A), s))) return rc;
  if (p->nlc.on) {
    const int64_t ds = p->drive ? abs_k : -1;
    if (precision == 0) {
      const bool rabi = p->rabi != nullptr && p->d.ncomp == 2;
      return nlc_apply(p, A, 1, last ? 0 : 1, p->nl[NLSE_SLOT_FULL], rabi, ds, s);
    }
    if ((rc = nlc_apply(p, A, 1, 0, p->nl[NLSE_SLOT_HALF_POST], false, ds, s))) return rc;
    return last ? NLSE_OK : nlc_apply(p, A, 0, 1, p->nl[NLSE_SLOT_HALF_PRE], false, -1, s);
  }
  RowArgs a = mid_row(p, plan_row_args(p, A), precision, last);
  a.has_drive = p->drive ? 1 : 0;
  if (p->drive) {
    a.drv_t0 = p->ft0[abs_k];
    a.drv_t1 = p->ft1[abs_k];
  }
  return launch_rows(p, p->d.ncomp, a, s);
}

static int run_checks(nlse_plan* p, void* A, int64_t nsteps, int precision, int64_t step0) {
  if (!p || !A || nsteps < 0 || (precision != 0 && precision != 1)) return fail(NLSE_ERR_ARG, "bad run arguments");
  int rc = check_ready(p, precision);
  if (rc) return rc;
  if (p->d.ndim == 3 && p->pkind == PROP_SEP3D && !p->pt)
    return fail(NLSE_ERR_STATE, "3-D temporal propagator factor not set");
  if (p->drive && p->d.ndim == 2 && step0 + nsteps > (int64_t)p->ft0.size())
    return fail(NLSE_ERR_ARG, "drive time profile too short (%zu for step %lld)", p->ft0.size(),
                (long long)(step0 + nsteps - 1));
  return NLSE_OK;
}

static void note_stream(nlse_plan* p, hipStream_t s) {
  p->last = s;
  p->ran = true;
}

int nlse_run(nlse_plan* p, void* A, int64_t nsteps, int precision, int64_t step0, void* stream) {
  int rc = run_checks(p, A, nsteps, precision, step0);
  if (rc || nsteps == 0) return rc;
  hipStream_t s = (hipStream_t)stream;
  note_stream(p, s);
  if (p->d.ndim == 1) return p->wide ? wrun1d(p, A, nsteps, precision, s) : run1d(p, A, nsteps, precision, s);
  if ((rc = chain_first(p, A, precision, s))) return rc;
  for (int64_t k = 0; k < nsteps; ++k)
    if ((rc = chain_step(p, A, precision, k == nsteps - 1, step0 + k, s))) return rc;
  return NLSE_OK;
}

// ------------------------------------------------------- graph replay
// The steady steps of a run are captured once per (field, precision,
// chunk, plan tables) into a hipGraph of `chunk` steps and replayed; the
// first sweep, the last step and the remainder are launched directly.  The
// key holds every pointer and flag the captured launches bake in, so a
// change of tables re-captures.
// Everything a captured step bakes into its launches: the field, every table
// and parameter pointer and the kinds that select kernels.  The values behind
// the pointers (propagator factors, nonlinear records, V) are read when the
// graph replays, so setters that rewrite a table in place keep the graph.
static std::vector<uint64_t> graph_key(const nlse_plan* p, const void* A, int precision, int64_t chunk) {
  std::vector<uint64_t> k = {(uint64_t)(uintptr_t)A, (uint64_t)precision, (uint64_t)chunk, (uint64_t)p->pkind,
                             (uint64_t)row_p(p), (uint64_t)nl_general(p),
                             (uint64_t)(uintptr_t)p->px, (uint64_t)(uintptr_t)p->py,
                             (uint64_t)(uintptr_t)p->ptab, (uint64_t)(uintptr_t)p->ptab128,
                             (uint64_t)(uintptr_t)p->pt, (uint64_t)(uintptr_t)p->V, (uint64_t)p->vkind,
                             (uint64_t)p->v_item_stride, (uint64_t)(uintptr_t)p->rabi,
                             (uint64_t)(uintptr_t)p->nlc.KT, (uint64_t)(uintptr_t)p->nlc.Z, (uint64_t)p->nlc.on,
                             (uint64_t)(uintptr_t)p->wn.K, (uint64_t)(uintptr_t)p->wn.Ic};
  for (void* q : p->nl) k.push_back((uint64_t)(uintptr_t)q);
  return k;
}

static void graph_free(nlse_plan* p) {
  if (p->gexec) (void)hipGraphExecDestroy(p->gexec);
  if (p->graph) (void)hipGraphDestroy(p->graph);
  p->gexec = nullptr;
  p->graph = nullptr;
  p->gkey.clear();
}

static int graph_capture(nlse_plan* p, void* A, int precision, int64_t chunk) {
  graph_free(p);
  if (!p->cap) HIP_TRY(hipStreamCreateWithFlags(&p->cap, hipStreamNonBlocking));
  HIP_TRY(hipStreamBeginCapture(p->cap, hipStreamCaptureModeThreadLocal));
  int rc = NLSE_OK;
  for (int64_t k = 0; k < chunk && !rc; ++k) rc = chain_step(p, A, precision, false, 0, p->cap);
  hipGraph_t g = nullptr;
  const hipError_t e = hipStreamEndCapture(p->cap, &g);
  if (rc) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  if (e != hipSuccess) return fail(NLSE_ERR_HIP, "hipStreamEndCapture failed: %s", hipGetErrorString(e));
  p->graph = g;
  HIP_TRY(hipGraphInstantiate(&p->gexec, g, nullptr, nullptr, 0));
  p->gkey = graph_key(p, A, precision, chunk);
  return NLSE_OK;
}

int nlse_run_graph(nlse_plan* p, void* A, int64_t nsteps, int precision, int64_t chunk, void* stream) {
  int rc = run_checks(p, A, nsteps, precision, 0);
  if (rc || nsteps == 0) return rc;
  if (chunk < 1) return fail(NLSE_ERR_ARG, "graph chunk must be >= 1");
  if (p->d.ndim == 1 || p->drive) return nlse_run(p, A, nsteps, precision, 0, stream);
  hipStream_t s = (hipStream_t)stream;
  note_stream(p, s);
  const int64_t steady = nsteps - 1;
  const int64_t reps = steady / chunk;
  if (reps > 0 && p->gkey != graph_key(p, A, precision, chunk) && (rc = graph_capture(p, A, precision, chunk)))
    return rc;
  if ((rc = chain_first(p, A, precision, s))) return rc;
  for (int64_t r = 0; r < reps; ++r) HIP_TRY(hipGraphLaunch(p->gexec, s));
  for (int64_t k = reps * chunk; k < nsteps; ++k)
    if ((rc = chain_step(p, A, precision, k == nsteps - 1, k, s))) return rc;
  return NLSE_OK;
}

int nlse_graph_prepare(nlse_plan* p, void* A, int precision, int64_t chunk, void* stream) {
  int rc = run_checks(p, A, 1, precision, 0);
  if (rc) return rc;
  if (chunk < 1) return fail(NLSE_ERR_ARG, "graph chunk must be >= 1");
  if (p->d.ndim == 1 || p->drive) return NLSE_OK;  // these plans run without a graph
  if (p->gkey != graph_key(p, A, precision, chunk) && (rc = graph_capture(p, A, precision, chunk))) return rc;
  // move the executable graph to the device now rather than at its first launch
  HIP_TRY(hipGraphUpload(p->gexec, (hipStream_t)stream));
  return NLSE_OK;
}

int nlse_run_pass(nlse_plan* p, void* A, int pass, int64_t count, int precision, void* stream) {
  if (!p || !A || count < 0 || pass < 0 || pass > 6 || (precision != 0 && precision != 1))
    return fail(NLSE_ERR_ARG, "bad run_pass arguments");
  if (p->d.ndim != 2) return fail(NLSE_ERR_ARG, "run_pass times the sweeps of 2-D plans");
  if (p->wide) return fail(NLSE_ERR_ARG, "run_pass times the sweeps of complex64 plans");
  int rc = check_ready(p, precision);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  note_stream(p, s);
  if (pass >= 2) {
    if (!p->nlc.on) return fail(NLSE_ERR_STATE, "passes 2-5 need a nonlocal response");
    if (pass == 4 && p->nlc.direct) return fail(NLSE_ERR_STATE, "direct nonlocal plans have no intensity sweep");
    const float inv_nx = (float)(1.0 / (double)p->d.nx);
    NlcArgs a = plan_nlc_args(p, A);
    a.out_scale = inv_nx;
    a.inverse_first = 1;
    a.forward_last = 1;
    a.nlp = precision == 1 ? p->nl[NLSE_SLOT_HALF_POST] : p->nl[NLSE_SLOT_FULL];
    ColArgs cz = nlc_col_args(p);
    cz.scale = (float)p->d.nx;
    for (int64_t k = 0; k < count && !rc; ++k) {
      if (pass == 2) rc = p->rops->nlc(1, a, s);
      else if (pass == 3) rc = band_launch(p, A, s);
      else if (pass == 4) rc = p->nlc.unpack ? p->nlc.zops->colu(cz, s) : p->nlc.zops->col(p->nlc.colw, false, cz, s);
      else if (pass == 6) rc = band_and_z(p, A, s, &cz);
      else rc = p->rops->nlc(2, a, s);
    }
    return rc;
  }
  // repeated sweeps of one kind: 1/N per sweep keeps the data at its scale
  // (in a run the 1/(NX NY) of the propagator normalises both transforms)
  RowArgs r = mid_row(p, plan_row_args(p, A), precision, false);
  r.out_scale = (float)(1.0 / (double)p->d.nx);
  ColArgs c = plan_col_args(p, A);
  c.scale = (float)(1.0 / (double)p->d.ny);
  for (int64_t k = 0; k < count; ++k) {
    rc = pass == 0 ? launch_rows(p, p->d.ncomp, r, s) : p->cops->col(p->colw, p->small, c, s);
    if (rc) return rc;
  }
  return NLSE_OK;
}

}  // extern "C"
