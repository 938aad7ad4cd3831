// Complex128 engine: per-length launchers of the wide kernels (wide.hpp),
// the 2-D nonlocal convolution and the complex128 reductions.
#include <hip/hip_runtime.h>

#include <map>
#include <mutex>

#include "lines.hpp"
#include "wide.hpp"

namespace nlse {

namespace {

// Kernels that need more than 64 KiB of dynamic LDS raise their limit once
// per device.
int lds_limit(const void* fn, size_t bytes) {
  if (bytes <= 64 * 1024) return NLSE_OK;
  if (bytes > 160 * 1024) return fail(NLSE_ERR_ARG, "complex128 kernel needs %zu bytes of LDS", bytes);
  static std::mutex mu;
  static std::map<std::pair<int, const void*>, bool> done;
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(mu);
  auto key = std::make_pair(dev, fn);
  if (!done[key]) {
    HIP_TRY(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    done[key] = true;
  }
  return NLSE_OK;
}

// Eight points per thread: radix-8 stages (the FP64 natural set of a
// two-component thread is then 64 VGPRs).
template <int N>
constexpr int wp() {
  return 8;
}

template <int N, int G>
int wrow_launch_g(const WRowArgs& a, hipStream_t s) {
  constexpr int P = wp<N>(), T = N / P;
  constexpr int L = T >= 128 / G ? 1 : (128 / G) / T;
  const size_t bytes = (size_t)L * G * WLine<N>::SIZE * sizeof(double2);
  auto fn = k_wrow<N, P, L, G>;
  int rc = lds_limit((const void*)fn, bytes);
  if (rc) return rc;
  const int64_t blocks = (a.ngroups + L - 1) / L;
  hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3(L * T), bytes, s, a);
  return launch_status("k_wrow");
}

template <int N>
int wrow_launch(int G, const WRowArgs& a, hipStream_t s) {
  return G == 1 ? wrow_launch_g<N, 1>(a, s) : wrow_launch_g<N, 2>(a, s);
}

template <int N, int WT>
int wcol_launch_w(const WColArgs& a, hipStream_t s) {
  constexpr int P = wp<N>(), T = N / P;
  const size_t bytes = (size_t)WT * ColLine<N, WT, double2>::SIZE * sizeof(double2);
  auto fn = k_wcol<N, P, WT>;
  int rc = lds_limit((const void*)fn, bytes);
  if (rc) return rc;
  const int64_t blocks = a.nslabs * (a.NX / WT);
  hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3(WT * T), bytes, s, a);
  return launch_status("k_wcol");
}

// Column tile: 8 adjacent columns (128-byte row segments) where the block
// stays within 512 threads and 150 KiB of LDS and the columns divide.
template <int N>
int wcol_launch(const WColArgs& a, hipStream_t s) {
  constexpr int T = N / wp<N>();
  constexpr size_t LINEB = WLine<N>::SIZE * sizeof(double2);
  auto fits = [&](int wt) { return wt * T <= 512 && wt * LINEB <= 150 * 1024 && a.NX % wt == 0; };
  if (fits(8)) return wcol_launch_w<N, 8>(a, s);
  if (fits(4)) return wcol_launch_w<N, 4>(a, s);
  if (fits(2)) return wcol_launch_w<N, 2>(a, s);
  return wcol_launch_w<N, 1>(a, s);
}

template <int N, int G>
int wline1d_launch_g(const WLine1DArgs& a, hipStream_t s) {
  constexpr int P = wp<N>(), T = N / P;
  constexpr int L = T >= 256 / G ? 1 : (256 / G) / T;
  const size_t bytes = (size_t)L * G * WLine<N>::SIZE * sizeof(double2);
  auto fn = k_wline1d<N, P, L, G>;
  int rc = lds_limit((const void*)fn, bytes);
  if (rc) return rc;
  const int64_t blocks = (a.ngroups + L - 1) / L;
  hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3(L * T), bytes, s, a);
  return launch_status("k_wline1d");
}

template <int N>
int wline1d_launch(int G, const WLine1DArgs& a, hipStream_t s) {
  return G == 1 ? wline1d_launch_g<N, 1>(a, s) : wline1d_launch_g<N, 2>(a, s);
}

template <int N>
WideOps make_wide_ops() {
  return WideOps{&get_twiddles<N>, &wrow_launch<N>, &wcol_launch<N>, &wline1d_launch<N>};
}

}  // namespace

__global__ __launch_bounds__(WCONV_TILE* WCONV_TILE) void k_wconv2d(WConvArgs a) {
  extern __shared__ double wconv_sm[];
  const int tilesx = (a.nx + WCONV_TILE - 1) / WCONV_TILE;
  const int tilesy = (a.ny + WCONV_TILE - 1) / WCONV_TILE;
  const int64_t b = blockIdx.x;
  const int64_t slab = b / ((int64_t)tilesx * tilesy);
  const int tb = (int)(b % ((int64_t)tilesx * tilesy));
  const int y0 = (tb / tilesx) * WCONV_TILE, x0 = (tb % tilesx) * WCONV_TILE;
  const int ty = threadIdx.x / WCONV_TILE, tx = threadIdx.x % WCONV_TILE;
  const int rh = a.kh / 2, rw = a.kw / 2;
  const double* I = a.I + slab * (int64_t)a.ny * a.nx;
  const int y = y0 + ty, x = x0 + tx;
  double acc = 0.0;
  if (a.lds) {
    const int hh = WCONV_TILE + 2 * rh, hw = WCONV_TILE + 2 * rw;
    for (int i = threadIdx.x; i < hh * hw; i += WCONV_TILE * WCONV_TILE) {
      const int sy = y0 - rh + i / hw, sx = x0 - rw + i % hw;
      wconv_sm[i] = (sy >= 0 && sy < a.ny && sx >= 0 && sx < a.nx) ? I[(int64_t)sy * a.nx + sx] : 0.0;
    }
    __syncthreads();
    // I(y + rh - ka, x + rw - kb) sits at tile row ty + 2 rh - ka, column tx + 2 rw - kb
    for (int ka = 0; ka < a.kh; ++ka) {
      const double* row = wconv_sm + (ty + 2 * rh - ka) * hw + tx + 2 * rw;
      const double* kr = a.K + (int64_t)ka * a.kw;
      for (int kb = 0; kb < a.kw; ++kb) acc = fma(kr[kb], row[-kb], acc);
    }
  } else if (y < a.ny && x < a.nx) {
    for (int ka = 0; ka < a.kh; ++ka) {
      const int sy = y + rh - ka;
      if (sy < 0 || sy >= a.ny) continue;
      const double* kr = a.K + (int64_t)ka * a.kw;
      for (int kb = 0; kb < a.kw; ++kb) {
        const int sx = x + rw - kb;
        if (sx >= 0 && sx < a.nx) acc = fma(kr[kb], I[(int64_t)sy * a.nx + sx], acc);
      }
    }
  }
  if (y < a.ny && x < a.nx) a.Ic[slab * (int64_t)a.ny * a.nx + (int64_t)y * a.nx + x] = acc;
}

// Ic on the FP64 matrix cores: a block of four waves owns 32 x 32 outputs,
// one 16 x 16 sub-tile per wave.  With the intensities staged from (y0 -
// rh, x0 - rw), kernel row u (flipped: KF[u][v] = K[kh-1-u][kw-1-v])
// contributes out[Y][X] += sum_j S[Y + u][X0 + j] KF[u][j - X] to the
// sub-tile at staged column X0: NCH products of 16 x 16 x 4
// (v_mfma_f64_16x16x4_f64) with A the staged rows and B a Toeplitz slice
// of the row, read from KP[u][t] = KF[u][t - 16] (zero outside [16, 16 +
// 2 rw]) at t = 4c + k - X + 16.  PAIR: rows u and kh-1-u are equal, their
// staged rows are added and take one product.  The next row's operands are
// loaded while the current row's products run.  Sums stay in FP64.
constexpr int WCONV_MT = 32;  // output tile edge (2 x 2 sub-tiles)

inline int wconv_mfma_pitch(int ws) { return ws + ((17 - ws % 16) % 16); }  // >= ws, = 1 mod 16 doubles
inline size_t wconv_mfma_lds(int rh, int rw, int kh) {
  const int nch = wconv_mfma_chunks(rw);
  const int ws = 16 + 4 * nch;
  return ((size_t)(WCONV_MT + 2 * rh) * wconv_mfma_pitch(ws) + (size_t)kh * (4 * nch + 16)) * sizeof(double);
}

typedef double wconv_d4 __attribute__((ext_vector_type(4)));

template <int NCH, bool PAIR>
__global__ __launch_bounds__(256) void k_wconv2d_mfma(WConvArgs a, int pitch, int tilesx, int tilesy) {
  extern __shared__ double wconv_sm[];
  constexpr int NTH = 256, STG = 8;
  constexpr int WS = 16 + 4 * NCH;  // staged columns (zeros beyond the halo)
  const int64_t per = (int64_t)tilesx * tilesy;
  const int64_t slab = blockIdx.x / per;
  const int tb = (int)(blockIdx.x % per);
  const int y0 = (tb / tilesx) * WCONV_MT, x0 = (tb % tilesx) * WCONV_MT;
  const int rh = a.kh / 2, rw = a.kw / 2, kpw = a.kpw;
  const int hrows = WCONV_MT + 2 * rh, wcols = WCONV_MT + 2 * rw;
  double* img = wconv_sm;
  double* kp = wconv_sm + (size_t)hrows * pitch;
  const double* I = a.I + slab * (int64_t)a.ny * a.nx;
  const int tid = threadIdx.x;
  const int nkp = a.kh * kpw;
  for (int e0 = 0; e0 < nkp; e0 += STG * NTH) {
    double kv[STG];
#pragma unroll
    for (int k = 0; k < STG; ++k) {
      const int e = e0 + k * NTH + tid;
      kv[k] = a.KP[e < nkp ? e : 0];
    }
#pragma unroll
    for (int k = 0; k < STG; ++k) {
      const int e = e0 + k * NTH + tid;
      if (e < nkp) kp[e] = kv[k];
    }
  }
  const int total = hrows * WS;
  for (int e0 = 0; e0 < total; e0 += STG * NTH) {
    double q[STG];
    int at[STG];
#pragma unroll
    for (int k = 0; k < STG; ++k) {
      const int e = e0 + k * NTH + tid;
      const int i = e / WS, j = e - i * WS;
      const int y = y0 - rh + i, x = x0 - rw + j;
      const bool ok = e < total && j < wcols && y >= 0 && y < a.ny && x >= 0 && x < a.nx;
      q[k] = I[ok ? (int64_t)y * a.nx + x : 0];
      q[k] = ok ? q[k] : 0.0;
      at[k] = e < total ? i * pitch + j : -1;
    }
#pragma unroll
    for (int k = 0; k < STG; ++k)
      if (at[k] >= 0) img[at[k]] = q[k];
  }
  __syncthreads();
  const int lane = tid & 63, wv = tid >> 6;
  const int sy = wv >> 1, sx = wv & 1;
  if (y0 + sy * 16 >= a.ny || x0 + sx * 16 >= a.nx) return;
  const int m = lane & 15, k = lane >> 4;
  const double* pa = img + (sy * 16 + m) * pitch + sx * 16 + k;
  const double* pb = kp + 16 + k - m;
  wconv_d4 d0 = {0.0, 0.0, 0.0, 0.0}, d1 = {0.0, 0.0, 0.0, 0.0};
  double xa[NCH], xc[NCH], xb[NCH], ya[NCH], yc[NCH], yb[NCH];
  auto load = [&](double (&ra)[NCH], double (&rc)[NCH], double (&rb)[NCH], int u) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      ra[c] = pa[u * pitch + 4 * c];
      if (PAIR) rc[c] = pa[(a.kh - 1 - u) * pitch + 4 * c];
      rb[c] = pb[u * kpw + 4 * c];
    }
  };
  auto step = [&](const double (&ra)[NCH], const double (&rc)[NCH], const double (&rb)[NCH], bool pair) {
#pragma unroll
    for (int c = 0; c < NCH; c += 2) {
      const double a0 = pair ? ra[c] + rc[c] : ra[c];
      const double a1 = pair ? ra[c + 1] + rc[c + 1] : ra[c + 1];
      d0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, rb[c], d0, 0, 0, 0);
      d1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, rb[c + 1], d1, 0, 0, 0);
    }
  };
  // row steps: PAIR takes rows (t, kh-1-t) for t < rh, then the middle row
  // rh alone; otherwise every row alone
  const int nsteps = PAIR ? rh + 1 : a.kh;
  auto is_pair = [&](int t) { return PAIR && t < rh; };
  load(xa, xc, xb, 0);
  int t = 0;
  for (; t + 2 <= nsteps; t += 2) {
    load(ya, yc, yb, t + 1);
    step(xa, xc, xb, is_pair(t));
    load(xa, xc, xb, t + 2 < nsteps ? t + 2 : nsteps - 1);
    step(ya, yc, yb, is_pair(t + 1));
  }
  if (t < nsteps) step(xa, xc, xb, is_pair(t));
  // D of the FP64 16 x 16 x 4 product: register i of a lane holds row
  // 4 * i + lane / 16, column lane % 16 (unlike the FP32 product, whose
  // lane holds four consecutive rows)
  const int x = x0 + sx * 16 + m;
  if (x >= a.nx) return;
  double* out = a.Ic + slab * (int64_t)a.ny * a.nx;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int y = y0 + sy * 16 + 4 * i + k;
    if (y < a.ny) out[(int64_t)y * a.nx + x] = d0[i] + d1[i];
  }
}

template <int NCH, bool PAIR>
int wconv_mfma_launch(const WConvArgs& a, hipStream_t s) {
  const int rh = a.kh / 2, rw = a.kw / 2;
  const int pitch = wconv_mfma_pitch(16 + 4 * NCH);
  const size_t bytes = wconv_mfma_lds(rh, rw, a.kh);
  const int tilesx = (a.nx + WCONV_MT - 1) / WCONV_MT, tilesy = (a.ny + WCONV_MT - 1) / WCONV_MT;
  auto fn = k_wconv2d_mfma<NCH, PAIR>;
  int rc = lds_limit((const void*)fn, bytes);
  if (rc) return rc;
  hipLaunchKernelGGL(fn, dim3((unsigned)(a.nslabs * tilesx * tilesy)), dim3(256), bytes, s, a, pitch, tilesx,
                     tilesy);
  return launch_status("k_wconv2d_mfma");
}

template <bool PAIR>
int wconv_mfma_dispatch(const WConvArgs& a, hipStream_t s) {
  switch (wconv_mfma_chunks(a.kw / 2)) {
    case 4: return wconv_mfma_launch<4, PAIR>(a, s);
    case 6: return wconv_mfma_launch<6, PAIR>(a, s);
    case 8: return wconv_mfma_launch<8, PAIR>(a, s);
    case 10: return wconv_mfma_launch<10, PAIR>(a, s);
    case 12: return wconv_mfma_launch<12, PAIR>(a, s);
    default: return fail(NLSE_ERR_ARG, "kernel too wide for the matrix-core convolution");
  }
}

const WideOps* wide_ops(int64_t n) {
  static const WideOps ops[] = {make_wide_ops<8>(),   make_wide_ops<16>(),  make_wide_ops<32>(),
                                make_wide_ops<64>(),  make_wide_ops<128>(), make_wide_ops<256>(),
                                make_wide_ops<512>(), make_wide_ops<1024>(), make_wide_ops<2048>(),
                                make_wide_ops<4096>()};
  if (!is_pow2(n) || n < 8 || n > 4096) return nullptr;
  int l = 0;
  while ((int64_t(1) << l) < n) ++l;
  return &ops[l - 3];
}

bool wide_conv2d_mfma_fits(int kh, int kw) {
  return wconv_mfma_chunks(kw / 2) <= WCONV_MFMA_MAX_CHUNKS && wconv_mfma_lds(kh / 2, kw / 2, kh) <= 64 * 1024;
}

int wide_conv2d(const WConvArgs& a0, hipStream_t s) {
  if (a0.KP) return a0.pair ? wconv_mfma_dispatch<true>(a0, s) : wconv_mfma_dispatch<false>(a0, s);
  WConvArgs a = a0;
  const int hh = WCONV_TILE + 2 * (a.kh / 2), hw = WCONV_TILE + 2 * (a.kw / 2);
  const size_t bytes = (size_t)hh * hw * sizeof(double);
  a.lds = bytes <= 150 * 1024 ? 1 : 0;
  if (a.lds) {
    int rc = lds_limit((const void*)k_wconv2d, bytes);
    if (rc) return rc;
  }
  const int64_t tiles =
      (int64_t)((a.ny + WCONV_TILE - 1) / WCONV_TILE) * ((a.nx + WCONV_TILE - 1) / WCONV_TILE);
  hipLaunchKernelGGL(k_wconv2d, dim3((unsigned)(a.nslabs * tiles)), dim3(WCONV_TILE * WCONV_TILE),
                     a.lds ? bytes : 0, s, a);
  return launch_status("k_wconv2d");
}

}  // namespace nlse

// ------------------------------------------- complex128 reductions (C ABI)
namespace {

constexpr int WSUM_THREADS = 256;
constexpr int64_t WSUM_CHUNK = 4096;

// Per-item FP64 sums of |A|^2 over chunks of WSUM_CHUNK points, then one
// block per item adds its chunk partials in order.
__global__ __launch_bounds__(WSUM_THREADS) void k_wsumsq_part(const double2* A, int64_t isz, int64_t nchunks,
                                                              double* part) {
  const int64_t item = blockIdx.x / nchunks, ch = blockIdx.x % nchunks;
  const double2* a = A + item * isz;
  const int64_t beg = ch * WSUM_CHUNK, end = beg + WSUM_CHUNK < isz ? beg + WSUM_CHUNK : isz;
  double acc = 0.0;
  for (int64_t i = beg + threadIdx.x; i < end; i += WSUM_THREADS) acc = fma(a[i].x, a[i].x, fma(a[i].y, a[i].y, acc));
  __shared__ double red[WSUM_THREADS];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = WSUM_THREADS / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(WSUM_THREADS) void k_wsum_final(const double* part, int64_t nchunks, double* out) {
  const double* p = part + blockIdx.x * nchunks;
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < nchunks; i += WSUM_THREADS) acc += p[i];
  __shared__ double red[WSUM_THREADS];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = WSUM_THREADS / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = red[0];
}

__global__ void k_wscale(double2* A, int64_t items, int64_t isz, int64_t str, nlse_bparam sp) {
  const int64_t n = items * isz;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t item = i / isz, j = i - item * isz;
    const double f = sp.v_dev[item * sp.stride];
    double2& a = A[item * str + j];
    a = make_double2(a.x * f, a.y * f);
  }
}

// delta_n of callbacks.py:57-82 on a complex128 field, in FP64 (the same
// operator order as the complex64 kernel: the imaginary part is scaled by
// c eps0/2 alone, callbacks.py:109).
__device__ __forceinline__ double wdelta_n_point(double2 a, double qc, double qe, double coef, double isat) {
  const double yy = a.y * a.y;
  const double im = qc != 0.0 ? ((yy * qc) * qe) * 0.5 : yy;
  const double q = a.x * a.x + im;
  return (coef * q) / (1.0 + q / isat);
}

__device__ __forceinline__ double wbp(const nlse_bparam& p, int64_t item) { return p.v_dev[item * p.stride]; }

__global__ void k_wdelta_n(const double2* A, int64_t items, int64_t isz, double qc, double qe, nlse_bparam coef,
                           nlse_bparam isat, double* out) {
  const int64_t n = items * isz;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t item = i / isz;
    out[i] = wdelta_n_point(A[i], qc, qe, wbp(coef, item), wbp(isat, item));
  }
}

__global__ __launch_bounds__(WSUM_THREADS) void k_wdelta_n_max(const double2* A, int64_t items, int64_t isz,
                                                               double qc, double qe, nlse_bparam coef,
                                                               nlse_bparam isat, double* part) {
  const int64_t n = items * isz;
  double m = -__builtin_inf();
  for (int64_t i = blockIdx.x * (int64_t)WSUM_THREADS + threadIdx.x; i < n; i += (int64_t)gridDim.x * WSUM_THREADS) {
    const int64_t item = i / isz;
    m = fmax(m, wdelta_n_point(A[i], qc, qe, wbp(coef, item), wbp(isat, item)));
  }
  __shared__ double red[WSUM_THREADS];
  red[threadIdx.x] = m;
  __syncthreads();
  for (int w = WSUM_THREADS / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(WSUM_THREADS) void k_wmax_final(const double* part, int64_t n, double* out) {
  double m = -__builtin_inf();
  for (int64_t i = threadIdx.x; i < n; i += WSUM_THREADS) m = fmax(m, part[i]);
  __shared__ double red[WSUM_THREADS];
  red[threadIdx.x] = m;
  __syncthreads();
  for (int w = WSUM_THREADS / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = red[0];
}

// One drive term on a complex128 cavity field (see nlse::wdrive).
__global__ void k_wdrive(double2* A, int64_t items, int64_t isz, int64_t str, const float2* Fr, float2 ft, float dz) {
  const int64_t n = items * isz;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t item = i / isz, j = i - item * isz;
    double2& a = A[item * str + j];
    a = nlse::wdrive(a, Fr[j], ft, dz);
  }
}

unsigned wgrid(int64_t n) {
  int64_t b = (n + 255) / 256;
  if (b > 65536) b = 65536;
  if (b < 1) b = 1;
  return (unsigned)b;
}

}  // namespace

extern "C" {

int nlse_sumsq_c128(const void* A, int64_t items, int64_t isz, double* out, void* stream) {
  using namespace nlse;
  if (!A || !out || items < 1 || isz < 1) return fail(NLSE_ERR_ARG, "bad sumsq_c128 arguments");
  const int64_t nchunks = (isz + WSUM_CHUNK - 1) / WSUM_CHUNK;
  double* part = nullptr;
  int rc = scratch_doubles((size_t)(items * nchunks), &part);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(k_wsumsq_part, dim3((unsigned)(items * nchunks)), dim3(WSUM_THREADS), 0, s,
                     (const double2*)A, isz, nchunks, part);
  hipLaunchKernelGGL(k_wsum_final, dim3((unsigned)items), dim3(WSUM_THREADS), 0, s, (const double*)part, nchunks,
                     out);
  return launch_status("k_wsumsq");
}

int nlse_scale_c128(void* A, int64_t items, int64_t isz, int64_t str, nlse_bparam sp, void* stream) {
  using namespace nlse;
  if (!A || items < 1 || isz < 1 || str < isz || !sp.v_dev) return fail(NLSE_ERR_ARG, "bad scale_c128 arguments");
  hipLaunchKernelGGL(k_wscale, dim3(wgrid(items * isz)), dim3(256), 0, (hipStream_t)stream, (double2*)A, items, isz,
                     str, sp);
  return launch_status("k_wscale");
}

int nlse_cavity_drive_c128(void* A, int64_t items, int64_t isz, int64_t str, const void* Fr, float ft_re,
                           float ft_im, double dz, void* stream) {
  using namespace nlse;
  if (!A || !Fr || items < 0 || isz < 0 || str < 0) return fail(NLSE_ERR_ARG, "bad cavity_drive_c128 arguments");
  const int64_t n = items * isz;
  if (n == 0) return NLSE_OK;
  hipLaunchKernelGGL(k_wdrive, dim3(wgrid(n)), dim3(256), 0, (hipStream_t)stream, (double2*)A, items, isz, str,
                     (const float2*)Fr, make_float2(ft_re, ft_im), (float)dz);
  return launch_status("k_wdrive");
}

int nlse_delta_n_c128(const void* A, int64_t items, int64_t isz, double qc, double qe, nlse_bparam coef,
                      nlse_bparam isat, double* out, void* stream) {
  using namespace nlse;
  if (!A || !out || items < 1 || isz < 1 || !coef.v_dev || !isat.v_dev)
    return fail(NLSE_ERR_ARG, "bad delta_n_c128 arguments");
  hipLaunchKernelGGL(k_wdelta_n, dim3(wgrid(items * isz)), dim3(256), 0, (hipStream_t)stream, (const double2*)A,
                     items, isz, qc, qe, coef, isat, out);
  return launch_status("k_wdelta_n");
}

int nlse_delta_n_max_c128(const void* A, int64_t items, int64_t isz, double qc, double qe, nlse_bparam coef,
                          nlse_bparam isat, double* out, void* stream) {
  using namespace nlse;
  if (!A || !out || items < 1 || isz < 1 || !coef.v_dev || !isat.v_dev)
    return fail(NLSE_ERR_ARG, "bad delta_n_max_c128 arguments");
  const unsigned g = wgrid(items * isz) > 1024 ? 1024 : wgrid(items * isz);
  double* part = nullptr;
  int rc = scratch_doubles(g, &part);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(k_wdelta_n_max, dim3(g), dim3(WSUM_THREADS), 0, s, (const double2*)A, items, isz, qc, qe, coef,
                     isat, part);
  hipLaunchKernelGGL(k_wmax_final, dim3(1), dim3(WSUM_THREADS), 0, s, (const double*)part, (int64_t)g, out);
  return launch_status("k_wdelta_n_max");
}

}  // extern "C"
