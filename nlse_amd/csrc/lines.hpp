// Per-line-length kernel dispatch: twiddle tables, launch configurations
// and launchers of every kernel templated on the line length N.  Each
// lines_*.hip translation unit instantiates make_ops<N> for its lengths, so
// the kernels of different lengths compile in parallel.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "common.hpp"
#include "passes_2d.hpp"

namespace nlse {

// Runtime-N dispatch table.  p: points per thread (radix plan) of a sweep.
struct LineOps {
  int (*twiddles)(const double2**);
  // x rows (G = 1, or component pairs G = 2) with p points per thread: p_row
  // by default, p_row_alt on request, p_row_small for small fields, p_row_large
  // for stacks of LARGE_STACK points
  int (*row)(int, int, const RowArgs&, hipStream_t);
  int p_row, p_row_alt, p_row_small, p_row_large;
  int (*line1d)(int, const Line1DArgs&, hipStream_t);
  int (*nlc)(int, const NlcArgs&, hipStream_t);
  // columns: tile width, small-field plan or not
  int (*col)(int, bool, const ColArgs&, hipStream_t);
  int (*colw)(int64_t, int, bool);
  int p_col, p_col_small;
  // intensity column sweep + band pass in one launch (1: not available for
  // this tile width, use the separate launches)
  int (*colz_band)(int, const ColArgs&, const BandArgs&, int, size_t, int64_t, hipStream_t);
  // full-torus intensity convolution of row-pair-packed spectra (k_colu)
  int (*colu)(const ColArgs&, hipStream_t);
};

// ------------------------------------------------------ twiddle tables
// One table per (device, line length): the ratio pairs of the stages of Plan<N,
// P> for P = 16, 8, 4 in that order (rt_base), evaluated and stored in FP64.

// Ratio pairs {c, s/c} of the stages of Plan<N, P> (rt_offset): for the levels r
// = R, R/2, .., 2 of a stage of radix R, w^(R/r) W_r^k with k < max(1, r/4) and
// w = exp(-2 pi i jm / (Ns R)), entry [i * Ns + jm] for the i-th pair.  The ratio
// is that of the exact sine to the rounded cosine, which the butterfly multiplies
// by: each part of a twiddle is rounded once.
template <int N, int P>
void build_ratio_twiddles(double2* rt) {
  if constexpr (P <= N) {
    using PL = Plan<N, P>;
    for (int s = 1; s < PL::NSTAGES; ++s) {
      const int R = PL::radix(s), NS = PL::ns(s);
      double2* out = rt + rt_base(N, P) + rt_offset(N, P, s);
      int i = 0;
      for (int r = R; r >= 2; r /= 2)
        for (int k = 0; k < (r >= 4 ? r / 4 : 1); ++k, ++i)
          for (int jm = 0; jm < NS; ++jm) {
            // angle / (-2 pi) = jm / (NS r) + k / r, in lowest terms of NS r
            const long double pi = 3.14159265358979323846264338327950288L;
            const long double ang = -2 * pi * (long double)(jm + (long)k * NS) / ((long double)NS * r);
            double c = (double)cosl(ang);
            if (std::fabs(c) < 1e-17) c = 6e-17;  // (a quarter turn: see bf2)
            out[i * NS + jm] = make_double2(c, (double)(sinl(ang) / (long double)c));
          }
    }
  }
}

template <int N>
std::vector<double2> build_twiddles() {
  std::vector<double2> tw(rt_size(N) > 0 ? rt_size(N) : 1, make_double2(0.0, 0.0));
  build_ratio_twiddles<N, 16>(tw.data());
  build_ratio_twiddles<N, 8>(tw.data());
  build_ratio_twiddles<N, 4>(tw.data());
  return tw;
}

static std::mutex g_tw_mu;
static std::map<std::pair<int, int>, double2*> g_tw;  // (device, N) -> table

template <int N>
static int get_twiddles(const double2** out) {
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_tw_mu);
  auto key = std::make_pair(dev, N);
  auto it = g_tw.find(key);
  if (it != g_tw.end()) {
    *out = it->second;
    return NLSE_OK;
  }
  std::vector<double2> h = build_twiddles<N>();
  double2* d = nullptr;
  HIP_TRY(hipMalloc(&d, h.size() * sizeof(double2)));
  HIP_TRY(hipMemcpy(d, h.data(), h.size() * sizeof(double2), hipMemcpyHostToDevice));
  g_tw[key] = d;
  *out = d;
  return NLSE_OK;
}

// -------------------------------------------------- kernel dispatchers
// Points per thread (P) of the nonlocal row kernels.  A smaller P puts more
// lanes on a line (a shorter chain of instructions per lane, what a field of
// few lines waits for), a larger P has fewer stages, i.e. fewer exchanges and
// conversions.  Nonlocal step with P = 4 / 8 / 16 in both kernels: 256^2 23.0 /
// 25.8 / 31.5 us, 128^2 22.0 / 24.4 / 30.9, 256 fields of 256^2 309 / 307 / 313;
// k_nlc_nl at 2048 points keeps 8 (26.7 against 29.6 us), k_nlc_z takes 16 there
// (90.7 against 91.9 us a step).
constexpr int pick_p(int n, int p8_upto) { return n <= 256 ? (n >= 32 ? 4 : 8) : (n < p8_upto ? 8 : 16); }
constexpr int lines_per_block(int threads, int t) { return threads / t >= 1 ? threads / t : 1; }

// Fields of at most this many points (all items and components) take the
// small-field plans of LineCfg: their sweeps are a few waves per CU, bound by
// the length of one lane's work.  One step (row + column sweep) of a local
// field, default against small-field plan: 256^2 14.0 -> 7.8 us; at the limit 4 x
// 256^2 11.0 -> 9.0, 16 x 128^2 10.6 -> 8.8, 64 x 64^2 11.8 -> 7.5, 512^2 11.5 ->
// 10.3.  Past it the plans cross at other sizes for each grid (24 x 128^2 11.2 /
// 9.8, 5 x 256^2 11.1 / 10.8, 4 x 512^2 14.9 / 14.1, but 3 x 512^2 14.1 / 15.1, 24 x
// 256^2 17.8 / 19.2): the line lies where all of them still gain.
constexpr int64_t SMALL_FIELD = 1 << 18;

// Fields of at most this many bytes are written through to memory: a kernel's
// end then has no dirty L2 lines left to write back before the next sweep,
// whose reads come from other XCDs, may start.  Step of a local field, stores
// back / through: 1024^2 25.2 -> 21.0 us, 2 x 1024^2 46.2 -> 31.8 us, 2048^2
// 59.7 -> 56.4 us, 6 x 1024^2 (48 MiB) 62.7 / 61.4; beyond the limit 7 x 1024^2
// 69.1 / 74.5, 12 x 1024^2 109 / 112, 28 x 1024^2 (235 MB) 280 / 298 us.
// Stores of fewer contiguous bytes than a line leave in as many pieces: 64 bytes
// (rows of 8 lanes, tiles of 8 columns) go through up to WRITE_THROUGH, 16 and 32
// up to WRITE_THROUGH_NARROW, single points never.  Whole calls with all stores
// back / through / by this rule: 8-byte rows, 3-D 512 x 512 x 16 2.74 / 3.43 / 2.65
// ms, 200 fields of 256 x 16 2.38 / 2.60 / 2.13; 8-byte columns, 4096 x 64 2.02 /
// 2.73 / 2.01, 4096 x 256 3.20 / 3.58 / 2.86; 16-byte rows, 512 x 256 x 32 (32 MiB)
// 2.29 / 2.62 / 2.25; 32-byte columns, 16 of 4096 x 64 (32 MiB) 4.63 / 5.74 / 4.63,
// 1024^2 (8 MiB) 25.2 / 21.0 / 21.0 us a step; 16-byte columns, cnlse 4096 x 256 (16
// MiB) 3.16 / 3.05 / 3.05.
constexpr int64_t WRITE_THROUGH = 48 << 20, WRITE_THROUGH_NARROW = 16 << 20;
constexpr int through_level(int64_t bytes) {
  return bytes <= WRITE_THROUGH_NARROW ? 2 : (bytes <= WRITE_THROUGH ? 1 : 0);
}

// Stacks of one-component fields of at least this many points take p_row_large
// in their row sweeps: 16 points per lane on 1024-point rows exchange once less
// through LDS (24 instead of 32 bytes written per point and sweep), which pays
// where enough waves hide one lane's longer chain.  Row sweep with 8 / 16
// points: one 1024^2 field 8.9 / 10.8 us, 2 fields 13.8 / 12.6, 4 fields 21.6 /
// 19.8, 28 fields 127 / 119 us (512-point rows: no difference).  A single field
// keeps its plan whatever its size: an uneven batch computes it in that plan.
constexpr int64_t LARGE_STACK = 1 << 21;

template <int N>
struct LineCfg {
  // column sweeps
  static constexpr int P = N >= 16 ? 16 : N;
  static constexpr int T = N / P;
  // small fields: up to 256 points 4 per thread, FP64 exchanges (one rounding
  // per transform, so the extra stages round nothing); 512 points 8
  static constexpr int PS = N <= 256 ? 4 : (N == 512 ? 8 : P);
  static constexpr int ARS = N <= 256 ? F64X : F64;
  // x rows
  static constexpr int PR = (N == 512 || N == 1024) ? 8 : P;
  static constexpr int PRS = N <= 256 ? 4 : PR;
  static constexpr int PRL = N == 1024 ? 16 : PR;
  // nonlocal row kernels (a thread group per line pair); up to NLC_FEW points
  // in the first lines of all pairs, lines of 512 and 1024 points take 4 per
  // thread: nonlocal step with 8 / 4, 1024^2 42.8 / 40.3 us, 512^2 27.9 / 26.8,
  // 4 fields of 512^2 39.8 / 39.1, 8 fields 53.4 / 55.8, 4 of 1024^2 92.9 / 96.7
  static constexpr int PZ = pick_p(N, 2048);
  static constexpr int PN = pick_p(N, 1 << 30);
  static constexpr int64_t NLC_FEW = N == 512 || N == 1024 ? 1 << 19 : 0;
  // whole 1-D runs; up to LINES1S lines (or line pairs), which leave a CU one
  // or two lines, take the small plan: few points per lane, FP64 exchanges
  // up to 1024 points, twiddles kept.  Per step, default against small plan:
  // 250 lines of 1024 4.2 -> 3.0 us (pairs 11.3 -> 5.9), 200 of 256 3.1 ->
  // 1.25, of 512 3.9 -> 2.0, of 2048 4.9 -> 3.7 us.  300 steps at and past the
  // limits, default / small plan, ms: 64 points 8192 lines 1.35 / 0.93, 12000 1.44 /
  // 1.32; 256: 2048 1.26 / 0.97, 2500 1.27 / 1.38; 512: 1024 1.52 / 1.05, 2048
  // 1.57 / 1.84, 2500 2.79 / 2.57; 1024: 512 1.57 / 1.43, 600 1.56 / 2.12; 2048: 256
  // 1.88 / 1.33, 300 1.88 / 2.39
  static constexpr int P1 = N >= 16 ? 16 : N;
  static constexpr int LPB1D1 = lines_per_block(256, N / P1);
  static constexpr int LPB1D2 = lines_per_block(128, N / P1);
  static constexpr int P1S = (N <= 256 || N == 1024) ? 4 : ((N == 512 || N == 2048) ? 8 : P1);
  static constexpr int AR1S = N <= 1024 ? F64X : F64;
  static constexpr int64_t LINES1S = P1S == P1 ? 0 : (N <= 1024 ? 1 << 17 : 1 << 16) / (N / P1S);
  // default column tile: 8 columns (64-byte row segments; narrower tiles
  // read 32-byte segments: 12.9 us against 8.5 us for an in-place copy of
  // a 2048^2 field); 2-D plans narrow it for small fields (nlse_plan_create)
  static constexpr int WDEF = 8;
};

// Column tile of W columns with PC points per thread: WT threads across, G =
// W/WT columns per thread, LDS rounds of GR columns per thread column.  One
// column per thread needs at most 128 VGPRs and takes blocks of up to 1024
// threads; several columns per thread take 512.
template <int N, int W, int PC, int AR>
struct ColCfg {
  static constexpr int T = N / PC;
  template <int WTX>
  static constexpr int lineb() { return ColLine<N, WTX, xchg_t<AR>>::SIZE * (int)sizeof(xchg_t<AR>); }
  static constexpr bool ONE = W * T <= 1024 && W * lineb<W>() <= 150 * 1024;
  static constexpr int WTMAX = lines_per_block(512, T);
  static constexpr int WT = ONE || W < WTMAX ? W : WTMAX;
  static constexpr int LINEB = lineb<WT>();  // bytes of a line
  static constexpr int G = W / WT;
  static constexpr int GRMAX = (150 * 1024) / (WT * LINEB);
  static constexpr int gr(int g) { return (g <= GRMAX || g == 1) ? g : gr(g / 2); }
  static constexpr int GR = gr(G);
  static constexpr bool OK = G >= 1 && G <= 4 && GR >= 1 && WT * GR * LINEB <= 160 * 1024;
};

// Row kernels with PR points per thread, 128 threads where a line has fewer.
template <int N, int PR, int AR>
static int row_launch_p(int G, const RowArgs& a, hipStream_t s) {
  constexpr int T = N / PR;
  constexpr int L = lines_per_block(128, T);
  const int64_t blocks = (a.ngroups + L - 1) / L;
  if (G == 2)
    hipLaunchKernelGGL((k_row<N, PR, L, 2, true, AR>), dim3((unsigned)blocks), dim3(L * T), 0, s, a);
  else if (a.general)
    hipLaunchKernelGGL((k_row<N, PR, L, 1, true, AR>), dim3((unsigned)blocks), dim3(L * T), 0, s, a);
  else
    hipLaunchKernelGGL((k_row<N, PR, L, 1, false, AR>), dim3((unsigned)blocks), dim3(L * T), 0, s, a);
  return launch_status("k_row");
}

// The alternative set size: 16 where the default is 8 and 8 where it is 16
// (lines of 16 points and more).
template <int N>
constexpr int row_p_alt() {
  return (LineCfg<N>::PR == 8 && N >= 16) ? 16 : (LineCfg<N>::PR == 16 ? 8 : LineCfg<N>::PR);
}

template <int N>
static int row_launch(int p, int G, const RowArgs& a, hipStream_t s) {
  using C = LineCfg<N>;
  if (p == C::PR) return row_launch_p<N, C::PR, F64>(G, a, s);
  if constexpr (row_p_alt<N>() != C::PR) {
    if (p == row_p_alt<N>()) return row_launch_p<N, row_p_alt<N>(), F64>(G, a, s);
  }
  if constexpr (C::PRS != C::PR) {
    if (p == C::PRS) return row_launch_p<N, C::PRS, C::ARS>(G, a, s);
  }
  return fail(NLSE_ERR_ARG, "no row kernel of %d points per thread for length %d", p, N);
}

template <int N, int P, int L1, int L2, int AR, bool KEEP>
static int line1d_launch_p(int G, const Line1DArgs& a, hipStream_t s) {
  constexpr int T = N / P;
  const int64_t blocks = G == 1 ? (a.ngroups + L1 - 1) / L1 : (a.ngroups + L2 - 1) / L2;
  if (G == 2)
    hipLaunchKernelGGL((k_line1d<N, P, L2, 2, true, AR, KEEP>), dim3((unsigned)blocks), dim3(L2 * T), 0, s, a);
  else if (a.general)
    hipLaunchKernelGGL((k_line1d<N, P, L1, 1, true, AR, KEEP>), dim3((unsigned)blocks), dim3(L1 * T), 0, s, a);
  else
    hipLaunchKernelGGL((k_line1d<N, P, L1, 1, false, AR, KEEP>), dim3((unsigned)blocks), dim3(L1 * T), 0, s, a);
  return launch_status("k_line1d");
}

template <int N>
static int line1d_launch(int G, const Line1DArgs& a, hipStream_t s) {
  using C = LineCfg<N>;
  if constexpr (C::P1S != C::P1) {
    if (a.ngroups <= C::LINES1S) {
      constexpr int L = lines_per_block(64, N / C::P1S);
      return line1d_launch_p<N, C::P1S, L, L, C::AR1S, true>(G, a, s);
    }
  }
  return line1d_launch_p<N, C::P1, C::LPB1D1, C::LPB1D2, F64, false>(G, a, s);
}

// Nonlocal line kernels: stage 1 (k_nlc_z) or stage 2 (k_nlc_nl), one
// line pair per N/P threads.
// (PZ, PN points per thread of k_nlc_z and k_nlc_nl, 128 threads per block)
template <int N, int PZ, int PN>
static void nlc_launch_p(int stage, const NlcArgs& a, hipStream_t s) {
  const bool full = a.full && a.ncomp == 1;
  if (stage == 1) {
    constexpr int T = N / PZ, L = lines_per_block(128, T);
    const int64_t blocks = (a.ngroups + L - 1) / L;
    if (full)
      hipLaunchKernelGGL((k_nlc_z<N, PZ, L, 1>), dim3((unsigned)blocks), dim3(L * T), 0, s, a);
    else
      hipLaunchKernelGGL((k_nlc_z<N, PZ, L>), dim3((unsigned)blocks), dim3(L * T), 0, s, a);
  } else {
    constexpr int T = N / PN, L = lines_per_block(128, T);
    const int64_t blocks = (a.ngroups + L - 1) / L;
    if (full)
      hipLaunchKernelGGL((k_nlc_nl<N, PN, L, 1, 1, true>), dim3((unsigned)blocks), dim3(L * T), 0, s, a);
    else if (a.ncomp != 1)
      hipLaunchKernelGGL((k_nlc_nl<N, PN, L, 2, 0, true>), dim3((unsigned)blocks), dim3(L * T), 0, s, a);
    else if (a.general)
      hipLaunchKernelGGL((k_nlc_nl<N, PN, L, 1, 0, true>), dim3((unsigned)blocks), dim3(L * T), 0, s, a);
    else
      hipLaunchKernelGGL((k_nlc_nl<N, PN, L, 1>), dim3((unsigned)blocks), dim3(L * T), 0, s, a);
  }
}

template <int N>
static int nlc_launch(int stage, const NlcArgs& a, hipStream_t s) {
  using C = LineCfg<N>;
  if constexpr (C::NLC_FEW > 0) {
    if ((int64_t)a.ngroups * N <= C::NLC_FEW) {
      nlc_launch_p<N, 4, 4>(stage, a, s);
      return launch_status(stage == 1 ? "k_nlc_z" : "k_nlc_nl");
    }
  }
  nlc_launch_p<N, C::PZ, C::PN>(stage, a, s);
  return launch_status(stage == 1 ? "k_nlc_z" : "k_nlc_nl");
}

// The default tile: at most the widest of one column per thread (4096^2, tile of 8
// columns, four per thread, against 4: column sweep 144 -> 115 us).
template <int N>
constexpr int col_width_default() {
  int w = LineCfg<N>::WDEF;
  while (w > 1 && w * LineCfg<N>::T > 1024) w /= 2;
  return w;
}

// Slabs past the reach of 32-bit offsets have instances for the default tile alone.
constexpr bool big_slab(int64_t n, int64_t ncols) { return n * ncols * 8 > (int64_t)0xffffffff; }

template <int N, int W, int PK, int PC, int AR, bool BIG = false>
static void col_launch_k(const ColArgs& a, hipStream_t s) {
  using K = ColCfg<N, W, PC, AR>;
  const int64_t blocks = a.nslabs * (a.NX / W);
  hipLaunchKernelGGL((k_col<N, PC, K::WT, K::G, K::GR, PK, AR, BIG>), dim3((unsigned)blocks), dim3(K::WT * K::T), 0, s,
                     a);
}

template <int N, int W>
static bool col_launch_w(bool small, const ColArgs& a, hipStream_t s) {
  using C = LineCfg<N>;
  if constexpr (ColCfg<N, W, C::PS, C::ARS>::OK && C::PS != C::P) {
    // small fields: the separable propagator's sweep
    if (small && a.do_prop && a.pkind == PROP_SEP64) {
      col_launch_k<N, W, PROP_SEP64, C::PS, C::ARS>(a, s);
      return true;
    }
  }
  if constexpr (ColCfg<N, W, C::P, F64>::OK) {
    // one instance per propagator kind (fewer live registers than a run-time
    // dispatch).  Step with a dense complex64 table, by a dispatch over all kinds
    // (228 VGPRs, or scratch in blocks of 1024 threads) / by its instance (104):
    // 2048^2 58.4 / 50.6 us, 4096^2 231 / 203, two components of 1024^2 35.6 / 31.5,
    // tiles of 16 columns at 2048^2 109 / 84 (107 before addresses by 64 bits)
    constexpr int P = C::P;
    const int kind = a.do_prop ? a.pkind : PK_NONE;
    if constexpr (W == col_width_default<N>()) {
      // of 3-D fields only
      if (big_slab(N, a.NX)) {
        switch (kind) {
          case PK_NONE: col_launch_k<N, W, PK_NONE, P, F64, true>(a, s); return true;
          case PROP_SEP3D: col_launch_k<N, W, PROP_SEP3D, P, F64, true>(a, s); return true;
          case PROP_C128: col_launch_k<N, W, PROP_C128, P, F64, true>(a, s); return true;
          default: return false;
        }
      }
    }
    switch (kind) {
      case PK_NONE: col_launch_k<N, W, PK_NONE, P, F64>(a, s); return true;
      case PROP_SEP64: col_launch_k<N, W, PROP_SEP64, P, F64>(a, s); return true;
      case PROP_C64: col_launch_k<N, W, PROP_C64, P, F64>(a, s); return true;
      case PROP_SEP3D: col_launch_k<N, W, PROP_SEP3D, P, F64>(a, s); return true;
      case PROP_C128: col_launch_k<N, W, PROP_C128, P, F64>(a, s); return true;
      case PROP_KREAL: col_launch_k<N, W, PROP_KREAL, P, F64>(a, s); return true;
      default: return false;
    }
  }
  return false;
}

template <int N>
static bool col_ok(int w, bool small) {
  using C = LineCfg<N>;
#define NLSE_COL_OK(W) (ColCfg<N, W, C::P, F64>::OK && (!small || ColCfg<N, W, C::PS, C::ARS>::OK))
  switch (w) {
    case 1: return NLSE_COL_OK(1);
    case 2: return NLSE_COL_OK(2);
    case 4: return NLSE_COL_OK(4);
    case 8: return NLSE_COL_OK(8);
    case 16: return NLSE_COL_OK(16);
    case 32: return NLSE_COL_OK(32);
    case 64: return NLSE_COL_OK(64);
    default: return false;
  }
#undef NLSE_COL_OK
}

template <int N>
static int col_width_for(int64_t ncols, int want, bool small) {
  int w = want > 0 && !big_slab(N, ncols) ? want : col_width_default<N>();
  if (w > 64) w = 64;
  while (w > 1 && (w > ncols || (ncols % w) != 0 || !col_ok<N>(w, small))) w >>= 1;
  return w;
}

template <int N>
static int col_launch(int W, bool small, const ColArgs& a, hipStream_t s) {
  bool ok = false;
  switch (W) {
    case 1: ok = col_launch_w<N, 1>(small, a, s); break;
    case 2: ok = col_launch_w<N, 2>(small, a, s); break;
    case 4: ok = col_launch_w<N, 4>(small, a, s); break;
    case 8: ok = col_launch_w<N, 8>(small, a, s); break;
    case 16: ok = col_launch_w<N, 16>(small, a, s); break;
    case 32: ok = col_launch_w<N, 32>(small, a, s); break;
    case 64: ok = col_launch_w<N, 64>(small, a, s); break;
    default: break;
  }
  if (!ok) return fail(NLSE_ERR_ARG, "unsupported column width %d for length %d", W, N);
  return launch_status("k_col");
}

template <int N, int WT, int G, int PITCH>
static int colz_band_launch_wp(const ColArgs& c, const BandArgs& b, size_t band_lds, int64_t nband,
                               hipStream_t s) {
  using C = LineCfg<N>;
  constexpr int W = WT * G;
  constexpr int THREADS = WT * C::T;
  static_assert(THREADS % (64 * BAND_WAVES) == 0, "shared launch blocks hold whole band tiles");
  constexpr int TPB = THREADS / (64 * BAND_WAVES);
  const int64_t ncol = c.nslabs * (c.NX / W);
  const int64_t nbb = (nband + TPB - 1) / TPB;
  const size_t col_bytes = sizeof(float2) * (size_t)col_lds_size<N, WT, 1, float2>();
  const size_t band_bytes = TPB * band_lds;
  const size_t bytes = col_bytes > band_bytes ? col_bytes : band_bytes;
  if (bytes > 160 * 1024) return 1;
  auto fn = k_colz_band<N, C::P, WT, G, PITCH>;
  if (bytes > 64 * 1024) {
    // raise the dynamic LDS limit once per device
    static bool done[64] = {};
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev));
    if (dev < 64 && !done[dev]) {
      HIP_TRY(hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
      done[dev] = true;
    }
  }
  // band tiles first for long intensity columns (2048^2 fields: 25.6 ->
  // 24.3 us), sweep tiles first below (1024^2: 8.9 vs 9.3 us)
  const int band_first = N >= 1024 ? 1 : 0;
  hipLaunchKernelGGL(fn, dim3((unsigned)(ncol + nbb)), dim3(THREADS), bytes, s, c, b, ncol, nband,
                     (int)(band_lds / sizeof(float)), band_first);
  return launch_status("k_colz_band");
}

template <int N, int WT, int G>
static int colz_band_launch_g(int pitch, const ColArgs& c, const BandArgs& b, size_t band_lds, int64_t nband,
                              hipStream_t s) {
  if (pitch == 128) return colz_band_launch_wp<N, WT, G, 128>(c, b, band_lds, nband, s);
  if (pitch == 256) return colz_band_launch_wp<N, WT, G, 256>(c, b, band_lds, nband, s);
  return colz_band_launch_wp<N, WT, G, 0>(c, b, band_lds, nband, s);
}

// The shared launch uses 256-thread blocks (one band tile each, so the band
// tiles keep the occupancy of their own kernel): column tiles of WT = 256/T
// columns, one per thread (two adjacent columns per thread, which needs two
// LDS rounds per stage within the band tiles' LDS, measured slower: 25.5 ->
// 28.3 us at 2048^2).  Below 4 columns per tile (intensity columns of 2048
// and more) the narrow tiles cost more than the overlap gains (4096^2:
// 192 -> 210 us), and the launches stay separate.
#ifndef NLSE_COLZ_G
#define NLSE_COLZ_G 1
#endif
template <int N>
static int colz_band_launch(int, const ColArgs& c, const BandArgs& b, int pitch, size_t band_lds, int64_t nband,
                            hipStream_t s) {
  constexpr int WT = 64 * BAND_WAVES / LineCfg<N>::T;
  if constexpr (WT >= 2 && WT <= 64 && WT * NLSE_COLZ_G >= 4) {
    if (c.NX % (WT * NLSE_COLZ_G) != 0) return 1;
    return colz_band_launch_g<N, WT, NLSE_COLZ_G>(pitch, c, b, band_lds, nband, s);
  } else {
    return 1;
  }
}

// k_colu: blocks of WT = NLSE_COLU_THREADS/T column pairs (at most 64).
// Wide tiles keep the two column runs of a tile long (8 pairs = 64-byte
// runs at NY = 2048): 256 / 512 / 1024 threads measured 46.8 / 40.6 /
// 27.6 us at 2048^2.
#ifndef NLSE_COLU_THREADS
#define NLSE_COLU_THREADS 1024
#endif
template <int N>
static int colu_launch(const ColArgs& a, hipStream_t s) {
  using C = LineCfg<N>;
  constexpr int WT0 = NLSE_COLU_THREADS / C::T;
  constexpr int WT = WT0 < 1 ? 1 : (WT0 > 64 ? 64 : WT0);
  if constexpr (C::P >= 4 && N >= 8) {
    const int64_t tiles = (a.NX / 2 + 1 + WT - 1) / WT;
    hipLaunchKernelGGL((k_colu<N, C::P, WT>), dim3((unsigned)(a.nslabs * tiles)), dim3(WT * C::T), 0, s, a);
    return launch_status("k_colu");
  } else {
    return fail(NLSE_ERR_ARG, "no packed intensity convolution for columns of %d", N);
  }
}

template <int N>
LineOps make_ops() {
  using C = LineCfg<N>;
  return LineOps{&get_twiddles<N>,  &row_launch<N>, C::PR,          row_p_alt<N>(), C::PRS, C::PRL,
                 &line1d_launch<N>, &nlc_launch<N>, &col_launch<N>, &col_width_for<N>,
                 C::P,              C::PS,          &colz_band_launch<N>, &colu_launch<N>};
}

// Dispatch table entry of a line length (engine.hip), or null.
const LineOps* line_ops_public(int64_t n);

// Defined in the lines_*.hip units.
LineOps make_ops_8();
LineOps make_ops_16();
LineOps make_ops_32();
LineOps make_ops_64();
LineOps make_ops_128();
LineOps make_ops_256();
LineOps make_ops_512();
LineOps make_ops_1024();
LineOps make_ops_2048();
LineOps make_ops_4096();

}  // namespace nlse
