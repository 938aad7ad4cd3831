// Nonlocal response of the split step (kernel built at nlse.py:143-153,
// applied at nlse.py:406-409,444-447, cnlse.py:243-249,317-323): the
// intensity |A|^2 is replaced by its zero-padded linear convolution with
// the normalised K0 profile, mode "same", before the nonlinear operator.
//
// 2-D fields.  The bulk is a circular convolution computed by FFT on a
// torus of M x NX points; the kernel is even in both axes, so its spectrum
// is real and is stored as one quadrant.  Two real intensity fields share
// one complex transform, Z = I_a + i I_b:
//   one component   I_a = rows [0, NY/2), I_b = rows [NY/2, NY)  (M = NY/2)
//   two components  I_a = |A1|^2, I_b = |A2|^2                   (M = NY)
// Circular and zero-padded linear convolution agree except within r = 3d
// points of the torus edges (rows y mod M in [0, r) or [M-r, M), columns in
// [0, r) or [NX-r, NX)).  Those band points are convolved directly, in
// FP64, by k_nl_band; when the bands would cover the torus (2r >= M or
// 2r >= NX, or M < 8) every point is a band point ("direct" mode).
//
// One nonlinear application with the nonlocal response is four launches:
//   k_nlc_z    [I_x of the field, stored in real space], Z, F_x(Z)
//   k_nl_band  direct convolution at the band points
//   k_col      (PROP_KREAL) F_y, x K^/(M NX), I_y of Z
//   k_nlc_nl   I_x(Z), band substitution, nonlinear operator, [F_x]
#pragma once
#include "fft_line.hpp"
#include "step_ops.hpp"

namespace nlse {

struct NlcArgs {
  float2* A;
  float2* Z;              // [items][M][NX] x-transformed packed intensities
  int64_t ngroups;        // items * M line groups
  int64_t M;              // torus rows
  int64_t ny;             // NY
  int ncomp;              // 1: row pairs (y, y+M); 2: component pairs
  const double2* tw;      // row twiddles
  // stage 1
  int inverse_first;      // apply I_x to the field (then store it)
  int write_z;            // build and transform Z (0 in direct mode)
  // stage 2
  int forward_last;       // apply F_x after the nonlinear operator
  int loss_sat;
  const void* nlp;        // NLParams1[items] or NLParams2[items*2]
  int has_rabi;
  int has_drive;
  const RabiParams* rabi;
  const void* V;
  int vkind;
  int64_t v_item_stride;
  const float2* drv_r0;
  const float2* drv_r1;
  float2 drv_t0;
  float2 drv_t1;
  float drv_dz;
  float out_scale;
  int general;            // the loss varies from point to point (see nl1_block_I)
  int through;            // level of the field's stores (through_level)
  // band values of the convolved intensity
  const int* rowmap;      // [NY] band row index, or -1
  const float* rowband;   // [slabs][nb][NX]
  const float* colband;   // [slabs][NY][2r]
  int nb;
  int r;
  int direct;
  // one component on the full NY x NX torus (a spectral response given in
  // Fourier space, no band points): the two rows of a pair keep separate
  // intensity rows Z[item][y] = I(y) + 0i, NY per item
  int full;
};

// Line groups of a block (see RowLines): a uniform base of the block's first
// group and this lane's 32-bit offset from there; the group's second line
// lies cs elements after its first.
struct NlcLines {
  int64_t base;          // uniform
  uint32_t d;
  int64_t cs;            // uniform
  uint32_t item, yp;
  uint32_t item0, yp0;   // uniform: the block's first group
  uint32_t slab[2], y[2];
};

__device__ __forceinline__ NlcLines nlc_lines(const NlcArgs& a, uint32_t g0, uint32_t gi, uint32_t n) {
  NlcLines L;
  const uint32_t M = (uint32_t)a.M, ny = (uint32_t)a.ny;
  const bool one = a.M >= a.ngroups;
  L.item0 = one ? 0u : g0 / M;
  L.yp0 = g0 - L.item0 * M;
  L.item = one ? 0u : gi / M;
  L.yp = gi - L.item * M;
  const uint32_t rows = ny * (uint32_t)a.ncomp;  // field rows of an item
  L.base = ((int64_t)L.item0 * rows + L.yp0) * n;
  L.d = ((L.item - L.item0) * rows + L.yp - L.yp0) * n;
  if (a.ncomp == 1) {
    L.slab[0] = L.slab[1] = L.item;
    L.y[0] = L.yp;
    L.y[1] = L.yp + M;
    L.cs = (int64_t)M * n;
  } else {
    L.slab[0] = 2 * L.item;
    L.slab[1] = 2 * L.item + 1;
    L.y[0] = L.y[1] = L.yp;
    L.cs = (int64_t)ny * n;
  }
  return L;
}

// Store a natural set at lane offset d, uniform offset u (bytes).
template <int P, int T>
__device__ __forceinline__ void put_line(const Buf& B, const float2 (&v)[P], uint32_t d, uint32_t u, int through) {
  if (through >= through_need(8 * T)) {
#pragma unroll
    for (int m = 0; m < P; ++m) B.store<ST_THROUGH>(v[m], d, u + 8u * m * T);
  } else {
#pragma unroll
    for (int m = 0; m < P; ++m) B.store(v[m], d, u + 8u * m * T);
  }
}

// Stage 1: [I_x] of the two field lines (stored back in real space), then
// Z = |A_a|^2 + i |A_b|^2 and its forward transform along x.
template <int N, int P, int LPB, int FULL = 0>
__global__ __launch_bounds__(LPB*(N / P)) void k_nlc_z(NlcArgs a) {
  using PL = Plan<N, P>;
  constexpr int T = PL::T;
  constexpr int LINE = LdsLine<N, NLSE_ROW_PADSH, 0>::SIZE;
  __shared__ float2 lds[LPB * LINE];
  constexpr int SYNC = T <= 64 ? SYNC_WAVE : SYNC_BLOCK;
  const int li = LPB == 1 ? 0 : threadIdx.x / T;
  const int t = LPB == 1 ? threadIdx.x : threadIdx.x % T;
  // groups past the end work on the last group and store nothing
  const uint32_t g0 = blockIdx.x * LPB, last = (uint32_t)a.ngroups - 1;
  const bool active = g0 + li <= last;
  const uint32_t gi = active ? g0 + li : last;
  const NlcLines L = nlc_lines(a, g0, gi, N);
  float2* lline = lds + li * LINE;
  const Buf A0(a.A + L.base), Z0(a.Z + (int64_t)g0 * N), tw(a.tw);
  const uint32_t d = 8u * (L.d + t), cs = 8u * (uint32_t)L.cs, zd = 8u * ((gi - g0) * N + t);

  float2 v[2][P];
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int m = 0; m < P; ++m) v[g][m] = A0.load<float2>(d, g * cs + 8u * m * T);
  const Twid<N, P> W = load_twiddles<N, P>(tw, t);
  if (a.inverse_first) {
    fft_line<N, P, 2, true, 1, NLSE_ROW_PADSH, F64, SYNC>(v, t, W, tw, lline, LINE);
    if (a.out_scale != 1.f) {
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int m = 0; m < P; ++m) v[g][m] = make_float2(v[g][m].x * a.out_scale, v[g][m].y * a.out_scale);
    }
    if (active) {
#pragma unroll
      for (int g = 0; g < 2; ++g) put_line<P, T>(A0, v[g], d, g * cs, a.through);
    }
  }
  if constexpr (FULL) {
    // one real intensity per complex line, each row on its own
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int m = 0; m < P; ++m) v[g][m] = make_float2(sqmag(v[g][m]), 0.f);
    fft_line<N, P, 2, false, 1, NLSE_ROW_PADSH, F64, SYNC>(v, t, W, tw, lline, LINE);
    if (active) {
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int m = 0; m < P; ++m) a.Z[((int64_t)L.item * a.ny + L.y[g]) * N + t + m * T] = v[g][m];
    }
  } else if (a.write_z) {
    float2 z[1][P];
#pragma unroll
    for (int m = 0; m < P; ++m) z[0][m] = make_float2(sqmag(v[0][m]), sqmag(v[1][m]));
    fft_line<N, P, 1, false, 1, NLSE_ROW_PADSH, F64, SYNC>(z, t, W, tw, lline, LINE);
    if (active) put_line<P, T>(Z0, z[0], zd, 0, a.through);
  }
}

// Stage 2: the nonlinear operator with the convolved intensities, then
// [Rabi, drive, F_x].  The intensity transform runs first, while the field
// loads are in flight.  One component (NC = 1): the two rows are finished
// one after the other (potential, nonlinear step, F_x, store), so only one
// row's working set is live at a time; two components (NC = 2) couple at
// every point and are transformed one line after the other.
// Both rows of a one-component pair transformed by one two-line F_x
// (measured 27.9 -> 27.0 us at 2048^2) rather than one after the other.

template <int N, int P, int LPB, int NC, int FULL = 0, bool GEN = false>
__global__ __launch_bounds__(LPB*(N / P)) void k_nlc_nl(NlcArgs a) {
  using PL = Plan<N, P>;
  constexpr int T = PL::T;
  constexpr int LINE = LdsLine<N, NLSE_ROW_PADSH, 0>::SIZE;
  __shared__ float2 lds[LPB * LINE];
  constexpr int SYNC = T <= 64 ? SYNC_WAVE : SYNC_BLOCK;
  const int li = LPB == 1 ? 0 : threadIdx.x / T;
  const int t = LPB == 1 ? threadIdx.x : threadIdx.x % T;
  // groups past the end work on the last group and store nothing
  const uint32_t g0 = blockIdx.x * LPB, last = (uint32_t)a.ngroups - 1;
  const bool active = g0 + li <= last;
  const uint32_t gi = active ? g0 + li : last;
  const NlcLines L = nlc_lines(a, g0, gi, N);
  float2* lline = lds + li * LINE;
  const Buf A0(a.A + L.base), Z0(a.Z + (int64_t)g0 * N), tw(a.tw);
  const uint32_t d = 8u * (L.d + t), cs = 8u * (uint32_t)L.cs, zd = 8u * ((gi - g0) * N + t);

  float2 z[1][P];
#pragma unroll
  for (int m = 0; m < P; ++m) z[0][m] = make_float2(0.f, 0.f);
  if (!a.direct) {
    // full: row y of an item's ny, else group g's row
#pragma unroll
    for (int m = 0; m < P; ++m)
      z[0][m] = FULL ? a.Z[((int64_t)L.item * a.ny + L.y[0]) * N + t + m * T] : Z0.load<float2>(zd, 8u * m * T);
  }
  float2 v[NC][P];
#pragma unroll
  for (int g = 0; g < NC; ++g)
#pragma unroll
    for (int m = 0; m < P; ++m) v[g][m] = A0.load<float2>(d, g * cs + 8u * m * T);
  const Twid<N, P> W = load_twiddles<N, P>(tw, t);
  if (!a.direct) fft_line<N, P, 1, true, 1, NLSE_ROW_PADSH, F64, SYNC>(z, t, W, tw, lline, LINE);
  // z.x: convolved intensity of line 0, z.y: of line 1; band points take
  // their band values: a band row from the row band, else the r points at
  // either end from the column band (uniform tests skip the other points)
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const int bi = a.rowmap[L.y[g]];
    const float* rb = a.rowband + ((int64_t)L.slab[g] * a.nb + bi) * N + t;
    const float* cb = a.colband + ((int64_t)L.slab[g] * a.ny + L.y[g]) * 2 * a.r + t;
#pragma unroll
    for (int m = 0; m < P; ++m) {
      float& c = g == 0 ? z[0][m].x : z[0][m].y;
      if (bi >= 0) c = rb[m * T];
      else if (m * T < a.r && t + m * T < a.r) c = cb[m * T];
      else if ((m + 1) * T > N - a.r && t + m * T >= N - a.r) c = cb[m * T - N + 2 * a.r];
    }
  }

  float vr[P], vi[P];
  auto load_row_v = [&](uint32_t y) __attribute__((always_inline)) {
    load_v_set<P, T, GEN>(a.V, a.vkind, L.item0 * a.v_item_stride + (int64_t)L.yp0 * N,
                     (L.item - L.item0) * (uint32_t)a.v_item_stride + (y - L.yp0) * N + t, vr, vi);
  };
  auto finish_line = [&](float2 (&w)[1][P], uint32_t c1) __attribute__((always_inline)) {
    if (a.forward_last) fft_line<N, P, 1, false, 1, NLSE_ROW_PADSH, F64, SYNC>(w, t, W, tw, lline, LINE);
    if (a.out_scale != 1.f) {
#pragma unroll
      for (int m = 0; m < P; ++m) w[0][m] = make_float2(w[0][m].x * a.out_scale, w[0][m].y * a.out_scale);
    }
    if (active) put_line<P, T>(A0, w[0], d, c1, a.through);
  };

  if constexpr (NC == 1) {
    const NLParams1 p = reinterpret_cast<const NLParams1*>(a.nlp)[L.item];
    float I[P];
    if constexpr (FULL) {
      // the second row's intensity line, transformed on its own; the first
      // row's goes to z.x (its imaginary part is zero)
      float2 z2[1][P];
#pragma unroll
      for (int m = 0; m < P; ++m)
        z2[0][m] = a.Z[((int64_t)L.item * a.ny + L.y[1]) * N + t + m * T];
      fft_line<N, P, 1, true, 1, NLSE_ROW_PADSH, F64, SYNC>(z2, t, W, tw, lline, LINE);
#pragma unroll
      for (int m = 0; m < P; ++m) z[0][m].y = z2[0][m].x;
    }
#pragma unroll
    for (int m = 0; m < P; ++m) I[m] = z[0][m].x;
    load_row_v(L.y[0]);
    nl1_block_I<P, GEN>(v[0], I, p, a.loss_sat, a.vkind == V_CPLX, vr, vi);
    // both rows' F_x in one two-line transform
    float2 u[2][P];
#pragma unroll
    for (int m = 0; m < P; ++m) {
      u[0][m] = v[0][m];
      u[1][m] = A0.load<float2>(d, cs + 8u * m * T);
      I[m] = z[0][m].y;
    }
    load_row_v(L.y[1]);
    nl1_block_I<P, GEN>(u[1], I, p, a.loss_sat, a.vkind == V_CPLX, vr, vi);
    if (a.forward_last) fft_line<N, P, 2, false, 1, NLSE_ROW_PADSH, F64, SYNC>(u, t, W, tw, lline, LINE);
    if (a.out_scale != 1.f) {
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int m = 0; m < P; ++m) u[g][m] = make_float2(u[g][m].x * a.out_scale, u[g][m].y * a.out_scale);
    }
    if (active) {
#pragma unroll
      for (int g = 0; g < 2; ++g) put_line<P, T>(A0, u[g], d, g * cs, a.through);
    }
  } else {
    const NLParams2* pp = reinterpret_cast<const NLParams2*>(a.nlp) + 2 * L.item;
    const NLParams2 p1 = pp[0], p2 = pp[1];
    float I1[P], I2[P];
#pragma unroll
    for (int m = 0; m < P; ++m) {
      I1[m] = z[0][m].x;
      I2[m] = z[0][m].y;
    }
    load_row_v(L.yp);
    nl2_block_I<P>(v[0], v[1], I1, I2, p1, p2, vr, vi);
    if (a.has_rabi) {
      const RabiParams rb = a.rabi[L.item];
#pragma unroll
      for (int m = 0; m < P; ++m) rabi(v[0][m], v[1][m], rb);
    }
    if (a.has_drive) {
#pragma unroll
      for (int m = 0; m < P; ++m) {
        const int64_t ri = (int64_t)L.yp * N + t + m * T;
        float2 q = cmul(a.drv_r0[ri], a.drv_t0);
        q = make_float2(q.x * a.drv_dz, q.y * a.drv_dz);
        v[1][m] = make_float2(v[1][m].x + q.y, v[1][m].y - q.x);
        q = cmul(a.drv_r1[ri], a.drv_t1);
        q = make_float2(q.x * a.drv_dz, q.y * a.drv_dz);
        v[1][m] = make_float2(v[1][m].x + q.y, v[1][m].y - q.x);
      }
    }
    float2 w[1][P];
#pragma unroll
    for (int m = 0; m < P; ++m) w[0][m] = v[0][m];
    finish_line(w, 0);
#pragma unroll
    for (int m = 0; m < P; ++m) w[0][m] = v[1][m];
    finish_line(w, cs);
  }
}

// ------------------------------------------------------------ band points
// Output rectangle of k_nl_band: rows [y0, y0 + nrows), columns
// [x0, x0 + ncols), ncols <= 64.  Lane l of each wave owns column
// x0 + l % ncols and the RB_BAND rows y0 + (l / ncols)*RB_BAND + j.
struct BandTile {
  int y0, x0, nrows, ncols;
};

#ifndef NLSE_RB_BAND
#define NLSE_RB_BAND 4
#endif
constexpr int RB_BAND = NLSE_RB_BAND;  // output rows per lane
constexpr int BAND_WAVES = 4;  // waves per block, splitting the kernel columns
constexpr int KU_BAND = 4;     // kernel rows per register window
#ifndef NLSE_BAND_MFMA
#define NLSE_BAND_MFMA 1  // band tiles on the matrix cores where their LDS fits
#endif

struct BandArgs {
  const float2* A;        // real-space field, slabs of NY x NX
  int ny, nx, r;
  const float* KT;        // [2r+1][kr] transposed kernel, entries u >= 2r+1 zero
  int kr;                 // padded kernel rows (multiple of KU_BAND)
  int kc;                 // kernel rows per LDS chunk (multiple of KU_BAND)
  const BandTile* tiles;
  int ntiles;             // tiles per slab
  const int* rowmap;
  int nb;
  float* rowband;
  float* colband;
  // matrix-core form (band_mfma_body): zero-padded kernel rows [2r+1][kpw]
  const float* KP;
  int kpw;
  int mfma;
};

// LDS of one k_nl_band block, in floats: staged intensities
// [groups*RB_BAND + kc - 1][pitch], the kernel chunk [2r+1][kc] and the
// per-wave partial sums [BAND_WAVES][64][RB_BAND] (double).
__host__ __device__ inline size_t band_lds_floats(int nc, int r, int kc, int pitch) {
  const size_t srows = (size_t)(64 / nc) * RB_BAND + kc - 1;
  const size_t p = pitch > 0 ? (size_t)pitch : (size_t)(nc + 2 * r);
  const size_t img = (srows * p + 3) & ~(size_t)3;
  const size_t kt = ((size_t)(2 * r + 1) * kc + 1) & ~(size_t)1;
  return img + kt + (size_t)BAND_WAVES * 64 * RB_BAND * 2;
}

// Direct convolution at the points of one band tile of one slab, by
// 64 * BAND_WAVES threads (local ids `tid`) with `smem` holding
// band_lds_floats() floats.  The intensities the tile needs are staged in
// LDS with a row pitch of PITCH floats (0: the tile's own width), per chunk
// of kc kernel rows.  The BAND_WAVES waves split the kernel columns; each
// lane slides a register window of RB_BAND + 3 rows down its column and
// reads four kernel rows at once, accumulating FP32 partial sums of at most
// 4 x 8 products that are added in FP64.  Every thread of the block passes
// the same barriers whatever its tile; `write` = false computes without
// storing (padding tiles of a shared launch).
template <int PITCH>
__device__ __forceinline__ void band_body(const BandArgs& b, int tile, int64_t slab, int tid, float* smem,
                                          bool write) {
  const BandTile tl = b.tiles[tile];
  const int lane = tid & 63;
  const int wv = tid >> 6;
  const int kw = 2 * b.r + 1;
  const int groups = 64 / tl.ncols;
  const int wcols = tl.ncols + 2 * b.r;
  const int pitch = PITCH > 0 ? PITCH : wcols;
  const int srows = groups * RB_BAND + b.kc - 1;
  float* img = smem;
  float* kt = smem + (((size_t)srows * pitch + 3) & ~(size_t)3);
  double* red = reinterpret_cast<double*>(kt + (((size_t)kw * b.kc + 1) & ~(size_t)1));
  const int c = lane % tl.ncols;
  const int g = lane / tl.ncols;
  const bool lane_ok = g < groups;
  const float2* a = b.A + slab * (int64_t)b.ny * b.nx;
  const int vper = (kw + BAND_WAVES - 1) / BAND_WAVES;
  const int v0 = wv * vper;
  const int v1 = v0 + vper < kw ? v0 + vper : kw;

  double acc[RB_BAND];
#pragma unroll
  for (int j = 0; j < RB_BAND; ++j) acc[j] = 0.0;

  const int total = srows * wcols;
  for (int u0 = 0; u0 < b.kr; u0 += b.kc) {
    const int kc = (b.kr - u0) < b.kc ? (b.kr - u0) : b.kc;
    __syncthreads();
    // kernel chunk, transposed: kt[v][u - u0]; four loads in flight per
    // thread before the stores
    for (int e0 = tid; e0 < kw * kc; e0 += 4 * 64 * BAND_WAVES) {
      float kv[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int e = e0 + k * 64 * BAND_WAVES;
        const int ec = e < kw * kc ? e : 0;
        const int v = ec / kc, u = ec - v * kc;
        kv[k] = b.KT[(int64_t)v * b.kr + u0 + u];
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (e0 + k * 64 * BAND_WAVES < kw * kc) kt[e0 + k * 64 * BAND_WAVES] = kv[k];
    }
    // staged row i holds field row y0 - r + u0 + i; column j holds x0 - r + j.
    // Eight loads per thread are issued back to back: out-of-range points
    // read element 0 and are zeroed after the load (a load under a branch
    // makes the compiler wait for it at the join), and (i, j) advance
    // incrementally instead of dividing by the tile width per element.
    constexpr int NTH = 64 * BAND_WAVES;
    const int di = NTH / wcols, dj = NTH - di * wcols;
    for (int base = 0; base < total; base += 8 * NTH) {
      const int e0 = base + tid;
      int i = e0 / wcols, j = e0 - i * wcols;
      float2 q[8];
      int at[8];
      bool ok[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int y = tl.y0 - b.r + u0 + i, x = tl.x0 - b.r + j;
        ok[k] = e0 + k * NTH < total && y >= 0 && y < b.ny && x >= 0 && x < b.nx;
        q[k] = a[ok[k] ? (int64_t)y * b.nx + x : 0];
        at[k] = i * pitch + j;
        i += di;
        j += dj;
        if (j >= wcols) {
          j -= wcols;
          ++i;
        }
      }
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (e0 + k * NTH < total) img[at[k]] = ok[k] ? sqmag(q[k]) : 0.f;
    }
    __syncthreads();
    if (lane_ok) {
      const float* col = img + g * RB_BAND * pitch + c;
      for (int q = 0; q < kc; q += KU_BAND) {
        for (int vc = v0; vc < v1; vc += 8) {
          const int vend = vc + 8 < v1 ? vc + 8 : v1;
          float s[RB_BAND];
#pragma unroll
          for (int j = 0; j < RB_BAND; ++j) s[j] = 0.f;
          for (int vv = vc; vv < vend; ++vv) {
            const float4 k4 = *reinterpret_cast<const float4*>(kt + vv * kc + q);
            const float* p = col + q * pitch + vv;
            float w[RB_BAND + KU_BAND - 1];
#pragma unroll
            for (int i = 0; i < RB_BAND + KU_BAND - 1; ++i) w[i] = p[i * pitch];
#pragma unroll
            for (int j = 0; j < RB_BAND; ++j) {
              s[j] = fmaf(k4.x, w[j], s[j]);
              s[j] = fmaf(k4.y, w[j + 1], s[j]);
              s[j] = fmaf(k4.z, w[j + 2], s[j]);
              s[j] = fmaf(k4.w, w[j + 3], s[j]);
            }
          }
#pragma unroll
          for (int j = 0; j < RB_BAND; ++j) acc[j] += (double)s[j];
        }
      }
    }
  }
  // sum the partial results of the waves
#pragma unroll
  for (int j = 0; j < RB_BAND; ++j) red[(wv * 64 + lane) * RB_BAND + j] = acc[j];
  __syncthreads();
  if (wv != 0 || !lane_ok || !write) return;
  const int x = tl.x0 + c;
#pragma unroll
  for (int j = 0; j < RB_BAND; ++j) {
    double sum = 0.0;
#pragma unroll
    for (int w2 = 0; w2 < BAND_WAVES; ++w2) sum += red[(w2 * 64 + lane) * RB_BAND + j];
    const int yo = g * RB_BAND + j;
    if (yo >= tl.nrows) break;
    const int y = tl.y0 + yo;
    const int bi = b.rowmap[y];
    float* out;
    if (bi >= 0)
      out = b.rowband + (slab * b.nb + bi) * (int64_t)b.nx + x;
    else
      out = b.colband + (slab * b.ny + y) * (int64_t)2 * b.r + (x < b.r ? x : x - b.nx + 2 * b.r);
    *out = (float)sum;
  }
}

// ------------------------------------------------ band points, matrix cores
// A block of 4 waves covers ty x tx sub-tiles of 16 x 16 output points (tx =
// 1, 2 or 4 sub-tiles across the tile's columns, ty = 4 / tx).  With the
// intensities staged from (y0 - r, x0 - r), one kernel row u contributes
//   out[Y][X] += sum_j S[Y + u][X0 + j] * K[u][j - X]     (j = X + v)
// to the sub-tile at staged column X0: a product of a 16 x J slice of the
// staged rows and a J x 16 Toeplitz slice of the kernel row (K zero outside
// [0, 2r]), J = 16 + 2r rounded up to 4, i.e. J/4 FP32 MFMAs of 16 x 16 x 4.
// The B operand is read from a copy of the kernel row with 16 zeros in
// front (KP[u][t] = K[u][t - 16]), so lane (k, X) reads KP[u][4c + k - X +
// 16].  The FP32 sum of one kernel row (pair of rows, band_mfma_rows; at
// most 2r+1 nonzero products) is added in FP64, as the VALU form adds its
// partial sums.
typedef float band_f4 __attribute__((ext_vector_type(4)));
#ifndef NLSE_BAND_STAGE
#define NLSE_BAND_STAGE 8
#endif
constexpr int BAND_STAGE = NLSE_BAND_STAGE;  // staging loads in flight per thread

__host__ __device__ inline int band_mfma_tx(int ncols) { return ncols > 32 ? 4 : (ncols > 16 ? 2 : 1); }
// chunks of 4 staged columns per kernel row: J = 16 + 2r rounded up to an
// even number of chunks (two accumulators take alternate chunks)
__host__ __device__ inline int band_mfma_chunks(int r) { return (16 + 2 * r + 7) / 8 * 2; }
constexpr int BAND_MFMA_MAX_CHUNKS = 18;
__host__ __device__ inline int band_mfma_kpw(int r) { return 4 * band_mfma_chunks(r) + 16; }
// staged columns of a tile (the last ones zero) and their LDS pitch: at
// least the width and 2 mod 32, so the 16 rows x 2 columns that a half-wave
// reads for one A operand fall in distinct banks of 32 four-byte banks
__host__ __device__ inline int band_mfma_ws(int tx, int r) { return 16 * (tx - 1) + 4 * band_mfma_chunks(r); }
__host__ __device__ inline int band_mfma_pitch(int ws) { return (ws + 29) / 32 * 32 + 2; }
__host__ __device__ inline size_t band_mfma_lds_floats(int tx, int r) {
  const size_t img = (size_t)(16 * (4 / tx) + 2 * r) * band_mfma_pitch(band_mfma_ws(tx, r));
  return ((img + 3) & ~(size_t)3) + (size_t)(2 * r + 1) * band_mfma_kpw(r);
}

// The kernel rows of one 16 x 16 sub-tile, NCH chunks per row.  The kernel
// is even in y (row u equals row 2r - u), so rows u and 2r - u take one
// product with their staged intensity rows added: r + 1 row steps, the last
// the middle row alone.  The next step's operands are loaded while the
// current step's MFMAs run (steps taken in pairs so two register sets
// alternate).  pa / pb: this lane's A / B operand of chunk 0 of row 0.
template <int NCH>
__device__ __forceinline__ void band_mfma_rows(const float* pa, const float* pb, int pitch, int kpw, int r,
                                               double (&acc)[4]) {
  static_assert(NCH % 2 == 0, "chunks alternate between two accumulators");
  float xa[NCH], xc[NCH], xb[NCH], ya[NCH], yc[NCH], yb[NCH];
  auto load = [&](float (&ra)[NCH], float (&rc)[NCH], float (&rb)[NCH], int u) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      ra[c] = pa[u * pitch + 4 * c];
      rc[c] = pa[(2 * r - u) * pitch + 4 * c];
      rb[c] = pb[u * kpw + 4 * c];
    }
  };
  auto step = [&](const float (&ra)[NCH], const float (&rc)[NCH], const float (&rb)[NCH], bool pair) {
    band_f4 d0 = {0.f, 0.f, 0.f, 0.f}, d1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < NCH; c += 2) {
      const float a0 = pair ? ra[c] + rc[c] : ra[c];
      const float a1 = pair ? ra[c + 1] + rc[c + 1] : ra[c + 1];
      d0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, rb[c], d0, 0, 0, 0);
      d1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, rb[c + 1], d1, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] += (double)d0[i] + (double)d1[i];
  };
  load(xa, xc, xb, 0);
  int t = 0;
  for (; t + 2 <= r; t += 2) {  // steps t and t + 1 are pairs
    load(ya, yc, yb, t + 1);
    step(xa, xc, xb, true);
    load(xa, xc, xb, t + 2);
    step(ya, yc, yb, true);
  }
  if (t < r) {  // t = r - 1: one pair, then the middle row
    load(ya, yc, yb, r);
    step(xa, xc, xb, true);
    step(ya, yc, yb, false);
  } else {  // t = r: the middle row
    step(xa, xc, xb, false);
  }
}

// Direct convolution at the points of one band tile of one slab on the
// matrix cores, by 64 * BAND_WAVES threads with `smem` holding
// band_mfma_lds_floats() floats for the tile's shape.  One barrier, passed
// by every thread; `write` = false stages without computing (padding tiles
// of a shared launch).
__device__ __forceinline__ void band_mfma_body(const BandArgs& b, int tile, int64_t slab, int tid, float* smem,
                                               bool write) {
  static_assert(BAND_WAVES == 4, "one 16 x 16 sub-tile per wave, four per tile");
  const BandTile tl = b.tiles[tile];
  const int r = b.r, kw = 2 * r + 1;
  const int tx = band_mfma_tx(tl.ncols), ty = 4 / tx;
  const int hrows = 16 * ty + 2 * r;
  const int wcols = 16 * tx + 2 * r;  // staged columns that hold field values
  const int ws = band_mfma_ws(tx, r);
  const int pitch = band_mfma_pitch(ws);
  const int nch = band_mfma_chunks(r);
  const int kpw = b.kpw;
  float* img = smem;
  float* kp = smem + (((size_t)hrows * pitch + 3) & ~(size_t)3);
  const float2* a = b.A + slab * (int64_t)b.ny * b.nx;
  constexpr int NTH = 64 * BAND_WAVES;
  // the kernel rows, BAND_STAGE loads per thread in flight
  const int nkp = kw * kpw;
  for (int e0 = 0; e0 < nkp; e0 += BAND_STAGE * NTH) {
    float kv[BAND_STAGE];
#pragma unroll
    for (int k = 0; k < BAND_STAGE; ++k) {
      const int e = e0 + k * NTH + tid;
      kv[k] = b.KP[e < nkp ? e : 0];
    }
#pragma unroll
    for (int k = 0; k < BAND_STAGE; ++k) {
      const int e = e0 + k * NTH + tid;
      if (e < nkp) kp[e] = kv[k];
    }
  }
  // staged row i holds field row y0 - r + i, column j field column x0 - r +
  // j; BAND_STAGE loads per thread in flight, out-of-range points read
  // element 0 and are zeroed after the load
  const int total = hrows * ws;
  const int di = NTH / ws, dj = NTH - di * ws;
  for (int base = 0; base < total; base += BAND_STAGE * NTH) {
    const int e0 = base + tid;
    int i = e0 / ws, j = e0 - i * ws;
    float2 q[BAND_STAGE];
    int at[BAND_STAGE];
    bool ok[BAND_STAGE];
#pragma unroll
    for (int k = 0; k < BAND_STAGE; ++k) {
      const int y = tl.y0 - r + i, x = tl.x0 - r + j;
      ok[k] = e0 + k * NTH < total && j < wcols && y >= 0 && y < b.ny && x >= 0 && x < b.nx;
      q[k] = a[ok[k] ? (int64_t)y * b.nx + x : 0];
      at[k] = i * pitch + j;
      i += di;
      j += dj;
      if (j >= ws) {
        j -= ws;
        ++i;
      }
    }
#pragma unroll
    for (int k = 0; k < BAND_STAGE; ++k)
      if (e0 + k * NTH < total) img[at[k]] = ok[k] ? sqmag(q[k]) : 0.f;
  }
  __syncthreads();
  const int lane = tid & 63, wv = tid >> 6;
  const int sy = wv / tx, sx = wv - sy * tx;
  if (!write || sy * 16 >= tl.nrows || sx * 16 >= tl.ncols) return;
  // band row indices of this lane's output rows, fetched before the products
  int bis[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int yo = sy * 16 + 4 * (lane >> 4) + i;
    bis[i] = b.rowmap[tl.y0 + (yo < tl.nrows ? yo : 0)];
  }
  // A: lane (m, k) = (lane % 16, lane / 16) supplies S[Y = m][4c + k];
  // B: the same lane supplies KP[u][4c + k - X + 16] with X = m
  const int m = lane & 15, k = lane >> 4;
  const float* pa = img + (sy * 16 + m) * pitch + sx * 16 + k;
  const float* pb = kp + 16 + k - m;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  switch (nch) {
    case 4: band_mfma_rows<4>(pa, pb, pitch, kpw, r, acc); break;
    case 6: band_mfma_rows<6>(pa, pb, pitch, kpw, r, acc); break;
    case 8: band_mfma_rows<8>(pa, pb, pitch, kpw, r, acc); break;
    case 10: band_mfma_rows<10>(pa, pb, pitch, kpw, r, acc); break;
    case 12: band_mfma_rows<12>(pa, pb, pitch, kpw, r, acc); break;
    case 14: band_mfma_rows<14>(pa, pb, pitch, kpw, r, acc); break;
    case 16: band_mfma_rows<16>(pa, pb, pitch, kpw, r, acc); break;
    default: band_mfma_rows<18>(pa, pb, pitch, kpw, r, acc); break;
  }
  // D: lane holds rows 4 * (lane / 16) + i, column lane % 16 of the sub-tile
  const int xo = sx * 16 + m;
  if (xo >= tl.ncols) return;
  const int x = tl.x0 + xo;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int yo = sy * 16 + 4 * k + i;
    if (yo >= tl.nrows) break;
    const int y = tl.y0 + yo;
    const int bi = bis[i];
    float* out;
    if (bi >= 0)
      out = b.rowband + (slab * b.nb + bi) * (int64_t)b.nx + x;
    else
      out = b.colband + (slab * b.ny + y) * (int64_t)2 * b.r + (x < b.r ? x : x - b.nx + 2 * b.r);
    *out = (float)acc[i];
  }
}

// ------------------------------------------------------------------ 1-D
// Zero-padded linear convolution of the intensities of the G lines owned
// by a thread group, through the line's LDS (N floats per line), FP64
// accumulation: I[g][m] = sum_j K[x - j + r] |A_g(j)|^2, x = t + m*T.
template <int N, int P, int G>
__device__ __forceinline__ void conv1d_intensity(const float2 (&v)[G][P], float (&I)[G][P], float* ib, int t,
                                                 const double* __restrict__ K, int r) {
  constexpr int T = N / P;
  __syncthreads();
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int m = 0; m < P; ++m) ib[g * N + t + m * T] = sqmag(v[g][m]);
  __syncthreads();
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int m = 0; m < P; ++m) {
      const int x = t + m * T;
      const int j0 = x - r < 0 ? 0 : x - r;
      const int j1 = x + r > N - 1 ? N - 1 : x + r;
      double acc = 0.0;
      for (int j = j0; j <= j1; ++j) acc = fma(K[x - j + r], (double)ib[g * N + j], acc);
      I[g][m] = (float)acc;
    }
  __syncthreads();
}

}  // namespace nlse
