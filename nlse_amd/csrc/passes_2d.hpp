// Fused line passes of the 2-D split step.
//
// Field layout in HBM: complex64, row-major (..., [2,] NY, NX), leading dims
// flattened into "items"; a 2-component field stores component c of item b
// at slab b*2 + c.  Between passes the field lives in the mixed domain
// B = F_x(A) (x spectral, y real).  One split step is then two sweeps:
//
//   column pass  C = I_y * diag(P/(NX NY)) * F_y      (strided columns)
//   row pass     R = F_x * Nl * I_x                    (contiguous rows)
//
// where Nl is the real-space operator of the step (nl_prop[_c], Rabi,
// drive).  The first row pass of a run omits I_x, the last omits F_x.
// Every sweep reads and writes the field once: 16 B per point, plus the
// real-space side inputs in the row pass.
#pragma once
#include "fft_line.hpp"
#include "nonlocal.hpp"
#include "step_ops.hpp"

namespace nlse {

enum : int { PROP_SEP64 = 0, PROP_C64 = 1, PROP_SEP3D = 2, PROP_C128 = 3, PROP_KREAL = 4 };
// compile-time kind of a column instance without a propagator (transforms only)
constexpr int PK_NONE = 16;

#ifndef NLSE_COL_PAIRED
#define NLSE_COL_PAIRED 1
#endif

struct RowArgs {
  float2* A;
  int64_t ngroups;        // rows (G=1) or row pairs (G=2)
  int64_t rows_per_item;  // NY: rows per item and component
  const double2* tw;      // twiddles of the row length (FP64 ratio pairs)
  int inverse_first;      // apply I_x (unnormalised) first
  int forward_last;       // apply F_x last
  int has_a;              // first nonlinear application (end of step k)
  int has_rabi;           // Rabi rotation after application a (G=2)
  int has_drive;          // cavity drive after the step (G=2, DDGPE)
  int has_b;              // second nonlinear application (start of step k+1)
  int loss_sat;           // single-component loss multiplied by sat
  const void* nlp_a;      // NLParams1[items] or NLParams2[items*2]
  const void* nlp_b;
  const RabiParams* rabi; // [items]
  const void* V;          // potential V' (k/2 V), broadcast over items
  int vkind;
  int64_t v_item_stride;  // elements between items of V (0: shared)
  // drive: A[...,1,:,:] -= F_r * F_t[step] * dz * 1j for (pump, probe)
  const float2* drv_r0;
  const float2* drv_r1;
  float2 drv_t0;
  float2 drv_t1;
  float drv_dz;
  float out_scale;        // applied to the stored result (1 or 1/N)
  int general;            // the loss varies from point to point (see nl1_block_I)
  int through;            // level of the field's stores (through_level)
};

// LDS entries of one row block.
template <int N, int LPB, int G>
constexpr int row_lds_size() {
  return LPB * G * LdsLine<N, NLSE_ROW_PADSH, 0>::SIZE;
}

// Line groups of a row block: a uniform element offset of the block's first
// group and 32-bit per-lane offsets from there (a block's groups span less
// than 2^29 elements: at most two items' worth of one component pair).
template <int N, int G>
struct RowLines {
  int64_t base;   // uniform: element offset of the first group's first line
  uint32_t d;     // this lane's group, relative to base
  int64_t cs;     // uniform: offset from line 0 to line 1 of a group (G = 2)
  uint32_t item;
  uint32_t item0, y0;  // uniform: item and row of the block's first group
  uint32_t y;
};

template <int N, int G>
__device__ __forceinline__ RowLines<N, G> row_lines(uint32_t g0, uint32_t g, uint32_t rows, bool one_item) {
  RowLines<N, G> L;
  L.item0 = one_item ? 0u : g0 / rows;
  L.item = one_item ? 0u : g / rows;
  L.y0 = g0 - L.item0 * rows;
  L.y = g - L.item * rows;
  L.cs = (int64_t)rows * N;
  if constexpr (G == 1) {
    L.base = (int64_t)g0 * N;
    L.d = (g - g0) * N;
  } else {
    L.base = ((int64_t)L.item0 * 2 * rows + L.y0) * N;
    L.d = ((L.item - L.item0) * 2 * rows + L.y - L.y0) * N;
  }
  return L;
}

// Row sweep body: LPB line groups starting at group `g0`.  Groups past the
// end work on the last group and store nothing.
template <int N, int P, int LPB, int G, bool GEN, int AR = F64>
__device__ __forceinline__ void row_body(const RowArgs& a, int64_t g0, xchg_t<AR>* lds) {
  using PL = Plan<N, P>;
  constexpr int T = PL::T;
  constexpr int LINE = LdsLine<N, NLSE_ROW_PADSH, 0>::SIZE;
  // the lanes of a line are one wave's or fewer: no block barriers
  constexpr int SYNC = T <= 64 ? SYNC_WAVE : SYNC_BLOCK;

  const int li = LPB == 1 ? 0 : threadIdx.x / T;
  const int t = LPB == 1 ? threadIdx.x : threadIdx.x % T;
  const uint32_t gi = (uint32_t)g0 + li, last = (uint32_t)a.ngroups - 1;
  const bool active = gi <= last;
  const RowLines<N, G> L =
      row_lines<N, G>((uint32_t)g0, active ? gi : last, (uint32_t)a.rows_per_item, a.rows_per_item >= a.ngroups);
  const uint32_t item = L.item;
  xchg_t<AR>* lline = lds + li * G * LINE;
  const Buf A0(a.A + L.base), tw(a.tw);
  const uint32_t d = 8u * (L.d + t), cs = 8u * (uint32_t)L.cs;

  float2 v[G][P];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int m = 0; m < P; ++m) v[g][m] = A0.load<float2>(d, g * cs + 8u * m * T);
  const Twid<N, P> W = load_twiddles<N, P>(tw, t);

  // side inputs of the real-space step, fetched with the field so that
  // their latency overlaps the inverse transform
  const bool has_nl = a.has_a || a.has_b;
  float vr[P], vi[P];
  load_v_set<P, T, GEN>(a.V, has_nl ? a.vkind : V_NONE, L.item0 * a.v_item_stride + (int64_t)L.y0 * N,
                   (item - L.item0) * (uint32_t)a.v_item_stride + (L.y - L.y0) * N + t, vr, vi);

  if (a.inverse_first) fft_line<N, P, G, true, G, NLSE_ROW_PADSH, AR, SYNC>(v, t, W, tw, lline, LINE);

  if constexpr (G == 1) {
    // one copy of the code for both applications
#pragma unroll 1
    for (int k = 0; k < 2; ++k) {
      if (k == 0 ? a.has_a : a.has_b) {
        const NLParams1 q = reinterpret_cast<const NLParams1*>(k == 0 ? a.nlp_a : a.nlp_b)[item];
        nl1_block<P, GEN>(v[0], q, a.loss_sat, a.vkind == V_CPLX, vr, vi);
      }
    }
  } else {
    if (a.has_a) {
      const NLParams2* p = reinterpret_cast<const NLParams2*>(a.nlp_a) + 2 * item;
      const NLParams2 p1 = p[0], p2 = p[1];
      nl2_block<P>(v[0], v[1], p1, p2, vr, vi);
      if (a.has_rabi) {
        const RabiParams rb = a.rabi[item];
#pragma unroll
        for (int m = 0; m < P; ++m) rabi(v[0][m], v[1][m], rb);
      }
    }
    if (a.has_drive) {
#pragma unroll
      for (int m = 0; m < P; ++m) {
        const int64_t ri = (int64_t)L.y * N + t + m * T;
        float2 q = cmul(a.drv_r0[ri], a.drv_t0);
        q = make_float2(q.x * a.drv_dz, q.y * a.drv_dz);
        v[1][m] = make_float2(v[1][m].x + q.y, v[1][m].y - q.x);
        q = cmul(a.drv_r1[ri], a.drv_t1);
        q = make_float2(q.x * a.drv_dz, q.y * a.drv_dz);
        v[1][m] = make_float2(v[1][m].x + q.y, v[1][m].y - q.x);
      }
    }
    if (a.has_b) {
      const NLParams2* p = reinterpret_cast<const NLParams2*>(a.nlp_b) + 2 * item;
      const NLParams2 p1 = p[0], p2 = p[1];
      nl2_block<P>(v[0], v[1], p1, p2, vr, vi);
    }
  }

  if (a.forward_last) fft_line<N, P, G, false, G, NLSE_ROW_PADSH, AR, SYNC>(v, t, W, tw, lline, LINE);

  if (a.out_scale != 1.f) {
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int m = 0; m < P; ++m) v[g][m] = make_float2(v[g][m].x * a.out_scale, v[g][m].y * a.out_scale);
  }
  if (active) {
    if (a.through >= through_need(8 * T)) {
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int m = 0; m < P; ++m) A0.store<ST_THROUGH>(v[g][m], d, g * cs + 8u * m * T);
    } else {
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int m = 0; m < P; ++m) A0.store(v[g][m], d, g * cs + 8u * m * T);
    }
  }
}

template <int N, int P, int LPB, int G, bool GEN = false, int AR = F64>
__global__ __launch_bounds__(LPB*(N / P)) void k_row(RowArgs a) {
  __shared__ xchg_t<AR> lds[row_lds_size<N, LPB, G>()];
  row_body<N, P, LPB, G, GEN, AR>(a, (int64_t)blockIdx.x * LPB, lds);
}

struct ColArgs {
  float2* A;
  int64_t nslabs;      // items * components
  int NX;              // columns per slab
  int ncomp;           // propagator component = slab % ncomp
  const double2* tw;   // twiddles of the column length (FP64 ratio pairs)
  int do_fwd;          // F_y
  int do_prop;         // multiply by the propagator (with `scale`)
  int do_inv;          // I_y
  int pkind;           // PROP_SEP64 or PROP_C64
  const double2* px;   // [ncomp][NX]   separable factors exp(-i phi_x)
  const double2* py;   // [ncomp][NY]   exp(-i phi_y)
  const float2* ptab;  // [ncomp][NY][NX] dense complex64 propagator
  const double2* pt;   // [NT] temporal factor of the 3-D propagator (PROP_SEP3D)
  const double2* ptab128;  // [N][NX] dense complex128 propagator (PROP_C128)
  const float* kq;     // [N/2+1][NX/2+1] real spectrum quadrant (PROP_KREAL)
  int nt;              // columns = NX * NT for PROP_SEP3D
  float scale;         // 1/(NX NY) folded into the propagator
  float out_scale;     // applied to the stored result when no propagator
  int through;         // level of the field's stores (through_level)
};

// Column sweep.  A block covers W = WT*G adjacent columns of one slab:
// WT threads across (consecutive lanes read consecutive columns), each
// thread owning G columns (c0 + g*WT + cw) so that twiddles and the y
// factor of the propagator are shared; LDS exchanges run in rounds of GR
// columns per thread column.
// LDS entries of one column block.
template <int N, int WT, int GR, typename X>
constexpr int col_lds_size() {
  return WT * GR * ColLine<N, WT, X>::SIZE;
}

// The propagator on the natural sets w of G columns c0 + g*CS: complex64
// products (float2 sets) for the complex64 propagators, FP64 products
// (double2) for the complex128 ones.
template <int KIND>
using prop_t = typename std::conditional<KIND == PROP_SEP3D || KIND == PROP_C128, double2, float2>::type;

template <int N, int P, int G, int CS, int KIND>
__device__ __forceinline__ void col_prop(const ColArgs& a, prop_t<KIND> (&w)[G][P], int comp, int t, int c0) {
  constexpr int T = N / P;
  if constexpr (KIND == PROP_SEP64) {
    const Buf pyb(a.py + comp * N);
    double2 px[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      px[g] = a.px[comp * a.NX + c0 + g * CS];
      px[g].x *= (double)a.scale;
      px[g].y *= (double)a.scale;
    }
#pragma unroll
    for (int m = 0; m < P; ++m) {
      const double2 py = pyb.load<double2>(16u * t, 16u * m * T);
#pragma unroll
      for (int g = 0; g < G; ++g) w[g][m] = prop_sep_c64(w[g][m], px[g], py);
    }
  } else if constexpr (KIND == PROP_SEP3D) {
    // column c = x*NT + t of an (NY, NX, NT) field: complex64(px*py)
    // times the complex128 temporal factor
    const Buf pyb(a.py);
    double2 px[G], pt[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int col = c0 + g * CS;
      px[g] = a.px[col / a.nt];
      pt[g] = a.pt[col % a.nt];
      pt[g].x *= (double)a.scale;
      pt[g].y *= (double)a.scale;
    }
#pragma unroll
    for (int m = 0; m < P; ++m) {
      const double2 py = pyb.load<double2>(16u * t, 16u * m * T);
#pragma unroll
      for (int g = 0; g < G; ++g) w[g][m] = prop_sep3d(w[g][m], px[g], py, pt[g]);
    }
  } else {
    static_assert(KIND == PROP_C128, "kinds addressed by column");
    const double2* pt = a.ptab128 + (int64_t)opaque((uint32_t)t) * a.NX + c0;
#pragma unroll
    for (int m = 0; m < P; ++m) {
#pragma unroll
      for (int g = 0; g < G; ++g)
        w[g][m] = prop_c128(w[g][m], pt[(int64_t)(m * T) * a.NX + g * CS], (double)a.scale);
      // no more than four rows of the table in registers
      if (m % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// A dense complex64 propagator read as the field is: from the tile's uniform
// address pt, the lane's offset d and the row stride rs.
template <int P, int G, int WT, bool PAIRED>
__device__ __forceinline__ void col_prop_dense(const Buf& pt, float2 (&w)[G][P], uint32_t d, uint32_t rs, float scale) {
#pragma unroll
  for (int m = 0; m < P; ++m) {
    if constexpr (PAIRED) {
      const float4 q = pt.load<float4>(d, m * rs);
      w[0][m] = prop_c64(w[0][m], make_float2(q.x, q.y), scale);
      w[1][m] = prop_c64(w[1][m], make_float2(q.z, q.w), scale);
    } else {
#pragma unroll
      for (int g = 0; g < G; ++g) w[g][m] = prop_c64(w[g][m], pt.load<float2>(d, m * rs + 8u * g * WT), scale);
    }
  }
}

// Column sweep body for tile `b` (tile index over slabs x tiles per slab).
// PK: the propagator kind compiled in.  BIG: slabs of 4 GiB and more, addressed
// by 64 bits.
template <int N, int P, int WT, int G, int GR, int PK, int FA = F64, bool BIG = false>
__device__ __forceinline__ void col_body(const ColArgs& a, int64_t b, xchg_t<FA>* lds) {
  using PL = Plan<N, P>;
  constexpr int T = PL::T;
  constexpr int LINE = ColLine<N, WT, xchg_t<FA>>::SIZE;
  constexpr int TILE = WT * G;

  const int cw = threadIdx.x % WT;
  const int t = threadIdx.x / WT;
  const uint32_t tiles = (uint32_t)a.NX / TILE;
  const uint32_t slab = (uint32_t)b / tiles;
  // column of line g: c0 + g * CS.  Two lines per thread take adjacent
  // columns (PAIRED, CS = 1), so a thread moves 16 bytes per row and a
  // wave's load covers whole 64-byte row segments; otherwise lines are WT
  // apart (a one-column tile, WT = G = 1, also has CS = 1 but is not paired)
  constexpr bool PAIRED = G == 2 && NLSE_COL_PAIRED;
  constexpr int CS = PAIRED ? 1 : WT;
  const int u0 = (int)((uint32_t)b - slab * tiles) * TILE;  // uniform: first column of the tile
  const int cl = PAIRED ? G * cw : cw;  // this thread's first column in the tile
  const int c0 = u0 + cl;
  // slabs below 4 GiB are addressed from a uniform descriptor (the launcher
  // chooses)
  float2* const A0 = a.A + (int64_t)slab * N * a.NX + u0;
  // (BIG: the lane's 64-bit address, found again for the stores)
  auto big_at = [&]() { return A0 + (int64_t)opaque((uint32_t)t) * a.NX + cl; };
  const Buf AB(A0), tw(a.tw);
  const uint32_t rs = 8u * (uint32_t)T * (uint32_t)a.NX;
  const uint32_t d = 8u * ((uint32_t)t * (uint32_t)a.NX + (uint32_t)cl);
  xchg_t<FA>* lline = lds + cw * GR * LINE;

  float2 v[G][P];
  const float2* const in = BIG ? big_at() : nullptr;
#pragma unroll
  for (int m = 0; m < P; ++m) {
    if constexpr (BIG) {
#pragma unroll
      for (int g = 0; g < G; ++g) v[g][m] = in[(int64_t)(m * T) * a.NX + g * CS];
    } else if constexpr (PAIRED) {
      const float4 q = AB.load<float4>(d, m * rs);
      v[0][m] = make_float2(q.x, q.y);
      v[1][m] = make_float2(q.z, q.w);
    } else {
#pragma unroll
      for (int g = 0; g < G; ++g) v[g][m] = AB.load<float2>(d, m * rs + 8u * g * WT);
    }
  }
  const Twid<N, P> W = load_twiddles<N, P>(tw, t);

  constexpr int PADSH = 3;
  if constexpr (PK != PK_NONE && PK != PROP_KREAL) {
    // F_y, propagator, I_y; with a complex128 propagator the field stays in
    // FP64 from the last forward stage to the first inverse one
    prop_t<PK> w[G][P];
    fft_line_io<N, P, G, false, GR, PADSH, FA, SYNC_BLOCK>(v, w, t, W, tw, lline, LINE);
    const int comp = (int)(slab % (uint32_t)a.ncomp);
    if constexpr (PK == PROP_C64) {
      col_prop_dense<P, G, WT, PAIRED>(Buf(a.ptab + (int64_t)comp * N * a.NX + u0), w, d, rs, a.scale);
    } else {
      col_prop<N, P, G, CS, PK>(a, w, comp, t, c0);
    }
    fft_line_io<N, P, G, true, GR, PADSH, FA, SYNC_BLOCK>(w, v, t, W, tw, lline, LINE);
  } else {
    if (a.do_fwd) fft_line<N, P, G, false, GR, PADSH, FA>(v, t, W, tw, lline, LINE);
    if (PK == PROP_KREAL && a.do_prop) {
      // even real spectrum: entry (ky, kx) of the quadrant table at
      // (min(ky, N-ky), min(kx, NX-kx))
      const int hx = a.NX / 2 + 1;
      int kx[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int col = c0 + g * CS;
        kx[g] = col <= a.NX / 2 ? col : a.NX - col;
      }
#pragma unroll
      for (int m = 0; m < P; ++m) {
        const int ky = t + m * T;
        const int kyq = ky <= N / 2 ? ky : N - ky;
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const float f = a.kq[kyq * hx + kx[g]] * a.scale;
          v[g][m] = make_float2(v[g][m].x * f, v[g][m].y * f);
        }
      }
    }
    if (a.do_inv) fft_line<N, P, G, true, GR, PADSH, FA>(v, t, W, tw, lline, LINE);
  }

  if (a.out_scale != 1.f) {
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int m = 0; m < P; ++m) v[g][m] = make_float2(v[g][m].x * a.out_scale, v[g][m].y * a.out_scale);
  }
  auto put = [&](auto st) __attribute__((always_inline)) {
    constexpr int ST = decltype(st)::value;
    float2* const out = BIG ? big_at() : nullptr;
#pragma unroll
    for (int m = 0; m < P; ++m) {
      if constexpr (BIG) {
#pragma unroll
        for (int g = 0; g < G; ++g) out[(int64_t)(m * T) * a.NX + g * CS] = v[g][m];
      } else if constexpr (PAIRED) {
        AB.template store<ST>(make_float4(v[0][m].x, v[0][m].y, v[1][m].x, v[1][m].y), d, m * rs);
      } else {
#pragma unroll
        for (int g = 0; g < G; ++g) AB.template store<ST>(v[g][m], d, m * rs + 8u * g * WT);
      }
    }
  };
  if (!BIG && a.through >= through_need(8 * TILE)) put(std::integral_constant<int, ST_THROUGH>{});
  else put(std::integral_constant<int, ST_BACK>{});
}

template <int N, int P, int WT, int G, int GR, int PK, int FA = F64, bool BIG = false>
__global__ __launch_bounds__(WT*(N / P)) void k_col(ColArgs a) {
  __shared__ xchg_t<FA> lds[col_lds_size<N, WT, GR, xchg_t<FA>>()];
  // XCD-aware tile order: workgroups are dealt round-robin to the 8 XCDs,
  // so block b runs on XCD b % 8; give each XCD a contiguous range of
  // tiles so that the two 64-byte halves of a 128-byte line are fetched
  // by neighbouring tiles on the same XCD (one L2 fill instead of two)
  const int64_t nblk = (int64_t)gridDim.x;
  const int64_t b = (nblk % 8 == 0) ? (int64_t)(blockIdx.x % 8) * (nblk / 8) + blockIdx.x / 8 : blockIdx.x;
  col_body<N, P, WT, G, GR, PK, FA, BIG>(a, b, lds);
}

// Intensity convolution over the full NY-row torus (a response given by
// its spectrum) for one-component fields whose intensity rows are packed
// in pairs (p, p + M), M = NY/2, along x:  Z(p, kx) = F_x(I_p + i I_{p+M}).
// Unit j in [0, NX/2] owns the columns a = j and b = (NX - j) mod NX: it
// unpacks the spectra of the two real rows,
//   X_p(j) = (Z(p,a) + conj Z(p,b)) / 2,   X_{p+M}(j) = (Z(p,a) - conj Z(p,b)) / 2i,
// into one NY-point column (a thread's set m < P/2 holds rows p = t + mT,
// m >= P/2 the rows p + M), applies I_y K^ F_y, and packs the result back
// into both columns (the convolved rows are real, so their spectra at -j
// are the conjugates).  Half the column work of transforming every row's
// intensity on its own.  Units past NX/2 in the last tile compute unit 0
// again without storing (every thread passes the barriers).
template <int N, int P, int WT>
__global__ __launch_bounds__(WT*(N / P)) void k_colu(ColArgs a) {
  using PL = Plan<N, P>;
  constexpr int T = PL::T;
  constexpr int LINE = ColLine<N, WT, float2>::SIZE;
  constexpr int H = P / 2;
  static_assert(H * T == N / 2, "the first half of a natural set covers rows [0, N/2)");
  __shared__ float2 lds[col_lds_size<N, WT, 1, float2>()];
  const int units = a.NX / 2 + 1;
  const int tiles = (units + WT - 1) / WT;
  const int64_t nblk = (int64_t)gridDim.x;
  const int64_t bb = (nblk % 8 == 0) ? (int64_t)(blockIdx.x % 8) * (nblk / 8) + blockIdx.x / 8 : blockIdx.x;
  const int64_t slab = bb / tiles;
  const int jt = (int)(bb % tiles) * WT;
  const uint32_t nx = (uint32_t)a.NX;
  const int cw = threadIdx.x % WT;
  const int t = threadIdx.x / WT;
  // this thread's unit and the byte offsets of its two columns; found again
  // after the transforms, which need every register of 1024-thread blocks
  struct Unit {
    int j;
    bool act, two;
    uint32_t da, db;
  };
  auto unit = [&]() __attribute__((always_inline)) {
    const uint32_t id = opaque(threadIdx.x);
    Unit u;
    const int j0 = jt + (int)(id % WT);
    u.act = j0 < units;
    u.j = u.act ? j0 : 0;
    const uint32_t cb = u.j == 0 ? 0u : nx - (uint32_t)u.j;
    u.two = cb != (uint32_t)u.j;
    u.da = 8u * (id / WT * nx + (uint32_t)u.j);
    u.db = 8u * (id / WT * nx + cb);
    return u;
  };
  float2* lline = lds + cw * LINE;
  // (a slab of Z and the spectrum quadrant are far below 4 GiB)
  const Buf Z(a.A + slab * (int64_t)(N / 2) * a.NX), kq(a.kq), tw(a.tw);
  const uint32_t rs = 8u * (uint32_t)T * (uint32_t)a.NX;
  const Twid<N, P> W = load_twiddles<N, P>(tw, t);

  float2 v[1][P];
  const Unit in = unit();
#pragma unroll
  for (int m = 0; m < H; ++m) {
    const float2 za = Z.load<float2>(in.da, m * rs), zb = Z.load<float2>(in.db, m * rs);
    v[0][m] = make_float2(0.5f * (za.x + zb.x), 0.5f * (za.y - zb.y));
    v[0][m + H] = make_float2(0.5f * (za.y + zb.y), 0.5f * (zb.x - za.x));
  }
  fft_line<N, P, 1, false, 1, 3, F64>(v, t, W, tw, lline, LINE);
  const int hx = a.NX / 2 + 1, jq = unit().j, tq = (int)(opaque(threadIdx.x) / WT);
#pragma unroll
  for (int m = 0; m < P; ++m) {
    const int ky = tq + m * T;
    const int kyq = ky <= N / 2 ? ky : N - ky;
    const float f = kq.load<float>(4u * (uint32_t)(kyq * hx + jq), 0) * a.scale;
    v[0][m] = make_float2(v[0][m].x * f, v[0][m].y * f);
  }
  fft_line<N, P, 1, true, 1, 3, F64>(v, t, W, tw, lline, LINE);
  // the results are rounded before the branches (else the last stage's FP64
  // values are kept through them, and spill)
#pragma unroll
  for (int m = 0; m < P; ++m) {
    v[0][m].x = __builtin_bit_cast(float, opaque(__builtin_bit_cast(uint32_t, v[0][m].x)));
    v[0][m].y = __builtin_bit_cast(float, opaque(__builtin_bit_cast(uint32_t, v[0][m].y)));
  }
  const Unit out = unit();
  if (out.act) {
#pragma unroll
    for (int m = 0; m < H; ++m)
      Z.store(make_float2(v[0][m].x - v[0][m + H].y, v[0][m].y + v[0][m + H].x), out.da, m * rs);
    if (out.two) {
#pragma unroll
      for (int m = 0; m < H; ++m)
        Z.store(make_float2(v[0][m].x + v[0][m + H].y, v[0][m + H].x - v[0][m].y), out.db, m * rs);
    }
  }
}

// Intensity-spectrum column sweep (PROP_KREAL) and the band pass of the
// nonlocal response in one launch: blocks [0, ncol) run column tiles of W =
// WT*G columns (one LDS round per line), the others run blockDim/256 band
// tiles each, so the band pass (matrix cores, or VALU for wide kernels)
// runs beside the sweep (VALU, LDS and memory) instead of after it.
// The two read disjoint data (Z; the real-space field) and write disjoint
// data (Z; the band values).  LDS is dynamic: the larger of the column
// tile's and the band tiles' needs.
template <int N, int P, int WT, int G, int PITCH>
__global__ __launch_bounds__(WT*(N / P)) void k_colz_band(ColArgs c, BandArgs b, int64_t ncol, int64_t nband,
                                                          int band_floats, int band_first) {
  extern __shared__ float4 smem4[];
  float* smem = reinterpret_cast<float*>(smem4);
  constexpr int TPB = WT * (N / P) / (64 * BAND_WAVES);
  const int64_t nbb = (nband + TPB - 1) / TPB;
  // band_first: the long-running band tiles are dispatched before the
  // sweep's tiles, which then fill in beside them
  const int64_t bx = band_first ? ((int64_t)blockIdx.x < nbb ? (int64_t)blockIdx.x + ncol : (int64_t)blockIdx.x - nbb)
                                : (int64_t)blockIdx.x;
  if (bx < ncol) {
    // XCD-aware order as in k_col
    const int64_t tb = (ncol % 8 == 0) ? (bx % 8) * (ncol / 8) + bx / 8 : bx;
    col_body<N, P, WT, G, 1, PROP_KREAL>(c, tb, reinterpret_cast<float2*>(smem));
  } else {
    const int sub = threadIdx.x / (64 * BAND_WAVES);
    const int64_t item = (bx - ncol) * TPB + sub;
    const bool real = item < nband;
    const int64_t it = real ? item : nband - 1;
    if (b.mfma)
      band_mfma_body(b, (int)(it % b.ntiles), it / b.ntiles, threadIdx.x % (64 * BAND_WAVES),
                     smem + (size_t)sub * band_floats, real);
    else
      band_body<PITCH>(b, (int)(it % b.ntiles), it / b.ntiles, threadIdx.x % (64 * BAND_WAVES),
                       smem + (size_t)sub * band_floats, real);
  }
}

// ----------------------------------------------------------------- 1-D
// Whole 1-D runs: every line is independent, so one launch performs all
// `nsteps` steps of LPB lines (G = 1 or component pairs G = 2) in
// registers and LDS: [N(dz/2)] F, * P/N (complex128 propagator, FP64
// multiply), I, N(dz or dz/2).  16 B per point for the whole run.
struct Line1DArgs {
  float2* A;
  int64_t ngroups;        // lines (G=1) or line pairs (G=2)
  const double2* tw;
  const double2* prop;    // [ncomp][N] complex128 propagator
  double scale;           // 1/N
  int64_t nsteps;
  int precision;          // 0 single, 1 double
  int loss_sat;
  const void* nl_full;    // NLParams1[items] / NLParams2[items*2]
  const void* nl_pre;
  const void* nl_post;
  const RabiParams* rabi; // [items] or null
  const void* V;          // [N] raw potential
  int vkind;
  const double* nlk;      // nonlocal kernel [2*nlr+1] (null: local response)
  int nlr;
  int general;            // the loss varies from point to point (see nl1_block_I)
};

// KEEP: the twiddles too stay in registers for the whole run.
template <int N, int P, int LPB, int G, bool GEN = false, int AR = F64, bool KEEP = false>
__global__ __launch_bounds__(LPB*(N / P)) void k_line1d(Line1DArgs a) {
  using PL = Plan<N, P>;
  constexpr int T = PL::T;
  constexpr int LINE = LdsLine<N, NLSE_ROW_PADSH, 0>::SIZE;
  constexpr int SYNC = T <= 64 ? SYNC_WAVE : SYNC_BLOCK;
  __shared__ xchg_t<AR> lds[LPB * G * LINE];
  const int li = threadIdx.x / T;
  const int t = threadIdx.x % T;
  const int64_t gi = (int64_t)blockIdx.x * LPB + li;
  const bool active = gi < a.ngroups;
  const int64_t item = active ? gi : 0;
  int64_t off[G];
  off[0] = item * G * N;
  if constexpr (G == 2) off[1] = off[0] + N;
  xchg_t<AR>* lline = lds + li * G * LINE;

  float2 v[G][P];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int m = 0; m < P; ++m) v[g][m] = active ? a.A[off[g] + t + m * T] : make_float2(0.f, 0.f);
  float vr[P], vi[P];
  load_v_set<P, T, GEN>(a.V, a.vkind, 0, (uint32_t)t, vr, vi);
  // the propagator and the parameters stay in registers for the whole run
  const Buf tw(a.tw);
  const Twid<N, P, KEEP> W = load_twiddles<N, P, KEEP>(tw, t);
  double2 pr[G][P];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int m = 0; m < P; ++m) {
      pr[g][m] = a.prop[g * N + t + m * T];
      pr[g][m].x *= a.scale;
      pr[g][m].y *= a.scale;
    }
  using NL = typename std::conditional<G == 1, NLParams1, NLParams2>::type;
  NL pre[G], post[G];  // (pre: "double" only)
#pragma unroll
  for (int g = 0; g < G; ++g) {
    post[g] = reinterpret_cast<const NL*>(a.precision == 1 ? a.nl_post : a.nl_full)[G * item + g];
    pre[g] = a.precision == 1 ? reinterpret_cast<const NL*>(a.nl_pre)[G * item + g] : post[g];
  }
  const bool has_rabi = G == 2 && a.rabi != nullptr && a.precision == 0;
  RabiParams rb{};
  if (has_rabi) rb = a.rabi[item];

  // Always inlined: left to the compiler, pairs of lines of 16 points per lane had
  // it as a function of its own, on a line in memory, and took twice as long (600
  // pairs of 1024, 200 steps: 2.8 -> 5.1 ms).  Two copies, for the local and the
  // convolved intensities: one for both took 5-8 % longer at 4 points per lane.
  auto apply_nl = [&](const NL (&p)[G]) __attribute__((always_inline)) {
    if (a.nlk != nullptr) {
      // nonlocal response: convolved intensities (nlse_1d.py:65-66 kernel)
      float I[G][P];
      conv1d_intensity<N, P, G>(v, I, reinterpret_cast<float*>(lline), t, a.nlk, a.nlr);
      if constexpr (G == 1) nl1_block_I<P, GEN>(v[0], I[0], p[0], a.loss_sat, a.vkind == V_CPLX, vr, vi);
      else nl2_block_I<P>(v[0], v[1], I[0], I[1], p[0], p[1], vr, vi);
    } else if constexpr (G == 1) {
      nl1_block<P, GEN>(v[0], p[0], a.loss_sat, a.vkind == V_CPLX, vr, vi);
    } else {
      nl2_block<P>(v[0], v[1], p[0], p[1], vr, vi);
    }
  };

  for (int64_t s = 0; s < a.nsteps; ++s) {
    if (a.precision == 1) apply_nl(pre);
    double2 w[G][P];
    fft_line_io<N, P, G, false, G, NLSE_ROW_PADSH, AR, SYNC>(v, w, t, W, tw, lline, LINE);
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int m = 0; m < P; ++m) w[g][m] = prop_c128(w[g][m], pr[g][m], 1.0);
    fft_line_io<N, P, G, true, G, NLSE_ROW_PADSH, AR, SYNC>(w, v, t, W, tw, lline, LINE);
    apply_nl(post);
    if (has_rabi) {
#pragma unroll
      for (int m = 0; m < P; ++m) rabi(v[0][m], v[G - 1][m], rb);
    }
  }
  if (active) {
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int m = 0; m < P; ++m) a.A[off[g] + t + m * T] = v[g][m];
  }
}

}  // namespace nlse
