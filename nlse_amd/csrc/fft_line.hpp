// Line FFT building blocks for gfx950 (CDNA4): complex64 Stockham transform
// of a power-of-two line held as a "natural set" in registers.
//
// A line of N points is owned by T = N/P threads; thread t holds
//     v[m] = x[t + m*T],   m = 0 .. P-1.
// Stage s (radix R, Ns = product of the radices of the stages before it)
// evaluates N/R butterflies j = t + b*T (b < P/R), whose inputs are exactly
// v[b + k*P/R] (k < R) -- a thread's own registers -- and whose outputs go to
// the Stockham positions (j/Ns)*Ns*R + j%Ns + k*Ns.  The first stage reads
// registers loaded straight from HBM, the last stage (Ns = N/R) lands again
// on the natural set, so a forward transform, a pointwise operator and an
// inverse transform chain without an extra exchange.  Middle stages exchange
// through LDS with one float2 of padding every 16 entries, which keeps the
// b64 accesses of each 16-lane group on distinct banks.
//
// Arithmetic: each stage converts its R inputs to FP64, applies the radix-R
// butterfly with its twiddles in FP64 (dft_fma), and rounds the R outputs once
// to complex64 when it stores them (to LDS, or to the natural set after the last
// stage); F64X transforms exchange FP64 and round once.  On gfx950 an FP64 add,
// multiply or FMA issues at the same rate as an FP32 one without packed math, so
// this costs no more than compensated FP32 butterflies, and it leaves one
// rounding per stage instead of one per butterfly level.  The long split-step
// runs accumulate this rounding noise as sqrt(steps), so fewer roundings per
// transform is what keeps a 2001-step run close to an exactly rounded transform.
// FP64 twiddles also remove the systematic gain bias a table rounded to
// complex64 would add (a mean |w|^2 - 1 of about -1e-8 per stage, -5e-8 per
// forward/inverse pair).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace nlse {

// ---------------------------------------------------------------- complex
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(fmaf(a.x, b.x, -a.y * b.y), fmaf(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ float sqmag(float2 a) { return a.x * a.x + a.y * a.y; }
__device__ __forceinline__ float2 conjf2(float2 a) { return make_float2(a.x, -a.y); }
// a * (-i)
__device__ __forceinline__ float2 mul_mi(float2 a) { return make_float2(a.y, -a.x); }

// FP64 butterfly arithmetic
__device__ __forceinline__ double2 to_f64(float2 a) { return make_double2((double)a.x, (double)a.y); }
__device__ __forceinline__ float2 to_f32(double2 a) { return make_float2((float)a.x, (float)a.y); }
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 mul_mi(double2 a) { return make_double2(a.y, -a.x); }
constexpr double K_R2 = 0.70710678118654752440084436210484904;  // 1/sqrt(2)
constexpr double K_C8 = 0.92387953251128675612818318939678829;  // cos(pi/8)
constexpr double K_S8 = 0.38268343236508977172845998403039887;  // sin(pi/8)

// ------------------------------------------------------------ radix plan
// Stages for N = 2^n with at most P points per thread: the remainder radix
// (2, 4 or 8) first, then radix-P stages.  P is 4, 8 or 16.
__host__ __device__ constexpr int ilog2c(int n) { return n <= 1 ? 0 : 1 + ilog2c(n >> 1); }

template <int N, int P>
struct Plan {
  static constexpr int LOGN = ilog2c(N);
  static constexpr int LOGP = ilog2c(P);
  static_assert((1 << LOGN) == N, "N must be a power of two");
  static_assert(P == 4 || P == 8 || P == 16, "P must be 4, 8 or 16");
  static_assert(N >= P, "line shorter than the per-thread set");
  static constexpr int FULL = LOGN / LOGP;        // radix-P stages
  static constexpr int REM = LOGN % LOGP;         // log2 of the remainder radix
  static constexpr int NSTAGES = FULL + (REM ? 1 : 0);
  static constexpr int T = N / P;                 // threads per line
  __host__ __device__ static constexpr int radix(int s) {
    return (REM && s == 0) ? (1 << REM) : P;
  }
  __host__ __device__ static constexpr int ns(int s) {  // product of radices before s
    int p = 1;
    for (int i = 0; i < s; ++i) p *= radix(i);
    return p;
  }
};

// Stores kept in the L2 until the kernel's end, or written through to memory
// (sc1) while the kernel runs: if the field's level (through_level) reaches what
// lanes that store `bytes` contiguous bytes need.
enum : int { ST_BACK = 0, ST_THROUGH = 16 };
constexpr int through_need(int bytes) { return bytes >= 64 ? 1 : (bytes >= 16 ? 2 : 3); }

// Memory seen from a uniform address: a buffer descriptor in scalar registers.
// An access is one instruction at a per-lane 32-bit byte offset plus a uniform
// one, without vector instructions for 64-bit addresses and without keeping
// the addresses of a line's loads for its stores.
struct Buf {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ explicit Buf(const void* p)
      : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(uniform(p)), 0, -1, 0x00027000)) {}
  static __device__ __forceinline__ const void* uniform(const void* p) {
    const uint64_t q = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)q);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(q >> 32));
    return reinterpret_cast<const void*>(((uint64_t)hi << 32) | lo);
  }
  template <typename T>
  __device__ __forceinline__ T load(uint32_t lane, uint32_t uni) const {
    static_assert(sizeof(T) == 4 || sizeof(T) == 8 || sizeof(T) == 16, "access width");
    if constexpr (sizeof(T) == 4) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, lane, uni, 0));
    else if constexpr (sizeof(T) == 8)
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, lane, uni, 0));
    else return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(r, lane, uni, 0));
  }
  template <int ST = ST_BACK>
  __device__ __forceinline__ void store(float2 x, uint32_t lane, uint32_t uni) const {
    typedef uint32_t u2 __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, x), r, lane, uni, ST);
  }
  template <int ST = ST_BACK>
  __device__ __forceinline__ void store(float4 x, uint32_t lane, uint32_t uni) const {
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, x), r, lane, uni, ST);
  }
};

// Padding of the row kernels' LDS lines (one float2 every 2^NLSE_ROW_PADSH
// entries); the column kernel passes its own.
#ifndef NLSE_ROW_PADSH
#define NLSE_ROW_PADSH 4
#endif

// LDS line layout: one float2 of padding every 2^PADSH entries, plus EXTRA
// float2 at the end of each line (staggers the lines of a multi-line
// block across banks).
template <int N, int PADSH, int EXTRA>
struct LdsLine {
  static constexpr int SIZE = N + (N >> PADSH) + EXTRA + 1;
};

// Lines of a tile of WT columns (entries of type X, padded every 8): lanes go
// over the columns first, and LDS serves the entries of 128 bytes at a time, so
// the lines of a tile start 128 bytes / WT apart modulo 128.  32 bytes apart
// whatever the tile, a 2048-point sweep of 8 columns counted 8192 clocks of
// bank conflicts per CU, of which other waves hid most: 2048^2 nonlocal step
// 92.6 -> 91.2 us, complex128 1024^2 37.2 -> 36.5, 2048^2 84.1 -> 82.6 us.
template <int N, int WT, typename X>
struct ColLine {
  static constexpr int ENTRIES = 128 / (int)sizeof(X);
  static constexpr int EXTRA = WT == 1 ? 0 : (WT < ENTRIES ? ENTRIES / WT - 1 : 0);
  static constexpr int SIZE = LdsLine<N, 3, EXTRA>::SIZE;
};

template <int PADSH>
__host__ __device__ __forceinline__ constexpr int lds_pad(int i) { return i + (i >> PADSH); }

// Ratio twiddles {cos, tan} of the factored butterflies (dft_fma): R/2 entries
// per stage of radix R and index jm, the stages of P = 16, 8 and 4 one after the
// other: one table per line length serves every number of points per thread.
__host__ __device__ constexpr int rt_offset(int n, int p, int stage) {
  const int logn = ilog2c(n), logp = ilog2c(p), rem = logn % logp;
  int off = 0, ns = rem ? (1 << rem) : p;
  for (int i = 1; i < stage; ++i) {
    off += p / 2 * ns;
    ns *= p;
  }
  return off;
}
__host__ __device__ constexpr int rt_size_np(int n, int p) {
  if (p > n) return 0;
  const int logn = ilog2c(n), logp = ilog2c(p);
  return rt_offset(n, p, logn / logp + (logn % logp ? 1 : 0));
}
__host__ __device__ constexpr int rt_base(int n, int p) {
  return (p < 16 ? rt_size_np(n, 16) : 0) + (p < 8 ? rt_size_np(n, 8) : 0);
}
__host__ __device__ constexpr int rt_size(int n) { return rt_size_np(n, 16) + rt_size_np(n, 8) + rt_size_np(n, 4); }

// Precision of a transform's exchanges: F64 rounds to complex64 once per stage,
// F64X carries FP64: one rounding per transform and no conversions between
// stages, for twice the LDS traffic.  Butterflies are FP64 in both.
enum FftArith : int { F64 = 0, F64X = 1 };

template <int AR>
using xchg_t = typename std::conditional<AR == F64X, double2, float2>::type;

// Who exchanges a line: the whole block (barriers), or one wave (the lines of
// a wave use their own LDS; the LDS operations of a wave complete in order, so
// a compiler fence is enough).
enum : int { SYNC_BLOCK = 0, SYNC_WAVE = 1 };

template <int SYNC>
__device__ __forceinline__ void line_sync() {
  if constexpr (SYNC == SYNC_BLOCK) {
    __syncthreads();
  } else {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

__device__ __forceinline__ double2 to_f64(double2 a) { return a; }
template <typename C>
__device__ __forceinline__ C from_f64(double2 a) {
  if constexpr (std::is_same<C, float2>::value) return to_f32(a);
  else return a;
}

// Radix-R butterfly in FP64 as log2 R layers of radix-2 ones, in the factored form
// for fused multiply-adds of E. Linzer and E. Feig (IEEE Trans. Signal Processing
// 41, 93, 1993): X[k] = E[k] +
// w W_R^k O[k], X[k + R/2] = E[k] - w W_R^k O[k] with E, O the transforms of
// the even and odd points for w^2.  A twiddle c + i s is applied as c (1 + i
// s/c), the c inside the additions: a butterfly is 6 FMAs where a complex
// product and two additions are 8, twiddles included: 12 operations per point
// of a twiddled radix-16 stage against 17 of the factored 4 x 4 form (VALU
// issue is what bounds the sweeps of large fields).  The R/2 pairs {c, s/c} of
// a stage: w W_R^k for k < R/4 (the others are -i times these), then the same
// for w^2 and R/2, and so on.  Where c is nearly zero s/c is as large and the
// product keeps its relative precision; c is never exactly zero (the table
// holds 6e-17 for a quarter turn).
__device__ __forceinline__ void bf2(double2 e, double2 o, double2 ct, bool mi, double2& x0, double2& x1) {
  const double vr = fma(-ct.y, o.y, o.x), vi = fma(ct.y, o.x, o.y);
  if (!mi) {
    x0 = make_double2(fma(ct.x, vr, e.x), fma(ct.x, vi, e.y));
    x1 = make_double2(fma(-ct.x, vr, e.x), fma(-ct.x, vi, e.y));
  } else {
    x0 = make_double2(fma(ct.x, vi, e.x), fma(-ct.x, vr, e.y));
    x1 = make_double2(fma(-ct.x, vi, e.x), fma(ct.x, vr, e.y));
  }
}
__device__ __forceinline__ void bf2(double2 e, double2 o, bool mi, double2& x0, double2& x1) {
  if (mi) o = mul_mi(o);
  x0 = cadd(e, o);
  x1 = csub(e, o);
}

// {cos, tan} of -2 pi k / R, k < R/4
template <int R, int K>
constexpr double2 const_ct() {
  static_assert(K > 0 && K < R / 4 && R <= 16, "W8, W16, W16^3");
  // (the tangents of the rounded cosines, as in the tables; 1 for W8, whose parts
  // then have one rounding in common and whose products are additions)
  constexpr double c = R == 8 || K == 2 ? K_R2 : (K == 1 ? K_C8 : K_S8);
  constexpr double t = R == 8 || K == 2 ? 1.0 : (K == 1 ? 0.41421356237309503 : 2.414213562373095);
  return double2{c, -t};
}

template <int R, bool TW, int K = 0>
__device__ __forceinline__ void dft_top(const double2* E, const double2* O, const double2* ct, double2* X) {
  if constexpr (K < R / 2) {
    constexpr int Q = R / 4;
    constexpr bool MI = R >= 4 && K >= Q;
    constexpr int KK = MI ? K - Q : K;
    if constexpr (TW) bf2(E[K], O[K], ct[KK], MI, X[K], X[K + R / 2]);
    else if constexpr (KK == 0) bf2(E[K], O[K], MI, X[K], X[K + R / 2]);
    else bf2(E[K], O[K], const_ct<R, KK>(), MI, X[K], X[K + R / 2]);
    dft_top<R, TW, K + 1>(E, O, ct, X);
  }
}

// points z(n) = ld(START + n * STEP), n < R
template <int R, bool TW, int START, int STEP, class Load>
__device__ __forceinline__ void dft_fma(Load ld, const double2* ct, double2* X) {
  if constexpr (R == 1) {
    X[0] = ld(START);
  } else {
    double2 E[R / 2], O[R / 2];
    constexpr int Q = R >= 4 ? R / 4 : 1;
    dft_fma<R / 2, TW, START, 2 * STEP>(ld, ct + Q, E);
    dft_fma<R / 2, TW, START + STEP, 2 * STEP>(ld, ct + Q, O);
    dft_top<R, TW>(E, O, ct, X);
  }
}

// The twiddles of a thread's stages, loaded once beside the field for lines of
// up to 512 points with less than 16 per thread (loads at each stage would
// expose their latency in the small fields these sets serve); else they would
// take the registers of a wave (16 per stage at P = 8), and each stage loads
// its own.
constexpr bool twid_kept(int n, int p) { return p < 16 && n <= 512; }

template <int N, int P, bool KEEP = twid_kept(N, P)>
struct Twid {
  static constexpr int NT = KEEP && Plan<N, P>::NSTAGES > 1 ? Plan<N, P>::NSTAGES - 1 : 1;
  double2 ct[NT][P / 2 > 0 ? P / 2 : 1];
};

// Byte offset of stage S's ratio pairs.
template <int N, int P, int S>
constexpr uint32_t stage_twiddles() {
  return 16u * (uint32_t)(rt_base(N, P) + rt_offset(N, P, S));
}

// A value the compiler cannot see through: what is computed from it is
// computed again (addresses, twiddle loads) instead of being kept in
// registers from one stage or transform to the next.
__device__ __forceinline__ uint32_t opaque(uint32_t x) {
  asm volatile("" : "+v"(x));
  return x;
}

template <int N, int P, int S>
__device__ __forceinline__ void load_stage_twiddles(double2 (&ct)[P / 2 > 0 ? P / 2 : 1], const Buf& tw, uint32_t jm) {
  constexpr int NS = Plan<N, P>::ns(S);
#pragma unroll
  for (int i = 0; i < P / 2; ++i) ct[i] = tw.load<double2>(16u * jm, stage_twiddles<N, P, S>() + 16u * i * NS);
}

template <int N, int P, bool KEEP, int S = 1>
__device__ __forceinline__ void load_twiddles_from(Twid<N, P, KEEP>& W, const Buf& tw, int t) {
  using PL = Plan<N, P>;
  if constexpr (S < PL::NSTAGES) {
    static_assert(PL::radix(S) == P, "only the first stage has another radix, and no twiddles");
    load_stage_twiddles<N, P, S>(W.ct[S - 1], tw, (uint32_t)(t & (PL::ns(S) - 1)));
    load_twiddles_from<N, P, KEEP, S + 1>(W, tw, t);
  }
}

template <int N, int P, bool KEEP = twid_kept(N, P)>
__device__ __forceinline__ Twid<N, P, KEEP> load_twiddles(const Buf& tw, int t) {
  Twid<N, P, KEEP> W;
  if constexpr (Plan<N, P>::NSTAGES > 1 && P >= 4 && KEEP) load_twiddles_from<N, P, KEEP>(W, tw, t);
  return W;
}

// One Stockham stage on G lines owned by the same thread, natural sets v in,
// w out (v and w may be the same registers).  Stages before the last exchange
// through LDS in rounds of GR lines (the LDS region holds GR lines per thread
// column: line g of round r lives at slot g - r*GR); the last stage (Ns = N/R)
// lands on the natural set.
template <int N, int P, int S, int G, int GR, int PADSH, int AR, int SYNC, bool KEEP, typename CI, typename CO>
__device__ __forceinline__ void fft_stage(CI (&v)[G][P], CO (&w)[G][P], int t, const Twid<N, P, KEEP>& W, const Buf& tw,
                                          xchg_t<AR>* lds, int lds_stride) {
  using PL = Plan<N, P>;
  constexpr int R = PL::radix(S);
  constexpr int NS = PL::ns(S);
  constexpr int NB = P / R;  // butterflies per thread
  constexpr bool LAST = (S == PL::NSTAGES - 1);
  constexpr int T = PL::T;
  static_assert(G % GR == 0, "lines per round must divide the lines per thread");
  // T a multiple of the padding period: no carry in lds_pad(t + m T)
  constexpr bool LDS_STEP = T % (1 << PADSH) == 0;
#pragma unroll
  for (int r = 0; r < G / GR; ++r) {
    if constexpr (!LAST) line_sync<SYNC>();  // the exchange before this one has been read
    const int ts = (int)opaque((uint32_t)t);
#pragma unroll
    for (int gg = 0; gg < GR; ++gg) {
      const int g = r * GR + gg;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int j = ts + b * T;
        const int jm = j & (NS - 1);
        // lds_pad(base + k NS) = lds_pad(base) + lds_pad(k NS): base mod
        // 2^PADSH and k NS mod 2^PADSH add without a carry (NS >= 2^PADSH,
        // or base mod NS R = jm < NS, or R divides 2^PADSH), so one address
        // serves all outputs through instruction offsets
        xchg_t<AR>* out = lds + gg * lds_stride + lds_pad<PADSH>((j / NS) * NS * R + jm);
        auto ld = [&](int k) { return to_f64(v[g][b + k * NB]); };
        auto st = [&](int k, double2 x) {
          if constexpr (LAST) w[g][b + k * NB] = from_f64<CO>(x);
          else out[lds_pad<PADSH>(k * NS)] = from_f64<xchg_t<AR>>(x);
        };
        double2 X[R];
        if constexpr (NS == 1) {
          dft_fma<R, false, 0, 1>(ld, (const double2*)nullptr, X);
        } else if constexpr (!KEEP) {
          double2 ct[P / 2];
          load_stage_twiddles<N, P, S>(ct, tw, opaque((uint32_t)jm));
          dft_fma<R, true, 0, 1>(ld, ct, X);
        } else {
          dft_fma<R, true, 0, 1>(ld, W.ct[S - 1], X);
        }
#pragma unroll
        for (int k = 0; k < R; ++k) st(k, X[k]);
      }
    }
    if constexpr (!LAST) {
      line_sync<SYNC>();
#pragma unroll
      for (int gg = 0; gg < GR; ++gg)
#pragma unroll
        for (int m = 0; m < P; ++m)
          w[r * GR + gg][m] = LDS_STEP ? lds[gg * lds_stride + lds_pad<PADSH>(ts) + lds_pad<PADSH>(m * T)]
                                       : lds[gg * lds_stride + lds_pad<PADSH>(ts + m * T)];
    }
  }
}

template <int N, int P, int S, int G, int GR, int PADSH, int AR, int SYNC, bool KEEP, typename CI, typename CO>
__device__ __forceinline__ void fft_stages_from(CI (&v)[G][P], CO (&w)[G][P], int t, const Twid<N, P, KEEP>& W, const Buf& tw,
                                                xchg_t<AR>* lds, int lds_stride) {
  if constexpr (S == Plan<N, P>::NSTAGES - 1) {
    fft_stage<N, P, S, G, GR, PADSH, AR, SYNC>(v, w, t, W, tw, lds, lds_stride);
  } else {
    xchg_t<AR> u[G][P];
    fft_stage<N, P, S, G, GR, PADSH, AR, SYNC>(v, u, t, W, tw, lds, lds_stride);
    fft_stages_from<N, P, S + 1, G, GR, PADSH, AR, SYNC>(u, w, t, W, tw, lds, lds_stride);
  }
}

template <int G, int P, typename C>
__device__ __forceinline__ void swap_parts(C (&v)[G][P]) {
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int m = 0; m < P; ++m) {
      C z = v[g][m];
      v[g][m].x = z.y;
      v[g][m].y = z.x;
    }
}

// Forward (INV=false) or unnormalised inverse (INV=true) DFT of G lines,
// natural set v in, natural set w out.  The inverse is swap(F(swap(x))) with
// swap(a + ib) = b + ia (= conj(F(conj x))), a register renaming.  An FP64
// input or output set is taken or left without rounding.
template <int N, int P, int G, bool INV, int GR, int PADSH, int AR, int SYNC, bool KEEP, typename CI, typename CO>
__device__ __forceinline__ void fft_line_io(CI (&v)[G][P], CO (&w)[G][P], int t, const Twid<N, P, KEEP>& W, const Buf& tw,
                                            xchg_t<AR>* lds, int lds_stride) {
  if constexpr (INV) swap_parts<G, P>(v);
  fft_stages_from<N, P, 0, G, GR, PADSH, AR, SYNC>(v, w, t, W, tw, lds, lds_stride);
  if constexpr (INV) swap_parts<G, P>(w);
}

template <int N, int P, int G, bool INV, int GR = G, int PADSH = NLSE_ROW_PADSH, int AR = F64, int SYNC = SYNC_BLOCK,
          bool KEEP>
__device__ __forceinline__ void fft_line(float2 (&v)[G][P], int t, const Twid<N, P, KEEP>& W, const Buf& tw,
                                         xchg_t<AR>* lds, int lds_stride) {
  fft_line_io<N, P, G, INV, GR, PADSH, AR, SYNC>(v, v, t, W, tw, lds, lds_stride);
}

}  // namespace nlse
