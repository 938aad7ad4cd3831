// Uneven batches of 2-D single-component fields (nlse_batch_*): many NLSE
// instances of different grid sizes and physical parameters advanced
// together, one launch per sweep and line length for the whole batch, or one
// per sweep.
//
// Work units are uniform in size whatever the grid: a row unit is
// 4096/NX rows of NX points (256 threads) and a column unit is 8192/NY
// columns of NY points (512 threads).  Every unit therefore moves the same
// bytes and does the same FFT work per point.  By default a block takes one
// pass of a unit; blocks of a smaller grid stride over the unit list, balanced
// without a work queue.  Each block reads its unit's instance descriptor (field
// pointer, tables, parameters) and runs the sweep body of that line length, in
// the plan (points per thread, exchange precision) that the member's own
// single-field run takes by default: small members (SMALL_FIELD) take the
// small-field plans, so every member gives bit for bit the result of its own
// run (row_points as given or tuned for that run aside).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "../../include/nlse_hip.h"
#include "common.hpp"
#include "lines.hpp"

namespace nlse {

struct BatchInst {
  RowArgs row;
  ColArgs col;
  const void* nl[3];  // NLParams1 of the three slots
  int nx, ny;
  int small;  // SMALL_FIELD
  float inv_nx, inv_ny;
};

struct BatchUnit {
  int inst;
  int pad;
  int64_t first;  // first row (row units) or column tile (column units)
};

struct BatchFlags {
  int inverse_first, forward_last, has_a, has_b, slot_a, slot_b;
  int timing;  // repeated sweeps: rescale by 1/N per sweep
};

// Row units of 4096/NX rows are PASSES row_body calls of LPB rows, column
// units of 8192/NY columns PASSES tiles of WT columns.  The per-length kernels
// deal out single passes, in blocks of THREADS threads: 256, or 512 for
// 2048-point columns (tiles of 4 columns, 32-byte row segments, at least).
// The kernels of all lengths (block sizes BROW_THREADS, BCOL_THREADS) deal out
// whole units.
constexpr int BROW_THREADS = 256;
constexpr int BCOL_THREADS = 512;

template <int N, bool SMALL>
struct BRow {
  using C = LineCfg<N>;
  static constexpr int P = SMALL ? C::PRS : C::PR;
  static constexpr int AR = SMALL ? C::ARS : F64;
  static constexpr int T = N / P;
  static constexpr int LPB = BROW_THREADS / T < 4096 / N ? BROW_THREADS / T : 4096 / N;
  static constexpr int PASSES = (4096 / N) / LPB;
  static constexpr int LDSB = row_lds_size<N, LPB, 1>() * (int)sizeof(xchg_t<AR>);
  static_assert(LPB * T == BROW_THREADS, "one block size for every length");
};

template <int N, bool SMALL, int THREADS = BCOL_THREADS>
struct BCol {
  using C = LineCfg<N>;
  static constexpr int P = SMALL ? C::PS : C::P;
  static constexpr int AR = SMALL ? C::ARS : F64;
  static constexpr int T = N / P;
  static constexpr int W = 8192 / N;
  static constexpr int WT = THREADS / T < W ? THREADS / T : W;
  static constexpr int PASSES = W / WT;
  static constexpr int LDSB = col_lds_size<N, WT, 1, xchg_t<AR>>() * (int)sizeof(xchg_t<AR>);
  static_assert(WT * T == THREADS, "whole blocks");
};
constexpr int bcol_threads(int n) { return n >= 2048 ? 512 : 256; }

static bool batch_len_ok(int64_t n) { return n == 128 || n == 256 || n == 512 || n == 1024 || n == 2048; }

// unit groups: line length, small-field plans or not
static int len_index(int64_t n, bool small) {
  return 2 * (n == 128 ? 0 : n == 256 ? 1 : n == 512 ? 2 : n == 1024 ? 3 : 4) + (small ? 1 : 0);
}
constexpr int NLEN = 10;

// Pass k of a unit of a row or column sweep.  GEN: some member's loss varies
// from point to point (see nl1_block_I).
template <int N, bool SMALL, bool GEN>
__device__ __forceinline__ void row_pass(const BatchInst& I, const BatchUnit& un, int k, const BatchFlags& f,
                                         void* lds) {
  using B = BRow<N, SMALL>;
  RowArgs a = I.row;
  a.inverse_first = f.inverse_first;
  a.forward_last = f.forward_last;
  a.has_a = f.has_a;
  a.has_b = f.has_b;
  a.nlp_a = I.nl[f.slot_a];
  a.nlp_b = I.nl[f.slot_b];
  a.out_scale = f.timing ? I.inv_nx : 1.f;
  row_body<N, B::P, B::LPB, 1, GEN, B::AR>(a, un.first + k * B::LPB, reinterpret_cast<xchg_t<B::AR>*>(lds));
}

template <int N, bool SMALL, int THREADS>
__device__ __forceinline__ void col_pass(const BatchInst& I, const BatchUnit& un, int k, const BatchFlags& f,
                                         void* lds) {
  using B = BCol<N, SMALL, THREADS>;
  ColArgs c = I.col;
  if (f.timing) c.scale = I.inv_ny;
  col_body<N, B::P, B::WT, 1, 1, PROP_SEP64, B::AR>(c, un.first * B::PASSES + k,
                                                    reinterpret_cast<xchg_t<B::AR>*>(lds));
}

// XCD-aware order: consecutive list entries (neighbouring column tiles,
// which share 128-byte lines when narrow) go to blocks on the same XCD
__device__ __forceinline__ int64_t xcd_block() {
  const int64_t grid = gridDim.x;
  return (grid % 8 == 0) ? (int64_t)(blockIdx.x % 8) * (grid / 8) + blockIdx.x / 8 : blockIdx.x;
}

// One kernel per line length: a single length per kernel keeps the register
// footprint of the plain sweeps (a kernel holding every length spills).  The
// blocks stride over the passes of the units.
template <int N, bool SMALL, bool GEN>
__global__ __launch_bounds__(BROW_THREADS) void k_batch_row(const BatchInst* __restrict__ inst,
                                                            const BatchUnit* __restrict__ units, int64_t nunits,
                                                            BatchFlags f) {
  using B = BRow<N, SMALL>;
  __shared__ double2 lds[B::LDSB / 16 + 1];
  for (int64_t u = blockIdx.x; u < nunits * B::PASSES; u += gridDim.x) {
    const BatchUnit un = units[u / B::PASSES];
    row_pass<N, SMALL, GEN>(inst[un.inst], un, (int)(u % B::PASSES), f, lds);
  }
}

template <int N, bool SMALL>
__global__ __launch_bounds__(bcol_threads(N)) void k_batch_col(const BatchInst* __restrict__ inst,
                                                               const BatchUnit* __restrict__ units, int64_t nunits,
                                                               BatchFlags f) {
  using B = BCol<N, SMALL, bcol_threads(N)>;
  __shared__ double2 lds[B::LDSB / 16 + 1];
  for (int64_t u = xcd_block(); u < nunits * B::PASSES; u += gridDim.x) {
    const BatchUnit un = units[u / B::PASSES];
    col_pass<N, SMALL, bcol_threads(N)>(inst[un.inst], un, (int)(u % B::PASSES), f, lds);
  }
}

// One persistent launch per sweep for the whole batch, whatever the line
// lengths: each unit's length picks the body (a block-uniform branch).  The
// bodies are separate (not inlined) functions, so the kernel's register
// allocation is the largest body's, not that of one giant inlined switch
// (which spilled), and the LDS array is the largest length's.
template <int N, bool SMALL, bool GEN>
__device__ __noinline__ void batch_row_unit(const BatchInst& I, const BatchUnit& un, const BatchFlags& f, void* lds) {
#pragma unroll 1
  for (int k = 0; k < BRow<N, SMALL>::PASSES; ++k) row_pass<N, SMALL, GEN>(I, un, k, f, lds);
}

template <int N, bool SMALL>
__device__ __noinline__ void batch_col_unit(const BatchInst& I, const BatchUnit& un, const BatchFlags& f, void* lds) {
#pragma unroll 1
  for (int k = 0; k < BCol<N, SMALL>::PASSES; ++k) col_pass<N, SMALL, BCOL_THREADS>(I, un, k, f, lds);
}

constexpr int cmax(int a, int b) { return a > b ? a : b; }
template <int N, bool SMALL>
using BColAll = BCol<N, SMALL, BCOL_THREADS>;
template <template <int, bool> class B>
constexpr int lds_all() {
  return cmax(cmax(cmax(B<128, false>::LDSB, B<128, true>::LDSB), cmax(B<256, false>::LDSB, B<256, true>::LDSB)),
              cmax(cmax(B<512, false>::LDSB, B<512, true>::LDSB), cmax(B<1024, false>::LDSB, B<2048, false>::LDSB)));
}

template <bool GEN>
__global__ __launch_bounds__(BROW_THREADS) void k_batch_row_all(const BatchInst* __restrict__ inst,
                                                                const BatchUnit* __restrict__ units, int64_t nunits,
                                                                BatchFlags f) {
  __shared__ double2 lds[lds_all<BRow>() / 16 + 1];
  for (int64_t u = blockIdx.x; u < nunits; u += gridDim.x) {
    const BatchUnit un = units[u];
    const BatchInst& I = inst[un.inst];
    switch (I.nx + (I.small ? 1 : 0)) {
      case 128: batch_row_unit<128, false, GEN>(I, un, f, lds); break;
      case 129: batch_row_unit<128, true, GEN>(I, un, f, lds); break;
      case 256: batch_row_unit<256, false, GEN>(I, un, f, lds); break;
      case 257: batch_row_unit<256, true, GEN>(I, un, f, lds); break;
      case 512:
      case 513: batch_row_unit<512, false, GEN>(I, un, f, lds); break;
      case 1024:
      case 1025: batch_row_unit<1024, false, GEN>(I, un, f, lds); break;
      default: batch_row_unit<2048, false, GEN>(I, un, f, lds); break;
    }
    __syncthreads();  // the lengths lay the LDS out differently
  }
}

__global__ __launch_bounds__(BCOL_THREADS) void k_batch_col_all(const BatchInst* __restrict__ inst,
                                                                const BatchUnit* __restrict__ units, int64_t nunits,
                                                                BatchFlags f) {
  __shared__ double2 lds[lds_all<BColAll>() / 16 + 1];
  for (int64_t u = xcd_block(); u < nunits; u += gridDim.x) {
    const BatchUnit un = units[u];
    const BatchInst& I = inst[un.inst];
    switch (I.ny + (I.small ? 1 : 0)) {
      case 128: batch_col_unit<128, false>(I, un, f, lds); break;
      case 129: batch_col_unit<128, true>(I, un, f, lds); break;
      case 256: batch_col_unit<256, false>(I, un, f, lds); break;
      case 257: batch_col_unit<256, true>(I, un, f, lds); break;
      case 512: batch_col_unit<512, false>(I, un, f, lds); break;
      case 513: batch_col_unit<512, true>(I, un, f, lds); break;
      case 1024:
      case 1025: batch_col_unit<1024, false>(I, un, f, lds); break;
      default: batch_col_unit<2048, false>(I, un, f, lds); break;
    }
    __syncthreads();
  }
}

}  // namespace nlse

using namespace nlse;

struct nlse_batch {
  int64_t count = 0;
  std::vector<BatchInst> h_inst;
  std::vector<int64_t> offsets;
  BatchInst* d_inst = nullptr;
  // units grouped by line length: rows by NX, columns by NY
  BatchUnit* d_row = nullptr;
  BatchUnit* d_col = nullptr;
  int64_t n_row = 0, n_col = 0;
  bool general = false;  // some member's loss varies from point to point
  int64_t row_off[NLEN + 1] = {0}, col_off[NLEN + 1] = {0};
  int row_grid[NLEN] = {0}, col_grid[NLEN] = {0};
  // one launch per sweep for every line length (k_batch_*_all) instead of
  // one per length present
  bool single = false;
  int row_grid_all = 0, col_grid_all = 0;
  std::vector<void*> owned;  // device tables
  const void* base = nullptr;
  hipStream_t cap = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  int gprec = -1;
  int64_t gchunk = 0;
};

static int batch_alloc(nlse_batch* b, void** dst, const void* src, size_t bytes) {
  HIP_TRY(hipMalloc(dst, bytes));
  b->owned.push_back(*dst);
  HIP_TRY(hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice));
  return NLSE_OK;
}

static void batch_graph_free(nlse_batch* b) {
  if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  b->gexec = nullptr;
  b->graph = nullptr;
  b->gprec = -1;
}

static BatchFlags row_flags(int precision, int stage) {
  // stage 0: first sweep, 1: steady, 2: last
  BatchFlags f;
  std::memset(&f, 0, sizeof f);
  f.inverse_first = stage > 0;
  f.forward_last = stage < 2;
  f.has_a = stage > 0;
  f.slot_a = precision == 1 ? NLSE_SLOT_HALF_POST : NLSE_SLOT_FULL;
  f.has_b = (precision == 1 && stage < 2) ? 1 : 0;
  f.slot_b = NLSE_SLOT_HALF_PRE;
  return f;
}

// Blocks of a per-length launch: one per pass where the grid covers the units
// (the default), else the grid given per CU (nlse_batch_set_grid), whose blocks
// stride over the passes.
static unsigned pass_grid(int64_t units, int passes, int grid) {
  return (unsigned)(grid >= units ? units * passes : grid);
}

template <int N, bool SMALL>
static void launch_row_n(nlse_batch* b, int li, const BatchFlags& f, hipStream_t s) {
  const BatchUnit* units = b->d_row + b->row_off[li];
  const int64_t n = b->row_off[li + 1] - b->row_off[li];
  const dim3 grid(pass_grid(n, BRow<N, SMALL>::PASSES, b->row_grid[li])), block(BROW_THREADS);
  if (b->general)
    hipLaunchKernelGGL((k_batch_row<N, SMALL, true>), grid, block, 0, s, b->d_inst, units, n, f);
  else
    hipLaunchKernelGGL((k_batch_row<N, SMALL, false>), grid, block, 0, s, b->d_inst, units, n, f);
}

template <int N, bool SMALL>
static void launch_col_n(nlse_batch* b, int li, const BatchFlags& f, hipStream_t s) {
  constexpr int TH = bcol_threads(N);
  const int64_t n = b->col_off[li + 1] - b->col_off[li];
  hipLaunchKernelGGL((k_batch_col<N, SMALL>), dim3(pass_grid(n, BCol<N, SMALL, TH>::PASSES, b->col_grid[li])),
                     dim3(TH), 0, s, b->d_inst, b->d_col + b->col_off[li], n, f);
}

// One launch per line length present in the batch, or one for all lengths
// (b->single).
static int batch_row(nlse_batch* b, const BatchFlags& f, hipStream_t s) {
  if (b->single) {
    hipLaunchKernelGGL(b->general ? k_batch_row_all<true> : k_batch_row_all<false>, dim3((unsigned)b->row_grid_all),
                       dim3(BROW_THREADS), 0, s, b->d_inst, b->d_row, b->n_row, f);
    return launch_status("k_batch_row_all");
  }
  // longest lines first
  for (int li = NLEN - 1; li >= 0; --li) {
    if (b->row_off[li + 1] == b->row_off[li]) continue;
    switch (li) {
      case 0: launch_row_n<128, false>(b, li, f, s); break;
      case 1: launch_row_n<128, true>(b, li, f, s); break;
      case 2: launch_row_n<256, false>(b, li, f, s); break;
      case 3: launch_row_n<256, true>(b, li, f, s); break;
      case 4:
      case 5: launch_row_n<512, false>(b, li, f, s); break;
      case 6:
      case 7: launch_row_n<1024, false>(b, li, f, s); break;
      default: launch_row_n<2048, false>(b, li, f, s); break;
    }
    int rc = launch_status("k_batch_row");
    if (rc) return rc;
  }
  return NLSE_OK;
}

static int batch_col(nlse_batch* b, hipStream_t s, int timing = 0) {
  BatchFlags f;
  std::memset(&f, 0, sizeof f);
  f.timing = timing;
  if (b->single) {
    hipLaunchKernelGGL(k_batch_col_all, dim3((unsigned)b->col_grid_all), dim3(BCOL_THREADS), 0, s, b->d_inst, b->d_col,
                       b->n_col, f);
    return launch_status("k_batch_col_all");
  }
  for (int li = NLEN - 1; li >= 0; --li) {
    if (b->col_off[li + 1] == b->col_off[li]) continue;
    switch (li) {
      case 0: launch_col_n<128, false>(b, li, f, s); break;
      case 1: launch_col_n<128, true>(b, li, f, s); break;
      case 2: launch_col_n<256, false>(b, li, f, s); break;
      case 3: launch_col_n<256, true>(b, li, f, s); break;
      case 4: launch_col_n<512, false>(b, li, f, s); break;
      case 5: launch_col_n<512, true>(b, li, f, s); break;
      case 6:
      case 7: launch_col_n<1024, false>(b, li, f, s); break;
      default: launch_col_n<2048, false>(b, li, f, s); break;
    }
    int rc = launch_status("k_batch_col");
    if (rc) return rc;
  }
  return NLSE_OK;
}

static int batch_steady(nlse_batch* b, int precision, hipStream_t s) {
  int rc = batch_col(b, s);
  return rc ? rc : batch_row(b, row_flags(precision, 1), s);
}

static int batch_bind(nlse_batch* b, void* base, hipStream_t s) {
  if (base == b->base) return NLSE_OK;
  // launches already queued may still read the table
  HIP_TRY(hipStreamSynchronize(s));
  for (int64_t i = 0; i < b->count; ++i) {
    float2* A = (float2*)base + b->offsets[i];
    b->h_inst[i].row.A = A;
    b->h_inst[i].col.A = A;
  }
  HIP_TRY(hipMemcpy(b->d_inst, b->h_inst.data(), b->h_inst.size() * sizeof(BatchInst), hipMemcpyHostToDevice));
  b->base = base;
  return NLSE_OK;
}

static int64_t batch_cus() {
  int dev = 0, ncu = 256;
  if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
  return ncu;
}

// All units at once: a block per pass (pass_grid).  64 fields of 256^2 to 1024^2
// (7168 and 3584 units at 1024 points): 366 us a step by 8 and 1 blocks per CU that
// stride over the units, 282 by a block per pass.
static void batch_default_grid(nlse_batch* b) {
  const int64_t ncu = batch_cus();
  for (int li = 0; li < NLEN; ++li) {
    b->row_grid[li] = (int)(b->row_off[li + 1] - b->row_off[li]);
    b->col_grid[li] = (int)(b->col_off[li + 1] - b->col_off[li]);
  }
  b->row_grid_all = (int)std::min<int64_t>(b->n_row, ncu * 4);
  b->col_grid_all = (int)std::min<int64_t>(b->n_col, ncu * 1);
}

extern "C" {

int nlse_batch_create(const nlse_batch_item* items, int64_t count, int loss_saturates, nlse_batch** out) {
  if (!items || !out || count < 1) return fail(NLSE_ERR_ARG, "bad batch arguments");
  *out = nullptr;
  for (int64_t i = 0; i < count; ++i) {
    const nlse_batch_item& it = items[i];
    if (!batch_len_ok(it.ny) || !batch_len_ok(it.nx))
      return fail(NLSE_ERR_ARG, "batch field %lld: grid (%lld, %lld) unsupported (128..2048, powers of two)",
                  (long long)i, (long long)it.ny, (long long)it.nx);
    if (!it.px || !it.py || it.offset < 0) return fail(NLSE_ERR_ARG, "batch field %lld: bad tables", (long long)i);
    if (it.v_kind != V_NONE && (!it.V_dev || (it.v_kind != V_REAL && it.v_kind != V_CPLX)))
      return fail(NLSE_ERR_ARG, "batch field %lld: bad potential", (long long)i);
  }
  nlse_batch* b = new nlse_batch();
  b->count = count;
  int rc = NLSE_OK;
  int64_t total = 0;
  std::vector<BatchUnit> rows_n[NLEN], cols_n[NLEN];
  for (int64_t i = 0; i < count && !rc; ++i) {
    const nlse_batch_item& it = items[i];
    BatchInst I;
    std::memset(&I, 0, sizeof I);
    I.nx = (int)it.nx;
    I.ny = (int)it.ny;
    I.small = it.nx * it.ny <= SMALL_FIELD;
    total += it.nx * it.ny;
    I.inv_nx = (float)(1.0 / (double)it.nx);
    I.inv_ny = (float)(1.0 / (double)it.ny);
    const double2 *twx = nullptr, *twy = nullptr;
    const LineOps* ox = line_ops_public(it.nx);
    const LineOps* oy = line_ops_public(it.ny);
    if ((rc = ox->twiddles(&twx)) || (rc = oy->twiddles(&twy))) break;
    void *px = nullptr, *py = nullptr, *nl = nullptr;
    if ((rc = batch_alloc(b, &px, it.px, sizeof(double2) * it.nx))) break;
    if ((rc = batch_alloc(b, &py, it.py, sizeof(double2) * it.ny))) break;
    NLParams1 h[3];
    for (int sl = 0; sl < 3; ++sl) {
      h[sl].adz = (float)it.nl[sl].adz;
      h[sl].gdz = (float)it.nl[sl].gdz;
      h[sl].inv_isat = std::isinf(it.nl[sl].inv_isat) ? 0.f : (float)it.nl[sl].inv_isat;
      h[sl].vdz = (float)it.nl[sl].vdz;
      h[sl].adz_i = (float)it.nl[sl].adz_i;
      h[sl].gdz_i = (float)it.nl[sl].gdz_i;
      h[sl].vdz_i = (float)it.nl[sl].vdz_i;
      h[sl].cplx = it.nl[sl].adz_i != 0.0 || it.nl[sl].gdz_i != 0.0 || it.nl[sl].vdz_i != 0.0;
      b->general = b->general || h[sl].cplx;
    }
    b->general = b->general || loss_saturates || it.v_kind == V_CPLX;
    if ((rc = batch_alloc(b, &nl, h, sizeof h))) break;
    for (int sl = 0; sl < 3; ++sl) I.nl[sl] = (const NLParams1*)nl + sl;
    RowArgs& r = I.row;
    r.ngroups = it.ny;
    r.rows_per_item = it.ny;
    r.tw = twx;
    r.loss_sat = loss_saturates;
    r.V = it.V_dev;
    r.vkind = it.v_kind;
    r.out_scale = 1.f;
    ColArgs& c = I.col;
    c.nslabs = 1;
    c.NX = (int)it.nx;
    c.ncomp = 1;
    c.tw = twy;
    c.do_fwd = c.do_prop = c.do_inv = 1;
    c.pkind = PROP_SEP64;
    c.px = (const double2*)px;
    c.py = (const double2*)py;
    c.scale = (float)(1.0 / ((double)it.nx * (double)it.ny));
    c.out_scale = 1.f;
    b->h_inst.push_back(I);
    b->offsets.push_back(it.offset);
    const int64_t lpb = 4096 / it.nx, w = 8192 / it.ny;
    for (int64_t y = 0; y < it.ny; y += lpb) rows_n[len_index(it.nx, I.small)].push_back(BatchUnit{(int)i, 0, y});
    for (int64_t t = 0; t < it.nx / w; ++t) cols_n[len_index(it.ny, I.small)].push_back(BatchUnit{(int)i, 0, t});
  }
  // both sweeps, tiles of 4 columns among them, go through up to WRITE_THROUGH.
  // Both through / both back / rows through and columns back, a step: 60 fields of
  // 256^2 (31 MB) 45 / 47 / 52 us, 3 of 2048 x 512 43 / 44 / 46, 20 of 512^2 54 / 52
  // / 53, 2048^2 55 / 52 / 53
  for (BatchInst& I : b->h_inst) I.row.through = I.col.through = total * 8 <= WRITE_THROUGH ? 2 : 0;
  std::vector<BatchUnit> rows, cols;
  for (int li = 0; li < NLEN; ++li) {
    b->row_off[li] = (int64_t)rows.size();
    b->col_off[li] = (int64_t)cols.size();
    rows.insert(rows.end(), rows_n[li].begin(), rows_n[li].end());
    cols.insert(cols.end(), cols_n[li].begin(), cols_n[li].end());
  }
  b->row_off[NLEN] = (int64_t)rows.size();
  b->col_off[NLEN] = (int64_t)cols.size();
  if (!rc) rc = batch_alloc(b, (void**)&b->d_inst, b->h_inst.data(), b->h_inst.size() * sizeof(BatchInst));
  if (!rc) rc = batch_alloc(b, (void**)&b->d_row, rows.data(), rows.size() * sizeof(BatchUnit));
  if (!rc) rc = batch_alloc(b, (void**)&b->d_col, cols.data(), cols.size() * sizeof(BatchUnit));
  if (rc) {
    nlse_batch_destroy(b);
    return rc;
  }
  b->n_row = (int64_t)rows.size();
  b->n_col = (int64_t)cols.size();
  batch_default_grid(b);
  *out = b;
  return NLSE_OK;
}

int nlse_batch_destroy(nlse_batch* b) {
  if (!b) return NLSE_OK;
  batch_graph_free(b);
  if (b->cap) (void)hipStreamDestroy(b->cap);
  for (void* q : b->owned) (void)hipFree(q);
  delete b;
  return NLSE_OK;
}

int nlse_batch_set_grid(nlse_batch* b, int row_blocks_per_cu, int col_blocks_per_cu) {
  if (!b || row_blocks_per_cu < 1 || col_blocks_per_cu < 1 || row_blocks_per_cu > 64 || col_blocks_per_cu > 64)
    return fail(NLSE_ERR_ARG, "bad batch grid (%d, %d blocks per CU)", row_blocks_per_cu, col_blocks_per_cu);
  const int64_t ncu = batch_cus();
  for (int li = 0; li < NLEN; ++li) {
    b->row_grid[li] = (int)std::min<int64_t>(b->row_off[li + 1] - b->row_off[li], ncu * row_blocks_per_cu);
    b->col_grid[li] = (int)std::min<int64_t>(b->col_off[li + 1] - b->col_off[li], ncu * col_blocks_per_cu);
  }
  b->row_grid_all = (int)std::min<int64_t>(b->n_row, ncu * row_blocks_per_cu);
  b->col_grid_all = (int)std::min<int64_t>(b->n_col, ncu * col_blocks_per_cu);
  batch_graph_free(b);  // the captured launches bake in the grid
  return NLSE_OK;
}

int nlse_batch_default_grid(nlse_batch* b) {
  if (!b) return fail(NLSE_ERR_ARG, "null batch");
  batch_default_grid(b);
  batch_graph_free(b);
  return NLSE_OK;
}

int nlse_batch_set_single_launch(nlse_batch* b, int on) {
  if (!b) return fail(NLSE_ERR_ARG, "null batch");
  if (b->single != (on != 0)) batch_graph_free(b);  // the captured launches differ
  b->single = on != 0;
  return NLSE_OK;
}

int nlse_batch_config(const nlse_batch* b, int64_t* row_units, int64_t* col_units, int* row_grid, int* col_grid) {
  if (!b) return fail(NLSE_ERR_ARG, "null batch");
  if (row_units) *row_units = b->n_row;
  if (col_units) *col_units = b->n_col;
  int rg = 0, cg = 0;
  for (int li = 0; li < NLEN; ++li) {
    rg += b->row_grid[li];
    cg += b->col_grid[li];
  }
  if (b->single) {
    rg = b->row_grid_all;
    cg = b->col_grid_all;
  }
  if (row_grid) *row_grid = rg;  // units taken at a time over the launches of one sweep
  if (col_grid) *col_grid = cg;
  return NLSE_OK;
}

// Capture `chunk` steady steps unless the graph for (precision, chunk) is
// already there; the kernels read the instance table, so a new field buffer
// only rewrites the table.
static int batch_capture(nlse_batch* b, int precision, int64_t chunk) {
  if (b->gexec && b->gprec == precision && b->gchunk == chunk) return NLSE_OK;
  batch_graph_free(b);
  if (!b->cap) HIP_TRY(hipStreamCreateWithFlags(&b->cap, hipStreamNonBlocking));
  HIP_TRY(hipStreamBeginCapture(b->cap, hipStreamCaptureModeThreadLocal));
  int rc = NLSE_OK;
  for (int64_t k = 0; k < chunk && !rc; ++k) rc = batch_steady(b, precision, b->cap);
  hipGraph_t g = nullptr;
  const hipError_t e = hipStreamEndCapture(b->cap, &g);
  if (rc) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  if (e != hipSuccess) return fail(NLSE_ERR_HIP, "hipStreamEndCapture failed: %s", hipGetErrorString(e));
  b->graph = g;
  HIP_TRY(hipGraphInstantiate(&b->gexec, g, nullptr, nullptr, 0));
  b->gprec = precision;
  b->gchunk = chunk;
  return NLSE_OK;
}

int nlse_batch_graph_prepare(nlse_batch* b, void* base, int precision, int64_t chunk, void* stream) {
  if (!b || !base || (precision != 0 && precision != 1) || chunk < 1)
    return fail(NLSE_ERR_ARG, "bad batch graph arguments");
  hipStream_t s = (hipStream_t)stream;
  int rc = batch_bind(b, base, s);
  if (!rc) rc = batch_capture(b, precision, chunk);
  if (!rc) HIP_TRY(hipGraphUpload(b->gexec, s));
  return rc;
}

int nlse_batch_run(nlse_batch* b, void* base, int64_t nsteps, int precision, int64_t chunk, void* stream) {
  if (!b || !base || nsteps < 0 || (precision != 0 && precision != 1) || chunk < 0)
    return fail(NLSE_ERR_ARG, "bad batch run arguments");
  if (nsteps == 0) return NLSE_OK;
  hipStream_t s = (hipStream_t)stream;
  int rc = batch_bind(b, base, s);
  if (rc) return rc;
  const int64_t reps = chunk > 0 ? (nsteps - 1) / chunk : 0;
  if (reps > 0 && (rc = batch_capture(b, precision, chunk))) return rc;
  if ((rc = batch_row(b, row_flags(precision, 0), s))) return rc;
  for (int64_t r = 0; r < reps; ++r) HIP_TRY(hipGraphLaunch(b->gexec, s));
  for (int64_t k = reps * chunk; k < nsteps; ++k) {
    if ((rc = batch_col(b, s))) return rc;
    if ((rc = batch_row(b, row_flags(precision, k == nsteps - 1 ? 2 : 1), s))) return rc;
  }
  return NLSE_OK;
}

int nlse_batch_run_pass(nlse_batch* b, void* base, int pass, int64_t count, void* stream) {
  if (!b || !base || count < 0 || (pass != 0 && pass != 1)) return fail(NLSE_ERR_ARG, "bad batch pass arguments");
  hipStream_t s = (hipStream_t)stream;
  int rc = batch_bind(b, base, s);
  BatchFlags f = row_flags(0, 1);
  f.timing = 1;
  for (int64_t k = 0; k < count && !rc; ++k) rc = pass == 0 ? batch_row(b, f, s) : batch_col(b, s, 1);
  return rc;
}

}  // extern "C"
