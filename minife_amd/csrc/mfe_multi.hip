// Many right-hand sides on one matrix: Y = A X for X with K columns (row-major
// n x K, K = 4, 8 or 16), and K simultaneous FP64 CG solves that share one
// SpMM per iteration (each column keeps its own alpha, beta and stopping test,
// cg_solve.hpp:69-229 per column, with tree-reduced dots).
//
// SpMM tile: L = K / CPL lanes per row, each lane owns CPL consecutive columns
// of the row (one 8*CPL-byte load per non-zero), so a row's K columns are one
// 8K-byte stretch of X per non-zero.  The L lanes of a row read the same
// value/column entry (a broadcast).  The row is walked in chunks of U entries
// whose loads are all issued before the first product; each column's sum runs
// in stored column order, so column k of Y equals A * X[:, k] from the
// single-vector SpMV bit for bit.  SELL tiles read the values and columns
// from the matrix's SELL-64 copy (slot-major: the loads of a wave's rows are
// contiguous) instead of the CSR arrays.  Staged tiles first copy the distinct
// X rows of 16 or 32 consecutive rows into LDS and gather from there (same
// arithmetic).
// The autotuner times every tile on the caller's matrix and keeps the fastest
// for that matrix and K.
#include <algorithm>
#include <cmath>
#include <vector>

#include "mfe_box.hpp"
#include "mfe_common.hpp"
#include "mfe_sell.hpp"

namespace mfe {

constexpr int kSellTile = -1;      // SpmmTile::rows of a tile reading the SELL-64 copy
constexpr int kSellLineTile = -2;  // the same, sharing X rows along grid lines
constexpr int kBoxTile = -3;       // the box layout, X planes of a block in LDS
constexpr int kLineStride = 16;    // ints per slice line record (count + 9 columns, 64 B)

struct SpmmTile {
  int cpl, unroll;
  int rows;  // 0: CSR, direct gathers; 16 or 32: rows per workgroup of a staged tile;
             // kSellTile: SELL-64 copy, direct gathers; kSellLineTile: SELL-64 copy,
             // line slices taking two of each three X rows from neighbouring lanes;
             // kBoxTile: box layout
  int box = 0;  // kBoxTile: the variant (kBoxVariants)
};

// Candidate tiles per K (index = tile id).
static const SpmmTile kTiles16[] = {{1, 9, 0},  {2, 9, 0},  {4, 9, 0},  {8, 9, 0},  {2, 3, 0},
                                    {4, 3, 0},  {8, 3, 0},  {16, 3, 0}, {1, 9, 16}, {2, 9, 16},
                                    {1, 9, 32}, {2, 9, 32}, {4, 9, 32}, {2, 9, kSellTile},
                                    {4, 9, kSellTile}, {8, 9, kSellTile}, {4, 9, kSellLineTile},
                                    {8, 9, kSellLineTile}, {4, 27, kBoxTile, 0},
                                    {4, 27, kBoxTile, 1}};
static const SpmmTile kTiles8[] = {{1, 9, 0},  {2, 9, 0},  {4, 9, 0},         {8, 9, 0},
                                   {2, 3, 0},  {4, 3, 0},  {8, 3, 0},         {1, 9, 16},
                                   {1, 9, 32}, {2, 9, 32}, {1, 9, kSellTile}, {2, 9, kSellTile},
                                   {4, 9, kSellTile}, {2, 9, kSellLineTile}, {4, 9, kSellLineTile},
                                   {2, 27, kBoxTile, 0}, {2, 27, kBoxTile, 1}};
static const SpmmTile kTiles4[] = {{1, 9, 0},  {2, 9, 0},  {4, 9, 0},         {2, 3, 0},
                                   {4, 3, 0},  {1, 9, 16}, {1, 9, 32},        {1, 9, kSellTile},
                                   {2, 9, kSellTile}, {1, 9, kSellLineTile}, {2, 9, kSellLineTile},
                                   {1, 27, kBoxTile, 0}, {1, 27, kBoxTile, 1}};
constexpr int kMaxTiles = 20;

static int tile_count(int K) {
  return K == 16 ? (int)(sizeof(kTiles16) / sizeof(SpmmTile))
                 : K == 8 ? (int)(sizeof(kTiles8) / sizeof(SpmmTile))
                          : (int)(sizeof(kTiles4) / sizeof(SpmmTile));
}
static SpmmTile tile_of(int K, int id) {
  return K == 16 ? kTiles16[id] : K == 8 ? kTiles8[id] : kTiles4[id];
}

// ------------------------------------------------------ staging plan --------
//
// A staged tile owns R consecutive rows (R = 16 or 32, one plan each).  The
// plan lists each tile's distinct columns (sorted, `ucols` from `uoff[tile]`)
// and rewrites every non-zero's column as its 16-bit position in that list
// (`lcols`).  The SpMM then copies those X rows into LDS once per tile and
// reads them from there: R rows along x of a 27-point stencil need 9 (R + 2)
// distinct X rows, about 10 per row instead of 27 gathers.

constexpr int kStageCap = 1024;  // non-zeros per tile the plan kernel sorts in LDS
constexpr int kStageLdsBytes = 60 * 1024;  // staged X rows; + the dot array stays <= 64 KiB

static int plan_slot(int rows) { return rows == 16 ? 0 : 1; }

struct SpmmPlan {
  const mfe_csr* A = nullptr;
  uint64_t gen = 0;
  bool built = false, ok = false;
  int rows = 0, ntiles = 0, maxu = 0;
  int* uoff = nullptr;
  int* ucols = nullptr;
  unsigned short* lcols = nullptr;
  void release() {
    (void)hipFree(uoff);
    (void)hipFree(ucols);
    (void)hipFree(lcols);
    uoff = ucols = nullptr;
    lcols = nullptr;
    built = ok = false;
    rows = ntiles = maxu = 0;
  }
};

// One workgroup per tile: sort the tile's columns in LDS (bitonic), mark the
// first of each value; pass 0 counts them, pass 1 writes them and the local
// indices.  Tiles with more than kStageCap non-zeros report -1.
__global__ __launch_bounds__(kBlock) void stage_plan_kernel(int n, int rows,
                                                            const int* __restrict__ ro,
                                                            const int* __restrict__ cols, int pass,
                                                            const int* __restrict__ uoff,
                                                            int* __restrict__ counts,
                                                            int* __restrict__ ucols,
                                                            unsigned short* __restrict__ lcols) {
  __shared__ int a[kStageCap];
  __shared__ int u[kStageCap];
  __shared__ int scan[kBlock];
  const int t = (int)threadIdx.x;
  const int tile = (int)blockIdx.x;
  const int r0 = tile * rows, r1 = min(r0 + rows, n);
  const int s0 = ro[r0], cnt = ro[r1] - s0;
  if (cnt > kStageCap) {
    if (pass == 0 && t == 0) counts[tile] = -1;
    return;
  }
  for (int i = t; i < kStageCap; i += kBlock) a[i] = i < cnt ? cols[s0 + i] : INT_MAX;
  __syncthreads();
  for (int k = 2; k <= kStageCap; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = t; i < kStageCap; i += kBlock) {
        const int ixj = i ^ j;
        if (ixj > i) {
          const int ai = a[i], aj = a[ixj];
          if ((i & k) == 0 ? ai > aj : ai < aj) {
            a[i] = aj;
            a[ixj] = ai;
          }
        }
      }
      __syncthreads();
    }
  constexpr int kPer = kStageCap / kBlock;  // 4 consecutive entries per thread
  int f[kPer], lsum = 0;
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int i = kPer * t + q;
    f[q] = a[i] != INT_MAX && (i == 0 || a[i] != a[i - 1]);
    lsum += f[q];
  }
  scan[t] = lsum;
  __syncthreads();
  for (int off = 1; off < kBlock; off <<= 1) {  // inclusive scan
    const int v = t >= off ? scan[t - off] : 0;
    __syncthreads();
    scan[t] += v;
    __syncthreads();
  }
  const int total = scan[kBlock - 1];
  if (pass == 0) {
    if (t == 0) counts[tile] = total;
    return;
  }
  int r = scan[t] - lsum;
  const int base = uoff[tile];
#pragma unroll
  for (int q = 0; q < kPer; ++q)
    if (f[q]) {
      u[r] = a[kPer * t + q];
      ucols[base + r] = a[kPer * t + q];
      ++r;
    }
  __syncthreads();
  for (int i = t; i < cnt; i += kBlock) {
    const int c = cols[s0 + i];
    int lo = 0, hi = total;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (u[mid] < c) lo = mid + 1;
      else hi = mid;
    }
    lcols[s0 + i] = (unsigned short)lo;
  }
}

// Sum over the lanes of one wave that hold the same column (lane % L), in a
// fixed butterfly order; valid in every lane.
template <int L>
__device__ __forceinline__ double sum_same_column(double v) {
#pragma unroll
  for (int off = kWave / 2; off >= L; off >>= 1) v += __shfl_xor(v, off, kWave);
  return v;
}

// out[0..CPL) = src[0..CPL), in 16-byte loads when CPL is even.
template <int CPL>
__device__ __forceinline__ void load_x_piece(const double* __restrict__ src, double (&out)[CPL]) {
  if constexpr (CPL % 2 == 0) {
#pragma unroll
    for (int q = 0; q < CPL; q += 2) {
      const double2 d = *reinterpret_cast<const double2*>(src + q);
      out[q] = d.x;
      out[q + 1] = d.y;
    }
  } else {
#pragma unroll
    for (int q = 0; q < CPL; ++q) out[q] = src[q];
  }
}

// Y = A X; with partials non-null also the workgroup partials of Y[:,k].P[:,k]
// (partials[block * K + k]), P = X here (the CG's p.Ap).
template <int K, int CPL, int U>
__global__ __launch_bounds__(kBlock) void spmm_kernel(int n, const int* __restrict__ ro,
                                                      const int* __restrict__ cols,
                                                      const double* __restrict__ vals,
                                                      const double* __restrict__ X,
                                                      double* __restrict__ Y,
                                                      double* __restrict__ partials,
                                                      const int* __restrict__ done) {
  if (done && *done) return;
  constexpr int L = K / CPL;
  constexpr int RPB = kBlock / L;  // rows per workgroup
  const int t = (int)threadIdx.x;
  const int row = (int)blockIdx.x * RPB + t / L;
  const int k0 = (t % L) * CPL;
  double acc[CPL];
#pragma unroll
  for (int q = 0; q < CPL; ++q) acc[q] = 0.0;
  if (row < n) {
    const int a = ro[row], len = ro[row + 1] - a;
    for (int j0 = 0; j0 < len; j0 += U) {
      int c[U];
      double v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = a + min(j0 + u, len - 1);
        c[u] = cols[j];
        v[u] = vals[j];
      }
      double xv[U][CPL];
#pragma unroll
      for (int u = 0; u < U; ++u) load_x_piece<CPL>(X + (int64_t)c[u] * K + k0, xv[u]);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (j0 + u < len) {
#pragma unroll
          for (int q = 0; q < CPL; ++q) acc[q] += v[u] * xv[u][q];
        }
    }
    double* dst = Y + (int64_t)row * K + k0;
#pragma unroll
    for (int q = 0; q < CPL; ++q) dst[q] = acc[q];
  }
  if (partials) {
    __shared__ double red[kBlock / kWave][K];
    double term[CPL];
#pragma unroll
    for (int q = 0; q < CPL; ++q)
      term[q] = row < n ? acc[q] * X[(int64_t)row * K + k0 + q] : 0.0;
    const int lane = t % kWave, wave = t / kWave;
#pragma unroll
    for (int q = 0; q < CPL; ++q) {
      const double s = sum_same_column<L>(term[q]);
      if (lane < L) red[wave][lane * CPL + q] = s;
    }
    __syncthreads();
    if (t < K) {
      double s = red[0][t];
#pragma unroll
      for (int w = 1; w < kBlock / kWave; ++w) s += red[w][t];
      partials[(int64_t)blockIdx.x * K + t] = s;
    }
  }
}

// Staged SpMM: one workgroup per R-row tile, L = K / CPL lanes per row.  The tile's distinct X rows are copied into LDS (sx[u * K + k], in the
// plan's column order), then each lane walks its row in chunks of U entries
// as spmm_kernel does, with the local column index in place of the global
// one: the same products added in the same order, so the same bits.
template <int K, int CPL, int U, int R>
__global__ __launch_bounds__(R * K / CPL) void spmm_staged_kernel(
    int n, const int* __restrict__ ro, const unsigned short* __restrict__ lcols,
    const double* __restrict__ vals, const int* __restrict__ uoff, const int* __restrict__ ucols,
    const double* __restrict__ X, double* __restrict__ Y, double* __restrict__ partials,
    const int* __restrict__ done) {
  if (done && *done) return;
  constexpr int L = K / CPL;
  constexpr int NT = R * L;
  constexpr int H = K / 2;  // 16-byte pieces per X row
  extern __shared__ __align__(16) double sx[];
  const int t = (int)threadIdx.x;
  const int tile = (int)blockIdx.x;
  const int u0 = uoff[tile], nu = uoff[tile + 1] - u0;
  for (int i = t; i < nu * H; i += NT) {
    const int u = i / H, h = i - u * H;
    const double2 d = *reinterpret_cast<const double2*>(X + (int64_t)ucols[u0 + u] * K + 2 * h);
    *reinterpret_cast<double2*>(sx + u * K + 2 * h) = d;
  }
  __syncthreads();
  const int row = tile * R + t / L;
  const int k0 = (t % L) * CPL;
  double acc[CPL];
#pragma unroll
  for (int q = 0; q < CPL; ++q) acc[q] = 0.0;
  if (row < n) {
    const int a = ro[row], len = ro[row + 1] - a;
    for (int j0 = 0; j0 < len; j0 += U) {
      int c[U];
      double v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = a + min(j0 + u, len - 1);
        c[u] = lcols[j];
        v[u] = vals[j];
      }
      double xv[U][CPL];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const double* src = sx + c[u] * K + k0;
        if constexpr (CPL % 2 == 0) {
#pragma unroll
          for (int q = 0; q < CPL; q += 2) {
            const double2 d = *reinterpret_cast<const double2*>(src + q);
            xv[u][q] = d.x;
            xv[u][q + 1] = d.y;
          }
        } else {
#pragma unroll
          for (int q = 0; q < CPL; ++q) xv[u][q] = src[q];
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (j0 + u < len) {
#pragma unroll
          for (int q = 0; q < CPL; ++q) acc[q] += v[u] * xv[u][q];
        }
    }
    double* dst = Y + (int64_t)row * K + k0;
#pragma unroll
    for (int q = 0; q < CPL; ++q) dst[q] = acc[q];
  }
  if (partials) {
    constexpr int NW = NT / kWave;
    __shared__ double red[NW][K];
    double term[CPL];
#pragma unroll
    for (int q = 0; q < CPL; ++q)
      term[q] = row < n ? acc[q] * X[(int64_t)row * K + k0 + q] : 0.0;
    const int lane = t % kWave, wave = t / kWave;
#pragma unroll
    for (int q = 0; q < CPL; ++q) {
      const double s = sum_same_column<L>(term[q]);
      if (lane < L) red[wave][lane * CPL + q] = s;
    }
    __syncthreads();
    if (t < K) {
      double s = red[0][t];
#pragma unroll
      for (int w = 1; w < NW; ++w) s += red[w][t];
      partials[(int64_t)tile * K + t] = s;
    }
  }
}

// Builds the R-row staging plan of A (synchronises ctx's stream).  A matrix
// with a tile of more than kStageCap non-zeros gets ok = false (its staged
// tiles of that R are then not offered); so does n = 0.
static int build_stage_plan(mfe_ctx* ctx, const mfe_csr* A, int R, SpmmPlan& p) {
  p.release();
  p.A = A;
  p.gen = A->plan_gen;
  p.built = true;
  p.rows = R;
  const int64_t n = A->nrows;
  if (n == 0 || n > INT_MAX - R) return MFE_OK;
  const int nt = (int)cdiv(n, R);
  hipStream_t s = ctx->stream;
  MFE_CHECK(ctx, dev_malloc(ctx, &p.uoff, sizeof(int) * ((size_t)nt + 1)));
  stage_plan_kernel<<<nt, kBlock, 0, s>>>((int)n, R, A->row_offsets, A->cols, 0, nullptr, p.uoff,
                                          nullptr, nullptr);
  MFE_LAUNCHED(ctx, "stage_plan_kernel count");
  std::vector<int> h(nt + 1);
  MFE_CHECK(ctx, hipMemcpyAsync(h.data(), p.uoff, sizeof(int) * nt, hipMemcpyDeviceToHost, s));
  MFE_CHECK(ctx, hipStreamSynchronize(s));
  int64_t total = 0;
  int maxu = 0;
  for (int i = 0; i < nt; ++i) {
    if (h[i] < 0) {  // a tile too long for the plan kernel
      p.release();
      p.A = A;
      p.gen = A->plan_gen;
      p.built = true;
      p.rows = R;
      return MFE_OK;
    }
    const int c = h[i];
    h[i] = (int)total;
    total += c;
    maxu = std::max(maxu, c);
  }
  h[nt] = (int)total;
  if (total > INT_MAX) return MFE_OK;
  MFE_CHECK(ctx, hipMemcpyAsync(p.uoff, h.data(), sizeof(int) * ((size_t)nt + 1),
                                hipMemcpyHostToDevice, s));
  MFE_CHECK(ctx, dev_malloc(ctx, &p.ucols, sizeof(int) * (size_t)std::max<int64_t>(total, 1)));
  MFE_CHECK(ctx, dev_malloc(ctx, &p.lcols, sizeof(unsigned short) * (size_t)std::max<int64_t>(A->nnz, 1)));
  stage_plan_kernel<<<nt, kBlock, 0, s>>>((int)n, R, A->row_offsets, A->cols, 1, p.uoff, nullptr,
                                          p.ucols, p.lcols);
  MFE_LAUNCHED(ctx, "stage_plan_kernel fill");
  MFE_CHECK(ctx, hipStreamSynchronize(s));
  p.ntiles = nt;
  p.maxu = maxu;
  p.ok = true;
  return MFE_OK;
}

// Operands of one SpMM launch; plans[plan_slot(R)] is the R-row staging plan
// (null: staged tiles of that R unavailable); svals null: no SELL tiles.
struct SpmmArgs {
  int n;
  const int* ro;
  const int* cols;
  const double* vals;
  const SpmmPlan* plans[2];
  int nslices;
  const int* soff;
  const unsigned char* slen;
  const int* scols;
  const double* svals;
  const int* lines;  // per-slice line records (null: line tiles unavailable)
  const double* bvals;  // box layout of the values (null: box tiles unavailable)
  BoxGeom bg;
  int cus;              // compute units (the box tile sizes its z chunks)
};

static bool stage_ok(const SpmmPlan* p, int K) {
  return p && p->ok && (int64_t)p->maxu * K * (int64_t)sizeof(double) <= kStageLdsBytes;
}

// spmm_kernel on the SELL-64 copy: thread (row, column group) reads slot j of
// its row at sell_pos (the L lanes of a row read the same entry, the rows of a
// wave consecutive entries); RPB rows per workgroup cover whole or parts of
// slices; rows past the last slice return at once, rows past n add nothing.
// With LINES, a slice that sell_lines_kernel recorded as a line slice takes
// the line path below instead; its products and their order are the same.
template <int K, int CPL, int U, bool LINES>
__global__ __launch_bounds__(kBlock) void spmm_sell_kernel(
    int n, int nslices, const int* __restrict__ soff, const unsigned char* __restrict__ slen,
    const int* __restrict__ scols, const double* __restrict__ svals,
    const int* __restrict__ lines, const double* __restrict__ X,
    double* __restrict__ Y, double* __restrict__ partials, const int* __restrict__ done) {
  if (done && *done) return;
  constexpr int L = K / CPL;
  constexpr int RPB = kBlock / L;
  const int t = (int)threadIdx.x;
  const int row = (int)blockIdx.x * RPB + t / L;
  const int k0 = (t % L) * CPL;
  const int slice = row / kWave, lane = row % kWave;
  const bool live = slice < nslices;
  double acc[CPL];
#pragma unroll
  for (int q = 0; q < CPL; ++q) acc[q] = 0.0;
  // a wave's rows lie in one slice: its line record is wave-uniform
  const int* rec = LINES && live
                       ? lines + (int64_t)__builtin_amdgcn_readfirstlane(slice) * kLineStride
                       : nullptr;
  const int ntr = rec ? rec[0] : 0;
  if (ntr > 0) {
    // Line slice: its 64 rows all have width w = 3 ntr, and slots 3g, 3g+1,
    // 3g+2 of row r hold columns c_g + r - 1, c_g + r, c_g + r + 1
    // (consecutive nodes of grid lines; c_g = rec[1 + g]).  Slot 3g's X row
    // of row r is slot 3g+1's X row of row r-1, and slot 3g+2's that of row
    // r+1: each lane loads its row's middle X row and takes the other two
    // from the lanes L below and above it; the lanes of the wave's first and
    // last rows load their missing one.  No column loads: the X loads go out
    // with the value loads.
    static_assert(U % 3 == 0, "line path unrolls whole slot triples");
    constexpr int G = U / 3;
    const int w = 3 * ntr;
    const int64_t o64 = (int64_t)soff[slice] * kWave;
    const int hl = t % kWave;
    const bool head = hl < L, tail = hl >= kWave - L;
    for (int g0 = 0; g0 < ntr; g0 += G) {
      double v[U];
      double xm[G][CPL], xe[G][CPL];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int gg = min(g0 + g, ntr - 1);
#pragma unroll
        for (int m = 0; m < 3; ++m) v[3 * g + m] = svals[sell_pos(o64, 3 * gg + m, w, lane)];
        const int c = rec[1 + gg] + lane;
        load_x_piece<CPL>(X + (int64_t)c * K + k0, xm[g]);
        if (head || tail) load_x_piece<CPL>(X + (int64_t)(head ? c - 1 : c + 1) * K + k0, xe[g]);
      }
#pragma unroll
      for (int g = 0; g < G; ++g)
        if (g0 + g < ntr) {
#pragma unroll
          for (int q = 0; q < CPL; ++q) {
            const double lo = __shfl_up(xm[g][q], L, kWave);
            const double hi = __shfl_down(xm[g][q], L, kWave);
            acc[q] += v[3 * g] * (head ? xe[g][q] : lo);
            acc[q] += v[3 * g + 1] * xm[g][q];
            acc[q] += v[3 * g + 2] * (tail ? xe[g][q] : hi);
          }
        }
    }
    double* dst = Y + (int64_t)row * K + k0;  // every row of a line slice is < n
#pragma unroll
    for (int q = 0; q < CPL; ++q) dst[q] = acc[q];
  } else if (live) {
    const int o = soff[slice], w = soff[slice + 1] - o;
    const int len = slen[row];
    const int64_t o64 = (int64_t)o * kWave;
    for (int j0 = 0; j0 < len; j0 += U) {
      int c[U];
      double v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t at = sell_pos(o64, min(j0 + u, w - 1), w, lane);
        c[u] = scols[at];
        v[u] = svals[at];
      }
      double xv[U][CPL];
#pragma unroll
      for (int u = 0; u < U; ++u) load_x_piece<CPL>(X + (int64_t)c[u] * K + k0, xv[u]);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (j0 + u < len) {
#pragma unroll
          for (int q = 0; q < CPL; ++q) acc[q] += v[u] * xv[u][q];
        }
    }
    if (row < n) {
      double* dst = Y + (int64_t)row * K + k0;
#pragma unroll
      for (int q = 0; q < CPL; ++q) dst[q] = acc[q];
    }
  }
  if (partials) {
    __shared__ double red[kBlock / kWave][K];
    double term[CPL];
#pragma unroll
    for (int q = 0; q < CPL; ++q)
      term[q] = row < n ? acc[q] * X[(int64_t)row * K + k0 + q] : 0.0;
    const int lw = t % kWave, wave = t / kWave;
#pragma unroll
    for (int q = 0; q < CPL; ++q) {
      const double s = sum_same_column<L>(term[q]);
      if (lw < L) red[wave][lw * CPL + q] = s;
    }
    __syncthreads();
    if (t < K) {
      double s = red[0][t];
#pragma unroll
      for (int w = 1; w < kBlock / kWave; ++w) s += red[w][t];
      partials[(int64_t)blockIdx.x * K + t] = s;
    }
  }
}

// Y = A X on the box layout of A's values (mfe_box.hpp).  A workgroup owns a
// block of MX x MY = 64 nodes, four lanes per node (CPL = K/4 columns each),
// and a range of z node planes; it streams the X planes of the block and a
// one-node ring ((MX+2) (MY+2) cells of K values) through LDS one at a time,
// so each X row leaves HBM about once per workgroup.  Step p holds X plane p
// (two buffers: plane p+1 is loaded during or after step p and stored into
// the other buffer, one barrier per step) and adds its terms to three rows
// per node in flight: the row of plane p+1 (its slots 0-8, which read plane
// p), of plane p (slots 9-17) and of plane p-1 (slots 18-26, after which that
// row is complete and stored).  Each row still adds its in-range products in
// ascending slot order from 0.0: per column, the bits of the single-vector
// SpMV.  A step goes line by line: three slots of each of the three rows, whose
// nine values are loaded one line ahead (every lane of a node loads them; one fetch
// per wave and address).  Partials: the dot of
// each completed row with X of its own node (held from the step that had that
// plane in LDS), per thread over its planes in order, then over the rows of
// the workgroup.  XCD: workgroup i runs on XCD i % 8, and each XCD takes a
// contiguous range of tiles numbered x-fastest within a z chunk; PF: X plane
// p+1 is loaded into registers before step p's arithmetic (else after it).
// The body for workgroup wg of nwg is a device function so that a persistent
// kernel can run it tile by tile.
constexpr int kBoxNodes = 64;  // nodes per box SpMM workgroup
template <int K, int MX, bool XCD, bool PF>
__device__ __forceinline__ void spmm_boxp_body(int wg, int nwg, BoxGeom g, int nbxm, int nzc,
                                               int zc, const double* __restrict__ V,
                                               const double* __restrict__ X,
                                               double* __restrict__ Y,
                                               double* __restrict__ partials) {
  constexpr int L = 4, CPL = K / L;
  constexpr int MY = kBoxNodes / MX, WX = MX + 2, MW = WX * (MY + 2);
  constexpr int NLD = (MW * K + kBlock - 1) / kBlock;  // X loads per thread per plane
  static_assert(MX * MY == kBoxNodes && kBoxNodes * L == kBlock, "four lanes per node");
  __shared__ double win[2][MW * K];
  int chunk, bx, by;
  if (XCD) {
    // workgroup i runs on XCD i % 8: give each XCD a contiguous range of
    // tiles numbered x-fastest within a z chunk, so the tiles that share value
    // lines and X halos meet in one L2
    const int per = nwg / 8, rem = nwg % 8, x = wg % 8;
    const int tile = x * per + min(x, rem) + wg / 8;
    const int nb = nwg / nzc;  // blocks per z chunk
    chunk = tile / nb;
    bx = (tile % nb) % nbxm;
    by = (tile % nb) / nbxm;
  } else {
    chunk = wg % nzc;
    const int blk = wg / nzc;
    bx = blk % nbxm;
    by = blk / nbxm;
  }
  const int t = (int)threadIdx.x;
  const int r = t / L, j = t % L;
  const int tx = r % MX, ty = r / MX;
  const int ix = bx * MX + tx, iy = by * MY + ty;
  const bool live = ix < g.gx && iy < g.gy;
  auto col = [&](int q) { return j * CPL + q; };  // this lane's q-th column
  const int vblk = (iy / kBoxBY) * g.nbx + ix / kBoxBX;
  const int vt = (ix % kBoxBX) + kBoxBX * (iy % kBoxBY);
  const int z0 = chunk * zc;
  const int z1 = min(z0 + zc, g.gz);
  const int64_t plane = (int64_t)g.gx * g.gy;
  double xr[NLD];
  auto fetch = [&](int p) {
    const bool zin = p >= 0 && p < g.gz;
#pragma unroll
    for (int k = 0; k < NLD; ++k) {
      const int e = t + k * kBlock;
      const int cell = e / K, c = e % K;
      const int wx = cell % WX, wy = cell / WX;
      const int nx = bx * MX + wx - 1, ny = by * MY + wy - 1;
      const bool ok = e < MW * K && zin && nx >= 0 && nx < g.gx && ny >= 0 && ny < g.gy;
      xr[k] = ok ? X[((int64_t)p * plane + nx + (int64_t)g.gx * ny) * K + c] : 0.0;
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int k = 0; k < NLD; ++k) {
      const int e = t + k * kBlock;
      if (e < MW * K) win[buf][e] = xr[k];
    }
  };
  const int c0 = (ty + 1) * WX + (tx + 1);
  double tsum[CPL], accA[CPL], accB[CPL], accC[CPL], xown[CPL];
#pragma unroll
  for (int q = 0; q < CPL; ++q) tsum[q] = accA[q] = accB[q] = accC[q] = xown[q] = 0.0;
  // The nine values of line sy of X plane p: three slots of each of the three
  // rows in flight (plane p + 1 - grp, slots 9 grp + 3 (sy + 1) ..).  They are
  // loaded one line ahead of their products.
  double vn[3][3];
  auto values = [&](int p, int sy) {
#pragma unroll
    for (int grp = 0; grp < 3; ++grp) {
      const int zrow = p + 1 - grp;
      const bool need = live && zrow >= z0 && zrow < z1;
#pragma unroll
      for (int i = 0; i < 3; ++i)
        vn[grp][i] = need ? V[box_at(g, vblk, zrow, grp * 9 + (sy + 1) * 3 + i, vt)] : 0.0;
    }
  };
  fetch(z0 - 1);
  values(z0 - 1, -1);
  put(0);
  __syncthreads();
  for (int p = z0 - 1; p <= z1; ++p) {
    const int buf = (p - z0 + 1) & 1;
    if (PF && p < z1) fetch(p + 1);
    const bool pin = p >= 0 && p < g.gz;  // X plane p exists: every slot reading it is in range in z
    // the row of plane q takes its slots (sz+1)*9 .. (sz+1)*9+8 at step q + sz
    const bool rowC = live && p - 1 >= z0 && p - 1 < z1;  // complete after this step
    const double* wp = win[buf];
    // one line of the plane at a time: each cell's X piece is read from LDS once
    // and goes into all three rows in flight.  Out of range the value and the X
    // entry are 0: adding +0.0 leaves a sum that started at +0.0 as it is; rows
    // that this chunk does not store are never read.
#pragma unroll 1
    for (int sy = -1; sy <= 1; ++sy) {
      double v[3][3];
#pragma unroll
      for (int grp = 0; grp < 3; ++grp)
#pragma unroll
        for (int i = 0; i < 3; ++i) v[grp][i] = vn[grp][i];
      if (sy < 1) values(p, sy + 1);
      else if (p < z1) values(p + 1, -1);
#pragma unroll
      for (int sx = -1; sx <= 1; ++sx) {
        const double* xp = wp + (c0 + sy * WX + sx) * K;
        double xv[CPL];
#pragma unroll
        for (int q = 0; q < CPL; ++q) xv[q] = xp[col(q)];
#pragma unroll
        for (int q = 0; q < CPL; ++q) accA[q] += v[0][sx + 1] * xv[q];
#pragma unroll
        for (int q = 0; q < CPL; ++q) accB[q] += v[1][sx + 1] * xv[q];
#pragma unroll
        for (int q = 0; q < CPL; ++q) accC[q] += v[2][sx + 1] * xv[q];
      }
    }
    if (rowC) {  // the row of plane p-1 is complete
      double* dst = Y + ((int64_t)(p - 1) * plane + ix + (int64_t)g.gx * iy) * K;
#pragma unroll
      for (int q = 0; q < CPL; ++q) {
        dst[col(q)] = accC[q];
        tsum[q] += accC[q] * xown[q];
      }
    }
    // this node's X of plane p, for the dot of the row of plane p (complete at step p+1)
    if (pin) {
#pragma unroll
      for (int q = 0; q < CPL; ++q) xown[q] = win[buf][c0 * K + col(q)];
    }
#pragma unroll
    for (int q = 0; q < CPL; ++q) {
      accC[q] = accB[q];
      accB[q] = accA[q];
      accA[q] = 0.0;
    }
    if (p < z1) {
      if (!PF) fetch(p + 1);
      put(buf ^ 1);
    }
    __syncthreads();
  }
  if (partials) {
    __shared__ double red[kBlock / kWave][K];
    const int lane = t % kWave, wave = t / kWave;
#pragma unroll
    for (int q = 0; q < CPL; ++q) {
      const double s = sum_same_column<L>(tsum[q]);
      if (lane < L) red[wave][col(q)] = s;
    }
    __syncthreads();
    if (t < K) {
      double s = red[0][t];
#pragma unroll
      for (int w = 1; w < kBlock / kWave; ++w) s += red[w][t];
      partials[(int64_t)wg * K + t] = s;
    }
  }
}

template <int K, int MX, bool XCD, bool PF, int MINB>
__global__ __launch_bounds__(kBlock, MINB) void spmm_boxp_kernel(
    BoxGeom g, int nbxm, int nzc, int zc, const double* __restrict__ V,
    const double* __restrict__ X, double* __restrict__ Y, double* __restrict__ partials,
    const int* __restrict__ done) {
  if (done && *done) return;
  spmm_boxp_body<K, MX, XCD, PF>((int)blockIdx.x, (int)gridDim.x, g, nbxm, nzc, zc, V, X, Y,
                                 partials);
}

// The box tiles the tuner tries: block width MX (MY = 64 / MX), XCD-contiguous
// tile order, X prefetch, and a minimum of MINB resident workgroups per CU
// (MINB 3: at most 168 VGPRs; the kernel needs 148 and 156, the next line's nine
// values among them).  Bound by the memory system: 1.0 GB per product at
// 128^3 x 16 (values 0.47, X 0.27, Y 0.27), 206 us at the rate of a copy.
// Measured there (us per SpMM, one MI355X): 8 x 8 prefetch 308, 16 x 4 XCD 326.
// With the values loaded slot by slot, nine loads of one row ahead of 9 K
// products, and each X piece read from LDS three times, the same tiles took 365
// and 360 (MINB 5, five workgroups per CU); that loop line by line but without
// the values ahead 304 and 384, with them and MINB 4 (21 VGPRs spilled) 468 for
// 16 x 4.  8 x 8 XCD with prefetch 310, without 315; 16 x 4 with prefetch 318.
// K = 8: 246 and 251 (before: 269 and 255).
struct BoxVariant {
  int mx;
  bool xcd, prefetch;
  int minb;
};
constexpr BoxVariant kBoxVariants[] = {{16, true, false, 3}, {8, false, true, 3}};
constexpr int kBoxVariantCount = 2;

template <int K, int V>
static const void* box_kernel_ptr() {
  constexpr BoxVariant bv = kBoxVariants[V];
  return (const void*)spmm_boxp_kernel<K, bv.mx, bv.xcd, bv.prefetch, bv.minb>;
}

// Blocks and z chunks of box variant V's launch (chunks filling whole rounds
// of the kernel's resident workgroups, at most one workgroup per row).
template <int K, int V>
static BoxGeom box_spmm_shape(const BoxGeom& g, int cus) {
  constexpr BoxVariant bv = kBoxVariants[V];
  BoxGeom m = g;
  m.nbx = (int)cdiv(g.gx, bv.mx);
  m.nby = (int)cdiv(g.gy, kBoxNodes / bv.mx);
  box_chunks(m, resident_groups(box_kernel_ptr<K, V>(), cus), (int64_t)g.gx * g.gy * g.gz);
  return m;
}

template <int K, int V>
static hipError_t launch_box_variant(const SpmmArgs& a, const double* X, double* Y,
                                     double* partials, const int* done, hipStream_t s,
                                     int* blocks_out) {
  constexpr BoxVariant bv = kBoxVariants[V];
  const BoxGeom m = box_spmm_shape<K, V>(a.bg, a.cus);
  const unsigned g = (unsigned)((int64_t)m.nbx * m.nby * m.nzc);
  if (blocks_out) *blocks_out = (int)g;
  if (a.n == 0) return hipSuccess;
  spmm_boxp_kernel<K, bv.mx, bv.xcd, bv.prefetch, bv.minb>
      <<<g, kBlock, 0, s>>>(a.bg, m.nbx, m.nzc, m.zc, a.bvals, X, Y, partials, done);
  return hipGetLastError();
}

// Line record of slice s, lines[s * kLineStride ...]: [0] = w / 3 when
// slice s can take spmm_sell_kernel's line path, else 0; then [1 + g] = slot
// 3g+1's column in the slice's first row.  The path applies when the 64 rows
// (all < n) have the slice's width w, a positive multiple of 3; slot j's
// column is slot j's column of the first row + lane; and slots 3g+1 and 3g+2
// hold slot 3g's column + 1 and + 2.  One wave per slice.
__global__ __launch_bounds__(kBlock) void sell_lines_kernel(int n, int nslices,
                                                            const int* __restrict__ soff,
                                                            const unsigned char* __restrict__ slen,
                                                            const int* __restrict__ scols,
                                                            int* __restrict__ lines) {
  const int slice = (int)blockIdx.x * (kBlock / kWave) + (int)threadIdx.x / kWave;
  const int lane = (int)threadIdx.x % kWave;
  if (slice >= nslices) return;  // whole waves
  const int o = soff[slice], w = soff[slice + 1] - o;
  const int64_t row = (int64_t)slice * kWave + lane;
  const int64_t o64 = (int64_t)o * kWave;
  int* const rec = lines + (int64_t)slice * kLineStride;
  bool ok = w > 0 && w % 3 == 0 && w / 3 < kLineStride && row < n && slen[row] == w;
  int prev = 0;
  for (int j = 0; j < w; ++j) {
    const int c = scols[sell_pos(o64, j, w, lane)];
    const int c0 = __shfl(c, 0, kWave);
    ok = ok && c == c0 + lane && (j % 3 == 0 || c == prev + 1);
    if (lane == 0 && j % 3 == 1 && 1 + j / 3 < kLineStride) rec[1 + j / 3] = c;
    prev = c;
  }
  const int all = __all(ok ? 1 : 0);
  if (lane == 0) rec[0] = all ? w / 3 : 0;
}

// The line flags of A's SELL-64 copy (built once per structure).
static int ensure_lines(mfe_ctx* ctx, const mfe_csr* Ac) {
  mfe_csr* A = const_cast<mfe_csr*>(Ac);
  if (!A->sell_ok || A->sell_lines_valid) return MFE_OK;
  const int ns = (int)A->sell_nslices;
  if (!A->sell_lines)
    MFE_CHECK(ctx, dev_alloc(ctx, &A->sell_lines, sizeof(int) * kLineStride * (size_t)std::max(ns, 1)));
  if (ns > 0) {
    sell_lines_kernel<<<(unsigned)cdiv(ns, kBlock / kWave), kBlock, 0, ctx->stream>>>(
        (int)A->nrows, ns, A->sell_off, A->sell_len, A->sell_cols, A->sell_lines);
    MFE_LAUNCHED(ctx, "sell_lines_kernel");
  }
  A->sell_lines_valid = true;
  return MFE_OK;
}

// Staged shapes need whole waves and at most 1024 threads: 64 <= R (K / CPL).
template <int K, int CPL, int U, int R>
static hipError_t launch_staged(const SpmmArgs& a, size_t lds, const double* X, double* Y,
                                double* partials, const int* done, hipStream_t s) {
  constexpr int NT = CPL <= K ? R * (K / CPL) : 0;
  if constexpr (NT >= kWave && NT <= 1024) {
    const SpmmPlan& p = *a.plans[plan_slot(R)];
    spmm_staged_kernel<K, CPL, U, R><<<p.ntiles, NT, lds, s>>>(a.n, a.ro, p.lcols, a.vals, p.uoff,
                                                                 p.ucols, X, Y, partials, done);
    return hipGetLastError();
  } else {
    return hipErrorInvalidValue;
  }
}

template <int K>
static hipError_t launch_spmm(int tile, const SpmmArgs& a, const double* X, double* Y,
                              double* partials, const int* done, hipStream_t s, int* blocks_out) {
  const SpmmTile T = tile_of(K, tile);
  const int n = a.n;
  if (T.rows == kBoxTile) {
    if (!a.bvals) return hipErrorInvalidValue;
    static_assert(kBoxVariantCount == 2, "one case per box variant");
    switch (T.box) {
      case 0: return launch_box_variant<K, 0>(a, X, Y, partials, done, s, blocks_out);
      case 1: return launch_box_variant<K, 1>(a, X, Y, partials, done, s, blocks_out);
      default: return hipErrorInvalidValue;
    }
  }
  if (T.rows == kSellTile || T.rows == kSellLineTile) {
    const bool lines = T.rows == kSellLineTile;
    if (!a.svals || (lines && !a.lines)) return hipErrorInvalidValue;
    const int rpb = kBlock / (K / T.cpl);
    const unsigned g = (unsigned)cdiv((int64_t)a.nslices * kWave, rpb);
    if (blocks_out) *blocks_out = (int)g;
    if (n == 0) return hipSuccess;
#define MFE_SELL_CASE(C, UU, LN)                                                                \
    if (T.cpl == C && T.unroll == UU && lines == LN) {                                         \
      spmm_sell_kernel<K, (C <= K ? C : K), UU, LN><<<g, kBlock, 0, s>>>(                      \
          n, a.nslices, a.soff, a.slen, a.scols, a.svals, a.lines, X, Y, partials, done);     \
      return hipGetLastError();                                                                \
    }
    MFE_SELL_CASE(1, 9, false)
    MFE_SELL_CASE(2, 9, false)
    MFE_SELL_CASE(4, 9, false)
    MFE_SELL_CASE(8, 9, false)
    MFE_SELL_CASE(1, 9, true)
    MFE_SELL_CASE(2, 9, true)
    MFE_SELL_CASE(4, 9, true)
    MFE_SELL_CASE(8, 9, true)
#undef MFE_SELL_CASE
    return hipErrorInvalidValue;
  }
  if (T.rows > 0) {
    const SpmmPlan* p = a.plans[plan_slot(T.rows)];
    if (!stage_ok(p, K) || p->rows != T.rows) return hipErrorInvalidValue;
    if (blocks_out) *blocks_out = p->ntiles;
    const size_t lds = (size_t)p->maxu * K * sizeof(double);
#define MFE_STAGED_CASE(C, UU, RR)                  \
    if (T.cpl == C && T.unroll == UU && T.rows == RR) \
      return launch_staged<K, C, UU, RR>(a, lds, X, Y, partials, done, s);
    MFE_STAGED_CASE(1, 9, 16)
    MFE_STAGED_CASE(2, 9, 16)
    MFE_STAGED_CASE(1, 9, 32)
    MFE_STAGED_CASE(2, 9, 32)
    MFE_STAGED_CASE(4, 9, 32)
#undef MFE_STAGED_CASE
    return hipErrorInvalidValue;
  }
  const int rpb = kBlock / (K / T.cpl);
  const unsigned g = (unsigned)cdiv(n, rpb);
  if (blocks_out) *blocks_out = (int)g;
  if (n == 0) return hipSuccess;
#define MFE_SPMM_CASE(C, UU)                                                                \
  if (T.cpl == C && T.unroll == UU) {                                                      \
    spmm_kernel<K, (C <= K ? C : K), UU><<<g, kBlock, 0, s>>>(n, a.ro, a.cols, a.vals, X, Y, \
                                                               partials, done);            \
    return hipGetLastError();                                                              \
  }
  MFE_SPMM_CASE(1, 9)
  MFE_SPMM_CASE(2, 9)
  MFE_SPMM_CASE(4, 9)
  MFE_SPMM_CASE(8, 9)
  MFE_SPMM_CASE(2, 3)
  MFE_SPMM_CASE(4, 3)
  MFE_SPMM_CASE(8, 3)
  MFE_SPMM_CASE(16, 3)
#undef MFE_SPMM_CASE
  return hipErrorInvalidValue;
}

static hipError_t launch_spmm_k(int K, int tile, const SpmmArgs& a, const double* X, double* Y,
                                double* partials, const int* done, hipStream_t s,
                                int* blocks_out) {
  switch (K) {
    case 16: return launch_spmm<16>(tile, a, X, Y, partials, done, s, blocks_out);
    case 8: return launch_spmm<8>(tile, a, X, Y, partials, done, s, blocks_out);
    case 4: return launch_spmm<4>(tile, a, X, Y, partials, done, s, blocks_out);
    default: return hipErrorInvalidValue;
  }
}

static int k_slot(int K) { return K == 16 ? 2 : K == 8 ? 1 : 0; }

// Tile `tile` can run on A for K with these operands.
static bool tile_available(int K, int tile, const SpmmArgs& a) {
  const int R = tile_of(K, tile).rows;
  if (R == kBoxTile) return a.bvals != nullptr && a.n > 0;
  if (R == kSellTile) return a.svals != nullptr && a.n > 0;
  if (R == kSellLineTile) return a.svals != nullptr && a.lines != nullptr && a.n > 0;
  return R == 0 || stage_ok(a.plans[plan_slot(R)], K);
}

// ---------------------------------------------------------- autotuner -------

struct SpmmTuning {
  const mfe_csr* A = nullptr;
  uint64_t gen = 0;
  int tile[3] = {-1, -1, -1};
  double ms[3][kMaxTiles] = {};
};

// Times every available tile for K on A (3 launches each after one warm-up,
// HIP events on ctx's stream) and keeps the fastest; unavailable tiles get
// ms = +inf.  X and Y are scratch of n*K.
static int tune_spmm(mfe_ctx* ctx, const SpmmArgs& a, int K, const double* X, double* Y,
                     SpmmTuning& tun) {
  hipStream_t s = ctx->stream;
  const int nt = tile_count(K);
  const int slot = k_slot(K);
  int best = 0;
  double best_ms = HUGE_VAL;
  for (int id = 0; id < nt; ++id) {
    if (!tile_available(K, id, a)) {
      tun.ms[slot][id] = HUGE_VAL;
      continue;
    }
    MFE_CHECK(ctx, launch_spmm_k(K, id, a, X, Y, nullptr, nullptr, s, nullptr));
    MFE_CHECK(ctx, hipEventRecord(ctx->t_start, s));
    const int reps = 3;
    for (int r = 0; r < reps; ++r)
      MFE_CHECK(ctx, launch_spmm_k(K, id, a, X, Y, nullptr, nullptr, s, nullptr));
    MFE_CHECK(ctx, hipEventRecord(ctx->t_stop, s));
    MFE_CHECK(ctx, hipEventSynchronize(ctx->t_stop));
    float ms = 0;
    MFE_CHECK(ctx, hipEventElapsedTime(&ms, ctx->t_start, ctx->t_stop));
    tun.ms[slot][id] = ms / reps;
    if (tun.ms[slot][id] < best_ms) {
      best_ms = tun.ms[slot][id];
      best = id;
    }
  }
  tun.tile[slot] = best;
  return MFE_OK;
}

// ------------------------------------------------------ column reductions ---

constexpr int kColStage = 1024;  // partial rows per stage-1 workgroup

// Sum over rows r of [r0, r1) of in[r*K + k], k = threadIdx.x % K, fixed order:
// thread (t / K) walks rows t/K, t/K + 256/K, ... (eight loads in flight: one at a
// time a first stage of 1,024 rows took 10.8 us at K = 16, so 6.7); then the 256/K
// threads of a column add up in a fixed tree.  Valid in the first K threads; sh:
// kBlock values.
template <int K>
__device__ __forceinline__ double sum_cols(const double* __restrict__ in, int r0, int r1,
                                           double* sh) {
  constexpr int G = kBlock / K;  // threads per column
  constexpr int U = 8;
  const int t = (int)threadIdx.x;
  const int k = t % K, g = t / K;
  double s = 0.0;
  int r = r0 + g;
  for (; r + (U - 1) * G < r1; r += U * G) {
    double v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = in[(int64_t)(r + u * G) * K + k];
#pragma unroll
    for (int u = 0; u < U; ++u) s += v[u];
  }
  for (; r < r1; r += G) s += in[(int64_t)r * K + k];
  sh[t] = s;
  __syncthreads();
  for (int w = G / 2; w > 0; w >>= 1) {
    if (g < w) sh[t] += sh[t + w * K];
    __syncthreads();
  }
  return sh[k];
}

// First stage: out[b*K + k] = the sum of rows [b*chunk, (b+1)*chunk).
template <int K>
__global__ __launch_bounds__(kBlock) void reduce_cols_kernel(const double* __restrict__ in,
                                                             int rows, int chunk,
                                                             double* __restrict__ out,
                                                             const int* __restrict__ done) {
  if (done && *done) return;
  __shared__ double sh[kBlock];
  const int r0 = (int)blockIdx.x * chunk, r1 = min(r0 + chunk, rows);
  const double s = sum_cols<K>(in, r0, r1, sh);
  if ((int)threadIdx.x < K) out[(int64_t)blockIdx.x * K + threadIdx.x] = s;
}

// ------------------------------------------------------------ CG state -------

// pending[c]: column c's update X += palpha[c] P of the last iteration is
// still to be applied (by the next P update, or by multi_finish_kernel).
struct MultiState {
  double rtrans[16], oldrtrans[16], pAp[16], alpha[16], beta[16], normr[16], tol[16], bnorm[16],
      palpha[16];
  int active[16], iters[16], breakdown[16], pending[16];
  int k, max_iter, done, pad;
};

__global__ void multi_init_kernel(MultiState* st, int K, int max_iter, double rel_tol,
                                  const double* bb, const double* rr) {
  const int c = (int)threadIdx.x;
  if (c == 0) {
    st->k = 1;
    st->max_iter = max_iter;
  }
  if (c < 16) {
    const bool live = c < K;
    st->rtrans[c] = live ? rr[c] : 0.0;
    st->oldrtrans[c] = 0.0;
    st->normr[c] = live ? sqrt(rr[c]) : 0.0;
    st->bnorm[c] = live ? sqrt(bb[c]) : 0.0;
    st->tol[c] = rel_tol * st->bnorm[c];
    st->alpha[c] = st->beta[c] = st->pAp[c] = 0.0;
    st->iters[c] = 0;
    st->breakdown[c] = 0;
    st->pending[c] = 0;
    st->palpha[c] = 0.0;
    st->active[c] = live && max_iter >= 1 && st->normr[c] > st->tol[c];
  }
  __syncthreads();
  if (c == 0) {
    int any = 0;
    for (int q = 0; q < K; ++q) any |= st->active[q];
    st->done = !any;
  }
}

// The last iteration's X += palpha P where pending, then P = R (k = 1) or
// P = R + beta P for active columns (grid-stride with a stride that is a
// multiple of K: a thread always sees the same column).
template <int K>
__global__ __launch_bounds__(kBlock) void multi_p_kernel(int64_t nk, const MultiState* st,
                                                         const double* __restrict__ R,
                                                         double* __restrict__ P,
                                                         double* __restrict__ X) {
  if (st->done) return;
  const bool first = st->k == 1;
  const int c = (int)(((int64_t)blockIdx.x * blockDim.x + threadIdx.x) % K);
  const bool pend = st->pending[c], act = st->active[c];
  const double a = st->palpha[c], b = st->beta[c];
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nk; i += stride) {
    if (pend) X[i] = 1.0 * X[i] + a * P[i];
    if (act) P[i] = first ? 1.0 * R[i] + 0.0 * R[i] : 1.0 * R[i] + b * P[i];
  }
}

// The update still pending when the loop has stopped.
template <int K>
__global__ __launch_bounds__(kBlock) void multi_finish_kernel(int64_t nk, const MultiState* st,
                                                              const double* __restrict__ P,
                                                              double* __restrict__ X) {
  const int c = (int)(((int64_t)blockIdx.x * blockDim.x + threadIdx.x) % K);
  if (!st->pending[c]) return;
  const double a = st->palpha[c];
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nk; i += stride)
    X[i] = 1.0 * X[i] + a * P[i];
}

// The second stage of the p.Ap reduction (nb rows of first-stage sums), then
// alpha per column.
template <int K>
__global__ __launch_bounds__(kBlock) void multi_alpha_kernel(MultiState* st, const double* part,
                                                             int nb) {
  if (st->done) return;
  __shared__ double sh[kBlock];
  const double pAp = sum_cols<K>(part, 0, nb, sh);
  const int c = (int)threadIdx.x;
  if (c < K && st->active[c]) {
    st->pAp[c] = pAp;
    if (!(pAp > 0.0)) {  // non-positive curvature: stop this column
      st->breakdown[c] = 1;
      st->active[c] = 0;
      st->alpha[c] = 0.0;
    } else {
      st->alpha[c] = st->rtrans[c] / pAp;
    }
  }
  if (c < K) {  // this iteration's X update, applied by the next P update
    st->pending[c] = st->active[c];
    st->palpha[c] = st->alpha[c];
  }
}

// R -= alpha AP for active columns, with R.R partials per column
// (grid-stride: a thread always sees the same column since the stride is a
// multiple of K).  X += alpha P is left to the next P update.
template <int K>
__global__ __launch_bounds__(kBlock) void multi_update_kernel(int64_t nk, const MultiState* st,
                                                              double* __restrict__ R,
                                                              const double* __restrict__ AP,
                                                              double* __restrict__ partials) {
  if (st->done) return;
  const int t = (int)threadIdx.x;
  const int c = t % K;
  const bool act = st->active[c];
  const double a = st->alpha[c];
  double s = 0.0;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + t; i < nk; i += stride) {
    double r = R[i];
    if (act) {
      r = 1.0 * r + (-a) * AP[i];
      R[i] = r;
    }
    s += r * r;
  }
  __shared__ double red[kBlock / kWave][K];
  s = sum_same_column<K>(s);
  const int lane = t % kWave, wave = t / kWave;
  if (lane < K) red[wave][lane] = s;
  __syncthreads();
  if (t < K) {
    double v = red[0][t];
#pragma unroll
    for (int w = 1; w < kBlock / kWave; ++w) v += red[w][t];
    partials[(int64_t)blockIdx.x * K + t] = v;
  }
}

// The second stage of the r.r reduction, then the end of the iteration per column.
template <int K>
__global__ __launch_bounds__(kBlock) void multi_next_kernel(MultiState* st, const double* part,
                                                            int nb) {
  if (st->done) return;
  __shared__ double sh[kBlock];
  const double rr = sum_cols<K>(part, 0, nb, sh);
  const int c = (int)threadIdx.x;
  const int k = st->k;
  __syncthreads();  // every thread has read k and done
  if (c < K && st->active[c]) {
    st->oldrtrans[c] = st->rtrans[c];
    st->rtrans[c] = rr;
    st->normr[c] = sqrt(rr);
    st->beta[c] = st->rtrans[c] / st->oldrtrans[c];
    st->iters[c] = k;
    if (!(st->normr[c] > st->tol[c]) || k + 1 > st->max_iter) st->active[c] = 0;
  }
  __syncthreads();
  if (c == 0) {
    int any = 0;
    for (int q = 0; q < K; ++q) any |= st->active[q];
    st->k = k + 1;
    st->done = !any;
  }
}

// R = B - Y elementwise.
__global__ __launch_bounds__(kBlock) void multi_resid_kernel(int64_t nk, const double* B,
                                                             const double* Y, double* R) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nk; i += stride)
    R[i] = 1.0 * B[i] + (-1.0) * Y[i];
}

// partials of column dots a[:,k].b[:,k]
template <int K>
__global__ __launch_bounds__(kBlock) void multi_dot_kernel(int64_t nk, const double* a,
                                                           const double* b, double* partials) {
  const int t = (int)threadIdx.x;
  double s = 0.0;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + t; i < nk; i += stride) s += a[i] * b[i];
  __shared__ double red[kBlock / kWave][K];
  s = sum_same_column<K>(s);
  const int lane = t % kWave, wave = t / kWave;
  if (lane < K) red[wave][lane] = s;
  __syncthreads();
  if (t < K) {
    double v = red[0][t];
#pragma unroll
    for (int w = 1; w < kBlock / kWave; ++w) v += red[w][t];
    partials[(int64_t)blockIdx.x * K + t] = v;
  }
}

struct MultiWorkspace {
  int64_t nk = -1;
  int K = 0;
  double *R = nullptr, *P = nullptr, *AP = nullptr, *part = nullptr, *part2 = nullptr,
         *res = nullptr;
  int64_t part_rows = 0;
  MultiState* st = nullptr;
  MultiState* h_st = nullptr;
  hipGraphExec_t exec = nullptr;
  hipGraph_t graph = nullptr;
  const void *kA = nullptr, *kX = nullptr;
  uint64_t kgen = 0;
  int ktile = -1;
  SpmmTuning tun;
  SpmmPlan plans[2];  // 16- and 32-row staging plans of one matrix (kept across nk changes)
  void drop_graph() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    exec = nullptr;
    graph = nullptr;
    kA = kX = nullptr;
  }
  void release() {
    drop_graph();
    (void)hipFree(R);
    (void)hipFree(P);
    (void)hipFree(AP);
    (void)hipFree(part);
    (void)hipFree(part2);
    (void)hipFree(res);
    (void)hipFree(st);
    if (h_st) (void)hipHostFree(h_st);
    R = P = AP = part = part2 = res = nullptr;
    st = nullptr;
    h_st = nullptr;
    nk = -1;
  }
};

static unsigned multi_vec_grid(int64_t nk) {
  const int64_t b = cdiv(nk, kBlock);
  return (unsigned)std::max<int64_t>(1, std::min<int64_t>(b, kVecBlocks));
}

// The R-row staging plan of A in ctx's workspace, rebuilt when A or its
// structure changed.  A rebuilt plan moves its arrays, so the captured CG
// graph (which holds their addresses) is dropped with it.
static int ensure_plan(mfe_ctx* ctx, const mfe_csr* A, int R) {
  if (!ctx->multi) ctx->multi = new MultiWorkspace();
  MultiWorkspace* w = ctx->multi;
  SpmmPlan& p = w->plans[plan_slot(R)];
  if (!p.built || p.A != A || p.gen != A->plan_gen) {
    w->drop_graph();
    const int st = build_stage_plan(ctx, A, R, p);
    if (st) {
      p.release();
      return st;
    }
  }
  return MFE_OK;
}

// Operands for A with the workspace's plans that belong to A (others null)
// and A's SELL-64 copy when it is current.
static SpmmArgs spmm_args(const mfe_csr* A, const MultiWorkspace* w) {
  SpmmArgs a{(int)A->nrows, A->row_offsets, A->cols, A->vals, {nullptr, nullptr},
             0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, BoxGeom{},
             A->ctx ? A->ctx->cu_count : 0};
  if (A->box_vals_valid && A->box_vals && A->box_elems[0] > 0) {
    a.bvals = A->box_vals;
    a.bg = A->box_geom;
  }
  if (w)
    for (int i = 0; i < 2; ++i)
      if (w->plans[i].built && w->plans[i].A == A && w->plans[i].gen == A->plan_gen)
        a.plans[i] = &w->plans[i];
  if (A->sell_ok && A->sell_vals_valid && A->sell_vals) {
    a.nslices = (int)A->sell_nslices;
    a.soff = A->sell_off;
    a.slen = A->sell_len;
    a.scols = A->sell_cols;
    a.svals = A->sell_vals;
    if (A->sell_lines_valid) a.lines = A->sell_lines;
  }
  return a;
}

static int multi_prepare(mfe_ctx* ctx, int64_t n, int K, MultiWorkspace** out) {
  if (!ctx->multi) ctx->multi = new MultiWorkspace();
  MultiWorkspace* w = ctx->multi;
  const int64_t nk = n * K;
  if (w->nk != nk || w->K != K) {
    w->release();
    const size_t bytes = sizeof(double) * (size_t)std::max<int64_t>(nk, 1);
    MFE_CHECK(ctx, dev_malloc(ctx, &w->R, bytes));
    MFE_CHECK(ctx, dev_malloc(ctx, &w->P, bytes));
    MFE_CHECK(ctx, dev_malloc(ctx, &w->AP, bytes));
    // partial rows: the SpMM's workgroups (at most n with one row each) or
    // the vector kernels' grid
    w->part_rows = std::max<int64_t>(n, kVecBlocks) + 1;
    MFE_CHECK(ctx, dev_malloc(ctx, &w->part, sizeof(double) * (size_t)(w->part_rows * K)));
    MFE_CHECK(ctx, dev_malloc(ctx, &w->part2, sizeof(double) * (size_t)((cdiv(w->part_rows, kColStage) + 1) * K)));
    MFE_CHECK(ctx, dev_malloc(ctx, &w->res, sizeof(double) * 64));
    MFE_CHECK(ctx, dev_malloc(ctx, &w->st, sizeof(MultiState)));
    MFE_CHECK(ctx, hipHostMalloc(&w->h_st, sizeof(MultiState), hipHostMallocDefault));
    w->nk = nk;
    w->K = K;
  }
  *out = w;
  return MFE_OK;
}

// Two-stage column reduction of part[rows][K] into out[K].
static hipError_t reduce_cols(int K, const double* part, int rows, double* part2, double* out,
                              const int* done, hipStream_t s) {
  const int nb = (int)std::max<int64_t>(1, cdiv(rows, kColStage));
  switch (K) {
    case 16:
      reduce_cols_kernel<16><<<nb, kBlock, 0, s>>>(part, rows, kColStage, part2, done);
      reduce_cols_kernel<16><<<1, kBlock, 0, s>>>(part2, nb, nb, out, done);
      break;
    case 8:
      reduce_cols_kernel<8><<<nb, kBlock, 0, s>>>(part, rows, kColStage, part2, done);
      reduce_cols_kernel<8><<<1, kBlock, 0, s>>>(part2, nb, nb, out, done);
      break;
    default:
      reduce_cols_kernel<4><<<nb, kBlock, 0, s>>>(part, rows, kColStage, part2, done);
      reduce_cols_kernel<4><<<1, kBlock, 0, s>>>(part2, nb, nb, out, done);
  }
  return hipGetLastError();
}

template <int K>
static hipError_t enqueue_multi_iteration(MultiWorkspace* w, const mfe_csr* A, double* X,
                                          int tile, hipStream_t s) {
  const int64_t nk = w->nk;
  const unsigned vg = multi_vec_grid(nk);
  const int* done = &w->st->done;
  // no sum: one element per thread (0.5% faster per solve than the grid-stride form)
  multi_p_kernel<K><<<(unsigned)cdiv(nk, kBlock), kBlock, 0, s>>>(nk, w->st, w->R, w->P, X);
  int nb = 0;
  hipError_t e = launch_spmm<K>(tile, spmm_args(A, w), w->P, w->AP, w->part, done, s, &nb);
  if (e != hipSuccess) return e;
  const int s1 = (int)std::max<int64_t>(1, cdiv(nb, kColStage));
  reduce_cols_kernel<K><<<s1, kBlock, 0, s>>>(w->part, nb, kColStage, w->part2, done);
  multi_alpha_kernel<K><<<1, kBlock, 0, s>>>(w->st, w->part2, s1);
  multi_update_kernel<K><<<vg, kBlock, 0, s>>>(nk, w->st, w->R, w->AP, w->part);
  const int s2 = (int)std::max<int64_t>(1, cdiv(vg, kColStage));
  reduce_cols_kernel<K><<<s2, kBlock, 0, s>>>(w->part, (int)vg, kColStage, w->part2, done);
  multi_next_kernel<K><<<1, kBlock, 0, s>>>(w->st, w->part2, s2);
  return hipGetLastError();
}

static hipError_t enqueue_multi(int K, MultiWorkspace* w, const mfe_csr* A, double* X, int tile,
                                hipStream_t s) {
  switch (K) {
    case 16: return enqueue_multi_iteration<16>(w, A, X, tile, s);
    case 8: return enqueue_multi_iteration<8>(w, A, X, tile, s);
    default: return enqueue_multi_iteration<4>(w, A, X, tile, s);
  }
}

static hipError_t launch_multi_finish(int K, MultiWorkspace* w, double* X, hipStream_t s) {
  const unsigned vg = multi_vec_grid(w->nk);
  switch (K) {
    case 16: multi_finish_kernel<16><<<vg, kBlock, 0, s>>>(w->nk, w->st, w->P, X); break;
    case 8: multi_finish_kernel<8><<<vg, kBlock, 0, s>>>(w->nk, w->st, w->P, X); break;
    default: multi_finish_kernel<4><<<vg, kBlock, 0, s>>>(w->nk, w->st, w->P, X);
  }
  return hipGetLastError();
}

static hipError_t launch_multi_dot(int K, int64_t nk, const double* a, const double* b,
                                   double* part, hipStream_t s) {
  const unsigned vg = multi_vec_grid(nk);
  switch (K) {
    case 16: multi_dot_kernel<16><<<vg, kBlock, 0, s>>>(nk, a, b, part); break;
    case 8: multi_dot_kernel<8><<<vg, kBlock, 0, s>>>(nk, a, b, part); break;
    default: multi_dot_kernel<4><<<vg, kBlock, 0, s>>>(nk, a, b, part);
  }
  return hipGetLastError();
}

static bool k_ok(int K) { return K == 4 || K == 8 || K == 16; }

static int ensure_tuned(mfe_ctx* ctx, const mfe_csr* A, int K, MultiWorkspace* w) {
  const int slot = k_slot(K);
  int st;
  if ((st = box_prepare(ctx, A)) || (st = sell_prepare(ctx, A)) || (st = ensure_lines(ctx, A)) ||
      (st = ensure_plan(ctx, A, 16)) || (st = ensure_plan(ctx, A, 32)))
    return st;
  if (w->tun.A == A && w->tun.gen == A->plan_gen && w->tun.tile[slot] >= 0) return MFE_OK;
  if (w->tun.A != A || w->tun.gen != A->plan_gen) {
    w->tun = SpmmTuning();
    w->tun.A = A;
    w->tun.gen = A->plan_gen;
  }
  // scratch operands: R (filled with ones) and AP
  MFE_CHECK(ctx, hipMemsetAsync(w->R, 0, sizeof(double) * (size_t)w->nk, ctx->stream));
  return tune_spmm(ctx, spmm_args(A, w), K, w->R, w->AP, w->tun);
}

}  // namespace mfe

using namespace mfe;

extern "C" {

int mfe_spmm_tune(mfe_ctx* ctx, const mfe_csr* A, int nrhs, int* tile, double* ms, int* ntiles) {
  if (!ctx || !A || !k_ok(nrhs)) return MFE_BAD_ARG;
  uses(ctx, A);
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  MultiWorkspace* w = nullptr;
  int st;
  if ((st = multi_prepare(ctx, A->nrows, nrhs, &w))) return st;
  w->tun = SpmmTuning();  // re-time on request
  if ((st = ensure_tuned(ctx, A, nrhs, w))) return st;
  const int slot = k_slot(nrhs);
  if (tile) *tile = w->tun.tile[slot];
  if (ntiles) *ntiles = tile_count(nrhs);
  if (ms)
    for (int i = 0; i < tile_count(nrhs); ++i) ms[i] = w->tun.ms[slot][i];
  return MFE_OK;
}

int mfe_spmm_select(mfe_ctx* ctx, const mfe_csr* A, int nrhs, int tile) {
  if (!ctx || !A || !k_ok(nrhs)) return MFE_BAD_ARG;
  uses(ctx, A);
  if (tile < 0 || tile >= tile_count(nrhs)) return fail(ctx, MFE_BAD_ARG, "spmm_select: no such tile");
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  MultiWorkspace* w = nullptr;
  int st;
  if ((st = multi_prepare(ctx, A->nrows, nrhs, &w))) return st;
  if ((st = box_prepare(ctx, A)) || (st = sell_prepare(ctx, A)) || (st = ensure_lines(ctx, A)) ||
      (st = ensure_plan(ctx, A, 16)) || (st = ensure_plan(ctx, A, 32)))
    return st;
  if (!tile_available(nrhs, tile, spmm_args(A, w)))
    return fail(ctx, MFE_BAD_ARG, "spmm_select: staged tile unavailable for this matrix");
  if (w->tun.A != A || w->tun.gen != A->plan_gen) {
    w->tun = SpmmTuning();
    w->tun.A = A;
    w->tun.gen = A->plan_gen;
  }
  w->tun.tile[k_slot(nrhs)] = tile;
  return MFE_OK;
}

int mfe_spmm_tile_info(int nrhs, int tile, int* cols_per_lane, int* unroll, int* rows_per_block,
                       int* kind) {
  if (!k_ok(nrhs) || tile < 0 || tile >= tile_count(nrhs)) return MFE_BAD_ARG;
  const SpmmTile T = tile_of(nrhs, tile);
  if (cols_per_lane) *cols_per_lane = T.cpl;
  if (unroll) *unroll = T.unroll;
  if (rows_per_block)
    *rows_per_block = T.rows > 0 ? T.rows : T.rows == kBoxTile ? kBoxNodes
                                                                : kBlock / (nrhs / T.cpl);
  if (kind)
    *kind = T.rows > 0 ? 1 : T.rows == kSellTile ? 2 : T.rows == kSellLineTile ? 3
          : T.rows == kBoxTile ? 4 : 0;
  return MFE_OK;
}

int mfe_spmm(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* X, mfe_vec* Y, int nrhs, int tile) {
  if (!ctx || !A || !X || !Y || !k_ok(nrhs)) return MFE_BAD_ARG;
  uses(ctx, A, X, Y);
  const int64_t nk = A->nrows * nrhs;
  if (X->n != nk || Y->n != nk) return fail(ctx, MFE_BAD_ARG, "spmm: X and Y need nrows*nrhs values");
  if (tile >= tile_count(nrhs)) return fail(ctx, MFE_BAD_ARG, "spmm: no such tile");
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  int st;
  if (tile < 0) {  // the tuned tile for this matrix and nrhs
    MultiWorkspace* w = nullptr;
    if ((st = multi_prepare(ctx, A->nrows, nrhs, &w)) || (st = ensure_tuned(ctx, A, nrhs, w)))
      return st;
    tile = w->tun.tile[k_slot(nrhs)];
  }
  const int R = tile_of(nrhs, tile).rows;
  if (R > 0) {
    if ((st = ensure_plan(ctx, A, R))) return st;
    if (!stage_ok(&ctx->multi->plans[plan_slot(R)], nrhs))
      return fail(ctx, MFE_BAD_ARG,
                  "spmm: staged tile unavailable for this matrix (a row tile has more than "
                  "1024 non-zeros or its distinct X rows exceed 64 KiB)");
  } else if (R == kSellTile || R == kSellLineTile) {
    if ((st = sell_prepare(ctx, A)) || (st = ensure_lines(ctx, A))) return st;
    if (!(A->sell_ok && A->sell_vals_valid) || A->nrows == 0)
      return fail(ctx, MFE_BAD_ARG,
                  "spmm: SELL tile unavailable for this matrix (CSR format, or a row longer "
                  "than 27 entries)");
  } else if (R == kBoxTile) {
    if ((st = box_prepare(ctx, A))) return st;
    if (!A->box_vals_valid || A->nrows == 0)
      return fail(ctx, MFE_BAD_ARG,
                  "spmm: box tile unavailable for this matrix (it does not hold a box's "
                  "generated structure, or its format is not MFE_SPMV_AUTO)");
  }
  MFE_CHECK(ctx, launch_spmm_k(nrhs, tile, spmm_args(A, ctx->multi), X->d, Y->d, nullptr, nullptr,
                               ctx->stream, nullptr));
  return MFE_OK;
}

int mfe_cg_solve_multi(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* B, mfe_vec* X, int nrhs,
                       int max_iter, double rel_tol, int* iters, double* rel_residual,
                       double* seconds) {
  if (!ctx || !A || !B || !X || !k_ok(nrhs) || max_iter < 0) return MFE_BAD_ARG;
  uses(ctx, A, B, X);
  if (!A->has_local_indices)
    return fail(ctx, MFE_NOT_LOCAL,
                "cg_solve_multi: A.has_local_indices is false; call make_local_matrix(A) first");
  const int K = nrhs;
  const int64_t n = A->nrows, nk = n * K;
  if (B->n != nk || X->n != nk)
    return fail(ctx, MFE_BAD_ARG, "cg_solve_multi: B and X need nrows*nrhs values (row-major)");
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  hipStream_t s = ctx->stream;
  MultiWorkspace* w = nullptr;
  int st;
  if ((st = multi_prepare(ctx, n, K, &w)) || (st = ensure_tuned(ctx, A, K, w))) return st;
  const int tile = w->tun.tile[k_slot(K)];
  MFE_CHECK(ctx, hipEventRecord(ctx->t_start, s));
  if (n > 0) {
    // R = B - A X ; tolerances from ||B[:,k]||, rtrans = ||R[:,k]||^2
    int nb = 0;
    MFE_CHECK(ctx, launch_spmm_k(K, tile, spmm_args(A, w), X->d, w->AP, nullptr, nullptr, s,
                                 &nb));
    multi_resid_kernel<<<multi_vec_grid(nk), kBlock, 0, s>>>(nk, B->d, w->AP, w->R);
    MFE_CHECK(ctx, launch_multi_dot(K, nk, B->d, B->d, w->part, s));
    MFE_CHECK(ctx, reduce_cols(K, w->part, (int)multi_vec_grid(nk), w->part2, w->res + 32, nullptr, s));
    MFE_CHECK(ctx, launch_multi_dot(K, nk, w->R, w->R, w->part, s));
    MFE_CHECK(ctx, reduce_cols(K, w->part, (int)multi_vec_grid(nk), w->part2, w->res + 48, nullptr, s));
    multi_init_kernel<<<1, 64, 0, s>>>(w->st, K, max_iter, rel_tol, w->res + 32, w->res + 48);
    MFE_LAUNCHED(ctx, "multi prologue");
    const bool reuse = w->exec && w->kA == A && w->kgen == A->plan_gen && w->kX == X->d &&
                       w->ktile == tile;
    if (!reuse) {
      w->drop_graph();
      MFE_CHECK(ctx, hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
      hipError_t ce = hipSuccess;
      for (int c = 0; c < 25 && ce == hipSuccess; ++c) ce = enqueue_multi(K, w, A, X->d, tile, s);
      hipGraph_t g = nullptr;
      hipError_t ee = hipStreamEndCapture(s, &g);
      if (ce != hipSuccess) {
        if (g) (void)hipGraphDestroy(g);
        return hip_fail(ctx, ce, "cg_solve_multi capture");
      }
      if (ee != hipSuccess) return hip_fail(ctx, ee, "hipStreamEndCapture");
      w->graph = g;
      MFE_CHECK(ctx, hipGraphInstantiate(&w->exec, g, nullptr, nullptr, 0));
      w->kA = A;
      w->kgen = A->plan_gen;
      w->kX = X->d;
      w->ktile = tile;
    }
    const int chunks = (int)cdiv(std::max(max_iter, 1), 25);
    for (int c = 0; c < chunks; ++c) {
      MFE_CHECK(ctx, hipGraphLaunch(w->exec, s));
      MFE_CHECK(ctx, hipMemcpyAsync(w->h_st, w->st, sizeof(MultiState), hipMemcpyDeviceToHost, s));
      MFE_CHECK(ctx, hipStreamSynchronize(s));
      if (w->h_st->done) break;
    }
    MFE_CHECK(ctx, launch_multi_finish(K, w, X->d, s));
  }
  MFE_CHECK(ctx, hipEventRecord(ctx->t_stop, s));
  MFE_CHECK(ctx, hipEventSynchronize(ctx->t_stop));
  float ms = 0;
  MFE_CHECK(ctx, hipEventElapsedTime(&ms, ctx->t_start, ctx->t_stop));
  if (seconds) *seconds = 1e-3 * ms;
  if (n == 0) return MFE_OK;
  const MultiState hs = *w->h_st;
  int brk = 0;
  for (int c = 0; c < K; ++c) {
    if (iters) iters[c] = hs.iters[c];
    if (rel_residual) rel_residual[c] = hs.bnorm[c] > 0 ? hs.normr[c] / hs.bnorm[c] : hs.normr[c];
    brk |= hs.breakdown[c];
  }
  if (brk) return fail(ctx, MFE_BREAKDOWN, "cg_solve_multi: CG breakdown in a column");
  return MFE_OK;
}

void mfe_multi_workspace_free(mfe_ctx* ctx) {
  if (ctx && ctx->multi) {
    ctx->multi->release();
    ctx->multi->plans[0].release();
    ctx->multi->plans[1].release();
    delete ctx->multi;
    ctx->multi = nullptr;
  }
}

}  // extern "C"
