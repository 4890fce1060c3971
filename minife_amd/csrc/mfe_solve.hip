// CSR SpMV, vector kernels and the conjugate-gradient solvers on gfx950.
//
// SpMV ("row-stream"): a workgroup owns 256 consecutive rows.  Its threads
// stream the rows' value/column arrays with coalesced loads, form every
// product vals[j] * x[cols[j]] (rounded, as the reference's a*b) and park it
// in LDS; then thread t adds up row r0+t's products in stored column order.
// That is exactly matvec_std's arithmetic (SparseMatrix_functions.hpp:566-572)
// with HBM traffic of one pass over vals/cols.  No MFMA: the operator is sparse.
//
// CG: one HIP stream, device-resident scalars and fused kernels, launched one by
// one behind the GPU's progress word (small systems) or in chunks of iterations
// captured in a HIP graph and replayed; every kernel checks a device "done" flag so
// the reference's data-dependent loop test (cg_solve.hpp:152) stops the work
// without host round trips.  The kernels are
// templated on the vector type: double for cg_solve, float for the inner solve
// of the mixed-precision refinement.
#include <algorithm>
#include <cfloat>
#include <climits>
#include <cmath>
#include <cstring>
#include <mutex>
#include <tuple>
#include <type_traits>

#include "mfe_box.hpp"
#include "mfe_boxsym.hpp"
#include "mfe_common.hpp"
#include "mfe_sell.hpp"

namespace mfe {

// ---------------------------------------------------------------- SpMV ------

// MODE (SpmvMode): kPlain, kDot with the partial of x.y at partials[tile],
// kResid with the partial of y.y.  ZERO_Y: start each row sum at
// 0*y[row] (matvec_std's beta*ycoefs[row]); otherwise at +0.0 without reading
// y.  Loads whose addresses do not depend on the column stream (row offsets,
// y[row], x[row], b[row]) are issued first, so no memory round trip sits
// between the LDS barrier and the row sums.
template <typename T, bool ZERO_Y, int MODE>
__global__ __launch_bounds__(kBlock) void spmv_stream_kernel(
    int n, const int* __restrict__ ro, const int* __restrict__ cols,
    const T* __restrict__ vals, const T* __restrict__ x, T* __restrict__ y,
    const T* __restrict__ bvec, T* __restrict__ partials, const int* __restrict__ done) {
  if (done && *done) return;
  __shared__ T prod[kSpmvMaxNnz];
  __shared__ T red[4];
  const int tile = (int)blockIdx.x;
  const int r0 = tile * kSpmvRows;
  const int r1 = min(r0 + kSpmvRows, n);
  const int t = (int)threadIdx.x;
  const int row = r0 + t;
  const bool valid = row < r1;
  const int rr = valid ? row : r1 - 1;
  const int ra = ro[rr], rb = ro[rr + 1];
  const T y0 = ZERO_Y ? y[rr] : T(0);
  const T xr = MODE == kDot ? x[rr] : T(0);
  const T br = MODE == kResid ? bvec[rr] : T(0);
  const int s = ro[r0];
  const int cnt = ro[r1] - s;
  if (cnt > 0) {
    // Every column and value load of the tile before the first use (indices
    // clamped into the tile, so all loads are unconditional), then every x
    // gather, then the products: 27 loads in flight per lane.
    constexpr int K = kSpmvMaxNnz / kBlock;
    int c[K];
    T v[K], xv[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int i = t + k * kBlock;
      const int j = s + (i < cnt ? i : 0);
      c[k] = cols[j];
      v[k] = vals[j];
    }
#pragma unroll
    for (int k = 0; k < K; ++k) xv[k] = x[c[k]];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int i = t + k * kBlock;
      if (i < cnt) prod[i] = v[k] * xv[k];
    }
  }
  __syncthreads();
  T sum = T(0);
  if (valid) {
    if (ZERO_Y) sum = T(0) * y0;
    const int a = ra - s, b = rb - s;
    int j = a;
    for (; j + 4 <= b; j += 4) {  // LDS reads ahead, additions still in order
      const T p0 = prod[j], p1 = prod[j + 1], p2 = prod[j + 2], p3 = prod[j + 3];
      sum += p0;
      sum += p1;
      sum += p2;
      sum += p3;
    }
    for (; j < b; ++j) sum += prod[j];
    if (MODE == kResid) sum = T(1) * br + T(-1) * sum;
    y[row] = sum;
  }
  if (MODE != kPlain) {
    const T term = MODE == kDot ? sum * xr : sum * sum;
    const T v0 = block_sum<T>(valid ? term : T(0), red);
    if (t == 0) partials[tile] = v0;
  }
}

// Fallback for matrices with a 256-row tile of more than 27*256 non-zeros:
// one thread per row, same per-row order, so the same bits.
template <typename T, bool ZERO_Y, int MODE>
__global__ __launch_bounds__(kBlock) void spmv_rowwise_kernel(
    int n, const int* __restrict__ ro, const int* __restrict__ cols,
    const T* __restrict__ vals, const T* __restrict__ x, T* __restrict__ y,
    const T* __restrict__ bvec, T* __restrict__ partials, const int* __restrict__ done) {
  if (done && *done) return;
  __shared__ T red[4];
  const int row = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  T sum = T(0);
  if (row < n) {
    if (ZERO_Y) sum = T(0) * y[row];
    for (int j = ro[row]; j < ro[row + 1]; ++j) sum += vals[j] * x[cols[j]];
    if (MODE == kResid) sum = T(1) * bvec[row] + T(-1) * sum;
    y[row] = sum;
  }
  if (MODE != kPlain) {
    const T term = row < n ? (MODE == kDot ? sum * x[row] : sum * sum) : T(0);
    const T v0 = block_sum<T>(term, red);
    if (threadIdx.x == 0) partials[blockIdx.x] = v0;
  }
}

// ------------------------------------------------------------ SELL-64 -------
//
// Slice s holds rows 64s..64s+63 (one per lane) with width w_s = its longest
// row, in the slot-pair layout of mfe_sell.hpp: coalesced 16-byte value and
// 8-byte column loads, no LDS, and on a stencil matrix the x gathers of one
// slot hit consecutive addresses.  Rows are summed in stored column order:
// the same bits as the CSR kernels.  Four slices per workgroup, so the
// partials match the CSR kernel's (one per 256 rows).

constexpr int kSlice = kWave;
constexpr int kSlicesPerBlock = kBlock / kSlice;

template <typename T, bool ZERO_Y, int MODE>
__global__ __launch_bounds__(kBlock) void spmv_sell_kernel(
    int n, int nslices, const int* __restrict__ soff, const unsigned char* __restrict__ slen,
    const int* __restrict__ cols, const T* __restrict__ vals, const T* __restrict__ x,
    T* __restrict__ y, const T* __restrict__ bvec, T* __restrict__ partials,
    const int* __restrict__ done) {
  if (done && *done) return;
  __shared__ T red[4];
  const int t = (int)threadIdx.x;
  const int slice = (int)blockIdx.x * kSlicesPerBlock + t / kSlice;
  const int row = slice * kSlice + t % kSlice;
  bool valid = false;
  T sum = T(0), xr = T(0);
  if (slice < nslices) {  // uniform per wave
    valid = row < n;
    const int rr = valid ? row : n - 1;
    const T y0 = ZERO_Y ? y[rr] : T(0);
    if (MODE == kDot) xr = x[rr];
    const T br = MODE == kResid ? bvec[rr] : T(0);
    const int o = soff[slice];
    const int w = soff[slice + 1] - o;
    const int len = slen[row];
    if (ZERO_Y) sum = T(0) * y0;
    sum = sell_row_sum<T>(cols, vals, x, (int64_t)o * kSlice, w, t % kSlice, len, sum);
    if (MODE == kResid) sum = T(1) * br + T(-1) * sum;
    if (valid) y[row] = sum;
  }
  if (MODE != kPlain) {
    const T term = valid ? (MODE == kDot ? sum * xr : sum * sum) : T(0);
    const T v0 = block_sum<T>(term, red);
    if (t == 0) partials[blockIdx.x] = v0;
  }
}

// Row lengths (clamped to 255) and slice widths.
__global__ __launch_bounds__(kBlock) void sell_len_kernel(int n, int nslices,
                                                          const int* __restrict__ ro,
                                                          unsigned char* __restrict__ slen,
                                                          int* __restrict__ width) {
  const int row = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const int slice = row / kSlice;
  if (slice >= nslices) return;  // whole waves
  const int len = row < n ? ro[row + 1] - ro[row] : 0;
  slen[row] = (unsigned char)(len < 255 ? len : 255);
  int m = len;
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) m = max(m, __shfl_xor(m, off, kWave));
  if (row % kSlice == 0) width[slice] = m;
}

// Scatter the CSR rows into the slices, one workgroup (one wave) per slice:
// the slice's CSR columns or values (S = int or double; at most 27 per row,
// contiguous) are read into LDS with coalesced loads first -- a row's entries
// are a whole row apart from the next lane's, so direct per-thread reads touch
// 64 cache lines per instruction -- then each lane writes its row's slots.
// D = int (columns), double or float (values, rounded).  Padding: value 0,
// column = the row itself (rows past n use n-1), so every gather stays in
// bounds.
template <typename S, typename D>
__global__ __launch_bounds__(kSlice) void sell_fill_kernel(
    int n, int nslices, const int* __restrict__ soff, const unsigned char* __restrict__ slen,
    const int* __restrict__ ro, const S* __restrict__ src, D* __restrict__ dst, bool columns) {
  __shared__ S ss[kSellMaxWidth * kSlice];
  const int slice = (int)blockIdx.x;
  if (slice >= nslices) return;
  const int lane = (int)threadIdx.x;
  const int r0 = slice * kSlice;
  const int rl = min(r0, n), rh = min(r0 + kSlice, n);
  const int s0 = ro[rl], cnt = ro[rh] - s0;
  for (int i = lane; i < cnt; i += kSlice) ss[i] = src[s0 + i];
  __syncthreads();
  const int row = r0 + lane;
  const int o = soff[slice], w = soff[slice + 1] - o;
  const int len = slen[row];
  const int start = row < n ? ro[row] - s0 : 0;
  const int pad = row < n ? row : n - 1;
  for (int j = 0; j < w; ++j) {
    const int64_t at = sell_pos((int64_t)o * kSlice, j, w, lane);
    const bool in = j < len;
    if (columns) dst[at] = in ? (D)ss[start + j] : (D)pad;
    else dst[at] = in ? (D)ss[start + j] : D(0);
  }
}

// ---------------------------------------------- SELL-64 with staged x -------
//
// Workgroup = 4 slices = a tile of 256 rows.  A plan lists each tile's
// distinct columns in increasing order, as runs of consecutive columns (first
// column, position in the list), and stores at every SELL slot the column's
// position in the tile's list as 16 bits; a slice whose slot-j positions are
// base_j + lane (the rows of one grid line) keeps only its 27 bases.  The SpMV
// copies the tile's runs of x into LDS (coalesced: a 256-row tile of the
// 27-point stencil has 9 runs, 2.3 K entries) while the slot loads (the HBM
// stream) are in flight, and after the barrier gathers x from LDS.  Index
// traffic drops from 4 bytes per slot to 2, or to none for slices with bases,
// and x comes from L2 once per tile instead of once per slot.  Sums are in
// stored column order: the other kernels' bits.

constexpr int kXCap = 8192;        // non-zeros per tile the plan kernel sorts in LDS
constexpr int kXMaxRuns = 128;     // runs per tile the SpMV keeps in LDS
constexpr int kXLdsBytes = 56 * 1024;  // staged x per tile (27 * 256 doubles fit)
constexpr int kXFirst = 10;  // x entries per thread requested before the slot loads
                             // (2560 per tile: a 27-point tile needs 9 * 258)
constexpr int kXTail = 2048;  // zero local columns after the last slot: the clamped
                              // loads' tail, and what slices with bases load instead

// Exclusive workgroup scan of two counts; totals in ta, tb.
__device__ __forceinline__ int2 block_scan2(int a, int b, int* sa, int* sb, int& ta, int& tb) {
  const int t = (int)threadIdx.x;
  sa[t] = a;
  sb[t] = b;
  __syncthreads();
  for (int off = 1; off < kBlock; off <<= 1) {
    const int va = t >= off ? sa[t - off] : 0, vb = t >= off ? sb[t - off] : 0;
    __syncthreads();
    sa[t] += va;
    sb[t] += vb;
    __syncthreads();
  }
  ta = sa[kBlock - 1];
  tb = sb[kBlock - 1];
  return make_int2(sa[t] - a, sb[t] - b);
}

// Column range (in columns) up to which a tile's distinct columns are found
// with a bitmap in LDS instead of a sort: 2^19 bits (64 KB, whose first 32 KB
// hold the sort's keys otherwise), enough for the tiles of a 400^3 mesh.
constexpr int kBmWords = 16384;
constexpr int64_t kBmRange = 32 * (int64_t)kBmWords;
static_assert(kBmWords >= kXCap, "the sort's keys live in the bitmap's storage");

// The slot loop of a plan's pass 1 (shared by both ways of listing the
// distinct columns): each lane's local column per slot, and per slice whether
// the slot's local columns are base_j + lane (saff, sbase).
template <typename Loc>
__device__ __forceinline__ void sellx_plan_slots(int n, int nslices, const int* __restrict__ ro,
                                                 const int* __restrict__ cols,
                                                 const int* __restrict__ soff,
                                                 const unsigned char* __restrict__ slen,
                                                 unsigned short* __restrict__ lcols,
                                                 unsigned char* __restrict__ saff,
                                                 unsigned short* __restrict__ sbase, Loc loc_of) {
  const int t = (int)threadIdx.x, tile = (int)blockIdx.x;
  const int slice = tile * kSlicesPerBlock + t / kSlice;
  if (slice >= nslices) return;
  const int row = tile * kSpmvRows + t;
  const int lane = t % kSlice;
  const int o = soff[slice], w = soff[slice + 1] - o;
  const int len = slen[row];
  const int start = row < n ? ro[row] : 0;
  bool affine = w > 0 && len == w;
  for (int j = 0; j < w; ++j) {  // w is uniform over the wave
    const int loc = j < len ? loc_of(cols[start + j]) : 0;
    lcols[sell_pos((int64_t)o * kSlice, j, w, lane)] = (unsigned short)loc;
    const int base = __shfl(loc, 0, kWave);
    affine = affine && loc == base + lane;
    if (lane == 0) sbase[(int64_t)slice * kSellBaseStride + j] = (unsigned short)base;
  }
  if (lane >= w && lane < kSellBaseStride) sbase[(int64_t)slice * kSellBaseStride + lane] = 0;
  const int all = __all(affine ? 1 : 0);
  if (lane == 0) saff[slice] = (unsigned char)(all ? 1 : 0);
}

// Bitmap path of sellx_plan_kernel (see there): bm = the first nw (<=
// kBmWords) words of LDS, bit c - cmin set for every column c of the tile.
// Thread t owns words [t * per, (t + 1) * per), per a multiple of 8 (the
// groups of gpre); words past nw read as 0.
__device__ void sellx_plan_bitmap(int n, int nslices, const int* __restrict__ ro,
                                  const int* __restrict__ cols, const int* __restrict__ soff,
                                  const unsigned char* __restrict__ slen, int pass,
                                  int2* __restrict__ counts, const int* __restrict__ roff,
                                  int* __restrict__ rcol, int* __restrict__ rpos,
                                  unsigned short* __restrict__ lcols,
                                  unsigned char* __restrict__ saff,
                                  unsigned short* __restrict__ sbase, unsigned* bm, int* gpre,
                                  int* sa, int* sb, int s0, int cnt, int cmin, int nw) {
  const int per = ((nw + kBlock - 1) / kBlock + 7) & ~7;
  const int t = (int)threadIdx.x, tile = (int)blockIdx.x;
  for (int i = t; i < nw; i += kBlock) bm[i] = 0u;
  __syncthreads();
  for (int i = t; i < cnt; i += kBlock) {
    const int d = cols[s0 + i] - cmin;
    atomicOr(&bm[d >> 5], 1u << (d & 31));
  }
  __syncthreads();
  const int w0 = t * per;
  auto word = [&](int w) { return w < nw ? bm[w] : 0u; };
  unsigned prev_msb = w0 > 0 ? word(w0 - 1) >> 31 : 0u;
  int nu = 0, nr = 0;
  for (int q = 0; q < per; ++q) {
    const unsigned wd = word(w0 + q);
    const unsigned st = wd & ~((wd << 1) | prev_msb);  // set bits whose predecessor is clear
    nu += __popc(wd);
    nr += __popc(st);
    prev_msb = wd >> 31;
  }
  int tu, tr;
  const int2 base = block_scan2(nu, nr, sa, sb, tu, tr);
  if (pass == 0) {
    if (t == 0) counts[tile] = make_int2(tu, tr);
    return;
  }
  // runs in increasing column order, and the set bits before each group of 8 words
  int u = base.x, r = base.y;
  const int rb = roff[tile];
  prev_msb = w0 > 0 ? word(w0 - 1) >> 31 : 0u;
  for (int q = 0; q < per; ++q) {
    if ((q & 7) == 0 && w0 + q < nw) gpre[(w0 + q) >> 3] = u;
    const unsigned wd = word(w0 + q);
    unsigned st = wd & ~((wd << 1) | prev_msb);
    while (st) {
      const int bit = __ffs(st) - 1;
      rcol[rb + r] = cmin + (w0 + q) * 32 + bit;
      rpos[rb + r] = u + __popc(wd & ((1u << bit) - 1u));
      ++r;
      st &= st - 1u;
    }
    u += __popc(wd);
    prev_msb = wd >> 31;
  }
  __syncthreads();
  sellx_plan_slots(n, nslices, ro, cols, soff, slen, lcols, saff, sbase, [&](int c) {
    const int d = c - cmin, wi = d >> 5;
    int p = gpre[wi >> 3];
    for (int k = wi & ~7; k < wi; ++k) p += __popc(bm[k]);
    return p + __popc(bm[wi] & ((1u << (d & 31)) - 1u));
  });
}

// One workgroup per tile.  The tile's distinct columns, in increasing order,
// come from a bitmap over [min column, max column] when that range is at most
// kBmRange (a mesh numbering's tiles span about two planes): each entry sets
// its column's bit, a set bit is a distinct column, a set bit after a clear one
// starts a run, and a column's position in the list is the number of set bits
// before it.  Wider tiles sort their columns in LDS (bitonic); a value is
// distinct where it differs from its predecessor and starts a run where the
// predecessor is not value - 1.  Both give the same lists.  Pass 0:
// counts[tile] = {distinct, runs}, or {-1, -1} past kXCap non-zeros.  Pass 1: the runs at roff[tile], the local
// columns at every slot of the tile's slices (padding slots: 0), and per slice
// (one wave) whether every row has the slice's width w > 0 and slot j's local
// column is base_j + lane for every j (saff = 1, bases in sbase; 0 past w).
__global__ __launch_bounds__(kBlock) void sellx_plan_kernel(
    int n, int nslices, const int* __restrict__ ro, const int* __restrict__ cols,
    const int* __restrict__ soff, const unsigned char* __restrict__ slen, int pass,
    int2* __restrict__ counts, const int* __restrict__ roff, int* __restrict__ rcol,
    int* __restrict__ rpos, unsigned short* __restrict__ lcols, unsigned char* __restrict__ saff,
    unsigned short* __restrict__ sbase) {
  __shared__ unsigned bmw[kBmWords];  // the bitmap, or (first kXCap) the sort's keys
  int* const a = reinterpret_cast<int*>(bmw);
  __shared__ int sa[kBlock], sb[kBlock];
  __shared__ int gpre[kBmWords / 8];  // bitmap path: set bits before each group of 8 words
  constexpr int kPer = kXCap / kBlock;
  const int t = (int)threadIdx.x, tile = (int)blockIdx.x;
  const int r0 = tile * kSpmvRows, r1 = min(r0 + kSpmvRows, n);
  const int s0 = ro[r0], cnt = ro[r1] - s0;
  if (cnt > kXCap) {
    if (pass == 0 && t == 0) counts[tile] = make_int2(-1, -1);
    return;
  }
  // the tile's column range
  int cmin = INT_MAX, cmax = -1;
  for (int i = t; i < cnt; i += kBlock) {
    const int c = cols[s0 + i];
    cmin = min(cmin, c);
    cmax = max(cmax, c);
  }
  sa[t] = cmin;
  sb[t] = cmax;
  __syncthreads();
  for (int off = kBlock / 2; off > 0; off >>= 1) {
    if (t < off) {
      sa[t] = min(sa[t], sa[t + off]);
      sb[t] = max(sb[t], sb[t + off]);
    }
    __syncthreads();
  }
  cmin = sa[0];
  cmax = sb[0];
  __syncthreads();
  if (cnt == 0 || (int64_t)cmax - cmin + 1 <= kBmRange) {
    sellx_plan_bitmap(n, nslices, ro, cols, soff, slen, pass, counts, roff, rcol, rpos, lcols,
                      saff, sbase, bmw, gpre, sa, sb, s0, cnt, cnt == 0 ? 0 : cmin,
                      cnt == 0 ? 0 : (int)(((int64_t)cmax - cmin + 32) >> 5));
    return;
  }
  for (int i = t; i < kXCap; i += kBlock) a[i] = i < cnt ? cols[s0 + i] : INT_MAX;
  __syncthreads();
  for (int k = 2; k <= kXCap; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = t; i < kXCap; i += kBlock) {
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
  int v[kPer];
  unsigned distinct = 0, starts = 0;
  int nu = 0, nr = 0;
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int i = kPer * t + q;
    v[q] = a[i];
    const int prev = i > 0 ? a[i - 1] : INT_MIN;
    const bool d = v[q] != INT_MAX && v[q] != prev;
    const bool r = d && (i == 0 || prev != v[q] - 1);
    distinct |= (unsigned)d << q;
    starts |= (unsigned)r << q;
    nu += d;
    nr += r;
  }
  int tu, tr;
  const int2 base = block_scan2(nu, nr, sa, sb, tu, tr);
  if (pass == 0) {
    if (t == 0) counts[tile] = make_int2(tu, tr);
    return;
  }
  __syncthreads();  // every thread holds its entries: compact the list in place
  int u = base.x, r = base.y;
  const int rb = roff[tile];
#pragma unroll
  for (int q = 0; q < kPer; ++q)
    if ((distinct >> q) & 1) {
      if ((starts >> q) & 1) {
        rcol[rb + r] = v[q];
        rpos[rb + r] = u;
        ++r;
      }
      a[u] = v[q];
      ++u;
    }
  __syncthreads();
  sellx_plan_slots(n, nslices, ro, cols, soff, slen, lcols, saff, sbase, [&](int c) {
    int lo = 0, hi = tu;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (a[mid] < c) lo = mid + 1;
      else hi = mid;
    }
    return lo;
  });
}

// spmv_sell_kernel's modes and results, x staged per tile (dynamic LDS:
// max(A->sellx_maxu, 64) entries of T).  A slice with bases (saff) reads its
// local columns as base_j + lane; its column loads go to the zero tail ltail
// (one cached region) so that every wave issues the same loads.  Order of
// work: the tile's run list goes to LDS; the thread's first kXFirst x entries
// are requested, then the lane's slot loads (memory returns loads in issue
// order, so the x entries can be written to LDS while the slot loads are
// still in flight); remaining x entries, if any, follow; after the barrier
// the slots are unpacked and summed.  Every local column in the array is
// below A->sellx_maxu, and a base + lane below max(A->sellx_maxu, 64), so the
// LDS reads of padding and of clamped loads stay inside the allocation.
template <typename T, bool ZERO_Y, int MODE>
__global__ __launch_bounds__(kBlock) void spmv_sellx_kernel(
    int n, int nslices, const int* __restrict__ soff, const unsigned char* __restrict__ slen,
    const unsigned short* __restrict__ lcols, const unsigned short* __restrict__ ltail,
    const unsigned char* __restrict__ saff, const unsigned short* __restrict__ sbase,
    const T* __restrict__ vals, const int* __restrict__ roff, const int* __restrict__ rcol,
    const int* __restrict__ rpos, const int* __restrict__ tnu, const T* __restrict__ x,
    T* __restrict__ y, const T* __restrict__ bvec, T* __restrict__ partials,
    const int* __restrict__ done) {
  if (done && *done) return;
  constexpr int CH = sizeof(T) == 8 ? 8 : 4;  // x loads in flight per thread while staging
  extern __shared__ __align__(16) unsigned char sx_bytes[];
  T* sx = reinterpret_cast<T*>(sx_bytes);
  __shared__ int run_col[kXMaxRuns], run_pos[kXMaxRuns + 1];
  __shared__ T red[4];
  const int t = (int)threadIdx.x, tile = (int)blockIdx.x;
  const int ra = roff[tile], nr = roff[tile + 1] - ra, nu = tnu[tile];
  const bool has_run = t < nr;
  const int my_col = has_run ? rcol[ra + t] : 0;
  const int my_pos = has_run ? rpos[ra + t] : 0;
  const int slice = tile * kSlicesPerBlock + t / kSlice;
  const int lane = t % kSlice;
  const int row = slice * kSlice + lane;
  const bool live = slice < nslices;  // uniform per wave
  const bool valid = live && row < n;
  const int rr = valid ? row : n - 1;
  const int sl = live ? slice : nslices - 1;
  const T y0 = ZERO_Y ? y[rr] : T(0);
  const T xr = MODE == kDot ? x[rr] : T(0);
  const T br = MODE == kResid ? bvec[rr] : T(0);
  const int o = soff[sl];
  const int w = live ? soff[sl + 1] - o : 0;
  const int len = live ? (int)slen[row] : 0;
  // per-wave values: the slice's flag and its 32 bases (64 bytes) are read
  // before the barrier, from a uniform address
  const int sl_u = __builtin_amdgcn_readfirstlane(sl);
  const bool aff = live && saff[sl_u];
  const uint4* sb4 = reinterpret_cast<const uint4*>(sbase + (int64_t)sl_u * kSellBaseStride);
  const uint4 q0 = sb4[0], q1 = sb4[1], q2 = sb4[2], q3 = sb4[3];
  const unsigned bw[16] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w,
                           q2.x, q2.y, q2.z, q2.w, q3.x, q3.y, q3.z, q3.w};
  if (has_run) {
    run_col[t] = my_col;
    run_pos[t] = my_pos;
  }
  if (t == 0) run_pos[nr] = nu;
  __syncthreads();
  int r = 0;  // run of entry i; i grows, so the run only moves forward
  T xf[kXFirst];
  {
    int g[kXFirst];
#pragma unroll
    for (int k = 0; k < kXFirst; ++k) {
      const int i = t + k * kBlock;
      while (r + 1 < nr && run_pos[r + 1] <= i) ++r;
      g[k] = i < nu ? run_col[r] + (i - run_pos[r]) : 0;
    }
#pragma unroll
    for (int k = 0; k < kXFirst; ++k) xf[k] = x[g[k]];
  }
  SellLocalRaw<T> raw;
  sell_load_local<T>(aff ? ltail : lcols, aff ? 0 : (int64_t)o * kSlice, vals,
                     (int64_t)o * kSlice, w, lane, raw);
#pragma unroll
  for (int k = 0; k < kXFirst; ++k)
    if (t + k * kBlock < nu) sx[t + k * kBlock] = xf[k];
  for (int i0 = t + kXFirst * kBlock; i0 < nu; i0 += kBlock * CH) {
    int g[CH];
#pragma unroll
    for (int k = 0; k < CH; ++k) {
      const int i = i0 + k * kBlock;
      while (r + 1 < nr && run_pos[r + 1] <= i) ++r;
      g[k] = i < nu ? run_col[r] + (i - run_pos[r]) : 0;
    }
    T xv[CH];
#pragma unroll
    for (int k = 0; k < CH; ++k) xv[k] = x[g[k]];
#pragma unroll
    for (int k = 0; k < CH; ++k)
      if (i0 + k * kBlock < nu) sx[i0 + k * kBlock] = xv[k];
  }
  __syncthreads();
  T sum = T(0);
  if (live) {
    if (ZERO_Y) sum = T(0) * y0;
    int c[kSellMaxWidth];
    T v[kSellMaxWidth], xv[kSellMaxWidth];
#pragma unroll
    for (int j = 0; j < kSellMaxWidth; ++j) {
      sell_slot<T>(raw, j, c[j], v[j]);
      if (aff) c[j] = (int)((bw[j >> 1] >> ((j & 1) * 16)) & 0xffffu) + lane;
    }
#pragma unroll
    for (int j = 0; j < kSellMaxWidth; ++j) xv[j] = sx[c[j]];
#pragma unroll
    for (int j = 0; j < kSellMaxWidth; ++j)
      if (j < len) sum += v[j] * xv[j];
    if (MODE == kResid) sum = T(1) * br + T(-1) * sum;
    if (valid) y[row] = sum;
  }
  if (MODE != kPlain) {
    const T term = valid ? (MODE == kDot ? sum * xr : sum * sum) : T(0);
    const T v0 = block_sum<T>(term, red);
    if (t == 0) partials[blockIdx.x] = v0;
  }
}

static void sellx_release(mfe_csr* A) {
  csr_free(A, A->sellx_lcols);
  csr_free(A, A->sellx_roff);
  csr_free(A, A->sellx_rcol);
  csr_free(A, A->sellx_rpos);
  csr_free(A, A->sellx_nu);
  csr_free(A, A->sellx_aff);
  csr_free(A, A->sellx_sbase);
  A->sellx_lcols = nullptr;
  A->sellx_roff = A->sellx_rcol = A->sellx_rpos = A->sellx_nu = nullptr;
  A->sellx_aff = nullptr;
  A->sellx_sbase = nullptr;
  A->sellx_valid = A->sellx_ok = false;
  A->sellx_maxu = 0;
  A->sellx_ntiles = A->sellx_runs = A->sellx_affine = A->sellx_explicit = 0;
}

void sell_release(mfe_csr* A) {
  A->plan_gen = next_plan_gen();
  sellx_release(A);
  csr_free(A, A->sell_off);
  csr_free(A, A->sell_len);
  csr_free(A, A->sell_cols);
  csr_free(A, A->sell_vals);
  csr_free(A, A->sell_vals32);
  csr_free(A, A->sell_lines);
  A->sell_lines = nullptr;
  A->sell_lines_valid = false;
  A->sell_off = nullptr;
  A->sell_len = nullptr;
  A->sell_cols = nullptr;
  A->sell_vals = nullptr;
  A->sell_vals32 = nullptr;
  A->sell_struct_valid = A->sell_ok = false;
  A->sell_vals_valid = A->sell_vals32_valid = false;
  A->sell_nslices = A->sell_slots = 0;
  A->sell_max_len = 0;
}

// The structure was examined and SELL does not apply (a long row, or no
// memory for the copy): free the copy, keep the longest-row figure.
static void sell_disable(mfe_csr* A) {
  const int maxw = A->sell_max_len;
  sell_release(A);
  A->sell_struct_valid = true;
  A->sell_max_len = maxw;
}

// False (and a null pointer) when memory is short: the plan then falls back to
// another format.
template <typename P>
static bool try_alloc(mfe_ctx* ctx, P** p, size_t bytes) {
  return dev_alloc(ctx, p, bytes) == hipSuccess;
}

// The staged-x plan of A's SELL structure (synchronises the stream).  Leaves
// sellx_ok false, and the plain SELL kernel in use, when a tile has more than
// kXMaxRuns runs or kXCap non-zeros, or the arrays do not fit in memory.
static int build_sellx(mfe_ctx* ctx, mfe_csr* A) {
  sellx_release(A);
  A->sellx_valid = true;
  const int64_t n = A->nrows;
  if (!A->sell_ok || n == 0) return MFE_OK;
  hipStream_t s = ctx->stream;
  const int nt = (int)cdiv(n, kSpmvRows);
  const int ns = (int)A->sell_nslices;
  int2* d_counts = nullptr;
  if (!try_alloc(ctx, &d_counts, sizeof(int2) * (size_t)nt)) return MFE_OK;
  sellx_plan_kernel<<<nt, kBlock, 0, s>>>((int)n, ns, A->row_offsets, A->cols, A->sell_off,
                                           A->sell_len, 0, d_counts, nullptr, nullptr, nullptr,
                                           nullptr, nullptr, nullptr);
  std::vector<int2> counts((size_t)nt);
  hipError_t e = hipGetLastError();
  int dst = e == hipSuccess ? download_bytes(ctx, counts.data(), d_counts, sizeof(int2) * (size_t)nt)
                            : MFE_OK;
  dev_free(ctx, d_counts);
  if (e != hipSuccess) return hip_fail(ctx, e, "sellx_plan_kernel count");
  if (dst) return dst;
  std::vector<int> roff((size_t)nt + 1), nu((size_t)nt);
  int64_t runs = 0;
  int maxu = 0;
  for (int i = 0; i < nt; ++i) {
    const int2 c = counts[(size_t)i];
    if (c.x < 0 || c.y > kXMaxRuns) return MFE_OK;
    roff[(size_t)i] = (int)runs;
    runs += c.y;
    nu[(size_t)i] = c.x;
    maxu = std::max(maxu, c.x);
  }
  roff[(size_t)nt] = (int)runs;
  if ((int64_t)maxu * (int64_t)sizeof(double) > kXLdsBytes || runs >= INT32_MAX) return MFE_OK;
  const size_t nl = (size_t)(A->sell_slots + kXTail);
  const bool ok = try_alloc(ctx, &A->sellx_lcols, sizeof(unsigned short) * nl) &&
                  try_alloc(ctx, &A->sellx_roff, sizeof(int) * ((size_t)nt + 1)) &&
                  try_alloc(ctx, &A->sellx_rcol, sizeof(int) * (size_t)std::max<int64_t>(runs, 1)) &&
                  try_alloc(ctx, &A->sellx_rpos, sizeof(int) * (size_t)std::max<int64_t>(runs, 1)) &&
                  try_alloc(ctx, &A->sellx_nu, sizeof(int) * (size_t)nt) &&
                  try_alloc(ctx, &A->sellx_aff, (size_t)ns) &&
                  try_alloc(ctx, &A->sellx_sbase, sizeof(unsigned short) * kSellBaseStride * (size_t)ns);
  if (!ok) {
    sellx_release(A);
    A->sellx_valid = true;
    return MFE_OK;
  }
  MFE_CHECK(ctx, hipMemsetAsync(A->sellx_lcols + A->sell_slots, 0,
                                sizeof(unsigned short) * kXTail, s));
  int ust;
  if ((ust = upload_bytes(ctx, A->sellx_roff, roff.data(), sizeof(int) * roff.size())) ||
      (ust = upload_bytes(ctx, A->sellx_nu, nu.data(), sizeof(int) * nu.size())))
    return ust;
  sellx_plan_kernel<<<nt, kBlock, 0, s>>>((int)n, ns, A->row_offsets, A->cols, A->sell_off,
                                           A->sell_len, 1, nullptr, A->sellx_roff, A->sellx_rcol,
                                           A->sellx_rpos, A->sellx_lcols, A->sellx_aff,
                                           A->sellx_sbase);
  MFE_LAUNCHED(ctx, "sellx_plan_kernel fill");
  // slices with bases, and the stored entries of the others (plan figures)
  std::vector<unsigned char> aff((size_t)ns);
  std::vector<int> soff((size_t)ns + 1);
  {
    int dst;
    if ((dst = download_bytes(ctx, aff.data(), A->sellx_aff, (size_t)ns)) ||
        (dst = download_bytes(ctx, soff.data(), A->sell_off, sizeof(int) * soff.size())))
      return dst;
  }
  int64_t naff = 0, nexp = 0;
  for (int i = 0; i < ns; ++i) {
    if (aff[(size_t)i]) ++naff;
    else nexp += (int64_t)(soff[(size_t)i + 1] - soff[(size_t)i]) * kSlice;
  }
  A->sellx_affine = naff;
  A->sellx_explicit = nexp;
  A->sellx_ok = true;
  A->sellx_maxu = maxu;
  A->sellx_ntiles = nt;
  A->sellx_runs = runs;
  return MFE_OK;
}

// CSR FP32 copy of the values (round to nearest).
__global__ void vals_to_f32_kernel(int64_t nnz, const double* __restrict__ v,
                                   float* __restrict__ v32) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nnz; i += stride)
    v32[i] = (float)v[i];
}

// Builds what the next SpMV launches need: the SELL structure, and its FP64
// and/or FP32 values; the CSR FP32 copy instead when SELL does not apply.
// Synchronises the stream (host-side scan of the slice widths); never called
// during graph capture.
// ---- box layout plan ---------------------------------------------------------

void box_release(mfe_csr* A) {
  csr_free(A, A->box_vals);
  csr_free(A, A->box_vals32);
  csr_free(A, A->boxsym_u);
  csr_free(A, A->boxsym_w);
  csr_free(A, A->boxsym_u32);
  csr_free(A, A->boxsym_w32);
  csr_free(A, A->boxsym_tab);
  csr_free(A, A->boxpack_pw);
  csr_free(A, A->boxpack_kq);
  csr_free(A, A->boxpack32_pw);
  csr_free(A, A->boxpack32_kq);
  csr_free(A, A->boxwpack_pw);
  csr_free(A, A->boxwpack_kq);
  A->box_vals = nullptr;
  A->box_vals32 = nullptr;
  A->boxsym_u = A->boxsym_w = nullptr;
  A->boxsym_u32 = A->boxsym_w32 = nullptr;
  A->boxsym_tab = nullptr;
  A->boxpack_pw = A->boxpack32_pw = nullptr;
  A->boxpack_kq = nullptr;
  A->boxpack32_kq = nullptr;
  A->boxwpack_pw = nullptr;
  A->boxwpack_kq = nullptr;
  A->boxwpack_form = kPackNone;
  A->boxpack_cap = A->boxpack32_cap = 0;
  A->box_vals_valid = A->box_vals32_valid = false;
  A->boxsym_state = 0;
  A->boxsym_valid = A->boxsym32_valid = false;
  A->boxpack_valid = A->boxpack32_valid = false;
  A->boxpack_form = A->boxpack32_form = kPackNone;
  A->box_geom = BoxGeom{};
}

// In-range stencil slots of node (ix, iy, iz) as a 27-bit mask (bit s set:
// neighbour s exists); the rank of slot s among them is its position in the
// row's stored entries.
__host__ __device__ inline unsigned box_mask(int ix, int iy, int iz, int gx, int gy, int gz) {
  unsigned m = 0;
  for (int sz = -1; sz <= 1; ++sz)
    for (int sy = -1; sy <= 1; ++sy)
      for (int sx = -1; sx <= 1; ++sx) {
        const int x = ix + sx, yy = iy + sy, zz = iz + sz;
        if (x >= 0 && x < gx && yy >= 0 && yy < gy && zz >= 0 && zz < gz)
          m |= 1u << ((sz + 1) * 9 + (sy + 1) * 3 + (sx + 1));
      }
  return m;
}
__device__ inline int slot_rank(unsigned mask, int s) { return __popc(mask & ((1u << s) - 1u)); }

// The tables of the symmetric layout: entry e = pair (t, s) of a block row t
// and a lower slot s whose neighbour is outside the 16 x 16 block, in (t, s)
// order; tab[e] = where the kernel writes its value (reading row t and the
// neighbour's mirrored slot) and its place in the packed boundary stream
// (sym_wcode), tab[kSymNB + t * 13 + s] = e or -1, and from kSymWListAt the
// entries of each lower slot s (kSymWListLen per slot, -1 after the last).
constexpr int kSymWListLen = 32;
constexpr int kSymWListAt = kSymNB + kBlock * 13;
static void boxsym_tables(std::vector<int>& tab) {
  tab.assign(kSymWListAt + kSymWGroups * kSymWListLen, -1);
  int e = 0, nb = 0;
  int len[kSymWGroups] = {};
  for (int t = 0; t < kBlock; ++t) {
    const int tx = t % kBoxBX, ty = t / kBoxBX;
    for (int s = 0; s < 13; ++s) {
      const int sz = s / 9 - 1, sy = (s / 3) % 3 - 1, sx = s % 3 - 1;
      if (tx + sx >= 0 && tx + sx < kBoxBX && ty + sy >= 0 && ty + sy < kBoxBY) continue;
      const int near = (kSymWNear >> s) & 1u;
      tab[(size_t)e] = (sz < 0 ? sym_code(t, 26 - s - 18, 0) : sym_code(t, 26 - s - 14, 1)) |
                       sym_wcode(nb, near, s);
      tab[(size_t)kSymNB + (size_t)t * 13 + (size_t)s] = e;
      tab[(size_t)kSymWListAt + (size_t)s * kSymWListLen + (size_t)len[s]++] = e;
      nb += near;
      ++e;
    }
  }
  if (e != kSymNB || nb != kSymWNearCount) tab.clear();  // (the geometry fixes both)
}

// The layout's blocks of kBoxBX x kBoxBY nodes (z chunks are chosen per
// launch, box_chunks).
static BoxGeom box_geometry(const mfe_csr* A) {
  BoxGeom g{};
  g.gx = A->box_elems[0] + 1;
  g.gy = A->box_elems[1] + 1;
  g.gz = A->box_elems[2] + 1;
  g.nbx = (int)cdiv(g.gx, kBoxBX);
  g.nby = (int)cdiv(g.gy, kBoxBY);
  return g;
}

// Workgroups of `kernel` (kBlock threads) resident on the whole GPU.
int resident_groups(const void* kernel, int cus) {
  static std::mutex mu;
  static std::vector<std::pair<const void*, int>> cache;
  std::lock_guard<std::mutex> lock(mu);
  for (const auto& e : cache)
    if (e.first == kernel) return e.second * std::max(cus, 1);
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kBlock, 0) != hipSuccess ||
      per_cu < 1) {
    (void)hipGetLastError();
    per_cu = 1;
  }
  cache.emplace_back(kernel, per_cu);
  return per_cu * std::max(cus, 1);
}

// Z chunks of a box-layout launch: the workgroups (blocks x chunks) should
// fill whole rounds of the `resident` slots -- a last round that runs a few
// workgroups alone costs a whole chunk's time -- while each chunk's first
// plane costs about one and a half plane steps more; never more workgroups
// than `cap` (the partial buffers).  Sets g.zc, g.nzc.
void box_chunks(BoxGeom& g, int resident, int64_t cap) {
  const int64_t nb = (int64_t)g.nbx * g.nby;
  const int64_t maxc = std::max<int64_t>(1, std::min<int64_t>(g.gz, cap / std::max<int64_t>(nb, 1)));
  double best = -1;
  g.zc = g.gz;
  g.nzc = 1;
  for (int64_t c = 1; c <= maxc; ++c) {
    const int zc = (int)cdiv(g.gz, c);
    const int nzc = (int)cdiv(g.gz, zc);
    if (nzc != c) continue;  // each distinct chunking once
    const int64_t items = nb * nzc;
    const int64_t rounds = cdiv(items, std::max(resident, 1));
    const double util = (double)items / (double)(rounds * std::max(resident, 1));
    const double score = util / (1.0 + 1.5 * (double)nzc / (double)g.gz);
    if (score > best + 1e-12) {
      best = score;
      g.zc = zc;
      g.nzc = nzc;
    }
  }
}

// Workgroups per CU that the z chunks of a symmetric SpMV are sized for.  The
// chunks are also the groups of its dot's partials, so the figure belongs to the
// format (precision, packed form, packed boundary stream) and is not asked of the
// occupancy query, whose answer follows the compiler's register allocation and
// would move the sums with it (and which counts no scalar registers: with the
// plane record in about 100 of them a SIMD holds at most six waves).  They are the
// chunks that the sums had before the products were handed over, not the fastest
// ones: FP32 all12 at 200^3 takes 71.3 us in chunks for five per CU, 67.8 for six,
// 83.3 for seven, but with other groups a mixed solve to 1e-11 there ended 1.0e-9
// (two of its own runs: 4e-10) from the x it had given.  The figure of the packed
// boundary stream also holds below kWPackRows, where the boundary is read in full.
static int sym_slots(bool f64, int pack, bool wpack, int cus) {
  const bool wide = pack == kPackAll16 || pack == kPackCube16Near32 || pack == kPackCube16;
  int per = f64 ? (wpack && wide ? 3 : 4)
          : pack == kPackNone || pack == kPackCube16 ? 7
          : pack == kPackAll16 || pack == kPackAll10 ? 6 : 5;
  return per * std::max(cus, 1);
}

static bool box_applies(const mfe_csr* A) {
  return A->spmv_format == MFE_SPMV_AUTO && A->box_elems[0] > 0 && A->nrows > 0 &&
         (int64_t)(A->box_elems[0] + 1) * (A->box_elems[1] + 1) * (A->box_elems[2] + 1) ==
             A->nrows;
}

// One workgroup per (block, plane): thread t's node takes its CSR row's
// entries, in order, into its in-range slots, and 0 into the others (also
// for threads past the box's edge), so every entry of V is written.  The
// block's rows of values (at most 27 x 256 entries, in row runs along x)
// are read from the CSR arrays into LDS with coalesced loads first.
template <typename Tout>
__global__ __launch_bounds__(kBlock) void box_fill_kernel(BoxGeom g, const int* __restrict__ ro,
                                                          const double* __restrict__ vals,
                                                          Tout* __restrict__ V) {
  const int blk = (int)(blockIdx.x / (unsigned)g.gz), z = (int)(blockIdx.x % (unsigned)g.gz);
  const int bx = blk % g.nbx, by = blk / g.nbx;
  const int t = (int)threadIdx.x, tx = t % kBoxBX, ty = t / kBoxBX;
  const int ix = bx * kBoxBX + tx, iy = by * kBoxBY + ty;
  const bool live = ix < g.gx && iy < g.gy;
  const int64_t row = ((int64_t)z * g.gy + iy) * g.gx + ix;
  const int lox = ix > 0 ? -1 : 0, hix = ix < g.gx - 1 ? 1 : 0;
  const int loy = iy > 0 ? -1 : 0, hiy = iy < g.gy - 1 ? 1 : 0;
  const int loz = z > 0 ? -1 : 0, hiz = z < g.gz - 1 ? 1 : 0;
  int k = live ? ro[row] : 0;
#pragma unroll
  for (int sz = -1; sz <= 1; ++sz)
#pragma unroll
    for (int sy = -1; sy <= 1; ++sy)
#pragma unroll
      for (int sx = -1; sx <= 1; ++sx) {
        const int sl = (sz + 1) * 9 + (sy + 1) * 3 + (sx + 1);
        const bool in = live && sx >= lox && sx <= hix && sy >= loy && sy <= hiy && sz >= loz &&
                        sz <= hiz;
        V[box_at(g, blk, z, sl, t)] = in ? (Tout)vals[k] : Tout(0);
        k += in ? 1 : 0;
      }
}

// Sets A->box_geom for A's current box, freeing the layouts (and forgetting
// the symmetry check) when it changes.  Every builder below relies on it.
static void box_set_geometry(mfe_csr* A) {
  const BoxGeom g = box_geometry(A);
  const bool same = A->box_geom.gx == g.gx && A->box_geom.gy == g.gy && A->box_geom.gz == g.gz;
  if (!same) {
    box_release(A);
    A->box_geom = g;
  }
}

// The box layout of A's values as T (synchronises nothing; on the stream).
// Returns MFE_OK with the layout absent when it does not fit in memory.
template <typename T>
static int build_box(mfe_ctx* ctx, mfe_csr* A) {
  const BoxGeom g = A->box_geom;
  T** dst;
  if constexpr (std::is_same<T, double>::value) dst = &A->box_vals;
  else dst = &A->box_vals32;
  if (!*dst && !try_alloc(ctx, dst, sizeof(T) * (size_t)box_entries(g))) return MFE_OK;
  box_fill_kernel<T><<<(unsigned)((int64_t)g.nbx * g.nby * g.gz), kBlock, 0, ctx->stream>>>(
      g, A->row_offsets, A->vals, *dst);
  MFE_LAUNCHED(ctx, "box_fill_kernel");
  if constexpr (std::is_same<T, double>::value) A->box_vals_valid = true;
  else A->box_vals32_valid = true;
  return MFE_OK;
}

// The packed form of a box layout's values (mfe_pack.hpp; SymPack: the
// symmetric layout's upper slots).  The layout's build finds per (block,
// plane, slot) group the least exponent qe of any value's lowest set bit
// (values other than +0.0 and 1.0; -0.0, infinities and NaNs make the slot
// unpackable in that group) and the least and greatest k = v / 2^qe.  The
// slot fits W bits in the group when every |k| < 2^53 (FP32: 2^24) and they
// span at most 2^W - 3 (W of kPackWidths; 32 for FP64 only).
template <typename T>
struct PackBits;
template <>
struct PackBits<double> {
  static constexpr double kLimit = 9007199254740992.0;  // 2^53
  static constexpr int kLeast = -1022;  // a q below the least normal number is not packed
  // exponent of the lowest set bit; INT_MAX for +0.0 and 1.0; INT_MIN if unpackable
  __device__ static int lowbit(double v) {
    const long long b = __double_as_longlong(v);
    if (b == 0 || v == 1.0) return INT_MAX;
    const int e = (int)((b >> 52) & 0x7FF);
    const long long m = b & 0xFFFFFFFFFFFFFLL;
    if (e == 0x7FF || (e == 0 && m == 0)) return INT_MIN;
    return e == 0 ? -1074 + __builtin_ctzll(m) : (e - 1075) + __builtin_ctzll(m | (1LL << 52));
  }
  __device__ static double pow2(int e) { return ldexp(1.0, e); }
  __device__ static bool same(double a, double b) {
    return __double_as_longlong(a) == __double_as_longlong(b);
  }
};
template <>
struct PackBits<float> {
  static constexpr float kLimit = 16777216.0f;  // 2^24
  static constexpr int kLeast = -126;
  __device__ static int lowbit(float v) {
    const int b = __float_as_int(v);
    if (b == 0 || v == 1.0f) return INT_MAX;
    const int e = (b >> 23) & 0xFF;
    const int m = b & 0x7FFFFF;
    if (e == 0xFF || (e == 0 && m == 0)) return INT_MIN;
    return e == 0 ? -149 + __builtin_ctz(m) : (e - 150) + __builtin_ctz(m | (1 << 23));
  }
  __device__ static float pow2(int e) { return ldexpf(1.0f, e); }
  __device__ static bool same(float a, float b) { return __float_as_int(a) == __float_as_int(b); }
};

// Least lowest-set-bit exponent and range of a group's values (+0.0 and 1.0
// apart; -0.0, infinities and NaNs set bad), 16 lanes per group.
template <typename T>
struct PackRange {
  using B = PackBits<T>;
  int lb = INT_MAX, bad = 0;
  T lo = T(0), hi = T(0);  // of the values seen so far (lb != INT_MAX)
  __device__ void add(T v) {
    const int l = B::lowbit(v);
    if (l == INT_MAX) return;
    if (l == INT_MIN) {
      bad = 1;
      return;
    }
    lo = lb == INT_MAX || v < lo ? v : lo;
    hi = lb == INT_MAX || v > hi ? v : hi;
    lb = min(lb, l);
  }
  __device__ void join16() {
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) {
      const int l = __shfl_xor(lb, off, kWave);
      const T ol = __shfl_xor(lo, off, kWave), oh = __shfl_xor(hi, off, kWave);
      bad |= __shfl_xor(bad, off, kWave);
      if (l == INT_MAX) continue;
      lo = lb == INT_MAX || ol < lo ? ol : lo;
      hi = lb == INT_MAX || oh > hi ? oh : hi;
      lb = min(lb, l);
    }
  }
  // The group's power of two and greatest multiple, and the widths of
  // kPackWidths (bit i) that hold it.  A multiple v / q is exact, and the
  // least and greatest one are those of the least and greatest value.
  __device__ unsigned widths(T& kmax, T& qv) const {
    bool ok = !bad;
    T kmin = T(0);
    kmax = T(0);
    qv = T(1);
    if (ok && lb != INT_MAX) {
      qv = B::pow2(lb);
      kmin = lo / qv;
      kmax = hi / qv;
      ok = lb >= B::kLeast && fabs(kmin) < B::kLimit && fabs(kmax) < B::kLimit;
    }
    const T span = kmax - kmin;  // exact: both are integers below the limit
    unsigned m = 0;
#pragma unroll
    for (int i = 0; i < kPackNumWidths; ++i) {
      const int w = kPackWidths[i];
      const bool allowed = sizeof(T) == 8 || w <= 24;
      if (ok && allowed && span <= T((double)((1ull << w) - 3ull))) m |= 1u << i;
    }
    return m;
  }
};

// Device words of a plan build (PlanWords at d_scalars + kPlanWordsAt).
struct PlanWords {
  unsigned asym;                     // 1: a mirrored pair differs
  unsigned pack_bad, wpack_bad;      // 1: a packed value does not decode to itself
  unsigned pad;
  unsigned fits[kPackNumWidths];     // per width of kPackWidths: the slots every group fits
  unsigned wfits[kPackNumWidths];    // the boundary stream's lower slots
};
constexpr int kPlanWordsAt = 16;
static_assert(sizeof(PlanWords) <= 32 * sizeof(double), "d_scalars holds 64 doubles");

__global__ void plan_words_kernel(PlanWords* w) {
  const int i = (int)threadIdx.x;
  if (i == 0) w->asym = w->pack_bad = w->wpack_bad = w->pad = 0u;
  if (i < kPackNumWidths) w->fits[i] = w->wfits[i] = ~0u;
}

// The symmetric layout of A's values and, in the same pass, what its packed
// form and its symmetry check need.  A workgroup owns one 16 x 16 block and a
// range of planes (g.zc); per plane thread t's node writes its 14 upper slots
// to U and its lower slots whose neighbour lies outside the block to W (entry
// inv[t * 13 + s]), 0 where the slot is out of range or the node past the
// box's edge, so every entry is written.
//   The block-plane's CSR rows are staged in LDS (16 lanes per grid line, whose
// rows' values are one contiguous run: coalesced loads instead of one
// 216-byte-strided row per thread), the next plane's loads in flight while
// this one is worked on; positions follow from the box's closed-form row
// offsets.
//   CHECK: every lower slot whose neighbour lies in the block must hold the
// bits of that neighbour's mirrored upper slot (from LDS: this plane's, or
// the plane before's kept in `up`); pairs across the block's edge are read
// from W, the row's own values, and need none.
//   With kq (and wkq: the boundary stream's groups), per (block, plane, slot)
// group the least exponent of any value's lowest set bit and the range of
// the values (16 threads per slot), giving kmax and q (kq[rec + 2 u], [+ 1];
// wkq[rec + 2 s], [+ 1]) and the widths every group fits.
//   What bounds it: HBM, 27 values read and 14 + 282/256 written per row (9.2
// GB at 300^3).  Filling one plane per workgroup and scanning U and W in two
// kernels of their own took 7.5 + 7.9 + 2.1 ms there (serial loads of one
// line after another, mirrored entries gathered from memory, 70 workgroup
// reductions per plane).
constexpr int kSymStage = 27 * kBlock;  // values of a block-plane's rows
template <typename T, bool CHECK>
__global__ __launch_bounds__(kBlock, 2) void boxsym_build_kernel(
    BoxGeom g, const double* __restrict__ vals, const int* __restrict__ tab, T* __restrict__ U,
    T* __restrict__ W, T* __restrict__ kq, T* __restrict__ wkq, PlanWords* words) {
  __shared__ double sv[kSymStage];  // the staged rows, then this plane's upper slots [u][t]
  __shared__ double up[CHECK ? 9 : 1][kBlock];  // the plane before's upper slots 18 + j
  __shared__ T sw[kSymNB];
  double(*const su)[kBlock] = reinterpret_cast<double(*)[kBlock]>(sv);
  const int wg = (int)blockIdx.x;
  const int chunk = wg % g.nzc, blk = wg / g.nzc;
  const int bx = blk % g.nbx, by = blk / g.nbx;
  const int t = (int)threadIdx.x, tx = t % kBoxBX, ty = t / kBoxBX;
  const int x0 = bx * kBoxBX, ix = x0 + tx, iy = by * kBoxBY + ty;
  const int nxl = min(kBoxBX, g.gx - x0);  // live nodes per line
  const bool lline = iy < g.gy, live = ix < g.gx && lline;
  const int z0 = chunk * g.zc, z1 = min(z0 + g.zc, g.gz);
  // entries before node i of an axis of g nodes, each with its in-range neighbours
  auto pre = [](int i, int gn) { return i == 0 ? 0 : 3 * i - 1 - (i == gn ? 1 : 0); };
  auto cnt = [](int i, int gn) { return 1 + (i > 0) + (i < gn - 1); };
  const int64_t Sx = pre(g.gx, g.gx), Sy = pre(g.gy, g.gy);
  const int cy = cnt(iy, g.gy);
  const int px = pre(ix < g.gx ? ix : x0, g.gx) - pre(x0, g.gx);
  const int lx = pre(x0 + nxl, g.gx) - pre(x0, g.gx);
  double v[27];
  auto load = [&](int z) {  // the 16 lanes of a line take its values in turn
    const int cz = cnt(z, g.gz);
    const int64_t first =
        lline ? pre(z, g.gz) * Sy * Sx + cz * (pre(iy, g.gy) * Sx + cy * (int64_t)pre(x0, g.gx)) : 0;
    const int len = lline ? cz * cy * lx : 0;
#pragma unroll
    for (int k = 0; k < 27; ++k) {
      const int i = tx + kBoxBX * k;
      v[k] = i < len ? vals[first + i] : 0.0;
    }
  };
  int e[13];
#pragma unroll
  for (int s = 0; s < 13; ++s) e[s] = tab[kSymNB + t * 13 + s];
  const int gs = t / 16, gp = t % 16;  // the slot and part this thread scans
  int we[2] = {-1, -1};
  if (gs < kSymWGroups) {
    we[0] = tab[kSymWListAt + gs * kSymWListLen + gp];
    we[1] = tab[kSymWListAt + gs * kSymWListLen + gp + 16];
  }
  unsigned fit = ~0u, wfit = ~0u;
  bool same = true;
  if (CHECK) {
#pragma unroll
    for (int j = 0; j < 9; ++j) up[CHECK ? j : 0][t] = 0.0;
  }
  const int zb = CHECK && z0 > 0 ? z0 - 1 : z0;  // one plane early for the checks across planes
  load(zb);
  for (int z = zb; z < z1; ++z) {
    const bool own = z >= z0;
#pragma unroll
    for (int k = 0; k < 27; ++k) sv[ty * (27 * kBoxBX) + tx + kBoxBX * k] = v[k];
    __syncthreads();
    const unsigned m = live ? box_mask(ix, iy, z, g.gx, g.gy, g.gz) : 0u;
    double r[27];
    {
      int at = ty * (27 * kBoxBX) + cnt(z, g.gz) * cy * px;
#pragma unroll
      for (int s = 0; s < 27; ++s) {
        const bool in = (m >> s) & 1u;
        r[s] = in ? sv[at] : 0.0;
        at += in ? 1 : 0;
      }
    }
    if (z + 1 < z1) load(z + 1);
    if (own) {
#pragma unroll
      for (int u = 0; u < kSymU; ++u) U[sym_at(g, blk, z, u, t)] = (T)r[13 + u];
      const int64_t wbase = ((int64_t)blk * g.gz + z) * kSymNB;
#pragma unroll
      for (int s = 0; s < 13; ++s) {
        if (e[s] >= 0) {
          W[wbase + e[s]] = (T)r[s];
          sw[e[s]] = (T)r[s];
        } else if (CHECK && s < 9 && ((m >> s) & 1u)) {
          const int sy = s / 3 - 1, sx = s % 3 - 1;
          const double c = up[CHECK ? 8 - s : 0][t + sy * kBoxBX + sx];
          same = same && __double_as_longlong(c) == __double_as_longlong(r[s]);
        }
      }
    }
    __syncthreads();  // the staged rows and the plane before's slots are read
#pragma unroll
    for (int u = 0; u < kSymU; ++u) su[u][t] = r[13 + u];
    if (CHECK) {
#pragma unroll
      for (int j = 0; j < 9; ++j) up[CHECK ? j : 0][t] = r[18 + j];
    }
    __syncthreads();
    if (own) {
      if (CHECK) {
#pragma unroll
        for (int s = 9; s < 13; ++s)
          if (e[s] < 0 && ((m >> s) & 1u)) {
            const int sy = (s - 9) / 3 - 1, sx = (s - 9) % 3 - 1;
            const double c = su[13 - s][t + sy * kBoxBX + sx];
            same = same && __double_as_longlong(c) == __double_as_longlong(r[s]);
          }
      }
      const int64_t gi = (int64_t)blk * g.gz + z;
      if (kq) {
        PackRange<T> pr;
        const int u = gs < kSymU ? gs : 0;
#pragma unroll 4
        for (int k = 0; k < 16; ++k) pr.add((T)su[u][gp + 16 * ((k + gs) & 15)]);
        pr.join16();
        T kmax, qv;
        const unsigned w = pr.widths(kmax, qv);
        if (gs < kSymU) {
          fit &= w;
          if (gp == 0) {
            kq[gi * kSymKRec + 2 * gs] = kmax;
            kq[gi * kSymKRec + 2 * gs + 1] = qv;
          }
        }
      }
      if (wkq) {
        PackRange<T> pr;
        if (we[0] >= 0) pr.add(sw[we[0]]);
        if (we[1] >= 0) pr.add(sw[we[1]]);
        pr.join16();
        T kmax, qv;
        const unsigned w = pr.widths(kmax, qv);
        if (gs < kSymWGroups) {
          wfit &= w;
          if (gp == 0) {
            wkq[gi * kSymWRec + 2 * gs] = kmax;
            wkq[gi * kSymWRec + 2 * gs + 1] = qv;
          }
        }
      }
    }
    __syncthreads();  // sv and sw are written by the next plane
  }
  if (CHECK && !same) words->asym = 1u;
  if (gp == 0) {
#pragma unroll
    for (int i = 0; i < kPackNumWidths; ++i) {
      if (kq && gs < kSymU && !((fit >> i) & 1u)) atomicAnd(&words->fits[i], ~(1u << gs));
      if (wkq && gs < kSymWGroups && !((wfit >> i) & 1u)) atomicAnd(&words->wfits[i], ~(1u << gs));
    }
  }
}

// The fields of PF's slots (each fits its width W in every group) from kb =
// kmax - (2^W - 1), so kb is an integer of at most kmax's size and every field
// lies between 2 (the codes' successor) and 2^W - 1; packed into words, kb q
// replaces kmax.  Every value is decoded as the SpMV decodes it and compared bit
// for bit (*bad = 1 on a mismatch).  The (block, plane)'s codes flag is 1 when
// any packed value took a code.
template <typename T, typename P, int PF>
__global__ __launch_bounds__(kBlock) void boxpack_pack_kernel(const T* __restrict__ U, T* kq,
                                                              unsigned* __restrict__ PW,
                                                              unsigned* bad) {
  using B = PackBits<T>;
  constexpr PackLayout<P, PF> L{};
  constexpr int NS = P::kSlots, kWords = L.words;
  const int64_t gi = blockIdx.x;
  const int t = (int)threadIdx.x;
  T* const rec = kq + gi * kSymKRec;
  // the record's slots go through LDS: threads 0 .. 13 read (kmax, q), and after
  // the barrier (every read is done: its value is in LDS) write the SymRec
  __shared__ T base[NS], qs[NS];
  if (t < NS) {
    base[t] = rec[2 * t] - T((double)((1ull << P::width(PF, t)) - 1ull));
    qs[t] = rec[2 * t + 1];
  }
  __syncthreads();
  unsigned* const rw = reinterpret_cast<unsigned*>(rec + NS);
  if (t < NS) {
    rec[t] = base[t] * qs[t];
    if constexpr (sizeof(T) == 8) rw[t] = (unsigned)__double2hiint(qs[t]);
    else rw[t] = __float_as_uint(qs[t]);
  }
  unsigned pw[kWords];
#pragma unroll
  for (int w = 0; w < kWords; ++w) pw[w] = 0;
  bool ok = true, coded = false;
#pragma unroll
  for (int u = 0; u < NS; ++u) {
    if (!L.width[u]) continue;
    const T v = U[(gi * NS + u) * kBlock + t];
    const T qv = qs[u];
    const bool special = B::lowbit(v) == INT_MAX;
    const bool zero = special && v == T(0);
    coded = coded || special;
    const unsigned f = special ? (zero ? 0u : 1u) : (unsigned)(long long)(v / qv - base[u]);
    ok = ok && B::same(pack_decode<T, true>(base[u] * qv, qv, f), v);
    const int w = L.word[u], sh = L.shift[u];
    pw[w] |= f << sh;
    if (L.straddle[u]) pw[w + 1] |= f >> (32 - sh);
  }
#pragma unroll
  for (int w = 0; w < kWords; ++w) PW[(gi * kWords + w) * kBlock + t] = pw[w];
  if (!ok) *bad = 1u;
  const int any = __syncthreads_or(coded ? 1 : 0);
  if (t == 0) rw[NS] = any ? 1u : 0u;
}

// The symmetric box layout of A's values as T, with the groups' bases and
// powers of two and the widths they fit (what build_boxpack needs); MFE_OK
// with the layout absent when it does not fit in memory.  The first build for
// A's current values also checks the symmetry the layout relies on
// (A->boxsym_state 1 or 2) and frees the layout again when it fails.
// Synchronises the stream.
template <typename T>
static int build_boxsym(mfe_ctx* ctx, mfe_csr* A) {
  constexpr bool f64 = std::is_same<T, double>::value;
  BoxGeom g = A->box_geom;
  if (!A->boxsym_tab) {
    std::vector<int> tab;
    boxsym_tables(tab);
    if (tab.empty()) return fail(ctx, MFE_UNSUPPORTED, "symmetric layout tables");
    if (!try_alloc(ctx, &A->boxsym_tab, sizeof(int) * tab.size())) return MFE_OK;
    if (int st = upload_bytes(ctx, A->boxsym_tab, tab.data(), sizeof(int) * tab.size())) return st;
  }
  T **du, **dw, **dk;
  if constexpr (f64) {
    du = &A->boxsym_u;
    dw = &A->boxsym_w;
    dk = &A->boxpack_kq;
  } else {
    du = &A->boxsym_u32;
    dw = &A->boxsym_w32;
    dk = &A->boxpack32_kq;
  }
  const int64_t groups = (int64_t)g.nbx * g.nby * g.gz;
  if (!*du && !try_alloc(ctx, du, sizeof(T) * (size_t)sym_entries(g))) return MFE_OK;
  if (!*dw && !try_alloc(ctx, dw, sizeof(T) * (size_t)sym_bnd_entries(g))) return MFE_OK;
  // without room for these the values stay at full width
  if (!*dk) (void)try_alloc(ctx, dk, sizeof(T) * (size_t)(groups * kSymKRec));
  T* wkq = nullptr;
  if constexpr (f64) {
    if (!A->boxwpack_kq) (void)try_alloc(ctx, &A->boxwpack_kq, sizeof(T) * (size_t)(groups * kSymWRec));
    wkq = A->boxwpack_kq;
  }
  const bool check = A->boxsym_state == 0;
  PlanWords* words = reinterpret_cast<PlanWords*>(ctx->d_scalars + kPlanWordsAt);
  plan_words_kernel<<<1, kWave, 0, ctx->stream>>>(words);
  auto run = [&](auto kern) {
    box_chunks(g, resident_groups((const void*)kern, ctx->cu_count), groups);
    kern<<<(unsigned)((int64_t)g.nbx * g.nby * g.nzc), kBlock, 0, ctx->stream>>>(
        g, A->vals, A->boxsym_tab, *du, *dw, *dk, wkq, words);
  };
  if (check) run(boxsym_build_kernel<T, true>);
  else run(boxsym_build_kernel<T, false>);
  MFE_LAUNCHED(ctx, "boxsym_build_kernel");
  PlanWords hw;
  if (int st = download_bytes(ctx, &hw, words, sizeof(hw))) return st;
  if (check) {
    A->boxsym_state = hw.asym ? 2 : 1;
    if (hw.asym) {  // not symmetric: the box layout with all 27 slots instead
      csr_free(A, *du);
      csr_free(A, *dw);
      *du = nullptr;
      *dw = nullptr;
      return MFE_OK;
    }
  }
  for (int i = 0; i < kPackNumWidths; ++i) {
    (f64 ? A->boxpack_fits : A->boxpack32_fits)[i] = *dk ? hw.fits[i] : 0u;
    if (f64) A->boxwpack_fits[i] = wkq ? hw.wfits[i] : 0u;
  }
  if constexpr (f64) A->boxsym_valid = true;
  else A->boxsym32_valid = true;
  return MFE_OK;
}

// f(std::integral_constant<int, form>) for a packed form that precision T
// has (FP32: no 32-bit fields); else hipErrorInvalidValue.
template <typename T, typename F>
static int with_pack_form(int form, F&& f) {
  using std::integral_constant;
  constexpr bool f64 = sizeof(T) == 8;
  switch (form) {
    case kPackAll16: return f(integral_constant<int, kPackAll16>{});
    case kPackCube16: return f(integral_constant<int, kPackCube16>{});
    case kPackAll12: return f(integral_constant<int, kPackAll12>{});
    case kPackAll10: return f(integral_constant<int, kPackAll10>{});
    case kPackCube16Near32:
      if constexpr (f64) return f(integral_constant<int, kPackCube16Near32>{});
      break;
    case kPackCube12Near24: return f(integral_constant<int, kPackCube12Near24>{});
    case kPackCube10Near22: return f(integral_constant<int, kPackCube10Near22>{});
    default: break;
  }
  return (int)hipErrorInvalidValue;
}

// The packed form of the symmetric layout U (precision T, `groups` (block,
// plane) groups), built after the layout: of the forms whose every field fits
// its width in every group (fits), the one with the fewest bytes per row
// (fields and full-width values), or none (kPackNone: the SpMV reads the full
// values).  *pw and *cap are the layout's words (allocated here); the form is
// left kPackNone when they do not fit in memory.  Enqueues the packing; the
// caller checks words->pack_bad.
template <typename T>
static int enqueue_pack(mfe_ctx* ctx, const mfe_csr* A, const T* U, int64_t groups,
                        const unsigned* fits, T* kq, unsigned** pw, int* cap, PlanWords* words,
                        int* form_out) {
  using P = SymPack;
  constexpr bool f64 = std::is_same<T, double>::value;
  *form_out = kPackNone;
  int form = kPackNone;
  int64_t best = 0;
  for (int f = 1; f < kPackForms; ++f) {
    if (!f64 && pack_wide(f) == 32) continue;  // FP32: fields below 2^24
    bool fits_all = true;
    int fulls = 0;
    for (int s = 0; s < P::kSlots; ++s) {
      const int w = P::width(f, s);
      if (w == 0) {
        ++fulls;
        continue;
      }
      int i = 0;
      while (kPackWidths[i] != w) ++i;
      fits_all = fits_all && ((fits[i] >> s) & 1u);
    }
    const int64_t bytes = 4 * (int64_t)P::words(f) + (int64_t)sizeof(T) * fulls;
    if (fits_all && (form == kPackNone || bytes < best)) {
      form = f;
      best = bytes;
    }
  }
  if (form == kPackNone) return MFE_OK;
  const int nw = P::words(form);
  if (*cap < nw) {
    csr_free(A, *pw);
    *pw = nullptr;
    *cap = 0;
    if (!try_alloc(ctx, pw, sizeof(unsigned) * (size_t)(groups * nw * kBlock))) return MFE_OK;
    *cap = nw;
  }
  with_pack_form<T>(form, [&](auto pf) {
    boxpack_pack_kernel<T, P, decltype(pf)::value>
        <<<(unsigned)groups, kBlock, 0, ctx->stream>>>(U, kq, *pw, &words->pack_bad);
    return 0;
  });
  MFE_LAUNCHED(ctx, "boxpack_pack_kernel");
  *form_out = form;
  return MFE_OK;
}

// The packed boundary stream (mfe_boxsym.hpp) in form F: the fields of the
// (block, plane)'s entries,
// assembled in LDS, each decoded as the SpMV decodes it and compared bit for
// bit (*bad = 1 on a mismatch); kb q replaces kmax, and the codes flag is set.
template <typename T, int F>
__global__ __launch_bounds__(kBlock) void boxwpack_pack_kernel(const T* __restrict__ W,
                                                               const int* __restrict__ tab,
                                                               T* __restrict__ wkq,
                                                               unsigned* __restrict__ WPW,
                                                               unsigned* bad) {
  using B = PackBits<T>;
  constexpr int wn = pack_narrow(F), ww = pack_all(F) ? wn : pack_wide(F);
  constexpr int kWords = sym_w_words(F);
  __shared__ unsigned acc[kWords];
  __shared__ T base[kSymWGroups], qs[kSymWGroups];
  const int64_t gi = blockIdx.x;
  const int t = (int)threadIdx.x;
  if (t < kWords) acc[t] = 0u;
  if (t < kSymWGroups) {
    const int wd = ((kSymWNear >> t) & 1u) ? ww : wn;
    base[t] = wkq[gi * kSymWRec + 2 * t] - T((double)((1ull << wd) - 1ull));
    qs[t] = wkq[gi * kSymWRec + 2 * t + 1];
  }
  __syncthreads();
  bool ok = true, coded = false;
  for (int e = t; e < kSymNB; e += kBlock) {
    const int code = tab[e];
    const int sl = (code >> 26) & 15, near = (code >> 25) & 1, nb = (code >> 16) & 511;
    const int wd = near ? ww : wn;
    const int off = (e - nb) * wn + nb * ww;
    const T v = W[gi * kSymNB + e];
    const bool special = B::lowbit(v) == INT_MAX;
    const bool zero = special && v == T(0);
    coded = coded || special;
    const unsigned f = special ? (zero ? 0u : 1u) : (unsigned)(long long)(v / qs[sl] - base[sl]);
    ok = ok && B::same(pack_decode<T, true>(base[sl] * qs[sl], qs[sl], f), v);
    const int sh = off & 31;
    atomicOr(&acc[off >> 5], f << sh);
    if (sh + wd > 32) atomicOr(&acc[(off >> 5) + 1], f >> (32 - sh));
  }
  __syncthreads();
  if (t < kWords) WPW[gi * kWords + t] = acc[t];
  if (!ok) *bad = 1u;
  const int any = __syncthreads_or(coded ? 1 : 0);
  if (t < kSymWGroups) wkq[gi * kSymWRec + 2 * t] = base[t] * qs[t];
  if (t == 0) wkq[gi * kSymWRec + 2 * kSymWGroups] = any ? T(1) : T(0);
}

// The FP64 boundary stream's packed form: of the forms that give every entry a
// field and whose widths every group fits, the one with the fewest words, or
// none (the SpMV reads the full values).  Enqueues the packing; the caller
// checks words->wpack_bad.
static int enqueue_wpack(mfe_ctx* ctx, mfe_csr* A, int64_t groups, PlanWords* words,
                         int* form_out) {
  *form_out = kPackNone;
  if (!A->boxwpack_pw &&
      !try_alloc(ctx, &A->boxwpack_pw, sizeof(unsigned) * (size_t)(groups * sym_w_words(kPackCube16Near32))))
    return MFE_OK;
  auto fit = [&](int wd, unsigned slots) {
    int i = 0;
    while (kPackWidths[i] != wd) ++i;
    return (A->boxwpack_fits[i] & slots) == slots;
  };
  const unsigned all = (1u << kSymWGroups) - 1u;
  int form = kPackNone;
  for (int f = 1; f < kPackForms; ++f) {
    if (f == kPackCube16) continue;
    const bool ok = pack_all(f) ? fit(pack_narrow(f), all)
                                : fit(pack_narrow(f), all & ~kSymWNear) && fit(pack_wide(f), kSymWNear);
    if (ok && (form == kPackNone || sym_w_words(f) < sym_w_words(form))) form = f;
  }
  if (form == kPackNone) return MFE_OK;
  with_pack_form<double>(form, [&](auto pf) {
    boxwpack_pack_kernel<double, decltype(pf)::value><<<(unsigned)groups, kBlock, 0, ctx->stream>>>(
        A->boxsym_w, A->boxsym_tab, A->boxwpack_kq, A->boxwpack_pw, &words->wpack_bad);
    return 0;
  });
  MFE_LAUNCHED(ctx, "boxwpack_pack_kernel");
  *form_out = form;
  return MFE_OK;
}

// The packed form of A's symmetric layout in precision T (after the layout):
// the upper values, and the boundary stream where the upper values are packed.
// A form whose fields do not give back every value is not used.  Synchronises
// the stream when something was packed.
template <typename T>
static int build_boxpack(mfe_ctx* ctx, mfe_csr* A) {
  constexpr bool f64 = std::is_same<T, double>::value;
  const BoxGeom g = A->box_geom;
  const int64_t groups = (int64_t)g.nbx * g.nby * g.gz;
  PlanWords* words = reinterpret_cast<PlanWords*>(ctx->d_scalars + kPlanWordsAt);
  plan_words_kernel<<<1, kWave, 0, ctx->stream>>>(words);
  int form = kPackNone, wform = kPackNone, st = MFE_OK;
  if constexpr (f64) {
    st = enqueue_pack<double>(ctx, A, A->boxsym_u, groups, A->boxpack_fits, A->boxpack_kq,
                              &A->boxpack_pw, &A->boxpack_cap, words, &form);
    if (!st && form != kPackNone) st = enqueue_wpack(ctx, A, groups, words, &wform);
  } else {
    st = enqueue_pack<float>(ctx, A, A->boxsym_u32, groups, A->boxpack32_fits, A->boxpack32_kq,
                             &A->boxpack32_pw, &A->boxpack32_cap, words, &form);
  }
  if (st) return st;
  if (form != kPackNone) {
    PlanWords hw;
    if ((st = download_bytes(ctx, &hw, words, sizeof(hw)))) return st;
    if (hw.wpack_bad) wform = kPackNone;
    if (hw.pack_bad) form = wform = kPackNone;
  }
  if constexpr (f64) {
    A->boxpack_form = form;
    A->boxwpack_form = wform;
    A->boxpack_valid = true;
  } else {
    A->boxpack32_form = form;
    A->boxpack32_valid = true;
  }
  return MFE_OK;
}

// allow_box false: the SELL/CSR plan even where the box layout applies (the
// many-RHS SELL tiles, comparison runs).
static int ensure_plan(mfe_ctx* ctx, const mfe_csr* Ac, bool need64, bool need32,
                       bool allow_box = true) {
  mfe_csr* A = const_cast<mfe_csr*>(Ac);
  hipStream_t s = ctx->stream;
  const int64_t n = A->nrows;
  if (allow_box && box_applies(A)) {
    int st;
    box_set_geometry(A);
    if (A->boxsym_state != 2) {  // symmetric, or not examined yet (the first build checks)
      if (need64 && !A->boxsym_valid && (st = build_boxsym<double>(ctx, A))) return st;
      if (need64 && A->boxsym_state == 1 && A->boxsym_valid && !A->boxpack_valid &&
          (st = build_boxpack<double>(ctx, A)))
        return st;
      if (need32 && !A->boxsym32_valid && A->boxsym_state != 2 &&
          (st = build_boxsym<float>(ctx, A)))
        return st;
      if (need32 && A->boxsym_state == 1 && A->boxsym32_valid && !A->boxpack32_valid &&
          (st = build_boxpack<float>(ctx, A)))
        return st;
      if (A->boxsym_state == 1 && (!need64 || A->boxsym_valid) &&
          (!need32 || A->boxsym32_valid))
        return MFE_OK;
    }
    if (need64 && !A->box_vals_valid && (st = build_box<double>(ctx, A))) return st;
    if (need32 && !A->box_vals32_valid && (st = build_box<float>(ctx, A))) return st;
    if ((!need64 || A->box_vals_valid) && (!need32 || A->box_vals32_valid)) return MFE_OK;
    // no room for the layout: the SELL/CSR plan below
  }
  const bool sell_format = A->spmv_format == MFE_SPMV_AUTO || A->spmv_format == MFE_SPMV_SELL;
  if (sell_format && !A->sell_struct_valid && n > 0) {
    sell_release(A);
    const int64_t ns = cdiv(n, kSlice);
    int* d_width = nullptr;
    bool ok = try_alloc(ctx, &A->sell_len, (size_t)(ns * kSlice)) &&
              try_alloc(ctx, &A->sell_off, sizeof(int) * (size_t)(ns + 1)) &&
              try_alloc(ctx, &d_width, sizeof(int) * (size_t)ns);
    if (ok) {
      sell_len_kernel<<<(unsigned)cdiv(ns * kSlice, kBlock), kBlock, 0, s>>>(
          (int)n, (int)ns, A->row_offsets, A->sell_len, d_width);
      MFE_LAUNCHED(ctx, "sell_len_kernel");
      std::vector<int> width((size_t)ns), off((size_t)ns + 1);
      {
        const int dst = download_bytes(ctx, width.data(), d_width, sizeof(int) * (size_t)ns);
        if (dst) {
          dev_free(ctx, d_width);
          return dst;
        }
      }
      int64_t acc = 0;
      int maxw = 0;
      for (int64_t i = 0; i < ns; ++i) {
        off[(size_t)i] = (int)acc;
        acc += width[(size_t)i];
        maxw = std::max(maxw, width[(size_t)i]);
      }
      off[(size_t)ns] = (int)acc;
      A->sell_max_len = maxw;
      A->sell_nslices = ns;
      A->sell_slots = acc * kSlice;
      ok = maxw <= kSellMaxWidth && acc < INT32_MAX &&
           try_alloc(ctx, &A->sell_cols, sizeof(int) * (size_t)(A->sell_slots + kSellTail));
      if (ok) {
        MFE_CHECK(ctx, hipMemsetAsync(A->sell_cols + A->sell_slots, 0, sizeof(int) * kSellTail, s));
        int ust = upload_bytes(ctx, A->sell_off, off.data(), sizeof(int) * (size_t)(ns + 1));
        if (ust) return ust;
        sell_fill_kernel<int, int><<<(unsigned)ns, kSlice, 0, s>>>(
            (int)n, (int)ns, A->sell_off, A->sell_len, A->row_offsets, A->cols, A->sell_cols,
            true);
        MFE_LAUNCHED(ctx, "sell_fill_kernel (columns)");
      }
    }
    dev_free(ctx, d_width);
    A->sell_struct_valid = true;
    if (ok) {
      A->sell_ok = true;
    } else {
      sell_disable(A);
    }
  }
  if (A->spmv_format == MFE_SPMV_AUTO && A->sell_ok && !A->sellx_valid && n > 0) {
    int st;
    if ((st = build_sellx(ctx, A))) return st;
  }
  const bool sell = sell_format && A->sell_ok && n > 0;
  const unsigned fg = (unsigned)A->sell_nslices;  // one wave per slice
  if (sell && need64 && !A->sell_vals_valid) {
    if (!A->sell_vals) {
      if (!try_alloc(ctx, &A->sell_vals, sizeof(double) * (size_t)(A->sell_slots + kSellTail))) {
        sell_disable(A);  // no room for the copy: CSR kernels
        return ensure_plan(ctx, A, need64, need32, allow_box);
      }
      MFE_CHECK(ctx, hipMemsetAsync(A->sell_vals + A->sell_slots, 0, sizeof(double) * kSellTail, s));
    }
    sell_fill_kernel<double, double><<<fg, kSlice, 0, s>>>(
        (int)n, (int)A->sell_nslices, A->sell_off, A->sell_len, A->row_offsets, A->vals,
        A->sell_vals, false);
    MFE_LAUNCHED(ctx, "sell_fill_kernel<double>");
    A->sell_vals_valid = true;
  }
  if (sell && need32 && !A->sell_vals32_valid) {
    if (!A->sell_vals32) {
      if (!try_alloc(ctx, &A->sell_vals32, sizeof(float) * (size_t)(A->sell_slots + kSellTail))) {
        sell_disable(A);
        return ensure_plan(ctx, A, need64, need32, allow_box);
      }
      MFE_CHECK(ctx, hipMemsetAsync(A->sell_vals32 + A->sell_slots, 0, sizeof(float) * kSellTail, s));
    }
    sell_fill_kernel<double, float><<<fg, kSlice, 0, s>>>(
        (int)n, (int)A->sell_nslices, A->sell_off, A->sell_len, A->row_offsets, A->vals,
        A->sell_vals32, false);
    MFE_LAUNCHED(ctx, "sell_fill_kernel<float>");
    A->sell_vals32_valid = true;
  }
  if (!sell && need32 && !A->vals32_valid) {
    if (!A->vals32)
      MFE_CHECK(ctx, dev_alloc(ctx, &A->vals32, sizeof(float) * (size_t)(A->nnz > 0 ? A->nnz : 1)));
    if (A->nnz > 0) {
      vals_to_f32_kernel<<<(unsigned)std::min<int64_t>(cdiv(A->nnz, kBlock), 65536), kBlock, 0,
                           s>>>(A->nnz, A->vals, A->vals32);
      MFE_LAUNCHED(ctx, "vals_to_f32_kernel");
    }
    A->vals32_valid = true;
  }
  return MFE_OK;
}

int sell_prepare(mfe_ctx* ctx, const mfe_csr* A) { return ensure_plan(ctx, A, true, false, false); }

int box_prepare(mfe_ctx* ctx, const mfe_csr* Ac) {
  mfe_csr* A = const_cast<mfe_csr*>(Ac);
  if (!box_applies(A)) return MFE_OK;
  box_set_geometry(A);
  if (A->box_vals_valid) return MFE_OK;
  return build_box<double>(ctx, A);
}

// Rows from which the packed boundary stream is read (measured at launch_spmv).
constexpr int64_t kWPackRows = 1 << 23;

// What one SpMV launch reads: the SELL copy when the plan has one for T,
// else the CSR arrays (FP64 values, or the CSR FP32 copy).
template <typename T>
struct SpmvOp {
  const mfe_csr* A = nullptr;
  uint64_t gen = 0;  // A->plan_gen when made
  int n = 0;
  const int* ro = nullptr;
  const int* cols = nullptr;
  const T* vals = nullptr;
  bool stream_ok = false;  // CSR row-stream kernel applies (else row-per-thread)
  int nslices = 0;
  const int* soff = nullptr;
  const unsigned char* slen = nullptr;
  const int* scols = nullptr;
  const T* svals = nullptr;  // non-null: SELL
  const unsigned short* xl = nullptr;  // non-null: SELL with staged x
  const unsigned short* xltail = nullptr;
  const unsigned char* xaff = nullptr;
  const unsigned short* xsbase = nullptr;
  const int *xroff = nullptr, *xrcol = nullptr, *xrpos = nullptr, *xnu = nullptr;
  int xmaxu = 0;
  int cus = 0;                // compute units (box launches size their z chunks)
  const T* bvals = nullptr;  // non-null: box layout (takes precedence)
  const T* symu = nullptr;   // non-null: symmetric box layout (takes precedence over both)
  const T* symw = nullptr;
  const int* symtab = nullptr;
  int pack = kPackNone;           // the symmetric layout's packed form (a PackForm), if used
  const unsigned* pw = nullptr;   // its words
  const T* pkq = nullptr;         // its (base, power of two) per (block, plane, slot)
  int wpack = kPackNone;          // the boundary stream's packed form, if there is one (with pack)
  int64_t wrows = kWPackRows;     // rows from which it is read
  const unsigned* wpw = nullptr;
  const T* wkq = nullptr;
  BoxGeom bg{};
  // All that a launch chooses its kernel by or hands to it: a captured graph may be
  // replayed for an operand that ties equal.  (Values that change in place stay
  // covered; a rebuilt plan may take another packed form in the same memory.)
  auto tie() const {
    return std::tie(A, gen, n, ro, cols, vals, stream_ok, nslices, soff, slen, scols, svals, xl,
                    xltail, xaff, xsbase, xroff, xrcol, xrpos, xnu, xmaxu, cus, bvals, symu, symw,
                    symtab, pack, pw, pkq, wpack, wrows, wpw, wkq, bg.gx, bg.gy, bg.gz, bg.nbx, bg.nby);
  }
};

// allow_sell false: the CSR kernels; allow_stage false: plain SELL even where
// the staged-x plan exists.
template <typename T>
static SpmvOp<T> spmv_op(const mfe_csr* A, bool allow_sell = true, bool allow_stage = true,
                         bool allow_box = true, bool allow_sym = true, bool allow_pack = true) {
  SpmvOp<T> op;
  op.A = A;
  op.gen = A->plan_gen;
  op.n = (int)A->nrows;
  op.ro = A->row_offsets;
  op.cols = A->cols;
  op.stream_ok = A->max_block_nnz >= 0 && A->max_block_nnz <= kSpmvMaxNnz;
  op.cus = A->ctx ? A->ctx->cu_count : 0;
  if (allow_box && allow_sell && allow_stage && box_applies(A)) {
    if (allow_sym && A->boxsym_state == 1) {
      if constexpr (std::is_same<T, double>::value) {
        if (A->boxsym_valid) {
          op.symu = A->boxsym_u;
          op.symw = A->boxsym_w;
          if (allow_pack && A->boxpack_valid && A->boxpack_form != kPackNone) {
            op.pack = A->boxpack_form;
            op.pw = A->boxpack_pw;
            op.pkq = A->boxpack_kq;
            if (A->boxwpack_form != kPackNone) {
              op.wpack = A->boxwpack_form;
              op.wpw = A->boxwpack_pw;
              op.wkq = A->boxwpack_kq;
            }
          }
        }
      } else {
        if (A->boxsym32_valid) {
          op.symu = A->boxsym_u32;
          op.symw = A->boxsym_w32;
          if (allow_pack && A->boxpack32_valid && A->boxpack32_form != kPackNone) {
            op.pack = A->boxpack32_form;
            op.pw = A->boxpack32_pw;
            op.pkq = A->boxpack32_kq;
          }
        }
      }
      if (op.symu) {
        op.symtab = A->boxsym_tab;
        op.bg = A->box_geom;
        return op;
      }
    }
    if constexpr (std::is_same<T, double>::value) {
      if (A->box_vals_valid) op.bvals = A->box_vals;
    } else {
      if (A->box_vals32_valid) op.bvals = A->box_vals32;
    }
    if (op.bvals) {
      op.bg = A->box_geom;
      return op;
    }
  }
  const bool sell = allow_sell && A->sell_ok &&
                    (A->spmv_format == MFE_SPMV_AUTO || A->spmv_format == MFE_SPMV_SELL);
  if constexpr (std::is_same<T, double>::value) {
    op.vals = A->vals;
    if (sell && A->sell_vals_valid) op.svals = A->sell_vals;
  } else {
    op.vals = A->vals32;
    if (sell && A->sell_vals32_valid) op.svals = A->sell_vals32;
  }
  if (op.svals) {
    op.nslices = (int)A->sell_nslices;
    op.soff = A->sell_off;
    op.slen = A->sell_len;
    op.scols = A->sell_cols;
    if (allow_stage && A->spmv_format == MFE_SPMV_AUTO && A->sellx_ok) {
      op.xl = A->sellx_lcols;
      op.xltail = A->sellx_lcols + A->sell_slots;
      op.xaff = A->sellx_aff;
      op.xsbase = A->sellx_sbase;
      op.xroff = A->sellx_roff;
      op.xrcol = A->sellx_rcol;
      op.xrpos = A->sellx_rpos;
      op.xnu = A->sellx_nu;
      op.xmaxu = A->sellx_maxu;
    }
  }
  return op;
}

// -------------------------------------------------------------- vectors -----

template <typename T>
__global__ __launch_bounds__(kBlock) void waxpby_kernel(int64_t n, T alpha, const T* x, T beta,
                                                        const T* y, T* w) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    w[i] = alpha * x[i] + beta * y[i];
}

// dst = (float)(src * scale)
__global__ __launch_bounds__(kBlock) void to_f32_kernel(int64_t n, const double* __restrict__ src,
                                                        double scale, float* __restrict__ dst) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    dst[i] = (float)(src[i] * scale);
}

// dst = (double)src
__global__ __launch_bounds__(kBlock) void to_f64_kernel(int64_t n, const float* __restrict__ src,
                                                        double* __restrict__ dst) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    dst[i] = (double)src[i];
}

// x = 1*x + a*(double)d : the refinement update in FP64.
__global__ __launch_bounds__(kBlock) void refine_update_kernel(int64_t n, double a,
                                                               const float* __restrict__ d,
                                                               double* __restrict__ x) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    x[i] = 1.0 * x[i] + a * (double)d[i];
}

// Per-thread partial sums over a fixed grid-stride pattern, then the fixed
// wave/workgroup tree: deterministic for a given n.
template <typename T>
__device__ __forceinline__ T grid_dot(int64_t n, const T* __restrict__ x, const T* __restrict__ y) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  T acc = T(0);
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    acc += x[i] * y[i];
  return acc;
}

template <typename T>
__global__ __launch_bounds__(kBlock) void dot_partial_kernel(int64_t n, const T* __restrict__ x,
                                                             const T* __restrict__ y,
                                                             T* __restrict__ partials) {
  __shared__ T red[4];
  const T acc = block_sum<T>(grid_dot<T>(n, x, y), red);
  if (threadIdx.x == 0) partials[blockIdx.x] = acc;
}

// Workgroup sum of p[0..np): each thread adds its strided values in index
// order (eight loads in flight per step), then the fixed workgroup tree.
template <typename T>
__device__ __forceinline__ T sum_partials(const T* __restrict__ p, int np, T* red) {
  T acc = T(0);
  int i = (int)threadIdx.x;
  for (; i + 7 * kBlock < np; i += 8 * kBlock) {
    T v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = p[i + u * kBlock];
#pragma unroll
    for (int u = 0; u < 8; ++u) acc += v[u];
  }
  for (; i < np; i += kBlock) acc += p[i];
  return block_sum<T>(acc, red);
}

// First stage of a two-stage reduction of nvec arrays of np partials: block j
// sums partials[v*np + j*kStage .. +kStage) into out[v*gridDim.x + j].
constexpr int kStage = 8 * kBlock;
template <typename T>
__global__ __launch_bounds__(kBlock) void reduce_stage_kernel(const T* __restrict__ partials,
                                                              int np, int nvec,
                                                              T* __restrict__ out,
                                                              const int* __restrict__ done) {
  if (done && *done) return;
  __shared__ T red[4];
  const int j = (int)blockIdx.x;
  const int lo = j * kStage;
  const int m = min(kStage, np - lo);
  for (int v = 0; v < nvec; ++v) {
    const T s = sum_partials<T>(partials + (int64_t)v * np + lo, m, red);
    if (threadIdx.x == 0) out[(int64_t)v * gridDim.x + j] = s;
  }
}

__global__ __launch_bounds__(kBlock) void finalize_kernel(const double* __restrict__ partials,
                                                          int np, int nvec,
                                                          double* __restrict__ out) {
  __shared__ double red[4];
  for (int v = 0; v < nvec; ++v) {
    const double s = sum_partials<double>(partials + (int64_t)v * np, np, red);
    if (threadIdx.x == 0) out[v] = s;
  }
}

// Sequential dot, the reference's left-to-right order (Vector_functions.hpp:
// 216-218): the workgroup stages products x[i]*y[i] into LDS in chunks and
// thread 0 adds them in index order.  One workgroup; for replay/parity use.
constexpr int kSeqChunk = 8 * kBlock;
__device__ double dot_sequential(int64_t n, const double* x, const double* y, double* buf) {
  double result = 0;
  for (int64_t base = 0; base < n; base += kSeqChunk) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int64_t i = base + threadIdx.x + k * kBlock;
      if (i < n) buf[threadIdx.x + k * kBlock] = x[i] * y[i];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      const int m = (int)((n - base) < kSeqChunk ? (n - base) : kSeqChunk);
      for (int j = 0; j < m; ++j) result += buf[j];
    }
    __syncthreads();
  }
  return result;  // valid in thread 0
}

__global__ __launch_bounds__(kBlock) void dot_seq_kernel(int64_t n, const double* x,
                                                         const double* y, double* out) {
  __shared__ double buf[kSeqChunk];
  const double r = dot_sequential(n, x, y, buf);
  if (threadIdx.x == 0) *out = r;
}

// ------------------------------------------------------------------- CG -----
//
// Per iteration k (fast mode), all on one stream:
//   advance    (k > 1) breakdown() if the norms were needed; end of k-1; loop
//              test; rtrans, beta, normr of k
//   p          x += alpha_{k-1} p_{k-1} (deferred, see below); p = 1*r + beta*y
//   spmv       Ap = A p, workgroup partials of p.Ap
//   reduce     first stage of the p.Ap reduction (large n only)
//   update     p.Ap; breakdown test; alpha = rtrans / p.Ap;
//              r = 1*r + (-alpha)*Ap, workgroup partials of r.r (and, only
//              when p.Ap < brkdown_tol, of ||Ap||^2 and ||p||^2)
// The scalars live in two records: `st` as an iteration begins (written by
// advance) and `mid` after its alpha (written by update).  A kernel reads one
// and its first workgroup writes the other, so every workgroup of the p update
// can do the advance step itself (from mid and the r.r partials: the same sums
// in the same order give all of them the same scalars) and the separate launch
// goes away; running it twice changes nothing.
// The per-operation timing mode runs the same sums as separate kernels
// (reduce, alpha, norms, norms-fin, update, next) on st alone.
// The reference updates x right after r (cg_solve.hpp:211-212).  Here the
// update x = 1*x + alpha*p of iteration k is applied by the next cg_p, which
// reads p anyway (or by cg_finish after the last iteration): the same
// operation on the same operands, so the same bits, one vector pass fewer.
// Scalars (rtrans, alpha, beta, ...) are kept in double for both vector types.

struct CgState {
  double rtrans, oldrtrans, pAp, alpha, beta, normr, brkdown_tol, tol;
  double alpha_prev;  // alpha of the iteration whose x update is pending
  double gamma;       // coefficient of r in the next p update (1 but after a resume)
  int k, max_iter, done, status, num_iters, need_norms, x_pending, pad;
};

// Prologue scalar step: rtrans = r0.r0, normr, and the loop test for k = 1.
__device__ void cg_begin_first(CgState* st, double rr) {
  st->rtrans = rr;
  st->normr = sqrt(rr);
  st->beta = 0.0;
  st->k = 1;
  if (!(1 <= st->max_iter && st->normr > st->tol)) st->done = 1;
}

// End of iteration k (r updated): its x update becomes pending, num_iters = k,
// then the reference's loop test with the normr of iteration k, and rtrans,
// beta, normr of iteration k+1 (cg_solve.hpp:152-165).
__device__ void cg_next(CgState* st, double rr) {
  st->x_pending = 1;
  st->alpha_prev = st->alpha;
  st->num_iters = st->k;
  const int k1 = st->k + 1;
  if (!(k1 <= st->max_iter && st->normr > st->tol)) {
    st->done = 1;
    return;
  }
  st->oldrtrans = st->rtrans;
  st->rtrans = rr;
  st->beta = st->rtrans / st->oldrtrans;
  st->normr = sqrt(st->rtrans);
  st->k = k1;
}

__device__ double* hist_row(const CgState* st, double* hist) {
  return hist + 4 * (int64_t)(st->k - 1);
}

// Record p.Ap and, unless the breakdown test needs the norms, alpha.
// (cg_solve.hpp:186-201)
__device__ void cg_alpha_or_defer(CgState* st, double pAp, double* hist) {
  st->x_pending = 0;  // cg_p of this iteration has applied it
  st->gamma = 1.0;
  st->pAp = pAp;
  double* h = hist_row(st, hist);
  h[0] = st->rtrans;
  h[1] = pAp;
  h[2] = 0.0;
  h[3] = st->beta;
  if (pAp < st->brkdown_tol) {
    if (pAp < 0) {
      st->status = MFE_BREAKDOWN;
      st->done = 1;
      return;
    }
    st->need_norms = 1;
    return;
  }
  st->alpha = st->rtrans / pAp;
  h[2] = st->alpha;
}

// breakdown() (cg_solve.hpp:49-67) with v = Ap, w = p, then alpha.
__device__ void cg_alpha_after_norms(CgState* st, double ApAp, double pp, double* hist) {
  st->need_norms = 0;
  const double vnorm = sqrt(ApAp), wnorm = sqrt(pp);
  if (fabs(st->pAp) <= 100 * vnorm * wnorm * DBL_EPSILON) {
    st->status = MFE_BREAKDOWN;
    st->done = 1;
    return;
  }
  st->brkdown_tol = 0.1 * st->pAp;
  st->alpha = st->rtrans / st->pAp;
  hist_row(st, hist)[2] = st->alpha;
}

__global__ void cg_init_kernel(CgState* st, int max_iter, double tol) {
  CgState s;
  memset(&s, 0, sizeof(s));
  s.max_iter = max_iter;
  s.tol = tol;
  s.brkdown_tol = DBL_EPSILON;
  s.gamma = 1.0;
  s.k = 1;
  *st = s;
}

// Fast mode scalar kernels (one workgroup each) ------------------------------
template <typename T>
__global__ __launch_bounds__(kBlock) void cg_first_fast_kernel(CgState* st, CgState* mid,
                                                               const T* partials, int np) {
  __shared__ T red[4];
  const T rr = sum_partials<T>(partials, np, red);
  if (threadIdx.x == 0) {
    cg_begin_first(st, (double)rr);
    *mid = *st;  // what advance reads if there is nothing to do
  }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void cg_alpha_fast_kernel(CgState* st, const T* partials,
                                                               int np, double* hist) {
  if (st->done) return;
  __shared__ T red[4];
  const T pAp = sum_partials<T>(partials, np, red);
  if (threadIdx.x == 0) cg_alpha_or_defer(st, (double)pAp, hist);
}

// ||Ap||^2 and ||p||^2 partials, only when the breakdown test needs them.
template <typename T>
__global__ __launch_bounds__(kBlock) void cg_norms_kernel(int64_t n, const CgState* st,
                                                          const T* __restrict__ Ap,
                                                          const T* __restrict__ p,
                                                          T* __restrict__ partials) {
  if (st->done || !st->need_norms) return;
  __shared__ T red[4];
  const T a = block_sum<T>(grid_dot<T>(n, Ap, Ap), red);
  const T b = block_sum<T>(grid_dot<T>(n, p, p), red);
  if (threadIdx.x == 0) {
    partials[blockIdx.x] = a;
    partials[gridDim.x + blockIdx.x] = b;
  }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void cg_norms_fin_kernel(CgState* st, const T* partials,
                                                              int np, double* hist) {
  if (st->done || !st->need_norms) return;
  __shared__ T red[4];
  const T ApAp = sum_partials<T>(partials, np, red);
  const T pp = sum_partials<T>(partials + np, np, red);
  if (threadIdx.x == 0) cg_alpha_after_norms(st, (double)ApAp, (double)pp, hist);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void cg_next_fast_kernel(CgState* st, const T* partials,
                                                              int np) {
  if (st->done) return;
  __shared__ T red[4];
  const T rr = sum_partials<T>(partials, np, red);
  if (threadIdx.x == 0) cg_next(st, (double)rr);
}

// Continue a stopped CG after its residual was replaced (the mixed solve's
// FP64 residual, rounded): rtrans = r.r of the new residual and beta = rtrans
// / rtrans of the last iteration.  The replaced r is no longer orthogonal to
// the kept p, so p first loses its r component, p <- p - (r.p / r.r) r (the
// "reliable update" of mixed-precision CG, Clark et al. 2010); folded into
// the next cg_p as p = gamma r + beta p with gamma = 1 - beta (r.p / r.r).
// k restarts at 1 (history rows stay in range; the captured iterations always
// take p = gamma r + beta p).
template <typename T>
__global__ __launch_bounds__(kBlock) void cg_resume_kernel(CgState* st, CgState* mid,
                                                           const T* partials, int np, int max_iter,
                                                           double tol) {
  __shared__ T red[4];
  const T rr = sum_partials<T>(partials, np, red);
  const T rp = sum_partials<T>(partials + np, np, red);
  if (threadIdx.x == 0) {
    st->oldrtrans = st->rtrans;
    st->rtrans = (double)rr;
    st->beta = st->oldrtrans > 0 ? st->rtrans / st->oldrtrans : 0.0;
    st->gamma = st->rtrans > 0 ? 1.0 - st->beta * ((double)rp / st->rtrans) : 1.0;
    st->normr = sqrt(st->rtrans);
    st->k = 1;
    st->max_iter = max_iter;
    st->tol = tol;
    st->done = !(st->normr > tol) || max_iter < 1;
    st->status = 0;
    st->num_iters = 0;
    st->need_norms = 0;
    st->x_pending = 0;
    *mid = *st;
  }
}

// Replay mode scalar kernels (sequential dots, FP64 only) -------------------------
__global__ __launch_bounds__(kBlock) void cg_first_seq_kernel(CgState* st, int64_t n,
                                                              const double* r) {
  __shared__ double buf[kSeqChunk];
  const double rr = dot_sequential(n, r, r, buf);
  if (threadIdx.x == 0) cg_begin_first(st, rr);
}

// End of iteration k, the loop test for k+1 and, only if it passes, the
// sequential r.r of iteration k+1.
__global__ __launch_bounds__(kBlock) void cg_next_seq_kernel(CgState* st, int64_t n,
                                                             const double* r) {
  __shared__ double buf[kSeqChunk];
  __shared__ int go;
  if (threadIdx.x == 0) {
    go = 0;
    if (!st->done) {
      st->x_pending = 1;
      st->alpha_prev = st->alpha;
      st->num_iters = st->k;
      const int k1 = st->k + 1;
      if (!(k1 <= st->max_iter && st->normr > st->tol)) st->done = 1;
      else go = 1;
    }
  }
  __syncthreads();
  if (!go) return;
  const double rr = dot_sequential(n, r, r, buf);
  if (threadIdx.x == 0) {
    st->oldrtrans = st->rtrans;
    st->rtrans = rr;
    st->beta = st->rtrans / st->oldrtrans;
    st->normr = sqrt(st->rtrans);
    st->k = st->k + 1;
  }
}

__global__ __launch_bounds__(kBlock) void cg_alpha_seq_kernel(CgState* st, int64_t n,
                                                              const double* Ap, const double* p,
                                                              double* hist) {
  __shared__ double buf[kSeqChunk];
  __shared__ int need;
  if (st->done) return;
  const double pAp = dot_sequential(n, Ap, p, buf);
  if (threadIdx.x == 0) {
    cg_alpha_or_defer(st, pAp, hist);
    need = st->need_norms;
  }
  __syncthreads();
  if (!need) return;
  const double ApAp = dot_sequential(n, Ap, Ap, buf);
  const double pp = dot_sequential(n, p, p, buf);
  if (threadIdx.x == 0) cg_alpha_after_norms(st, ApAp, pp, hist);
}

// x = 1*x + alpha_prev*p if an x update is pending; then p = 1*r + beta*y
// (y = r for k = 1, y = p afterwards; cg_solve.hpp:153-161, 211).
template <typename T>
__global__ __launch_bounds__(kBlock) void cg_p_kernel(int64_t n, const CgState* st, const T* r,
                                                      const T* y, T* p, T* x) {
  if (st->done) return;
  const T beta = (T)st->beta;
  const T gamma = (T)st->gamma;  // 1 (the reference's waxpby) except after a resume
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (st->x_pending) {
    const T a = (T)st->alpha_prev;
    for (int64_t i = i0; i < n; i += stride) {
      const T pi = p[i];
      // x is not read again until the next iteration's cg_p: stream it past
      // the caches the SpMV's gathers of p are about to use
      __builtin_nontemporal_store(T(1) * x[i] + a * pi, x + i);
      p[i] = gamma * r[i] + beta * (y == p ? pi : y[i]);
    }
  } else {
    for (int64_t i = i0; i < n; i += stride) p[i] = gamma * r[i] + beta * y[i];
  }
}

// After the last iteration: apply the pending x update.
template <typename T>
__global__ __launch_bounds__(kBlock) void cg_finish_kernel(int64_t n, const CgState* st,
                                                           const T* __restrict__ p,
                                                           T* __restrict__ x) {
  if (!st->x_pending) return;
  const T a = (T)st->alpha_prev;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    x[i] = T(1) * x[i] + a * p[i];
}

// r = 1*r + (-alpha)*Ap (cg_solve.hpp:212); with DOT, partials of the new r.r.
template <typename T, bool DOT>
__global__ __launch_bounds__(kBlock) void cg_update_kernel(int64_t n, const CgState* st,
                                                           T* __restrict__ r,
                                                           const T* __restrict__ Ap,
                                                           T* __restrict__ partials) {
  if (st->done) return;
  __shared__ T red[4];
  const T malpha = (T)(-st->alpha);
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  T acc = T(0);
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const T ri = T(1) * r[i] + malpha * Ap[i];
    r[i] = ri;
    if (DOT) acc += ri * ri;
  }
  if (DOT) {
    acc = block_sum<T>(acc, red);
    if (threadIdx.x == 0) partials[blockIdx.x] = acc;
  }
}

// Up to this many groups of kStage SpMV partials, the fast iteration sums
// p.Ap straight from the tile partials in each r-update workgroup (no
// reduce_stage_kernel launch); beyond, from reduce_stage_kernel's group sums.
constexpr int kInlineGroups = 4;

// p.Ap in the order of reduce_stage_kernel + cg_alpha_fast_kernel: the tile
// partials summed in groups of kStage by sum_partials, then the group sums by
// sum_partials.  red2 != nullptr: the group sums are given (ng of them);
// otherwise they are formed here from partials[0, np) (np <= kInlineGroups *
// kStage).  Every workgroup that calls it gets the same bits.
template <typename T>
__device__ T pap_two_stage(const T* partials, int np, const T* red2, int ng, T* red) {
  if (red2) return sum_partials<T>(red2, ng, red);
  __shared__ T grp[kInlineGroups];
  const int ngi = (int)cdiv(np, kStage);
  for (int g = 0; g < ngi; ++g) {
    const T sg = sum_partials<T>(partials + g * kStage, min(kStage, np - g * kStage), red);
    if (threadIdx.x == 0) grp[g] = sg;
  }
  if (ngi == 1) return T(0) + grp[0];  // what the second stage gives (thread 0)
  __syncthreads();
  return sum_partials<T>(grp, ngi, red);
}

// The fast iteration's alpha step folded into the r update: every workgroup
// forms p.Ap (pap_two_stage) and alpha = rtrans / p.Ap itself, workgroup 0
// records them in mid (cg_alpha_or_defer).  p.Ap < 0: breakdown, nothing updated.
// p.Ap < brkdown_tol: the breakdown test's norms are needed; alpha does not
// depend on them (cg_solve.hpp:186-201), so r is updated at once and the
// partials of ||Ap||^2 and ||p||^2 go beside those of r.r for
// advance, which decides before anything else of the iteration
// becomes visible (x is updated only once the iteration has ended, and r is
// internal).  Partials: r.r at out[b], ||Ap||^2 at out[G + b], ||p||^2 at
// out[2G + b] (G = the grid), the same per-workgroup sums as cg_update_kernel
// and cg_norms_kernel.
// PRE: at most kUpdPre elements per thread (small n), whose loads do not depend
// on alpha and are in flight while p.Ap is summed; else a grid-stride loop (for
// which loading ahead measured slower: FP32 at 200^3 136 against 131 us per
// iteration).
constexpr int kUpdPre = 4;
template <typename T, bool PRE>
__global__ __launch_bounds__(kBlock) void cg_update_alpha_kernel(
    int64_t n, const CgState* st, CgState* mid, T* __restrict__ r, const T* __restrict__ Ap, const T* __restrict__ p,
    const T* partials, int np, const T* red2, int ng, double* hist, T* __restrict__ out) {
  __shared__ T red[4];
  __shared__ double s_pap;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  T rv[kUpdPre], av[kUpdPre];
  if (PRE) {
#pragma unroll
    for (int u = 0; u < kUpdPre; ++u) {
      const int64_t i = i0 + u * stride;
      rv[u] = i < n ? r[i] : T(0);
      av[u] = i < n ? Ap[i] : T(0);
    }
  }
  if (st->done) return;
  const double rtrans = st->rtrans, btol = st->brkdown_tol;
  const T pap_t = pap_two_stage<T>(partials, np, red2, ng, red);  // valid in thread 0
  if (threadIdx.x == 0) {
    s_pap = (double)pap_t;
    if (blockIdx.x == 0) {
      CgState c = *st;
      cg_alpha_or_defer(&c, (double)pap_t, hist);
      *mid = c;
    }
  }
  __syncthreads();
  const double pAp = s_pap;
  if (pAp < btol && pAp < 0) return;
  const bool need = pAp < btol;
  const T malpha = (T)(-(rtrans / pAp));
  T acc = T(0);
  if (PRE) {
#pragma unroll
    for (int u = 0; u < kUpdPre; ++u) {
      const int64_t i = i0 + u * stride;
      if (i >= n) break;
      const T ri = T(1) * rv[u] + malpha * av[u];
      r[i] = ri;
      acc += ri * ri;
    }
  } else {
    for (int64_t i = i0; i < n; i += stride) {
      const T ri = T(1) * r[i] + malpha * Ap[i];
      r[i] = ri;
      acc += ri * ri;
    }
  }
  acc = block_sum<T>(acc, red);
  if (threadIdx.x == 0) out[blockIdx.x] = acc;
  if (!need) return;
  const T a = block_sum<T>(grid_dot<T>(n, Ap, Ap), red);
  const T b = block_sum<T>(grid_dot<T>(n, p, p), red);
  if (threadIdx.x == 0) {
    out[gridDim.x + blockIdx.x] = a;
    out[2 * gridDim.x + blockIdx.x] = b;
  }
}

// The scalars an iteration begins with, for every thread of the workgroup.
struct CgBegin {
  double beta, gamma, alpha_prev;
  int done, x_pending, k;
};

// The step from mid (iteration k after its update) to the start of k + 1: the
// breakdown test's norms if they were needed (cg_alpha_after_norms: breakdown
// ends the solve before the iteration counts), then cg_next with r.r.  The
// partials are the G r.r values (then G of ||Ap||^2 and G of ||p||^2) that
// cg_update_alpha_kernel left at out.  Every workgroup gets the same bits; the
// first one records them in st.
template <typename T>
__device__ __forceinline__ CgBegin cg_advance(const CgState* mid, CgState* st, const T* out, int G,
                                              double* hist, T* red) {
  __shared__ CgBegin begin;
  const int need = mid->need_norms;
  const T rr = sum_partials<T>(out, G, red);
  T ApAp = T(0), pp = T(0);
  if (need) {
    ApAp = sum_partials<T>(out + G, G, red);
    pp = sum_partials<T>(out + 2 * G, G, red);
  }
  if (threadIdx.x == 0) {
    CgState s = *mid;
    if (!s.done) {
      if (need) cg_alpha_after_norms(&s, (double)ApAp, (double)pp, hist);
      if (!s.done) cg_next(&s, (double)rr);
    }
    begin = CgBegin{s.beta, s.gamma, s.alpha_prev, s.done, s.x_pending, s.k};
    if (blockIdx.x == 0) *st = s;
  }
  __syncthreads();
  return begin;
}

template <typename T>
__global__ __launch_bounds__(kBlock) void cg_advance_kernel(const CgState* mid, CgState* st,
                                                            const T* out, int G, double* hist) {
  __shared__ T red[4];
  (void)cg_advance<T>(mid, st, out, G, hist, red);
}

// advance and the p update (cg_p_kernel) in one launch, four elements per
// thread; their loads do not depend on the scalars and are in flight while the
// partials are summed.
constexpr int kFoldPer = 4;
template <typename T>
__global__ __launch_bounds__(kBlock) void cg_p_next_kernel(int64_t n, const CgState* mid,
                                                           CgState* st, const T* out, int G,
                                                           double* hist, const T* __restrict__ r,
                                                           T* __restrict__ p, T* __restrict__ x,
                                                           unsigned long long* progress) {
  __shared__ T red[4];
  const int64_t i0 = (int64_t)blockIdx.x * (kBlock * kFoldPer) + threadIdx.x;
  T rv[kFoldPer], pv[kFoldPer], xv[kFoldPer];
#pragma unroll
  for (int u = 0; u < kFoldPer; ++u) {
    const int64_t i = i0 + u * kBlock;
    const bool in = i < n;
    rv[u] = in ? r[i] : T(0);
    pv[u] = in ? p[i] : T(0);
    xv[u] = in ? x[i] : T(0);
  }
  const CgBegin c = cg_advance<T>(mid, st, out, G, hist, red);
  if (blockIdx.x == 0 && threadIdx.x == 0)  // the host reads it from pinned memory
    __hip_atomic_store(progress, (unsigned long long)c.k | ((unsigned long long)(c.done != 0) << 32),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  if (c.done) return;
  const T beta = (T)c.beta, gamma = (T)c.gamma, a = (T)c.alpha_prev;
#pragma unroll
  for (int u = 0; u < kFoldPer; ++u) {
    const int64_t i = i0 + u * kBlock;
    if (i >= n) break;
    if (c.x_pending) x[i] = T(1) * xv[u] + a * pv[u];
    p[i] = gamma * rv[u] + beta * pv[u];
  }
}

// y = A x on stream; *tiles_out = the number of partials written (one per
// 256 rows in the CSR and SELL formats, one per workgroup in the box layout,
// never more than max(kVecBlocks, one per 256 rows)).
template <typename T, bool ZERO_Y, int MODE>
static int launch_spmv(const SpmvOp<T>& op, const T* x, T* y, const T* bvec, T* partials,
                       const int* done, hipStream_t stream, int* tiles_out) {
  const int n = op.n;
  if (n == 0) {
    if (tiles_out) *tiles_out = 0;
    return 0;
  }
  const int64_t cap = std::max<int64_t>(kVecBlocks, cdiv(n, kSpmvRows));
  if (op.symu) {
    BoxGeom g = op.bg;
    {
      if (op.pack) {
        auto run = [&](auto kern) {
          box_chunks(g, sym_slots(sizeof(T) == 8, op.pack, !ZERO_Y && op.wpack, op.cus), cap);
          const int groups = g.nbx * g.nby * g.nzc;
          kern<<<groups, kBlock, 0, stream>>>(g, op.symu, op.symw, op.symtab, x, y, bvec,
                                               partials, done, op.pw, op.pkq, op.wpw, op.wkq,
                                               op.wpack);
          if (tiles_out) *tiles_out = groups;
          return (int)hipGetLastError();
        };
        return with_pack_form<T>(op.pack, [&](auto pf) {
          // The packed boundary stream only where it was measured faster: FP64
          // without ZERO_Y (the CG's kernel) on matrices that the 256 MB of
          // last-level cache cannot hold with their vectors; elsewhere its decode
          // costs more than the bytes it saves (packed against full: 300^3 309
          // and 324 us, 200^3 100 and 100, 128^3 36.6 and 34.2, 64^3 12.4 and
          // 11.0; matvec_std at 300^3 385 and 371).
          if constexpr (!ZERO_Y && std::is_same<T, double>::value)
            if (op.wpack && n >= op.wrows) return run(spmv_boxsym_kernel<T, ZERO_Y, MODE, decltype(pf)::value, true>);
          return run(spmv_boxsym_kernel<T, ZERO_Y, MODE, decltype(pf)::value, false>);
        });
      }
    }
    box_chunks(g, sym_slots(sizeof(T) == 8, kPackNone, false, op.cus), cap);
    const int groups = g.nbx * g.nby * g.nzc;
    spmv_boxsym_kernel<T, ZERO_Y, MODE><<<groups, kBlock, 0, stream>>>(
        g, op.symu, op.symw, op.symtab, x, y, bvec, partials, done);
    if (tiles_out) *tiles_out = groups;
    return (int)hipGetLastError();
  }
  if (op.bvals) {
    BoxGeom g = op.bg;
    box_chunks(g, resident_groups((const void*)spmv_box_kernel<T, ZERO_Y, MODE>, op.cus), cap);
    const int groups = g.nbx * g.nby * g.nzc;
    spmv_box_kernel<T, ZERO_Y, MODE><<<groups, kBlock, 0, stream>>>(g, op.bvals, x, y, bvec,
                                                                     partials, done);
    if (tiles_out) *tiles_out = groups;
    return (int)hipGetLastError();
  }
  const int tiles = (int)cdiv(n, kSpmvRows);
  // operands the plan did not prepare (an FP32 CSR copy that was never made):
  // refuse rather than launch on a null array
  if (!op.svals && (!op.vals || !op.ro || !op.cols)) return (int)hipErrorInvalidValue;
  if (op.xl) {
    // padding slots read entry 0, slots past the width of a slice with bases entry lane
    const size_t lds = sizeof(T) * (size_t)std::max(op.xmaxu, kSlice);
    spmv_sellx_kernel<T, ZERO_Y, MODE><<<tiles, kBlock, lds, stream>>>(
        n, op.nslices, op.soff, op.slen, op.xl, op.xltail, op.xaff, op.xsbase, op.svals, op.xroff,
        op.xrcol, op.xrpos, op.xnu, x, y, bvec, partials, done);
  } else if (op.svals) {
    spmv_sell_kernel<T, ZERO_Y, MODE><<<tiles, kBlock, 0, stream>>>(
        n, op.nslices, op.soff, op.slen, op.scols, op.svals, x, y, bvec, partials, done);
  } else if (op.stream_ok) {
    spmv_stream_kernel<T, ZERO_Y, MODE><<<tiles, kBlock, 0, stream>>>(
        n, op.ro, op.cols, op.vals, x, y, bvec, partials, done);
  } else {
    spmv_rowwise_kernel<T, ZERO_Y, MODE><<<tiles, kBlock, 0, stream>>>(
        n, op.ro, op.cols, op.vals, x, y, bvec, partials, done);
  }
  if (tiles_out) *tiles_out = tiles;
  return (int)hipGetLastError();
}

// --------------------------------------------------------- workspace -----

// Attribution of GPU time to the reference's CG timer slots (WAXPY, DOT,
// MATVEC; mytimer.hpp:36-43) with events recorded between kernel groups on
// the solve's stream.  Eager mode only: events cannot split a graph launch.
struct OpTimer {
  std::vector<hipEvent_t> ev;
  std::vector<int> cat;  // slot of the interval that ends at ev[i]
  size_t used = 0;
  hipStream_t s = nullptr;
  bool on = false;
  // The reference's MINIFE_FUSED build (cg_solve.hpp:172-175): the SpMV and
  // its p.Ap sum are one timed operation (MATVECDOT), not MATVEC + DOT.
  bool fused = false;
  ~OpTimer() {
    for (hipEvent_t e : ev) hipEventDestroy(e);
  }
  bool grow(size_t need) {
    while (ev.size() < need) {
      hipEvent_t e;
      if (hipEventCreate(&e) != hipSuccess) return false;
      ev.push_back(e);
      cat.push_back(-1);
    }
    return true;
  }
  void begin(hipStream_t st, bool fused_timing) {
    s = st;
    fused = fused_timing;
    used = 0;
    on = grow(1) && hipEventRecord(ev[0], s) == hipSuccess;
    used = on ? 1 : 0;
  }
  void mark(int slot) {
    if (!on) return;
    if (!grow(used + 1) || hipEventRecord(ev[used], s) != hipSuccess) {
      on = false;
      return;
    }
    cat[used++] = slot;
  }
  void accumulate(double* times) {
    if (!on || used < 2 || hipEventSynchronize(ev[used - 1]) != hipSuccess) return;
    for (size_t i = 1; i < used; ++i) {
      float ms = 0;
      if (hipEventElapsedTime(&ms, ev[i - 1], ev[i]) == hipSuccess && cat[i] >= 0)
        times[cat[i]] += 1e-3 * ms;
    }
    on = false;
  }
};

template <typename T>
struct VecSet {
  int64_t n = -1;
  T *r = nullptr, *p = nullptr, *Ap = nullptr;
  T* partials = nullptr;  // 4 x max(tiles, kVecBlocks)
  int64_t part_base = 0;  // max(tiles, kVecBlocks): the fast iteration's second region
  T* red2 = nullptr;      // ceil(tiles / kStage)
  void release() {
    hipFree(r);
    hipFree(p);
    hipFree(Ap);
    hipFree(partials);
    hipFree(red2);
    r = p = Ap = partials = red2 = nullptr;
    n = -1;
  }
};

template <typename T>
struct GraphSlot {
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  SpmvOp<T> op;           // what the captured SpMVs read
  const T* x = nullptr;   // what the captured p updates write (besides the workspace)
  void drop() {
    if (exec) hipGraphExecDestroy(exec);
    if (graph) hipGraphDestroy(graph);
    exec = nullptr;
    graph = nullptr;
  }
};

struct CgWorkspace {
  VecSet<double> v64;
  VecSet<float> v32;
  float *f_rhs = nullptr, *f_x = nullptr;  // inner system of the mixed solve
  int64_t f_n = -1;
  CgState* st = nullptr;   // as an iteration begins; [1]: mid, after its alpha
  CgState* h_st = nullptr;  // pinned
  unsigned long long* h_progress = nullptr;  // pinned: k, and done in bit 32 (cg_p_next_kernel)
  double* hist = nullptr;
  int64_t hist_cap = 0;
  GraphSlot<double> g64;
  GraphSlot<float> g32;
  OpTimer timer;
};

constexpr int kGraphChunk = 25;  // CG iterations per captured graph

static void ws_free(CgWorkspace* w) {
  w->g64.drop();
  w->g32.drop();
  w->v64.release();
  w->v32.release();
  hipFree(w->f_rhs);
  hipFree(w->f_x);
  hipFree(w->st);
  hipFree(w->hist);
  if (w->h_st) hipHostFree(w->h_st);
  if (w->h_progress) hipHostFree(w->h_progress);
  delete w;
}

template <typename T>
static int vecset_prepare(mfe_ctx* ctx, VecSet<T>& v, int64_t n, GraphSlot<T>& g) {
  if (v.n == n) return MFE_OK;
  g.drop();
  v.release();
  const int64_t tiles = cdiv(n, kSpmvRows);
  const size_t bytes = sizeof(T) * (size_t)(n > 0 ? n : 1);
  MFE_CHECK(ctx, dev_malloc(ctx, &v.r, bytes));
  MFE_CHECK(ctx, dev_malloc(ctx, &v.p, bytes));
  MFE_CHECK(ctx, dev_malloc(ctx, &v.Ap, bytes));
  v.part_base = tiles > kVecBlocks ? tiles : kVecBlocks;
  MFE_CHECK(ctx, dev_malloc(ctx, &v.partials, sizeof(T) * 4 * (size_t)v.part_base));
  const int64_t n2 = cdiv(tiles, kStage) > 0 ? cdiv(tiles, kStage) : 1;
  MFE_CHECK(ctx, dev_malloc(ctx, &v.red2, sizeof(T) * (size_t)n2));
  v.n = n;
  return MFE_OK;
}

static int ws_get(mfe_ctx* ctx, int max_iter, CgWorkspace** out) {
  if (!ctx->cg) ctx->cg = new CgWorkspace();
  CgWorkspace* w = ctx->cg;
  // each by itself: an earlier call may have failed at any of them
  if (!w->st) MFE_CHECK(ctx, dev_malloc(ctx, &w->st, 2 * sizeof(CgState)));
  if (!w->h_st) MFE_CHECK(ctx, hipHostMalloc(&w->h_st, sizeof(CgState), hipHostMallocDefault));
  if (!w->h_progress)
    MFE_CHECK(ctx, hipHostMalloc(&w->h_progress, sizeof(*w->h_progress), hipHostMallocCoherent));
  const int64_t hneed = 4 * (int64_t)(max_iter > 0 ? max_iter : 1);
  if (w->hist_cap < hneed) {
    w->g64.drop();
    w->g32.drop();
    hipFree(w->hist);
    w->hist = nullptr;
    w->hist_cap = 0;
    MFE_CHECK(ctx, dev_malloc(ctx, &w->hist, sizeof(double) * (size_t)hneed));
    w->hist_cap = hneed;
  }
  *out = w;
  return MFE_OK;
}

static unsigned vec_grid(int64_t n) {
  const int64_t b = cdiv(n, kBlock);
  return (unsigned)(b < kVecBlocks ? (b > 0 ? b : 1) : kVecBlocks);
}

// Grids of the FP64 CG's vector kernels.  The p update (no sum) runs one
// element per thread: measured at n = 27.3 M it moves its 40n bytes in 181 us
// this way against 199-222 us for grid-stride loops over 1,024-16,384
// workgroups.  (The FP32 CG of the mixed solve measured faster with the
// 2,048-workgroup grid-stride form for both kernels: 0.917 against 0.947 ms
// per inner iteration at 300^3, so it keeps vec_grid.)
static unsigned stream_grid(int64_t n) {
  const int64_t b = cdiv(n, kBlock);
  return (unsigned)(b > 0 ? b : 1);
}

// The r update (with its r.r partials) is fastest as a grid-stride loop over
// 1,024 workgroups (115 us for 24n bytes at n = 27.3 M; 127-135 us over 2,048-
// 8,192).  The breakdown norms use the same grid, so their partials line up.
constexpr int kUpdBlocks = 1024;
static unsigned upd_grid(int64_t n) {
  const int64_t b = cdiv(n, kBlock);
  return (unsigned)(b < kUpdBlocks ? (b > 0 ? b : 1) : kUpdBlocks);
}

static inline void mark(OpTimer* tm, int slot) {
  if (tm) tm->mark(slot);
}

// One CG iteration of replay mode or of the per-operation timing mode, all
// scalars in st (k = 1 when y_for_p == r, k >= 2 when y_for_p == p).
template <typename T>
static hipError_t enqueue_iteration(const SpmvOp<T>& op, VecSet<T>& v, CgState* st,
                                    double* hist, T* x, const T* y_for_p, bool replay,
                                    hipStream_t s, OpTimer* tm) {
  const int64_t n = v.n;
  constexpr bool kF64 = sizeof(T) == 8;
  const unsigned vg = kF64 ? upd_grid(n) : vec_grid(n);
  cg_p_kernel<T><<<kF64 ? stream_grid(n) : vg, kBlock, 0, s>>>(n, st, v.r, y_for_p, v.p, x);
  mark(tm, MFE_T_WAXPY);
  int tiles = 0;
  const int* done = &st->done;
  const bool fused = tm && tm->fused;
  if constexpr (std::is_same<T, double>::value) {
    if (replay) {
      launch_spmv<double, true, kPlain>(op, v.p, v.Ap, nullptr, nullptr, done, s, &tiles);
      if (!fused) mark(tm, MFE_T_MATVEC);
      cg_alpha_seq_kernel<<<1, kBlock, 0, s>>>(st, n, v.Ap, v.p, hist);
      mark(tm, fused ? MFE_T_MATVECDOT : MFE_T_DOT);
      cg_update_kernel<double, false><<<vg, kBlock, 0, s>>>(n, st, v.r, v.Ap, nullptr);
      mark(tm, MFE_T_WAXPY);
      cg_next_seq_kernel<<<1, kBlock, 0, s>>>(st, n, v.r);
      mark(tm, MFE_T_DOT);
      return hipGetLastError();
    }
  }
  launch_spmv<T, false, kDot>(op, v.p, v.Ap, nullptr, v.partials, done, s, &tiles);
  if (!fused) mark(tm, MFE_T_MATVEC);
  const int nb2 = (int)cdiv(tiles, kStage);
  // Timed per operation: the dot products stay kernels of their own.
  reduce_stage_kernel<T><<<nb2, kBlock, 0, s>>>(v.partials, tiles, 1, v.red2, done);
  cg_alpha_fast_kernel<T><<<1, kBlock, 0, s>>>(st, v.red2, nb2, hist);
  // Fused timing: the breakdown test's norms are untimed, as breakdown()
  // is in the reference (slot -1).
  if (fused) mark(tm, MFE_T_MATVECDOT);
  cg_norms_kernel<T><<<vg, kBlock, 0, s>>>(n, st, v.Ap, v.p, v.partials);
  cg_norms_fin_kernel<T><<<1, kBlock, 0, s>>>(st, v.partials, (int)vg, hist);
  mark(tm, fused ? -1 : MFE_T_DOT);
  cg_update_kernel<T, true><<<vg, kBlock, 0, s>>>(n, st, v.r, v.Ap, v.partials);
  mark(tm, MFE_T_WAXPY);
  cg_next_fast_kernel<T><<<1, kBlock, 0, s>>>(st, v.partials, (int)vg);
  mark(tm, MFE_T_DOT);
  return hipGetLastError();
}

// Rows up to which every workgroup of the p update does the advance step itself
// (cg_p_next_kernel): each reads the r.r partials (8 KB), 4 us of a launch less
// per iteration (100^3 42.0 -> 40.4 us, 200^3 198 -> 194).
constexpr int64_t kFoldRows = 1 << 23;
// Rows up to which the host launches the iterations one by one, following the
// GPU's progress: a captured chunk costs 170 us per solve with new vectors, a
// stop every 25 iterations and empty iterations past the end, as much as the
// launches it saves (30^3 to 1e-10: 1.26 ms against 1.38 captured; 128^3 20.2
// against 19.8, so from there on captured).
constexpr int64_t kEagerRows = 1500000;
// Iterations the host may be ahead of the one the GPU reports to have begun (8
// measured no better, and up to this many run empty past the last one).
constexpr int kFoldAhead = 4;

// One fast CG solve's launches (see the kernels' overview): the same sums in the
// same order as the timing mode's.
template <typename T>
struct FastCg {
  const SpmvOp<T>& op;
  VecSet<T>& v;
  CgState *st, *mid;
  double* hist;
  T* x;
  hipStream_t s;
  unsigned long long* progress;
  static constexpr bool kF64 = sizeof(T) == 8;
  int64_t n() const { return v.n; }
  unsigned ug() const { return kF64 ? upd_grid(v.n) : vec_grid(v.n); }
  T* out() const { return v.partials + v.part_base; }  // past the SpMV's partials

  // p.Ap's first stage where it has one, then the r update (and alpha)
  hipError_t update(int tiles) const {
    const int nb2 = (int)cdiv(tiles, kStage);
    const bool inline_groups = nb2 <= kInlineGroups;
    if (!inline_groups)
      reduce_stage_kernel<T><<<nb2, kBlock, 0, s>>>(v.partials, tiles, 1, v.red2, &st->done);
    auto run = [&](auto kern) {
      kern<<<ug(), kBlock, 0, s>>>(n(), st, mid, v.r, v.Ap, v.p, v.partials, tiles,
                                   inline_groups ? nullptr : v.red2, nb2, hist, out());
    };
    if (n() <= (int64_t)ug() * kBlock * kUpdPre) run(cg_update_alpha_kernel<T, true>);
    else run(cg_update_alpha_kernel<T, false>);
    return hipGetLastError();
  }
  // the solve's first iteration: p from y (r, or the kept p) by the scalars in st
  hipError_t first(const T* y) const {
    cg_p_kernel<T><<<kF64 ? stream_grid(n()) : vec_grid(n()), kBlock, 0, s>>>(n(), st, v.r, y, v.p,
                                                                              x);
    int tiles = 0;
    launch_spmv<T, false, kDot>(op, v.p, v.Ap, nullptr, v.partials, &st->done, s, &tiles);
    return update(tiles);
  }
  // a later one
  hipError_t next() const {
    if (n() <= kFoldRows) {
      cg_p_next_kernel<T><<<(unsigned)cdiv(n(), kBlock * kFoldPer), kBlock, 0, s>>>(
          n(), mid, st, out(), (int)ug(), hist, v.r, v.p, x, progress);
    } else {
      cg_advance_kernel<T><<<1, kBlock, 0, s>>>(mid, st, out(), (int)ug(), hist);
      cg_p_kernel<T><<<kF64 ? stream_grid(n()) : vec_grid(n()), kBlock, 0, s>>>(n(), st, v.r, v.p,
                                                                                v.p, x);
    }
    int tiles = 0;
    launch_spmv<T, false, kDot>(op, v.p, v.Ap, nullptr, v.partials, &st->done, s, &tiles);
    return update(tiles);
  }
  // the scalars after the last iteration
  hipError_t settle() const {
    cg_advance_kernel<T><<<1, kBlock, 0, s>>>(mid, st, out(), (int)ug(), hist);
    return hipGetLastError();
  }
};

// The captured chunk of iterations after the first, kept in slot for the same
// operand and x.
template <typename T, typename F>
static int capture_chunk(mfe_ctx* ctx, const FastCg<T>& f, GraphSlot<T>& slot, F&& enqueue) {
  hipStream_t s = ctx->stream;
  if (slot.exec && slot.op.tie() == f.op.tie() && slot.x == f.x) return MFE_OK;
  slot.drop();
  MFE_CHECK(ctx, hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
  hipError_t ce = enqueue();
  hipGraph_t g = nullptr;
  hipError_t ee = hipStreamEndCapture(s, &g);
  if (ce != hipSuccess) {
    if (g) (void)hipGraphDestroy(g);
    return hip_fail(ctx, ce, "cg capture");
  }
  if (ee != hipSuccess) return hip_fail(ctx, ee, "hipStreamEndCapture");
  slot.graph = g;
  MFE_CHECK(ctx, hipGraphInstantiate(&slot.exec, g, nullptr, nullptr, 0));
  slot.op = f.op;
  slot.x = f.x;
  return MFE_OK;
}

// The iterations after the first, up to number `last`: launched one by one behind
// the GPU's progress word, or in captured chunks.
template <typename T>
static int run_cg_rest(mfe_ctx* ctx, const FastCg<T>& f, int last, bool eager, CgWorkspace* w,
                       GraphSlot<T>& slot) {
  hipStream_t s = ctx->stream;
  if (f.n() <= kEagerRows) {
    volatile unsigned long long* prog = w->h_progress;
    unsigned long long seen = 0;
    for (int k = 2; k <= last && !(seen >> 32); ++k) {
      if (hipError_t e = f.next()) return hip_fail(ctx, e, "cg iteration");
      seen = *prog;
      for (int spin = 0; !(seen >> 32) && (int)(seen & 0xffffffffu) < k - kFoldAhead; seen = *prog)
        if (++spin % (1 << 16) == 0) {  // not for ever: the stream may have failed
          const hipError_t e = hipStreamQuery(s);
          if (e == hipSuccess) break;
          if (e != hipErrorNotReady) return hip_fail(ctx, e, "cg iteration");
        }
    }
    if (hipError_t e = f.settle()) return hip_fail(ctx, e, "cg_advance_kernel");
    return MFE_OK;
  }
  if (eager) {
    for (int k = 2; k <= last; ++k) {
      if (hipError_t e = f.next()) return hip_fail(ctx, e, "cg iteration");
      if (k % kGraphChunk == 0) {
        if (hipError_t e = f.settle()) return hip_fail(ctx, e, "cg_advance_kernel");
        MFE_CHECK(ctx, hipMemcpyAsync(w->h_st, w->st, sizeof(CgState), hipMemcpyDeviceToHost, s));
        MFE_CHECK(ctx, hipStreamSynchronize(s));
        if (w->h_st->done) break;
      }
    }
    if (hipError_t e = f.settle()) return hip_fail(ctx, e, "cg_advance_kernel");
    return MFE_OK;
  }
  const int chunks = (int)cdiv(std::max(last - 1, 0), kGraphChunk);
  if (chunks == 0) {
    if (hipError_t e = f.settle()) return hip_fail(ctx, e, "cg_advance_kernel");
    return MFE_OK;
  }
  if (int st = capture_chunk<T>(ctx, f, slot, [&] {
        hipError_t e = hipSuccess;
        for (int c = 0; c < kGraphChunk && e == hipSuccess; ++c) e = f.next();
        return e == hipSuccess ? f.settle() : e;
      }))
    return st;
  for (int c = 0; c < chunks; ++c) {
    MFE_CHECK(ctx, hipGraphLaunch(slot.exec, s));
    if (c + 1 < chunks) {
      MFE_CHECK(ctx, hipMemcpyAsync(w->h_st, w->st, sizeof(CgState), hipMemcpyDeviceToHost, s));
      MFE_CHECK(ctx, hipStreamSynchronize(s));
      if (w->h_st->done) break;
    }
  }
  return MFE_OK;
}

// The pending x update and the final state in w->h_st.
template <typename T>
static int finish_cg(mfe_ctx* ctx, const FastCg<T>& f, CgWorkspace* w) {
  hipStream_t s = ctx->stream;
  cg_finish_kernel<T><<<stream_grid(f.n()), kBlock, 0, s>>>(f.n(), w->st, f.v.p, f.x);
  MFE_LAUNCHED(ctx, "cg_finish_kernel");
  MFE_CHECK(ctx, hipMemcpyAsync(w->h_st, w->st, sizeof(CgState), hipMemcpyDeviceToHost, s));
  MFE_CHECK(ctx, hipStreamSynchronize(s));
  return MFE_OK;
}

// Unpreconditioned CG (cg_solve.hpp:69-229) on vectors of type T from the
// initial x.  Leaves the final state in w->h_st.
template <typename T>
static int run_cg(mfe_ctx* ctx, const SpmvOp<T>& op, const T* b, T* x, int max_iter,
                  double tol, bool replay, bool eager, CgWorkspace* w, VecSet<T>& v,
                  GraphSlot<T>& slot, double* times = nullptr, bool fused = false) {
  hipStream_t s = ctx->stream;
  const int64_t n = v.n;
  OpTimer* tm = (eager && times) ? &w->timer : nullptr;
  if (tm) tm->begin(s, fused);
  cg_init_kernel<<<1, 1, 0, s>>>(w->st, max_iter, tol);
  MFE_LAUNCHED(ctx, "cg_init_kernel");
  if (n > 0) {
    const unsigned vg = vec_grid(n);
    // p = 1*x + 0*x ; Ap = A p ; r = 1*b + (-1)*Ap ; rtrans = r.r  (cg_solve.hpp:124-136)
    waxpby_kernel<T><<<vg, kBlock, 0, s>>>(n, T(1), x, T(0), x, v.p);
    mark(tm, MFE_T_WAXPY);
    // The reference's Ap starts as a zero vector, so its 0*Ap[row] is +0.0:
    // start the sums at +0.0 instead of reading the workspace.
    int e = launch_spmv<T, false, kPlain>(op, v.p, v.Ap, nullptr, nullptr, nullptr, s, nullptr);
    if (e) return hip_fail(ctx, (hipError_t)e, "cg prologue spmv");
    mark(tm, MFE_T_MATVEC);
    waxpby_kernel<T><<<vg, kBlock, 0, s>>>(n, T(1), b, T(-1), v.Ap, v.r);
    mark(tm, MFE_T_WAXPY);
    bool seq = false;
    if constexpr (std::is_same<T, double>::value) seq = replay;
    if (seq) {
      if constexpr (std::is_same<T, double>::value)
        cg_first_seq_kernel<<<1, kBlock, 0, s>>>(w->st, n, v.r);
    } else {
      dot_partial_kernel<T><<<vg, kBlock, 0, s>>>(n, v.r, v.r, v.partials);
      cg_first_fast_kernel<T><<<1, kBlock, 0, s>>>(w->st, w->st + 1, v.partials, (int)vg);
    }
    mark(tm, MFE_T_DOT);
    MFE_LAUNCHED(ctx, "cg prologue");
    if (!seq && !tm) {
      *w->h_progress = 1;  // nothing that writes it is in flight: every solve ends synchronised
      FastCg<T> f{op, v, w->st, w->st + 1, w->hist, x, s, w->h_progress};
      // Iteration 1: p = 1*r + 0*r.
      if (hipError_t he = f.first(v.r)) return hip_fail(ctx, he, "cg iteration 1");
      if (int st = run_cg_rest<T>(ctx, f, max_iter, eager, w, slot)) return st;
      return finish_cg<T>(ctx, f, w);
    }
    for (int k = 1; k <= max_iter; ++k) {
      hipError_t he =
          enqueue_iteration<T>(op, v, w->st, w->hist, x, k == 1 ? v.r : v.p, replay, s, tm);
      if (he != hipSuccess) return hip_fail(ctx, he, "cg iteration");
      if (k % kGraphChunk == 0) {
        MFE_CHECK(ctx, hipMemcpyAsync(w->h_st, w->st, sizeof(CgState), hipMemcpyDeviceToHost, s));
        MFE_CHECK(ctx, hipStreamSynchronize(s));
        if (w->h_st->done) break;
      }
    }
    cg_finish_kernel<T><<<stream_grid(n), kBlock, 0, s>>>(n, w->st, v.p, x);
    mark(tm, MFE_T_WAXPY);
    MFE_LAUNCHED(ctx, "cg_finish_kernel");
  }
  MFE_CHECK(ctx, hipMemcpyAsync(w->h_st, w->st, sizeof(CgState), hipMemcpyDeviceToHost, s));
  MFE_CHECK(ctx, hipStreamSynchronize(s));
  if (tm) tm->accumulate(times);
  return MFE_OK;
}

// Resume the stopped CG held in w->st with v.r just replaced and x (the
// correction) zeroed by the caller: up to max_iter more iterations to
// ||r|| <= tol.  Uses the same captured chunk as run_cg's k >= 2 iterations.
template <typename T>
static int run_cg_resume(mfe_ctx* ctx, const SpmvOp<T>& op, T* x, int max_iter, double tol,
                         CgWorkspace* w, VecSet<T>& v, GraphSlot<T>& slot) {
  hipStream_t s = ctx->stream;
  const int64_t n = v.n;
  if (n == 0) return MFE_OK;
  const unsigned vg = vec_grid(n);
  FastCg<T> f{op, v, w->st, w->st + 1, w->hist, x, s, w->h_progress};
  *w->h_progress = 1;
  dot_partial_kernel<T><<<vg, kBlock, 0, s>>>(n, v.r, v.r, v.partials);
  dot_partial_kernel<T><<<vg, kBlock, 0, s>>>(n, v.r, v.p, v.partials + vg);
  cg_resume_kernel<T><<<1, kBlock, 0, s>>>(w->st, w->st + 1, v.partials, (int)vg, max_iter, tol);
  MFE_LAUNCHED(ctx, "cg_resume_kernel");
  if (hipError_t he = f.first(v.p)) return hip_fail(ctx, he, "cg iteration 1");
  if (int st = run_cg_rest<T>(ctx, f, max_iter, false, w, slot)) return st;
  return finish_cg<T>(ctx, f, w);
}

// ---- allocation-free SpMV + dot ---------------------------------------------
//
// mfe_matvec_and_dot_noalloc keeps its per-tile partials in `scratch`, a
// file-scope device array of kScratchPartials doubles (1 MiB, one per 256-row
// tile: matrices up to 33,554,432 rows), instead of the context's partial
// buffer that mfe_matvec_and_dot grows with hipMalloc.  Each GPU holds its own
// copy at its own address, looked up once per device by
// noalloc_scratch_init (called by mfe_ctx_create with the device current);
// host code only ever passes that looked-up address, never the array's name.
// Calls on one GPU share the array: calls that overlap on one GPU (two
// contexts' streams) race.  Every launch writes all the partials it later
// reads, so nothing needs clearing between calls.
constexpr int64_t kScratchPartials = int64_t(1) << 17;
constexpr int kScratchDevices = 64;
static __device__ __align__(256) double scratch[kScratchPartials];
static std::mutex g_scratch_mu;
static double* g_scratch_dev[kScratchDevices];  // per-device address of `scratch`

int noalloc_scratch_init(mfe_ctx* ctx) {
  if (ctx->device < 0 || ctx->device >= kScratchDevices)
    return fail(ctx, MFE_UNSUPPORTED, "device index beyond the scratch table");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_dev[ctx->device]) return MFE_OK;
  void* ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr) return hip_fail(ctx, e, "hipGetSymbolAddress(scratch)");
  g_scratch_dev[ctx->device] = static_cast<double*>(ptr);
  return MFE_OK;
}

static double* scratch_of(const mfe_ctx* ctx) {
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  return g_scratch_dev[ctx->device];
}

// True when ensure_plan(ctx, A, true, false) has nothing left to build, i.e.
// an FP64 SpMV on A launches without allocating.
static bool plan_ready64(const mfe_csr* A) {
  if (A->nrows == 0) return true;
  if (box_applies(A) && (A->box_vals_valid || (A->boxsym_state == 1 && A->boxsym_valid)))
    return true;
  const bool sell_format = A->spmv_format == MFE_SPMV_AUTO || A->spmv_format == MFE_SPMV_SELL;
  if (!sell_format) return true;
  if (!A->sell_struct_valid) return false;
  if (!A->sell_ok) return true;
  if (A->spmv_format == MFE_SPMV_AUTO && !A->sellx_valid) return false;
  return A->sell_vals_valid;
}

__global__ void store_zero_kernel(double* out) { *out = 0.0; }

}  // namespace mfe

using namespace mfe;

extern "C" {

void mfe_cg_workspace_free(mfe_ctx* ctx) {
  if (ctx && ctx->cg) {
    ws_free(ctx->cg);
    ctx->cg = nullptr;
  }
}

static int check_vec(mfe_ctx* ctx, const mfe_vec* v, int64_t n, const char* what) {
  if (!v || v->n != n) return fail(ctx, MFE_BAD_ARG, std::string(what) + ": length mismatch");
  uses(ctx, v);
  return MFE_OK;
}

static int ensure_partials(mfe_ctx* ctx, int64_t count) {
  if ((int64_t)ctx->partials_cap >= count) return MFE_OK;
  hipFree(ctx->d_partials);
  ctx->d_partials = nullptr;
  ctx->partials_cap = 0;
  MFE_CHECK(ctx, dev_malloc(ctx, &ctx->d_partials, sizeof(double) * (size_t)count));
  ctx->partials_cap = (size_t)count;
  return MFE_OK;
}

static int read_scalar(mfe_ctx* ctx, const double* d, double* out) {
  MFE_CHECK(ctx, hipMemcpyAsync(ctx->h_scalars, d, sizeof(double), hipMemcpyDeviceToHost,
                                ctx->stream));
  MFE_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  *out = ctx->h_scalars[0];
  return MFE_OK;
}

int mfe_spmv_plan(mfe_ctx* ctx, mfe_csr* A, int format, int64_t info[8]) {
  if (!ctx || !A || (format != MFE_SPMV_AUTO && format != MFE_SPMV_CSR && format != MFE_SPMV_SELL))
    return MFE_BAD_ARG;
  uses(ctx, A);
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  if (format != A->spmv_format) {
    MFE_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    sell_release(A);
    box_release(A);
    A->spmv_format = format;
  }
  int st;
  if ((st = ensure_plan(ctx, A, true, false))) return st;
  if (info) {
    const SpmvOp<double> op = spmv_op<double>(A);
    if (op.bvals || op.symu) {  // box layout: stored entries; the CG kernel's launch
      BoxGeom g = op.bg;
      const int slots = op.symu ? sym_slots(true, op.pack, op.wpack != kPackNone, op.cus)
                                : resident_groups((const void*)spmv_box_kernel<double, false, kDot>,
                                                  op.cus);
      box_chunks(g, slots, std::max<int64_t>(kVecBlocks, cdiv(A->nrows, kSpmvRows)));
      info[0] = op.pack ? 6 : op.symu ? 5 : 4;
      info[1] = op.symu ? sym_entries(g) + sym_bnd_entries(g) : box_entries(g);
      info[2] = (int64_t)g.nbx * g.nby * g.nzc;
      // 6: the packed forms (PackForm), FP64 in bits 0-7 and FP32 (once built) in 8-15
      info[3] = op.pack ? (int64_t)op.pack |
                              ((int64_t)(A->boxpack32_valid ? A->boxpack32_form : 0) << 8) |
                              ((int64_t)op.wpack << 16)
                        : 27;
      info[4] = g.zc;
      info[5] = g.nbx;
      info[6] = g.nby;
      info[7] = g.nzc;
      return MFE_OK;
    }
    info[0] = op.xl ? 3 : op.svals ? 1 : (op.stream_ok ? 0 : 2);
    info[1] = op.svals ? A->sell_slots : A->nnz;
    info[2] = op.svals ? A->sell_nslices : cdiv(A->nrows, kSpmvRows);
    int64_t longest = A->sell_max_len;
    if (!A->sell_struct_valid) {  // CSR-only plan: measure on the host
      std::vector<int> ro((size_t)A->nrows + 1);
      MFE_CHECK(ctx, hipMemcpyAsync(ro.data(), A->row_offsets, sizeof(int) * ro.size(),
                                    hipMemcpyDeviceToHost, ctx->stream));
      MFE_CHECK(ctx, hipStreamSynchronize(ctx->stream));
      longest = 0;
      for (int64_t r = 0; r < A->nrows; ++r) longest = std::max<int64_t>(longest, ro[r + 1] - ro[r]);
    }
    info[3] = longest;
    info[4] = op.xl ? A->sellx_runs : 0;
    info[5] = op.xl ? A->sellx_maxu : 0;
    info[6] = op.xl ? A->sellx_explicit : 0;
    info[7] = op.xl ? A->sellx_affine : 0;
  }
  MFE_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  return MFE_OK;
}

int mfe_matvec(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* x, mfe_vec* y) {
  if (!ctx || !A) return MFE_BAD_ARG;
  uses(ctx, A);
  int st;
  if ((st = check_vec(ctx, x, A->nrows, "matvec x")) || (st = check_vec(ctx, y, A->nrows, "matvec y")))
    return st;
  if ((st = ensure_plan(ctx, A, true, false))) return st;
  int e = launch_spmv<double, true, kPlain>(spmv_op<double>(A), x->d, y->d, nullptr, nullptr,
                                            nullptr, ctx->stream, nullptr);
  if (e) return hip_fail(ctx, (hipError_t)e, "spmv");
  return MFE_OK;
}

int mfe_matvec_and_dot(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* x, mfe_vec* y,
                       double* result) {
  if (!ctx || !A || !result) return MFE_BAD_ARG;
  uses(ctx, A);
  int st;
  if ((st = check_vec(ctx, x, A->nrows, "matvec x")) || (st = check_vec(ctx, y, A->nrows, "matvec y")))
    return st;
  const int64_t tiles = cdiv(A->nrows, kSpmvRows);
  if ((st = ensure_partials(ctx, std::max<int64_t>(tiles, kVecBlocks)))) return st;
  if ((st = ensure_plan(ctx, A, true, false))) return st;
  int nt = 0;
  int e = launch_spmv<double, true, kDot>(spmv_op<double>(A), x->d, y->d, nullptr,
                                          ctx->d_partials, nullptr, ctx->stream, &nt);
  if (e) return hip_fail(ctx, (hipError_t)e, "spmv_dot");
  if (nt == 0) {
    *result = 0;
    return MFE_OK;
  }
  finalize_kernel<<<1, kBlock, 0, ctx->stream>>>(ctx->d_partials, nt, 1, ctx->d_scalars);
  MFE_LAUNCHED(ctx, "finalize_kernel");
  return read_scalar(ctx, ctx->d_scalars, result);
}

int mfe_matvec_and_dot_noalloc(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* x, mfe_vec* y,
                               double* result_device) {
  if (!ctx || !A || !result_device) return MFE_BAD_ARG;
  uses(ctx, A);
  int st;
  if ((st = check_vec(ctx, x, A->nrows, "matvec x")) || (st = check_vec(ctx, y, A->nrows, "matvec y")))
    return st;
  const int64_t tiles = cdiv(A->nrows, kSpmvRows);
  if (tiles > kScratchPartials)
    return fail(ctx, MFE_BAD_ARG,
                "matvec_and_dot_noalloc: more than 33,554,432 rows (the scratch holds one "
                "partial per 256 rows, 131,072 in all)");
  if (!plan_ready64(A))
    return fail(ctx, MFE_BAD_ARG,
                "matvec_and_dot_noalloc: the matrix's SpMV plan is not built; call "
                "mfe_spmv_plan (or any SpMV) after the last change of the matrix");
  double* part = scratch_of(ctx);
  if (!part) return fail(ctx, MFE_HIP_ERROR, "matvec_and_dot_noalloc: scratch not set up");
  int nt = 0;
  int e = launch_spmv<double, true, kDot>(spmv_op<double>(A), x->d, y->d, nullptr, part, nullptr,
                                          ctx->stream, &nt);
  if (e) return hip_fail(ctx, (hipError_t)e, "spmv_dot (noalloc)");
  if (nt == 0) {
    store_zero_kernel<<<1, 1, 0, ctx->stream>>>(result_device);
    MFE_LAUNCHED(ctx, "store_zero_kernel");
    return MFE_OK;
  }
  finalize_kernel<<<1, kBlock, 0, ctx->stream>>>(part, nt, 1, result_device);
  MFE_LAUNCHED(ctx, "finalize_kernel (noalloc)");
  return MFE_OK;
}

int mfe_matvec_fp32(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* x, mfe_vec* y) {
  if (!ctx || !A) return MFE_BAD_ARG;
  uses(ctx, A);
  int st;
  if ((st = check_vec(ctx, x, A->nrows, "matvec x")) || (st = check_vec(ctx, y, A->nrows, "matvec y")))
    return st;
  const int64_t n = A->nrows;
  if (n == 0) return MFE_OK;
  CgWorkspace* w = nullptr;
  if ((st = ws_get(ctx, 1, &w)) || (st = vecset_prepare<float>(ctx, w->v32, n, w->g32))) return st;
  if ((st = ensure_plan(ctx, A, false, true))) return st;
  const unsigned vg = vec_grid(n);
  to_f32_kernel<<<vg, kBlock, 0, ctx->stream>>>(n, x->d, 1.0, w->v32.p);
  int e = launch_spmv<float, false, kPlain>(spmv_op<float>(A), w->v32.p, w->v32.Ap, nullptr,
                                            nullptr, nullptr, ctx->stream, nullptr);
  if (e) return hip_fail(ctx, (hipError_t)e, "spmv fp32");
  to_f64_kernel<<<vg, kBlock, 0, ctx->stream>>>(n, w->v32.Ap, y->d);
  MFE_LAUNCHED(ctx, "to_f64_kernel");
  return MFE_OK;
}

int mfe_time_matvec(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* x, mfe_vec* y, int variant,
                    int reps, double* avg_ms) {
  if (!ctx || !A || !avg_ms || reps <= 0 || variant < 0 || variant > 13) return MFE_BAD_ARG;
  uses(ctx, A);
  int st;
  if ((st = check_vec(ctx, x, A->nrows, "matvec x")) || (st = check_vec(ctx, y, A->nrows, "matvec y")))
    return st;
  const int64_t n = A->nrows;
  const int64_t tiles = cdiv(n, kSpmvRows);
  if ((st = ensure_partials(ctx, std::max<int64_t>(tiles, kVecBlocks)))) return st;
  const bool f32 = variant == 2 || variant == 4 || variant == 8 || variant == 10 || variant == 12;
  const bool csr_only = variant == 3 || variant == 4;
  // variants 7, 8: variants 1, 2 on the SELL/staged-x plan where the box
  // layout applies (built for the comparison); 9, 10: on the box layout with
  // all 27 slots stored where the symmetric one applies
  const bool no_box = variant == 7 || variant == 8;
  const bool no_sym = variant == 9 || variant == 10;
  // variants 11, 12: variants 1, 2 on the symmetric layout's full values
  // where their 16-bit form is used
  const bool no_pack = variant == 11 || variant == 12;
  // variant 5: variant 1 with the CG's done flag (clear), as inside the solve
  const int* done = nullptr;
  if (variant == 5) {
    int* d = reinterpret_cast<int*>(ctx->d_scalars + 8);
    MFE_CHECK(ctx, hipMemsetAsync(d, 0, sizeof(int), ctx->stream));
    done = d;
  }
  if ((st = ensure_plan(ctx, A, !f32, f32, !no_box && variant != 6))) return st;
  if (no_sym && box_applies(A)) {
    mfe_csr* Am = const_cast<mfe_csr*>(A);
    box_set_geometry(Am);
    if (!f32 && !A->box_vals_valid && (st = build_box<double>(ctx, Am))) return st;
    if (f32 && !A->box_vals32_valid && (st = build_box<float>(ctx, Am))) return st;
  }
  // variant 6: variant 1 on the SELL kernel without the staged x; variant 13:
  // variant 1 on the packed boundary stream however few rows there are
  SpmvOp<double> op64 = spmv_op<double>(A, !csr_only, variant != 6, !no_box, !no_sym, !no_pack);
  if (variant == 13) op64.wrows = 0;
  SpmvOp<float> op32 = spmv_op<float>(A, !csr_only, true, !no_box, !no_sym, !no_pack);
  CgWorkspace* w = nullptr;
  if (f32) {
    if ((st = ws_get(ctx, 1, &w)) || (st = vecset_prepare<float>(ctx, w->v32, n, w->g32))) return st;
    if (csr_only && !A->vals32_valid) {  // CSR FP32 copy for the comparison run
      mfe_csr* Am = const_cast<mfe_csr*>(A);
      const int keep = Am->spmv_format;
      Am->spmv_format = MFE_SPMV_CSR;
      st = ensure_plan(ctx, Am, false, true);
      Am->spmv_format = keep;
      if (st) return st;
      op32 = spmv_op<float>(A, false);
    }
    to_f32_kernel<<<vec_grid(n), kBlock, 0, ctx->stream>>>(n, x->d, 1.0, w->v32.p);
    MFE_LAUNCHED(ctx, "to_f32_kernel");
  }
  MFE_CHECK(ctx, hipEventRecord(ctx->t_start, ctx->stream));
  for (int i = 0; i < reps; ++i) {
    int e;
    if (variant == 0)
      e = launch_spmv<double, true, kPlain>(op64, x->d, y->d, nullptr, nullptr, nullptr,
                                            ctx->stream, nullptr);
    else if (!f32)
      e = launch_spmv<double, false, kDot>(op64, x->d, y->d, nullptr, ctx->d_partials, done,
                                           ctx->stream, nullptr);
    else
      e = launch_spmv<float, false, kDot>(op32, w->v32.p, w->v32.Ap, nullptr, w->v32.partials,
                                          nullptr, ctx->stream, nullptr);
    if (e) return hip_fail(ctx, (hipError_t)e, "spmv");
  }
  MFE_CHECK(ctx, hipEventRecord(ctx->t_stop, ctx->stream));
  MFE_CHECK(ctx, hipEventSynchronize(ctx->t_stop));
  float ms = 0;
  MFE_CHECK(ctx, hipEventElapsedTime(&ms, ctx->t_start, ctx->t_stop));
  *avg_ms = (double)ms / reps;
  return MFE_OK;
}

int mfe_dot(mfe_ctx* ctx, const mfe_vec* x, const mfe_vec* y, double* result) {
  if (!ctx || !x || !y || !result) return MFE_BAD_ARG;
  uses(ctx, x, y);
  if (y->n < x->n) return fail(ctx, MFE_BAD_ARG, "dot: y shorter than x");
  const int64_t n = x->n;
  const unsigned g = vec_grid(n);
  int st;
  if ((st = ensure_partials(ctx, g))) return st;
  dot_partial_kernel<double><<<g, kBlock, 0, ctx->stream>>>(n, x->d, y->d, ctx->d_partials);
  MFE_LAUNCHED(ctx, "dot_partial_kernel");
  finalize_kernel<<<1, kBlock, 0, ctx->stream>>>(ctx->d_partials, (int)g, 1, ctx->d_scalars);
  MFE_LAUNCHED(ctx, "finalize_kernel");
  return read_scalar(ctx, ctx->d_scalars, result);
}

int mfe_dot_replay(mfe_ctx* ctx, const mfe_vec* x, const mfe_vec* y, double* result) {
  if (!ctx || !x || !y || !result) return MFE_BAD_ARG;
  uses(ctx, x, y);
  if (y->n < x->n) return fail(ctx, MFE_BAD_ARG, "dot: y shorter than x");
  dot_seq_kernel<<<1, kBlock, 0, ctx->stream>>>(x->n, x->d, y->d, ctx->d_scalars);
  MFE_LAUNCHED(ctx, "dot_seq_kernel");
  return read_scalar(ctx, ctx->d_scalars, result);
}

int mfe_waxpby(mfe_ctx* ctx, double alpha, const mfe_vec* x, double beta, const mfe_vec* y,
               mfe_vec* w) {
  if (!ctx || !x || !y || !w) return MFE_BAD_ARG;
  uses(ctx, x, y, w);
  if (y->n < x->n || w->n < x->n) return fail(ctx, MFE_BAD_ARG, "waxpby: y and w must be at least as long as x");
  if (x->n == 0) return MFE_OK;
  waxpby_kernel<double><<<vec_grid(x->n), kBlock, 0, ctx->stream>>>(x->n, alpha, x->d, beta, y->d,
                                                                    w->d);
  MFE_LAUNCHED(ctx, "waxpby_kernel");
  return MFE_OK;
}

int mfe_cg_solve(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* b, mfe_vec* x, int max_iter,
                 double tolerance, unsigned flags, int* num_iters, double* normr,
                 double* times, double* history) {
  if (!ctx || !A || !num_iters || !normr) return MFE_BAD_ARG;
  uses(ctx, A);
  if (!A->has_local_indices)
    return fail(ctx, MFE_NOT_LOCAL,
                "cg_solve: A.has_local_indices is false; call make_local_matrix(A) first");
  const int64_t n = A->nrows;
  int st;
  if ((st = check_vec(ctx, b, n, "cg b")) || (st = check_vec(ctx, x, n, "cg x"))) return st;
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  const bool replay = (flags & MFE_CG_REPLAY) != 0;
  const bool eager = (flags & MFE_CG_EAGER) != 0;

  double tol = tolerance;
  if (flags & MFE_CG_TOL_RELATIVE) {
    double bb = 0;
    if ((st = mfe_dot(ctx, b, b, &bb))) return st;
    tol = tolerance * std::sqrt(bb);
  }
  CgWorkspace* w = nullptr;
  if ((st = ws_get(ctx, max_iter, &w)) || (st = vecset_prepare<double>(ctx, w->v64, n, w->g64)))
    return st;
  *num_iters = 0;
  double op_times[5] = {0, 0, 0, 0, 0};
  MFE_CHECK(ctx, hipEventRecord(ctx->t_start, ctx->stream));
  if ((st = ensure_plan(ctx, A, true, false))) return st;
  st = run_cg<double>(ctx, spmv_op<double>(A), b->d, x->d, max_iter, tol, replay, eager, w,
                      w->v64, w->g64, times ? op_times : nullptr,
                      (flags & MFE_CG_FUSED) != 0);
  if (st) return st;
  MFE_CHECK(ctx, hipEventRecord(ctx->t_stop, ctx->stream));
  MFE_CHECK(ctx, hipEventSynchronize(ctx->t_stop));
  const CgState hs = *w->h_st;
  *num_iters = hs.num_iters;
  *normr = hs.normr;
  if (times) {
    float ms = 0;
    MFE_CHECK(ctx, hipEventElapsedTime(&ms, ctx->t_start, ctx->t_stop));
    for (int i = 0; i < 5; ++i) times[i] = op_times[i];
    times[MFE_T_TOTAL] = 1e-3 * ms;
  }
  const int rows = hs.num_iters + (hs.status == MFE_BREAKDOWN ? 1 : 0);
  if (history && rows > 0) {
    MFE_CHECK(ctx, hipMemcpy(history, w->hist, sizeof(double) * 4 * (size_t)rows,
                             hipMemcpyDeviceToHost));
  }
  return hs.status == MFE_BREAKDOWN ? MFE_BREAKDOWN : MFE_OK;
}

int mfe_cg_solve_mixed_ex(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* b, mfe_vec* x,
                          int max_outer, int max_inner, double inner_tol, double outer_tol,
                          unsigned flags, int* outer_iters, int* inner_iters,
                          double* rel_residual, double* times) {
  if (!ctx || !A || !outer_iters || !inner_iters || !rel_residual || max_outer < 0 || max_inner < 0)
    return MFE_BAD_ARG;
  uses(ctx, A);
  const bool keep = (flags & MFE_MIXED_KEEP_DIRECTION) != 0;
  if (!A->has_local_indices)
    return fail(ctx, MFE_NOT_LOCAL,
                "cg_solve_mixed: A.has_local_indices is false; call make_local_matrix(A) first");
  const int64_t n = A->nrows;
  int st;
  if ((st = check_vec(ctx, b, n, "cg b")) || (st = check_vec(ctx, x, n, "cg x"))) return st;
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  hipStream_t s = ctx->stream;
  *outer_iters = 0;
  *inner_iters = 0;
  *rel_residual = 0;
  CgWorkspace* w = nullptr;
  if ((st = ws_get(ctx, max_inner, &w)) || (st = vecset_prepare<double>(ctx, w->v64, n, w->g64)) ||
      (st = vecset_prepare<float>(ctx, w->v32, n, w->g32)))
    return st;
  if (w->f_n != n) {
    hipFree(w->f_rhs);
    hipFree(w->f_x);
    w->f_rhs = w->f_x = nullptr;
    w->f_n = -1;
    w->g32.drop();
    MFE_CHECK(ctx, dev_malloc(ctx, &w->f_rhs, sizeof(float) * (size_t)(n > 0 ? n : 1)));
    MFE_CHECK(ctx, dev_malloc(ctx, &w->f_x, sizeof(float) * (size_t)(n > 0 ? n : 1)));
    w->f_n = n;
  }
  MFE_CHECK(ctx, hipEventRecord(ctx->t_start, s));
  if ((st = ensure_plan(ctx, A, true, true))) return st;
  const SpmvOp<double> op64 = spmv_op<double>(A);
  const SpmvOp<float> op32 = spmv_op<float>(A);
  if (n == 0) return MFE_OK;
  const unsigned vg = vec_grid(n);
  double bb = 0;
  if ((st = mfe_dot(ctx, b, b, &bb))) return st;
  const double nb = std::sqrt(bb);
  VecSet<double>& v = w->v64;
  // r = 1*b + (-1)*(A x) in FP64 with the partials of r.r, fused in the SpMV
  // (as many partials as the launch wrote: the layouts group rows differently).
  auto residual = [&](double* rnorm) -> int {
    int tiles = 0;
    int e = launch_spmv<double, false, kResid>(op64, x->d, v.r, b->d, v.partials, nullptr,
                                               s, &tiles);
    if (e) return hip_fail(ctx, (hipError_t)e, "residual spmv");
    finalize_kernel<<<1, kBlock, 0, s>>>(v.partials, tiles, 1, ctx->d_scalars);
    MFE_LAUNCHED(ctx, "finalize_kernel");
    double rr = 0;
    int r2 = read_scalar(ctx, ctx->d_scalars, &rr);
    *rnorm = std::sqrt(rr);
    return r2;
  };
  double rn = 0;
  if ((st = residual(&rn))) return st;
  double rel = nb > 0 ? rn / nb : rn;
  int status = MFE_OK;
  int outer = 0, inner_total = 0;
  while (rel > outer_tol) {
    if (outer >= max_outer) {
      status = MFE_UNSUPPORTED;
      fail(ctx, MFE_UNSUPPORTED, "cg_solve_mixed: not converged within max_outer refinements");
      break;
    }
    // Inner system A d = r / ||r|| in FP32 from d = 0, to inner_tol -- or,
    // when less than that is still needed to reach outer_tol, to a tenth of
    // the remaining reduction (the inner solve's FP32 recursive residual runs
    // ahead of the true one by a small factor).
    const double need = 0.1 * outer_tol / rel;
    const double tol_k = need > inner_tol ? std::min(need, 0.1) : inner_tol;
    // Keeping the direction: the inner system is A d = r itself (no scaling,
    // so the kept p and rtrans stay in the same units), and every refinement
    // after the first resumes the stopped FP32 CG with r replaced by the
    // rounded FP64 residual (reliable updates).
    const double scale = keep ? 1.0 : rn;
    MFE_CHECK(ctx, hipMemsetAsync(w->f_x, 0, sizeof(float) * (size_t)n, s));
    if (keep && outer > 0) {
      to_f32_kernel<<<vg, kBlock, 0, s>>>(n, v.r, 1.0, w->v32.r);
      MFE_LAUNCHED(ctx, "to_f32_kernel");
      if ((st = run_cg_resume<float>(ctx, op32, w->f_x, max_inner, tol_k * rn, w, w->v32, w->g32)))
        return st;
    } else {
      to_f32_kernel<<<vg, kBlock, 0, s>>>(n, v.r, 1.0 / scale, w->f_rhs);
      MFE_LAUNCHED(ctx, "to_f32_kernel");
      if ((st = run_cg<float>(ctx, op32, w->f_rhs, w->f_x, max_inner, tol_k * (keep ? rn : 1.0),
                              false, false, w, w->v32, w->g32)))
        return st;
    }
    const CgState hs = *w->h_st;
    inner_total += hs.num_iters;
    if (hs.num_iters == 0) {
      status = MFE_BREAKDOWN;
      fail(ctx, MFE_BREAKDOWN, "cg_solve_mixed: inner solve made no progress");
      break;
    }
    refine_update_kernel<<<vg, kBlock, 0, s>>>(n, scale, w->f_x, x->d);
    MFE_LAUNCHED(ctx, "refine_update_kernel");
    ++outer;
    if ((st = residual(&rn))) return st;
    rel = nb > 0 ? rn / nb : rn;
    if (hs.status == MFE_BREAKDOWN && rel > outer_tol) {
      status = MFE_BREAKDOWN;
      fail(ctx, MFE_BREAKDOWN, "cg_solve_mixed: inner solve broke down");
      break;
    }
  }
  MFE_CHECK(ctx, hipEventRecord(ctx->t_stop, s));
  MFE_CHECK(ctx, hipEventSynchronize(ctx->t_stop));
  *outer_iters = outer;
  *inner_iters = inner_total;
  *rel_residual = rel;
  if (times) {
    float ms = 0;
    MFE_CHECK(ctx, hipEventElapsedTime(&ms, ctx->t_start, ctx->t_stop));
    for (int i = 0; i < 5; ++i) times[i] = 0;
    times[MFE_T_TOTAL] = 1e-3 * ms;
  }
  return status;
}

int mfe_cg_solve_mixed(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* b, mfe_vec* x,
                       int max_outer, int max_inner, double inner_tol, double outer_tol,
                       int* outer_iters, int* inner_iters, double* rel_residual, double* times) {
  return mfe_cg_solve_mixed_ex(ctx, A, b, x, max_outer, max_inner, inner_tol, outer_tol, 0u,
                               outer_iters, inner_iters, rel_residual, times);
}

}  // extern "C"
