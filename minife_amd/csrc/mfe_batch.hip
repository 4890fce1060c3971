// Batched miniFE: many independent box problems of uneven size, assembled and
// solved by FP64 CG together: every launch works on all problems that are not
// done.
//
// A problem's rows fall into tiles of kBlock rows; a workgroup owns a few
// consecutive tiles of one problem, the same ones in every launch.  The problems
// are laid out with the ones expected to iterate longest first (the largest
// side), so that the launches can end before the first problem of the tail that
// is done.  (Laying a launch over the XCDs in contiguous ranges, so that a problem
// stays within one L2, took 112.5 instead of 110.5 ms at 64 boxes: problems that
// are done leave their XCD idle.)
//
// Per problem (same arithmetic as the single-box path, so the assembled
// operator is bit-identical to the reference's):
//   1. element matrices K_e (k = 1) and source vectors F_e into scratch (SoA);
//   2. one thread per row: the row's entries summed in ascending element id,
//      both Dirichlet passes (u = 0 on bc_rows_0, then u = 1 on bc_rows_1,
//      row-local because the BC sets are faces of the box), stored straight
//      into the problem's SELL-64 slices and, for the CG, in an exact packed
//      form (below); x = 0, r = b;
//   3. CG (cg_solve.hpp:69-229 with the fast, tree-reduced dots), three launches
//      per iteration: the last iteration's x update and the p update, SpMV with
//      p.Ap partials, r update with r.r partials.  Every workgroup sums its
//      problem's partials in the same order, so all of them take the same
//      scalars; the problem's first one writes the state.  The host launches a
//      few iterations ahead of the GPU, which reports the iteration it is in and
//      the problems that are done in pinned words.
//
// Against one cooperative launch whose workgroups each ran their problem's whole
// CG, meeting at problem-local barriers (3.9 us each, and the phases
// of a problem as slow as its slowest workgroup): 64 boxes of 16..96 171 ms, so 110;
// two 150^3 110, so 72; 12 of 20..64 13.1, so 7.2; one 30^3 1.26, so 0.87.

// A row or a column of a Dirichlet face (all six faces are) is the identity's, so
// the operator couples interior nodes only, and an interior row has all its 27
// neighbours.  The CG keeps p = 0 on the faces in the vector that rows gather
// from and a face node's own p in its entry of A p (which equals it), so an
// interior row sums its 27 products without a look at where it lies: the skipped
// terms of a masked sum are the +-0.0 that leave this one unchanged.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <vector>

#include "mfe_common.hpp"
#include "mfe_hex8.hpp"
#include "mfe_pack.hpp"
#include "mfe_sell.hpp"

namespace mfe {

struct BatchProb {
  int Nx, Ny, Nz;  // elements per side
  int n;           // rows = (Nx+1)(Ny+1)(Nz+1)
  int ne;          // elements
  int nslices;     // ceil(n / 64)
  int b0, nb;      // first workgroup, workgroup count
  int tpb, ntiles; // tiles per workgroup and in all
  int64_t row0;    // base of the problem's rows in the vectors
  int64_t soff0;   // base of its nslices+1 slice offsets
  int64_t slot0;   // base of its SELL entries
  int64_t elem0;   // base of its element scratch (44 doubles per element)
  int64_t part0;   // base of its 2*nb partials: nb of r.r, nb of p.Ap
  int64_t tile0;   // index of its first tile's record and packed words
};

// The packed stencil values of a tile (kBlock consecutive rows), interior entries
// of interior rows only.  Slot s of the tile holds base[s] + f q, f a field of
// the form's width, q the largest power of two that divides all of the slot's
// values, base their least: the assembled values of one slot differ by rounding
// only, and both products and sums of the decoding are exact.  Widths needed:
// 8 to 10 bits for boxes of up to about 100 elements a side, 14 to 18 for the
// slots that are analytically zero (a cube's face neighbours, N x N x 2N's edge
// neighbours).  Per row 36, 44 or 68 bytes instead of the 216 that a tile which
// fits no form reads from its SELL slices.
constexpr int kBSlots = 27;
constexpr unsigned kBNear = (1u << 4) | (1u << 10) | (1u << 12) | (1u << 14) | (1u << 16) | (1u << 22);
struct BatchRec {
  double base[kBSlots];
  uint64_t inner[kBlock / kWave];  // the wave's lanes on interior nodes
  unsigned qhi[kBSlots];           // q's high word (the low one is 0)
  int form;                        // BatchForm
};
enum BatchForm { kBFull = 0, kB10 = 1, kB10Near22 = 2, kB20 = 3 };
// Form of bits N per slot, NN for the near ones: the fields follow each other in
// slot order; word w of the tile's row t is at w * kBlock + t.
template <int N, int NN>
struct BatchPack {
  static constexpr int width(int s) { return (kBNear >> s) & 1u ? NN : N; }
  static constexpr int bit(int s) {
    return s * N + __builtin_popcount(kBNear & ((1u << s) - 1u)) * (NN - N);
  }
  static constexpr int words = (kBSlots * N + 6 * (NN - N) + 31) / 32;
};
using BPack10 = BatchPack<10, 10>;      // 9 words
using BPack10N22 = BatchPack<10, 22>;   // 11
using BPack20 = BatchPack<20, 20>;      // 17
constexpr int kBWords = BPack20::words;  // words kept per row of a tile

struct BatchState {  // per problem, zeroed before each solve
  unsigned done_at;    // iteration at which the problem ended; 0: it has not
  int iters, status;   // status: 0 converged or max_iter, 1 breakdown
  int pad;
  double normr, tol, bnorm;
  double alpha;        // of the last complete iteration
  double rtrans[2];    // r.r at the start of iteration k at [k & 1]
  uint64_t t_begin, t_end;  // wall clock of the problem's first workgroup
  // that workgroup's clock ticks per phase: element math, row assembly,
  // x and p update, SpMV, r update
  uint64_t t_phase[5];
};

constexpr int kPPad = 2;    // entries of p before and after the problems' (packed_pair_sum)
constexpr int kUnroll = 4;  // tiles per step of the vector loops
constexpr int kMaxPart = 1024;  // a problem's workgroups (every one sums all partials)
constexpr int kBatchProblemsPerCu = 2;  // more are refused
constexpr unsigned kAhead = 6;  // iterations the host launches ahead of the GPU's

// Sum of a problem's nb partials in a fixed order (the same in every workgroup).
__device__ double sum_partials_all(const double* pp, int nb, double* red) {
  double s = 0.0;
  for (int i = (int)threadIdx.x; i < nb; i += kBlock) s += pp[i];
  const double t = block_sum<double>(s, red);
  __shared__ double s_tot;
  if (threadIdx.x == 0) s_tot = t;
  __syncthreads();
  const double r = s_tot;
  __syncthreads();
  return r;
}

// Assemble row `id` of problem P (element scratch K/F) into acc, apply both
// Dirichlet passes, store it into the SELL slices; returns b[id].
__device__ __forceinline__ double assemble_row(const BatchProb& P, int id, const double* K,
                                               const double* F, const int* soff, int* scols,
                                               double* svals, double (&acc)[kBSlots]) {
  const int Nx = P.Nx, Ny = P.Ny, Nz = P.Nz;
  const int gx = Nx + 1, gy = Ny + 1;
  const int64_t ne = P.ne;
  const int ix = id % gx, iy = (id / gx) % gy, iz = id / (gx * gy);
  const int lox = ix > 0 ? -1 : 0, hix = ix < Nx ? 1 : 0;
  const int loy = iy > 0 ? -1 : 0, hiy = iy < Ny ? 1 : 0;
  const int loz = iz > 0 ? -1 : 0, hiz = iz < Nz ? 1 : 0;
#pragma unroll
  for (int s = 0; s < kBSlots; ++s) acc[s] = 0.0;
  double accb = 0.0;
#pragma unroll
  for (int dz = -1; dz <= 0; ++dz)
#pragma unroll
    for (int dy = -1; dy <= 0; ++dy)
#pragma unroll
      for (int dx = -1; dx <= 0; ++dx) {
        const int ex = ix + dx, ey = iy + dy, ez = iz + dz;
        if (ex < 0 || ex >= Nx || ey < 0 || ey >= Ny || ez < 0 || ez >= Nz) continue;
        const int64_t e = ex + (int64_t)Nx * (ey + (int64_t)Ny * ez);
        const int cx = -dx, cy = -dy, cz = -dz;
        const int li = corner_of(cx, cy, cz);
#pragma unroll
        for (int lj = 0; lj < 8; ++lj) {
          const int s = (corner_z(lj) - cz + 1) * 9 + (corner_y(lj) - cy + 1) * 3 +
                        (corner_x(lj) - cx + 1);
          acc[s] += K[(int64_t)packed(li, lj) * ne + e];
        }
        accb += F[(int64_t)li * ne + e];
      }
  // Dirichlet, pass 0 (value 0) then pass 1 (value 1): impose_dirichlet's
  // row rule (SparseMatrix_functions.hpp:431-480) on this row.
  const bool in0 = ix == 0 || iy == 0 || iz == 0 || iy == gy - 1 || iz == Nz;
  const bool in1 = ix == gx - 1;
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const double value = pass == 0 ? 0.0 : 1.0;
    const bool row_bc = pass == 0 ? in0 : in1;
    double sum = 0.0;
#pragma unroll
    for (int sz = -1; sz <= 1; ++sz)
#pragma unroll
      for (int sy = -1; sy <= 1; ++sy)
#pragma unroll
        for (int sx = -1; sx <= 1; ++sx) {
          const int s = (sz + 1) * 9 + (sy + 1) * 3 + (sx + 1);
          const bool in = sx >= lox && sx <= hix && sy >= loy && sy <= hiy && sz >= loz && sz <= hiz;
          if (!in) continue;
          if (row_bc) {
            acc[s] = (sx == 0 && sy == 0 && sz == 0) ? 1.0 : 0.0;
          } else {
            const int jx = ix + sx, jy = iy + sy, jz = iz + sz;
            const bool col_bc = pass == 0
                                    ? (jx == 0 || jy == 0 || jz == 0 || jy == gy - 1 || jz == Nz)
                                    : (jx == gx - 1);
            if (col_bc) {
              sum += acc[s];
              acc[s] = 0.0;
            }
          }
        }
    if (row_bc)
      accb = value;
    else
      accb -= sum * value;
  }
  // Store in ascending column order into the row's SELL slots; pad the rest.
  const int slice = id / kWave, lane = id % kWave;
  const int o = soff[slice], w = soff[slice + 1] - o;
  const int64_t o64 = P.slot0 + (int64_t)o * kWave;
  int pos = 0;
#pragma unroll
  for (int sz = -1; sz <= 1; ++sz)
#pragma unroll
    for (int sy = -1; sy <= 1; ++sy)
#pragma unroll
      for (int sx = -1; sx <= 1; ++sx) {
        const int s = (sz + 1) * 9 + (sy + 1) * 3 + (sx + 1);
        const bool in = sx >= lox && sx <= hix && sy >= loy && sy <= hiy && sz >= loz && sz <= hiz;
        if (!in) continue;
        const int64_t at = sell_pos(o64, pos, w, lane);
        svals[at] = acc[s];
        scols[at] = (ix + sx) + gx * ((iy + sy) + gy * (iz + sz));
        ++pos;
      }
  for (; pos < w; ++pos) {
    const int64_t at = sell_pos(o64, pos, w, lane);
    svals[at] = 0.0;
    scols[at] = id;
  }
  return accb;
}

// Padding of a row slot past n in the problem's last slice: value 0 and a
// valid column, so the SpMV's unconditional loads and gathers stay in bounds.
__device__ void pad_row(const BatchProb& P, int id, const int* soff, int* scols, double* svals) {
  const int slice = id / kWave, lane = id % kWave;
  const int o = soff[slice], w = soff[slice + 1] - o;
  const int64_t o64 = P.slot0 + (int64_t)o * kWave;
  for (int j = 0; j < w; ++j) {
    const int64_t at = sell_pos(o64, j, w, lane);
    svals[at] = 0.0;
    scols[at] = P.n - 1;
  }
}

// The exponent of the lowest set bit of v (v != 0), as of a value 1.f * 2^e.
__device__ __forceinline__ int low_bit_exponent(double v) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  const int ex = (int)((u >> 52) & 0x7ff);
  const uint64_t m = (u & 0xfffffffffffffull) | (ex ? 1ull << 52 : 0ull);
  return (ex ? ex : 1) - 1075 + __builtin_ctzll(m);
}

// The packed words of form BP of one row: field s = (v[s] - base[s]) / q, exact.
template <typename BP>
__device__ __forceinline__ void pack_row(const double (&v)[kBSlots], const double* base,
                                         const double* inv_q, unsigned* w) {
  unsigned cur = 0;
#pragma unroll
  for (int s = 0; s < kBSlots; ++s) {
    const unsigned f = (unsigned)((v[s] - base[s]) * inv_q[s]);
    const int sh = BP::bit(s) % 32, word = BP::bit(s) / 32;
    cur |= f << sh;
    if (sh + BP::width(s) >= 32) {
      w[(int64_t)word * kBlock] = cur;
      cur = sh + BP::width(s) > 32 ? f >> ((32 - sh) & 31) : 0u;
    }
  }
  if ((BP::bit(kBSlots - 1) + BP::width(kBSlots - 1)) % 32)
    w[(int64_t)(BP::words - 1) * kBlock] = cur;
}

// The record and packed words of one tile from its rows' values (all threads of
// the workgroup; `in`: this thread's row is interior).  pw null: no packed form.
// An interior row's entries in columns on the faces are 0.0 and are skipped by
// the gathered p = 0 as well, so they take no part: any field does.
__device__ __forceinline__ void pack_tile(const BatchProb& P, int id, bool in,
                                          double (&v)[kBSlots], BatchRec* rec, unsigned* pw) {
  __shared__ double lo[kBSlots][kBlock / kWave], hi[kBSlots][kBlock / kWave];
  __shared__ int low[kBSlots][kBlock / kWave];
  __shared__ double base[kBSlots], inv_q[kBSlots];
  __shared__ int bits[kBSlots];
  __shared__ int form_sh;
  const int t = (int)threadIdx.x, lane = t % kWave, wave = t / kWave;
  const uint64_t m = __ballot(in);
  if (lane == 0) rec->inner[wave] = m;
  const int gx = P.Nx + 1, gy = P.Ny + 1;
  const int ix = id % gx, iy = (id / gx) % gy, iz = id / (gx * gy);
  const double inf = __longlong_as_double(0x7ff0000000000000ll);
  unsigned has = 0;  // slots whose column is interior
#pragma unroll
  for (int s = 0; s < kBSlots; ++s) {
    const int jx = ix + s % 3 - 1, jy = iy + (s / 3) % 3 - 1, jz = iz + s / 9 - 1;
    const bool h = in && jx > 0 && jx < P.Nx && jy > 0 && jy < P.Ny && jz > 0 && jz < P.Nz;
    has |= (h ? 1u : 0u) << s;
    double a = h ? v[s] : inf, b = h ? v[s] : -inf;
    int e = h && v[s] != 0.0 ? low_bit_exponent(v[s]) : 4096;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      a = fmin(a, __shfl_xor(a, d));
      b = fmax(b, __shfl_xor(b, d));
      e = min(e, __shfl_xor(e, d));
    }
    if (lane == 0) {
      lo[s][wave] = a;
      hi[s][wave] = b;
      low[s][wave] = e;
    }
  }
  __syncthreads();
  if (t < kBSlots) {
    double a = lo[t][0], b = hi[t][0];
    int e = low[t][0];
#pragma unroll
    for (int w = 1; w < kBlock / kWave; ++w) {
      a = fmin(a, lo[t][w]);
      b = fmax(b, hi[t][w]);
      e = min(e, low[t][w]);
    }
    int need = 0;
    if (a > b) {  // the slot is in no interior row's range
      a = 0.0;
      e = 0;
    } else if (e == 4096) {  // every value is 0.0
      e = 0;
    } else if (!(e > -1000 && e < 900)) {  // 2^e and 2^-e are not both normal
      need = 64;
      e = 0;
    } else {
      const double r = (b - a) * ldexp(1.0, -e);  // too large a range only rounds to one
      need = r <= 1023.0 ? 10 : r <= 1048575.0 ? 20 : r <= 4194303.0 ? 22 : 64;
    }
    const double q = ldexp(1.0, e);
    base[t] = a;
    inv_q[t] = ldexp(1.0, -e);
    bits[t] = need;
    rec->base[t] = a;
    rec->qhi[t] = (unsigned)__double2hiint(q);
  }
  __syncthreads();
  if (t == 0) {
    int all = 0, cube = 0, near = 0;
    for (int s = 0; s < kBSlots; ++s) {
      all = max(all, bits[s]);
      if ((kBNear >> s) & 1u) near = max(near, bits[s]);
      else cube = max(cube, bits[s]);
    }
    const int f = !pw ? kBFull
                      : all <= 10 ? kB10 : cube <= 10 && near <= 22 ? kB10Near22
                                               : all <= 20 ? kB20 : kBFull;
    form_sh = f;
    rec->form = f;
  }
  __syncthreads();
  const int form = form_sh;
  if (form == kBFull) return;
#pragma unroll
  for (int s = 0; s < kBSlots; ++s)
    if (!((has >> s) & 1u)) v[s] = base[s];
  if (form == kB10) pack_row<BPack10>(v, base, inv_q, pw + t);
  else if (form == kB10Near22) pack_row<BPack10N22>(v, base, inv_q, pw + t);
  else pack_row<BPack20>(v, base, inv_q, pw + t);
}

// The 27 entries of p around row `row` of a problem whose planes hold `plane`
// nodes; an unsigned byte offset from a pointer that is the same for every lane
// (rows < 2^29: the matrix alone takes 324 bytes a row).
__device__ __forceinline__ void gather27(const double* pv, int row, int gx, int plane,
                                         double (&xv)[kBSlots]) {
  const unsigned off = 8u * (unsigned)row;
#pragma unroll
  for (int s = 0; s < kBSlots; ++s) {
    const double* q = pv + ((s % 3 - 1) + gx * ((s / 3) % 3 - 1) + (int64_t)plane * (s / 9 - 1));
    xv[s] = *reinterpret_cast<const double*>(reinterpret_cast<const char*>(q) + off);
  }
}

// (A p)[row] of an interior row, its 27 entries in ascending column order, from
// the packed words w of the row's tile.
template <typename BP>
__device__ __forceinline__ double packed_row_sum(const unsigned* __restrict__ w,
                                                 const BatchRec* __restrict__ rec,
                                                 const double* pv, int row, int gx, int plane,
                                                 double* own) {
  unsigned f[BP::words];
#pragma unroll
  for (int i = 0; i < BP::words; ++i) f[i] = w[i * kBlock];
  double xv[kBSlots];
  gather27(pv, row, gx, plane, xv);
  double sum = 0.0;
#pragma unroll
  for (int s = 0; s < kBSlots; ++s) {
    const unsigned u = pack_field(f + BP::bit(s) / 32, BP::width(s), BP::bit(s) % 32);
    const double v = (double)u * __hiloint2double((int)rec->qhi[s], 0) + rec->base[s];
    sum += v * xv[s];
  }
  *own = xv[kBSlots / 2];
  return sum;
}

struct __attribute__((aligned(8))) PairD {
  double a, b;
};

// (A p) of rows `row` and row + 1, each over its 27 entries in ascending column
// order, from the packed words w of row `row` in its tile (row even there).  The
// rows of a line share their neighbours: four entries of p, two loads, serve both.
// A row that is not interior gets a sum that is not used; its neighbour's loads
// reach at most one entry past the problem's rows.
template <typename BP>
__device__ __forceinline__ void packed_pair_sum(const unsigned* __restrict__ w,
                                                const BatchRec* __restrict__ rec,
                                                const double* pv, int row, int gx, int plane,
                                                double (&sum)[2], double (&own)[2]) {
  unsigned f0[BP::words], f1[BP::words];
#pragma unroll
  for (int i = 0; i < BP::words; ++i) {
    const uint2 v = *reinterpret_cast<const uint2*>(w + i * kBlock);
    f0[i] = v.x;
    f1[i] = v.y;
  }
  const unsigned off = 8u * (unsigned)row;
  double x[9][4];
#pragma unroll
  for (int l = 0; l < 9; ++l) {
    const double* q = pv + (gx * (l % 3 - 1) + (int64_t)plane * (l / 3 - 1));
    const PairD lo = *reinterpret_cast<const PairD*>(reinterpret_cast<const char*>(q - 1) + off);
    const PairD hi = *reinterpret_cast<const PairD*>(reinterpret_cast<const char*>(q + 1) + off);
    x[l][0] = lo.a;
    x[l][1] = lo.b;
    x[l][2] = hi.a;
    x[l][3] = hi.b;
  }
  sum[0] = sum[1] = 0.0;
#pragma unroll
  for (int s = 0; s < kBSlots; ++s) {
    const double q = __hiloint2double((int)rec->qhi[s], 0), base = rec->base[s];
    const int at = BP::bit(s) / 32, sh = BP::bit(s) % 32;
    const double v0 = (double)pack_field(f0 + at, BP::width(s), sh) * q + base;
    const double v1 = (double)pack_field(f1 + at, BP::width(s), sh) * q + base;
    sum[0] += v0 * x[s / 3][s % 3];
    sum[1] += v1 * x[s / 3][s % 3 + 1];
  }
  own[0] = x[4][1];
  own[1] = x[4][2];
}

// One row from its SELL values (27 of them: its slice is as wide).
__device__ __forceinline__ double full_row_sum(const BatchProb& P, const int* __restrict__ soff,
                                               const double* __restrict__ svals,
                                               const double* pv, int row, int gx, int plane,
                                               double* own) {
  const int slice = row / kWave, lane = row % kWave;
  const int o = soff[slice], w = soff[slice + 1] - o;
  const int64_t o64 = P.slot0 + (int64_t)o * kWave;
  double v[kBSlots], xv[kBSlots];
#pragma unroll
  for (int s = 0; s < kBSlots; ++s) v[s] = svals[sell_pos(o64, s, w, lane)];
  gather27(pv, row, gx, plane, xv);
  double sum = 0.0;
#pragma unroll
  for (int s = 0; s < kBSlots; ++s) sum += v[s] * xv[s];
  *own = xv[kBSlots / 2];
  return sum;
}

// What a workgroup works on.
struct BatchWg {
  int pi, i;   // problem, index within it
  int t0, t1;  // tiles
};
__device__ __forceinline__ BatchWg batch_wg(const BatchProb* __restrict__ probs,
                                            const int* __restrict__ blk2prob) {
  const int wg = (int)blockIdx.x;
  BatchWg w;
  w.pi = blk2prob[wg];
  const BatchProb& P = probs[w.pi];
  w.i = wg - P.b0;
  w.t0 = w.i * P.tpb;
  w.t1 = min(w.t0 + P.tpb, P.ntiles);
  return w;
}

// Element matrices and source vectors of every problem (Hex8 element math, k = 1).
__global__ __launch_bounds__(kBlock) void batch_elements_kernel(
    const BatchProb* __restrict__ probs, const int* __restrict__ blk2prob, HexTables tab,
    double* KF, BatchState* states) {
  const BatchWg wg = batch_wg(probs, blk2prob);
  const BatchProb P = probs[wg.pi];
  const int i = wg.i, t = (int)threadIdx.x;
  const int64_t ne = P.ne;
  double* K = KF + P.elem0;
  double* F = K + 36 * ne;
  const uint64_t tc = wall_clock64();
  const double hx = 1.0 / P.Nx, hy = 1.0 / P.Ny, hz = 1.0 / P.Nz;
  for (int64_t e = (int64_t)i * kBlock + t; e < ne; e += (int64_t)P.nb * kBlock) {
    const int ex = (int)(e % P.Nx);
    const int ey = (int)((e / P.Nx) % P.Ny);
    const int ez = (int)(e / ((int64_t)P.Nx * P.Ny));
    const double x0 = 1.0 * ex / P.Nx;
    const double y0 = 1.0 * ey / P.Ny;
    const double z0 = (1.0 * ez) / P.Nz;
    const double x1 = x0 + hx, y1 = y0 + hy, z1 = z0 + hz;
    const double c[24] = {x0, y0, z0, x1, y0, z0, x1, y1, z0, x0, y1, z0,
                          x0, y0, z1, x1, y0, z1, x1, y1, z1, x0, y1, z1};
    double Ke[36], Fe[8];
    hex8_element(c, tab, 1.0, Ke, Fe);
#pragma unroll
    for (int q = 0; q < 36; ++q) K[(int64_t)q * ne + e] = Ke[q];
#pragma unroll
    for (int q = 0; q < 8; ++q) F[(int64_t)q * ne + e] = Fe[q];
  }
  if (i == 0 && t == 0) {
    BatchState* st = states + wg.pi;
    st->t_begin = tc;
    st->t_phase[0] = wall_clock64() - tc;
  }
}

// Rows of every problem: gather, Dirichlet, SELL store, packed form; x = 0,
// r = b, p = 0 (the faces keep it), and the partials of b.b.
__global__ __launch_bounds__(kBlock) void batch_rows_kernel(
    const BatchProb* __restrict__ probs, const int* __restrict__ blk2prob,
    const int* __restrict__ soff_all, const double* __restrict__ KF, int* scols, double* svals,
    BatchRec* recs, unsigned* words, double* b, double* x, double* r, double* p,
    double* partials, BatchState* states) {
  __shared__ double red[4];
  const BatchWg wg = batch_wg(probs, blk2prob);
  const BatchProb P = probs[wg.pi];
  const int t = (int)threadIdx.x;
  const double* K = KF + P.elem0;
  const double* F = K + 36 * (int64_t)P.ne;
  const int* soff = soff_all + P.soff0;
  const int gx = P.Nx + 1, gy = P.Ny + 1;
  const uint64_t tc = wall_clock64();
  double acc = 0.0;
  for (int tile = wg.t0; tile < wg.t1; ++tile) {
    const int row = tile * kBlock + t;
    double v[kBSlots];
    bool in = false;
    if (row < P.n) {
      const double bv = assemble_row(P, row, K, F, soff, scols, svals, v);
      const int ix = row % gx, iy = (row / gx) % gy, iz = row / (gx * gy);
      in = ix > 0 && ix < P.Nx && iy > 0 && iy < P.Ny && iz > 0 && iz < P.Nz;
      b[P.row0 + row] = bv;
      x[P.row0 + row] = 0.0;
      r[P.row0 + row] = bv;
      p[P.row0 + row] = 0.0;
      acc += bv * bv;
    } else if (row < P.nslices * kWave) {
      pad_row(P, row, soff, scols, svals);
    }
    pack_tile(P, row, in, v, recs + P.tile0 + tile,
              words ? words + (P.tile0 + tile) * (int64_t)(kBWords * kBlock) : nullptr);
  }
  const double v0 = block_sum<double>(acc, red);
  if (t == 0) partials[P.part0 + wg.i] = v0;
  if (wg.i == 0 && t == 0) states[wg.pi].t_phase[1] = wall_clock64() - tc;
}

// A row's own p: in p on interior nodes, in A p on the faces.
__device__ __forceinline__ double* own_p(const BatchRec* __restrict__ rec, int wave, int lane,
                                         double* pp, double* App) {
  return (rec->inner[wave] >> lane) & 1u ? pp : App;
}

// The problem's first workgroup at its end in iteration k.
__device__ __forceinline__ void batch_end(BatchState* st, int* host, int pi, unsigned k,
                                          double normr, int status) {
  st->done_at = k;
  st->iters = (int)(k - 1);
  st->normr = normr;
  st->status = status;
  st->t_end = wall_clock64();
  __hip_atomic_store(host + 1 + pi, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Start of iteration k: the convergence test, x += alpha p of the iteration
// before, and p = r + beta p unless the problem is done.  x rides along because
// p is read here anyway (40 bytes per row; with x in the r update 24 + 48
// instead of 40 + 24 for the two).  The loads of the first tiles are issued
// before the sum of the partials.
__global__ __launch_bounds__(kBlock) void batch_p_kernel(
    const BatchProb* __restrict__ probs, const int* __restrict__ blk2prob,
    const BatchRec* __restrict__ recs, double* __restrict__ x, const double* __restrict__ r,
    double* p, double* Ap, const double* __restrict__ partials, BatchState* states, int* host,
    unsigned k, int max_iter, double rel_tol) {
  __shared__ double red[4];
  const int t = (int)threadIdx.x;
  if (blockIdx.x == 0 && t == 0)
    __hip_atomic_store(host, (int)k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  const uint64_t tc = wall_clock64();
  const BatchWg wg = batch_wg(probs, blk2prob);
  const BatchProb& P = probs[wg.pi];
  BatchState* st = states + wg.pi;
  // (the first workgroup may be writing done_at = k)
  const unsigned done_at = st->done_at;
  if (done_at && done_at < k) return;
  const int lane = t % kWave, wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const BatchRec* prec = recs + P.tile0;
  const int n = P.n;
  double* xp = x + P.row0;
  const double* rp = r + P.row0;
  double* pp = p + P.row0;
  double* App = Ap + P.row0;
  double rv[kUnroll], pv[kUnroll], xv[kUnroll];
  auto load = [&](int tile) {
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int row = (tile + u) * kBlock + t;
      const bool ok = tile + u < wg.t1 && row < n;
      rv[u] = ok ? rp[row] : 0.0;
      pv[u] = ok && k > 1 ? own_p(prec + tile + u, wave, lane, pp, App)[row] : 0.0;
      xv[u] = ok && k > 1 ? xp[row] : 0.0;
    }
  };
  load(wg.t0);
  const double rtrans = sum_partials_all(partials + P.part0, P.nb, red);
  const double normr = sqrt(rtrans);
  const double tol = k == 1 ? rel_tol * normr : st->tol;
  const double alpha = k == 1 ? 0.0 : st->alpha;
  const double beta = k == 1 ? 0.0 : rtrans / st->rtrans[(k - 1) & 1];
  const bool stop = k > (unsigned)max_iter || !(normr > tol);
  for (int tile = wg.t0; tile < wg.t1;) {
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int row = (tile + u) * kBlock + t;
      if (tile + u < wg.t1 && row < n) {
        if (k > 1) xp[row] = 1.0 * xv[u] + alpha * pv[u];
        if (!stop)
          own_p(prec + tile + u, wave, lane, pp, App)[row] =
              k == 1 ? 1.0 * rv[u] + 0.0 * rv[u] : 1.0 * rv[u] + beta * pv[u];
      }
    }
    tile += kUnroll;
    if (tile < wg.t1) load(tile);
  }
  if (wg.i == 0 && t == 0) {
    st->rtrans[k & 1] = rtrans;
    if (k == 1) {
      st->tol = tol;
      st->bnorm = normr;
    }
    if (stop) batch_end(st, host, wg.pi, k, normr, 0);
    st->t_phase[2] += wall_clock64() - tc;
  }
}

// A p and the partials of p.Ap.  Two 150^3, row by row: 76 bytes per row read (46 of
// packed values and records, p by several XCDs; a cube's form) and 8 written, 4.1
// TB/s, 33 vector memory instructions per 64 rows, waves waiting half their time.
// PAIR: two rows per thread, whose lines share their entries (27 per 128 rows):
// their whole solve 72.2 ms, so 64.4; 64 boxes of 16..96 110.6, so 106.6.
// Workgroups of neighbouring tiles on one XCD (groups of 4 to 64) change nothing.
// For launches of few tiles (one per workgroup) PAIR
// leaves half the waves idle: 12 of 20..64 7.5 ms, row by row 7.2.
// 128 registers (four waves per SIMD): three 108 ms, five 121 (64 boxes).  With p
// staged in LDS, three windows for four tiles at a time, row by row: 115 to 124.
template <bool PAIR>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4, 8))) void batch_spmv_kernel(
    const BatchProb* __restrict__ probs, const int* __restrict__ blk2prob,
    const int* __restrict__ soff_all, const double* __restrict__ svals,
    const BatchRec* __restrict__ recs, const unsigned* __restrict__ words,
    const double* __restrict__ p, double* Ap, double* __restrict__ partials,
    BatchState* states) {
  __shared__ double red[4];
  const uint64_t tc = wall_clock64();
  const BatchWg wg = batch_wg(probs, blk2prob);
  const BatchProb& P = probs[wg.pi];
  BatchState* st = states + wg.pi;
  if (st->done_at) return;
  const int t = (int)threadIdx.x;
  const int lane = t % kWave, wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const int* soff = soff_all + P.soff0;
  const int n = P.n, gx = P.Nx + 1, plane = gx * (P.Ny + 1);
  const double* pp = p + P.row0;
  double* App = Ap + P.row0;
  double acc = 0.0;
  if constexpr (PAIR) {
    // two waves per tile, two rows per thread
    for (int tile = wg.t0 + wave / 2; tile < wg.t1; tile += kBlock / kWave / 2) {
      const int half = wave % 2, row = tile * kBlock + half * 2 * kWave + 2 * lane;
      const BatchRec* rec = recs + P.tile0 + tile;
      const int form = rec->form;
      const uint64_t m0 = rec->inner[2 * half], m1 = rec->inner[2 * half + 1];
      const unsigned in = (unsigned)((lane < kWave / 2 ? m0 : m1) >> (2 * lane % kWave)) & 3u;
      double sum[2], own[2];
      if (in) {
        const unsigned* w = words + (P.tile0 + tile) * (int64_t)(kBWords * kBlock) +
                            (half * 2 * kWave + 2 * lane);
        if (form == kB10) packed_pair_sum<BPack10>(w, rec, pp, row, gx, plane, sum, own);
        else if (form == kB10Near22)
          packed_pair_sum<BPack10N22>(w, rec, pp, row, gx, plane, sum, own);
        else if (form == kB20) packed_pair_sum<BPack20>(w, rec, pp, row, gx, plane, sum, own);
        else {
#pragma unroll
          for (int h = 0; h < 2; ++h)
            if ((in >> h) & 1u) sum[h] = full_row_sum(P, soff, svals, pp, row + h, gx, plane, &own[h]);
        }
      }
      if (in == 3u) {
        *reinterpret_cast<PairD*>(App + row) = PairD{sum[0], sum[1]};
        acc += sum[0] * own[0];
        acc += sum[1] * own[1];
      } else {
#pragma unroll
        for (int h = 0; h < 2; ++h)
          if ((in >> h) & 1u) {
            App[row + h] = sum[h];
            acc += sum[h] * own[h];
          } else if (row + h < n) {
            const double pv = App[row + h];
            acc += pv * pv;
          }
      }
    }
  } else {
    for (int tile = wg.t0; tile < wg.t1; ++tile) {
      const int row = tile * kBlock + t;
      const BatchRec* rec = recs + P.tile0 + tile;
      const int form = rec->form;
      if ((rec->inner[wave] >> lane) & 1u) {
        const unsigned* w = words + (P.tile0 + tile) * (int64_t)(kBWords * kBlock) + t;
        double sum, own;
        if (form == kB10) sum = packed_row_sum<BPack10>(w, rec, pp, row, gx, plane, &own);
        else if (form == kB10Near22)
          sum = packed_row_sum<BPack10N22>(w, rec, pp, row, gx, plane, &own);
        else if (form == kB20) sum = packed_row_sum<BPack20>(w, rec, pp, row, gx, plane, &own);
        else sum = full_row_sum(P, soff, svals, pp, row, gx, plane, &own);
        App[row] = sum;
        acc += sum * own;
      } else if (row < n) {
        const double own = App[row];
        acc += own * own;
      }
    }
  }
  const double v0 = block_sum<double>(acc, red);
  if (t == 0) partials[P.part0 + P.nb + wg.i] = v0;
  if (wg.i == 0 && t == 0) st->t_phase[3] += wall_clock64() - tc;
}

// alpha = r.r / p.Ap, r -= alpha Ap, and the partials of r.r.
__global__ __launch_bounds__(kBlock) void batch_r_kernel(
    const BatchProb* __restrict__ probs, const int* __restrict__ blk2prob,
    double* __restrict__ r, const double* __restrict__ Ap, double* partials, BatchState* states,
    int* host, unsigned k) {
  __shared__ double red[4];
  const uint64_t tc = wall_clock64();
  const BatchWg wg = batch_wg(probs, blk2prob);
  const BatchProb& P = probs[wg.pi];
  BatchState* st = states + wg.pi;
  if (st->done_at) return;  // (also what a breakdown of this iteration may have written)
  const int t = (int)threadIdx.x, n = P.n;
  double* rp = r + P.row0;
  const double* App = Ap + P.row0;
  double rv[kUnroll], av[kUnroll];
  auto load = [&](int tile) {
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int row = (tile + u) * kBlock + t;
      const bool ok = tile + u < wg.t1 && row < n;
      rv[u] = ok ? rp[row] : 0.0;
      av[u] = ok ? App[row] : 0.0;
    }
  };
  load(wg.t0);
  const double pAp = sum_partials_all(partials + P.part0 + P.nb, P.nb, red);
  const double rtrans = st->rtrans[k & 1];
  if (!(pAp > 0.0)) {  // non-positive curvature: the operator is not SPD here
    if (wg.i == 0 && t == 0) batch_end(st, host, wg.pi, k, sqrt(rtrans), 1);
    return;
  }
  const double alpha = rtrans / pAp;
  double acc = 0.0;
  for (int tile = wg.t0; tile < wg.t1;) {
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int row = (tile + u) * kBlock + t;
      if (tile + u < wg.t1 && row < n) {
        const double r1 = 1.0 * rv[u] + (-alpha) * av[u];
        rp[row] = r1;
        acc += r1 * r1;
      }
    }
    tile += kUnroll;
    if (tile < wg.t1) load(tile);
  }
  const double v0 = block_sum<double>(acc, red);
  if (t == 0) partials[P.part0 + wg.i] = v0;
  if (wg.i == 0 && t == 0) {
    st->alpha = alpha;
    st->t_phase[4] += wall_clock64() - tc;
  }
}

}  // namespace mfe

using namespace mfe;

struct mfe_batch {
  mfe_ctx* ctx = nullptr;
  int nprob = 0, grid = 0;
  bool pairs = false;  // the SpMV takes two rows per thread
  double tick_seconds = 1e-8;  // wall clock period
  std::vector<double> last_seconds;  // per problem, previous solve
  std::vector<double> last_phases;   // per problem x 6 phases, previous solve
  std::vector<BatchProb> probs;
  std::vector<int> soff;      // all problems' slice offsets
  std::vector<int> blk2prob;  // problem of each workgroup
  std::vector<int> order;     // the problems as they are laid out
  BatchProb* d_probs = nullptr;
  int* d_blk2prob = nullptr;
  int* d_soff = nullptr;
  int* d_scols = nullptr;
  double* d_svals = nullptr;
  double* d_KF = nullptr;
  BatchRec* d_recs = nullptr;
  unsigned* d_words = nullptr;  // null: every tile reads its SELL slices
  double *d_b = nullptr, *d_x = nullptr, *d_r = nullptr, *d_p = nullptr, *d_Ap = nullptr;
  double* d_part = nullptr;
  BatchState* d_states = nullptr;
  int* h_words = nullptr;  // pinned: the iteration the GPU is in, then a flag per problem
  int64_t rows = 0, slots = 0;
  void release() {
    (void)hipFree(d_probs);
    (void)hipFree(d_blk2prob);
    (void)hipFree(d_soff);
    (void)hipFree(d_scols);
    (void)hipFree(d_svals);
    (void)hipFree(d_KF);
    (void)hipFree(d_recs);
    (void)hipFree(d_words);
    (void)hipFree(d_b);
    (void)hipFree(d_x);
    (void)hipFree(d_r);
    (void)hipFree(d_p ? d_p - kPPad : nullptr);
    (void)hipFree(d_Ap);
    (void)hipFree(d_part);
    (void)hipFree(d_states);
    if (h_words) (void)hipHostFree(h_words);
  }
};

static int host_axis_len(int i, int g) { return 1 + (i > 0) + (i < g - 1); }

// The problems' workgroups: the problems in descending order of their largest
// side.  Up to 4 tiles per workgroup where that still leaves 16 workgroups per CU
// (one step of the vector loops, and fewer partials for each to sum: 64 boxes of
// 16..96 take 112 ms, with 2 tiles 127, with 8 113), more where a problem would
// have more than kMaxPart.
static void batch_layout(mfe_batch* B, int cus) {
  int64_t tiles = 0;
  for (const BatchProb& P : B->probs) tiles += P.ntiles;
  const int least = (int)std::max<int64_t>(1, std::min<int64_t>(kUnroll, tiles / (16 * cus)));
  B->pairs = least >= 2;
  auto side = [&](int q) {
    const BatchProb& P = B->probs[(size_t)q];
    return std::max(P.Nx, std::max(P.Ny, P.Nz));
  };
  B->order.resize((size_t)B->nprob);
  for (int q = 0; q < B->nprob; ++q) B->order[(size_t)q] = q;
  std::stable_sort(B->order.begin(), B->order.end(),
                   [&](int a, int b) { return side(a) > side(b); });
  int64_t part0 = 0;
  for (int q : B->order) {
    BatchProb& P = B->probs[(size_t)q];
    P.tpb = std::max(least, (int)cdiv(P.ntiles, kMaxPart));
    P.b0 = (int)B->blk2prob.size();
    P.nb = (int)cdiv(P.ntiles, P.tpb);
    P.part0 = part0;
    part0 += 2 * (int64_t)P.nb;
    B->blk2prob.insert(B->blk2prob.end(), (size_t)P.nb, q);
  }
  B->grid = (int)B->blk2prob.size();
}

static int batch_upload_layout(mfe_ctx* ctx, mfe_batch* B) {
  hipStream_t s = ctx->stream;
  MFE_CHECK(ctx, hipMemcpyAsync(B->d_probs, B->probs.data(), sizeof(BatchProb) * B->probs.size(),
                                hipMemcpyHostToDevice, s));
  MFE_CHECK(ctx, hipMemcpyAsync(B->d_blk2prob, B->blk2prob.data(),
                                sizeof(int) * B->blk2prob.size(), hipMemcpyHostToDevice, s));
  MFE_CHECK(ctx, hipStreamSynchronize(s));
  return MFE_OK;
}

extern "C" {

int mfe_batch_create(mfe_ctx* ctx, int nprob, const int* dims, mfe_batch** out) {
  if (!ctx || !out || nprob <= 0 || !dims) return MFE_BAD_ARG;
  *out = nullptr;
  for (int q = 0; q < 3 * nprob; ++q)
    if (dims[q] < 1 || dims[q] > 1024)
      return fail(ctx, MFE_BAD_ARG, "batch_create: box sides must be in [1, 1024] elements");
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  if (nprob > kBatchProblemsPerCu * ctx->cu_count)
    return fail(ctx, MFE_UNSUPPORTED, "batch_create: more than two problems per compute unit");
  mfe_batch* B = new mfe_batch();
  B->ctx = ctx;
  B->nprob = nprob;
  // Problem layout and slice widths (closed form: a row's length is the
  // product of its per-axis neighbour counts).
  int64_t row0 = 0, soff0 = 0, slot0 = 0, elem0 = 0, tile0 = 0;
  for (int q = 0; q < nprob; ++q) {
    BatchProb P{};
    P.Nx = dims[3 * q];
    P.Ny = dims[3 * q + 1];
    P.Nz = dims[3 * q + 2];
    const int gx = P.Nx + 1, gy = P.Ny + 1, gz = P.Nz + 1;
    P.n = gx * gy * gz;
    P.ne = P.Nx * P.Ny * P.Nz;
    P.nslices = (int)cdiv(P.n, kWave);
    P.row0 = row0;
    P.soff0 = soff0;
    P.slot0 = slot0;
    P.elem0 = elem0;
    P.tile0 = tile0;
    int acc = 0;
    for (int s = 0; s < P.nslices; ++s) {
      B->soff.push_back(acc);
      int w = 0;
      for (int l = 0; l < kWave; ++l) {
        const int id = s * kWave + l;
        if (id >= P.n) break;
        const int ix = id % gx, iy = (id / gx) % gy, iz = id / (gx * gy);
        w = std::max(w, host_axis_len(ix, gx) * host_axis_len(iy, gy) * host_axis_len(iz, gz));
      }
      acc += w;
    }
    B->soff.push_back(acc);
    row0 += P.n;
    soff0 += P.nslices + 1;
    slot0 += (int64_t)acc * kWave + kSellTail;  // each problem keeps its own over-read tail
    elem0 += 44 * (int64_t)P.ne;
    P.ntiles = (int)cdiv((int64_t)P.nslices * kWave, kBlock);
    tile0 += P.ntiles;
    B->probs.push_back(P);
  }
  B->rows = row0;
  B->slots = slot0;
  batch_layout(B, ctx->cu_count);
  hipStream_t s = ctx->stream;
  auto fail_oom = [&](hipError_t e) {
    B->release();
    delete B;
    return hip_fail(ctx, e, "batch_create: hipMalloc");
  };
  hipError_t e;
#define BALLOC(ptr, bytes) \
  if ((e = dev_malloc(ctx, &(ptr), (bytes))) != hipSuccess) return fail_oom(e)
  BALLOC(B->d_probs, sizeof(BatchProb) * (size_t)nprob);
  BALLOC(B->d_blk2prob, sizeof(int) * B->blk2prob.size());
  BALLOC(B->d_soff, sizeof(int) * B->soff.size());
  BALLOC(B->d_scols, sizeof(int) * (size_t)B->slots);
  BALLOC(B->d_svals, sizeof(double) * (size_t)B->slots);
  BALLOC(B->d_KF, sizeof(double) * (size_t)elem0);
  BALLOC(B->d_recs, sizeof(BatchRec) * (size_t)tile0);
  BALLOC(B->d_b, sizeof(double) * (size_t)B->rows);
  BALLOC(B->d_x, sizeof(double) * (size_t)B->rows);
  BALLOC(B->d_r, sizeof(double) * (size_t)B->rows);
  BALLOC(B->d_p, sizeof(double) * ((size_t)B->rows + 2 * kPPad));
  B->d_p += kPPad;
  BALLOC(B->d_Ap, sizeof(double) * (size_t)B->rows);
  BALLOC(B->d_part, sizeof(double) * 2 * B->blk2prob.size());
  BALLOC(B->d_states, sizeof(BatchState) * (size_t)nprob);
#undef BALLOC
  if ((e = hipHostMalloc(&B->h_words, sizeof(int) * (1 + (size_t)nprob),
                         hipHostMallocCoherent)) != hipSuccess)
    return fail_oom(e);
  // the packed words last: a batch that fits without them still runs
  const char* pack = std::getenv("MINIFE_BATCH_PACK");
  if (!(pack && std::atoi(pack) == 0) &&
      dev_malloc(ctx, &B->d_words, sizeof(unsigned) * kBWords * kBlock * (size_t)tile0) != hipSuccess)
    B->d_words = nullptr;
  // zero everything once: the per-problem tails stay value 0, column 0
  auto fill = [&]() -> int {
    MFE_CHECK(ctx, hipMemsetAsync(B->d_scols, 0, sizeof(int) * (size_t)B->slots, s));
    MFE_CHECK(ctx, hipMemsetAsync(B->d_svals, 0, sizeof(double) * (size_t)B->slots, s));
    if (int st2 = batch_upload_layout(ctx, B)) return st2;
    MFE_CHECK(ctx, hipMemcpyAsync(B->d_soff, B->soff.data(), sizeof(int) * B->soff.size(),
                                  hipMemcpyHostToDevice, s));
    MFE_CHECK(ctx, hipStreamSynchronize(s));
    return MFE_OK;
  };
  if (int st = fill()) {
    (void)hipStreamSynchronize(s);
    B->release();
    delete B;
    return st;
  }
  ctx_retain(ctx);
  *out = B;
  return MFE_OK;
}

void mfe_batch_destroy(mfe_batch* B) {
  if (!B) return;
  (void)hipStreamSynchronize(B->ctx->stream);
  B->release();
  mfe_ctx* ctx = B->ctx;
  delete B;
  ctx_release(ctx);
}

int mfe_batch_info(const mfe_batch* B, int p, int64_t info[6]) {
  if (!B || !info || p < -1 || p >= B->nprob) return MFE_BAD_ARG;
  if (p == -1) {
    info[0] = B->nprob;
    info[1] = B->grid;
    info[2] = B->rows;
    info[3] = B->slots;
    int64_t nnz = 0;
    for (const BatchProb& P : B->probs)
      nnz += (int64_t)(3 * P.Nx + 1) * (3 * P.Ny + 1) * (3 * P.Nz + 1);
    info[4] = nnz;
    info[5] = 0;
    return MFE_OK;
  }
  const BatchProb& P = B->probs[(size_t)p];
  info[0] = P.n;
  info[1] = (int64_t)(3 * P.Nx + 1) * (3 * P.Ny + 1) * (3 * P.Nz + 1);
  info[2] = P.ne;
  info[3] = P.nb;
  info[4] = P.b0;
  info[5] = (int64_t)B->soff[(size_t)(P.soff0 + P.nslices)] * kWave;
  return MFE_OK;
}

int mfe_batch_solve(mfe_ctx* ctx, mfe_batch* B, int max_iter, double rel_tol, int* iters,
                    double* rel_residual, double* seconds) {
  if (!ctx || !B || B->ctx != ctx || max_iter < 0 || !(rel_tol >= 0)) return MFE_BAD_ARG;
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  hipStream_t s = ctx->stream;
  MFE_CHECK(ctx, hipMemsetAsync(B->d_states, 0, sizeof(BatchState) * (size_t)B->nprob, s));
  std::fill(B->h_words, B->h_words + 1 + B->nprob, 0);  // nothing is in flight
  int rate_khz = 0;
  MFE_CHECK(ctx, hipDeviceGetAttribute(&rate_khz, hipDeviceAttributeWallClockRate, ctx->device));
  if (rate_khz <= 0) rate_khz = 100000;
  B->tick_seconds = 1.0 / (1e3 * (double)rate_khz);
  HexTables tab;
  host_tables(tab);
  MFE_CHECK(ctx, hipEventRecord(ctx->t_start, s));
  const unsigned grid = (unsigned)B->grid;
  batch_elements_kernel<<<grid, kBlock, 0, s>>>(B->d_probs, B->d_blk2prob, tab, B->d_KF,
                                                B->d_states);
  MFE_CHECK(ctx, hipGetLastError());
  batch_rows_kernel<<<grid, kBlock, 0, s>>>(B->d_probs, B->d_blk2prob, B->d_soff, B->d_KF,
                                            B->d_scols, B->d_svals, B->d_recs, B->d_words,
                                            B->d_b, B->d_x, B->d_r, B->d_p, B->d_part,
                                            B->d_states);
  MFE_CHECK(ctx, hipGetLastError());
  volatile int* host = B->h_words;
  int active = B->nprob;  // problems order[0 .. active) are launched
  for (unsigned k = 1; k <= (unsigned)max_iter + 1; ++k) {
    while (active > 0 && host[1 + B->order[(size_t)active - 1]]) --active;
    if (active == 0) break;
    const BatchProb& last = B->probs[(size_t)B->order[(size_t)active - 1]];
    const unsigned g = (unsigned)(last.b0 + last.nb);
    batch_p_kernel<<<g, kBlock, 0, s>>>(B->d_probs, B->d_blk2prob, B->d_recs, B->d_x, B->d_r,
                                        B->d_p, B->d_Ap, B->d_part, B->d_states, B->h_words, k,
                                        max_iter, rel_tol);
    if (k <= (unsigned)max_iter) {
      auto spmv = B->pairs ? batch_spmv_kernel<true> : batch_spmv_kernel<false>;
      spmv<<<g, kBlock, 0, s>>>(B->d_probs, B->d_blk2prob, B->d_soff, B->d_svals, B->d_recs,
                                B->d_words, B->d_p, B->d_Ap, B->d_part, B->d_states);
      batch_r_kernel<<<g, kBlock, 0, s>>>(B->d_probs, B->d_blk2prob, B->d_r, B->d_Ap, B->d_part,
                                          B->d_states, B->h_words, k);
    }
    MFE_CHECK(ctx, hipGetLastError());
    for (unsigned spin = 1; (unsigned)host[0] + kAhead < k; ++spin)
      if (spin % (1 << 16) == 0) {  // not for ever: the stream may have failed
        const hipError_t e = hipStreamQuery(s);
        if (e == hipSuccess) break;
        if (e != hipErrorNotReady) return hip_fail(ctx, e, "batch_solve: iteration");
      }
  }
  MFE_CHECK(ctx, hipEventRecord(ctx->t_stop, s));
  MFE_CHECK(ctx, hipEventSynchronize(ctx->t_stop));
  float ms = 0;
  MFE_CHECK(ctx, hipEventElapsedTime(&ms, ctx->t_start, ctx->t_stop));
  if (seconds) *seconds = 1e-3 * ms;
  std::vector<BatchState> hs((size_t)B->nprob);
  MFE_CHECK(ctx, hipMemcpy(hs.data(), B->d_states, sizeof(BatchState) * hs.size(),
                           hipMemcpyDeviceToHost));
  int status = MFE_OK;
  B->last_seconds.assign((size_t)B->nprob, 0.0);
  B->last_phases.assign((size_t)B->nprob * 6, 0.0);
  for (int q = 0; q < B->nprob; ++q) {
    B->last_seconds[(size_t)q] =
        (double)(hs[(size_t)q].t_end - hs[(size_t)q].t_begin) * B->tick_seconds;
    double rest = B->last_seconds[(size_t)q];  // between its workgroups of two launches
    for (int ph = 0; ph < 5; ++ph) {
      const double sec = (double)hs[(size_t)q].t_phase[ph] * B->tick_seconds;
      B->last_phases[(size_t)q * 6 + ph] = sec;
      rest -= sec;
    }
    B->last_phases[(size_t)q * 6 + 5] = std::max(rest, 0.0);
    if (iters) iters[q] = hs[(size_t)q].iters;
    if (rel_residual)
      rel_residual[q] = hs[(size_t)q].bnorm > 0 ? hs[(size_t)q].normr / hs[(size_t)q].bnorm
                                                : hs[(size_t)q].normr;
    if (hs[(size_t)q].status == 1) status = MFE_BREAKDOWN;
  }
  if (status == MFE_BREAKDOWN) fail(ctx, MFE_BREAKDOWN, "batch_solve: CG breakdown in a problem");
  return status;
}

int mfe_batch_timing(const mfe_batch* B, double* seconds, double* phases) {
  if (!B) return MFE_BAD_ARG;
  for (int q = 0; q < B->nprob; ++q) {
    const bool have = (size_t)q < B->last_seconds.size();
    if (seconds) seconds[q] = have ? B->last_seconds[(size_t)q] : 0.0;
    if (phases)
      for (int ph = 0; ph < 6; ++ph)
        phases[q * 6 + ph] = have ? B->last_phases[(size_t)q * 6 + ph] : 0.0;
  }
  return MFE_OK;
}

int mfe_batch_download(mfe_ctx* ctx, const mfe_batch* B, int p, int* row_offsets, int* cols,
                       double* vals, double* b, double* x) {
  if (!ctx || !B || p < 0 || p >= B->nprob) return MFE_BAD_ARG;
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  const BatchProb& P = B->probs[(size_t)p];
  if (b) MFE_CHECK(ctx, hipMemcpy(b, B->d_b + P.row0, sizeof(double) * (size_t)P.n, hipMemcpyDeviceToHost));
  if (x) MFE_CHECK(ctx, hipMemcpy(x, B->d_x + P.row0, sizeof(double) * (size_t)P.n, hipMemcpyDeviceToHost));
  if (!row_offsets && !cols && !vals) return MFE_OK;
  const int* so = B->soff.data() + P.soff0;
  const int64_t nslot = (int64_t)so[P.nslices] * kWave;
  std::vector<int> sc((size_t)nslot);
  std::vector<double> sv((size_t)nslot);
  MFE_CHECK(ctx, hipMemcpy(sc.data(), B->d_scols + P.slot0, sizeof(int) * (size_t)nslot,
                           hipMemcpyDeviceToHost));
  MFE_CHECK(ctx, hipMemcpy(sv.data(), B->d_svals + P.slot0, sizeof(double) * (size_t)nslot,
                           hipMemcpyDeviceToHost));
  const int gx = P.Nx + 1, gy = P.Ny + 1, gz = P.Nz + 1;
  int64_t pos = 0;
  for (int id = 0; id < P.n; ++id) {
    const int ix = id % gx, iy = (id / gx) % gy, iz = id / (gx * gy);
    const int len = host_axis_len(ix, gx) * host_axis_len(iy, gy) * host_axis_len(iz, gz);
    if (row_offsets) row_offsets[id] = (int)pos;
    const int s = id / kWave, l = id % kWave;
    for (int j = 0; j < len; ++j, ++pos) {
      const int64_t at = sell_pos((int64_t)so[s] * kWave, j, so[s + 1] - so[s], l);
      if (cols) cols[pos] = sc[(size_t)at];
      if (vals) vals[pos] = sv[(size_t)at];
    }
  }
  if (row_offsets) row_offsets[P.n] = (int)pos;
  return MFE_OK;
}

}  // extern "C"
