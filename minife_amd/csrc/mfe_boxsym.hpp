// The symmetric box layout: the box layout (mfe_box.hpp) for a box matrix
// whose entries satisfy A[r][c] == A[c][r] bit for bit (the assembled
// operator does: both are sums of the same element terms in the same order,
// and impose_dirichlet zeroes a boundary row and the matching column; the
// plan checks every pair before using this layout).
//
// Each row stores only its 14 upper slots s = 13..26 (the diagonal, the
// same-plane neighbours after it, the next plane's nine), 256 rows per
// (block, plane, slot) as in the box layout.  Lower slot s of row r is
// upper slot 26 - s of the neighbour r + off(s).  A neighbour in the block forms
// the product with its own x entry and leaves it in LDS for row r; a lower
// value whose neighbour lies outside the block comes from a second stream of
// kSymNB values per (block, plane) -- the row's own CSR entry -- and the thread
// that loads it leaves its product with the ring's x entry in the same place.
// About 15 values per row instead of 27; every row's products are still added in
// ascending slot order over its in-range slots, so y has the bits of matvec_std.
//
// The LDS arrays are indexed by the reading row: up[j][t] and sm[i][t] hold the
// product row t adds for the lower slot whose mirrored slot is 18 + j of the plane
// before (its own column's stays in a register) or 14 + i of the same plane, so
// every read is stride-1 and the arrays hold 256 entries per slot (32 KB with the
// three planes of x for FP64, a little more with the packed boundary stream: four
// workgroups per CU).
#pragma once

#include <type_traits>

#include "mfe_box.hpp"
#include "mfe_pack.hpp"

namespace mfe {

constexpr int kSymU = 14;    // upper slots stored per row
constexpr int kSymNB = 282;  // lower slots of a 16 x 16 block whose neighbour is outside it

__host__ __device__ inline int64_t sym_at(const BoxGeom& g, int blk, int z, int u, int t) {
  return (((int64_t)blk * g.gz + z) * kSymU + u) * kBlock + t;
}
__host__ __device__ inline int64_t sym_entries(const BoxGeom& g) {
  return (int64_t)g.nbx * g.nby * g.gz * kSymU * kBlock;
}
__host__ __device__ inline int64_t sym_bnd_entries(const BoxGeom& g) {
  return (int64_t)g.nbx * g.nby * g.gz * kSymNB;
}

// Boundary table entry e (kernel side): where its value goes in LDS.
// bits 0-8 reading row t, bits 9-12 slot within the array, bit 13: 1 = the
// same-plane array, 0 = the previous plane's array; for the packed boundary
// stream (below) bits 16-24 the near entries before e, bit 25 whether e is
// a near entry (lower slot 10 or 12), bits 26-29 its lower slot s.
__host__ __device__ inline int sym_code(int t, int slot, int same) {
  return t | (slot << 9) | (same << 13);
}
__host__ __device__ inline int sym_wcode(int near_before, int near, int s) {
  return (near_before << 16) | (near << 25) | (s << 26);
}

// The packed form of the boundary stream W (kSymNB values per (block,
// plane)): entry e's value is a field of the form's width (mfe_pack.hpp) --
// wide for the near entries, whose lower slot s mirrors a near-zero upper
// slot (s = 10, 12: upper slots 16, 14), narrow for the others -- with a
// base and a power of two per (block, plane, lower slot) (kSymWGroups groups:
// KQ[rec * kSymWRec + 2 s], [+ 1], and the codes flag at [+ 2 kSymWGroups]).
// The fields follow each other in entry order from bit 0 of the (block,
// plane)'s first word: entry e with nb near entries before it starts at bit
// (e - nb) * narrow + nb * wide.  One more word pads each (block, plane), so
// a field's second word is always there.  Only forms that give every entry a
// field.  The SpMV tests every boundary field for the codes (two selects per
// entry); the flag is kept for symmetry with the upper values' record.
constexpr unsigned kSymWNear = (1u << 10) | (1u << 12);
constexpr int kSymWGroups = 13;
constexpr int kSymWRec = 2 * kSymWGroups + 1;
constexpr int kSymWNearCount = 32;  // entries of slots 10 and 12 (16 each)
__host__ __device__ constexpr int sym_w_words(int f) {
  return ((kSymNB - kSymWNearCount) * pack_narrow(f) +
          kSymWNearCount * (pack_all(f) ? pack_narrow(f) : pack_wide(f)) + 31) / 32 + 1;
}

// The upper values' record of a (block, plane), kSymKRec values of T at KQ[rec *
// kSymKRec]: the bases kb q of the 14 slots, then as 32-bit words the powers of
// two q (FP64: the high word, the low one being 0) and the codes flag (1: some
// packed value is +0.0 or 1.0).
constexpr int kSymKRec = 2 * kSymU + 2;
template <typename T>
struct SymRec {
  T kb[kSymU];
  unsigned q[kSymU];
  unsigned codes;
  // the record at p, the same for every lane (scalar loads)
  __device__ static SymRec load(const T* p) {
    SymRec r;
    const unsigned* w = reinterpret_cast<const unsigned*>(p + kSymU);
#pragma unroll
    for (int u = 0; u < kSymU; ++u) {
      r.kb[u] = p[u];
      r.q[u] = w[u];
    }
    r.codes = w[kSymU];
    return r;
  }
  __device__ T pow2(int u) const {
    if constexpr (sizeof(T) == 8) return __hiloint2double((int)q[u], 0);
    else return __uint_as_float(q[u]);
  }
};

// One workgroup per (block, z chunk), one node column per thread.  Lower slot s
// of row r is upper slot 26 - s of the neighbour n = r + off(s), and both its
// value and its x entry are n's own: n forms the product v x_n and hands it to
// r through LDS (up: from the plane before; sm: from the same plane), so a row
// reads 8 + 4 products and the next plane's 9 x entries from LDS instead of
// 12 values and 27 x entries; its upper same-plane x entries are the ones it
// read as next-plane entries the step before, and the product from its own
// column stays in a register.  A boundary entry (a lower slot whose neighbour
// is outside the block) is multiplied by the ring's x entry by the thread that
// loaded it.  Products and their order are those of a row-by-row sum.
//   PF != kPackNone: the upper values are read in the packed form of
// mfe_pack.hpp (SymPack: slot u is upper slot u, one word group); a plane's
// record is the same for every lane and is read with scalar loads, issued when
// the plane before has been decoded (43 scalar registers).  With WPK
// (and PF) the boundary stream too, in form wform, from WPW and WKQ (a
// template argument: the choice between the two loads of the boundary values
// costs registers where it is made at run time); its records differ from lane
// to lane and are staged in LDS.
//   Every load runs one plane step ahead of its use.
template <typename T, bool ZERO_Y, int MODE, int PF = kPackNone, bool WPK = false>
__global__ __launch_bounds__(kBlock) void spmv_boxsym_kernel(
    BoxGeom g, const T* __restrict__ U, const T* __restrict__ W, const int* __restrict__ btab,
    const T* __restrict__ x, T* __restrict__ y, const T* __restrict__ bvec,
    T* __restrict__ partials, const int* __restrict__ done, const unsigned* __restrict__ PW = nullptr,
    const T* __restrict__ KQ = nullptr, const unsigned* __restrict__ WPW = nullptr,
    const T* __restrict__ WKQ = nullptr, int wform = kPackNone) {
  using P = SymPack;
  static_assert(P::kSlots == kSymU, "one packed slot per upper slot");
  constexpr PackLayout<P, PF> L{};
  constexpr unsigned kMask = L.mask;  // slots with a field
  constexpr int kWords = L.words;
  constexpr bool kHasKQ = PF != kPackNone;
  constexpr bool wpk = kHasKQ && WPK;
  const int stop = done ? *done : 0;  // tested once the first loads are in flight
  __shared__ T xw[3][kBoxWin];
  __shared__ T up[8][kBlock];  // products of the plane before's upper slots 18 + j
                               // (j != 4), by reading row
  __shared__ T sm[4][kBlock];  // products of this plane's upper slots 14 + i, by reading row
  __shared__ T red[4];
  // the boundary stream's record, double-buffered by plane parity: plane z+1's
  // is stored during step z
  __shared__ T kqs[2][wpk ? kSymWRec : 1];
  // each XCD takes a contiguous range of tiles numbered block-fastest within a z
  // chunk: neighbouring blocks then meet in one L2, which serves their x rings
  // and merges the lines of y that two blocks write (16 nodes start mid-line).
  // At 300^3 this reads 1.04 GB instead of 1.24 and takes 0.347 ms instead of 0.362.
  const int tile = xcd_contiguous((int)blockIdx.x, (int)gridDim.x), nblk = g.nbx * g.nby;
  const int chunk = tile / nblk, blk = tile % nblk;
  const int wg = blk * g.nzc + chunk;  // index of this workgroup's partial
  const int bx = blk % g.nbx, by = blk / g.nbx;
  const int t = (int)threadIdx.x;
  const int tx = t % kBoxBX, ty = t / kBoxBX;
  const int ix = bx * kBoxBX + tx, iy = by * kBoxBY + ty;
  const bool live = ix < g.gx && iy < g.gy;
  const int z0 = chunk * g.zc;
  const int z1 = min(z0 + g.zc, g.gz);
  const int64_t plane = (int64_t)g.gx * g.gy;
  const int64_t rec0 = (int64_t)blk * g.gz;  // (block, plane) index of plane 0
  // window cells this thread loads, and its boundary entries: where the value's
  // product goes and the ring cell of its x entry
  int woff[2], bcode[2], bcell[2];
  bool wok[2], bok[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int w = t + k * kBlock;
    const int wx = w % kBoxWX, wy = w / kBoxWX;
    const int nx = bx * kBoxBX + wx - 1, ny = by * kBoxBY + wy - 1;
    wok[k] = w < kBoxWin && nx >= 0 && nx < g.gx && ny >= 0 && ny < g.gy;
    woff[k] = wok[k] ? nx + g.gx * ny : 0;
    bok[k] = w < kSymNB;
    bcode[k] = bok[k] ? btab[w] : 0;
    const int rt = bcode[k] & 511, s = (bcode[k] >> 26) & 15;
    bcell[k] = (rt / kBoxBX + 1 + (s / 3) % 3 - 1) * kBoxWX + (rt % kBoxBX + 1 + s % 3 - 1);
  }
  // boundary entry k's field: bit offset (from its table code, recomputed
  // where used rather than held in registers)
  const int wn = pack_narrow(wform), wwd = pack_all(wform) ? wn : pack_wide(wform);
  const int wwords = wpk ? sym_w_words(wform) : 0;
  auto bfield_off = [&](int k) {
    const int nb = (bcode[k] >> 16) & 511;
    return (t + k * kBlock - nb) * wn + nb * wwd;
  };
  auto x_plane = [&](int z, T* dst) {
    const bool zin = z >= 0 && z < g.gz;
#pragma unroll
    for (int k = 0; k < 2; ++k)
      dst[k] = zin && wok[k] ? x[(int64_t)z * plane + woff[k]] : T(0);
  };
  auto put_plane = [&](int slot, const T* src) {
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (t + k * kBlock < kBoxWin) xw[slot][t + k * kBlock] = src[k];
  };
  const int lox = ix > 0 ? -1 : 0, hix = ix < g.gx - 1 ? 1 : 0;
  const int loy = iy > 0 ? -1 : 0, hiy = iy < g.gy - 1 ? 1 : 0;
  const int c0 = (ty + 1) * kBoxWX + (tx + 1);
  // The loads of plane z's upper values: the packed words and the full values
  // of the other slots (kFull of them).
  constexpr int kFull = kSymU - __builtin_popcount(kMask);
  struct Raw {
    unsigned pw[kWords > 0 ? kWords : 1];
    T full[kFull > 0 ? kFull : 1];
  };
  auto load_raw = [&](int z, int lo, int cnt, Raw& r) {
#pragma unroll
    for (int w = 0; w < kWords; ++w)
      if (L.needed(w, lo, cnt)) r.pw[w] = PW[((rec0 + z) * kWords + w) * kBlock + t];
#pragma unroll
    for (int u = lo; u < lo + cnt; ++u)
      if (!((kMask >> u) & 1u)) r.full[u - pack_rank(kMask, u)] = U[sym_at(g, blk, z, u, t)];
  };
  // upper slots lo .. lo+cnt-1 of a plane from its loads; its codes flag
  // chooses a branch of the whole workgroup
  auto decode_as = [&](int lo, int cnt, const Raw& r, const SymRec<T>& rec, T* dst, auto codes) {
#pragma unroll
    for (int i = 0; i < cnt; ++i) {
      const int u = lo + i;
      if (L.width[u]) {
        const unsigned f = pack_field(r.pw + L.word[u], L.width[u], L.shift[u]);
        dst[i] = pack_decode<T, decltype(codes)::value>(rec.kb[u], rec.pow2(u), f);
      } else {
        dst[i] = r.full[u - pack_rank(kMask, u)];
      }
    }
  };
  auto decode = [&](int lo, int cnt, const Raw& r, const SymRec<T>& rec, T* dst) {
    if (kHasKQ && rec.codes) decode_as(lo, cnt, r, rec, dst, std::true_type{});
    else decode_as(lo, cnt, r, rec, dst, std::false_type{});
  };
  SymRec<T> rec;
  auto load_rec = [&](int z) {
    if (kHasKQ) rec = SymRec<T>::load(KQ + (rec0 + z) * kSymKRec);
  };
  // this row's upper slot (dy, dx) of the next plane is read by the block row at
  // (tx+dx, ty+dy); its own column's stays in pc
  T pc = T(0);
  auto put_up = [&](const T* u9, T xo) {
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      const int rx = tx + j % 3 - 1, ry = ty + j / 3 - 1;
      const T p = u9[j] * xo;
      if (j == 4) pc = p;
      else if (rx >= 0 && rx < kBoxBX && ry >= 0 && ry < kBoxBY)
        up[j < 4 ? j : j - 1][rx + kBoxBX * ry] = p;
    }
  };
  T xn[2], wqn = T(0), y0n = T(0), brn = T(0);
  // boundary entry k: its value's bits, or the two words holding its field
  unsigned long long bn[2] = {0ull, 0ull};
  Raw rn;
  auto fetch = [&](int z) {  // x plane z+1, what step z reads, the boundary record of plane z+1
    x_plane(z + 1, xn);
    if (live) load_raw(z, 0, kSymU, rn);
    if (wpk) {
      const unsigned* wp = WPW + (rec0 + z) * wwords;
#pragma unroll
      for (int k = 0; k < 2; ++k)
        if (bok[k]) {
          const int wi = bfield_off(k) >> 5;
          bn[k] = ((unsigned long long)wp[wi + 1] << 32) | wp[wi];
        }
    } else {
      const int64_t wbase = (rec0 + z) * kSymNB;
#pragma unroll
      for (int k = 0; k < 2; ++k)
        if (bok[k]) {
          const T v = W[wbase + t + k * kBlock];
          if constexpr (sizeof(T) == 8) bn[k] = (unsigned long long)__double_as_longlong(v);
          else bn[k] = __float_as_uint(v);
        }
    }
    if (live) {
      const int64_t row = (int64_t)z * plane + ix + (int64_t)g.gx * iy;
      if (ZERO_Y) y0n = y[row];
      if (MODE == kResid) brn = bvec[row];
    }
    // issued last: the compiler's waits for the loads above (before their
    // registers are reset) would otherwise include it
    if (wpk && t < kSymWRec && z + 1 < z1) wqn = WKQ[(rec0 + z + 1) * kSymWRec + t];
  };
  T tsum = T(0);
  // Every product starts at +0.0: the ones that no row writes (a neighbour past
  // the box's edge inside the block, the plane below the box's first) stay +0.0.
#pragma unroll
  for (int j = 0; j < 8; ++j) up[j][t] = T(0);
#pragma unroll
  for (int j = 0; j < 4; ++j) sm[j][t] = T(0);
  T xa[2], xb[2];
  Raw r0;
  x_plane(z0 - 1, xa);
  x_plane(z0, xb);
  if (z0 > 0 && live) load_raw(z0 - 1, 5, 9, r0);
  if (wpk && t < kSymWRec) kqs[z0 & 1][t] = WKQ[(rec0 + z0) * kSymWRec + t];
  fetch(z0);
  SymRec<T> rprev{};
  if (kHasKQ && z0 > 0) rprev = SymRec<T>::load(KQ + (rec0 + z0 - 1) * kSymKRec);
  load_rec(z0);
  put_plane((z0 + 2) % 3, xa);
  put_plane(z0 % 3, xb);
  if (stop) return;
  __syncthreads();
  if (z0 > 0 && live) {
    T u9[9];
    decode(5, 9, r0, rprev, u9);
    put_up(u9, xw[(z0 + 2) % 3][c0]);
  }
  T xs[5];  // x of this row and of its upper same-plane neighbours, slots 13 .. 17
#pragma unroll
  for (int i = 0; i < 5; ++i)
    xs[i] = xw[z0 % 3][c0 + (i < 2 ? i : kBoxWX + i - 3)];
  for (int z = z0; z < z1; ++z) {
    // the boundary products first (into the LDS entries of the rows that read
    // them), while few registers are live
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (bok[k]) {
        T v;
        if constexpr (sizeof(T) == 8) v = __longlong_as_double((long long)bn[k]);
        else v = __uint_as_float((unsigned)bn[k]);
        if (wpk) {
          const T* rec = kqs[z & 1];
          const int wd = ((bcode[k] >> 25) & 1) ? wwd : wn, sl = (bcode[k] >> 26) & 15;
          const unsigned mask = wd >= 32 ? ~0u : (1u << wd) - 1u;
          const unsigned f = (unsigned)(bn[k] >> (bfield_off(k) & 31)) & mask;
          v = pack_decode<T, true>(rec[2 * sl], rec[2 * sl + 1], f);
        }
        const int rt = bcode[k] & 511, j = (bcode[k] >> 9) & 15;
        const bool same = (bcode[k] >> 13) & 1;
        const T p = v * xw[same ? z % 3 : (z + 2) % 3][bcell[k]];
        if (same) sm[j][rt] = p;
        else up[j < 4 ? j : j - 1][rt] = p;
      }
    T u[kSymU];
    if (live) {
      decode(0, kSymU, rn, rec, u);
      // same-plane upper slots 14 + i at (dy, dx) = (0, 1), (1, -1), (1, 0),
      // (1, 1): read by the block row at (tx+dx, ty+dy)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int dy = i == 0 ? 0 : 1, dx = i == 0 ? 1 : i - 2;
        const int rx = tx + dx, ry = ty + dy;
        const T p = u[1 + i] * xs[0];
        if (rx < kBoxBX && rx >= 0 && ry < kBoxBY) sm[i][rx + kBoxBX * ry] = p;
      }
    }
    load_rec(min(z + 1, z1 - 1));
    // the boundary record of plane z+1: its buffer was last read by step z-1's products,
    // before step z-1's barriers, and is read after this step's
    if (wpk && t < kSymWRec && z + 1 < z1) kqs[(z + 1) & 1][t] = wqn;
    put_plane((z + 1) % 3, xn);
    const T y0 = y0n, br = brn;
    if (z + 1 < z1) fetch(z + 1);
    __syncthreads();
    const T xo = xs[0];
    if (live) {
      const int loz = z > 0 ? -1 : 0, hiz = z < g.gz - 1 ? 1 : 0;
      T sum = ZERO_Y ? T(0) * y0 : T(0);
      // Out of range: the product is +-0.0, which leaves a sum that started at
      // +0.0 unchanged (a sum of round-to-nearest additions from +0.0 is
      // never -0.0); a sum that starts at 0*y (ZERO_Y) may be -0.0 and skips
      // the term.
      auto add = [&](int s, T p) {
        const int sz = s / 9 - 1, sy = (s / 3) % 3 - 1, sx = s % 3 - 1;
        const bool in = sx >= lox && sx <= hix && sy >= loy && sy <= hiy && sz >= loz && sz <= hiz;
        const T next = sum + p;
        sum = (ZERO_Y && !in) ? sum : next;
      };
#pragma unroll
      for (int s = 0; s < 9; ++s) add(s, s == 4 ? pc : up[s < 4 ? 7 - s : 8 - s][t]);
#pragma unroll
      for (int s = 9; s < 13; ++s) add(s, sm[12 - s][t]);
#pragma unroll
      for (int i = 0; i < 5; ++i) add(13 + i, u[i] * xs[i]);
      const T* wp = xw[(z + 1) % 3];
#pragma unroll
      for (int j = 0; j < 9; ++j) {
        const T xv = wp[c0 + (j / 3 - 1) * kBoxWX + j % 3 - 1];
        add(18 + j, u[5 + j] * xv);
        if (j >= 4) xs[j - 4] = xv;
      }
      if (MODE == kResid) sum = T(1) * br + T(-1) * sum;
      y[(int64_t)z * plane + ix + (int64_t)g.gx * iy] = sum;
      if (MODE == kDot) tsum += sum * xo;
      if (MODE == kResid) tsum += sum * sum;
    }
    __syncthreads();
    if (live) put_up(u + 5, xo);
  }
  if (MODE != kPlain) {
    const T s = block_sum<T>(tsum, red);
    if (t == 0) partials[wg] = s;
  }
}

}  // namespace mfe
