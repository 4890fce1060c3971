// Assembly of the structured hex8 box on gfx950: CSR structure, per-element
// diffusion matrix + source vector summed into CSR, Dirichlet.
//
// Bit-exactness: every entry A[r][c] of the reference is the sum, from 0.0 and
// in ascending element id, of K_e[loc(r)][loc(c)] over the elements sharing
// nodes r and c (perform_element_loop.hpp:78-100 iterates elements in
// ascending id; sum_into_row adds one term per element).  The element loop
// below computes each element's K and F (Hex8::diffusionMatrix_symm /
// sourceVector with the reference's operation order; -ffp-contract=off keeps
// every product rounded) and adds them into each node's row in ascending
// element id, so it performs the same additions in the same order.
#include <cmath>
#include <cstring>

#include "mfe_common.hpp"
#include "mfe_hex8.hpp"

namespace mfe {

int csr_alloc(mfe_ctx* ctx, mfe_csr* A, int64_t nrows, int64_t nnz);  // mfe_api.hip

// Jacobian column tables of the element loop: for each axis, element index
// i along it (coordinates i/N and i/N + h, as get_elem_nodes_and_coords forms
// them, Hex8_box_utils.hpp:101-159) and
// Gauss point q, the three sums of jac_column at [(off + i) * 24 + 3q + a],
// off = 0, Nx, Nx + Ny for x, y, z.
__global__ __launch_bounds__(kBlock) void jac_table_kernel(int Nx, int Ny, int Nz, double hx,
                                                           double hy, double hz,
                                                           const HexTables* __restrict__ tab,
                                                           double* __restrict__ out) {
  const int idx = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const int total = (Nx + Ny + Nz) * 8;
  if (idx >= total) return;
  const int line = idx / 8, q = idx % 8;
  int axis, i, N;
  double h;
  if (line < Nx) {
    axis = 0, i = line, N = Nx, h = hx;
  } else if (line < Nx + Ny) {
    axis = 1, i = line - Nx, N = Ny, h = hy;
  } else {
    axis = 2, i = line - Nx - Ny, N = Nz, h = hz;
  }
  const double c0 = 1.0 * i / N;
  jac_column(*tab, q, axis, c0, c0 + h, out + (int64_t)line * 24 + 3 * q);
}

// The element tables from the kernel arguments into device memory (on the
// stream, so no host copy is needed).
__global__ void copy_tables_kernel(HexTables tab, HexTables* __restrict__ out) {
  const double* src = reinterpret_cast<const double*>(&tab);
  double* dst = reinterpret_cast<double*>(out);
  for (int i = (int)threadIdx.x; i < (int)(sizeof(HexTables) / sizeof(double)); i += blockDim.x)
    dst[i] = src[i];
}

// The element loop and the gather in one pass (K and F never reach memory).
// A workgroup owns a tile of 16 x 16 elements in (x, y) -- element
// (15 bx + tx, 15 by + ty), one per thread -- and a range [z0, z1) of node
// planes, and marches through the element layers z0-1 .. z1-1.  Each step
// computes one layer's elements in registers and hands their entries to the
// tile's nodes through LDS: the 15 x 15 nodes whose four elements of the
// layer all lie in the tile (node (15 bx + i, 15 by + j), i, j in 1..15; the
// first tile of an axis also takes node 0, whose lower element does not
// exist), so a tile recomputes one row and one column of its neighbours'
// elements.  Node rows are summed in ascending element id: a row of plane z gets layer z-1's terms at step z-1 (its slots
// in plane z-1 are then complete and stored; its slots in plane z are
// carried in registers) and layer z's terms at step z, after which the rest
// of the row is stored.  LDS holds two phases of 16 x 16 elements' entries: first every
// entry with a lower-face corner (the 4 x 4 lower block packed, 10; the
// lower x upper block, 16; the lower corners' source terms, 4), then the
// upper block (10) and the upper source terms (4).
constexpr int kFuseSide = 16;                    // elements per tile side
constexpr int kFuseStep = kFuseSide - 1;         // tile pitch in elements
constexpr int kFuseA = 30;                       // LDS entries per element (the first phase's)
__host__ __device__ constexpr int tri4(int a, int b) {  // packed 4 x 4 upper triangle, a <= b
  return a * 4 - a * (a - 1) / 2 + (b - a);
}
// phase A slot of K entry (m, n), m <= n, m a lower corner
__host__ __device__ constexpr int fuse_a(int m, int n) { return n < 4 ? tri4(m, n) : 10 + m * 4 + (n - 4); }

// Bound by the FP64 operations of the elements (about 3,000 vector instructions
// per 64 elements, 57% of the issue slots) and the waits of two waves per SIMD:
// element loop at 300^3 5.73 ms with the Gauss tables read through the scalar
// cache and every Jacobian entry used, 5.12 with constant tables, 4.96 without
// the entries that are zero (into memory that was written before; the first time
// 6.2-6.6 ms, so 5.6-5.8).  (Three workgroups per CU, 168 registers and 224
// bytes of scratch: 7.27.)
template <bool ZERO_START>
// (launch bounds: two workgroups per CU, which the 60 KB of LDS allow, so at
// most 256 registers per lane)
__global__ __launch_bounds__(kBlock, 2) void element_gather_kernel(
    int Nx, int Ny, int Nz, int tiles_x, int nzc, int zc, const double* __restrict__ jac, const double* __restrict__ kappa, double Q,
    const int* __restrict__ ro, double* __restrict__ vals, double* __restrict__ b) {
  static_assert(kFuseSide * kFuseSide == kBlock, "one element per thread");
  __shared__ double sh[kFuseA][kBlock];
  const int gx = Nx + 1, gy = Ny + 1, gz = Nz + 1;
  const int wg = (int)blockIdx.x;
  const int chunk = wg % nzc, tile = wg / nzc;
  const int bx = tile % tiles_x, by = tile / tiles_x;
  const int t = (int)threadIdx.x;
  const int tx = t % kFuseSide, ty = t / kFuseSide;
  const int z0 = chunk * zc, z1 = min(z0 + zc, gz);
  // this thread's element (x, y) and node
  const int ex = bx * kFuseStep + tx, ey = by * kFuseStep + ty;
  const bool elive = ex < Nx && ey < Ny;
  const int ix = ex, iy = ey;  // node (ix, iy): elements local (tx-1..tx, ty-1..ty)
  const bool nlive = ix < gx && iy < gy && (tx > 0 || bx == 0) && (ty > 0 || by == 0);
  const int lox = ix > 0 ? -1 : 0, hix = ix < Nx ? 1 : 0;
  const int loy = iy > 0 ? -1 : 0, hiy = iy < Ny ? 1 : 0;
  const int64_t plane = (int64_t)gx * gy;
  const int64_t node_xy = ix + (int64_t)gx * iy;
  // in-range in-plane slots (sy, sx) of the node's row, and how many per z part
  auto in_xy = [&](int sy, int sx) { return sx >= lox && sx <= hix && sy >= loy && sy <= hiy; };
  const int part_len = (hiy - loy + 1) * (hix - lox + 1);
  double cr[9], bc = 0.0;
#pragma unroll
  for (int q = 0; q < 9; ++q) cr[q] = 0.0;
  // the start of a part's sums: 0.0, or the row's existing values (every
  // index below is a compile-time constant, so the arrays stay in registers)
  auto start_part = [&](double (&dst)[9], int64_t row, int part) {
#pragma unroll
    for (int q = 0; q < 9; ++q) dst[q] = 0.0;
    if (!ZERO_START) {
      const int loz = row >= plane ? -1 : 0;
      int64_t pos = ro[row] + (int64_t)(part - loz) * part_len;
#pragma unroll
      for (int sy = -1; sy <= 1; ++sy)
#pragma unroll
        for (int sx = -1; sx <= 1; ++sx)
          if (in_xy(sy, sx)) dst[(sy + 1) * 3 + (sx + 1)] = vals[pos++];
    }
  };
  auto store_part = [&](const double (&src)[9], int64_t& pos) {
#pragma unroll
    for (int sy = -1; sy <= 1; ++sy)
#pragma unroll
      for (int sx = -1; sx <= 1; ++sx)
        if (in_xy(sy, sx)) vals[pos++] = src[(sy + 1) * 3 + (sx + 1)];
  };
  for (int ez = z0 - 1; ez < z1; ++ez) {
    const bool layer = ez >= 0 && ez < Nz;
    const bool own0 = ez >= z0;      // plane ez is this tile's: completed at this step
    const bool own1 = ez + 1 < z1;   // plane ez + 1 is this tile's: started at this step
    double K[36], F[8];
    if (layer && elive) {
      const int64_t e = ex + (int64_t)Nx * (ey + (int64_t)Ny * ez);
      hex8_element_jac(jac + (int64_t)ex * 24, jac + (int64_t)(Nx + ey) * 24,
                             jac + (int64_t)(Nx + Ny + ez) * 24, kappa ? kappa[e] : 1.0, K,
                             F, Q);
    }
    __syncthreads();  // the previous step's reads are done
    if (layer && elive) {
#pragma unroll
      for (int m = 0; m < 4; ++m) {
#pragma unroll
        for (int n = m; n < 8; ++n) sh[fuse_a(m, n)][t] = K[packed(m, n)];
        sh[26 + m][t] = F[m];
      }
    }
    __syncthreads();
    const int64_t row0 = ez * plane + node_xy;  // the node of plane ez
    if (own0 && nlive) {
      // plane ez: its z = ez slots (carried) and z = ez+1 slots get layer ez's
      // terms, then the row is stored
      double up[9];
      if (layer && ez < Nz) start_part(up, row0, 1);
      if (layer) {
#pragma unroll
        for (int dy = 0; dy <= 1; ++dy)
#pragma unroll
          for (int dx = 0; dx <= 1; ++dx) {
            const int ux = tx - 1 + dx, uy = ty - 1 + dy;  // element local
            if (ux < 0 || uy < 0 || ex - 1 + dx >= Nx || ey - 1 + dy >= Ny) continue;
            const int el = uy * kFuseSide + ux;
            const int cx = 1 - dx, cy = 1 - dy;  // the node's corner: (cx, cy, 0)
            const int li = corner_of(cx, cy, 0);
#pragma unroll
            for (int sy = -1; sy <= 1; ++sy)
#pragma unroll
              for (int sx = -1; sx <= 1; ++sx) {
                const int ax = cx + sx, ay = cy + sy;
                if (ax < 0 || ax > 1 || ay < 0 || ay > 1) continue;
                const int q = (sy + 1) * 3 + (sx + 1);
                const int l0 = corner_of(ax, ay, 0), l1 = corner_of(ax, ay, 1);
                cr[q] += sh[fuse_a(min(li, l0), max(li, l0))][el];
                up[q] += sh[fuse_a(li, l1)][el];
              }
            bc += sh[26 + li][el];
          }
      }
      // store the row's z parts 0 and +1 (if ez < Nz); part -1 went out at
      // step ez - 1
      int64_t pos = ro[row0] + (ez > 0 ? part_len : 0);
      store_part(cr, pos);
      if (ez < Nz) store_part(up, pos);
      b[row0] = bc;
    }
    const int64_t row1 = row0 + plane;  // the node of plane ez + 1
    if (own1 && nlive) {
      if (!layer) {  // ez = -1: plane 0 starts from nothing
        start_part(cr, row1, 0);
        bc = b[row1];
      } else {
        // plane ez+1's z = ez slots: layer ez's terms only, then stored
        double lo[9];
        start_part(lo, row1, -1);
#pragma unroll
        for (int dy = 0; dy <= 1; ++dy)
#pragma unroll
          for (int dx = 0; dx <= 1; ++dx) {
            const int ux = tx - 1 + dx, uy = ty - 1 + dy;
            if (ux < 0 || uy < 0 || ex - 1 + dx >= Nx || ey - 1 + dy >= Ny) continue;
            const int el = uy * kFuseSide + ux;
            const int cx = 1 - dx, cy = 1 - dy;  // the node's corner: (cx, cy, 1)
            const int li = corner_of(cx, cy, 1);
#pragma unroll
            for (int sy = -1; sy <= 1; ++sy)
#pragma unroll
              for (int sx = -1; sx <= 1; ++sx) {
                const int ax = cx + sx, ay = cy + sy;
                if (ax < 0 || ax > 1 || ay < 0 || ay > 1) continue;
                lo[(sy + 1) * 3 + (sx + 1)] += sh[fuse_a(corner_of(ax, ay, 0), li)][el];
              }
          }
        int64_t pos = ro[row1];
        store_part(lo, pos);
      }
    }
    if (layer && own1) {
      __syncthreads();  // phase A's reads are done
      if (elive) {
#pragma unroll
        for (int m = 4; m < 8; ++m) {
#pragma unroll
          for (int n = m; n < 8; ++n) sh[tri4(m - 4, n - 4)][t] = K[packed(m, n)];
          sh[10 + m - 4][t] = F[m];
        }
      }
      __syncthreads();
      if (nlive) {
        // plane ez+1's z = ez+1 slots and b start with layer ez's terms
        start_part(cr, row1, 0);
        bc = b[row1];
#pragma unroll
        for (int dy = 0; dy <= 1; ++dy)
#pragma unroll
          for (int dx = 0; dx <= 1; ++dx) {
            const int ux = tx - 1 + dx, uy = ty - 1 + dy;
            if (ux < 0 || uy < 0 || ex - 1 + dx >= Nx || ey - 1 + dy >= Ny) continue;
            const int el = uy * kFuseSide + ux;
            const int cx = 1 - dx, cy = 1 - dy;
            const int li = corner_of(cx, cy, 1);
#pragma unroll
            for (int sy = -1; sy <= 1; ++sy)
#pragma unroll
              for (int sx = -1; sx <= 1; ++sx) {
                const int ax = cx + sx, ay = cy + sy;
                if (ax < 0 || ax > 1 || ay < 0 || ay > 1) continue;
                const int l1 = corner_of(ax, ay, 1);
                cr[(sy + 1) * 3 + (sx + 1)] += sh[tri4(min(li, l1) - 4, max(li, l1) - 4)][el];
              }
            bc += sh[10 + li - 4][el];
          }
      }
    }
  }
}

// generate_matrix_structure + MatrixInitOp: one thread per node.  The row
// offset has a closed form: per axis a node has cnt(i) = 2 (ends) or 3
// in-range neighbours and the running count before index i is 3i-1 (i>0).
__device__ __forceinline__ int64_t axis_cnt(int i, int g) { return 1 + (i > 0) + (i < g - 1); }
__device__ __forceinline__ int64_t axis_pre(int i) { return i > 0 ? 3 * (int64_t)i - 1 : 0; }

__global__ __launch_bounds__(kBlock) void structure_kernel(int gx, int gy, int gz,
                                                           int* __restrict__ rows,
                                                           int* __restrict__ ro,
                                                           int* __restrict__ cols) {
  // A row's (up to 27) columns are written to LDS first and the workgroup's
  // 256 rows of columns, contiguous in cols, are stored with coalesced writes
  // (rows are 108 bytes apart, so per-thread stores would touch 64 cache
  // lines per instruction).
  __shared__ int sc[kSpmvMaxNnz];
  __shared__ int64_t s_end;
  const int64_t n = (int64_t)gx * gy * gz;
  const int64_t r0 = (int64_t)blockIdx.x * blockDim.x;
  const int64_t id = r0 + threadIdx.x;
  const int64_t Sx = 3 * (int64_t)gx - 2, Sy = 3 * (int64_t)gy - 2;
  const int64_t last = (r0 + kBlock < n ? r0 + kBlock : n) - 1;
  int64_t off = 0, s0 = 0;
  if (id <= last) {
    const int ix = (int)(id % gx);
    const int iy = (int)((id / gx) % gy);
    const int iz = (int)(id / ((int64_t)gx * gy));
    const int64_t cz = axis_cnt(iz, gz), cy = axis_cnt(iy, gy);
    off = axis_pre(iz) * Sy * Sx + cz * axis_pre(iy) * Sx + cz * cy * axis_pre(ix);
    const int64_t len = cz * cy * axis_cnt(ix, gx);
    rows[id] = (int)id;
    ro[id] = (int)off;
    if (id == n - 1) ro[n] = (int)(off + len);
    if (id == last) s_end = off + len;
  }
  // the tile's first offset (thread 0's row), shared through LDS; a tile holds
  // at most 27 * 256 = kSpmvMaxNnz columns
  __shared__ int64_t s_begin;
  if (threadIdx.x == 0) s_begin = off;
  __syncthreads();
  s0 = s_begin;
  if (id <= last) {
    const int ix = (int)(id % gx);
    const int iy = (int)((id / gx) % gy);
    const int iz = (int)(id / ((int64_t)gx * gy));
    int pos = (int)(off - s0);
#pragma unroll
    for (int sz = -1; sz <= 1; ++sz)
#pragma unroll
      for (int sy = -1; sy <= 1; ++sy)
#pragma unroll
        for (int sx = -1; sx <= 1; ++sx) {
          const int x = ix + sx, y = iy + sy, z = iz + sz;
          if (x < 0 || y < 0 || z < 0 || x >= gx || y >= gy || z >= gz) continue;
          sc[pos++] = (int)(x + (int64_t)gx * y + (int64_t)gx * gy * z);
        }
  }
  __syncthreads();
  const int cnt = (int)(s_end - s0);
  for (int i = (int)threadIdx.x; i < cnt; i += kBlock) cols[s0 + i] = sc[i];
}

// Sets *bad when a row's offsets or columns differ from structure_kernel's.
__global__ __launch_bounds__(kBlock) void structure_check_kernel(int gx, int gy, int gz,
                                                                 const int* __restrict__ ro,
                                                                 const int* __restrict__ cols,
                                                                 unsigned* bad) {
  const int64_t n = (int64_t)gx * gy * gz;
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= n) return;
  const int ix = (int)(id % gx);
  const int iy = (int)((id / gx) % gy);
  const int iz = (int)(id / ((int64_t)gx * gy));
  const int64_t Sx = 3 * (int64_t)gx - 2, Sy = 3 * (int64_t)gy - 2;
  const int64_t cz = axis_cnt(iz, gz), cy = axis_cnt(iy, gy);
  const int64_t off = axis_pre(iz) * Sy * Sx + cz * axis_pre(iy) * Sx + cz * cy * axis_pre(ix);
  const int64_t len = cz * cy * axis_cnt(ix, gx);
  bool ok = ro[id] == off && ro[id + 1] == off + len;
  int64_t pos = off;
  for (int sz = -1; sz <= 1 && ok; ++sz)
    for (int sy = -1; sy <= 1 && ok; ++sy)
      for (int sx = -1; sx <= 1 && ok; ++sx) {
        const int x = ix + sx, y = iy + sy, z = iz + sz;
        if (x < 0 || y < 0 || z < 0 || x >= gx || y >= gy || z >= gz) continue;
        ok = cols[pos++] == (int)(x + (int64_t)gx * y + (int64_t)gx * gy * z);
      }
  if (!ok) atomicOr(bad, 1u);
}

__global__ void bc_flag_kernel(int64_t nbc, const int* __restrict__ bc, int64_t n,
                               unsigned char* __restrict__ flags) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nbc) return;
  const int r = bc[k];
  if (r >= 0 && r < n) flags[r] = 1;
}

// impose_dirichlet (SparseMatrix_functions.hpp:431-480), one thread per row.
// BC rows: b = value and identity row (zero_row_and_put_1_on_diagonal).
// Other rows: sum the BC-column coefficients in column order, zero them, and
// b -= sum * value.  Rows are independent, so one pass does both loops.
__global__ __launch_bounds__(kBlock) void dirichlet_kernel(int64_t n, const int* __restrict__ ro,
                                                           const int* __restrict__ cols,
                                                           double* __restrict__ vals,
                                                           double* __restrict__ b,
                                                           const unsigned char* __restrict__ flags,
                                                           double value) {
  const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= n) return;
  const int j0 = ro[row], j1 = ro[row + 1];
  if (flags[row]) {
    b[row] = value;
    for (int j = j0; j < j1; ++j) vals[j] = (cols[j] == row) ? 1.0 : 0.0;
    return;
  }
  double sum = 0;
  for (int j = j0; j < j1; ++j) {
    if (flags[cols[j]]) {
      sum += vals[j];
      vals[j] = 0;
    }
  }
  b[row] -= sum * value;
}

// impose_dirichlet for matrices whose 256-row tiles hold at most kSpmvMaxNnz
// entries: the tile's columns are read into LDS with coalesced loads (the
// per-thread row loop above touches 64 cache lines per load instruction);
// values are read and written only where the row or column is a BC row.
// Same operations in the same order as dirichlet_kernel.
__global__ __launch_bounds__(kBlock) void dirichlet_tile_kernel(
    int64_t n, const int* __restrict__ ro, const int* __restrict__ cols,
    double* __restrict__ vals, double* __restrict__ b, const unsigned char* __restrict__ flags,
    double value) {
  __shared__ int sc[kSpmvMaxNnz];
  const int64_t r0 = (int64_t)blockIdx.x * blockDim.x;
  const int64_t r1 = r0 + kBlock < n ? r0 + kBlock : n;
  const int64_t s0 = ro[r0];
  const int cnt = (int)(ro[r1] - s0);
  for (int i = (int)threadIdx.x; i < cnt; i += kBlock) sc[i] = cols[s0 + i];
  __syncthreads();
  const int64_t row = r0 + threadIdx.x;
  if (row >= r1) return;
  const int j0 = (int)(ro[row] - s0), j1 = (int)(ro[row + 1] - s0);
  if (flags[row]) {
    b[row] = value;
    for (int j = j0; j < j1; ++j) vals[s0 + j] = (sc[j] == row) ? 1.0 : 0.0;
    return;
  }
  double sum = 0;
  for (int j = j0; j < j1; ++j) {
    if (flags[sc[j]]) {
      sum += vals[s0 + j];
      vals[s0 + j] = 0;
    }
  }
  b[row] -= sum * value;
}

// On a structurally symmetric matrix (the box stencil) the rows that hold a
// BC column are the columns of the BC rows: mark them (every writer stores
// 1, so overlapping marks need no atomics).  (Half a wave per row, a lane per
// entry, takes 71 us instead of 51 for 300^3's 90,601 rows of the u = 1 face.)
__global__ void bc_touch_kernel(int64_t nbc, const int* __restrict__ bc, int64_t n,
                                const int* __restrict__ ro, const int* __restrict__ cols,
                                unsigned char* __restrict__ touch) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nbc) return;
  const int r = bc[k];
  if (r < 0 || r >= n) return;  // ignored, as by bc_flag_kernel
  for (int j = ro[r]; j < ro[r + 1]; ++j) touch[cols[j]] = 1;
}

// dirichlet_kernel for the marked rows of a box matrix: any other row has no BC
// column, and dirichlet_kernel would leave it as it is (its sum stays 0 and
// b[row] - 0 * value is b[row]).  A wave looks at 64 rows and takes the marked ones
// two at a time, half a wave per row, a lane per entry; the BC columns' values
// are added in column order from the lanes that hold them.  Bound by the marked
// rows' lines (4% of the rows at 300^3): a thread per row walked its 27 entries
// one dependent load at a time with most lanes idle, 0.62 ms per call, so 0.21.
constexpr int kHalf = kWave / 2;  // >= the 27 entries of a box row
__global__ __launch_bounds__(kBlock) void dirichlet_touched_kernel(
    int64_t n, const int* __restrict__ ro, const int* __restrict__ cols,
    double* __restrict__ vals, double* __restrict__ b, const unsigned char* __restrict__ flags,
    const unsigned char* __restrict__ touch, double value) {
  const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = (int)threadIdx.x % kWave, half = lane / kHalf, l = lane % kHalf;
  uint64_t marked = __ballot(row < n && (touch[row] | flags[row]));
  while (marked) {
    const int r0 = __builtin_ctzll(marked);
    marked &= marked - 1;
    const bool two = marked != 0;
    const int r1 = two ? __builtin_ctzll(marked) : r0;
    marked &= marked - 1;
    const bool mine = half == 0 || two;
    const int64_t r = row - lane + (half == 0 ? r0 : r1);
    const int j = ro[r] + l;
    const bool in = mine && j < ro[r + 1];
    const int c = in ? cols[j] : 0;
    if (flags[r]) {
      if (in) vals[j] = c == r ? 1.0 : 0.0;
      if (mine && l == 0) b[r] = value;
    } else {
      const bool bc = in && flags[c];
      const double v = bc ? vals[j] : 0.0;
      unsigned set = (unsigned)(__ballot(bc) >> (half * kHalf));
      double sum = 0;
      for (; set; set &= set - 1) sum += __shfl(v, half * kHalf + __builtin_ctz(set));
      if (bc) vals[j] = 0;
      if (mine && l == 0) b[r] -= sum * value;
    }
  }
}

// grad[e] = -lambda_e^T K_e(1) utilde_e, one thread per element.
__global__ __launch_bounds__(kBlock) void element_gradient_kernel(
    int Nx, int Ny, int Nz, double hx, double hy, double hz, HexTables tab,
    const double* __restrict__ lambda, const double* __restrict__ ut, double* __restrict__ grad,
    int64_t ne) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= ne) return;
  const int ex = (int)(e % Nx);
  const int ey = (int)((e / Nx) % Ny);
  const int ez = (int)(e / ((int64_t)Nx * Ny));
  const double x0 = 1.0 * ex / Nx;
  const double y0 = 1.0 * ey / Ny;
  const double z0 = (1.0 * ez) / Nz;
  const double x1 = x0 + hx, y1 = y0 + hy, z1 = z0 + hz;
  const double c[24] = {x0, y0, z0, x1, y0, z0, x1, y1, z0, x0, y1, z0,
                        x0, y0, z1, x1, y0, z1, x1, y1, z1, x0, y1, z1};
  double K[36], F[8];
  hex8_element(c, tab, 1.0, K, F);
  const int64_t gx = Nx + 1, gxy = (int64_t)(Nx + 1) * (Ny + 1);
  const int64_t node0 = ex + gx * ey + gxy * ez;
  double lam[8], u[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int64_t id = node0 + corner_x(i) + gx * corner_y(i) + gxy * corner_z(i);
    lam[i] = lambda[id];
    u[i] = ut[id];
  }
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    double t = 0.0;
#pragma unroll
    for (int j = 0; j < 8; ++j) t += K[packed(i, j)] * u[j];
    s += lam[i] * t;
  }
  grad[e] = -s;
}

static bool box_ok(const int* g) {
  return g && g[0] == 0 && g[2] == 0 && g[4] == 0 && g[1] > 0 && g[3] > 0 && g[5] > 0;
}
static bool same_box(const int* a, const int* b) {
  for (int i = 0; i < 6; ++i)
    if (a[i] != b[i]) return false;
  return true;
}

}  // namespace mfe

using namespace mfe;

extern "C" {

int mfe_generate_matrix_structure(mfe_ctx* ctx, const int gbox[6], const int lbox[6],
                                  mfe_csr* A) {
  if (!ctx || !A || !box_ok(gbox) || !lbox) return MFE_BAD_ARG;
  if (!same_box(gbox, lbox))
    return fail(ctx, MFE_UNSUPPORTED, "one rank: local box must equal the global box");
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  const int gx = gbox[1] + 1, gy = gbox[3] + 1, gz = gbox[5] + 1;
  const int64_t n = (int64_t)gx * gy * gz;
  const int64_t nnz = (3 * (int64_t)gx - 2) * (3 * (int64_t)gy - 2) * (3 * (int64_t)gz - 2);
  int st = csr_alloc(ctx, A, n, nnz);
  if (st) return st;
  structure_kernel<<<(unsigned)cdiv(n, kBlock), kBlock, 0, ctx->stream>>>(gx, gy, gz, A->rows,
                                                                          A->row_offsets, A->cols);
  MFE_LAUNCHED(ctx, "structure_kernel");
  MFE_CHECK(ctx, hipMemsetAsync(A->vals, 0, sizeof(double) * (size_t)nnz, ctx->stream));
  A->has_local_indices = false;
  A->num_cols = 0;
  csr_structure_changed(A);
  A->vals_zero = true;
  A->box_elems[0] = gbox[1];
  A->box_elems[1] = gbox[3];
  A->box_elems[2] = gbox[5];
  return plan_spmv(ctx, A);
}

static int element_loop(mfe_ctx* ctx, const int gbox[6], const int ebox[6], mfe_csr* A,
                        mfe_vec* b, const mfe_vec* kappa, double source);

int mfe_perform_element_loop(mfe_ctx* ctx, const int gbox[6], const int ebox[6], mfe_csr* A,
                             mfe_vec* b, const mfe_vec* kappa) {
  return element_loop(ctx, gbox, ebox, A, b, kappa, 1.0);
}

static int element_loop(mfe_ctx* ctx, const int gbox[6], const int ebox[6], mfe_csr* A,
                        mfe_vec* b, const mfe_vec* kappa, double source) {
  if (!ctx || !A || !b || !box_ok(gbox) || !ebox) return MFE_BAD_ARG;
  uses(ctx, A, b);
  if (kappa) uses(ctx, kappa);
  if (!same_box(gbox, ebox))
    return fail(ctx, MFE_UNSUPPORTED, "one rank: the element box must be the global box");
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  const int Nx = gbox[1], Ny = gbox[3], Nz = gbox[5];
  const int64_t n = (int64_t)(Nx + 1) * (Ny + 1) * (Nz + 1);
  const int64_t nnz = (3 * (int64_t)Nx + 1) * (3 * (int64_t)Ny + 1) * (3 * (int64_t)Nz + 1);
  const int64_t ne = (int64_t)Nx * Ny * Nz;
  if (A->nrows != n || A->nnz != nnz || b->n != n)
    return fail(ctx, MFE_BAD_ARG, "A/b do not hold this box's structure");
  if (A->box_elems[0] != Nx || A->box_elems[1] != Ny || A->box_elems[2] != Nz) {
    // a structure from elsewhere (an upload): accepted if it is the box's
    unsigned* bad = reinterpret_cast<unsigned*>(ctx->d_scalars);
    MFE_CHECK(ctx, hipMemsetAsync(bad, 0, sizeof(unsigned), ctx->stream));
    structure_check_kernel<<<(unsigned)cdiv(n, kBlock), kBlock, 0, ctx->stream>>>(
        Nx + 1, Ny + 1, Nz + 1, A->row_offsets, A->cols, bad);
    MFE_LAUNCHED(ctx, "structure_check_kernel");
    MFE_CHECK(ctx, hipMemcpyAsync(ctx->h_scalars, bad, sizeof(unsigned), hipMemcpyDeviceToHost,
                                  ctx->stream));
    MFE_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    unsigned hbad = 0;
    std::memcpy(&hbad, ctx->h_scalars, sizeof(hbad));
    if (hbad)
      return fail(ctx, MFE_BAD_ARG,
                  "A's structure is not the box's (generate_matrix_structure's rows and columns)");
    A->box_elems[0] = Nx;
    A->box_elems[1] = Ny;
    A->box_elems[2] = Nz;
  }
  if (kappa && kappa->n != ne) return fail(ctx, MFE_BAD_ARG, "kappa must have one value per element");
  HexTables tab;
  host_tables(tab);
  // the Jacobian column tables, then the Gauss tables (read by every element)
  const int64_t njac = 24 * ((int64_t)Nx + Ny + Nz);
  double* djac = nullptr;
  hipError_t e1 = dev_alloc(ctx, &djac, sizeof(double) * (size_t)njac + sizeof(HexTables));
  if (e1 != hipSuccess) return hip_fail(ctx, e1, "hipMalloc(element tables)");
  HexTables* dtab = reinterpret_cast<HexTables*>(djac + njac);
  copy_tables_kernel<<<1, kBlock, 0, ctx->stream>>>(tab, dtab);
  int st = MFE_OK;
  jac_table_kernel<<<(unsigned)cdiv((Nx + Ny + Nz) * 8, kBlock), kBlock, 0, ctx->stream>>>(
      Nx, Ny, Nz, 1.0 / Nx, 1.0 / Ny, 1.0 / Nz, dtab, djac);
  // tiles of 16 x 16 elements at a pitch of 15, z chunks filling whole rounds
  // of the resident workgroups
  const bool zero = A->vals_zero;
  const void* kfn = zero ? (const void*)element_gather_kernel<true>
                         : (const void*)element_gather_kernel<false>;
  BoxGeom m{};
  m.nbx = (int)cdiv(Nx, kFuseStep);
  m.nby = (int)cdiv(Ny, kFuseStep);
  m.gz = Nz + 1;
  box_chunks(m, resident_groups(kfn, ctx->cu_count), (int64_t)m.nbx * m.nby * m.gz);
  const unsigned grid = (unsigned)((int64_t)m.nbx * m.nby * m.nzc);
  if (zero)
    element_gather_kernel<true><<<grid, kBlock, 0, ctx->stream>>>(
        Nx, Ny, Nz, m.nbx, m.nzc, m.zc, djac, kappa ? kappa->d : nullptr, source,
        A->row_offsets, A->vals, b->d);
  else
    element_gather_kernel<false><<<grid, kBlock, 0, ctx->stream>>>(
        Nx, Ny, Nz, m.nbx, m.nzc, m.zc, djac, kappa ? kappa->d : nullptr, source,
        A->row_offsets, A->vals, b->d);
  hipError_t le = hipGetLastError();
  csr_values_changed(A);
  if (le != hipSuccess) st = hip_fail(ctx, le, "element_gather_kernel");
  hipError_t se = hipStreamSynchronize(ctx->stream);
  if (st == MFE_OK && se != hipSuccess) st = hip_fail(ctx, se, "assembly");
  dev_free(ctx, djac);
  return st;
}

int mfe_assemble_FE_data(mfe_ctx* ctx, const int gbox[6], const int lbox[6], mfe_csr* A,
                         mfe_vec* b, const mfe_vec* kappa) {
  if (!ctx || !box_ok(gbox) || !lbox) return MFE_BAD_ARG;
  if (!same_box(gbox, lbox))
    return fail(ctx, MFE_UNSUPPORTED, "one rank: local box must equal the global box");
  // One rank: the ghost layer of assemble_FE_data.hpp:59-72 is empty.
  return mfe_perform_element_loop(ctx, gbox, lbox, A, b, kappa);
}

int mfe_assemble_FE_data_ex(mfe_ctx* ctx, const int gbox[6], const int lbox[6], mfe_csr* A,
                            mfe_vec* b, const mfe_vec* kappa, double source) {
  if (!ctx || !box_ok(gbox) || !lbox) return MFE_BAD_ARG;
  if (!same_box(gbox, lbox))
    return fail(ctx, MFE_UNSUPPORTED, "one rank: local box must equal the global box");
  return element_loop(ctx, gbox, lbox, A, b, kappa, source);
}

int mfe_impose_dirichlet(mfe_ctx* ctx, double value, mfe_csr* A, mfe_vec* b, int gnx, int gny,
                         int gnz, const int* bc_rows, int64_t nbc) {
  (void)gnx;
  (void)gny;
  (void)gnz;
  if (!ctx || !A || !b || nbc < 0 || (nbc > 0 && !bc_rows)) return MFE_BAD_ARG;
  uses(ctx, A, b);
  if (b->n != A->nrows) return fail(ctx, MFE_BAD_ARG, "b length != rows");
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  const int64_t n = A->nrows;
  if (n == 0) return MFE_OK;
  int* stage = nullptr;
  if (nbc > 0) {
    int sst = stage_buffer(ctx, reinterpret_cast<void**>(&stage));
    if (sst) return sst;
  }
  unsigned char* flags = nullptr;
  // flags[0, n): BC rows; flags[n, 2n): rows that may hold a BC column
  hipError_t e = dev_alloc(ctx, &flags, 2 * (size_t)n);
  if (e != hipSuccess) return hip_fail(ctx, e, "hipMalloc(bc flags)");
  unsigned char* const touch = flags + n;
  // the box stencil is structurally symmetric: only the BC rows' neighbours
  // can hold BC columns
  const bool box = A->box_elems[0] > 0;
  int st = MFE_OK;
  do {
    e = hipMemsetAsync(flags, 0, 2 * (size_t)n, ctx->stream);
    if (e != hipSuccess) { st = hip_fail(ctx, e, "bc flags memset"); break; }
    // the kernels read the row list from the context's pinned buffer, a chunk
    // at a time (no copy engine involved)
    const int64_t chunk = (int64_t)(kStageBytes / sizeof(int));
    for (int64_t off = 0; off < nbc && st == MFE_OK; off += chunk) {
      const int64_t cnt = nbc - off < chunk ? nbc - off : chunk;
      if (off > 0 && (e = hipStreamSynchronize(ctx->stream)) != hipSuccess) {
        st = hip_fail(ctx, e, "bc rows");  // the previous chunk is still read
        break;
      }
      std::memcpy(stage, bc_rows + off, sizeof(int) * (size_t)cnt);
      bc_flag_kernel<<<(unsigned)cdiv(cnt, kBlock), kBlock, 0, ctx->stream>>>(cnt, stage, n, flags);
      if (box)
        bc_touch_kernel<<<(unsigned)cdiv(cnt, kBlock), kBlock, 0, ctx->stream>>>(
            cnt, stage, n, A->row_offsets, A->cols, touch);
      if ((e = hipGetLastError()) != hipSuccess) st = hip_fail(ctx, e, "bc_flag_kernel");
    }
    if (st) break;
    csr_values_changed(A);
    if (box)
      dirichlet_touched_kernel<<<(unsigned)cdiv(n, kBlock), kBlock, 0, ctx->stream>>>(
          n, A->row_offsets, A->cols, A->vals, b->d, flags, touch, value);
    else if (A->max_block_nnz >= 0 && A->max_block_nnz <= kSpmvMaxNnz)
      dirichlet_tile_kernel<<<(unsigned)cdiv(n, kBlock), kBlock, 0, ctx->stream>>>(
          n, A->row_offsets, A->cols, A->vals, b->d, flags, value);
    else
      dirichlet_kernel<<<(unsigned)cdiv(n, kBlock), kBlock, 0, ctx->stream>>>(
          n, A->row_offsets, A->cols, A->vals, b->d, flags, value);
    if ((e = hipGetLastError()) != hipSuccess) { st = hip_fail(ctx, e, "dirichlet_kernel"); break; }
  } while (0);
  hipError_t se = hipStreamSynchronize(ctx->stream);
  if (st == MFE_OK && se != hipSuccess) st = hip_fail(ctx, se, "impose_dirichlet");
  dev_free(ctx, flags);
  return st;
}

}  // extern "C"

extern "C" int mfe_element_gradient(mfe_ctx* ctx, const int gbox[6], const mfe_vec* lambda,
                                    const mfe_vec* utilde, mfe_vec* grad) {
  if (!ctx || !box_ok(gbox) || !lambda || !utilde || !grad) return MFE_BAD_ARG;
  uses(ctx, lambda, utilde, grad);
  const int Nx = gbox[1], Ny = gbox[3], Nz = gbox[5];
  const int64_t n = (int64_t)(Nx + 1) * (Ny + 1) * (Nz + 1);
  const int64_t ne = (int64_t)Nx * Ny * Nz;
  if (lambda->n != n || utilde->n != n || grad->n != ne)
    return fail(ctx, MFE_BAD_ARG, "element_gradient: lambda/utilde need one value per node, "
                                  "grad one per element");
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  HexTables tab;
  host_tables(tab);
  element_gradient_kernel<<<(unsigned)cdiv(ne, kBlock), kBlock, 0, ctx->stream>>>(
      Nx, Ny, Nz, 1.0 / Nx, 1.0 / Ny, 1.0 / Nz, tab, lambda->d, utilde->d, grad->d, ne);
  MFE_LAUNCHED(ctx, "element_gradient_kernel");
  return MFE_OK;
}
