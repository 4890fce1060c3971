// Internal definitions shared by the libminife_hip.so translation units.
// Everything here is compiled for gfx950 with -ffp-contract=off, so each
// a*b+c of the reference stays two rounded operations (bit-identical results).
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <cstdio>
#include <string>
#include <vector>

#include "minife_hip.h"

namespace mfe {

constexpr int kWave = 64;          // CDNA wavefront width
constexpr int kBlock = 256;        // threads per workgroup (4 waves)
constexpr int kNumXcd = 8;         // MI355X: 8 XCDs, one L2 each
constexpr int kSpmvRows = 256;     // rows per SpMV workgroup (one per thread)
constexpr int kSpmvMaxNnz = 27 * kSpmvRows;  // LDS product slots per workgroup
constexpr int kVecBlocks = 2048;   // fixed grid of the vector kernels
constexpr int kSellBaseStride = 32;  // per-slice local-column bases (27 used)
constexpr int kSellMaxWidth = 27;  // longest row the SELL SpMV takes (27-point stencil)

struct CgWorkspace;     // mfe_solve.hip
struct MultiWorkspace;  // mfe_multi.hip

// SpMV variants.  kPlain: y = A x.  kDot: also the workgroup partial of x.y
// (p.Ap in CG).  kResid: y = 1*b + (-1)*(A x) (the reference's r = b - Ap
// waxpby, fused) and the partial of y.y.
enum SpmvMode { kPlain = 0, kDot = 1, kResid = 2 };

// Geometry of the box layout (mfe_box.hpp) and of one launch on it.
struct BoxGeom {
  int gx, gy, gz;  // nodes per side
  int nbx, nby;    // blocks of kBoxBX x kBoxBY nodes per side
  int zc, nzc;     // a launch's planes per z chunk and chunks
};

}  // namespace mfe

struct mfe_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  hipEvent_t t_start = nullptr, t_stop = nullptr;
  std::string err;
  double* d_partials = nullptr;  // reduction partials (3 x kPartialsCap)
  size_t partials_cap = 0;
  double* d_scalars = nullptr;   // small device scalar area
  double* h_scalars = nullptr;   // pinned host mirror
  void* h_stage = nullptr;       // pinned staging for small uploads (lazy, kStageBytes)
  mfe::CgWorkspace* cg = nullptr;
  mfe::MultiWorkspace* multi = nullptr;
  int cu_count = 0;
  // The caller's reference (dropped by mfe_ctx_destroy) plus one per live
  // matrix, vector or batch made on this context: the context is freed when
  // the last of them goes, so handles may be destroyed in any order.
  std::atomic<int> refs{1};
};

struct mfe_csr {
  mfe_ctx* ctx = nullptr;
  mutable std::atomic<bool> shared{false};  // see uses()
  int64_t nrows = 0, nnz = 0;
  int* rows = nullptr;
  int* row_offsets = nullptr;
  int* cols = nullptr;
  double* vals = nullptr;
  float* vals32 = nullptr;  // FP32 copy for the mixed-precision solve (lazy)
  bool vals32_valid = false;
  bool has_local_indices = false;
  int64_t num_cols = 0;
  // SpMV plan: largest nnz of any kSpmvRows-row block (-1 = not computed).
  int64_t max_block_nnz = -1;
  // Elements per side of the box whose stencil generate_matrix_structure wrote
  // (0 after any other change of structure): the element loop writes each
  // row's entries at the positions that structure gives them.
  int box_elems[3] = {0, 0, 0};
  // Every value is +0.0 (set by generate_matrix_structure, cleared by any
  // change of the values).
  bool vals_zero = false;
  // SELL-64 copy of the matrix for the SpMV (sliced ELLPACK: slices of 64
  // rows, one row per lane, slot j of a slice stored as 64 consecutive
  // entries), derived lazily from the CSR arrays and rebuilt after changes.
  int spmv_format = MFE_SPMV_AUTO;
  // Process-unique stamp, renewed whenever the arrays an SpMV launch reads
  // move: (matrix, plan_gen) names one structure even across a matrix freed
  // and another created at its address.
  uint64_t plan_gen = 0;
  bool sell_struct_valid = false;  // sell_off/len/cols match the CSR structure
  bool sell_ok = false;            // every row fits kSellMaxWidth and the copy fits memory
  bool sell_vals_valid = false, sell_vals32_valid = false;
  int sell_max_len = 0;
  int64_t sell_nslices = 0, sell_slots = 0;
  int* sell_off = nullptr;           // nslices+1, in units of 64-entry slot columns
  unsigned char* sell_len = nullptr;  // nslices*64 row lengths
  int* sell_cols = nullptr;
  double* sell_vals = nullptr;
  float* sell_vals32 = nullptr;
  // SELL-64 with the x entries of each 256-row tile staged in LDS: the tile's
  // distinct columns as runs of consecutive columns, and every slot's column
  // as its 16-bit position in the tile's list (same slot layout as sell_cols).
  bool sellx_valid = false;  // examined for the current SELL structure
  bool sellx_ok = false;     // every tile fits (runs, LDS) and the copy fits memory
  int sellx_maxu = 0;        // most distinct columns of any tile
  int64_t sellx_ntiles = 0, sellx_runs = 0;
  unsigned short* sellx_lcols = nullptr;  // sell_slots + tail
  int* sellx_roff = nullptr;              // ntiles+1: first run of each tile
  int* sellx_rcol = nullptr;              // runs: first column of the run
  int* sellx_rpos = nullptr;              // runs: its position in the tile's list
  int* sellx_nu = nullptr;                // ntiles: distinct columns of the tile
  // Slices whose 64 rows all have the slice's width and whose slot-j local
  // columns are base_j + lane (rows of one grid line on a stencil): the SpMV
  // reads the 27 bases instead of 64 x 27 local columns.
  int64_t sellx_affine = 0;                // such slices
  int64_t sellx_explicit = 0;              // stored entries of the other slices
  unsigned char* sellx_aff = nullptr;      // nslices: 1 = bases apply
  unsigned short* sellx_sbase = nullptr;   // nslices x kSellBaseStride bases (0 past the width)
  // Per slice, whether its rows are 64 consecutive nodes of grid lines in the
  // form the SpMM's line tiles use, and their columns (built for those tiles,
  // mfe_multi.hip).
  bool sell_lines_valid = false;
  int* sell_lines = nullptr;
  // Box layout (mfe_box.hpp) of the values, for a matrix that holds the box
  // structure (box_elems set): made on first use, stale after any change.
  bool box_vals_valid = false, box_vals32_valid = false;
  mfe::BoxGeom box_geom{};
  double* box_vals = nullptr;
  float* box_vals32 = nullptr;
  // Symmetric box layout (mfe_boxsym.hpp): 0 = not examined for the current
  // values, 1 = every A[r][c] equals A[c][r] bit for bit, 2 = not symmetric.
  int boxsym_state = 0;
  bool boxsym_valid = false, boxsym32_valid = false;
  double *boxsym_u = nullptr, *boxsym_w = nullptr;
  float *boxsym_u32 = nullptr, *boxsym_w32 = nullptr;
  int* boxsym_tab = nullptr;  // kernel table (kSymNB) + fill table (256 x 13)
  // The packed form of the symmetric layout's upper values (mfe_boxsym.hpp),
  // per precision: boxpack_form (a PackForm; kPackNone: the SpMV reads the
  // full values), the packed words (boxpack_cap words per row allocated), and
  // a record of kSymKRec values per (block, plane) (SymRec: the slots' bases,
  // then their powers of two and the codes flag as 32-bit words; until the
  // packing each slot's greatest multiple and power of two, side by side).
  bool boxpack_valid = false, boxpack32_valid = false;
  // Per field width (mfe_pack.hpp's kPackWidths), the upper slots (and the FP64
  // boundary stream's lower slots) whose every group fits it, found while the
  // layout is built.
  unsigned boxpack_fits[6] = {}, boxpack32_fits[6] = {}, boxwpack_fits[6] = {};
  int boxpack_form = 0, boxpack32_form = 0;
  int boxpack_cap = 0, boxpack32_cap = 0;
  unsigned *boxpack_pw = nullptr, *boxpack32_pw = nullptr;
  double* boxpack_kq = nullptr;
  float* boxpack32_kq = nullptr;
  // the FP64 boundary stream's packed form (with the upper values' form;
  // kPackNone: full values), its words and (base, power of two) records
  int boxwpack_form = 0;
  unsigned* boxwpack_pw = nullptr;
  double* boxwpack_kq = nullptr;
};

struct mfe_vec {
  mfe_ctx* ctx = nullptr;
  mutable std::atomic<bool> shared{false};  // see uses()
  int64_t n = 0;
  double* d = nullptr;
  bool owns = true;  // false for mfe_vec_wrap views
};

namespace mfe {

int fail(mfe_ctx* ctx, int status, const std::string& msg);
// A handle made on ctx holds a reference to it until the handle is destroyed.
inline void ctx_retain(mfe_ctx* ctx) { ctx->refs.fetch_add(1, std::memory_order_relaxed); }
void ctx_release(mfe_ctx* ctx);  // frees ctx when its last reference goes
// Looks up this device's copy of the allocation-free entry point's scratch
// array (once per device; mfe_solve.hip); ctx's device must be current.
int noalloc_scratch_init(mfe_ctx* ctx);
// ctx's pinned host buffer of kStageBytes (allocated on first use), which
// kernels can read directly; the caller waits for them before refilling it.
constexpr size_t kStageBytes = 1 << 20;
int stage_buffer(mfe_ctx* ctx, void** out);
// Host <-> device copies through the pinned buffer done by a kernel that
// reads or writes it (for the index arrays and counts the plans move; no copy
// engine involved); on ctx's stream, complete on return (mfe_api.hip).
int upload_bytes(mfe_ctx* ctx, void* dst, const void* src, size_t bytes);
int download_bytes(mfe_ctx* ctx, void* dst, const void* src, size_t bytes);
int hip_fail(mfe_ctx* ctx, hipError_t e, const char* what);
// Device memory of matrices, vectors and their plans (mfe_api.hip).  dev_free
// keeps the block for the next dev_alloc of about its size on the same context:
// work on a context is ordered on its one stream, so a block can be handed out
// again while kernels that used it are still queued.  What another context's
// stream may have used (shared, see uses()) goes to hipFree, which waits for the
// device.  Blocks kept on a device are at most an eighth of its memory together
// (the oldest go first), all of them go when an allocation of the library fails
// or mfe_trim_memory asks for it, and a context's go with it.  Safe from several
// threads.
hipError_t dev_alloc_bytes(mfe_ctx* ctx, void** out, size_t bytes);
template <typename P>
inline hipError_t dev_alloc(mfe_ctx* ctx, P** out, size_t bytes) {
  return dev_alloc_bytes(ctx, reinterpret_cast<void**>(out), bytes);
}
void dev_free(mfe_ctx* ctx, void* p, bool shared = false);
// hipMalloc of memory that is not kept (workspaces; hipFree frees it) and, when
// that fails, once more after the kept blocks have gone back.
hipError_t dev_malloc_bytes(mfe_ctx* ctx, void** out, size_t bytes);
template <typename P>
inline hipError_t dev_malloc(mfe_ctx* ctx, P** out, size_t bytes) {
  return dev_malloc_bytes(ctx, reinterpret_cast<void**>(out), bytes);
}
// A block of A's own.
inline void csr_free(const mfe_csr* A, void* p) { dev_free(A->ctx, p, A->shared); }
// Every entry point says which handles it is about to use on ctx: one that was
// made on another context is marked for good, and its memory is not kept.
inline void uses(const mfe_ctx* ctx, const mfe_csr* A) {
  if (A->ctx != ctx) A->shared = true;
}
inline void uses(const mfe_ctx* ctx, const mfe_vec* v) {
  if (v->ctx != ctx) v->shared = true;
}
template <typename H, typename... Hs>
inline void uses(const mfe_ctx* ctx, const H* h, const Hs*... hs) {
  uses(ctx, h);
  uses(ctx, hs...);
}
// Recompute A->max_block_nnz on the device (synchronises the stream).
int plan_spmv(mfe_ctx* ctx, mfe_csr* A);

__host__ __device__ inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

inline uint64_t next_plan_gen() {
  static std::atomic<uint64_t> g{0};
  return ++g;
}

// Derived copies (FP32 values, SELL plan) are stale after these.
inline void csr_values_changed(mfe_csr* A) {
  A->vals_zero = false;
  A->vals32_valid = false;
  A->sell_vals_valid = false;
  A->sell_vals32_valid = false;
  A->box_vals_valid = false;
  A->box_vals32_valid = false;
  A->boxsym_state = 0;
  A->boxsym_valid = false;
  A->boxsym32_valid = false;
  A->boxpack_valid = false;
  A->boxpack32_valid = false;
}
inline void csr_structure_changed(mfe_csr* A) {
  csr_values_changed(A);
  A->box_elems[0] = A->box_elems[1] = A->box_elems[2] = 0;
  A->plan_gen = next_plan_gen();
  A->max_block_nnz = -1;
  A->sell_struct_valid = false;
  A->sell_ok = false;
}
// Frees the SELL arrays (mfe_solve.hip).
void sell_release(mfe_csr* A);
// Frees the box-layout values (mfe_solve.hip).
void box_release(mfe_csr* A);
// Builds A's SELL-64 copy with FP64 values if its format uses one and it is
// stale (mfe_solve.hip; synchronises the stream, not for graph capture).
// Leaves A->sell_ok false when the format is CSR or SELL does not apply.
int sell_prepare(mfe_ctx* ctx, const mfe_csr* A);
// Builds A's box layout with FP64 values when A holds a box's structure and
// the layout is stale (mfe_solve.hip); A->box_vals_valid tells whether it
// exists afterwards.
int box_prepare(mfe_ctx* ctx, const mfe_csr* A);
// Workgroups of kBlock threads of `kernel` resident on `cus` compute units,
// and the z chunks of a box-layout launch over g.nbx x g.nby blocks that fill
// whole rounds of them (sets g.zc, g.nzc; at most `cap` workgroups).
int resident_groups(const void* kernel, int cus);
void box_chunks(BoxGeom& g, int resident, int64_t cap);

}  // namespace mfe

#define MFE_CHECK(ctx, call)                                       \
  do {                                                             \
    hipError_t e_ = (call);                                        \
    if (e_ != hipSuccess) return ::mfe::hip_fail((ctx), e_, #call); \
  } while (0)

#define MFE_LAUNCHED(ctx, what)                                     \
  do {                                                              \
    hipError_t e_ = hipGetLastError();                              \
    if (e_ != hipSuccess) return ::mfe::hip_fail((ctx), e_, (what)); \
  } while (0)

namespace mfe {

// Workgroup i of a launch is dispatched to XCD (i mod 8).  This maps the
// dispatch index to a logical tile index so that each XCD sweeps one
// contiguous range of tiles: neighbouring rows then share their x-vector
// lines in the same L2.  A bijection on [0, n).
__device__ __forceinline__ int xcd_contiguous(int bid, int n) {
  const int q = n / kNumXcd, r = n % kNumXcd;
  const int xcd = bid % kNumXcd, local = bid / kNumXcd;
  return xcd * q + (xcd < r ? xcd : r) + local;
}

// Wave64 sum in a fixed butterfly order (deterministic).
template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
  return v;
}

// Workgroup sum for kBlock threads: wave butterflies, then the four wave
// totals added in wave order by thread 0.  Result valid in thread 0.
template <typename T>
__device__ __forceinline__ T block_sum(T v, T* lds4) {
  v = wave_sum(v);
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  if (lane == 0) lds4[wave] = v;
  __syncthreads();
  T t = 0;
  if (threadIdx.x == 0) t = ((lds4[0] + lds4[1]) + lds4[2]) + lds4[3];
  __syncthreads();
  return t;
}

}  // namespace mfe
