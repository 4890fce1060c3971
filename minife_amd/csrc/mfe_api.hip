// Context, handle, timer and verification entry points of libminife_hip.so.
#include <cmath>
#include <condition_variable>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <tuple>
#include <unordered_map>

#include "mfe_common.hpp"

namespace mfe {

int fail(mfe_ctx* ctx, int status, const std::string& msg) {
  if (ctx) ctx->err = msg;
  return status;
}

int hip_fail(mfe_ctx* ctx, hipError_t e, const char* what) {
  std::string m = std::string(what) + ": " + hipGetErrorString(e);
  return fail(ctx, e == hipErrorOutOfMemory ? MFE_OOM : MFE_HIP_ERROR, m);
}

// ---- device memory kept between objects ---------------------------------------
//
// A new matrix of 300^3 takes 14 GB with its plan.  Allocating and freeing that
// for every matrix of a parameter study costs more than assembling it: memory
// given back to the driver is cleared before it is handed out again (assembly
// and first product at 300^3: 371 ms, of which 18 in kernels at the time; with
// kept memory and 11 ms of kernels 11.4).  A process's first matrix is not helped
// by it: 14.6 ms, in memory that the driver had ready.

namespace {
struct DevPool {
  struct Block {
    void* p;
    size_t bytes;
    mfe_ctx* ctx;
  };
  std::mutex mu;
  std::condition_variable left;                // leaving became 0
  size_t leaving = 0;                          // blocks on their way to hipFree
  std::unordered_map<void*, size_t> live;      // blocks handed out
  std::map<uint64_t, Block> idle;              // kept blocks by age
  std::set<std::tuple<mfe_ctx*, size_t, uint64_t>> fit;  // the same by context, bytes, age
  size_t idle_bytes = 0, cap = 0;
  uint64_t clock = 0;
  // Keeps a block (mu held).
  void keep(mfe_ctx* ctx, void* p, size_t bytes) {
    fit.emplace(ctx, bytes, clock);
    idle[clock++] = Block{p, bytes, ctx};
    idle_bytes += bytes;
  }
  // Takes a kept block out (mu held).
  std::map<uint64_t, Block>::iterator take(std::map<uint64_t, Block>::iterator it,
                                           std::vector<void*>& out) {
    out.push_back(it->second.p);
    fit.erase({it->second.ctx, it->second.bytes, it->first});
    idle_bytes -= it->second.bytes;
    return idle.erase(it);
  }
  // Gives blocks back to the driver, without the mutex (the caller counted them as
  // leaving while it held it): hipFree waits for the device, other contexts' work
  // included, and their threads go on meanwhile.  No stream is waited for by name:
  // another thread may be capturing it.
  void release(const std::vector<void*>& blocks) {
    for (void* p : blocks) (void)hipFree(p);
    std::lock_guard<std::mutex> lock(mu);
    leaving -= blocks.size();
    if (leaving == 0) left.notify_all();
  }
};
constexpr int kPoolDevices = 64;
DevPool g_pools[kPoolDevices];
DevPool* pool_of(const mfe_ctx* ctx) {
  return ctx->device >= 0 && ctx->device < kPoolDevices ? &g_pools[ctx->device] : nullptr;
}
}  // namespace

// Gives every block kept on ctx's device back to the driver; their bytes.  On
// return what other threads were giving back is free too.
static size_t dev_trim(mfe_ctx* ctx) {
  DevPool* P = pool_of(ctx);
  if (!P) return 0;
  std::vector<void*> all;
  size_t bytes = 0;
  {
    std::lock_guard<std::mutex> lock(P->mu);
    bytes = P->idle_bytes;
    for (auto it = P->idle.begin(); it != P->idle.end();) it = P->take(it, all);
    P->leaving += all.size();
  }
  P->release(all);
  std::unique_lock<std::mutex> lock(P->mu);
  P->left.wait(lock, [&] { return P->leaving == 0; });
  return bytes;
}

hipError_t dev_malloc_bytes(mfe_ctx* ctx, void** out, size_t bytes) {
  hipError_t e = hipMalloc(out, bytes);
  if (e == hipSuccess) return e;
  (void)hipGetLastError();
  (void)dev_trim(ctx);
  e = hipMalloc(out, bytes);  // (also where another thread gave the memory back)
  if (e != hipSuccess) {
    (void)hipGetLastError();  // nothing sticky: the caller decides
    *out = nullptr;
  }
  return e;
}

hipError_t dev_alloc_bytes(mfe_ctx* ctx, void** out, size_t bytes) {
  *out = nullptr;
  DevPool* P = pool_of(ctx);
  if (!P) return dev_malloc_bytes(ctx, out, bytes);
  const size_t unit = bytes < (size_t(1) << 20) ? 512 : size_t(2) << 20;
  const size_t want = (bytes + unit - 1) / unit * unit;
  std::unique_lock<std::mutex> lock(P->mu);
  // the smallest kept block of at most 1/8 more, the oldest of those
  const auto best = P->fit.lower_bound({ctx, want, 0});
  if (best != P->fit.end() && std::get<0>(*best) == ctx &&
      std::get<1>(*best) - want <= want / 8) {
    std::vector<void*> block;
    const size_t got = std::get<1>(*best);
    P->take(P->idle.find(std::get<2>(*best)), block);
    *out = block[0];
    P->live[*out] = got;
    return hipSuccess;
  }
  lock.unlock();
  const hipError_t e = dev_malloc_bytes(ctx, out, want);
  if (e != hipSuccess) return e;
  lock.lock();
  P->live[*out] = want;
  return hipSuccess;
}

void dev_free(mfe_ctx* ctx, void* p, bool shared) {
  if (!p) return;
  DevPool* P = pool_of(ctx);
  if (!P) {
    (void)hipFree(p);
    return;
  }
  std::vector<void*> gone;
  {
    std::lock_guard<std::mutex> lock(P->mu);
    auto it = P->live.find(p);
    const size_t bytes = it == P->live.end() ? 0 : it->second;
    if (it != P->live.end()) P->live.erase(it);
    if (shared || bytes == 0) {
      gone.push_back(p);
    } else {
      if (!P->cap) {
        size_t free_b = 0, total = 0;
        if (hipMemGetInfo(&free_b, &total) == hipSuccess) P->cap = total / 8;
      }
      P->keep(ctx, p, bytes);
      for (auto old = P->idle.begin(); P->idle_bytes > P->cap && old != P->idle.end();)
        old = P->take(old, gone);
    }
    P->leaving += gone.size();
  }
  P->release(gone);
}

// The blocks kept for ctx go (its stream has drained).
static void dev_drop(mfe_ctx* ctx) {
  DevPool* P = pool_of(ctx);
  if (!P) return;
  std::vector<void*> gone;
  {
    std::lock_guard<std::mutex> lock(P->mu);
    for (auto it = P->idle.begin(); it != P->idle.end();)
      it = it->second.ctx == ctx ? P->take(it, gone) : std::next(it);
    P->leaving += gone.size();
  }
  P->release(gone);
}

// Largest non-zero count of any kSpmvRows-row tile: ro[min(r0+R,n)] - ro[r0].
__global__ void tile_nnz_max_kernel(int64_t n, const int* __restrict__ ro, int64_t ntiles,
                                    unsigned long long* out) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntiles) return;
  int64_t r0 = t * kSpmvRows;
  int64_t r1 = r0 + kSpmvRows < n ? r0 + kSpmvRows : n;
  long long c = (long long)ro[r1] - (long long)ro[r0];
  atomicMax(out, (unsigned long long)(c < 0 ? 0 : c));
}

// Uploads from pageable host memory start the runtime's copy machinery,
// which costs several ms the first time in a process; small host lists the
// kernels only read once (impose_dirichlet's BC rows) are read by the kernels
// straight from this pinned buffer instead.
int stage_buffer(mfe_ctx* ctx, void** out) {
  if (!ctx->h_stage) MFE_CHECK(ctx, hipHostMalloc(&ctx->h_stage, kStageBytes, hipHostMallocDefault));
  *out = ctx->h_stage;
  return MFE_OK;
}

// dst[i] = src[i] for i < nb, four bytes per thread.
__global__ void copy_bytes_kernel(int64_t nb, const unsigned char* __restrict__ src,
                                  unsigned char* __restrict__ dst) {
  const int64_t i0 = 4 * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (i0 + k < nb) dst[i0 + k] = src[i0 + k];
}

static int staged_copy(mfe_ctx* ctx, void* dst, const void* src, size_t bytes, bool up) {
  if (bytes == 0) return MFE_OK;
  void* stage = nullptr;
  int st = stage_buffer(ctx, &stage);
  if (st) return st;
  const unsigned char* s = static_cast<const unsigned char*>(src);
  unsigned char* d = static_cast<unsigned char*>(dst);
  unsigned char* pin = static_cast<unsigned char*>(stage);
  for (size_t off = 0; off < bytes; off += kStageBytes) {
    const size_t len = bytes - off < kStageBytes ? bytes - off : kStageBytes;
    if (up) std::memcpy(pin, s + off, len);
    copy_bytes_kernel<<<(unsigned)cdiv((int64_t)cdiv((int64_t)len, 4), kBlock), kBlock, 0,
                        ctx->stream>>>((int64_t)len, up ? pin : s + off, up ? d + off : pin);
    MFE_LAUNCHED(ctx, "copy_bytes_kernel");
    MFE_CHECK(ctx, hipStreamSynchronize(ctx->stream));  // the buffer is reused next
    if (!up) std::memcpy(d + off, pin, len);
  }
  return MFE_OK;
}

int upload_bytes(mfe_ctx* ctx, void* dst, const void* src, size_t bytes) {
  return staged_copy(ctx, dst, src, bytes, true);
}

int download_bytes(mfe_ctx* ctx, void* dst, const void* src, size_t bytes) {
  return staged_copy(ctx, dst, src, bytes, false);
}

int plan_spmv(mfe_ctx* ctx, mfe_csr* A) {
  if (A->nrows == 0) {
    A->max_block_nnz = 0;
    return MFE_OK;
  }
  int64_t ntiles = cdiv(A->nrows, kSpmvRows);
  unsigned long long* d = reinterpret_cast<unsigned long long*>(ctx->d_scalars);
  MFE_CHECK(ctx, hipMemsetAsync(d, 0, sizeof(*d), ctx->stream));
  tile_nnz_max_kernel<<<(unsigned)cdiv(ntiles, kBlock), kBlock, 0, ctx->stream>>>(
      A->nrows, A->row_offsets, ntiles, d);
  MFE_LAUNCHED(ctx, "tile_nnz_max_kernel");
  MFE_CHECK(ctx, hipMemcpyAsync(ctx->h_scalars, d, sizeof(*d), hipMemcpyDeviceToHost,
                                ctx->stream));
  MFE_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  unsigned long long v;
  std::memcpy(&v, ctx->h_scalars, sizeof(v));
  A->max_block_nnz = (int64_t)v;
  return MFE_OK;
}

}  // namespace mfe

using namespace mfe;

extern "C" {

int mfe_ctx_create(int device, mfe_ctx** out) {
  if (!out) return MFE_BAD_ARG;
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return MFE_HIP_ERROR;
  if (device < 0 || device >= ndev) return MFE_BAD_ARG;
  mfe_ctx* c = new mfe_ctx();
  c->device = device;
  auto bail = [&](int st) {
    mfe_ctx_destroy(c);
    return st;
  };
  if (hipSetDevice(device) != hipSuccess) return bail(MFE_HIP_ERROR);
  // Default-priority, non-blocking stream (no priority variants are used).
  if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess)
    return bail(MFE_HIP_ERROR);
  if (hipEventCreate(&c->t_start) != hipSuccess || hipEventCreate(&c->t_stop) != hipSuccess)
    return bail(MFE_HIP_ERROR);
  if (dev_malloc(c, &c->d_scalars, 64 * sizeof(double)) != hipSuccess) return bail(MFE_OOM);
  if (hipHostMalloc(&c->h_scalars, 64 * sizeof(double), hipHostMallocDefault) != hipSuccess)
    return bail(MFE_OOM);
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) == hipSuccess) c->cu_count = prop.multiProcessorCount;
  if (int st = noalloc_scratch_init(c)) return bail(st);
  *out = c;
  return MFE_OK;
}

void mfe_cg_workspace_free(mfe_ctx* ctx);     // mfe_solve.hip
void mfe_multi_workspace_free(mfe_ctx* ctx);  // mfe_multi.hip

void mfe_ctx_destroy(mfe_ctx* c) {
  if (c) ctx_release(c);
}

}  // extern "C"

namespace mfe {
void ctx_release(mfe_ctx* c) {
  if (c->refs.fetch_sub(1, std::memory_order_acq_rel) != 1) return;
  hipSetDevice(c->device);
  if (c->stream) hipStreamSynchronize(c->stream);
  dev_drop(c);
  mfe_cg_workspace_free(c);
  mfe_multi_workspace_free(c);
  if (c->d_partials) hipFree(c->d_partials);
  if (c->d_scalars) hipFree(c->d_scalars);
  if (c->h_scalars) hipHostFree(c->h_scalars);
  if (c->h_stage) hipHostFree(c->h_stage);
  if (c->t_start) hipEventDestroy(c->t_start);
  if (c->t_stop) hipEventDestroy(c->t_stop);
  if (c->stream) hipStreamDestroy(c->stream);
  delete c;
}
}  // namespace mfe

extern "C" {

const char* mfe_last_error(const mfe_ctx* ctx) { return ctx ? ctx->err.c_str() : "null ctx"; }

int mfe_ctx_synchronize(mfe_ctx* ctx) {
  if (!ctx) return MFE_BAD_ARG;
  MFE_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  return MFE_OK;
}

int mfe_trim_memory(mfe_ctx* ctx, int64_t* bytes) {
  if (!ctx) return MFE_BAD_ARG;
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  const size_t freed = dev_trim(ctx);
  if (bytes) *bytes = (int64_t)freed;
  return MFE_OK;
}

int mfe_device_info(mfe_ctx* ctx, char* name, int name_len, int* cu_count, int64_t* hbm) {
  if (!ctx) return MFE_BAD_ARG;
  hipDeviceProp_t prop;
  MFE_CHECK(ctx, hipGetDeviceProperties(&prop, ctx->device));
  if (name && name_len > 0) {
    std::snprintf(name, (size_t)name_len, "%s (%s)", prop.name, prop.gcnArchName);
  }
  if (cu_count) *cu_count = prop.multiProcessorCount;
  if (hbm) *hbm = (int64_t)prop.totalGlobalMem;
  return MFE_OK;
}

int mfe_timer_start(mfe_ctx* ctx) {
  if (!ctx) return MFE_BAD_ARG;
  MFE_CHECK(ctx, hipEventRecord(ctx->t_start, ctx->stream));
  return MFE_OK;
}

int mfe_timer_stop(mfe_ctx* ctx, double* ms) {
  if (!ctx || !ms) return MFE_BAD_ARG;
  MFE_CHECK(ctx, hipEventRecord(ctx->t_stop, ctx->stream));
  MFE_CHECK(ctx, hipEventSynchronize(ctx->t_stop));
  float f = 0;
  MFE_CHECK(ctx, hipEventElapsedTime(&f, ctx->t_start, ctx->t_stop));
  *ms = f;
  return MFE_OK;
}

// ---- CSRMatrix ------------------------------------------------------------

static void csr_release(mfe_csr* A) {
  for (void* p : {(void*)A->rows, (void*)A->row_offsets, (void*)A->cols, (void*)A->vals,
                  (void*)A->vals32})
    csr_free(A, p);
  A->rows = A->row_offsets = A->cols = nullptr;
  A->vals = nullptr;
  A->vals32 = nullptr;
  sell_release(A);
  box_release(A);
  csr_structure_changed(A);
  A->nrows = A->nnz = 0;
  A->has_local_indices = false;
  A->num_cols = 0;
}

int mfe_csr_create(mfe_ctx* ctx, mfe_csr** out) {
  if (!ctx || !out) return MFE_BAD_ARG;
  *out = new mfe_csr();
  (*out)->ctx = ctx;
  (*out)->plan_gen = next_plan_gen();
  ctx_retain(ctx);
  return MFE_OK;
}

void mfe_csr_destroy(mfe_csr* A) {
  if (!A) return;
  hipSetDevice(A->ctx->device);
  hipStreamSynchronize(A->ctx->stream);
  csr_release(A);
  mfe_ctx* ctx = A->ctx;
  delete A;
  ctx_release(ctx);
}

int mfe_csr_shape(const mfe_csr* A, int64_t* nrows, int64_t* nnz) {
  if (!A) return MFE_BAD_ARG;
  if (nrows) *nrows = A->nrows;
  if (nnz) *nnz = A->nnz;
  return MFE_OK;
}

}  // extern "C"

namespace mfe {
// (Re)allocate A's arrays for nrows/nnz; contents undefined.
int csr_alloc(mfe_ctx* ctx, mfe_csr* A, int64_t nrows, int64_t nnz) {
  uses(ctx, A);
  MFE_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  csr_release(A);
  if (nrows < 0 || nnz < 0 || nnz > INT32_MAX || nrows >= INT32_MAX)
    return fail(ctx, MFE_UNSUPPORTED, "matrix exceeds int32 ordinals");
  MFE_CHECK(ctx, dev_alloc(ctx, &A->rows, sizeof(int) * (size_t)(nrows > 0 ? nrows : 1)));
  MFE_CHECK(ctx, dev_alloc(ctx, &A->row_offsets, sizeof(int) * (size_t)(nrows + 1)));
  MFE_CHECK(ctx, dev_alloc(ctx, &A->cols, sizeof(int) * (size_t)(nnz > 0 ? nnz : 1)));
  MFE_CHECK(ctx, dev_alloc(ctx, &A->vals, sizeof(double) * (size_t)(nnz > 0 ? nnz : 1)));
  A->nrows = nrows;
  A->nnz = nnz;
  return MFE_OK;
}

__global__ void iota_kernel(int64_t n, int* out) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = (int)i;
}
}  // namespace mfe

extern "C" {

int mfe_csr_upload(mfe_ctx* ctx, mfe_csr* A, int64_t nrows, int64_t nnz, const int* rows,
                   const int* row_offsets, const int* cols, const double* vals) {
  if (!ctx || !A || !row_offsets || (nnz > 0 && (!cols || !vals))) return MFE_BAD_ARG;
  if (nrows < 0 || nnz < 0) return fail(ctx, MFE_BAD_ARG, "csr_upload: negative nrows or nnz");
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  if (row_offsets[0] != 0 || row_offsets[nrows] != nnz)
    return fail(ctx, MFE_BAD_ARG, "row_offsets must start at 0 and end at nnz");
  for (int64_t i = 0; i < nrows; ++i)
    if (row_offsets[i + 1] < row_offsets[i])
      return fail(ctx, MFE_BAD_ARG, "row_offsets must be non-decreasing");
  for (int64_t j = 0; j < nnz; ++j)
    if (cols[j] < 0 || cols[j] >= nrows)
      return fail(ctx, MFE_BAD_ARG, "column index out of range (one rank: cols < nrows)");
  // One rank owns rows 0..nrows-1 (first_local_row = 0): impose_dirichlet,
  // the element loop and verify_solution index rows by position, as the
  // reference does through rows[i] - first_local_row
  // (SparseMatrix_functions.hpp:446-478).
  if (rows)
    for (int64_t i = 0; i < nrows; ++i)
      if (rows[i] != (int)i)
        return fail(ctx, MFE_BAD_ARG, "rows[i] must equal i (one rank owns rows 0..nrows-1)");
  int st = csr_alloc(ctx, A, nrows, nnz);
  if (st) return st;
  hipStream_t s = ctx->stream;
  if (rows) {
    MFE_CHECK(ctx, hipMemcpyAsync(A->rows, rows, sizeof(int) * nrows, hipMemcpyHostToDevice, s));
  } else if (nrows > 0) {
    iota_kernel<<<(unsigned)cdiv(nrows, kBlock), kBlock, 0, s>>>(nrows, A->rows);
    MFE_LAUNCHED(ctx, "iota_kernel");
  }
  MFE_CHECK(ctx, hipMemcpyAsync(A->row_offsets, row_offsets, sizeof(int) * (nrows + 1),
                                hipMemcpyHostToDevice, s));
  if (nnz > 0) {
    MFE_CHECK(ctx, hipMemcpyAsync(A->cols, cols, sizeof(int) * nnz, hipMemcpyHostToDevice, s));
    MFE_CHECK(ctx,
              hipMemcpyAsync(A->vals, vals, sizeof(double) * nnz, hipMemcpyHostToDevice, s));
  }
  A->has_local_indices = false;
  A->num_cols = nrows;
  return plan_spmv(ctx, A);
}

int mfe_csr_download(mfe_ctx* ctx, const mfe_csr* A, int* rows, int* row_offsets, int* cols,
                     double* vals) {
  if (!ctx || !A) return MFE_BAD_ARG;
  uses(ctx, A);
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  hipStream_t s = ctx->stream;
  if (rows && A->nrows)
    MFE_CHECK(ctx, hipMemcpyAsync(rows, A->rows, sizeof(int) * A->nrows, hipMemcpyDeviceToHost, s));
  if (row_offsets && A->row_offsets)
    MFE_CHECK(ctx, hipMemcpyAsync(row_offsets, A->row_offsets, sizeof(int) * (A->nrows + 1),
                                  hipMemcpyDeviceToHost, s));
  if (cols && A->nnz)
    MFE_CHECK(ctx, hipMemcpyAsync(cols, A->cols, sizeof(int) * A->nnz, hipMemcpyDeviceToHost, s));
  if (vals && A->nnz)
    MFE_CHECK(ctx,
              hipMemcpyAsync(vals, A->vals, sizeof(double) * A->nnz, hipMemcpyDeviceToHost, s));
  MFE_CHECK(ctx, hipStreamSynchronize(s));
  return MFE_OK;
}

int mfe_make_local_matrix(mfe_ctx* ctx, mfe_csr* A) {
  if (!ctx || !A) return MFE_BAD_ARG;
  // One rank (make_local_matrix.hpp:437-441): every column is local.
  A->num_cols = A->nrows;
  A->has_local_indices = true;
  return MFE_OK;
}

// ---- Vector ----------------------------------------------------------------

int mfe_vec_create(mfe_ctx* ctx, int64_t n, mfe_vec** out) {
  if (!ctx || !out || n < 0) return MFE_BAD_ARG;
  *out = nullptr;
  MFE_CHECK(ctx, hipSetDevice(ctx->device));
  mfe_vec* v = new mfe_vec();
  v->ctx = ctx;
  v->n = n;
  hipError_t e = dev_alloc(ctx, &v->d, sizeof(double) * (size_t)(n > 0 ? n : 1));
  if (e != hipSuccess) {
    delete v;
    return hip_fail(ctx, e, "hipMalloc(vector)");
  }
  e = hipMemsetAsync(v->d, 0, sizeof(double) * (size_t)(n > 0 ? n : 1), ctx->stream);
  if (e != hipSuccess) {
    dev_free(ctx, v->d);
    delete v;
    return hip_fail(ctx, e, "hipMemsetAsync(vector)");
  }
  ctx_retain(ctx);
  *out = v;
  return MFE_OK;
}

void mfe_vec_destroy(mfe_vec* v) {
  if (!v) return;
  hipSetDevice(v->ctx->device);
  hipStreamSynchronize(v->ctx->stream);
  if (v->owns) dev_free(v->ctx, v->d, v->shared);
  mfe_ctx* ctx = v->ctx;
  delete v;
  ctx_release(ctx);
}

int mfe_vec_wrap(mfe_ctx* ctx, double* device_ptr, int64_t n, mfe_vec** out) {
  if (!ctx || !out || n < 0 || (n > 0 && !device_ptr)) return MFE_BAD_ARG;
  hipPointerAttribute_t attr;
  if (n > 0 && (hipPointerGetAttributes(&attr, device_ptr) != hipSuccess ||
                attr.type != hipMemoryTypeDevice || attr.device != ctx->device))
    return fail(ctx, MFE_BAD_ARG, "mfe_vec_wrap: not device memory of this context's GPU");
  mfe_vec* v = new mfe_vec();
  v->ctx = ctx;
  v->n = n;
  v->d = device_ptr;
  v->owns = false;
  ctx_retain(ctx);
  *out = v;
  return MFE_OK;
}

int64_t mfe_vec_size(const mfe_vec* v) { return v ? v->n : -1; }

int mfe_vec_upload(mfe_ctx* ctx, mfe_vec* v, const double* host, int64_t n) {
  if (!ctx || !v || (n > 0 && !host) || n != v->n) return MFE_BAD_ARG;
  uses(ctx, v);
  if (n) MFE_CHECK(ctx, hipMemcpyAsync(v->d, host, sizeof(double) * n, hipMemcpyHostToDevice,
                                       ctx->stream));
  MFE_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  return MFE_OK;
}

int mfe_vec_download(mfe_ctx* ctx, const mfe_vec* v, double* host, int64_t n) {
  if (!ctx || !v || (n > 0 && !host) || n != v->n) return MFE_BAD_ARG;
  uses(ctx, v);
  if (n) MFE_CHECK(ctx, hipMemcpyAsync(host, v->d, sizeof(double) * n, hipMemcpyDeviceToHost,
                                       ctx->stream));
  MFE_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  return MFE_OK;
}

}  // extern "C"

namespace mfe {
__global__ void fill_kernel(int64_t n, double v, double* __restrict__ out) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = v;
}
}  // namespace mfe

extern "C" {

int mfe_vec_fill(mfe_ctx* ctx, mfe_vec* v, double value) {
  if (!ctx || !v) return MFE_BAD_ARG;
  uses(ctx, v);
  if (v->n == 0) return MFE_OK;
  fill_kernel<<<(unsigned)cdiv(v->n, kBlock), kBlock, 0, ctx->stream>>>(v->n, value, v->d);
  MFE_LAUNCHED(ctx, "fill_kernel");
  return MFE_OK;
}

// ---- verification (host) -----------------------------------------------------

// analytic_soln.hpp:51-112: the Fourier series (Carslaw & Jaeger) of the
// steady temperature in the unit cube held at 1 on the face x = 1 and at 0 on
// the other five, over odd wave numbers a = 2p+1 in y and c = 2q+1 in z:
//   u = 16/pi^2 sum_a sum_c sinh(lam x)/sinh(lam) sin(a pi y)/a sin(c pi z)/c,
//   lam = pi sqrt(a^2 + c^2).
// A term that is NaN (sinh overflows for large lam) ends its inner sum.  The
// products are grouped as the reference groups them, so the verification
// error has the reference's bits.
double mfe_soln(double x, double y, double z, int max_p, int max_q) {
  const double pi = 3.141592653589793238462;
  const double pi2 = pi * pi;
  double total = 0;
  for (int p = 0; p <= max_p; ++p) {
    const int a = 2 * p + 1;
    const double wy = std::sin(a * pi * y) / a;
    for (int q = 0; q <= max_q; ++q) {
      const int c = 2 * q + 1;
      const double wz = std::sin(c * pi * z) / c;
      const double lam = std::sqrt(a * a * pi2 + c * c * pi2);
      const double term = (std::sinh(lam * x) * wy) * (wz / std::sinh(lam));
      if (std::isnan(term)) break;
      total += term;
    }
  }
  return 16.0 / pi2 * total;
}

// verify_solution.hpp:55-174.  Only the checked nodes are copied to the host.
int mfe_verify_solution(mfe_ctx* ctx, const int g[6], const mfe_vec* xv, double tolerance,
                        int whole, double* max_err) {
  return mfe_verify_solution_ex(ctx, g, xv, tolerance, whole, 1, max_err);
}

int mfe_verify_solution_ex(mfe_ctx* ctx, const int g[6], const mfe_vec* xv, double tolerance,
                           int whole, int hot_face, double* max_err) {
  if (!ctx || !g || !xv) return MFE_BAD_ARG;
  uses(ctx, xv);
  const int gx = g[1] + 1, gy = g[3] + 1, gz = g[5] + 1;
  if (g[0] != 0 || g[2] != 0 || g[4] != 0 || (int64_t)gx * gy * gz != xv->n)
    return fail(ctx, MFE_BAD_ARG, "verify_solution: box does not match x");
  const int xdiv = gx > 1 ? gx - 1 : 1, ydiv = gy > 1 ? gy - 1 : 1, zdiv = gz > 1 ? gz - 1 : 1;
  MFE_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  std::vector<double> host;
  if (whole) {
    host.resize((size_t)xv->n);
    int st = mfe_vec_download(ctx, xv, host.data(), xv->n);
    if (st) return st;
  }
  double maxe = 0.0;
  for (int iz = 0; iz < gz; ++iz) {
    double z = (1.0 * iz) / zdiv;
    if (!whole && !(std::abs(z - 0.5) < 0.05)) continue;
    for (int iy = 0; iy < gy; ++iy) {
      double y = 1.0 * iy / ydiv;
      if (!whole && !(std::abs(y - 0.5) < 0.05)) continue;
      for (int ix = 0; ix < gx; ++ix) {
        double x = 1.0 * ix / xdiv;
        if (!whole && !(std::abs(x - 0.5) < 0.05)) continue;
        int64_t id = ix + (int64_t)gx * iy + (int64_t)gx * gy * iz;
        double computed;
        if (whole) {
          computed = host[(size_t)id];
        } else {
          MFE_CHECK(ctx, hipMemcpy(&computed, xv->d + id, sizeof(double), hipMemcpyDeviceToHost));
        }
        // hot_face 0 (u = 1 on x = 0): the mirrored solution soln(1 - x, y, z)
        double a;
        if (hot_face ? x == 1.0 : x == 0.0) a = 1;
        else if (x == 0.0 || x == 1.0 || y == 0.0 || z == 0.0) a = 0;
        else if (y == 1.0 || z == 1.0) a = 0;
        else a = mfe_soln(hot_face ? x : 1.0 - x, y, z, 300, 300);
        double err = std::abs(a - computed);
        if (err > maxe) maxe = err;
      }
    }
  }
  if (max_err) *max_err = maxe;
  return maxe > tolerance ? 1 : 0;
}

}  // extern "C"
