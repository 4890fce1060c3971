/*
 * minife_hip.h -- C-ABI of libminife_hip.so, the MI355X (gfx950) implementation
 * of miniFE's assemble-and-solve path.
 *
 * The reference (Mantevo miniFE, ref/) has no FFI: its operators are C++
 * templates in namespace miniFE.  Each entry point below replaces one of them;
 * the comment names the reference interface (file:line, relative to the
 * reference root).  The C++ layer minife_amd/host/miniFE_hip.hpp keeps the
 * reference names and signatures on top of these entry points.
 *
 * Conventions
 *   - Plain C types only; every call returns an mfe_status (0 = MFE_OK).
 *     mfe_last_error(ctx) holds a message for the last failure on ctx.
 *   - One rank: local box == global box (the id->row map of
 *     simple_mesh_description is the identity).  Boxes are int[6] =
 *     {x0,x1,y0,y1,z0,z1} in elements, as ref/utils/Box.hpp.
 *   - Ordinals are int32 and Scalar is double, as ref/src/Makefile.gnu.serial;
 *     nnz must stay below 2^31 (the reference's LocalOrdinal is int).
 *   - Handles own device memory.  What destroyed matrices and vectors held is
 *     kept for later ones on the same context, at most an eighth of the
 *     device's memory over all contexts, until an allocation of the library
 *     fails, mfe_trim_memory is called or the context goes; the memory of one that was used on another context than
 *     its own goes back to the driver when it is destroyed.  Host pointers are
 *     borrowed for the call.
 *     Calls on one ctx are ordered on its single HIP stream; a ctx is not
 *     thread-safe.  No C++ exception crosses this boundary.
 */
#ifndef MINIFE_HIP_H
#define MINIFE_HIP_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef enum mfe_status {
  MFE_OK = 0,
  MFE_BREAKDOWN = 1,   /* cg_solve.hpp:186-200 numerical breakdown */
  MFE_NOT_LOCAL = 2,   /* cg_solve.hpp:99-104 !A.has_local_indices */
  MFE_OOM = 3,         /* generate_matrix_structure.hpp:80-147 allocation failure */
  MFE_HIP_ERROR = 4,
  MFE_BAD_ARG = 5,
  MFE_UNSUPPORTED = 6
} mfe_status;

typedef struct mfe_ctx mfe_ctx;
typedef struct mfe_csr mfe_csr;
typedef struct mfe_vec mfe_vec;
typedef struct mfe_batch mfe_batch;

/* cg_solve flags */
#define MFE_CG_REPLAY       0x1u /* sequential dots: reference's exact trajectory */
#define MFE_CG_TOL_RELATIVE 0x2u /* stop on ||r|| <= tol*||b|| instead of ||r|| <= tol */
#define MFE_CG_EAGER        0x4u /* launch kernels one by one, whatever the size, no HIP graphs */
/* With MFE_CG_EAGER: time as the reference's MINIFE_FUSED build does
 * (cg_solve.hpp:172-175,206-209): each iteration's SpMV and p.Ap sum in
 * MFE_T_MATVECDOT instead of MATVEC + DOT, the breakdown test's norms untimed.
 * The arithmetic is the same either way (matvec_and_dot returns dot(Ap, p)). */
#define MFE_CG_FUSED        0x8u

/* Timer slots of cg_solve's times[5] (ref/utils/mytimer.hpp:36-43). */
#define MFE_T_WAXPY 0
#define MFE_T_DOT 1
#define MFE_T_MATVEC 2
#define MFE_T_MATVECDOT 3
#define MFE_T_TOTAL 4

/* ---- context ----------------------------------------------------------- */
int mfe_ctx_create(int device, mfe_ctx** out);
/* Drops the caller's reference.  Matrices, vectors and batches made on ctx
 * keep it alive until they are destroyed, so handles may be destroyed in any
 * order; the context's stream, graphs and buffers go with the last one. */
void mfe_ctx_destroy(mfe_ctx* ctx);
const char* mfe_last_error(const mfe_ctx* ctx);
int mfe_ctx_synchronize(mfe_ctx* ctx);
/* Gives the memory kept for later matrices and vectors on ctx's device (of all
 * contexts) back to the driver, where other allocators of the process find it;
 * bytes (nullable) receives how much that was. */
int mfe_trim_memory(mfe_ctx* ctx, int64_t* bytes);
/* Device name, compute-unit count and HBM bytes of ctx's device. */
int mfe_device_info(mfe_ctx* ctx, char* name, int name_len, int* cu_count,
                    int64_t* hbm_bytes);
/* Stream-ordered timer on ctx's stream (hipEvent pair): start, then stop
 * returns the elapsed milliseconds between the two marks. */
int mfe_timer_start(mfe_ctx* ctx);
int mfe_timer_stop(mfe_ctx* ctx, double* elapsed_ms);

/* ---- CSRMatrix (ref/src/CSRMatrix.hpp:40-129) --------------------------- */
/* CSRMatrix() constructor, CSRMatrix.hpp:45-54: empty matrix. */
int mfe_csr_create(mfe_ctx* ctx, mfe_csr** out);
void mfe_csr_destroy(mfe_csr* A);
/* rows.size() and num_nonzeros(), CSRMatrix.hpp:84-87. */
int mfe_csr_shape(const mfe_csr* A, int64_t* nrows, int64_t* nnz);
/* Copy a host CSR in.  Replaces contents.  One rank owns rows 0..nrows-1, so
 * rows is NULL or rows[i] == i (MFE_BAD_ARG otherwise); row_offsets must start
 * at 0, not decrease and end at nnz, and 0 <= cols[j] < nrows. */
int mfe_csr_upload(mfe_ctx* ctx, mfe_csr* A, int64_t nrows, int64_t nnz, const int* rows,
                   const int* row_offsets, const int* cols, const double* vals);
/* Copy any subset of the arrays out (NULL pointers are skipped). */
int mfe_csr_download(mfe_ctx* ctx, const mfe_csr* A, int* rows, int* row_offsets,
                     int* cols, double* vals);

/* ---- Vector (ref/src/Vector.hpp:36-61) ---------------------------------- */
/* Vector(startIdx, local_sz), Vector.hpp:42-50: zero-filled. */
int mfe_vec_create(mfe_ctx* ctx, int64_t n, mfe_vec** out);
void mfe_vec_destroy(mfe_vec* v);
int64_t mfe_vec_size(const mfe_vec* v);
/* A vector over caller-owned device memory (e.g. a torch tensor's storage);
 * mfe_vec_destroy releases the handle only.  The memory must stay valid and
 * must not be written by other streams while the library uses it. */
int mfe_vec_wrap(mfe_ctx* ctx, double* device_ptr, int64_t n, mfe_vec** out);
int mfe_vec_upload(mfe_ctx* ctx, mfe_vec* v, const double* host, int64_t n);
int mfe_vec_download(mfe_ctx* ctx, const mfe_vec* v, double* host, int64_t n);
int mfe_vec_fill(mfe_ctx* ctx, mfe_vec* v, double value);

/* ---- assemble ------------------------------------------------------------ */
/* generate_matrix_structure(mesh, A), generate_matrix_structure.hpp:47-149
 * (+ MatrixInitOp<CSRMatrix> MatrixInitOp.hpp:127-156): rows, row_offsets,
 * ascending 27-stencil cols, zero coefficients.  Bit-exact. */
int mfe_generate_matrix_structure(mfe_ctx* ctx, const int global_box[6],
                                  const int local_box[6], mfe_csr* A);

/* perform_element_loop(mesh, elem_box, A, b, params),
 * perform_element_loop.hpp:40-104: hex8 diffusion matrix and source vector per
 * element (Hex8.hpp:259-410), added onto A's values and b (sum_into_row
 * adds).  Each entry receives its elements' contributions in ascending
 * element id, so the result is bit-identical to the reference.  A must hold
 * the box's structure: the one mfe_generate_matrix_structure writes (a copy
 * uploaded with mfe_csr_upload is verified on the device first); otherwise
 * MFE_BAD_ARG.  kappa (nullable, one double per element) is the per-element
 * conductivity k of Hex8.hpp:273 (reference: 1.0). */
int mfe_perform_element_loop(mfe_ctx* ctx, const int global_box[6], const int elem_box[6],
                             mfe_csr* A, mfe_vec* b, const mfe_vec* kappa);
/* assemble_FE_data(mesh, A, b, params), assemble_FE_data.hpp:38-73. */
int mfe_assemble_FE_data(mfe_ctx* ctx, const int global_box[6], const int local_box[6],
                         mfe_csr* A, mfe_vec* b, const mfe_vec* kappa);
/* assemble_FE_data with the element source Q (sourceVector's Q, Hex8.hpp:379;
 * the reference uses 1.0, which mfe_assemble_FE_data passes; 0 gives the
 * source-free problem).  Q = 1.0 gives the same bits as mfe_assemble_FE_data. */
int mfe_assemble_FE_data_ex(mfe_ctx* ctx, const int global_box[6], const int local_box[6],
                            mfe_csr* A, mfe_vec* b, const mfe_vec* kappa, double source);

/* impose_dirichlet(value, A, b, gnx, gny, gnz, bc_rows),
 * SparseMatrix_functions.hpp:431-480: bc_rows is the reference's std::set as a
 * sorted host array.  BC rows become identity rows with b = value; other rows
 * drop their BC columns and subtract their (column-ordered) sum * value. */
int mfe_impose_dirichlet(mfe_ctx* ctx, double prescribed_value, mfe_csr* A, mfe_vec* b,
                         int global_nx, int global_ny, int global_nz, const int* bc_rows,
                         int64_t num_bc_rows);

/* make_local_matrix(A), make_local_matrix.hpp:42-442 (one rank: num_cols =
 * nrows, has_local_indices = true). */
int mfe_make_local_matrix(mfe_ctx* ctx, mfe_csr* A);

/* ---- solve --------------------------------------------------------------- */
/* SpMV storage plan (no reference counterpart: the reference always runs its
 * CSR loop).  MFE_SPMV_AUTO (default), when A holds the structure
 * generate_matrix_structure writes for a box (or the element loop has verified
 * that it does), keeps the values in the box layout: per block of 16 x 16
 * nodes, per z plane and per stencil slot, 256 consecutive values (rows padded
 * to 27 slots); the SpMV marches each block along z with three planes of x in
 * LDS and reads no column indices.  When every A[r][c] equals A[c][r] bit for
 * bit (checked when the plan is built; the assembled operator is symmetric)
 * each row stores only its 14 upper slots and takes the other 13 from its
 * neighbours' (the symmetric box layout, about 15 values per row instead of
 * 27).  Its upper values (FP64, and the FP32 copy of the mixed solve) are
 * further packed: per (block, plane, stencil slot) a power of two q that
 * divides every value and a base kb, and per value an unsigned field f of
 * 10, 12 or 16 bits (22 or 24, or for FP64 32, for the 3 analytically zero
 * face-neighbour slots), the value being (kb + f) * q exactly; +0.0 and 1.0
 * have codes of their own.  The assembled operator's entries vary only in
 * their last bits from node to node, so narrow fields hold them; the plan
 * takes, of the forms every value fits, the one with the fewest bytes per
 * row, and checks every value; other matrices keep the full values.
 * Otherwise MFE_SPMV_AUTO keeps a SELL-64 copy of A beside the CSR
 * arrays -- slices of 64 rows, one row per lane, slot j of a slice stored as
 * 64 consecutive values/columns -- built on first use and rebuilt after the
 * values or structure change -- and, per 256-row tile, a staged-x plan: the
 * tile's distinct columns as runs of consecutive columns, with 16-bit local
 * columns per slot (or, for a slice whose local columns are base_j + lane,
 * just the 27 bases), so the SpMV copies the tile's x entries into LDS once
 * and gathers from there.  A tile with more than 128 runs leaves the matrix on
 * plain SELL-64; a row longer than 27 entries, or a copy that does not fit in
 * device memory, on the CSR kernels.  MFE_SPMV_SELL: SELL-64 without the
 * staged x.  MFE_SPMV_CSR frees the copies and uses the CSR kernels only.
 * Every format sums each row in stored column order, so results are
 * bit-identical. */
#define MFE_SPMV_AUTO 0
#define MFE_SPMV_CSR 1
#define MFE_SPMV_SELL 2
/* Sets A's format and builds its FP64 plan now (so later solves do not pay
 * for it).  info (nullable) receives {kernel in use: 0 CSR row-stream,
 * 1 SELL-64, 2 CSR row-per-thread, 3 SELL-64 with staged x, 4 box layout,
 * 5 symmetric box layout, 6 symmetric box layout with packed upper values;
 * stored entries incl. padding; slices (box: workgroups); longest row (6:
 * the packed form of the FP64 values in bits 0-7 -- 1 all 14 slots in 16
 * bits, 2 eleven in 16 and the three near-zero ones in 32, 3 eleven in 16
 * (the three at full width), 4 all in 12, 5 eleven in 12 and three in 24, 6
 * all in 10, 7 eleven in 10 and three in 22 -- and, once the FP32 copy
 * exists, of the FP32 values in bits 8-15; the FP64 boundary stream's form
 * in bits 16-23, 0 where it has none -- the CG reads it so from 2^23 rows on,
 * and at full width below); and
 * for the staged-x plan (else 0): runs; most distinct columns of a 256-row
 * tile; stored entries whose local columns are read; slices read as base +
 * lane instead (every row of the slice as wide as the slice, slot j's local
 * column = base_j + lane) -- for the box layout: planes per z chunk, blocks
 * along x, blocks along y, z chunks}.  Workgroup partial sums (p.Ap in the
 * fast CG) group rows per 256-row tile in the CSR and SELL formats and per
 * workgroup in the box layout, so fast-mode dots may differ in the last bits
 * between the two; replay mode's dots do not depend on the format. */
int mfe_spmv_plan(mfe_ctx* ctx, mfe_csr* A, int format, int64_t info[8]);
/* matvec_std<CSRMatrix>::operator()(A, x, y), SparseMatrix_functions.hpp:545-578.
 * Each row's products are summed in stored column order: bit-identical. */
int mfe_matvec(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* x, mfe_vec* y);
/* matvec_and_dot(A, x, y), SparseMatrix_functions.hpp:491-536: y = A x and
 * returns x.y (two-level tree reduction). */
int mfe_matvec_and_dot(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* x, mfe_vec* y,
                       double* result);
/* No counterpart in the reference: mfe_matvec_and_dot for callers that cannot
 * allocate device memory (code under HIP graph capture, serving loops,
 * harnesses that forbid hipMalloc).  It calls no hipMalloc/hipFree: the
 * per-tile partials live in a fixed 1 MiB device array of the library (one
 * copy per GPU, held until the process ends), so A may have at most
 * 33,554,432 rows (MFE_BAD_ARG beyond), and A's SpMV plan must already be
 * built (mfe_spmv_plan or any SpMV after A's last change; MFE_BAD_ARG
 * otherwise).  y = A x as mfe_matvec_and_dot computes it; x.y (the same bits)
 * is written to result_device, one double of device memory, on ctx's stream,
 * without synchronising.  Calls that overlap on one GPU (from two contexts)
 * share the array and race. */
int mfe_matvec_and_dot_noalloc(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* x, mfe_vec* y,
                               double* result_device);
/* dot(x, y), Vector_functions.hpp:194-226, as a deterministic two-level
 * (wave64 shuffle + LDS) tree reduction. */
int mfe_dot(mfe_ctx* ctx, const mfe_vec* x, const mfe_vec* y, double* result);
/* dot(x, y) summed strictly left to right, as the reference: bit-identical. */
int mfe_dot_replay(mfe_ctx* ctx, const mfe_vec* x, const mfe_vec* y, double* result);
/* waxpby(alpha, x, beta, y, w), Vector_functions.hpp:127-150. */
int mfe_waxpby(mfe_ctx* ctx, double alpha, const mfe_vec* x, double beta, const mfe_vec* y,
               mfe_vec* w);

/* cg_solve(A, b, x, matvec_std, max_iter, tolerance, num_iters, normr, times),
 * cg_solve.hpp:69-229: unpreconditioned CG from the initial x.  Iteration k
 * runs while k <= max_iter and the residual norm computed at the start of the
 * previous iteration exceeds tolerance (the reference's loop test), so
 * num_iters and normr mean what they mean there.  Returns MFE_OK or
 * MFE_BREAKDOWN (num_iters = last completed k).  times (nullable) receives
 * seconds in the MFE_T_* slots: TOTAL always; WAXPY, DOT and MATVEC (and
 * MATVECDOT with MFE_CG_FUSED) only with MFE_CG_EAGER (GPU time between kernel
 * groups; otherwise they stay 0: the fused kernels and graph launches cannot be
 * split).  history (nullable) receives 4 doubles per iteration k (entry k-1): {rtrans, p_ap_dot, alpha, beta}.
 * flags: MFE_CG_REPLAY reproduces the reference's sequential dot products and
 * hence its scalar trajectory bit for bit; the default fast mode uses tree
 * reductions (deterministic, not bit-identical to the serial sum). */
int mfe_cg_solve(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* b, mfe_vec* x, int max_iter,
                 double tolerance, unsigned flags, int* num_iters, double* normr,
                 double* times, double* history);

/* ---- adjoint (extension; no counterpart in the reference) ------------------
 * grad[e] = -lambda_e^T K_e(1) utilde_e for every element e of the global box:
 * K_e(1) is Hex8::diffusionMatrix_symm with k = 1 (Hex8.hpp:259-361), the
 * derivative of the assembled operator with respect to the element
 * conductivity kappa_e; lambda and utilde are nodal vectors (n = nodes), grad
 * has one entry per element.  With lambda the adjoint solution (zero on
 * Dirichlet rows) and utilde the solution with its bc_rows_0 entries set to 0
 * (the values the reference's Dirichlet lifting uses), grad is dL/dkappa.
 * Sum order per element: for i: t = sum_j K_ij utilde_j (j ascending);
 * s += lambda_i t; grad = -s. */
int mfe_element_gradient(mfe_ctx* ctx, const int global_box[6], const mfe_vec* lambda,
                         const mfe_vec* utilde, mfe_vec* grad);

/* ---- mixed precision (extension; no counterpart in the reference) --------
 * Iterative refinement around cg_solve: the inner solve is unpreconditioned
 * CG entirely in FP32 (FP32 copy of A's values sharing the int32 columns;
 * SpMV products, row sums, axpys and dot products in FP32) on the residual
 * scaled to unit norm, run to ||r_in|| <= inner_tol (looser, a tenth of the
 * remaining reduction, when that is all that is still needed) or max_inner
 * iterations; the outer loop computes r = b - A x, x += ||r|| d and the norms
 * in FP64 on the GPU, until ||b - A x||_2 <= outer_tol * ||b||_2 or max_outer
 * refinements.  Returns MFE_OK when converged, MFE_BREAKDOWN if an inner
 * solve broke down, MFE_UNSUPPORTED if it did not converge in max_outer. */
int mfe_cg_solve_mixed(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* b, mfe_vec* x,
                       int max_outer, int max_inner, double inner_tol, double outer_tol,
                       int* outer_iters, int* inner_iters, double* rel_residual, double* times);
/* y = A x evaluated as the mixed solve's inner SpMV: FP32 values, x rounded
 * to FP32, FP32 products summed in stored column order, y widened to FP64. */
int mfe_matvec_fp32(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* x, mfe_vec* y);
/* mfe_cg_solve_mixed with flags.  MFE_MIXED_KEEP_DIRECTION: the inner FP32 CG
 * is not restarted at a refinement; its residual is replaced by the rounded
 * FP64 residual b - A x, its direction loses its component along the new
 * residual, and it continues (reliable updates, Clark et al. 2010), so the
 * inner iterations total about what FP64 CG needs.  It wants frequent
 * replacements: inner_tol (the reduction per refinement) about 0.1; at 1e-5
 * the FP32 recursion drifts too far from the true residual between two. */
#define MFE_MIXED_KEEP_DIRECTION 0x1u
int mfe_cg_solve_mixed_ex(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* b, mfe_vec* x,
                          int max_outer, int max_inner, double inner_tol, double outer_tol,
                          unsigned flags, int* outer_iters, int* inner_iters,
                          double* rel_residual, double* times);

/* Kernel timing mode, the counterpart of time_kernels (time_kernels.hpp:42-134):
 * launches `reps` back-to-back SpMV kernels y = A x on ctx's stream between two
 * hipEvents and returns the mean kernel time in ms.  variant 0 = matvec_std's
 * kernel (row sums start at 0*y[row]); variant 1 = the kernel inside the fast
 * cg_solve (sums start at +0.0, plus workgroup partials of x.y); variant 2 =
 * the FP32 kernel inside mfe_cg_solve_mixed's inner CG (x is used as its
 * FP32 copy, converted before the timed launches).  Variants 3 and 4 are 1
 * and 2 on the CSR kernels whatever A's plan (for comparison); variant 5 is
 * 1 reading the CG's (clear) done flag first, as it does inside the solve;
 * variant 6 is 1 on plain SELL-64 where A's plan stages x (for comparison);
 * variants 7 and 8 are 1 and 2 on the SELL-64 / staged-x plan where the box
 * layout applies, 9 and 10 are 1 and 2 on the box layout with all 27 slots
 * stored where the symmetric one applies, 11 and 12 are 1 and 2 on the
 * symmetric layout's full-width values where their packed form is read (for
 * comparison), 13 is 1 on the packed boundary stream, where there is one,
 * whatever the number of rows (1 reads it from 2^23 rows on). */
int mfe_time_matvec(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* x, mfe_vec* y, int variant,
                    int reps, double* avg_ms);

/* ---- batched boxes --------------------------------------------------------- */
/* Many independent miniFE box problems (no reference counterpart: the
 * reference solves one box per run).  Problem p is the unit cube meshed with
 * dims[3p..3p+2] = (nx, ny, nz) hex8 elements, unit conductivity, the
 * reference's source and Dirichlet faces.  mfe_batch_solve assembles every
 * problem and solves it with FP64 CG to ||r|| <= rel_tol * ||b||, all problems
 * that are not done in the same launches; each assembled operator is
 * bit-identical to the reference's (generate_matrix_structure +
 * assemble_FE_data + both impose_dirichlet passes, driver.hpp:181-218).  At
 * most two problems per compute unit (else MFE_UNSUPPORTED).
 * The CG reads the stencil values in an exact packed form where they fit one; with
 * MINIFE_BATCH_PACK=0 in the environment when the batch is created it reads them at
 * full width, with the same results (for comparison). */
int mfe_batch_create(mfe_ctx* ctx, int nprob, const int* dims, mfe_batch** out);
void mfe_batch_destroy(mfe_batch* batch);
/* p = -1: {problems, workgroups, total rows, stored SELL entries, total
 * non-zeros, 0}; p >= 0: {rows, non-zeros, elements, workgroups, first
 * workgroup, stored SELL entries} of problem p. */
int mfe_batch_info(const mfe_batch* batch, int p, int64_t info[6]);
/* iters[nprob], rel_residual[nprob] (recursive ||r||/||b||) and the solve's
 * GPU time in seconds (all nullable).  MFE_BREAKDOWN if a problem hit
 * non-positive p.Ap. */
int mfe_batch_solve(mfe_ctx* ctx, mfe_batch* batch, int max_iter, double rel_tol, int* iters,
                    double* rel_residual, double* seconds);
/* seconds[nprob]: each problem's time in the last solve (its first
 * workgroup's wall clock from the first launch to its end); phases[6*nprob]
 * (nullable): the seconds of that workgroup in its own kernels -- elements
 * (element math), rows (row assembly), xp_update (x and p updates), spmv,
 * r_update -- and outside_first_workgroup, the rest: the time in which the
 * problem's other workgroups and the other problems run, and between launches. */
int mfe_batch_timing(const mfe_batch* batch, double* seconds, double* phases);
/* Problem p's assembled operator as CSR (row_offsets[n+1], cols[nnz],
 * vals[nnz]), its right-hand side b[n] and solution x[n]; any may be NULL. */
int mfe_batch_download(mfe_ctx* ctx, const mfe_batch* batch, int p, int* row_offsets, int* cols,
                       double* vals, double* b, double* x);

/* ---- many right-hand sides on one matrix ----------------------------------- */
/* (no reference counterpart: the reference solves one right-hand side.)
 * Block vectors are row-major n x nrhs mfe_vecs of n*nrhs values; nrhs is 4,
 * 8 or 16.  SpMM tiles: `tile` < 0 picks the autotuned tile for A and nrhs
 * (tuned on first use); tile >= 0 forces one (for comparison).  Column k of
 * Y = A X is bit-identical to mfe_matvec's A * X[:, k] for every tile. */
int mfe_spmm(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* X, mfe_vec* Y, int nrhs, int tile);
/* Autotuner: times every candidate tile on A (3 launches each, HIP events),
 * keeps the fastest for A and nrhs; tile, ms[ntiles] and ntiles nullable. */
int mfe_spmm_tune(mfe_ctx* ctx, const mfe_csr* A, int nrhs, int* tile, double* ms, int* ntiles);
/* Pins `tile` as the tuned tile of A for nrhs (mfe_spmm with tile -1 and
 * mfe_cg_solve_multi use it) without timing; fails for an unavailable tile.
 * Kept until A's structure changes or another matrix is tuned on ctx. */
int mfe_spmm_select(mfe_ctx* ctx, const mfe_csr* A, int nrhs, int tile);
/* Shape of a tile: columns per lane, non-zeros per unrolled chunk, rows per
 * workgroup, and kind: 0 = CSR arrays, each lane gathering its X pieces;
 * 1 = staged, the distinct X rows of 16 or 32 consecutive rows copied into
 * LDS first (available when no such row tile has more than 1024 non-zeros and
 * its X rows fit 64 KiB); 2 = SELL, values and columns read from A's SELL-64
 * copy (available unless A's format is CSR-only or a row is longer than 27);
 * 3 = SELL with grid-line slices (same availability as 2): a slice of 64
 * consecutive nodes on grid lines, whose entries 3g, 3g+1, 3g+2 are the
 * columns c-1, c, c+1, loads only the middle X row of each triple and takes
 * the other two from the neighbouring rows' lanes (the same products, added
 * in the same order: the bits of kind 2); 4 = box, A's box layout (27 values
 * per row, no column indices) with the X planes of a 64-node tile streamed
 * through LDS along z (available when A holds a box's generated or verified
 * structure and its format is MFE_SPMV_AUTO).  Every kind gives each column
 * the bits of mfe_matvec.
 * The tuner reports ms = +inf for an unavailable tile, and mfe_spmm rejects
 * it.  Outputs nullable. */
int mfe_spmm_tile_info(int nrhs, int tile, int* cols_per_lane, int* unroll, int* rows_per_block,
                       int* kind);

/* nrhs simultaneous FP64 CG solves A X[:, k] = B[:, k] from the given X,
 * sharing one SpMM per iteration; column k stops once ||r_k|| <= rel_tol *
 * ||B[:, k]|| (cg_solve.hpp's loop test per column) or after max_iter.
 * iters[nrhs], rel_residual[nrhs] (recursive), seconds: nullable. */
int mfe_cg_solve_multi(mfe_ctx* ctx, const mfe_csr* A, const mfe_vec* B, mfe_vec* X, int nrhs,
                       int max_iter, double rel_tol, int* iters, double* rel_residual,
                       double* seconds);

/* ---- verification (host) -------------------------------------------------- */
/* soln(x, y, z, max_p, max_q), analytic_soln.hpp:80-112. */
double mfe_soln(double x, double y, double z, int max_p, int max_q);
/* verify_solution(mesh, x, tol, whole), verify_solution.hpp:55-174: returns 0
 * when the max abs error over the checked nodes is <= tolerance, else 1;
 * *max_err (nullable) receives that error. */
int mfe_verify_solution(mfe_ctx* ctx, const int global_box[6], const mfe_vec* x,
                        double tolerance, int verify_whole_domain, double* max_err);
/* verify_solution for either choice of the u = 1 face: hot_face 1 = x=1 (the
 * reference), 0 = x=0, checked against the mirrored series soln(1-x, y, z). */
int mfe_verify_solution_ex(mfe_ctx* ctx, const int global_box[6], const mfe_vec* x,
                           double tolerance, int verify_whole_domain, int hot_face,
                           double* max_err);

#ifdef __cplusplus
}
#endif
#endif
