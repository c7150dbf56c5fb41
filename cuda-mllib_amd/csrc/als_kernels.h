// als_kernels.h -- internal interface between the host driver and the
// gfx950 kernels of the ALS half-sweep.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cumf {

// One unit of work for a wavefront: `count` ratings of row `row`, starting
// at rating index `start` of the CSR (absolute, so that no row-pointer load
// precedes the first gather; rating indices fit int32 like the CSR's own).  slot < 0: the task covers the
// whole row and solves it; slot >= 0: it writes a partial Gram to
// partial[slot].  row < 0: nothing to do (the tail of a list sized by a bound).
struct Task {
  int32_t row;
  int32_t start;
  int32_t count;
  int32_t slot;
};

// A row whose Gram is the sum of `nchunks` partials starting at `slot`
// (row < 0: none).
struct HeavyRow {
  int32_t row;
  int32_t slot;
  int32_t nchunks;
  int32_t pad;
};

struct SweepArgs {
  const int32_t* row_ptr;  // CSR of the side being solved (m+1)
  const int32_t* col;      // column indices into theta (nnz)
  const float* val;        // ratings (nnz)
  const float* theta;      // factors of the other side, row stride ldf
  float* x;                // factors being solved, row stride ldf
  int64_t ldf;             // factor row stride in floats (multiple of 4, >= f)
  const Task* tasks;
  int64_t ntasks;
  const HeavyRow* heavy;
  int64_t nheavy;
  float* partial;          // partial Grams, partial_floats_per_slot(f) each
  int* fail_counter;       // rows whose factorisation met a non-positive pivot
  int f;
  float lambda;
  // precision != 0: Gram from BF16 shadow factors (theta_b, row stride ldb,
  // zero padded); solutions are also written to x_b in BF16.
  int precision;
  int64_t ldb;
  const uint16_t* theta_b;
  uint16_t* x_b;
  // solver != 0: FP16 conjugate gradients inside FP32 refinement with an
  // FP64 residual, warm-started from x; Cholesky for rows that do not reach
  // ||b - A x|| <= cg_tol ||b|| within cg_rounds rounds of cg_iters steps.
  int solver;
  int cg_iters;
  int cg_rounds;
  float cg_tol;
  int* cg_fallback;        // rows that fell back to Cholesky
  // CG start: 0 the current factor, 1 zero, 2 x0 (row stride ldf), 3 the
  // better of the current factor and x0 by FP64 residual.
  int warm;
  const float* x0;
  float* cg_trace;         // optional, 4 floats per row: initial / final relative residual, rounds, fell back
  // Rows the CG pass hands to the Cholesky fallback kernel: entry = row, or
  // -1 - index into heavy for a split row; fb_count = list length.
  int* fb_list;
  int* fb_count;
  // != 0: FP32 rows in the f x f system whatever their length (a tile table's
  // Cholesky); 0: short ones in the dual form.
  int primal;
  // Longest whole FP32 row that the launch solves in the dual form (0: none);
  // the launchers set it (fp32_dual_limit).
  int dual_limit;
  // persistent > 0: launch that many wavefronts, each taking tasks from
  // *task_counter (zero before the launch) until ntasks are taken.
  // launch_rows_kernel: that many work-groups over the rows 0 .. ntasks of
  // row_ptr; task_counter[0] and [2] zero before the launch.
  int persistent;
  int* task_counter;
  // occupancy > 0 (one-task-per-group launches): at most that many
  // wavefronts per CU, enforced through the LDS each group requests.
  int occupancy;
  // Dual-form launches: 32-rating chunks staged per row, 1 (rows of at
  // most 31 ratings), 2 (at most 63) or 3 (at most 95); dual_partial != 0
  // if a task of the launch is a split row's chunk (its partial Gram is
  // formed: two or three chunks only).
  int dual_chunks;
  int dual_partial;
};

// A range of count >= 1 ratings in chunks of `size`: how many there are, and
// the position of a chunk's i-th rating, to be compared with the count as an
// unsigned number.  Exact up to INT_MAX ratings and for the few chunks past
// the end that a prefetch asks about, whose positions no longer fit an int.
__host__ __device__ constexpr int chunks_of(int count, int size) { return (count - 1) / size + 1; }
__host__ __device__ constexpr uint32_t position_in(int ch, int size, int i) { return (uint32_t)ch * size + i; }

// Rows up to this length are solved whole, whatever the matrix: the finest cut
// that adaptive_split makes by itself, and the longest row that one wavefront
// of launch_rows_kernel solves.  One constant, so that both give the same
// factors up to it; the value is not a measured optimum.
constexpr int kWholeRowMax = 2048;

// Longest row the dual form takes (three staged chunks of 32 ratings).
constexpr int kDualMaxRatingsHost = 95;

// Length classes of the device planner (planner.hip): every length below 256
// by itself, then eighths of an octave up to INT_MAX.
constexpr int kPlanClasses = 256 + 8 * 23;
__host__ __device__ inline int plan_class(int n) {
  if (n < 256) return n;
  const int e = 31 - __builtin_clz((unsigned)n);  // 8 .. 30
  return 256 + 8 * (e - 8) + ((n >> (e - 3)) & 7);
}
// What the host needs of a plan made on the device.
struct PlanSummary {
  int32_t ntasks, nheavy, nslots;
  int32_t bad_row;              // first row whose pointers decrease (INT_MAX: none)
  int32_t first, last;          // row_ptr[0], row_ptr[m]
  int32_t start[kPlanClasses];  // tasks of longer classes: where each class begins in the task list
};
size_t plan_work_bytes();
// Plans m rows into tasks[0 .. task_cap) and heavy[0 .. heavy_cap), entries
// past the plan naming row -1; with bad row pointers (see the summary) every
// entry does.  task_cap >= m + nnz / split and heavy_cap >= nnz / (split + 1);
// `work` holds plan_work_bytes() of device memory, `out` is host memory the
// device can write, valid once the stream has passed.
hipError_t launch_plan(const int32_t* row_ptr, int64_t m, int64_t nnz, int split, Task* tasks, int64_t task_cap,
                       HeavyRow* heavy, int64_t heavy_cap, void* work, PlanSummary* out, hipStream_t s);

// LDS of one CU, and the range of occupancy caps a launch accepts.
constexpr int kLdsBytesPerCU = 160 * 1024;
constexpr int kMinOccupancy = 3, kMaxOccupancy = 16;
// LDS a group requests so that at most n groups fit one CU: more than a
// (n+1)-th of the CU's LDS, in 512-byte steps.
inline size_t occupancy_lds_bytes(int n) { return (size_t)(kLdsBytesPerCU / (n + 1) / 512 + 1) * 512; }

// The reference-reproducing path (compat.hip): one work-group per row.
struct CompatArgs {
  const int32_t* row_ptr;
  const int32_t* col;
  const float* val;
  const float* theta;      // row stride ldf
  float* x;                // row stride ldf
  int64_t ldf;
  const int32_t* rows;     // optional list of rows (NULL: rows 0..nrows-1)
  double* dump;            // optional: write [M | b] (f*(f+1) doubles per row) and stop
  int* fail_counter;       // rows with a zero pivot
  int f;
  float lambda;
};
hipError_t prepare_compat(int f);
hipError_t launch_compat(const CompatArgs& a, int64_t nrows, hipStream_t s);

int sweep_nb(int f);
// First of the two columns (high and low part) that the rating takes in the
// BF16 layout of NB column blocks: f, or the last block's first column where f
// lies before that block (f % 16 above 12): the solves read the right-hand
// side from the last block.
__host__ __device__ constexpr int bf16_rating_col(int f, int NB) { return f > 16 * (NB - 1) ? f : 16 * (NB - 1); }
// Wavefronts per SIMD that the launches without a tile table are built for:
// two while the accumulator tiles leave room for the solver's registers (up
// to 8 column blocks, f <= 124), one beyond (the two-wavefront build spills
// several hundred bytes per lane).
__host__ __device__ constexpr int default_waves(int NB) { return NB >= 9 ? 1 : 2; }
size_t partial_floats_per_slot(int f);
int dump_dim(int f);
// Clears n <= 64 ints (CG fallback-list length, persistent task counters).
hipError_t launch_fallback_reset(int* count, int n, hipStream_t s);
// Half-sweep kernels (als_sweep.hip), one set per register budget:
// w2 = two wavefronts per SIMD, w1 = one.
// Launchers of the sweep kernels, per register budget (w1, w2) and solver
// family (chol: Cholesky task/finish kernels and the CG path's fallback;
// cg: CG task/finish kernels; chol also holds the dual-form task kernel
// for rows of at most 95 ratings, BF16 factors only, and the kernel over
// whole rows without a plan, FP32 only).
#define CUMF_SWEEP_LAUNCHERS                                                \
  namespace chol {                                                          \
  hipError_t launch_task_kernel(const SweepArgs& a, hipStream_t s);         \
  hipError_t launch_finish_kernel(const SweepArgs& a, hipStream_t s);       \
  hipError_t launch_fallback_kernel(const SweepArgs& a, hipStream_t s);     \
  hipError_t launch_dual_kernel(const SweepArgs& a, hipStream_t s);         \
  hipError_t launch_rows_kernel(const SweepArgs& a, hipStream_t s);         \
  }                                                                         \
  namespace cg {                                                            \
  hipError_t launch_task_kernel(const SweepArgs& a, hipStream_t s);         \
  hipError_t launch_finish_kernel(const SweepArgs& a, hipStream_t s);       \
  }
namespace w1 { CUMF_SWEEP_LAUNCHERS }
namespace w2 { CUMF_SWEEP_LAUNCHERS }
#undef CUMF_SWEEP_LAUNCHERS
// Half-sweep for 140 < f <= 256 (FP32 Gram + FP32 Cholesky, one 256-thread
// work-group per row: the whole-row tasks a.tasks[0 .. rows), or rows
// 0 .. rows-1 of row_ptr when a.tasks is null); large_lds_bytes(f) of LDS.
// prepare_large_kernel(f) raises the kernel's dynamic LDS limit to
// large_lds_bytes(f); call it outside any stream capture before launching.
hipError_t launch_large_kernel(const SweepArgs& a, int64_t rows, hipStream_t s);
hipError_t prepare_large_kernel(int f);
size_t large_lds_bytes(int f);
// The dual form for 140 < f <= 256: one wavefront per whole-row task
// a.tasks[0 .. ntasks), each of at most kDualMaxRatingsHost ratings (FP32).
hipError_t launch_large_dual_kernel(const SweepArgs& a, int64_t ntasks, hipStream_t s);
// The dual form on the work-group for 140 < f <= 256: whole-row tasks
// a.tasks[0 .. ntasks) of more than kDualMaxRatingsHost ratings whose
// systems have nbd = (n + 16) / 16 row blocks (7 .. kLargeDualWgMaxBlocks).
// prepare_large_kernel raises the LDS limits of these kernels too.
constexpr int kLargeDualWgMaxBlocks = 16;
hipError_t launch_large_dual_wg_kernel(const SweepArgs& a, int64_t ntasks, int nbd, hipStream_t s);
hipError_t launch_dump_kernel(const SweepArgs& a, const int32_t* rows, int64_t nrows, float* out,
                              hipStream_t s);
hipError_t launch_rmse(const int32_t* u, const int32_t* v, const float* r, int64_t cnt, const float* X,
                       const float* T, int64_t ldf, int f, double* partial, int nblocks, double* out,
                       hipStream_t s);
hipError_t launch_mfma_layout(float* out, hipStream_t s);
hipError_t launch_mfma_bf16_layout(float* out, hipStream_t s);
hipError_t launch_to_bf16(const float* src, int64_t ldf, void* dst, int64_t ldb, int64_t rows, int f,
                          hipStream_t s);
// Device rows of `cols` floats, stride lds -> stride ldd (zero padded), ldd <= 4096.
hipError_t launch_restride(const float* src, int64_t lds, float* dst, int64_t ldd, int64_t rows, int cols,
                           hipStream_t s);
hipError_t launch_copy(const void* src, void* dst, int64_t bytes, hipStream_t s);

}  // namespace cumf
