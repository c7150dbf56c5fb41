// planner.hip -- the task planner on the device (host counterpart:
// plan_tasks in als_api.cpp, which the resident handle uses, where the row
// pointers are in host memory anyway and the plan outlives the call).
//
// The device entry points get a rating matrix per call, so its plan is part
// of every call.  Read back and sorted on the host, the plan of 480,189 rows
// took 18 ms beside a half-sweep of 16.5 ms; here it is a counting sort in
// device memory, 0.04 ms, and nothing but the summary crosses the bus.
//
// Same tasks as plan_tasks: a row of at most `split` ratings is one task, a
// longer one ceil(n / split) chunks of near-equal size in consecutive
// partial-Gram slots.  The order is by length class, longest first: every
// length below 256 is a class of its own (so the dual forms' ranges, edges 32
// .. 256, are exact), longer ones fall into eighths of an octave.  Within a
// class the order is that of arrival: it moves no result, since every task is
// solved by itself and a split row's chunks are summed in slot order.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <climits>

#include "als_kernels.h"

namespace cumf {
namespace {

// One block plans matrices up to this many rows: one launch and no global
// counters (600 rows, f = 32: 60 us a call with the host planner, 28 us with this).
// Beyond it the count and the placement are spread over the chip.
constexpr int64_t kOneBlockRows = 16384;
constexpr int kBlockRows = 2048;  // rows per block of the counting and placing kernels

struct Cut {
  int chunks, base, rem;  // the first rem chunks have base + 1 ratings, the others base
};
__device__ __forceinline__ Cut cut_row(int n, int split) {
  if (n <= split) return {1, n, 0};
  const int nc = (int)(((int64_t)n + split - 1) / split);
  return {nc, n / nc, n % nc};
}

// Shared state of the planning kernels; in device memory for the many-block
// form.
struct Work {
  int hist[kPlanClasses];
  int cursor[kPlanClasses];
  int slots, heavy;  // next free slot / heavy-row entry
  int bad_row;
  int ntasks;
};

__device__ __forceinline__ void count_row(const int32_t* rp, int64_t u, int split, int* hist, int* bad) {
  const int64_t n = (int64_t)rp[u + 1] - rp[u];
  if (n < 0) atomicMin(bad, (int)u);
  if (n < 0 || n > INT_MAX) return;  // (past INT_MAX: another row decreases, or the ends are wrong)
  const Cut c = cut_row((int)n, split);
  if (c.chunks > c.rem) atomicAdd(&hist[plan_class(c.base)], c.chunks - c.rem);
  if (c.rem > 0) atomicAdd(&hist[plan_class(c.base + 1)], c.rem);
}

// Exclusive scan from the longest class down: cursor[b] = tasks of classes
// above b.  512 threads take part; returns with the block synchronised.
__device__ __forceinline__ void scan_classes(const int* hist, int* cursor, int* tmp) {
  const int t = threadIdx.x;
  static_assert(kPlanClasses <= 512, "one thread per class");
  // tmp[i] = hist of class kPlanClasses - 1 - i
  if (t < 512) tmp[t] = t < kPlanClasses ? hist[kPlanClasses - 1 - t] : 0;
  __syncthreads();
  for (int d = 1; d < 512; d <<= 1) {
    const int v = (t < 512 && t >= d) ? tmp[t - d] : 0;
    __syncthreads();
    if (t < 512) tmp[t] += v;
    __syncthreads();
  }
  if (t < kPlanClasses) cursor[kPlanClasses - 1 - t] = t > 0 ? tmp[t - 1] : 0;
  __syncthreads();
}

// A split row's places.  Its chunks have at most two lengths, so one add each
// reserves them: with an add per chunk, one after the other, the call for one
// row of 30 million ratings in 1,832 chunks took 1.5 ms (f = 8), now 1.3 ms,
// and one of 2 million in 285,715 chunks 205 ms, now 115 ms.
struct SplitRow {
  int row, start, slot, at_long, at_short;
  Cut c;
  __device__ __forceinline__ void reserve(int64_t u, int s, int n, int split, int* cursor, int* slots, int* heavy,
                                          HeavyRow* hv) {
    row = (int)u;
    start = s;
    c = cut_row(n, split);
    slot = atomicAdd(slots, c.chunks);
    hv[atomicAdd(heavy, 1)] = HeavyRow{row, slot, c.chunks, 0};
    at_long = c.rem > 0 ? atomicAdd(&cursor[plan_class(c.base + 1)], c.rem) : 0;
    at_short = atomicAdd(&cursor[plan_class(c.base)], c.chunks - c.rem);
  }
  __device__ __forceinline__ void place(int k, Task* tasks) const {
    const bool lng = k < c.rem;
    tasks[lng ? at_long + k : at_short + (k - c.rem)] =
        Task{row, start + k * c.base + (lng ? k : c.rem), c.base + (lng ? 1 : 0), slot + k};
  }
};
// Up to this many chunks a lane places its row by itself, beside the rows of
// the other lanes; longer ones are placed by a wavefront together.
constexpr int kLaneChunks = 64;

// Places the rows of more than kLaneChunks chunks among 64 rows from u0 on, one
// after the other, by the wavefront together.
__device__ __forceinline__ void place_long_rows(const int32_t* rp, int64_t u0, int64_t m, int split, int* cursor,
                                                int* slots, int* heavy, Task* tasks, HeavyRow* hv) {
  const int lane = threadIdx.x & 63;
  const int64_t u = u0 + lane;
  const int start = u < m ? rp[u] : 0, n = u < m ? rp[u + 1] - start : 0;
  SplitRow r{};
  const bool lng = n > split && cut_row(n, split).chunks > kLaneChunks;
  if (lng) r.reserve(u, start, n, split, cursor, slots, heavy, hv);
  for (uint64_t todo = __ballot(lng); todo; todo &= todo - 1) {
    const int l = __builtin_ctzll(todo);
    const SplitRow w{__shfl(r.row, l), __shfl(r.start, l), __shfl(r.slot, l), __shfl(r.at_long, l),
                     __shfl(r.at_short, l), {__shfl(r.c.chunks, l), __shfl(r.c.base, l), __shfl(r.c.rem, l)}};
    for (int k = lane; k < w.c.chunks; k += 64) w.place(k, tasks);
  }
}

// A row of at most kLaneChunks chunks, by a lane (false: a longer one, left to
// place_long_rows).
__device__ __forceinline__ bool place_row(const int32_t* rp, int64_t u, int split, int* cursor, int* slots, int* heavy,
                                          Task* tasks, HeavyRow* hv) {
  const int start = rp[u], n = rp[u + 1] - start;
  if (n <= split) {
    tasks[atomicAdd(&cursor[plan_class(n)], 1)] = Task{(int32_t)u, start, n, -1};
    return true;
  }
  if (cut_row(n, split).chunks > kLaneChunks) return false;
  SplitRow r;
  r.reserve(u, start, n, split, cursor, slots, heavy, hv);
  for (int k = 0; k < r.c.chunks; ++k) r.place(k, tasks);
  return true;
}

// The matrix as one block sees it, and the summary for the host.
__device__ __forceinline__ void write_summary(PlanSummary* out, const int* cursor, int ntasks, int bad, int first,
                                              int last) {
  for (int b = threadIdx.x; b < kPlanClasses; b += blockDim.x) out->start[b] = cursor[b];
  if (threadIdx.x == 0) {
    out->ntasks = ntasks;
    out->bad_row = bad;
    out->first = first;
    out->last = last;
  }
}

__global__ __launch_bounds__(1024) void plan_one_block_kernel(const int32_t* __restrict__ rp, int64_t m, int64_t nnz,
                                                              int split, Task* tasks, int64_t task_cap, HeavyRow* hv,
                                                              int64_t heavy_cap, PlanSummary* out) {
  __shared__ int hist[kPlanClasses], cursor[kPlanClasses], tmp[512];
  __shared__ int slots, heavy, bad, any_long;
  for (int b = threadIdx.x; b < kPlanClasses; b += 1024) hist[b] = 0;
  if (threadIdx.x == 0) {
    slots = heavy = any_long = 0;
    bad = INT_MAX;
  }
  __syncthreads();
  for (int64_t u = threadIdx.x; u < m; u += 1024) count_row(rp, u, split, hist, &bad);
  __syncthreads();
  scan_classes(hist, cursor, tmp);
  const int ntasks = tmp[511];
  const int first = rp[0], last = rp[m];
  write_summary(out, cursor, ntasks, bad, first, last);
  __syncthreads();  // the summary holds the starts; placing moves the cursors
  const bool ok = bad == INT_MAX && first == 0 && (int64_t)last == nnz;
  if (ok)
    for (int64_t u = threadIdx.x; u < m; u += 1024)
      if (!place_row(rp, u, split, cursor, &slots, &heavy, tasks, hv)) any_long = 1;
  __syncthreads();
  if (any_long) {
    for (int64_t u0 = threadIdx.x & ~63; u0 < m; u0 += 1024)
      place_long_rows(rp, u0, m, split, cursor, &slots, &heavy, tasks, hv);
    __syncthreads();
  }
  // Entries past the plan (all of them, if the row pointers are bad) name no row.
  for (int64_t i = (ok ? ntasks : 0) + (int)threadIdx.x; i < task_cap; i += 1024) tasks[i] = Task{-1, 0, 0, -1};
  for (int64_t i = (ok ? heavy : 0) + (int)threadIdx.x; i < heavy_cap; i += 1024) hv[i] = HeavyRow{-1, 0, 0, 0};
  if (threadIdx.x == 0) {
    out->nheavy = heavy;
    out->nslots = slots;
  }
}

__global__ __launch_bounds__(512) void plan_clear_kernel(Work* w) {
  const int t = threadIdx.x;
  if (t < kPlanClasses) w->hist[t] = 0;
  if (t == 0) {
    w->slots = w->heavy = 0;
    w->bad_row = INT_MAX;
  }
}

__global__ __launch_bounds__(256) void plan_count_kernel(const int32_t* __restrict__ rp, int64_t m, int split, Work* w) {
  __shared__ int hist[kPlanClasses];
  __shared__ int bad, nslots, nheavy;
  for (int b = threadIdx.x; b < kPlanClasses; b += 256) hist[b] = 0;
  if (threadIdx.x == 0) {
    bad = INT_MAX;
    nslots = nheavy = 0;
  }
  __syncthreads();
  const int64_t u0 = (int64_t)blockIdx.x * kBlockRows, u1 = u0 + kBlockRows < m ? u0 + kBlockRows : m;
  for (int64_t u = u0 + threadIdx.x; u < u1; u += 256) {
    count_row(rp, u, split, hist, &bad);
    const int64_t n = (int64_t)rp[u + 1] - rp[u];
    if (n > split && n <= INT_MAX) {
      atomicAdd(&nslots, cut_row((int)n, split).chunks);
      atomicAdd(&nheavy, 1);
    }
  }
  __syncthreads();
  for (int b = threadIdx.x; b < kPlanClasses; b += 256)
    if (hist[b]) atomicAdd(&w->hist[b], hist[b]);
  if (threadIdx.x == 0) {
    if (bad != INT_MAX) atomicMin(&w->bad_row, bad);
    if (nheavy) {
      atomicAdd(&w->slots, nslots);
      atomicAdd(&w->heavy, nheavy);
    }
  }
}

__global__ __launch_bounds__(512) void plan_scan_kernel(const int32_t* __restrict__ rp, int64_t m, int64_t nnz, Work* w,
                                                        PlanSummary* out) {
  __shared__ int cursor[kPlanClasses], tmp[512];
  scan_classes(w->hist, cursor, tmp);
  if (threadIdx.x < kPlanClasses) w->cursor[threadIdx.x] = cursor[threadIdx.x];
  const int first = rp[0], last = rp[m];
  write_summary(out, cursor, tmp[511], w->bad_row, first, last);
  if (threadIdx.x == 0) {
    out->nheavy = w->heavy;
    out->nslots = w->slots;
    const bool ok = w->bad_row == INT_MAX && first == 0 && (int64_t)last == nnz;
    w->ntasks = ok ? tmp[511] : 0;
    if (!ok) w->bad_row = 0;  // (the placing kernel's refusal, whatever the fault)
    w->slots = w->heavy = 0;  // now the next free slot and entry
  }
}

// Reserves the block's places in each class with one global add per class,
// then places its rows.  A chunk of a split row takes its place directly.
__global__ __launch_bounds__(256) void plan_place_kernel(const int32_t* __restrict__ rp, int64_t m, int split, Work* w,
                                                         Task* tasks, int64_t task_cap) {
  __shared__ int hist[kPlanClasses];
  const bool ok = w->bad_row == INT_MAX;
  for (int64_t i = w->ntasks + (int64_t)blockIdx.x * 256 + threadIdx.x; i < task_cap; i += (int64_t)gridDim.x * 256)
    tasks[i] = Task{-1, 0, 0, -1};
  if (!ok) return;
  const int64_t u0 = (int64_t)blockIdx.x * kBlockRows, u1 = u0 + kBlockRows < m ? u0 + kBlockRows : m;
  for (int b = threadIdx.x; b < kPlanClasses; b += 256) hist[b] = 0;
  __syncthreads();
  for (int64_t u = u0 + threadIdx.x; u < u1; u += 256) {
    const int n = rp[u + 1] - rp[u];
    if (n <= split) atomicAdd(&hist[plan_class(n)], 1);
  }
  __syncthreads();
  for (int b = threadIdx.x; b < kPlanClasses; b += 256)
    if (hist[b]) hist[b] = atomicAdd(&w->cursor[b], hist[b]);
  __syncthreads();
  for (int64_t u = u0 + threadIdx.x; u < u1; u += 256) {
    const int start = rp[u], n = rp[u + 1] - start;
    if (n <= split) tasks[atomicAdd(&hist[plan_class(n)], 1)] = Task{(int32_t)u, start, n, -1};
  }
}

// The split rows (few: a launch of its own keeps their global atomics out of
// the placing kernel's loop).
__global__ __launch_bounds__(256) void plan_place_heavy_kernel(const int32_t* __restrict__ rp, int64_t m, int split,
                                                               Work* w, Task* tasks, HeavyRow* hv) {
  if (w->bad_row != INT_MAX) return;
  for (int64_t u0 = (int64_t)blockIdx.x * 256 + (threadIdx.x & ~63); u0 < m; u0 += (int64_t)gridDim.x * 256) {
    const int64_t u = u0 + (threadIdx.x & 63);
    const bool heavy = u < m && rp[u + 1] - rp[u] > split;
    if (__ballot(heavy && !place_row(rp, u, split, w->cursor, &w->slots, &w->heavy, tasks, hv)))
      place_long_rows(rp, u0, m, split, w->cursor, &w->slots, &w->heavy, tasks, hv);
  }
}

__global__ __launch_bounds__(256) void plan_pad_heavy_kernel(const Work* w, HeavyRow* hv, int64_t heavy_cap) {
  for (int64_t i = w->heavy + (int64_t)blockIdx.x * 256 + threadIdx.x; i < heavy_cap; i += (int64_t)gridDim.x * 256)
    hv[i] = HeavyRow{-1, 0, 0, 0};
}

}  // namespace

size_t plan_work_bytes() { return sizeof(Work); }

hipError_t launch_plan(const int32_t* row_ptr, int64_t m, int64_t nnz, int split, Task* tasks, int64_t task_cap,
                       HeavyRow* heavy, int64_t heavy_cap, void* work, PlanSummary* out, hipStream_t s) {
  if (m < 1 || split < 1 || task_cap < m) return hipErrorInvalidValue;
  if (m <= kOneBlockRows) {
    hipLaunchKernelGGL(plan_one_block_kernel, dim3(1), dim3(1024), 0, s, row_ptr, m, nnz, split, tasks, task_cap, heavy,
                       heavy_cap, out);
    return hipGetLastError();
  }
  Work* w = static_cast<Work*>(work);
  const dim3 grid((unsigned)((m + kBlockRows - 1) / kBlockRows));
  hipLaunchKernelGGL(plan_clear_kernel, dim3(1), dim3(512), 0, s, w);
  hipLaunchKernelGGL(plan_count_kernel, grid, dim3(256), 0, s, row_ptr, m, split, w);
  hipLaunchKernelGGL(plan_scan_kernel, dim3(1), dim3(512), 0, s, row_ptr, m, nnz, w, out);
  hipLaunchKernelGGL(plan_place_kernel, grid, dim3(256), 0, s, row_ptr, m, split, w, tasks, task_cap);
  if (heavy_cap > 0) {
    hipLaunchKernelGGL(plan_place_heavy_kernel, dim3(256), dim3(256), 0, s, row_ptr, m, split, w, tasks, heavy);
    const dim3 pad((unsigned)(heavy_cap < 256 * 256 ? (heavy_cap + 255) / 256 : 256));
    hipLaunchKernelGGL(plan_pad_heavy_kernel, pad, dim3(256), 0, s, w, heavy, heavy_cap);
  }
  return hipGetLastError();
}

}  // namespace cumf
