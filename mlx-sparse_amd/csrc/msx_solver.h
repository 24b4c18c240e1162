// msx_solver.h - device-side building blocks of the Krylov solver loops
// (csr_cg.hip, csr_krylov.hip): workgroup sizes, the reproducible
// partial-sum protocol and the grid-stride loop with loads in flight.
//
// Sums: each workgroup reduces its grid-stride share in double and writes
// one partial per slot; every workgroup of the NEXT pass adds those
// partials in workgroup order, so all workgroups see the same bits and
// take the same scalar decisions, and no workgroup waits on another inside
// a kernel.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>

#include "msx_device.h"
#include "msx_internal.h"

namespace msx {
namespace solver {

constexpr int kSolverThreads = 512;
constexpr int kSolverMaxBlocks = 512;  // two workgroups per CU at most (partials re-read by each)
constexpr int kSlots = 4;              // partial sums per pass
constexpr int kUnroll = 4;             // independent loads in flight per thread

__device__ inline bool fin(float v) { return isfinite(v); }
__device__ inline bool fin(double v) { return isfinite(v); }

// std::max(v, 0) of the reference loops: a NaN stays NaN (fmax would drop it).
__device__ inline double max0(double v) { return v < 0.0 ? 0.0 : v; }
__device__ inline float max0(float v) { return v < 0.0f ? 0.0f : v; }

__device__ inline double wave_sum(double v) {
  // butterfly: every lane ends with the same value (each level adds a
  // commutative pair)
  for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
  return v;
}

// Workgroup sums of v[] -> part[k * kSolverMaxBlocks + blockIdx.x].
__device__ inline void write_partials(double (&v)[kSlots], double *part) {
  __shared__ double sh[kSlots][kSolverThreads / kWave];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  for (int k = 0; k < kSlots; ++k) {
    const double w = wave_sum(v[k]);
    if (lane == 0) sh[k][wave] = w;
  }
  __syncthreads();
  if (threadIdx.x < kSlots) {
    double s = 0.0;
    for (int w = 0; w < kSolverThreads / kWave; ++w) s += sh[threadIdx.x][w];
    part[threadIdx.x * kSolverMaxBlocks + blockIdx.x] = s;
  }
}

// Totals of the previous pass's `nparts` partials, the same bits in every
// workgroup (fixed order, written by an earlier kernel).  In two steps, so
// that a kernel can issue its own element loads between them: loads are
// waited on in issue order, so partials loaded after the elements would wait
// for the elements too.
__device__ inline void load_partials(const double *part, int nparts, double (&v)[kSlots]) {
  // all kSlots loads at once (clamped index, no branch)
  const int idx = static_cast<int>(threadIdx.x) < nparts ? static_cast<int>(threadIdx.x) : 0;
#pragma unroll
  for (int k = 0; k < kSlots; ++k) v[k] = part[k * kSolverMaxBlocks + idx];
}

__device__ inline void reduce_partials(const double (&v)[kSlots], int nparts, double (&t)[kSlots]) {
  // The loops of one workgroup pass a literal 1: load_partials gave every thread
  // the one partial.  Not a test at run time, which cost bi_v and bi_r 0.4 us of 8.
  if (__builtin_constant_p(nparts) && nparts == 1) {
    for (int k = 0; k < kSlots; ++k) t[k] = v[k];
    __syncthreads();  // what follows may write the solver state that was read before
    return;
  }
  __shared__ double sh[kSlots][kSolverThreads / kWave];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const bool mine = static_cast<int>(threadIdx.x) < nparts;
#pragma unroll
  for (int k = 0; k < kSlots; ++k) {
    const double w = wave_sum(mine ? v[k] : 0.0);
    if (lane == 0) sh[k][wave] = w;
  }
  __syncthreads();
  for (int k = 0; k < kSlots; ++k) {
    double s = 0.0;
    for (int w = 0; w < kSolverThreads / kWave; ++w) s += sh[k][w];
    t[k] = s;
  }
  __syncthreads();
}

__device__ inline void read_totals(const double *part, int nparts, double (&t)[kSlots]) {
  double v[kSlots];
  load_partials(part, nparts, v);
  reduce_partials(v, nparts, t);
}

// Grid-stride over [0, n) with kUnroll coalesced elements per round.
// A thread whose kUnroll elements all lie below n runs them without a
// per-element test, so the compiler issues all of their loads before the
// first use (a test per element made it wait for each load in turn); the
// last, partial group tests each element.
#define MSX_SOLVER_LOOP(...)                                                                    \
  {                                                                                          \
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kSolverThreads;                     \
    for (int64_t base = static_cast<int64_t>(blockIdx.x) * kSolverThreads + threadIdx.x; base < n; \
         base += kUnroll * stride) {                                                         \
      if (base + (kUnroll - 1) * stride < n) {                                               \
        _Pragma("unroll") for (int u = 0; u < kUnroll; ++u) {                                \
          const int64_t i = base + u * stride;                                               \
          __VA_ARGS__                                                                        \
        }                                                                                    \
      } else {                                                                               \
        _Pragma("unroll") for (int u = 0; u < kUnroll; ++u) {                                \
          const int64_t i = base + u * stride;                                               \
          if (i < n) { __VA_ARGS__ }                                                         \
        }                                                                                    \
      }                                                                                      \
    }                                                                                        \
  }

// A pass whose arithmetic needs the previous pass's totals issues, in this
// order, that pass's partial loads (load_partials), the loads of its own
// first round of elements (load_round: kUnroll grid-stride elements of each
// of NV vectors; an index past n reads the thread's first element, or
// element 0), then reduces the partials (reduce_partials) and runs
// for_rounds: op(i, e) for every element i of the thread in grid-stride
// order, e holding its NV values - the first round from those registers,
// each later round loaded whole before its first use.  The reduction's
// wave sums and barriers then overlap the element loads.
template <int NV>
struct Round {
  float e[kUnroll][NV];
};

template <int NV>
__device__ inline void load_round(const float *const (&vec)[NV], int64_t base, int64_t n,
                                  Round<NV> &r) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kSolverThreads;
#pragma unroll
  for (int u = 0; u < kUnroll; ++u) {
    const int64_t j = base + u * stride < n ? base + u * stride : (base < n ? base : 0);
#pragma unroll
    for (int k = 0; k < NV; ++k) r.e[u][k] = vec[k][j];
  }
}

__device__ inline int64_t first_base() {
  return static_cast<int64_t>(blockIdx.x) * kSolverThreads + threadIdx.x;
}

template <int NV, class Op>
__device__ inline void for_rounds(const float *const (&vec)[NV], int64_t n, const Round<NV> &first,
                                  Op op) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kSolverThreads;
  const int64_t base0 = first_base();
#pragma unroll
  for (int u = 0; u < kUnroll; ++u)
    if (base0 + u * stride < n) op(base0 + u * stride, first.e[u]);
  for (int64_t base = base0 + kUnroll * stride; base < n; base += kUnroll * stride) {
    Round<NV> r;
    load_round<NV>(vec, base, n, r);
#pragma unroll
    for (int u = 0; u < kUnroll; ++u)
      if (base + u * stride < n) op(base + u * stride, r.e[u]);
  }
}

// Host side: iterations to enqueue before the next read of the solver
// state.  An iteration enqueued past the solve's stop still runs its SpMVs
// in full (only the vector passes return early), while a read costs a round
// trip to the host; so the batch doubles (1, 2, 4, ... kMaxBatch) until two
// reads give a rate of residual decrease, and from then on covers the
// iterations that rate needs to reach the tolerance (at most kMaxBatch).
// The device alone decides where the solve stops, so results do not depend
// on the batches.
class BatchSchedule {
 public:
  static constexpr int64_t kMaxBatch = 32;
  // `completed` iterations done, their residual norm, the solve's tolerance.
  int64_t next(int64_t completed, double residual, double tol) {
    int64_t b = doubling_;
    if (k_ >= 0 && completed > k_ && residual > tol && tol > 0.0 && residual < res_) {
      const double rate = std::log(residual / res_) / static_cast<double>(completed - k_);
      const double need = std::ceil(std::log(tol / residual) / rate);
      b = need >= static_cast<double>(kMaxBatch) ? kMaxBatch : (need < 1.0 ? 1 : static_cast<int64_t>(need));
    }
    doubling_ = doubling_ * 2 < kMaxBatch ? doubling_ * 2 : kMaxBatch;
    k_ = completed;
    res_ = residual;
    return b;
  }

 private:
  int64_t doubling_ = 1;
  int64_t k_ = -1;
  double res_ = 0.0;
};

// ---------------------------------------------------------------------------
// Small systems in one workgroup.  Below some thousands of rows an iteration's
// four to seven kernels take 4 to 5 us each however little they do, and a
// launch's gap between them; one workgroup that runs the product and the
// passes of many iterations in turn pays a barrier in their place, at one
// compute unit's rate.  The passes are the kernels' own, over one block.  The
// matrix stays in registers for the launch (kValues values a thread), its row
// pointers in LDS, so a product is one round of gathers of x.
// Only for row-block plans without rows of more than kGroupRowValues values: a
// row is one thread's sum in stored order, as in the row blocks, which take
// lanes and a tree of sums for blocks that average more than that.
// Whole solves to 1e-5, kernels -> one workgroup, us: CG, Laplacian 30^2 712
// -> 309, 63^2 707 -> 492; MINRES 35^2 955 -> 434, 40^2 982 -> 468 (48 values a
// thread do not fit the registers beside its passes, 63^2 981 -> 951 with them,
// so MINRES and BiCGSTAB stop at 16); BiCGSTAB 40^2 919 -> 456.  A pass takes
// about 2.5 us, the latency of its two reductions.
constexpr int64_t kGroupRows = 4608;
constexpr int64_t kGroupRowValues = 32;
constexpr int64_t kGroupBatch = 128;  // iterations a launch: it ends with the solve
constexpr int kGroupFew = 16, kGroupMany = 48;  // values a thread

template <class I>
struct GroupMatrix {
  const float *data;
  const I *indices;
  const I *indptr;
  int64_t n, nnz;
};

// `values`: the most values a thread that the solver's loop is built for.
inline bool in_one_group(const msx_csr_plan *plan, int64_t n, int64_t nnz, int values) {
  return plan != nullptr && plan->longest <= kGroupRowValues && plan->n_panels == 0 &&
         plan->n_slices == 0 && n <= kGroupRows && nnz <= int64_t{values} * kSolverThreads;
}

// LDS of a launch: the products of all values, then n + 1 row pointers.
inline size_t group_lds(int64_t n, int64_t nnz) {
  return static_cast<size_t>(nnz + n + 1) * sizeof(float);
}
inline hipError_t group_lds_limit(const void *kernel) {
  return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                             static_cast<int>(group_lds(kGroupRows, int64_t{kGroupMany} * kSolverThreads)));
}

template <class I, class System>
GroupMatrix<I> group_matrix(const System &s) {
  return {s.data, static_cast<const I *>(s.indices), static_cast<const I *>(s.indptr), s.n, s.nnz};
}

template <int kValues>
struct GroupValues {
  int32_t col[kValues];  // -1: no value, or a column out of range
  float val[kValues];
};

// The thread's values (positions threadIdx.x + u * kSolverThreads) into
// registers and the row pointers, held to [0, nnz], into LDS.
template <int kValues, class I>
__device__ inline void group_load(const GroupMatrix<I> &a, GroupValues<kValues> &m, float *lds) {
  const int tid = static_cast<int>(threadIdx.x);
  const uint32_t lim = col_limit32(a.n);
#pragma unroll
  for (int u = 0; u < kValues; ++u) {
    const int64_t p = tid + u * kSolverThreads;
    m.col[u] = -1;
    m.val[u] = 0.0f;
    if (p < a.nnz) {
      const I c = a.indices[p];
      m.col[u] = col_ok(c, a.n, lim) ? static_cast<int32_t>(c) : -1;
      m.val[u] = a.data[p];
    }
  }
  int32_t *ip = reinterpret_cast<int32_t *>(lds + a.nnz);
  for (int64_t r = tid; r <= a.n; r += kSolverThreads) {
    const int64_t p = static_cast<int64_t>(a.indptr[r]);
    ip[r] = static_cast<int32_t>(p < 0 ? 0 : (p > a.nnz ? a.nnz : p));
  }
  __syncthreads();
}

// y = A x in one workgroup: all products in LDS, then a row a thread, in
// stored order, rows of one to four values from their first product.
template <int kValues, class I>
__device__ inline void group_spmv(const GroupMatrix<I> &a, const GroupValues<kValues> &m,
                                  const float *x, float *y, float *lds) {
  const int tid = static_cast<int>(threadIdx.x);
  const int nnz = static_cast<int>(a.nnz), n = static_cast<int>(a.n);
  const int32_t *ip = reinterpret_cast<const int32_t *>(lds + nnz);
  float xv[kValues];
#pragma unroll
  for (int u = 0; u < kValues; ++u) xv[u] = x[m.col[u] < 0 ? 0 : m.col[u]];
#pragma unroll
  for (int u = 0; u < kValues; ++u)
    if (tid + u * kSolverThreads < nnz)
      lds[tid + u * kSolverThreads] = m.col[u] < 0 ? 0.0f : m.val[u] * xv[u];
  __syncthreads();
  constexpr int U = 8;
  for (int r = tid; r < n; r += kSolverThreads) {
    int i = ip[r];
    const int end = ip[r + 1];
    float sum = i < end && end - i <= 4 ? lds[i++] : 0.0f;
    for (; i < end; i += U) {
      float t[U];
#pragma unroll
      for (int u = 0; u < U; ++u) t[u] = lds[i + u < end ? i + u : i];
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (i + u < end) sum = sum + t[u];
    }
    y[r] = sum;
  }
  __syncthreads();
}

// Whether the solve still runs, read after the pass before.
template <class State>
__device__ inline bool group_running(const State *st) {
  __syncthreads();
  return *const_cast<const volatile int32_t *>(&st->running) != 0;
}

// Workgroups of a solver pass over n elements (kUnroll per thread and round).
inline uint32_t blocks_for(int64_t n) {
  const int64_t per_block = static_cast<int64_t>(kUnroll) * kSolverThreads;
  const int64_t blocks = (n + per_block - 1) / per_block;
  return static_cast<uint32_t>(blocks < 1 ? 1 : (blocks > kSolverMaxBlocks ? kSolverMaxBlocks : blocks));
}

}  // namespace solver
}  // namespace msx
