// Block ILU numeric factorisation and the L/U triangular sweeps on a 6x6 BSR
// pattern (replaces cusparseXbsrilu02 and cusparseXbsrsv2,
// examples/iterative/gmres.cu:374-465 and :609-625).
//
// Semantics: in-place incomplete LU on the given block pattern, equal to
// scalar ILU on the block-expanded pattern: strictly-lower blocks hold L_ik,
// the diagonal block holds unit-lower L_ii below and U_ii on/above its
// diagonal, upper blocks hold U_ij.  The L sweep has a unit diagonal, the U
// sweep a non-unit one.
//
// Schedules
//   factorisation: rows ordered by dependency level on the host (the levels
//     of the factorisation equal those of the L sweep).  Default (dataflow):
//     a few launches, each over a run of levels, in which a workgroup takes
//     the next row in level order from a counter and waits, pivot by pivot,
//     only for the pivot rows it is about to use (a per-row completion flag,
//     released after the row is written); no level waits for the whole
//     previous level.  GPUFEM_ILU_SCHEDULE=level runs one launch per level
//     instead.  The arithmetic of a row is the same either way, so the two
//     schedules give bitwise-identical factors.
//   sweeps: over groups of up to eight rows of a chain (trsv_group_kernel,
//     below) or, for patterns without such chains, over rows; small systems
//     in one workgroup (trsv_small_kernel).  Otherwise one
//     persistent launch per sweep, synchronised through the data:
//     the output vector is pre-filled with a signalling-NaN sentinel, each
//     entry is written once with a relaxed agent-scope atomic store, and a
//     row polls the entries it needs with relaxed agent-scope atomic loads
//     until none holds the sentinel.  No fence and no flag array: each entry
//     validates itself, so a dependency hop costs one store and one load
//     round trip, without L2 write-back or invalidation.  Rows are handed out
//     in level order, in chunks, from a 64-bit counter, so every row waited
//     on is already held by a running wavefront and the sweep cannot
//     deadlock.  The level-by-level sweep stays available (GPUFEM_TRSV=level)
//     as an independent schedule for parity checks.
#include <algorithm>
#include <future>
#include <mutex>
#include <cstdlib>
#include <string>
#include <vector>

#include "common.h"
#include "krylov.h"
#include "symbolic.h"

struct gf_ilu_s {
  gf_context ctx = nullptr;
  int n = 0, nnzb = 0;
  int *rowp = nullptr, *cols = nullptr, *diag = nullptr;
  int *lrows = nullptr, *urows = nullptr;  // rows ordered by level
  std::vector<int> lptr, uptr;             // level offsets (host)
  int* pivot = nullptr;                    // first zero-pivot row (device)
  int max_row_len = 0;
  std::vector<int> lmaxlen;                // longest row of each L level
  // sync-free sweep state
  int *lchunk = nullptr, *uchunk = nullptr; // chunk offsets (see below)
  int4 *lmeta = nullptr, *umeta = nullptr;  // {row, k0, k1, level} per
                                            // position in hand-out order
  int nlchunk = 0, nuchunk = 0;
  bool lchains = false, uchains = false;  // chunks are chains in row order
  unsigned long long* counter = nullptr;   // chunk dispenser (monotonic)
  int* err = nullptr;  // set when a bounded wait expires: [0] sweeps,
                      // [1] factorisation
  unsigned long long base = 0;   // value of counter 0 (factorisation, groups)
  unsigned long long wbase = 0;  // of the counters after it (other sweeps)
  int grid = 0;                            // workgroups per sweep launch
  bool level_sweeps = false;
  // dataflow factorisation: done[i] == epoch once row i is final
  int* done = nullptr;
  int epoch = 0;
  // sweeps over row groups (trsv_group_kernel; none: nlgroup == 0)
  int *lgroup = nullptr, *ugroup = nullptr;  // group records
  int *lgrows = nullptr, *ugrows = nullptr;  // and their rows
  int nlgroup = 0, nugroup = 0, ggrid = 0;
  // small system: both sweeps by one workgroup (trsv_small_kernel) over the
  // level-ordered rows of lmeta and umeta
  bool small = false;
  // dependency level of every group, or of every chunk where there are no
  // groups (host; batched sweeps merge the items of several systems level by
  // level)
  std::vector<int> llevel, ulevel;
};

namespace gf {
namespace {

// Longest row (blocks) the factorisation takes: the column indices and two
// pivots' position lists of a row live in LDS (3 ints per block of the
// longest row, 96 KB at this limit).
constexpr int kMaxRowBlocks = 8192;

// Dataflow schedule of the factorisation (kFlow kernels).  Every workgroup
// takes exactly one ticket from the counter; ticket t factors
// level_rows[t].  Tickets follow level order, so the pivot rows a row waits
// for were handed out before it to workgroups that are already running, and
// the lowest unfinished ticket never waits: the schedule cannot deadlock.
struct Flow {
  unsigned long long* counter = nullptr;
  unsigned long long base = 0;  // counter value at the launch
  int* done = nullptr;          // done[row] == epoch: row is final
  int epoch = 0;
  int* err = nullptr;           // set when a bounded wait expires
};
constexpr unsigned kFlowSpinLimit = 1u << 23;  // polls per wait (seconds)

// The bits of T, for relaxed agent-scope atomic accesses: such a load reads
// past the caches of this XCD, such a store writes through them.
template <typename T> struct BitsOf;
template <> struct BitsOf<double> { using type = unsigned long long; };
template <> struct BitsOf<float> { using type = unsigned int; };
template <typename T>
__device__ __forceinline__ T load_agent(const T* p) {
  using B = typename BitsOf<T>::type;
  return __builtin_bit_cast(
      T, __hip_atomic_load(reinterpret_cast<const B*>(p), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT));
}
template <typename T>
__device__ __forceinline__ void store_agent(T* p, T v) {
  using B = typename BitsOf<T>::type;
  __hip_atomic_store(reinterpret_cast<B*>(p), __builtin_bit_cast(B, v),
                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// lane l's value, to every lane (v_readlane: a few cycles, where a
// ds_bpermute shuffle takes an LDS round trip)
__device__ __forceinline__ double read_lane(double v, int l) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)u, l);
  const unsigned hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), l);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ float read_lane(float v, int l) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_readlane(__builtin_bit_cast(unsigned, v), l));
}

// The row this workgroup factors (dataflow) or blockIdx.x's row (levels).
template <bool kFlow>
__device__ __forceinline__ int flow_row(const int* level_rows, int nrows,
                                        const Flow& f, int* s_row) {
  if (!kFlow) return blockIdx.x < nrows ? level_rows[blockIdx.x] : -1;
  if (threadIdx.x == 0) {
    const long long t = (long long)(atomicAdd(f.counter, 1ull) - f.base);
    const bool ok = t >= 0 && t < nrows;
    *s_row = ok ? level_rows[t] : -1;
    // each workgroup takes one ticket of [0, nrows): anything else means
    // the counter was not where the host expected it
    if (!ok)
      __hip_atomic_store(f.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  return *s_row;
}

// Wait until the pivot rows piv[0..target] are final.  s_rdy[par] holds the
// length of the prefix of piv known to be final; wavefront 0 extends it
// 64 flags per load (one ballot), sleeping between polls while the next
// pivot row is not done, and publishes the new prefix in the other slot,
// s_rdy[par ^ 1]: every thread reads s_rdy[par] to decide whether to wait,
// so it must not change until all have passed the barrier.
// Uniform: every thread of the workgroup calls it with the same target.
// kFence: the wait ends with an agent-scope acquire (it invalidates this
// XCD's L2); without it the caller reads the pivot rows under the rules
// below.
//
// Pivot rows without cache maintenance.  The rows are exchanged between the
// XCDs, whose L2 caches are not coherent with each other.  An agent-scope
// release and acquire pair per row writes back and invalidates the L2, so
// nothing stays cached: the pattern and the U rows, which hundreds of rows
// re-read, come from memory each time.  Instead
//   - a row's final D and U values are written with agent-scope stores
//     (through the L2), and its flag is set once every wavefront has waited
//     for its stores (flow_publish);
//   - a row is read only once its flag is set, so no L2 or L1 can hold an
//     older copy of a line inside the row, except the owner's own XCD, whose
//     caches its stores have passed through;
//   - a line at either end of a row is shared with the next row and may have
//     been cached earlier, by a reader or the owner of that neighbour: the
//     blocks that touch the first or last kEdgeBytes of a row are read with
//     agent-scope loads (edge_block).
// Cached lines of final rows stay valid, so the L2 serves the re-reads.
constexpr int kEdgeBytes = 256;  // two 128-byte lines
// blocks of a row, from either end, that touch its first or last kEdgeBytes
template <typename T>
constexpr int kEdgeBlocks = (kEdgeBytes + 36 * (int)sizeof(T) - 1) /
                            (36 * (int)sizeof(T));
// block t of the nu blocks of a U part lies at an end of its row (the
// diagonal block comes before block 0)
template <typename T>
__device__ __forceinline__ bool edge_block(int t, int nu) {
  return t >= nu - kEdgeBlocks<T> || t < kEdgeBlocks<T> - 1;
}
template <typename T, bool kFlow>
__device__ __forceinline__ T load_pivot(const T* p, bool edge) {
  return kFlow && edge ? load_agent(p) : *p;
}
// a row's final value: written through for the rows that wait for it
template <typename T, bool kFlow>
__device__ __forceinline__ void store_final(T* p, T v) {
  if (kFlow)
    store_agent(p, v);
  else
    *p = v;
}
template <bool kFence>
__device__ __forceinline__ void flow_wait(const int* piv, int npiv,
                                          int target, int* s_rdy, int& par,
                                          const Flow& f) {
  if (s_rdy[par] > target) return;
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    int rdy = s_rdy[par];
    unsigned spins = 0;
    int nap = 1;
    while (rdy <= target) {
      const int t = rdy + lane;
      const bool pend =
          t < npiv && __hip_atomic_load(f.done + piv[t], __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT) != f.epoch;
      const unsigned long long m = __ballot(pend);
      if (m == 0) {
        rdy = min(rdy + 64, npiv);
        continue;
      }
      rdy += __ffsll((long long)m) - 1;
      if (rdy > target) break;
      ++spins;
      const bool failed =
          spins > kFlowSpinLimit ||
          (spins % 256 == 0 && __hip_atomic_load(f.err, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT));
      if (failed) {
        // give up: the factors are reported invalid, the grid drains
        if (lane == 0)
          __hip_atomic_store(f.err, 1, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
        rdy = npiv;
        break;
      }
      for (int z = 0; z < nap; z++) __builtin_amdgcn_s_sleep(1);
      nap = nap * 2 > 8 ? 8 : nap * 2;
    }
    if (kFence)
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    else
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    if (lane == 0) s_rdy[par ^ 1] = rdy;
  }
  __syncthreads();
  par ^= 1;
}

// Publish row i as final, once every wavefront's stores of the row have
// completed: released at agent scope (kFence), or written through by
// store_final and waited for.
template <bool kFence>
__device__ __forceinline__ void flow_publish(int i, const Flow& f) {
  if (kFence)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
  else
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    if (kFence)
      __hip_atomic_store(f.done + i, f.epoch, __ATOMIC_RELEASE,
                         __HIP_MEMORY_SCOPE_AGENT);
    else
      __hip_atomic_store(f.done + i, f.epoch, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  }
}

// LU of a 6 x 6 diagonal block without pivoting by wavefront 0 (all 64 lanes
// call it): lane r < 6 holds row r in d.  Each step's multipliers are formed
// by the lanes at once, so five divisions are on the chain instead of
// fifteen.
template <typename T>
__device__ __forceinline__ void factor_diag(T (&d)[6], int lane, int i,
                                            int* pivot) {
  bool live = true;  // (uniform) no zero pivot so far
#pragma unroll
  for (int c = 0; c < 6; c++) {
    if (!live) continue;
    T u[6];
#pragma unroll
    for (int m = c; m < 6; m++) u[m] = read_lane(d[m], c);
    if (u[c] == T(0)) {
      if (lane == 0) atomicMin(pivot, i);
      live = false;
      continue;
    }
    if (c == 5) continue;  // no row below
    const T l = d[c] / u[c];
    if (lane > c) {
      d[c] = l;
#pragma unroll
      for (int m = c + 1; m < 6; m++) d[m] = d[m] - l * u[m];
    }
  }
}

// One 256-thread workgroup per row of the current level.  The row's column
// indices are staged in LDS (positions of U(k) in row i are found by binary
// search there), L_ik is kept in LDS for the update, and the next k's
// pattern bounds are loaded while the current update runs.
// 512 threads with two register pairs each measured fastest on the 400x400
// plate, AMD + ILU(16): 293 ms a factorisation (256 x 4: 311, 256 x 2: 306,
// 128 x 4: 350, 128 x 2: 366).  Forming the next pivot's L_ik while the
// current update runs (one more barrier a pivot) measured slower (312 ms).
#ifndef GPUFEM_ILU_THREADS
#define GPUFEM_ILU_THREADS 512
#endif
constexpr int kIluThreads = GPUFEM_ILU_THREADS;
template <typename T, bool kFlow>
__global__ void __launch_bounds__(kIluThreads)
    ilu_row_kernel(const int* __restrict__ level_rows, int nrows,
                   const int* __restrict__ rowp, const int* __restrict__ cols,
                   const int* __restrict__ diag, T* vals, int* pivot,
                   Flow f, int maxlen) {
  // dynamic LDS: column indices of row i, and the positions in row i of
  // the current and next pivot's U-part columns (maxlen = longest row)
  extern __shared__ int ilu_gdyn[];
  int* scol = ilu_gdyn;
  int* const pos[2] = {ilu_gdyn + maxlen, ilu_gdyn + 2 * maxlen};
  __shared__ int ub[2][2];               // U-part bounds [u0, u1) per buffer
  __shared__ T udg[2][36];               // U_kk per buffer
  __shared__ T udi[2][6];                // 1 / diagonal of U_kk per buffer
  __shared__ T lik[36];
  __shared__ int s_row, s_rdy[2];
  const int i = flow_row<kFlow>(level_rows, nrows, f, &s_row);
  if (i < 0) return;
  const int tid = threadIdx.x;
  const int r0 = rowp[i], r1 = rowp[i + 1], di = diag[i];
  for (int t = tid; t < r1 - r0; t += blockDim.x) scol[t] = cols[r0 + t];
  if (tid == 0) s_rdy[0] = 0;
  int par = 0;
  __syncthreads();
  // dataflow: pivot row scol[kl] is waited for before it is staged (kl) or
  // used (L_ik reads U_kk staged from it; the update reads U_kj)
  auto wait_for = [&](int kl) {
    if (kFlow) flow_wait<true>(scol, di - r0, kl, s_rdy, par, f);
  };
  // everything about pivot row k (its U part, U_kk, the positions of its
  // columns in row i) is final before this row starts, so it is staged for
  // the next k while the current k's update runs
  auto stage = [&](int kk, int buf) {
    const int k = scol[kk - r0];
    const int u0 = diag[k] + 1, u1 = rowp[k + 1];
    if (tid == 0) {
      ub[buf][0] = u0;
      ub[buf][1] = u1;
    }
    if (tid < 36) {
      const T u = vals[36 * (size_t)diag[k] + tid];
      udg[buf][tid] = u;
      if (tid % 7 == 0) udi[buf][tid / 7] = T(1) / u;
    }
    for (int t = tid; t < u1 - u0; t += blockDim.x) {
      const int j = cols[u0 + t];
      int lo = kk + 1 - r0, hi = r1 - r0;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (scol[mid] < j)
          lo = mid + 1;
        else
          hi = mid;
      }
      pos[buf][t] = (lo < r1 - r0 && scol[lo] == j) ? r0 + lo : -1;
    }
  };
  if (r0 < di) {
    wait_for(0);
    stage(r0, 0);
  }
  __syncthreads();
  for (int kk = r0; kk < di; kk++) {
    const int cur = (kk - r0) & 1;
    if (kk + 1 < di) wait_for(kk + 1 - r0);
    T* Aik = vals + 36 * (size_t)kk;
    const T* Ukk = udg[cur];
    const T* Ui = udi[cur];
    // L_ik = A_ik U_kk^-1 (row r by forward substitution over columns) on
    // lanes 0-5, the next k staged by the other lanes meanwhile
    if (tid < 6) {
      const int r = tid;
      T x[6];
#pragma unroll
      for (int c = 0; c < 6; c++) {
        T v = Aik[6 * r + c];
#pragma unroll
        for (int m = 0; m < c; m++) v -= x[m] * Ukk[6 * m + c];
        x[c] = v * Ui[c];
      }
#pragma unroll
      for (int c = 0; c < 6; c++) {
        Aik[6 * r + c] = x[c];
        lik[6 * r + c] = x[c];
      }
    } else if (kk + 1 < di) {
      // lanes 6.. stage the next pivot row (tid - 6 as the local index)
      const int k = scol[kk + 1 - r0];
      const int u0 = diag[k] + 1, u1 = rowp[k + 1];
      const int tl = tid - 6, nth = blockDim.x - 6;
      if (tl == 0) {
        ub[cur ^ 1][0] = u0;
        ub[cur ^ 1][1] = u1;
      }
      if (tl < 36) {
        const T u = vals[36 * (size_t)diag[k] + tl];
        udg[cur ^ 1][tl] = u;
        if (tl % 7 == 0) udi[cur ^ 1][tl / 7] = T(1) / u;
      }
      for (int t = tl; t < u1 - u0; t += nth) {
        const int j = cols[u0 + t];
        int lo = kk + 2 - r0, hi = r1 - r0;
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (scol[mid] < j)
            lo = mid + 1;
          else
            hi = mid;
        }
        pos[cur ^ 1][t] = (lo < r1 - r0 && scol[lo] == j) ? r0 + lo : -1;
      }
    }
    __syncthreads();
    // A_ij -= L_ik U_kj, kBatch entries per thread at a time: every load of
    // a batch is issued before its stores (the U_kj blocks and the targets
    // are in the same array, so the compiler would otherwise serialise each
    // entry's loads behind the previous entry's store)
    const int u0 = ub[cur][0], nu = ub[cur][1] - u0;
    constexpr int kBatch = 4;
    for (int w0 = 0; w0 < 36 * nu; w0 += kBatch * (int)blockDim.x) {
      T uk[kBatch][6], av[kBatch];
      long long dst[kBatch];
      int ee[kBatch];
#pragma unroll
      for (int bq = 0; bq < kBatch; bq++) {
        const int w = w0 + bq * blockDim.x + tid;
        const int t = w / 36, e = w % 36, c = e % 6;
        const int p = w < 36 * nu ? pos[cur][t] : -1;
        dst[bq] = p < 0 ? -1 : 36LL * p + e;
        ee[bq] = e;
        const T* Ukj = vals + 36 * (size_t)(u0 + (p < 0 ? 0 : t));
#pragma unroll
        for (int m = 0; m < 6; m++) uk[bq][m] = p < 0 ? T(0) : Ukj[6 * m + c];
        av[bq] = p < 0 ? T(0) : vals[(size_t)dst[bq]];
      }
#pragma unroll
      for (int bq = 0; bq < kBatch; bq++) {
        if (dst[bq] < 0) continue;
        const int r = ee[bq] / 6;
        T v = 0;
#pragma unroll
        for (int m = 0; m < 6; m++) v += lik[6 * r + m] * uk[bq][m];
        vals[(size_t)dst[bq]] = av[bq] - v;
      }
    }
    __syncthreads();
  }
  // factor the diagonal block (no pivoting)
  T* D = vals + 36 * (size_t)di;
  if (tid == 0) {
    for (int c = 0; c < 6; c++) {
      const T piv = D[6 * c + c];
      if (piv == T(0)) {
        atomicMin(pivot, i);
        break;
      }
      for (int r = c + 1; r < 6; r++) {
        const T l = D[6 * r + c] / piv;
        D[6 * r + c] = l;
        for (int m = c + 1; m < 6; m++) D[6 * r + m] -= l * D[6 * c + m];
      }
    }
  }
  __syncthreads();
  // U_ij = L_ii^-1 A_ij for the blocks right of the diagonal
  const int nr = r1 - (di + 1);
  for (int w = tid; w < 6 * nr; w += blockDim.x) {
    const int t = w / 6, c = w % 6;
    T* A = vals + 36 * (size_t)(di + 1 + t);
    T x[6];
#pragma unroll
    for (int r = 0; r < 6; r++) {
      T s = A[6 * r + c];
#pragma unroll
      for (int m = 0; m < r; m++) s -= D[6 * r + m] * x[m];
      x[r] = s;
    }
#pragma unroll
    for (int r = 0; r < 6; r++) A[6 * r + c] = x[r];
  }
  if (kFlow) flow_publish<true>(i, f);
}

// Rows too long for LDS, with the pivots applied in runs.  The values of row
// i stay in global memory.  A window of up to 2 nbatch pivots is prepared
// ahead, final or not: where the columns of their U parts lie in row i depends
// on the pattern alone.  Up to nbatch pivots of the window that are final form
// a run: wavefront 0 forms their L_ik in order, each applied at once to the
// run's own later L-part blocks (held in LDS), while the other wavefronts
// prepare the pivots that enter the window; then one pass reads every block of
// the rest of the row that a pivot of the run updates once, subtracts the
// run's contributions L_ik U_kj in pivot order and writes it once.  Every
// entry sees the operations of ilu_row_kernel in the same order, so the
// factors agree bit for bit.
// A thread takes kBatchCols columns of a block: it loads whole rows of U_kj
// in wide loads (one column per thread takes four times the load
// instructions, each touching as many lines), the next pivot's while the
// current one is applied, and shares each value of L_ik read from LDS among
// them.
// Dynamic LDS per position of row i: its column index, its place in the list
// of the run's blocks, and per pivot of the window the index (+ 1) of the
// position in the pivot's U part (0: not updated).
// What bounds it: memory.  400x400 plate, AMD + ILU(96), FP64: 352 GB read and
// written (PMC) in 60.6 ms, 5.8 TB/s, more than a copy reaches (4.95): a block
// update reads its U_kj from outside the L2, and rows share nothing.  FP32
// moves 160 GB in 41.4 ms, 3.9 TB/s, and its rows' own time counts as well:
// 9,266 rows of 370 to 1,750 blocks, 2.5 ms each on 512 places; a run of 7.7
// pivots took 42 us with the window of one run, 9 of them preparing the next
// one after it, 6 forming L_ik, 5 loading the pivots' edges, 12 the update, 9
// waiting.
#ifndef GPUFEM_ILU_BATCH
#define GPUFEM_ILU_BATCH 8
#endif
constexpr int kIluBatch = GPUFEM_ILU_BATCH;
constexpr int kIluPairSlots = kIluBatch * (kIluBatch - 1) / 2;
// slot of the pivot pair (p, q), p < q < kIluBatch
__device__ __forceinline__ int batch_pair(int p, int q) {
  return p * (2 * kIluBatch - p - 1) / 2 + (q - p - 1);
}
// dynamic LDS of a row of at most maxlen positions, runs of nbatch
__host__ __device__ constexpr int batch_stride(int maxlen) {
  return (maxlen + 7) / 8 * 8;
}
__host__ __device__ constexpr size_t batch_lds(int nbatch, int maxlen) {
  return (sizeof(short) * (size_t)(2 * nbatch + 1) + sizeof(int)) *
         batch_stride(maxlen);
}
// 400x400 plate, AMD + ILU(96), whole factorisation, columns per thread:
// FP64 1 / 2 / 3 / 6: 96 / 89 / 122 / 126 ms (3 and 6 leave room for one
// workgroup a CU), FP32 2 / 3 / 6: 78 / 78 / 101 ms; 256 or 1,024 threads
// 102 or 109 ms FP64.  (One column per thread, batches that waited for all
// their pivots' lists, and the row's pairs found by walking the U parts:
// 111 ms FP64, 97 ms FP32.)  Those with rows in LDS up to its whole size and a
// window of one run; up to half of it 83 / 65 ms, and with the next run
// prepared while L_ik are formed 72.7 / 54.9 ms (256x256 FP64 28.2 -> 23.7).
// Two columns a lane searched for at once; one or four 0.4 or 2 ms more.
constexpr int kBatchThreads = 512;
// A run waits for this many pivots unless it is the row's last one: rows far
// behind the chain would otherwise be read and written once a pivot.  75x150
// cylinder, FP64, with 1 / 2 / 4 / 8: 10.65 / 10.06 / 9.84 / 10.7 ms; plates
// the same within 1%.
constexpr int kRunLeast = 4;
template <typename T> constexpr int kBatchCols = sizeof(T) == 8 ? 2 : 3;
template <typename T, bool kFlow>
__global__ void __launch_bounds__(kBatchThreads, 4)
    ilu_row_batch_kernel(const int* __restrict__ level_rows, int nrows,
                         const int* __restrict__ rowp,
                         const int* __restrict__ cols,
                         const int* __restrict__ diag, T* vals, int* pivot,
                         Flow f, int nbatch, int maxlen) {
  constexpr int C = kBatchCols<T>, S = 6 / C;
  // blocks of a pivot's U part that load_pivot reads past the caches: its
  // first kHead and last kTail ones go through LDS
  constexpr int kTail = kEdgeBlocks<T>, kHead = kEdgeBlocks<T> - 1;
  constexpr int kEdge = 1 + kTail + kHead;  // with the diagonal block
  extern __shared__ __align__(16) unsigned char ilu_bdyn[];
  __shared__ int s_u0[2 * kIluBatch], s_nu[2 * kIluBatch];  // per window slot
  __shared__ __align__(16) T s_edge[kIluBatch][kEdge][36];
  __shared__ T s_udi[kIluBatch][6];  // 1 / diagonal of U_kk
  __shared__ __align__(16) T s_lik[kIluBatch][36];
  __shared__ T s_ab[kIluBatch][36];       // A_ik of the run's pivots
  __shared__ T s_uq[kIluPairSlots][36];   // U_kp,kq, p < q in the run
  __shared__ int s_row, s_rdy[2], s_cnt;
  const int i = flow_row<kFlow>(level_rows, nrows, f, &s_row);
  if (i < 0) return;
  const int tid = threadIdx.x, nth = kBatchThreads;
  const int r0 = rowp[i], r1 = rowp[i + 1], nb = r1 - r0, dl = diag[i] - r0;
  // hit[s * stride + pl] = 1 + index in U(k) of position pl for the pivot k
  // in slot s, or 0
  const int stride = batch_stride(maxlen), nwin = 2 * nbatch;
  unsigned short* hit = reinterpret_cast<unsigned short*>(ilu_bdyn);
  unsigned short* list = hit + (size_t)nwin * stride;
  int* scol = reinterpret_cast<int*>(list + stride);
  for (int t = tid; t < nb; t += nth) scol[t] = cols[r0 + t];
  for (int e = tid; e < nwin * stride / 8; e += nth)
    reinterpret_cast<int4*>(hit)[e] = make_int4(0, 0, 0, 0);
  if (tid == 0) s_rdy[0] = s_cnt = 0;
  int par = 0;
  __syncthreads();
  // pivots [k0, k1) of the row into their slots (pivot k: slot k % nwin, its
  // hits cleared) by wavefronts w0 .. 7: segments of kSeg columns of their U
  // parts in turn, kFind columns a lane in flight, searched for together
  constexpr int kFind = 2, kSeg = 64 * kFind;
  auto prepare = [&](int k0, int k1, int w0) {
    const int lane = tid % 64, nw = nth / 64 - w0;
    int lu0 = 0, lnu = 0;
    if (lane < k1 - k0) {
      const int k = scol[k0 + lane];
      lu0 = diag[k] + 1;
      lnu = rowp[k + 1] - lu0;
    }
    if (tid / 64 == w0 && lane < k1 - k0) {
      s_u0[(k0 + lane) % nwin] = lu0;
      s_nu[(k0 + lane) % nwin] = lnu;
    }
    int turn = tid / 64 - w0;
    for (int k = k0; k < k1; k++) {
      const int u0 = __builtin_amdgcn_readlane(lu0, k - k0);
      const int nu = __builtin_amdgcn_readlane(lnu, k - k0);
      unsigned short* const h = hit + (k % nwin) * stride;
      const int lo0 = k + 1;
      int top = 1;
      while (2 * top <= nb - lo0) top *= 2;
      int b = kSeg * turn;
      for (; b < nu; b += kSeg * nw) {
        int j[kFind], lo[kFind];
#pragma unroll
        for (int z = 0; z < kFind; z++) {
          const int t = b + 64 * z + lane;
          j[z] = t < nu ? cols[u0 + t] : 0;
          lo[z] = lo0;
        }
        for (int st = top; st > 0; st /= 2)
#pragma unroll
          for (int z = 0; z < kFind; z++) {
            const int at = lo[z] + st;
            if (at <= nb && scol[at - 1] < j[z]) lo[z] = at;
          }
#pragma unroll
        for (int z = 0; z < kFind; z++) {
          const int t = b + 64 * z + lane;
          if (t < nu && lo[z] < nb && scol[lo[z]] == j[z])
            h[lo[z]] = (unsigned short)(t + 1);
        }
      }
      turn = (b - nu) / kSeg;  // segments past this pivot's end
    }
  };
  // prepared pivots [kb, kw): runs are of at most nbatch, so that the next
  // ones can be prepared while a run's L_ik are formed
  int kb = 0, kw = min(nwin, dl);
  if (dl > 0) {
    prepare(0, kw, 0);
    __syncthreads();
  }
  while (kb < dl) {
    int pe = min(kw, kb + nbatch);  // the run [kb, pe)
    if (kFlow) {
      flow_wait<false>(scol, dl, pe < dl ? min(pe, kb + kRunLeast) - 1 : kb, s_rdy,
                       par, f);
      pe = min(pe, s_rdy[par]);
    }
    const int np = pe - kb, sb = kb % nwin;
    const int kn = min(kb + nwin, dl);  // pivots [kw, kn) are prepared now
    // slot of the run's pivot p
    auto slot = [&](int p) { return sb + p >= nwin ? sb + p - nwin : sb + p; };
    for (int e = tid; e < (kn - kw) * (stride / 8); e += nth) {
      const int s = (kw + e / (stride / 8)) % nwin;
      reinterpret_cast<int4*>(hit + s * stride)[e % (stride / 8)] =
          make_int4(0, 0, 0, 0);
    }
    // U_kk and the edge blocks of the pivots' U parts, and A_ik
    for (int e = tid; e < 36 * kEdge * np; e += nth) {
      const int p = e / (36 * kEdge), b = e / 36 % kEdge, q = e % 36;
      const int nu = s_nu[slot(p)], u0 = s_u0[slot(p)];
      // block of the row part D U: the diagonal, the head, the tail
      const int blk = b <= kHead ? b - 1 : nu - (kEdge - b);
      if (b > 0 && (blk < 0 || blk >= nu)) continue;
      const T u =
          load_pivot<T, kFlow>(vals + 36 * (size_t)(u0 + blk) + q, true);
      s_edge[p][b][q] = u;
      if (b == 0) {
        if (q % 7 == 0) s_udi[p][q / 7] = T(1) / u;
        s_ab[p][q] = vals[36 * (size_t)(r0 + kb + p) + q];
      }
    }
    // U_kp,kq for the pairs of the run
    if (np > 1)
      for (int e = tid; e < 36 * np * np; e += nth) {
        const int pq = e / 36, m = e % 36, p = pq / np, q = pq % np;
        if (q <= p) continue;
        const int v = hit[slot(p) * stride + kb + q];
        if (v)
          s_uq[batch_pair(p, q)][m] = load_pivot<T, kFlow>(
              vals + 36 * (size_t)(s_u0[slot(p)] + v - 1) + m,
              edge_block<T>(v - 1, s_nu[slot(p)]));
      }
    // the blocks past the run's L part that a pivot of the run updates
    for (int pl = pe + tid; pl < nb; pl += nth) {
      unsigned any = 0;
      for (int p = 0; p < np; p++) any |= hit[slot(p) * stride + pl];
      if (any) list[atomicAdd(&s_cnt, 1)] = (unsigned short)pl;
    }
    __syncthreads();
    const int items = S * s_cnt;
    // this thread's item: its block of the row, its columns, its values
    T a[6][C], u[6][C];
    int pl = -1, c0 = 0;
    T* A = nullptr;
    auto load_u = [&](int p) {  // false: pivot p does not update the block
      const int s = slot(p);
      const int tt = pl >= 0 ? (int)hit[s * stride + pl] - 1 : -1;
      if (tt < 0) return false;
      const int nu = s_nu[s];
      if (kFlow && edge_block<T>(tt, nu)) {
        const T* U = s_edge[p][tt >= nu - kTail ? kEdge - (nu - tt) : 1 + tt];
#pragma unroll
        for (int m = 0; m < 6; m++)
#pragma unroll
          for (int c = 0; c < C; c++) u[m][c] = U[6 * m + c0 + c];
      } else {
        const T* U = vals + 36 * (size_t)(s_u0[s] + tt) + c0;
#pragma unroll
        for (int m = 0; m < 6; m++)
#pragma unroll
          for (int c = 0; c < C; c++) u[m][c] = U[6 * m + c];
      }
      return true;
    };
    bool on = false;
    auto load_item = [&](int w) {
      pl = -1;
      if (w < items) {
        pl = list[w / S];
        c0 = C * (w % S);
        A = vals + 36 * (size_t)(r0 + pl) + c0;
#pragma unroll
        for (int r = 0; r < 6; r++)
#pragma unroll
          for (int c = 0; c < C; c++) a[r][c] = A[6 * r + c];
      }
      on = load_u(0);
    };
    load_item(tid);
    if (tid >= 64) {
      if (kn > kw) prepare(kw, kn, 1);
    } else {
      // wavefront 0: L_ik of each pivot, each applied to the run's later
      // L-part blocks before the next is formed
      for (int p = 0; p < np; p++) {
        if (tid < 6) {
          const int r = tid;
          T x[6];
#pragma unroll
          for (int c = 0; c < 6; c++) {
            T v = s_ab[p][6 * r + c];
#pragma unroll
            for (int m = 0; m < c; m++) v -= x[m] * s_edge[p][0][6 * m + c];
            x[c] = v * s_udi[p][c];
          }
#pragma unroll
          for (int c = 0; c < 6; c++) {
            s_ab[p][6 * r + c] = x[c];
            s_lik[p][6 * r + c] = x[c];
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (int e = tid; e < 36 * (np - 1 - p); e += 64) {
          const int q = p + 1 + e / 36, r = e % 36 / 6, c = e % 6;
          if (!hit[slot(p) * stride + kb + q]) continue;
          const T* U = s_uq[batch_pair(p, q)];
          T acc = 0;
#pragma unroll
          for (int m = 0; m < 6; m++) acc += s_lik[p][6 * r + m] * U[6 * m + c];
          s_ab[q][6 * r + c] = s_ab[q][6 * r + c] - acc;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
    }
    __syncthreads();
    if (tid == 0) s_cnt = 0;
    for (int e = tid; e < 36 * np; e += nth)
      vals[36 * (size_t)(r0 + kb + e / 36) + e % 36] = s_ab[e / 36][e % 36];
    for (int w = tid; w < items; w += nth) {
      if (w > tid) load_item(w);
      for (int p = 0; p < np; p++) {
        T uc[6][C];
        const bool now = on;
#pragma unroll
        for (int m = 0; m < 6; m++)
#pragma unroll
          for (int c = 0; c < C; c++) uc[m][c] = u[m][c];
        if (p + 1 < np) on = load_u(p + 1);
        if (now) {
#pragma unroll
          for (int r = 0; r < 6; r++) {
            T l[6];
#pragma unroll
            for (int m = 0; m < 6; m++) l[m] = s_lik[p][6 * r + m];
#pragma unroll
            for (int c = 0; c < C; c++) {
              T v = 0;
#pragma unroll
              for (int m = 0; m < 6; m++) v += l[m] * uc[m][c];
              a[r][c] = a[r][c] - v;
            }
          }
        }
      }
#pragma unroll
      for (int r = 0; r < 6; r++)
#pragma unroll
        for (int c = 0; c < C; c++) A[6 * r + c] = a[r][c];
    }
    __syncthreads();
    kb = pe;
    kw = kn;
  }
  __syncthreads();
  // factor the diagonal block (no pivoting); meanwhile the first pairs of the
  // U part are loaded
  T* D = vals + 36 * (size_t)(r0 + dl);
  T* Dl = s_ab[0];
  const int nr = nb - (dl + 1);
  constexpr int K = 4;  // (block, column) pairs per thread in flight
  T x[K][6];
  auto load_u_part = [&](int w0) {
#pragma unroll
    for (int z = 0; z < K; z++) {
      const int w = w0 + z * nth + tid;
      const T* B = D + 36 * (size_t)(1 + (w < 6 * nr ? w / 6 : 0)) + w % 6;
#pragma unroll
      for (int r = 0; r < 6; r++) x[z][r] = w < 6 * nr ? B[6 * r] : T(0);
    }
  };
  load_u_part(0);
  if (tid < 64) {
    const int r = tid < 6 ? tid : 5;
    T d[6];
#pragma unroll
    for (int m = 0; m < 6; m++) d[m] = D[6 * r + m];
    factor_diag(d, tid, i, pivot);
    if (tid < 6) {
#pragma unroll
      for (int m = 0; m < 6; m++) {
        Dl[6 * r + m] = d[m];
        store_final<T, kFlow>(D + 6 * r + m, d[m]);
      }
    }
  }
  __syncthreads();
  // U_ij = L_ii^-1 A_ij for the blocks right of the diagonal
  for (int w0 = 0; w0 < 6 * nr; w0 += K * nth) {
    if (w0 > 0) load_u_part(w0);
#pragma unroll
    for (int z = 0; z < K; z++) {
      const int w = w0 + z * nth + tid;
      if (w >= 6 * nr) continue;
#pragma unroll
      for (int r = 1; r < 6; r++)
#pragma unroll
        for (int m = 0; m < r; m++) x[z][r] -= Dl[6 * r + m] * x[z][m];
      T* B = D + 36 * (size_t)(1 + w / 6) + w % 6;
#pragma unroll
      for (int r = 0; r < 6; r++) store_final<T, kFlow>(B + 6 * r, x[z][r]);
    }
  }
  if (kFlow) flow_publish<false>(i, f);
}

// The same factorisation with row i held in LDS for the whole row: L_ik is
// formed from, and the updates A_ij -= L_ik U_kj are applied to, the LDS
// copy, so the only global accesses inside the pivot loop are reads of the
// final rows k.  Those are pipelined: the U-part bounds of every pivot row
// are read into LDS once; while pivot k is processed, the column indices of
// pivot k+2 and, if it is final by then, U_kk and each thread's U_kj columns
// of pivot k+1 are loaded into registers, and the positions of pivot k+1's
// columns in row i are searched.  The row is written back once at the end,
// D and U first.
// Arithmetic is that of ilu_row_kernel, operation for operation.
// Dynamic LDS: 36 * nb values, nb column indices, 2 * nl pivot bounds.
#ifndef GPUFEM_ILU_PAIRS
#define GPUFEM_ILU_PAIRS 2
#endif
constexpr int kIluPairs = GPUFEM_ILU_PAIRS;  // (block, column) pairs of U_kj per thread
constexpr int kIluCols = 4;   // prefetched column indices per staging thread
// Short rows (levels whose rows, and so their pivot rows' U parts, are
// short) run in 256-thread workgroups: the kernel's registers allow 12
// wavefronts a CU, one 512-thread row or three 256-thread ones, and a short
// row spends its time in per-row latency (ticket, loads of its pattern and
// pivot bounds, diagonal factorisation, write-back and release), not in its
// few pivot updates.  400x400 plate, AMD + ILU(96), FP64 / FP32
// factorisation: 83.4 / 59.1 ms with 512 threads throughout, 76.8 / 58.9 with
// rows up to 128 blocks in 256-thread workgroups, 73.0 / 55.4 up to 256; 75x150
// cylinder FP64 10.33, 9.93 and 9.86.  (The staging
// threads hold 4 * (256 - 6) column indices: pivot U parts up to 1,000.)
constexpr int kIluShortThreads = 256;
constexpr int kIluShortRow = 256;  // longest row (blocks) taken that way
template <typename T, bool kFlow, int kThreads = kIluThreads>
__global__ void __launch_bounds__(kThreads)
    ilu_row_lds_kernel(const int* __restrict__ level_rows, int nrows,
                       const int* __restrict__ rowp,
                       const int* __restrict__ cols,
                       const int* __restrict__ diag, T* vals, int* pivot,
                       Flow f, int maxlen) {
  extern __shared__ __align__(16) unsigned char ilu_dyn[];
  __shared__ T udg[2][36];
  __shared__ T udi[2][6];  // 1 / diagonal of U_kk
  __shared__ T lik[36];
  __shared__ int s_row, s_rdy[2];
  const int i = flow_row<kFlow>(level_rows, nrows, f, &s_row);
  if (i < 0) return;
  const int tid = threadIdx.x, nth = blockDim.x;
  const int r0 = rowp[i], r1 = rowp[i + 1], nb = r1 - r0, dl = diag[i] - r0;
  T* row = reinterpret_cast<T*>(ilu_dyn);
  int* scol = reinterpret_cast<int*>(row + 36 * (size_t)nb);
  int* ubs = scol + nb;  // [2 * kl]: U part [u0, u1) of pivot row scol[kl]
  // local positions in row i of two pivots' U-part columns, or -1
  int* const pos[2] = {ubs + 2 * nb, ubs + 2 * nb + maxlen};
  for (int e = tid; e < 36 * nb; e += nth) row[e] = vals[36 * (size_t)r0 + e];
  for (int t = tid; t < nb; t += nth) {
    const int j = cols[r0 + t];
    scol[t] = j;
    if (t < dl) {
      ubs[2 * t] = diag[j] + 1;
      ubs[2 * t + 1] = rowp[j + 1];
    }
  }
  if (tid == 0) s_rdy[0] = 0;
  int par = 0;
  __syncthreads();
  // dataflow: pivot kl is waited for when its turn comes; its values are read
  // one pivot ahead where it is known to be final by then
  auto wait_for = [&](int kl) {
    if (kFlow) flow_wait<false>(scol, dl, kl, s_rdy, par, f);
  };
  auto ready = [&](int kl) { return !kFlow || s_rdy[par] > kl; };
  const int ts = tid - 6, ns = nth - 6;  // staging threads (tid >= 6)
  // position of column j among scol[lo..nb), or -1
  auto find = [&](int j, int lo) {
    int hi = nb;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (scol[mid] < j)
        lo = mid + 1;
      else
        hi = mid;
    }
    return (lo < nb && scol[lo] == j) ? lo : -1;
  };
  // registers: this thread's U_kj columns for the current and next pivot,
  // and (staging threads) the column indices of the pivot after next and the
  // U_kk entry of the next
  T uv[kIluPairs][6], un[kIluPairs][6];
  int pc[kIluCols];
  T pd = T(0);
  // (block, column) pairs of a pivot: w0, w0 + sn, ...  Where the last pivot
  // was waited for (a chain), they are left to wavefronts 1 .., and wavefront
  // 0 updates the diagonal block and factors it meanwhile: 0.7 us of the 5.2
  // of a row of the chain.
  bool split = false;
  auto load_u = [&](int kl, T (&dst)[kIluPairs][6]) {
    const int u0 = kl < dl ? ubs[2 * kl] : 0;
    const int nu = kl < dl ? ubs[2 * kl + 1] - u0 : 0;
    const int w0 = split ? tid - 64 : tid, sn = split ? nth - 64 : nth;
#pragma unroll
    for (int sp = 0; sp < kIluPairs; sp++) {
      const int w = w0 + sp * sn;
      const bool ok = w0 >= 0 && w < 6 * nu;
      const T* U =
          vals + 36 * (size_t)(u0 + (ok ? w / 6 : 0)) + (ok ? w % 6 : 0);
      const bool edge = edge_block<T>(w / 6, nu);
#pragma unroll
      for (int m = 0; m < 6; m++)
        dst[sp][m] = ok ? load_pivot<T, kFlow>(U + 6 * m, edge) : T(0);
    }
  };
  auto load_cols = [&](int kl) {
    const int u0 = kl < dl ? ubs[2 * kl] : 0;
    const int nu = kl < dl ? ubs[2 * kl + 1] - u0 : 0;
#pragma unroll
    for (int q = 0; q < kIluCols; q++) {
      const int t = ts + q * ns;
      pc[q] = (ts >= 0 && t < nu) ? cols[u0 + t] : -1;
    }
  };
  // positions of pivot kl into buffer buf from the registers
  auto stage_from_regs = [&](int kl, int buf) {
    const int u0 = ubs[2 * kl], nu = ubs[2 * kl + 1] - u0;
#pragma unroll
    for (int q = 0; q < kIluCols; q++) {
      const int t = ts + q * ns;
      if (t < nu) pos[buf][t] = find(pc[q], kl + 1);
    }
    for (int t = ts + kIluCols * ns; t < nu; t += ns)
      pos[buf][t] = find(cols[u0 + t], kl + 1);
  };
  // U_kk of pivot kl (threads 6 .. 41), into buffer buf
  auto load_diag = [&](int kl) {
    if (ts >= 0 && ts < 36)
      pd = load_pivot<T, kFlow>(vals + 36 * (size_t)(ubs[2 * kl] - 1) + ts,
                                true);
  };
  auto stage_diag = [&](int buf) {
    if (ts >= 0 && ts < 36) {
      udg[buf][ts] = pd;
      if (ts % 7 == 0) udi[buf][ts / 7] = T(1) / pd;
    }
  };
  if (dl > 0) {
    const int u0 = ubs[0], nu = ubs[1] - u0;
    for (int t = tid; t < nu; t += nth) pos[0][t] = find(cols[u0 + t], 1);
    load_cols(1);
  }
  // the diagonal block (no pivoting), by wavefront 0
  T* const D = row + 36 * dl;
  auto factor = [&]() {
    const int r = tid < 6 ? tid : 5;
    T d[6];
#pragma unroll
    for (int m = 0; m < 6; m++) d[m] = D[6 * r + m];
    factor_diag(d, tid, i, pivot);
    if (tid < 6) {
#pragma unroll
      for (int m = 0; m < 6; m++) D[6 * r + m] = d[m];
    }
  };
  bool have = false;  // pivot kl's values are staged
  __syncthreads();
  for (int kl = 0; kl < dl; kl++) {
    const int cur = kl & 1;
    const int u0 = ubs[2 * kl], nu = ubs[2 * kl + 1] - u0;
    bool upd = false;  // the last pivot updates the diagonal block
    // wavefront 0, which has no pairs of it: column tid % 6 of U_ki into uv[0]
    auto load_ud = [&]() {
      int at = -1;
      for (int t = 0; t < nu && at < 0; t += 64) {
        const unsigned long long m =
            __ballot(t + tid < nu && pos[cur][t + tid] == dl);
        if (m) at = t + __ffsll((long long)m) - 1;
      }
      upd = at >= 0;
      if (!upd) return;
      const T* U = vals + 36 * (size_t)(u0 + at) + tid % 6;
      const bool edge = edge_block<T>(at, nu);
#pragma unroll
      for (int m = 0; m < 6; m++)
        uv[0][m] = load_pivot<T, kFlow>(U + 6 * m, edge);
    };
    if (!have) {
      wait_for(kl);
      split = kFlow && kl == dl - 1;
      load_u(kl, uv);
      load_diag(kl);
      if (split && tid < 64) load_ud();
      stage_diag(cur);
      __syncthreads();
    }
    // the next pivot's values, if it is known to be final (waiting for it
    // here would hold back this pivot: in a chain, the last two pivots of a
    // row would be applied after the last one had become final)
    const bool next = kl + 1 < dl && ready(kl + 1);
    if (next) {
      load_u(kl + 1, un);
      load_diag(kl + 1);
    }
    if (tid < 6) {
      const int r = tid;
      const T* Ukk = udg[cur];
      const T* Ui = udi[cur];
      T* Aik = row + 36 * kl;
      T x[6];
#pragma unroll
      for (int c = 0; c < 6; c++) {
        T v = Aik[6 * r + c];
#pragma unroll
        for (int m = 0; m < c; m++) v -= x[m] * Ukk[6 * m + c];
        x[c] = v * Ui[c];
      }
#pragma unroll
      for (int c = 0; c < 6; c++) {
        Aik[6 * r + c] = x[c];
        lik[6 * r + c] = x[c];
      }
    } else if (kl + 1 < dl) {
      stage_from_regs(kl + 1, cur ^ 1);
      load_cols(kl + 2);
    }
    __syncthreads();
    // A_ij -= L_ik U_kj on the LDS row
    const int w0 = split ? tid - 64 : tid, sn = split ? nth - 64 : nth;
    if (split && tid < 64) {
      if (upd && tid < 36) {
        const int r = tid / 6;
        T v = 0;
#pragma unroll
        for (int m = 0; m < 6; m++) v += lik[6 * r + m] * uv[0][m];
        row[36 * dl + tid] -= v;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      factor();
    }
#pragma unroll
    for (int sp = 0; sp < kIluPairs; sp++) {
      const int w = w0 + sp * sn;
      if (w0 >= 0 && w < 6 * nu) {
        const int pl = pos[cur][w / 6], c = w % 6;
        if (pl >= 0 && !(split && pl == dl)) {
#pragma unroll
          for (int r = 0; r < 6; r++) {
            T v = 0;
#pragma unroll
            for (int m = 0; m < 6; m++) v += lik[6 * r + m] * uv[sp][m];
            row[36 * pl + 6 * r + c] -= v;
          }
        }
      }
    }
    for (int w = w0 + kIluPairs * sn; w0 >= 0 && w < 6 * nu; w += sn) {
      const int pl = pos[cur][w / 6], c = w % 6;
      if (pl < 0 || (split && pl == dl)) continue;
      const T* U = vals + 36 * (size_t)(u0 + w / 6) + c;
      const bool edge = edge_block<T>(w / 6, nu);
      T um[6];
#pragma unroll
      for (int m = 0; m < 6; m++) um[m] = load_pivot<T, kFlow>(U + 6 * m, edge);
#pragma unroll
      for (int r = 0; r < 6; r++) {
        T v = 0;
#pragma unroll
        for (int m = 0; m < 6; m++) v += lik[6 * r + m] * um[m];
        row[36 * pl + 6 * r + c] -= v;
      }
    }
    if (next) stage_diag(cur ^ 1);
    __syncthreads();
#pragma unroll
    for (int sp = 0; sp < kIluPairs; sp++)
#pragma unroll
      for (int m = 0; m < 6; m++) uv[sp][m] = un[sp][m];
    have = next;
  }
  if (!split) {
    if (tid < 64) factor();
    __syncthreads();
  }
  // U_ij = L_ii^-1 A_ij for the blocks right of the diagonal
  const int nr = nb - (dl + 1);
  for (int w = tid; w < 6 * nr; w += nth) {
    const int t = w / 6, c = w % 6;
    T* A = row + 36 * (dl + 1 + t);
    T x[6];
#pragma unroll
    for (int r = 0; r < 6; r++) {
      T sv = A[6 * r + c];
#pragma unroll
      for (int m = 0; m < r; m++) sv -= D[6 * r + m] * x[m];
      x[r] = sv;
    }
#pragma unroll
    for (int r = 0; r < 6; r++) A[6 * r + c] = x[r];
  }
  __syncthreads();
  // the rows that wait read D and U only: L follows the flag
  for (int e = 36 * dl + tid; e < 36 * nb; e += nth)
    store_final<T, kFlow>(vals + 36 * (size_t)r0 + e, row[e]);
  if (kFlow) flow_publish<false>(i, f);
  for (int e = tid; e < 36 * dl; e += nth) vals[36 * (size_t)r0 + e] = row[e];
}

// Six lanes per row (lane = scalar row r), ten rows per wave.
template <typename T, bool kLower>
__global__ void __launch_bounds__(256)
    trsv_level_kernel(const int* __restrict__ level_rows, int nrows,
                      const int* __restrict__ rowp,
                      const int* __restrict__ cols,
                      const int* __restrict__ diag, const T* __restrict__ lu,
                      const T* __restrict__ b, T* __restrict__ x) {
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int li = (blockIdx.x * (blockDim.x / 64) + wave) * 10 + lane / 6;
  const int r = lane % 6;
  const bool active = lane < 60 && li < nrows;
  const int i = active ? level_rows[li] : 0;
  T s = 0;
  int di = 0;
  if (active) {
    di = diag[i];
    s = b[6 * (size_t)i + r];
    const int k0 = kLower ? rowp[i] : di + 1;
    const int k1 = kLower ? di : rowp[i + 1];
    for (int k = k0; k < k1; k++) {
      const T* a = lu + 36 * (size_t)k + 6 * r;
      const T* xk = x + 6 * (size_t)cols[k];
#pragma unroll
      for (int c = 0; c < 6; c++) s -= a[c] * xk[c];
    }
  }
  // diagonal block solve across the six lanes of the row
  const int base = lane - r;  // first lane of this row's group
  const T* D = lu + 36 * (size_t)di + 6 * r;
  if (kLower) {
#pragma unroll
    for (int c = 0; c < 5; c++) {
      const T yc = __shfl(s, base + c, 64);
      if (active && r > c) s -= D[c] * yc;
    }
  } else {
    const T dinv = active ? T(1) / D[r] : T(0);
#pragma unroll
    for (int c = 5; c >= 0; c--) {
      if (active && r == c) s *= dinv;
      const T yc = __shfl(s, base + c, 64);
      if (active && r < c) s -= D[c] * yc;
    }
  }
  if (active) x[6 * (size_t)i + r] = s;
}


constexpr int kSweepThreads = 256;        // 4 wavefronts per workgroup
// Batches of 10 blocks of a pass whose factor values are loaded into
// registers before the row waits; blocks beyond them are loaded after the
// wait, on the row's critical path.  With passes of 128 blocks
// (400x400 plate, AMD + ILU(16), L+U pair): 3 -> 4.33 ms, 4 -> 4.09,
// 6 -> 3.71, 8 -> 3.48, 10 -> 3.36, 12 -> 3.29 (256 VGPRs).  At ILU(96)
// (rows of hundreds of blocks, so most passes are full): 12 batches of a
// 128-block pass 7.32 ms, 13 (the whole pass) 6.83 ms, passes of 64 blocks
// with 7 batches (the whole pass, 178 VGPRs) 5.99 ms: no load is left
// after the wait, and the wait gathers half as many dependencies.
#ifndef GPUFEM_SWEEP_ITER
#define GPUFEM_SWEEP_ITER 7
#endif
#ifndef GPUFEM_SWEEP_MINWAVES
#define GPUFEM_SWEEP_MINWAVES 1
#endif
// Waiting on the latest-level dependency alone before gathering the others
// cuts polling traffic but adds a round trip per row: 4.70 vs 3.54 ms a sweep
// pair on the 400x400 plate (AMD, ILU(12)).
// longest sleep between polls, x 64 cycles: L+U pair on the 400x400 plate
// (ILU(16), 4 batches) 16 -> 4.14 ms, 8 -> 4.09, 4 -> 4.06, 2 -> 4.06,
// 1 -> 4.07; with 12 batches 8 -> 3.29, 2 -> 3.26; ILU(96), entries of a
// dependency in consecutive lanes: 1 -> 5.29, 2 -> 5.26, 4 -> 5.25
#ifndef GPUFEM_SWEEP_BACKOFF
#define GPUFEM_SWEEP_BACKOFF 2
#endif
// A waiting row polls only its pending entries, one poll in flight.  Two
// interleaved streams of polls of all the row's entries, the second half a
// round trip after the first, took the L+U pair of the 400x400 plate (AMD +
// ILU(96)) from 5.69 to 8.8 ms: polling traffic delays the stores and loads
// on the critical path more than the earlier detection gains.
// wavefronts per compute unit for a sweep launch: fewer waiting wavefronts
// mean less polling and counter traffic; measured on the 400x400 plate
// (AMD + ILU(12)): 16 -> 4.37 ms per L+U pair, 4 -> 3.62, 3 -> 3.51,
// 2 -> 3.64, 1 -> 5.17; with 12 register batches (ILU(16)): 2 -> 3.55,
// 3 -> 3.26, 4 -> 3.31, 5 -> 3.61; with 64-block passes (ILU(96)): 3 -> 5.99,
// 4 -> 5.95, 6 -> 6.13, 8 -> 6.19; with the entries of a dependency in
// consecutive lanes (fewer memory requests per wavefront): 3 -> 5.26,
// 4 -> 5.12, 5 -> 5.29, 6 -> 5.30
#ifndef GPUFEM_SWEEP_WAVES_PER_CU
#define GPUFEM_SWEEP_WAVES_PER_CU 4
#endif
constexpr int kSweepIter = GPUFEM_SWEEP_ITER;  // block batches in registers
constexpr int kCounterStride = 32;        // 256 bytes between the counters
constexpr int kGather = 64;               // dependency blocks per pass
// blocks next to the diagonal taken as a row's last pass: ILU(96) plate,
// L+U pair 5.99 ms without, 5.90 / 5.82 / 5.84 / 5.87 / 5.89 ms with 4 / 6 /
// 8 / 16 / 24 in every row longer than that, 5.77 ms with 8 in the rows of
// more than one pass (a row of at most kGather blocks keeps its one pass);
// with the entries of a dependency in consecutive lanes 5 / 8 / 10: 5.27 /
// 5.26 / 5.26 ms
#ifndef GPUFEM_SWEEP_NEAR
#define GPUFEM_SWEEP_NEAR 8
#endif
constexpr int kNearPass = GPUFEM_SWEEP_NEAR;
static_assert(kGather % 64 == 0, "a pass spreads over whole wavefronts");
constexpr unsigned kSpinLimit = 1u << 20; // bounded polls per batch

// Sentinel values: signalling NaNs.  Arithmetic never produces a signalling
// NaN (results are quiet), so an output entry that holds the sentinel has not
// been written yet in the current sweep.
template <typename T> struct Sentinel;
template <> struct Sentinel<double> {
  using Bits = unsigned long long;
  static constexpr Bits value = 0x7FF4A5A5A5A5A5A5ull;
};
template <> struct Sentinel<float> {
  using Bits = unsigned int;
  static constexpr Bits value = 0x7FA5A5A5u;
};

template <typename T>
__device__ __forceinline__ typename Sentinel<T>::Bits load_bits(const T* p) {
  using B = typename Sentinel<T>::Bits;
  return __hip_atomic_load(reinterpret_cast<const B*>(p), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void store_value(T* p, T v) {
  using B = typename Sentinel<T>::Bits;
  __hip_atomic_store(reinterpret_cast<B*>(p), __builtin_bit_cast(B, v),
                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename T>
__global__ void fill_sentinel_kernel(size_t n, T* x) {
  using B = typename Sentinel<T>::Bits;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) reinterpret_cast<B*>(x)[i] = Sentinel<T>::value;
}

// Sync-free sweep.  The output vector is filled with the sentinel before the
// launch; every output entry is written exactly once, with a relaxed
// agent-scope atomic store, and a row reads each entry it depends on with
// relaxed agent-scope atomic loads until the value is no longer the sentinel.
// Each entry validates itself, so no fences or flags are needed.
//
// Rows are taken from a monotonic 64-bit counter in chunks, either chunks of
// rows of one level in level order (order = the level-sorted rows), or
// chains of consecutive rows in sweep order (order = null).  Either way every
// dependency of a row lies in an earlier chunk, handed out earlier to a
// running wavefront, or earlier in the same chunk, so the sweep cannot
// deadlock whatever the number of resident workgroups.
//
// Per row, in passes of up to kGather dependency blocks: the pass's factor
// blocks are loaded into registers, then its dependencies' entries (six
// consecutive lanes per dependency) are loaded together, polled until none
// holds the sentinel and parked in LDS, so a pass costs about two memory
// round trips (column indices, then dependency entries) whatever its
// length; slot t = lane / 6 (0..9) takes blocks t, t+10, ... of the pass
// with r = lane % 6 the scalar row; the 6x6 diagonal block is solved by
// lanes 0-5 (v_readlane broadcasts with one row per wavefront).  The row
// last solved by the wavefront is kept in registers (a row often depends on
// the row just before it).
//
// fill_next (lower sweep only, may be null): the entries of the row in the
// upper sweep's output are set to the sentinel once the row's rhs is read,
// which allows that output to alias the rhs.
//
// kBatched: one launch sweeps the systems of several solves.  Chunk kc of
// the launch is chunk merged[kc].y of system merged[kc].x, whose arrays are
// in slots[merged[kc].x]; the merged list takes the systems' chunks level by
// level, so every row waited on is still in an earlier chunk.
template <typename T, bool kLower, int kRows, bool kBatched = false>
__global__ void __launch_bounds__(kSweepThreads, GPUFEM_SWEEP_MINWAVES)
    trsv_syncfree_kernel(const int4* __restrict__ meta_,
                         const int* __restrict__ cols_,
                         const int* __restrict__ chunk_ptr_, int nchunks,
                         const T* __restrict__ lu_, const T* b_, T* x_,
                         T* fill_next_, unsigned long long* counter,
                         unsigned long long base, int* err,
                         const SweepSlot<T>* __restrict__ slots = nullptr,
                         const int2* __restrict__ merged = nullptr) {
  using B = typename Sentinel<T>::Bits;
  const int4* __restrict__ meta = meta_;
  const int* __restrict__ cols = cols_;
  const int* __restrict__ chunk_ptr = chunk_ptr_;
  const T* __restrict__ lu = lu_;
  const T* b = b_;
  T* x = x_;
  T* fill_next = fill_next_;
  int cur_slot = -1;
  constexpr int G = 64 / kRows;        // lanes per row
  constexpr int kS = G / 6;            // block slots per row (10 or 5)
  constexpr int kH = kGather / G;      // dependency blocks per lane per pass
  constexpr bool kUseCache = kRows == 1;
  __shared__ T xs_all[kSweepThreads / 64][kRows][kGather][6];
  const int lane = threadIdx.x % 64;
  const int grp = lane / G, gl = lane % G, g0 = grp * G;
  const int t = gl / 6, r = gl % 6;
  const bool act = gl < 6 * kS;
  T(&xs)[kGather][6] = xs_all[threadIdx.x / 64][grp];
  // the last row solved by this wavefront (one row per wavefront only): a
  // chain's row usually depends on the row just before it
  int cid = -1;
  T cx[6];
#pragma unroll
  for (int c = 0; c < 6; c++) cx[c] = T(0);
  auto cached = [&](int j) { return kUseCache && cid == j; };
  // Wavefront c of a workgroup draws the chunks c, c + kCounters, ... from
  // counter c: atomics on one address take 12 ns each, 1.8 ms a sweep with a
  // ticket per row of the 400x400 plate.  Every workgroup has a wavefront of
  // each class, so the lowest unfinished chunk is always held, or next in
  // line for a wavefront that holds no unfinished chunk.
  constexpr int kCounters = kBatched ? 1 : kSweepThreads / 64;
  const int cls = kBatched ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  counter += kCounterStride * cls;
  const int ntk = (nchunks + kCounters - 1) / kCounters;
  unsigned long long tk = 0;
  if (lane == 0) tk = atomicAdd(counter, 1ull);
  tk = __shfl(tk, 0, 64);
  long long kc = (long long)(tk - base);
  for (; kc < ntk; kc = (long long)(tk - base)) {
    // take the next chunk now: the counter round trip overlaps this chunk
    unsigned long long tn = 0;
    if (lane == 0) tn = atomicAdd(counter, 1ull);
    int lc = (int)kc * kCounters + cls;
    if (lc >= nchunks) {
      tk = __shfl(tn, 0, 64);
      continue;
    }
    if constexpr (kBatched) {
      const int2 mc = merged[kc];
      lc = mc.y;
      if (*slots[mc.x].go != 1) {  // this system takes no step now
        tk = __shfl(tn, 0, 64);
        continue;
      }
      if (mc.x != cur_slot) {
        cur_slot = mc.x;
        const SweepSlot<T>& S = slots[mc.x];
        meta = kLower ? S.lmeta : S.umeta;
        chunk_ptr = kLower ? S.lchunk : S.uchunk;
        cols = S.cols;
        lu = S.lu;
        b = kLower ? S.b : S.tmp;
        x = kLower ? S.tmp : S.x;
        fill_next = kLower ? S.x : nullptr;
        cid = -1;  // the cached row belongs to another system
      }
    }
    const int p0 = chunk_ptr[lc], p1 = chunk_ptr[lc + 1];
    int4 mnext = (p0 + grp < p1) ? meta[p0 + grp] : make_int4(0, 0, 0, 0);
    for (int pb = p0; pb < p1; pb += kRows) {
      // rows pb + grp of one level (independent when kRows > 1)
      const bool live = pb + grp < p1;
      const int4 m = mnext;
      if (pb + kRows + grp < p1) mnext = meta[pb + kRows + grp];
      const int i = m.x, k0 = live ? m.y : 0, k1 = live ? m.z : 0;
      const int di = kLower ? m.z : m.y - 1;
      T s = (live && gl < 6) ? b[6 * (size_t)i + gl] : T(0);
      if (kLower && fill_next && live && gl < 6)
        reinterpret_cast<B*>(fill_next)[6 * (size_t)i + gl] =
            Sentinel<T>::value;
      T drow[6];
#pragma unroll
      for (int mm = 0; mm < 6; mm++)
        drow[mm] = (live && gl < 6) ? lu[36 * (size_t)di + 6 * gl + mm] : T(0);
      // reciprocal of this lane's diagonal entry, formed before any wait
      T dd = T(1);
#pragma unroll
      for (int mm = 0; mm < 6; mm++)
        if (gl == mm) dd = drow[mm];
      const T dinv = (!kLower && live && gl < 6) ? T(1) / dd : T(0);
      // the compiler would otherwise sink the division (a dozen dependent
      // instructions) past the waits onto the critical path: 400x400 plate,
      // AMD + ILU(96), L+U pair 5.78 -> 5.69 ms
      asm volatile("" ::"v"(dinv));
      // Per pass of up to kGather blocks: the first kSweepIter*kS blocks'
      // values are loaded before anything waits; the pass's column indices
      // are read (lane q: blocks q, q+G, ...) and the dependencies' entries
      // are loaded at once, polled until no sentinel is left, and parked in
      // LDS; then lanes (t, r) accumulate A[q][r][:] . x[col_q][:].
      T acc = T(0);
      const int nb = k1 - k0;
      // The row's latest dependency is usually its nearest row: the last
      // block of an L row, the first of a U row.  In rows of more than one
      // pass the kNearPass blocks next to the diagonal form the last pass,
      // so that little work is left once the latest dependency arrives; the
      // rest go in passes of kGather blocks, U rows taking theirs last to
      // first, so that the passes that wait longest come last and the
      // others overlap with the wait.
      const bool split = kNearPass > 0 && kRows == 1 && nb > kGather;
      const int nfar = split ? nb - kNearPass : nb;
      const int nfp = (nfar + kGather - 1) / kGather;
      int npass = nfp + (split ? 1 : 0);
      // every row group of the wavefront runs the same number of passes
#pragma unroll
      for (int o = G; o < 64; o <<= 1)
        npass = max(npass, __shfl_xor(npass, o, 64));
      for (int pi = 0; pi < npass; pi++) {
        int g0b, ng;
        if (split && pi == npass - 1) {
          g0b = kLower ? k1 - kNearPass : k0;
          ng = kNearPass;
        } else {
          const int j = kLower ? pi : nfp - 1 - pi;
          const int fb = kLower ? k0 : k0 + (split ? kNearPass : 0);
          const int fe = kLower ? (split ? k1 - kNearPass : k1) : k1;
          g0b = fb + j * kGather;
          ng = max(0, min(kGather, fe - g0b));
        }
        T a[kSweepIter][6];
#pragma unroll
        for (int it = 0; it < kSweepIter; it++) {
          const int q = kS * it + t;
          const bool ok = act && q < ng;
          const T* ap = lu + 36 * (size_t)(ok ? g0b + q : 0) + 6 * r;
#pragma unroll
          for (int c = 0; c < 6; c++) a[it][c] = ok ? ap[c] : T(0);
        }
        // The pass's dependency entries, kE per lane.  One row per
        // wavefront: lane l holds entries e = l + 64 k of the pass's 6 ng
        // (dependency e / 6, component e % 6), so the six entries of a
        // dependency sit in consecutive lanes and each load instruction
        // touches a sixth as many cache lines as with a dependency per lane;
        // several rows per wavefront: lane gl holds the six entries of
        // dependencies gl + G h.  400x400 plate, AMD + ILU(96), L+U pair:
        // 5.69 ms with a dependency per lane, 5.26 ms with its entries in
        // consecutive lanes (each poll of a waiting row is then one or two
        // requests instead of six).
        constexpr bool kT = kRows == 1;
        constexpr int kE = 6 * kH;
        int jq[kE], jc[kE], jj[kE];
        B xb[kE];
#pragma unroll
        for (int k = 0; k < kE; k++) {
          if constexpr (kT) {
            jq[k] = (lane + 64 * k) / 6;
            jc[k] = (lane + 64 * k) % 6;
          } else {
            jq[k] = gl + G * (k / 6);
            jc[k] = k % 6;
          }
          jj[k] = jq[k] < ng ? cols[g0b + jq[k]] : -1;
        }
#pragma unroll
        for (int k = 0; k < kE; k++)
          xb[k] = (jj[k] >= 0 && !cached(jj[k]))
                      ? load_bits(x + 6 * (size_t)jj[k] + jc[k])
                      : B(0);
        unsigned spins = 0;
        int nap = 1;
        for (;;) {
          bool pending = false;
#pragma unroll
          for (int k = 0; k < kE; k++)
            pending |= xb[k] == Sentinel<T>::value;
          if (!__any(pending)) break;
          if (++spins > kSpinLimit) {
            if (lane == 0)
              __hip_atomic_store(err, 1, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int k = 0; k < kE; k++) xb[k] = B(0);
            break;
          }
          // back off while the dependencies are not ready: many waiting
          // wavefronts polling at full rate load the memory system
          for (int z = 0; z < nap; z++) __builtin_amdgcn_s_sleep(1);
          nap = nap * 2 > GPUFEM_SWEEP_BACKOFF ? GPUFEM_SWEEP_BACKOFF : nap * 2;
#pragma unroll
          for (int k = 0; k < kE; k++)
            if (xb[k] == Sentinel<T>::value)
              xb[k] = load_bits(x + 6 * (size_t)jj[k] + jc[k]);
        }
        // park the dependencies in this row group's LDS slice
#pragma unroll
        for (int k = 0; k < kE; k++) {
          if (jq[k] < ng) {
            T v = __builtin_bit_cast(T, xb[k]);
            if (cached(jj[k])) {
              // cx[jc[k]] without a dynamically indexed register array
              v = cx[0];
#pragma unroll
              for (int cc = 1; cc < 6; cc++)
                if (jc[k] == cc) v = cx[cc];
            }
            xs[jq[k]][jc[k]] = v;
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int it = 0; it < kSweepIter; it++) {
          const int q = kS * it + t;
          if (act && q < ng) {
#pragma unroll
            for (int c = 0; c < 6; c++) acc += a[it][c] * xs[q][c];
          }
        }
        for (int q = kS * kSweepIter + t; act && q < ng; q += kS) {
          const T* ap = lu + 36 * (size_t)(g0b + q) + 6 * r;
#pragma unroll
          for (int c = 0; c < 6; c++) acc += ap[c] * xs[q][c];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
      // sum the slots of scalar row r into lane r of the group
      T rs = T(0);
#pragma unroll
      for (int u = 0; u < kS; u++) rs += __shfl(acc, g0 + 6 * u + (gl % 6), 64);
      s -= (gl < 6) ? rs : T(0);
      // the diagonal block solve is on the critical path of every level:
      // with one row per wavefront the source lane is uniform and
      // v_readlane broadcasts it (400x400 plate, AMD + ILU(96): L+U pair
      // 7.75 -> 7.34 ms against ds_bpermute shuffles)
      auto bcast = [&](T v, int l) {
        if constexpr (kRows == 1)
          return read_lane(v, l);
        else
          return __shfl(v, g0 + l, 64);
      };
      if (kLower) {
#pragma unroll
        for (int mm = 0; mm < 5; mm++) {
          const T ym = bcast(s, mm);
          if (gl < 6 && gl > mm) s -= drow[mm] * ym;
        }
      } else {
#pragma unroll
        for (int mm = 5; mm >= 0; mm--) {
          if (gl == mm) s *= dinv;
          const T ym = bcast(s, mm);
          if (gl < 6 && gl < mm) s -= drow[mm] * ym;
        }
      }
      if (live && gl < 6) store_value(x + 6 * (size_t)i + gl, s);
      if (kUseCache) {
        cid = i;
#pragma unroll
        for (int c = 0; c < 6; c++) cx[c] = read_lane(s, c);
      }
    }
    tk = __shfl(tn, 0, 64);
  }
}

// ---- both sweeps of a small system in one workgroup ----
// A level of the kernels above costs a trip through memory from one CU to
// another, and a small system has little else.  Here one workgroup takes the
// whole pair: the solution stays in LDS, a level ends at a barrier, and a
// wavefront takes every sixteenth row in level order and keeps the blocks of
// its next rows in flight, so that what follows a barrier is the
// dependencies' entries from LDS, their products, three adds across eight
// lanes and the 6 x 6 triangle.  Lane 8 r + t (r < 6) takes scalar row r of
// the row's block t.  No sentinel: tmp is not used.
// What bounds it: the chain of a level (0.5 us) in the smallest systems,
// then one CU's loads (0.08 us a row and sweep).  Natural-order ILU(0) of a
// 10x10 plate (31 levels a sweep), FP64: sentinel, L and U kernels 4 + 36 +
// 38 us, so 36 us.  16 wavefronts with 3 rows each in flight, 8 with 5: the
// same at 121 rows, 120 and 133 us at 625; one row in flight is no slower at
// 121 rows.
constexpr int kSmallThreads = 1024;
constexpr int kSmallBlocks = 8;  // blocks of a row on either side, at most
constexpr int kSmallRing = 3;    // rows of a wavefront whose blocks are in flight

// Sum over eight consecutive lanes, in each of them.
template <int kCtrl, typename T>
__device__ __forceinline__ T dpp_move(T v) {
  if constexpr (sizeof(T) == 4) {
    return __builtin_bit_cast(
        T, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), kCtrl, 0xf,
                                    0xf, true));
  } else {
    const long long b = __builtin_bit_cast(long long, v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, kCtrl, 0xf, 0xf, true);
    const int hi =
        __builtin_amdgcn_mov_dpp((int)(b >> 32), kCtrl, 0xf, 0xf, true);
    return __builtin_bit_cast(T, ((long long)hi << 32) | (unsigned)lo);
  }
}
template <typename T>
__device__ __forceinline__ T sum8(T v) {
  v += dpp_move<0xb1>(v);           // lanes 1 0 3 2
  v += dpp_move<0x4e>(v);           // lanes 2 3 0 1
  return v + dpp_move<0x141>(v);    // lanes 7 .. 0 of each eight
}

// A barrier for data in LDS alone: __syncthreads also waits for the loads
// and stores that the wavefront has in flight to memory.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ int4 uniform(int4 v) {
  return make_int4(__builtin_amdgcn_readfirstlane(v.x),
                   __builtin_amdgcn_readfirstlane(v.y),
                   __builtin_amdgcn_readfirstlane(v.z),
                   __builtin_amdgcn_readfirstlane(v.w));
}

template <typename T, bool kLower>
__device__ __forceinline__ void small_sweep(const SweepSlot<T>& S, int nlev,
                                            T* xs) {
  const int4* __restrict__ meta = kLower ? S.lmeta : S.umeta;
  const int* __restrict__ cols = S.cols;
  const T* __restrict__ lu = S.lu;
  constexpr int R = kSmallRing, nw = kSmallThreads / 64;
  const int lane = threadIdx.x % 64;
  const int r = lane >> 3, t = lane & 7, rr = r < 6 ? r : 5;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  constexpr int kNone = 0x7fffffff;  // level of no row
  // the ring: rows w + nw (R k + s) of the level order in slot s, their
  // descriptors (m: of the row held, mv: of the next row, not yet waited for),
  // blocks, diagonal blocks and right-hand sides
  int4 m[R], mv[R];
  T a[R][6], d[R][6], b[R];
  int col[R];
  auto fetch = [&](int p) {
    return p < S.n ? meta[p] : make_int4(0, 0, 0, kNone);
  };
  // lanes without a block of the row load nothing and what they hold is
  // dropped; lane 8 r alone has row r of the diagonal block
  auto load = [&](int s) {
    if (m[s].w == kNone) return;
    const int di = kLower ? m[s].z : m[s].y - 1;
    const int q = m[s].y + t;
    if (r < 6 && q < m[s].z) {
      col[s] = cols[q];
      const T* ap = lu + 36 * (size_t)q + 6 * r;
#pragma unroll
      for (int c = 0; c < 6; c++) a[s][c] = ap[c];
    }
    if (r < 6 && t == 0) {
      const T* dp = lu + 36 * (size_t)di + 6 * r;
#pragma unroll
      for (int c = 0; c < 6; c++) d[s][c] = dp[c];
      if constexpr (kLower) b[s] = S.b[6 * (size_t)m[s].x + r];
    }
  };
#pragma unroll
  for (int s = 0; s < R; s++) mv[s] = fetch(w + nw * s);
#pragma unroll
  for (int s = 0; s < R; s++) {
    m[s] = uniform(mv[s]);
    load(s);
    mv[s] = fetch(w + nw * (R + s));
  }
  int lev = 0, next = w + nw * 2 * R;
  for (;;) {
#pragma unroll
    for (int s = 0; s < R; s++) {
      const int4 mm = m[s];
      if (mm.w == kNone) goto done;
      for (; lev < mm.w; lev++) lds_barrier();
      T v = kLower ? b[s] : xs[6 * mm.x + rr], dinv = T(0);
      T acc = T(0);
      if (r < 6 && mm.y + t < mm.z) {
        const T* xv = xs + 6 * col[s];
#pragma unroll
        for (int c = 0; c < 6; c++) acc += a[s][c] * xv[c];
      }
      if constexpr (!kLower) {
        T dd = d[s][0];
#pragma unroll
        for (int c = 1; c < 6; c++) dd = rr == c ? d[s][c] : dd;
        dinv = T(1) / dd;
      }
      v -= sum8(acc);
      if constexpr (kLower) {
#pragma unroll
        for (int c = 0; c < 5; c++) {
          const T y = read_lane(v, 8 * c);
          v = r > c ? v - d[s][c] * y : v;
        }
      } else {
#pragma unroll
        for (int c = 5; c >= 0; c--) {
          v = r == c ? v * dinv : v;
          const T y = read_lane(v, 8 * c);
          v = r < c ? v - d[s][c] * y : v;
        }
      }
      if (r < 6 && t == 0) {
        xs[6 * mm.x + r] = v;
        if constexpr (!kLower) S.x[6 * (size_t)mm.x + r] = v;
      }
      m[s] = uniform(mv[s]);
      load(s);
      mv[s] = fetch(next);
      next += nw;
    }
  }
done:
  for (; lev < nlev; lev++) lds_barrier();
}

// kBatched: workgroup k takes system k of the slots, if it is a small one.
template <typename T, bool kBatched>
__global__ void __launch_bounds__(kSmallThreads)
    trsv_small_kernel(SweepSlot<T> one, const SweepSlot<T>* __restrict__ slots) {
  extern __shared__ __align__(16) unsigned char small_lds[];
  T* xs = reinterpret_cast<T*>(small_lds);
  const SweepSlot<T> S = kBatched ? slots[blockIdx.x] : one;
  if (kBatched && (S.nllev == 0 || *S.go != 1)) return;
  small_sweep<T, true>(S, S.nllev, xs);
  small_sweep<T, false>(S, S.nulev, xs);
}

// Neither infinite nor NaN.  Sweep pair of a 256x256 plate, RCM ILU(3), with
// the check in front of a group's stores, integer comparison / v_cmp_class /
// no check: FP64 2.41 / 2.44 / 2.37 ms, FP32 2.53 / 2.46 / 2.43 ms.
__device__ __forceinline__ bool finite(double v) {
  const unsigned hi =
      (unsigned)(__builtin_bit_cast(unsigned long long, v) >> 32);
  return hi << 1 < 0xffe00000u;
}
__device__ __forceinline__ bool finite(float v) {
  return !__builtin_amdgcn_classf(v, 0x207);
}

// ---- sweeps over row groups ----
// A level of a few rows costs a row's whole latency, from a dependency's
// store to the row's own (1.2 us on an idle device, 1.6-2.1 us under load).
// Most of the rows of the narrow levels are chains: row i's first U column
// is its parent row, which depends on it.  Up to kGroupRows rows of such a
// chain form a group, solved by one workgroup: wavefront p sums the external
// dependencies (rows outside the group) of row p as trsv_syncfree_kernel
// does, and the last wavefront then solves the rows one after another in
// registers, lane 6p + a holding scalar row a of row p, so that a dependency
// inside a group costs six v_readlane/fma steps (0.1 us) instead of a round
// trip through memory.  Each row's entries are stored as soon as the row is
// solved.  Fewer rows than wavefronts: each row gets several.
// What bounds it now: 2.5-3 us a group level (0.9 us from the last store to
// its being seen, 0.5 us for the pass, 0.4 us to the solver, 0.7-1 us the
// chain), and in the wide levels the 5-9 us latency of a record at two
// workgroups a CU.  L+U pair, row by row -> groups: 400x400 plate AMD +
// ILU(96) (1,372 row levels, 181 group levels) FP64 5.15 -> 2.17 ms, FP32
// 4.88 -> 1.96 ms; 101x101 ILU(64) FP64 1.77 -> 0.50 ms; 45x45 ILU(64)
// 0.79 -> 0.23 ms; complete LU of a 24,390-node wingbox (3,876 -> 489
// levels) 10.5 -> 2.65 ms.
//
// Group record (kGroupInts ints, rows in solve order): [0] rows n,
// [8 + p] row, [16 + p], [24 + p] its dependency blocks [k0, k1) (internal
// ones included: their columns are skipped), [32 + 8 p + q] block index of
// (row p, row q) for q < p, of the diagonal block for q == p, -1 for none.
constexpr int kGroupRows = 8;
constexpr int kGroupInts = 96;
constexpr int kGroupThreads = 64 * kGroupRows;
constexpr int kGroupNear = 16;  // blocks next to the diagonal, last pass
// Groups are used for patterns with at least kGroupRatio row levels per group
// level: a group level costs 2.5-3 us, a row level 1.2-1.6 us.  FP64 pair row
// by row / in groups on a 256x256 plate: natural ILU(0) (ratio 1.4) 1.88 /
// 2.44 ms, AMD ILU(0) (0.2) 0.41 / 0.60 ms, AMD ILU(3) (5.6) 0.75 / 0.58 ms,
// RCM ILU(3) (5.0) 5.9 / 2.3 ms; RCM ILU(3) of a wingbox (1.6) 7.1 / 6.0 ms.
constexpr double kGroupRatio = 1.5;
// records of a sweep at most, a bound of their memory (416 bytes each with its
// rows): a pattern that would need more is swept row by row
inline size_t group_records_max(size_t n) { return n / 4 + 64; }
// kBatched: the groups of several systems, merged[q] = {system, group}; the
// arrays of a system are in its slot.
template <typename T, bool kLower, bool kBatched = false>
__global__ void __launch_bounds__(kGroupThreads, 4)
    trsv_group_kernel(const int* __restrict__ groups, int ngroups,
                      const int* __restrict__ cols_, const T* __restrict__ lu_,
                      const T* b_, T* x_, T* fill_next_,
                      unsigned long long* counter, unsigned long long base,
                      int* err,
                      const SweepSlot<T>* __restrict__ slots = nullptr,
                      const int2* __restrict__ merged = nullptr) {
  using B = typename Sentinel<T>::Bits;
  const int* __restrict__ cols = cols_;
  const T* __restrict__ lu = lu_;
  const T* b = b_;
  T* x = x_;
  T* fill_next = fill_next_;
  // batches of ten blocks whose values a pass holds in registers, blocks of a
  // pass, dependency entries per lane.  Two workgroups a CU take at most 128
  // registers: 400x400 plate, FP64 pair 2.15 ms with 2 batches, 2.19 ms with
  // 3 (which spill), 2.25 / 2.31 ms with 4 / 6 and one workgroup a CU.
  constexpr int kIter = sizeof(T) == 8 ? 2 : 4;
  constexpr int kPass = 10 * kIter;
  constexpr int kE = (6 * kPass + 63) / 64;
  __shared__ T xs_all[kGroupRows][kPass][6];
  __shared__ T ext[kGroupRows][60];    // external sums of a wavefront's slots
  __shared__ T coef[6 * kGroupRows][6 * kGroupRows];  // [column][scalar row]
  __shared__ T diag[6 * kGroupRows];   // U: diagonal entries
  // of a row: bit q: block (row, row q) exists; row; dependency blocks
  __shared__ int4 info[kGroupRows];
  // group count for which a wavefront has written its coefficients, its sums
  __shared__ int staged[kGroupRows], arrived[kGroupRows];
  __shared__ int s_ticket;
  const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
  const int t = lane / 6, r = lane % 6;
  const bool act = lane < 60;
  if (threadIdx.x < kGroupRows)
    staged[threadIdx.x] = arrived[threadIdx.x] = 0;
  // A workgroup holds the ticket of its next group while it works on one,
  // and every wavefront has the next record in two registers by then (lane l:
  // ints l and 64 + l), so that neither round trip is waited for.
  auto ticket = [&]() {  // thread 0: a group, or -1 once there is none left
    const long long q = (long long)(atomicAdd(counter, 1ull) - base);
    return q >= 0 && q < ngroups ? (int)q : -1;
  };
  int ra = 0, rb = 0, next_sys = 0;
  auto load_record = [&](int g) {
    const int* rec;
    if constexpr (kBatched) {
      const int2 mg = merged[g];
      next_sys = mg.x;
      rec = (kLower ? slots[mg.x].lgroup : slots[mg.x].ugroup) +
            (size_t)kGroupInts * mg.y;
    } else {
      rec = groups + (size_t)kGroupInts * g;
    }
    ra = rec[lane];
    rb = lane < kGroupInts - 64 ? rec[64 + lane] : -1;
  };
  int tk = -1;  // thread 0: the ticket after the one in s_ticket
  if (threadIdx.x == 0) {
    s_ticket = ticket();
    if (s_ticket >= 0) tk = ticket();
  }
  __syncthreads();
  int g = s_ticket;
  if (g >= 0) load_record(g);
  __syncthreads();
  for (int seq = 1; g >= 0; seq++) {
    const int rec0 = ra, rec1 = rb, sys = next_sys;
    if (threadIdx.x == 0) s_ticket = tk;
    __syncthreads();
    g = s_ticket;  // the next group
    if (g >= 0) {
      if (threadIdx.x == 0) tk = ticket();
      load_record(g);
    }
    // rows of the group; none where this system takes no step now
    int n = __builtin_amdgcn_readlane(rec0, 0);
    if constexpr (kBatched) {
      const SweepSlot<T>& S = slots[sys];
      if (*S.go != 1) n = 0;
      cols = S.cols;
      lu = S.lu;
      b = kLower ? S.b : S.tmp;
      x = kLower ? S.tmp : S.x;
      fill_next = kLower ? S.x : nullptr;
    }
    if (n > 0) {
      const int p = w % n, part = w / n;
      const int nparts = (kGroupRows - p + n - 1) / n;
      int mem[kGroupRows];  // the group's rows: internal dependencies
#pragma unroll
      for (int q = 0; q < kGroupRows; q++)
        mem[q] = q < n ? __builtin_amdgcn_readlane(rec0, 8 + q) : -1;
      const int k0 = __builtin_amdgcn_readlane(rec0, 16 + p);
      const int k1 = __builtin_amdgcn_readlane(rec0, 24 + p);
      const bool solver = w == kGroupRows - 1;
      // the solver's lane 6 p + a is scalar row a of the group's row p
      const int sp = lane / 6, sa = lane % 6;
      const bool live = solver && lane < 6 * n;
      int srow = 0;
      T s = T(0);
      if (solver) {
        srow = __shfl(rec0, live ? 8 + sp : 8, 64);
        if (live) s = b[6 * (size_t)srow + sa];
        if (kLower && fill_next && live)
          reinterpret_cast<B*>(fill_next)[6 * (size_t)srow + sa] =
              Sentinel<T>::value;
      }
      // coefficients of row p for the solver: the internal blocks (p, q),
      // q < p, and the strict triangle of the diagonal block, one LDS row per
      // scalar column
      if (part == 0) {
        T v[5];
        int at[5];
#pragma unroll
        for (int z = 0; z < 5; z++) {
          const int e = 64 * z + lane, q = e / 36;
          const int i = 32 + 8 * p + (q < 8 ? q : 7);
          const int b0 = __shfl(rec0, i & 63, 64),
                    b1 = __shfl(rec1, i & 63, 64);
          const int bi = q <= p ? (i < 64 ? b0 : b1) : -1;
          v[z] = bi >= 0 ? lu[36 * (size_t)bi + e % 36] : T(0);
          at[z] = q;
        }
#pragma unroll
        for (int z = 0; z < 5; z++) {
          const int q = at[z], rc = (64 * z + lane) % 36, a = rc / 6,
                    c = rc % 6;
          if (q >= kGroupRows) continue;
          if (q == p && a == c) diag[6 * p + a] = v[z];
          if (q == p && (kLower ? c >= a : c <= a)) v[z] = T(0);
          coef[6 * q + c][6 * p + a] = v[z];
        }
        const int i = 32 + 8 * p + lane % 8;
        const int b0 = __shfl(rec0, i & 63, 64), b1 = __shfl(rec1, i & 63, 64);
        const unsigned blocks = (unsigned)__ballot((i < 64 ? b0 : b1) >= 0);
        const int row = __builtin_amdgcn_readlane(rec0, 8 + p);
        if (lane == 0) info[p] = make_int4(blocks & 255, row, k0, k1);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        if (lane == 0)
          __hip_atomic_store(&staged[w], seq, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      // the solver forms its reciprocal diagonal before the waits
      const int lc = lane < 6 * kGroupRows ? lane : 0;
      T dinv = T(1);
      if (solver) {
        // every row's coefficients (wavefronts 0 .. n - 1)
        for (;;) {
          const int v = lane < n
                            ? __hip_atomic_load(&staged[lane], __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_WORKGROUP)
                            : seq;
          if (!__any(v != seq)) break;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        if (!kLower && live) dinv = T(1) / diag[lc];
        asm volatile("" : "+v"(dinv), "+v"(s));
      }
      T(&xs)[kPass][6] = xs_all[w];
      T acc = T(0);
      const int nb = k1 - k0;
      // passes as in trsv_syncfree_kernel: the blocks next to the diagonal
      // last, the others in passes of kPass, all dealt out over the parts, U
      // rows taking theirs last to first
      const bool split = nb > kPass;
      const int nfar = split ? nb - kGroupNear : nb;
      const int nfp = (nfar + kPass - 1) / kPass;
      const int npass = nfp + (split ? 1 : 0);
      for (int pi = part; pi < npass; pi += nparts) {
        int g0b, ng;
        const int j = kLower ? pi : nfp - 1 - pi;
        if (pi == nfp) {
          g0b = kLower ? k1 - kGroupNear : k0;
          ng = kGroupNear;
        } else {
          const int fb = kLower ? k0 : k0 + (split ? kGroupNear : 0);
          const int fe = kLower ? (split ? k1 - kGroupNear : k1) : k1;
          g0b = fb + j * kPass;
          ng = max(0, min(kPass, fe - g0b));
        }
        T a[kIter][6];
#pragma unroll
        for (int it = 0; it < kIter; it++) {
          const int q = 10 * it + t;
          const bool ok = act && q < ng;
          const T* ap = lu + 36 * (size_t)(ok ? g0b + q : 0) + 6 * r;
#pragma unroll
          for (int c = 0; c < 6; c++) a[it][c] = ok ? ap[c] : T(0);
        }
        int jj[kE];
        B xb[kE];
#pragma unroll
        for (int k = 0; k < kE; k++) {
          const int q = (lane + 64 * k) / 6;
          int j2 = q < ng ? cols[g0b + q] : -1;
#pragma unroll
          for (int u = 0; u < kGroupRows; u++) j2 = j2 == mem[u] ? -1 : j2;
          jj[k] = j2;
        }
#pragma unroll
        for (int k = 0; k < kE; k++)
          xb[k] = jj[k] >= 0
                      ? load_bits(x + 6 * (size_t)jj[k] + (lane + 64 * k) % 6)
                      : B(0);
        unsigned spins = 0;
        int nap = 1;
        for (;;) {
          bool pending = false;
#pragma unroll
          for (int k = 0; k < kE; k++)
            pending |= xb[k] == Sentinel<T>::value;
          if (!__any(pending)) break;
          if (++spins > kSpinLimit) {
            if (lane == 0)
              __hip_atomic_store(err, 1, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int k = 0; k < kE; k++)
              if (xb[k] == Sentinel<T>::value) xb[k] = B(0);
            break;
          }
          for (int z = 0; z < nap; z++) __builtin_amdgcn_s_sleep(1);
          nap = nap * 2 > GPUFEM_SWEEP_BACKOFF ? GPUFEM_SWEEP_BACKOFF : nap * 2;
#pragma unroll
          for (int k = 0; k < kE; k++)
            if (xb[k] == Sentinel<T>::value)
              xb[k] = load_bits(x + 6 * (size_t)jj[k] + (lane + 64 * k) % 6);
        }
#pragma unroll
        for (int k = 0; k < kE; k++) {
          const int q = (lane + 64 * k) / 6;
          if (q < ng) xs[q][(lane + 64 * k) % 6] = __builtin_bit_cast(T, xb[k]);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int it = 0; it < kIter; it++) {
          const int q = 10 * it + t;
          if (act && q < ng) {
#pragma unroll
            for (int c = 0; c < 6; c++) acc += a[it][c] * xs[q][c];
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
      // the ten slots' sums go to the solver
      if (act) ext[w][lane] = acc;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      if (lane == 0)
        __hip_atomic_store(&arrived[w], seq, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
      if (solver) {
        T cf[2][6];  // coefficients of this row's columns and the next row's
#pragma unroll
        for (int m = 0; m < 6; m++) cf[0][m] = coef[m][lc];
        // the wavefronts p, p + n, ... sum row p: their sums are added in that
        // order, once all of them have arrived, and subtracted when row p's turn
        // comes (the result does not depend on the order of arrival)
        unsigned mine = 0;
        for (int u = sp; u < kGroupRows; u += n) mine |= 1u << u;
        bool taken = !live;
        T es = T(0);  // external sum of this lane's row
        const T s0 = s;
        unsigned arr = 0;  // wavefronts seen to have arrived
#pragma unroll
        for (int q = 0; q < kGroupRows; q++) {
          if (q < n) {
            unsigned need = 0;
            for (int u = q; u < kGroupRows; u += n) need |= 1u << u;
            while ((arr & need) != need) {
              const int v = lane < kGroupRows
                                ? __hip_atomic_load(&arrived[lane],
                                                    __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_WORKGROUP)
                                : 0;
              const unsigned now = (unsigned)__ballot(v == seq);
              if (now == arr) continue;
              arr = now;
              __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
              if (!taken && (arr & mine) == mine) {
                taken = true;
                for (int u = sp; u < kGroupRows; u += n) {
                  T e[10];
#pragma unroll
                  for (int z = 0; z < 10; z++) e[z] = ext[u][6 * z + sa];
#pragma unroll
                  for (int z = 0; z < 10; z++) es += e[z];
                }
              }
            }
            if (q + 1 < kGroupRows)
#pragma unroll
              for (int m = 0; m < 6; m++)
                cf[(q + 1) & 1][m] = coef[6 * (q + 1) + m][lc];
            s -= sp == q ? es : T(0);
            // L: unit diagonal.  U: x = s / diagonal (a lane's s is final once
            // its own step is reached)
#pragma unroll
            for (int z = 0; z < 6; z++) {
              const int m = kLower ? z : 5 - z;
              const T y = read_lane(kLower ? s : s * dinv, 6 * q + m);
              s -= cf[q & 1][m] * y;
            }
            // Blocks that do not exist, the other triangle and the group's
            // own blocks in the external sums are products with a zero, NaN
            // where the other factor is infinite or NaN: a finite value is
            // right, the others are formed again below.
            const T v = kLower ? s : s * dinv;
            if (sp == q && finite(v))
              store_value(x + 6 * (size_t)srow + sa, v);
          }
        }
        const bool odd = live && !finite(kLower ? s : s * dinv);
        if (__any(odd)) {
          // the record once more, without products that are not in the sums
          const int lr = live ? sp : 0;
          const int4 in = info[lr];
          if (live && !finite(es)) {
            bool inf = false;  // in a coefficient of the group's own blocks
            for (int c = 0; c < 6 * lr; c++) inf |= !finite(coef[c][lc]);
            if (inf) {
              es = T(0);
              for (int k = in.z; k < in.w; k++) {
                const int j = cols[k];
                bool own = false;
                for (int u = 0; u < n; u++) own |= j == info[u].y;
                for (int c = 0; c < 6 && !own; c++)
                  es += lu[36 * (size_t)k + 6 * sa + c] *
                        __builtin_bit_cast(T, load_bits(x + 6 * (size_t)j + c));
              }
            }
          }
          s = s0 - es;
#pragma unroll 1
          for (int q = 0; q < n; q++) {
            const bool below = sp > q && (in.x >> q & 1);
#pragma unroll 1
            for (int z = 0; z < 6; z++) {
              const int m = kLower ? z : 5 - z;
              const T y = read_lane(kLower ? s : s * dinv, 6 * q + m);
              const bool tri = sp == q && (kLower ? sa > m : sa < m);
              if (live && (below || tri)) s -= coef[6 * q + m][lc] * y;
            }
          }
          if (odd)
            store_value(x + 6 * (size_t)srow + sa, kLower ? s : s * dinv);
        }
      }
    }
    __syncthreads();  // s_ticket and the LDS buffers are rewritten next
  }
}

// The records of a sweep's groups from their rows, a wavefront each: lane
// 8 p + q looks row q up in row p's blocks.  (Analysis of a 256x256 plate, RCM
// ILU(3), with the records formed on the host and uploaded: 4.3 ms, so 2.1.)
__global__ void __launch_bounds__(256)
    group_records_kernel(int nrec, bool lower, const int* __restrict__ rows,
                         const int* __restrict__ rowp,
                         const int* __restrict__ cols,
                         const int* __restrict__ diag, int* records) {
  const int r = (int)(blockIdx.x * 256 + threadIdx.x) / 64;
  const int lane = threadIdx.x % 64, p = lane / 8, q = lane % 8;
  if (r >= nrec) return;
  const int i = rows[kGroupRows * (size_t)r + p];
  const int j = rows[kGroupRows * (size_t)r + q];
  int k0 = -1, k1 = -1, blk = -1;
  if (i >= 0) {
    const int d = diag[i];
    k0 = lower ? rowp[i] : d + 1;
    k1 = lower ? d : rowp[i + 1];
    if (q == p) {
      blk = d;
    } else if (q < p) {
      int lo = k0, hi = k1;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (cols[mid] < j)
          lo = mid + 1;
        else
          hi = mid;
      }
      if (lo < k1 && cols[lo] == j) blk = lo;
    }
  }
  const int n = __popcll(__ballot(i >= 0)) / 8;
  int* const rec = records + kGroupInts * (size_t)r;
  rec[32 + lane] = blk;
  if (q < 4)
    rec[8 * q + p] = q == 0 ? (p == 0 ? n : -1) : q == 1 ? i : q == 2 ? k0 : k1;
}

// Row groups of a pattern (host).  A row joins the group of the child whose
// first U column it is (the child latest in level order, when it has
// several), as long as the group stays free of cycles: no row outside the
// group with an index below the joining row may depend on a member, or be a
// dependency of a member in the U sweep.  Then ordering the groups by their
// last row is a valid order of both sweeps.
struct SweepGroup {
  int n = 0;            // rows
  int row[kGroupRows];  // ascending
};
struct SweepGroups {
  std::vector<SweepGroup> g;
  std::vector<int> gid;    // group of a row
  std::vector<int> llev;   // group level of the lower sweep
  int nllev = 0;
  std::vector<int> order;  // groups by last row
};
// The groups, and each row's level in the lower sweep (lev, returned: their
// number).  One pass over the L part: the group levels are kept per row, with
// the rows of row i's own group at -1 meanwhile, so that an entry costs two
// loads and a store (400x400 plate, AMD + ILU(96), one core: 14 ms; 23 with
// the levels first and the group of every entry looked up).
int sweep_groups(int n, const int* rowp, const int* cols, const int* diag,
                 SweepGroups& sg, std::vector<int>& levels) {
  levels.assign(n, 0);
  sg.gid.assign(n, -1);
  sg.g.clear();
  sg.g.reserve(n / 2 + 1);
  sg.llev.clear();
  sg.llev.reserve(n / 2 + 1);
  sg.nllev = 0;
  // child of which a row is the first U column; group level of a row; U
  // blocks of a row up to here are known to be in its group; a row outside
  // the group depends on the row
  std::vector<int> best_(n, -1), glev_(n), next_(n);
  std::vector<unsigned char> used_(n, 0);
  int *lev = levels.data(), *gid = sg.gid.data(), *best = best_.data(),
      *glev = glev_.data(), *next = next_.data();
  unsigned char* used = used_.data();
  int nlev = 0;
  for (int i = 0; i < n; i++) {
    const int c = best[i], d = diag[i];
    int g = -1;
    if (c >= 0) {
      g = gid[c];
      const SweepGroup& m = sg.g[g];
      bool ok = m.n < kGroupRows && m.row[m.n - 1] == c;
      if (c < i - 1) {  // (no row between them otherwise)
        for (int q = 0; ok && q < m.n; q++) ok = !used[m.row[q]];
        for (int q = 0; ok && q < m.n; q++) {
          const int r = m.row[q], k1 = rowp[r + 1];
          int k = next[r];
          while (k < k1 && cols[k] < i && gid[cols[k]] == g) k++;
          next[r] = k;
          ok = k == k1 || cols[k] >= i;
        }
      }
      if (!ok) g = -1;
    }
    if (g < 0) {
      g = (int)sg.g.size();
      sg.g.emplace_back();
      sg.llev.push_back(0);
    }
    SweepGroup& m = sg.g[g];
    // the groups this row depends on take no more rows, so their levels are
    // final
    int l = 0, gl = -1, k = rowp[i];
    const int first = m.n ? m.row[0] : i;
    for (; k < d && cols[k] < first; k++) {
      const int j = cols[k];
      l = std::max(l, lev[j] + 1);
      gl = std::max(gl, glev[j]);
      used[j] = 1;
    }
    for (; k < d; k++) {  // its own group's rows among others
      const int j = cols[k];
      l = std::max(l, lev[j] + 1);
      if (gid[j] == g) continue;
      gl = std::max(gl, glev[j]);
      used[j] = 1;
    }
    lev[i] = l;
    gid[i] = g;
    next[i] = d + 1;
    m.row[m.n++] = i;
    glev[i] = sg.llev[g];
    if (gl + 1 > sg.llev[g]) {
      sg.llev[g] = gl + 1;
      for (int q = 0; q < m.n; q++) glev[m.row[q]] = gl + 1;
    }
    sg.nllev = std::max(sg.nllev, sg.llev[g] + 1);
    nlev = std::max(nlev, l + 1);
    if (d + 1 < rowp[i + 1]) {
      const int j = cols[d + 1];
      if (best[j] < 0 || l >= lev[best[j]]) best[j] = i;
    }
  }
  sg.order.clear();
  sg.order.reserve(sg.g.size());
  for (int i = 0; i < n; i++) {
    const SweepGroup& m = sg.g[gid[i]];
    if (m.row[m.n - 1] == i) sg.order.push_back(gid[i]);
  }
  return nlev;
}

// Group levels of the upper sweep; returns their number.
int upper_group_levels(const int* rowp, const int* cols, const int* diag,
                       const SweepGroups& sg, std::vector<int>& lev) {
  std::vector<int> glev(sg.gid.size(), -1);  // of a row
  lev.assign(sg.g.size(), 0);
  int nlev = 0;
  for (size_t q = sg.order.size(); q-- > 0;) {
    const SweepGroup& m = sg.g[sg.order[q]];
    int l = -1;
    for (int z = 0; z < m.n; z++)
      for (int k = diag[m.row[z]] + 1; k < rowp[m.row[z] + 1]; k++)
        l = std::max(l, glev[cols[k]]);
    l++;
    for (int z = 0; z < m.n; z++) glev[m.row[z]] = l;
    lev[sg.order[q]] = l;
    nlev = std::max(nlev, l + 1);
  }
  return nlev;
}

// Rows of the group records of one sweep, kGroupRows each (-1: none), in
// hand-out order (by group level).
// lev, nlev: the groups' levels; level: the level of each record.
void group_rows(const SweepGroups& sg, bool lower, const std::vector<int>& lev,
                int nlev, std::vector<int>& out, std::vector<int>& level) {
  const int ng = (int)sg.g.size();
  std::vector<int> ptr(nlev + 1, 0);
  for (int g = 0; g < ng; g++) ptr[lev[g] + 1]++;
  for (int l = 0; l < nlev; l++) ptr[l + 1] += ptr[l];
  std::vector<int> order(ng);
  for (int q = 0; q < ng; q++) {
    const int g = sg.order[lower ? q : ng - 1 - q];
    order[ptr[lev[g]]++] = g;  // ptr[l] moves to the end of level l
  }
  // Groups of one level share a record as long as it holds their rows: the
  // largest group left, then the largest that still fit.
  out.clear();
  out.reserve(sg.gid.size() + sg.gid.size() / 2 + 64);
  level.clear();
  std::vector<int> bySize[kGroupRows + 1];
  for (int l = 0, q0 = 0; l < nlev; q0 = ptr[l++]) {
    for (int q = ptr[l] - 1; q >= q0; q--)
      bySize[sg.g[order[q]].n].push_back(order[q]);
    for (;;) {
      int used = 0;
      for (int sz = kGroupRows; sz > 0;) {
        if (sz > kGroupRows - used || bySize[sz].empty()) {
          sz--;
          continue;
        }
        const int* row = sg.g[bySize[sz].back()].row;
        bySize[sz].pop_back();
        if (!used) level.push_back(l);
        for (int z = 0; z < sz; z++)
          out.push_back(row[lower ? z : sz - 1 - z]);
        used += sz;
      }
      if (!used) break;
      out.resize(out.size() + (kGroupRows - used), -1);
    }
  }
}

}  // namespace

// Which systems trsv_small_kernel sweeps: those whose rows fit its lanes
// (kSmallBlocks a side) and LDS, with few enough rows a level.  FP64 pair in
// one workgroup / by the kernels of larger systems, with the host's calls:
// plates in natural order, ILU(0), 10x10 (121 rows, 31 levels) 55 / 99 us,
// 24x24 (625, 73) 140 / 198, 35x35 (1,296, 106) 250 / 276; RCM 24x24 (625,
// 96) 152 / 200; AMD 10x10 (121, 14) 45 / 55, 16x16 (289, 18) 68 / 68,
// 32x32 (1,089, 18) 167 / 70.
constexpr int kSmallRows = 1300;  // 6 FP64 values a row in 64 KB of LDS
constexpr int kSmallWidth = 12;   // rows a level, on average
static bool small_sweeps(int n, int nlev) {
  return n <= kSmallRows && n <= kSmallWidth * nlev;
}
size_t ilu_counter_bytes() {
  return sizeof(unsigned long long) * kCounterStride *
         (1 + kSweepThreads / 64);
}
size_t ilu_group_row_bytes(size_t nrec) {
  return sizeof(int) * kGroupRows * nrec;
}
size_t ilu_group_bytes(size_t nrec) { return sizeof(int) * kGroupInts * nrec; }
// Host analysis of a pattern: its levels, and how the sweeps run.
int ilu_plan(int n, const int* rowp, const int* cols, IluPlan& pl,
             std::string* why) {
  auto fail = [&](const std::string& msg) {
    if (why) *why = "ilu_create: " + msg;
    return GF_ERR_INVALID;
  };
  pl = IluPlan{};
  pl.diag.resize(n);
  int maxlen = 0;
  int side = 0;  // most blocks of a row on one side of the diagonal
  for (int i = 0; i < n; i++) {
    const int k0 = rowp[i], k1 = rowp[i + 1];
    bool bad = k1 > k0 && (cols[k0] < 0 || cols[k1 - 1] >= n);
    for (int k = k0 + 1; k < k1; k++) bad |= cols[k] <= cols[k - 1];
    if (bad) return fail("row " + std::to_string(i) + " not sorted/in range");
    const int d = (int)(std::lower_bound(cols + k0, cols + k1, i) - cols);
    if (d >= k1 || cols[d] != i)
      return fail("row " + std::to_string(i) + " has no diagonal block");
    pl.diag[i] = d;
    maxlen = std::max(maxlen, k1 - k0);
    side = std::max({side, d - k0, k1 - d - 1});
  }
  if (maxlen > kMaxRowBlocks)
    return fail("row length " + std::to_string(maxlen) + " exceeds " +
                std::to_string(kMaxRowBlocks) + " blocks");
  pl.max_row_len = maxlen;
  const int* diag = pl.diag.data();
  const char* tenv = getenv("GPUFEM_TRSV");
  const std::string mode = tenv ? tenv : "";
  pl.chains = mode == "chains";
  pl.levels = mode == "level";
  // The levels of the two sweeps of a large pattern are found at the same time
  // (here, one after the other, if the library can start no thread).
  // gf_ilu_create without row groups / with the groups' levels and records
  // found on the host, row by row / now: 400x400 plate, AMD + ILU(96) (14 M
  // blocks) 30.8 / 41.8 / 19.7 ms, 256x256 plate RCM ILU(3) 2.90 / 5.07 /
  // 2.13 ms, 45x45 AMD ILU(12) 0.27 / 0.40 / 0.23 ms.
  const auto policy = rowp[n] >= 200000
                          ? std::launch::async | std::launch::deferred
                          : std::launch::deferred;
  auto upper = std::async(policy, [&] {
    level_schedule(n, rowp, cols, false, pl.uptr, pl.urows);
  });
  // groups: whatever their ratio.  Any value but these: row by row.
  const bool force = mode == "groups";
  const bool small_fits = side <= kSmallBlocks && n <= kSmallRows;
  const bool groups = !tenv || force || mode == "small";
  SweepGroups sg;
  if (groups && (force || !small_fits)) {
    std::vector<int> lev;
    const int nlev = sweep_groups(n, rowp, cols, diag, sg, lev);
    order_levels(n, lev, nlev, true, pl.lptr, pl.lrows);
  } else {
    level_schedule(n, rowp, cols, true, pl.lptr, pl.lrows);
  }
  upper.get();
  pl.lmaxlen.assign(pl.lptr.size() - 1, 0);
  for (size_t l = 0; l + 1 < pl.lptr.size(); l++)
    for (int q = pl.lptr[l]; q < pl.lptr[l + 1]; q++)
      pl.lmaxlen[l] = std::max(
          pl.lmaxlen[l], rowp[pl.lrows[q] + 1] - rowp[pl.lrows[q]]);
  const int nlev = (int)std::max(pl.lptr.size(), pl.uptr.size()) - 1;
  if (small_fits && !force)
    pl.small = mode == "small" || (!tenv && small_sweeps(n, nlev));
  if (!groups || pl.small) return GF_OK;
  if (sg.g.empty()) {
    std::vector<int> lev;
    sweep_groups(n, rowp, cols, diag, sg, lev);
  }
  auto pays = [&](int glev) { return force || kGroupRatio * glev <= nlev; };
  if (!pays(sg.nllev)) return GF_OK;
  std::vector<int> ulev;
  const int nulev = upper_group_levels(rowp, cols, diag, sg, ulev);
  if (!pays(nulev)) return GF_OK;
  group_rows(sg, true, sg.llev, sg.nllev, pl.lgroup, pl.llevel);
  group_rows(sg, false, ulev, nulev, pl.ugroup, pl.ulevel);
  if (std::max(pl.llevel.size(), pl.ulevel.size()) > group_records_max(n))
    for (auto* v : {&pl.lgroup, &pl.ugroup, &pl.llevel, &pl.ulevel})
      v->clear();
  return GF_OK;
}
}  // namespace gf

extern "C" {

int gf_ilu_create(gf_context ctx, int n, const int* rowp, const int* cols,
                  gf_ilu* out) {
  if (!ctx || n <= 0 || !rowp || !cols || !out)
    return gf::set_error(ctx, GF_ERR_INVALID, "ilu_create: bad args");
  gf::IluPlan pl;
  std::string why;
  const int st = gf::ilu_plan(n, rowp, cols, pl, &why);
  if (st != GF_OK) return gf::set_error(ctx, st, "%s", why.c_str());
  return gf::ilu_create_planned(ctx, n, rowp, cols, pl, out);
}

}  // extern "C"

namespace gf {
int ilu_create_planned(gf_context ctx, int n, const int* rowp,
                       const int* cols, IluPlan& pl, gf_ilu* out) {
  auto* h = new gf_ilu_s;
  h->ctx = ctx;
  h->n = n;
  h->nnzb = rowp[n];
  h->max_row_len = pl.max_row_len;
  h->lptr.swap(pl.lptr);
  h->uptr.swap(pl.uptr);
  h->lmaxlen.swap(pl.lmaxlen);
  h->small = pl.small;
  h->level_sweeps = pl.levels;
  const std::vector<int>&diag = pl.diag, &lrows = pl.lrows, &urows = pl.urows;
  // chunks: runs of rows of one level, sized so that a level still spreads
  // over the resident wavefronts (one row per chunk for small levels)
  const int target_waves =
      GPUFEM_SWEEP_WAVES_PER_CU * std::max(ctx->num_cus, 1);
  const char* cenv = getenv("GPUFEM_TRSV_MINCHUNK");
  const int min_chunk = cenv ? std::max(1, atoi(cenv)) : 1;
  auto chunks = [&](const std::vector<int>& lp, std::vector<int>& out) {
    out.assign(1, 0);
    for (size_t l = 0; l + 1 < lp.size(); l++) {
      const int cnt = lp[l + 1] - lp[l];
      const int csz =
          std::max(std::min(min_chunk, (cnt + 63) / 64),
                   std::max(1, std::min(16, cnt / target_waves)));
      for (int a = lp[l]; a < lp[l + 1]; a += csz)
        out.push_back(std::min(a + csz, lp[l + 1]));
    }
  };
  // chains: maximal runs of consecutive rows (in sweep order) where each row
  // depends on the one before it
  auto chains = [&](bool lower, std::vector<int>& out) {
    out.assign(1, 0);
    for (int t = 1; t < n; t++) {
      const int i = lower ? t : n - 1 - t;
      bool dep = false;
      if (lower) {
        for (int k = rowp[i]; k < diag[i]; k++) dep |= cols[k] == i - 1;
      } else {
        for (int k = diag[i] + 1; k < rowp[i + 1]; k++) dep |= cols[k] == i + 1;
      }
      if (!dep) out.push_back(t);
    }
    out.push_back(n);
  };
  // Rows are handed out by level, in chunks of rows of one level.  Handing
  // out whole chains in row order instead (GPUFEM_TRSV=chains; each
  // wavefront forwards a chain's rows in registers) serialises the rows of a
  // chain behind each other's memory latency and measured 1.7x slower on the
  // natural-order plates.
  std::vector<int> lch, uch;
  const bool use_chains = pl.chains;
  h->lchains = h->uchains = use_chains;
  h->nlgroup = (int)pl.llevel.size();
  h->nugroup = (int)pl.ulevel.size();
  if (h->nlgroup) {
    h->llevel.swap(pl.llevel);
    h->ulevel.swap(pl.ulevel);
  } else if (use_chains) {
    chains(true, lch);
    chains(false, uch);
  } else {
    chunks(h->lptr, lch);
    chunks(h->uptr, uch);
    auto levels_of = [](const std::vector<int>& ch, const std::vector<int>& lp,
                        std::vector<int>& out) {
      out.resize(ch.size() - 1);
      size_t l = 0;
      for (size_t c = 0; c + 1 < ch.size(); c++) {
        while (l + 2 < lp.size() && lp[l + 1] <= ch[c]) l++;
        out[c] = (int)l;
      }
    };
    levels_of(lch, h->lptr, h->llevel);
    levels_of(uch, h->uptr, h->ulevel);
  }
  // row descriptors in hand-out order, one 16-byte load per row: {row, first
  // block, end block, level}; the diagonal block is the end (L) or one before the
  // first (U).  Row groups need neither these nor the chunks.
  std::vector<int4> lm, um;
  if (!h->nlgroup) {
    h->nlchunk = (int)lch.size() - 1;
    h->nuchunk = (int)uch.size() - 1;
    lm.resize(n);
    um.resize(n);
    for (int p = 0; p < n; p++) {
      const int li = use_chains ? p : lrows[p];
      lm[p] = make_int4(li, rowp[li], diag[li], 0);
      const int ui = use_chains ? n - 1 - p : urows[p];
      um[p] = make_int4(ui, diag[ui] + 1, rowp[ui + 1], 0);
    }
    auto levels_into = [](const std::vector<int>& lp, std::vector<int4>& mt) {
      for (size_t l = 0; l + 1 < lp.size(); l++)
        for (int p = lp[l]; p < lp[l + 1]; p++) mt[p].w = (int)l;
    };
    if (!use_chains) {
      levels_into(h->lptr, lm);
      levels_into(h->uptr, um);
    }
  }
  // (ProblemPlan::device_bytes mirrors the list; what is empty stays null)
  auto up = [&](int** dst, const int* src, size_t cnt) -> int {
    if (!cnt) return GF_OK;
    GF_TRY(gf::dmalloc(ctx, (void**)dst, sizeof(int) * cnt));
    GF_HIP(ctx, hipMemcpyAsync(*dst, src, sizeof(int) * cnt,
                               hipMemcpyHostToDevice, ctx->stream));
    return GF_OK;
  };
  int st = GF_OK;
  if ((st = up(&h->lgrows, pl.lgroup.data(), pl.lgroup.size())) ||
      (st = up(&h->ugrows, pl.ugroup.data(), pl.ugroup.size())) ||
      (st = up(&h->rowp, rowp, n + 1)) || (st = up(&h->cols, cols, rowp[n])) ||
      (st = up(&h->diag, diag.data(), n)) ||
      (st = up(&h->lrows, lrows.data(), n)) ||
      (st = up(&h->urows, urows.data(), n)) ||
      (st = up(&h->lchunk, lch.data(), lch.size())) ||
      (st = up((int**)&h->lmeta, (const int*)lm.data(), 4 * lm.size())) ||
      (st = up((int**)&h->umeta, (const int*)um.data(), 4 * um.size())) ||
      (st = up(&h->uchunk, uch.data(), uch.size())) ||
      (h->nlgroup &&
       ((st = gf::dmalloc(ctx, (void**)&h->lgroup,
                          ilu_group_bytes(h->nlgroup))) ||
        (st = gf::dmalloc(ctx, (void**)&h->ugroup,
                          ilu_group_bytes(h->nugroup))))) ||
      (st = gf::dmalloc(ctx, (void**)&h->pivot, sizeof(int))) ||
      (st = gf::dmalloc(ctx, (void**)&h->counter, gf::ilu_counter_bytes())) ||
      (st = gf::dmalloc(ctx, (void**)&h->err, 2 * sizeof(int))) ||
      (st = gf::dmalloc(ctx, (void**)&h->done, sizeof(int) * (size_t)n)) ||
      (st = gf::check_hip(ctx, hipMemsetAsync(h->done, 0, sizeof(int) * (size_t)n,
                                              ctx->stream), "memset")) ||
      (st = gf::check_hip(ctx, hipMemsetAsync(h->counter, 0, gf::ilu_counter_bytes(),
                                              ctx->stream), "memset")) ||
      (st = gf::check_hip(ctx, hipMemsetAsync(h->err, 0, 2 * sizeof(int), ctx->stream),
                          "memset"))) {
    gf_ilu_destroy(h);
    return st;
  }
  if (h->nlgroup) {
    auto records = [&](bool lower, int nrec, const int* rows, int* out) {
      hipLaunchKernelGGL(group_records_kernel, dim3(div_up(nrec, 4)), dim3(256),
                         0, ctx->stream, nrec, lower, rows, h->rowp, h->cols,
                         h->diag, out);
    };
    records(true, h->nlgroup, h->lgrows, h->lgroup);
    records(false, h->nugroup, h->ugrows, h->ugroup);
    if ((st = check_launch(ctx, "group_records_kernel"))) {
      gf_ilu_destroy(h);
      return st;
    }
  }
  {
    // enough wavefronts to cover the device, capped by the chunks and by
    // eight mean level widths: wavefronts further ahead than that mostly
    // wait, and on small matrices they would take the device from
    // concurrent solves on other streams
    const int nlev = (int)std::max(h->lptr.size(), h->uptr.size()) - 1;
    const int mean_w = (n + std::max(nlev, 1) - 1) / std::max(nlev, 1);
    const int waves = std::max(
        1, std::min({std::max(h->nlchunk, h->nuchunk), target_waves,
                     std::max(64, 8 * mean_w)}));
    h->grid = (waves + 3) / 4;
    // Workgroups of a group sweep: two a CU where each has dozens of
    // records to take (400x400 plate 2.15 against 2.25 ms a pair), one
    // otherwise (wingbox of 24,390 nodes 2.65 against 2.82 ms), fewer for a
    // small system, which would only wait in them (45x45 plate: 0.25 ms with
    // 64, 128 or 256) and take the device from other streams.
    const int nrec = std::max(h->nlgroup, h->nugroup);
    const int cus = std::max(1, ctx->num_cus);
    h->ggrid = std::min({nrec, nrec >= 32 * cus ? 2 * cus : cus,
                         std::max(64, nrec / 6)});
  }
  st = gf::check_hip(ctx, hipStreamSynchronize(ctx->stream), "ilu upload");
  if (st) {
    gf_ilu_destroy(h);
    return st;
  }
  *out = h;
  return GF_OK;
}
}  // namespace gf

extern "C" {

int gf_ilu_destroy(gf_ilu h) {
  if (!h) return GF_OK;
  gf::dfree(h->ctx, h->rowp);
  gf::dfree(h->ctx, h->cols);
  gf::dfree(h->ctx, h->diag);
  gf::dfree(h->ctx, h->lrows);
  gf::dfree(h->ctx, h->urows);
  gf::dfree(h->ctx, h->pivot);
  gf::dfree(h->ctx, h->lchunk);
  gf::dfree(h->ctx, h->lmeta);
  gf::dfree(h->ctx, h->umeta);
  gf::dfree(h->ctx, h->lgroup);
  gf::dfree(h->ctx, h->ugroup);
  gf::dfree(h->ctx, h->lgrows);
  gf::dfree(h->ctx, h->ugrows);
  gf::dfree(h->ctx, h->uchunk);
  gf::dfree(h->ctx, h->counter);
  gf::dfree(h->ctx, h->err);
  gf::dfree(h->ctx, h->done);
  delete h;
  return GF_OK;
}

int gf_ilu_info(gf_ilu h, int* nnzb, int* nl, int* nu) {
  if (!h) return GF_ERR_INVALID;
  if (getenv("GPUFEM_ILU_VERBOSE"))
    fprintf(stderr,
            "ilu: n=%d nnzb=%d levels L=%d U=%d %s L=%d %s U=%d\n", h->n,
            h->nnzb, (int)h->lptr.size() - 1, (int)h->uptr.size() - 1,
            h->lchains ? "chains" : "chunks", h->nlchunk,
            h->uchains ? "chains" : "chunks", h->nuchunk);
  if (nnzb) *nnzb = h->nnzb;
  if (nl) *nl = (int)h->lptr.size() - 1;
  if (nu) *nu = (int)h->uptr.size() - 1;
  return GF_OK;
}
int gf_ilu_sweep_info(gf_ilu h, int* kind, int* nlower, int* nupper) {
  if (!h) return GF_ERR_INVALID;
  const bool levels = h->small || h->level_sweeps;
  if (kind)
    *kind = h->small          ? GF_SWEEP_SMALL
            : h->level_sweeps ? GF_SWEEP_LEVELS
            : h->nlgroup      ? GF_SWEEP_GROUPS
            : h->lchains      ? GF_SWEEP_CHAINS
                              : GF_SWEEP_ROWS;
  const auto items = [&](const std::vector<int>& lptr, int groups, int chunks) {
    return levels ? (int)lptr.size() - 1 : groups ? groups : chunks;
  };
  if (nlower) *nlower = items(h->lptr, h->nlgroup, h->nlchunk);
  if (nupper) *nupper = items(h->uptr, h->nugroup, h->nuchunk);
  return GF_OK;
}

const int* gf_ilu_device_rowp(gf_ilu h) { return h ? h->rowp : nullptr; }

int gf_ilu_check(gf_ilu h) {
  if (!h) return GF_ERR_INVALID;
  int e = 0;
  GF_HIP(h->ctx, hipMemcpyAsync(&e, h->err, sizeof(int), hipMemcpyDeviceToHost,
                                h->ctx->stream));
  GF_HIP(h->ctx, hipStreamSynchronize(h->ctx->stream));
  if (e) {
    const int zero = 0;
    hipMemcpyAsync(h->err, &zero, sizeof(int), hipMemcpyHostToDevice,
                   h->ctx->stream);
    hipStreamSynchronize(h->ctx->stream);
    return gf::set_error(h->ctx, GF_ERR_TIMEOUT,
                         "triangular sweep: a dependency wait expired");
  }
  return GF_OK;
}
const int* gf_ilu_device_cols(gf_ilu h) { return h ? h->cols : nullptr; }

}  // extern "C"

namespace gf {
unsigned long long sweep_sentinel_bits(bool fp64) {
  return fp64 ? Sentinel<double>::value : Sentinel<float>::value;
}
int* ilu_sweep_err(gf_ilu h) { return h ? h->err : nullptr; }
gf_context ilu_context(gf_ilu h) { return h ? h->ctx : nullptr; }

int ilu_view(gf_ilu h, IluView* v) {
  if (!h || !v || h->lchains || h->uchains) return GF_ERR_INVALID;
  v->n = h->n;
  v->lmeta = h->lmeta;
  v->umeta = h->umeta;
  v->lchunk = h->lchunk;
  v->uchunk = h->uchunk;
  v->cols = h->cols;
  v->lgroup = h->nlgroup ? h->lgroup : nullptr;
  v->ugroup = h->nlgroup ? h->ugroup : nullptr;
  v->llevel = &h->llevel;
  v->ulevel = &h->ulevel;
  v->grid = h->grid;
  v->nllev = h->small ? (int)h->lptr.size() - 1 : 0;
  v->nulev = h->small ? (int)h->uptr.size() - 1 : 0;
  return GF_OK;
}

__global__ void reset_counters_kernel(unsigned long long* c, int n) {
  if ((int)threadIdx.x < n) c[threadIdx.x] = 0ull;
}

// One L and one U sweep over several systems (see SweepItems): the chunks of
// the systems without row groups, then the groups of the others.  The
// counters are zeroed first by a kernel (no memset: the launches may be
// captured in a graph), so the tickets start at 0 in every replay.
template <typename T>
int launch_batch_sweeps(hipStream_t s, const SweepSlot<T>* slots,
                        const SweepItems& it, int grid, int ggrid,
                        unsigned long long* counters, int* err) {
  hipLaunchKernelGGL(reset_counters_kernel, dim3(1), dim3(64), 0, s, counters,
                     kBatchCounters);
  auto sweep = [&](auto lower) {
    constexpr bool kLower = decltype(lower)::value;
    const int2* items = kLower ? it.l : it.u;
    const int nc = kLower ? it.lc : it.uc, ng = kLower ? it.lg : it.ug;
    unsigned long long* c = counters + (kLower ? 0 : 2);
    if (nc > 0)
      hipLaunchKernelGGL((trsv_syncfree_kernel<T, kLower, 1, true>),
                         dim3(grid), dim3(kSweepThreads), 0, s,
                         (const int4*)nullptr, (const int*)nullptr,
                         (const int*)nullptr, nc, (const T*)nullptr,
                         (const T*)nullptr, (T*)nullptr, (T*)nullptr, c, 0ull,
                         err, slots, items);
    if (ng > 0)
      hipLaunchKernelGGL((trsv_group_kernel<T, kLower, true>),
                         dim3(std::min(ggrid, ng)), dim3(kGroupThreads), 0, s,
                         (const int*)nullptr, ng, (const int*)nullptr,
                         (const T*)nullptr, (const T*)nullptr, (T*)nullptr,
                         (T*)nullptr, c + 1, 0ull, err, slots, items + nc);
  };
  sweep(std::true_type{});
  sweep(std::false_type{});
  if (it.small_rows > 0)
    hipLaunchKernelGGL((trsv_small_kernel<T, true>), dim3(it.nslots),
                       dim3(kSmallThreads), sizeof(T) * 6 * it.small_rows, s,
                       SweepSlot<T>{}, slots);
  return hipGetLastError() == hipSuccess ? GF_OK : GF_ERR_DEVICE;
}
template int launch_batch_sweeps<double>(hipStream_t, const SweepSlot<double>*,
                                         const SweepItems&, int, int,
                                         unsigned long long*, int*);
template int launch_batch_sweeps<float>(hipStream_t, const SweepSlot<float>*,
                                        const SweepItems&, int, int,
                                        unsigned long long*, int*);
}  // namespace gf

namespace {
template <typename T>
int ilu_factor(gf_ilu h, T* vals, int* zero_pivot) {
  if (!h || !vals) return GF_ERR_INVALID;
  gf_context ctx = h->ctx;
  const int big = 0x7fffffff;
  GF_HIP(ctx, hipMemcpyAsync(h->pivot, &big, sizeof(int),
                             hipMemcpyHostToDevice, ctx->stream));
  // rows whose values fit in LDS (dynamic LDS per level: its longest row)
  // are factored there; the other levels run ilu_row_kernel
  static size_t lds_cap[2] = {0, 0}, lds_half[2] = {0, 0};
  static size_t batch_cap[2] = {0, 0}, batch_cap2[2] = {0, 0};
  static std::once_flag once[2];
  const int ti = sizeof(T) == 8 ? 0 : 1;
  std::call_once(once[ti], [&] {
    const void* fns[4] = {
        (const void*)gf::ilu_row_lds_kernel<T, false>,
        (const void*)gf::ilu_row_lds_kernel<T, true>,
        (const void*)gf::ilu_row_lds_kernel<T, true, gf::kIluShortThreads>,
        (const void*)gf::ilu_row_lds_kernel<T, false, gf::kIluShortThreads>};
    hipDeviceProp_t prop{};
    if (hipGetDeviceProperties(&prop, ctx->device) != hipSuccess) return;
    const size_t total = std::min<size_t>(prop.sharedMemPerBlock, 160 * 1024);
    size_t cap = total;
    for (const void* fn : fns) {
      hipFuncAttributes fa{};
      if (hipFuncGetAttributes(&fa, fn) != hipSuccess) return;
      if (total <= fa.sharedSizeBytes + 1024) return;
      cap = std::min(cap, total - fa.sharedSizeBytes);
    }
    for (const void* fn : fns)
      if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)cap) != hipSuccess) {
        hipGetLastError();
        cap = std::min<size_t>(cap, 48 * 1024);
      }
    // the global-memory kernels' column and position lists
    const void* gfns[2] = {(const void*)gf::ilu_row_kernel<T, false>,
                           (const void*)gf::ilu_row_kernel<T, true>};
    for (const void* fn : gfns)
      if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)(3 * sizeof(int) * gf::kMaxRowBlocks)) !=
          hipSuccess)
        hipGetLastError();
    const void* bfns[2] = {(const void*)gf::ilu_row_batch_kernel<T, false>,
                           (const void*)gf::ilu_row_batch_kernel<T, true>};
    size_t bcap = total;
    for (const void* fn : bfns) {
      hipFuncAttributes fa{};
      if (hipFuncGetAttributes(&fa, fn) != hipSuccess ||
          total <= fa.sharedSizeBytes) {
        bcap = 0;
        break;
      }
      bcap = std::min(bcap, total - fa.sharedSizeBytes);
    }
    for (const void* fn : bfns)
      if (bcap > 0 &&
          hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)bcap) != hipSuccess) {
        hipGetLastError();
        bcap = 0;
      }
    batch_cap[ti] = bcap;
    // dynamic LDS that lets two workgroups share a CU
    const size_t stat = total - bcap;
    batch_cap2[ti] = total / 2 > stat ? total / 2 - stat : 0;
    lds_cap[ti] = cap;
    lds_half[ti] = cap > total / 2 ? cap - total / 2 : cap;
  });
  const int maxlen = h->max_row_len;
  const size_t gdyn = 3 * sizeof(int) * (size_t)maxlen;
  const bool no_lds = getenv("GPUFEM_ILU_GLOBAL") != nullptr;
  // rows in global memory: pivots applied in batches (ilu_row_batch_kernel)
  // of as many pivots as the LDS holds position lists for (at most
  // kIluBatch); GPUFEM_ILU_BATCH_N lowers the batch (a test hook), and
  // GPUFEM_ILU_GLOBAL_KERNEL=pivot selects ilu_row_kernel (one pass over the
  // row per pivot)
  int nbatch = 0;
  {
    // two workgroups per CU where the LDS allows
    const size_t cap2 = std::min(batch_cap[ti], batch_cap2[ti]);
    for (int nbt = gf::kIluBatch; nbt >= 1 && !nbatch; nbt--)
      if (gf::batch_lds(nbt, maxlen) <= cap2) nbatch = nbt;
    for (int nbt = gf::kIluBatch; nbt >= 1 && !nbatch; nbt--)
      if (gf::batch_lds(nbt, maxlen) <= batch_cap[ti]) nbatch = nbt;
    if (const char* benv = getenv("GPUFEM_ILU_BATCH_N"))
      nbatch = std::min(nbatch, std::max(1, atoi(benv)));
    const char* kenv = getenv("GPUFEM_ILU_GLOBAL_KERNEL");
    if (kenv && std::string(kenv) == "pivot") nbatch = 0;
  }
  const size_t bdyn = gf::batch_lds(nbatch, maxlen);
  auto launch_global = [&](bool flow, const int* rows, int cnt,
                           const gf::Flow& f) {
    if (nbatch > 0) {
      if (flow)
        hipLaunchKernelGGL((gf::ilu_row_batch_kernel<T, true>), dim3(cnt),
                           dim3(gf::kBatchThreads), bdyn, ctx->stream, rows,
                           cnt, h->rowp, h->cols, h->diag, vals, h->pivot, f,
                           nbatch, maxlen);
      else
        hipLaunchKernelGGL((gf::ilu_row_batch_kernel<T, false>), dim3(cnt),
                           dim3(gf::kBatchThreads), bdyn, ctx->stream, rows,
                           cnt, h->rowp, h->cols, h->diag, vals, h->pivot, f,
                           nbatch, maxlen);
    } else if (flow) {
      hipLaunchKernelGGL((gf::ilu_row_kernel<T, true>), dim3(cnt),
                         dim3(gf::kIluThreads), gdyn, ctx->stream, rows, cnt,
                         h->rowp, h->cols, h->diag, vals, h->pivot, f, maxlen);
    } else {
      hipLaunchKernelGGL((gf::ilu_row_kernel<T, false>), dim3(cnt),
                         dim3(gf::kIluThreads), gdyn, ctx->stream, rows, cnt,
                         h->rowp, h->cols, h->diag, vals, h->pivot, f, maxlen);
    }
  };
  // GPUFEM_ILU_LDS_CAP (bytes) lowers the LDS budget of a row, so that one
  // factorisation mixes LDS and global-memory rows (a test hook)
  size_t cap = lds_cap[ti];
  if (const char* cenv = getenv("GPUFEM_ILU_LDS_CAP"))
    cap = std::min<size_t>(cap, (size_t)std::max(0L, atol(cenv)));
  const char* senv = getenv("GPUFEM_ILU_SCHEDULE");
  const bool short_off = getenv("GPUFEM_ILU_SHORT_OFF") != nullptr;
  const bool by_level = senv && std::string(senv) == "level";
  const int nl = (int)h->lptr.size() - 1;
  // row values, column indices and pivot bounds of the level's longest
  // row, and two position lists as long as the longest row
  auto dyn_of = [&](int l) {
    return (size_t)h->lmaxlen[l] * (36 * sizeof(T) + 3 * sizeof(int)) +
           2 * sizeof(int) * (size_t)maxlen;
  };
  if (by_level) {
    for (int l = 0; l < nl; l++) {
      const int cnt = h->lptr[l + 1] - h->lptr[l];
      const size_t dyn = dyn_of(l);
      if (!no_lds && dyn <= cap)
        hipLaunchKernelGGL((gf::ilu_row_lds_kernel<T, false>), dim3(cnt),
                           dim3(gf::kIluThreads), dyn, ctx->stream,
                           h->lrows + h->lptr[l], cnt, h->rowp, h->cols,
                           h->diag, vals, h->pivot, gf::Flow{}, maxlen);
      else
        launch_global(false, h->lrows + h->lptr[l], cnt, gf::Flow{});
    }
  } else {
    // Dataflow: one launch per phase.  Levels before the first level with a
    // row too long for LDS run the LDS kernel, in phases whose LDS need
    // stays within twice that of their first level or 40 KB (so the wide
    // early levels keep several workgroups per CU); every level from there
    // on runs the global-memory kernel in one phase (row lengths of a
    // complete factorisation oscillate around the LDS limit, and a launch
    // boundary is a barrier for every row).  Launch boundaries order the
    // phases.
    if (++h->epoch <= 0) {
      GF_HIP(ctx, hipMemsetAsync(h->done, 0, sizeof(int) * (size_t)h->n,
                                 ctx->stream));
      h->epoch = 1;
    }
    // A row that takes more than half of a CU's LDS has the CU to itself,
    // where two workgroups of the global-memory kernel fit: such levels run
    // there unless they are chains (fewer than 1.25 rows a level), where only
    // a row's latency counts.  Half / all of the LDS: 400x400 plate ILU(96)
    // FP32 65 / 75 ms, FP64 83 / 86 ms; 101x101 ILU(64) FP32 6.0 / 7.6 ms;
    // complete LU of a wingbox of 24,390 nodes FP64 26.5 / 20.3 ms.
    auto levels_within = [&](size_t lim) {
      int l = 0;
      while (l < nl && !no_lds && dyn_of(l) <= lim) l++;
      return l;
    };
    int first_global = levels_within(std::min(cap, lds_half[ti]));
    if (4 * (h->n - h->lptr[first_global]) < 5 * (nl - first_global))
      first_global = levels_within(cap);
    // longest row up to each level: it bounds the U part of every pivot row
    // of the rows up to there
    std::vector<int> pmax(nl + 1, 0);
    for (int l = 0; l < nl; l++) pmax[l + 1] = std::max(pmax[l], h->lmaxlen[l]);
    int l0 = 0;
    while (l0 < nl) {
      const bool lds = l0 < first_global;
      const size_t d0 = dyn_of(l0);
      const size_t lim = std::max<size_t>(2 * d0, 40 * 1024);
      size_t dyn = d0;
      int l1 = l0 + 1;
      if (lds) {
        for (; l1 < first_global && dyn_of(l1) <= lim; l1++)
          dyn = std::max(dyn, dyn_of(l1));
      } else {
        l1 = nl;
      }
      const int r0 = h->lptr[l0], cnt = h->lptr[l1] - r0;
      gf::Flow f;
      f.counter = h->counter;
      f.base = h->base;
      f.done = h->done;
      f.epoch = h->epoch;
      f.err = h->err + 1;
      if (lds && pmax[l1] <= gf::kIluShortRow && !short_off) {
        // short rows: 256-thread workgroups, position lists as long as the
        // longest row so far
        int lmax = 0;
        for (int l = l0; l < l1; l++) lmax = std::max(lmax, h->lmaxlen[l]);
        const size_t dyn_s =
            (size_t)lmax * (36 * sizeof(T) + 3 * sizeof(int)) +
            2 * sizeof(int) * (size_t)pmax[l1];
        hipLaunchKernelGGL(
            (gf::ilu_row_lds_kernel<T, true, gf::kIluShortThreads>),
            dim3(cnt), dim3(gf::kIluShortThreads), dyn_s, ctx->stream,
            h->lrows + r0, cnt, h->rowp, h->cols, h->diag, vals, h->pivot, f,
            pmax[l1]);
      } else if (lds) {
        hipLaunchKernelGGL((gf::ilu_row_lds_kernel<T, true>), dim3(cnt),
                           dim3(gf::kIluThreads), dyn, ctx->stream,
                           h->lrows + r0, cnt, h->rowp, h->cols, h->diag, vals,
                           h->pivot, f, maxlen);
      } else {
        launch_global(true, h->lrows + r0, cnt, f);
      }
      h->base += (unsigned long long)cnt;
      l0 = l1;
    }
  }
  GF_TRY(gf::check_launch(ctx, "ilu_row_kernel"));
  int piv = big, werr = 0;
  GF_HIP(ctx, hipMemcpyAsync(&piv, h->pivot, sizeof(int),
                             hipMemcpyDeviceToHost, ctx->stream));
  GF_HIP(ctx, hipMemcpyAsync(&werr, h->err + 1, sizeof(int),
                             hipMemcpyDeviceToHost, ctx->stream));
  GF_HIP(ctx, hipStreamSynchronize(ctx->stream));
  if (werr) {
    const int zero = 0;
    GF_HIP(ctx, hipMemcpyAsync(h->err + 1, &zero, sizeof(int),
                               hipMemcpyHostToDevice, ctx->stream));
    GF_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return gf::set_error(ctx, GF_ERR_TIMEOUT,
                         "ILU factorisation: a dependency wait expired");
  }
  if (zero_pivot) *zero_pivot = piv == big ? -1 : piv;
  if (piv != big)
    return gf::set_error(ctx, GF_ERR_ZERO_PIVOT,
                         "ILU: zero pivot in diagonal block of row %d", piv);
  return GF_OK;
}

template <typename T>
int ilu_apply(gf_ilu h, const T* lu, const T* b, T* tmp, T* x) {
  if (!h || !lu || !b || !tmp || !x || b == tmp || tmp == x)
    return GF_ERR_INVALID;
  gf_context ctx = h->ctx;
  if (h->small) {
    gf::SweepSlot<T> one{};
    one.lmeta = h->lmeta;
    one.umeta = h->umeta;
    one.cols = h->cols;
    one.lu = lu;
    one.b = b;
    one.x = x;
    one.n = h->n;
    one.nllev = (int)h->lptr.size() - 1;
    one.nulev = (int)h->uptr.size() - 1;
    hipLaunchKernelGGL((gf::trsv_small_kernel<T, false>), dim3(1),
                       dim3(gf::kSmallThreads), sizeof(T) * 6 * (size_t)h->n,
                       ctx->stream, one, (const gf::SweepSlot<T>*)nullptr);
    return gf::check_launch(ctx, "trsv_small_kernel");
  }
  if (!h->level_sweeps) {
    const size_t N = 6 * (size_t)h->n;
    hipLaunchKernelGGL(gf::fill_sentinel_kernel<T>, dim3(gf::div_up(N, 256)),
                       dim3(256), 0, ctx->stream, N, tmp);
    if (h->nlgroup) {
      hipLaunchKernelGGL((gf::trsv_group_kernel<T, true>), dim3(h->ggrid),
                         dim3(gf::kGroupThreads), 0, ctx->stream, h->lgroup,
                         h->nlgroup, h->cols, lu, b, tmp, x, h->counter,
                         h->base, h->err);
      h->base += (unsigned long long)(h->nlgroup + h->ggrid);
      hipLaunchKernelGGL((gf::trsv_group_kernel<T, false>), dim3(h->ggrid),
                         dim3(gf::kGroupThreads), 0, ctx->stream, h->ugroup,
                         h->nugroup, h->cols, lu, tmp, x, (T*)nullptr,
                         h->counter, h->base, h->err);
      h->base += (unsigned long long)(h->nugroup + h->ggrid);
      return gf::check_launch(ctx, "trsv_group_kernel");
    }
    // one row per wavefront: two rows of a level per wavefront
    // (trsv_syncfree_kernel<T, L, 2>) measured slower, 4.8 vs 3.5 ms a pair
    // on the 400x400 plate
    unsigned long long* const ctr = h->counter + gf::kCounterStride;
    hipLaunchKernelGGL((gf::trsv_syncfree_kernel<T, true, 1>), dim3(h->grid),
                       dim3(gf::kSweepThreads), 0, ctx->stream, h->lmeta,
                       h->cols, h->lchunk, h->nlchunk, lu, b, tmp, x, ctr,
                       h->wbase, h->err);
    h->wbase += gf::div_up(h->nlchunk, gf::kSweepThreads / 64) +
                (unsigned long long)h->grid;
    hipLaunchKernelGGL((gf::trsv_syncfree_kernel<T, false, 1>), dim3(h->grid),
                       dim3(gf::kSweepThreads), 0, ctx->stream, h->umeta,
                       h->cols, h->uchunk, h->nuchunk, lu, tmp, x, (T*)nullptr,
                       ctr, h->wbase, h->err);
    h->wbase += gf::div_up(h->nuchunk, gf::kSweepThreads / 64) +
                (unsigned long long)h->grid;
    return gf::check_launch(ctx, "trsv_syncfree_kernel");
  }
  const int nl = (int)h->lptr.size() - 1;
  for (int l = 0; l < nl; l++) {
    const int cnt = h->lptr[l + 1] - h->lptr[l];
    hipLaunchKernelGGL((gf::trsv_level_kernel<T, true>),
                       dim3(gf::div_up(cnt, 40)), dim3(256), 0, ctx->stream,
                       h->lrows + h->lptr[l], cnt, h->rowp, h->cols, h->diag,
                       lu, b, tmp);
  }
  const int nu = (int)h->uptr.size() - 1;
  for (int l = 0; l < nu; l++) {
    const int cnt = h->uptr[l + 1] - h->uptr[l];
    hipLaunchKernelGGL((gf::trsv_level_kernel<T, false>),
                       dim3(gf::div_up(cnt, 40)), dim3(256), 0, ctx->stream,
                       h->urows + h->uptr[l], cnt, h->rowp, h->cols, h->diag,
                       lu, tmp, x);
  }
  return gf::check_launch(ctx, "trsv_level_kernel");
}
}  // namespace

extern "C" {
int gf_bsr_ilu_factor_f64(gf_ilu h, double* vals, int* zp) {
  return ilu_factor<double>(h, vals, zp);
}
int gf_bsr_ilu_factor_f32(gf_ilu h, float* vals, int* zp) {
  return ilu_factor<float>(h, vals, zp);
}
int gf_bsr_ilu_apply_f64(gf_ilu h, const double* lu, const double* b,
                         double* tmp, double* x) {
  return ilu_apply<double>(h, lu, b, tmp, x);
}
int gf_bsr_ilu_apply_f32(gf_ilu h, const float* lu, const float* b,
                         float* tmp, float* x) {
  return ilu_apply<float>(h, lu, b, tmp, x);
}
}  // extern "C"
