// gb_cg.hip -- device side of the conjugate-gradient solver.
//
// Reference: src/cgd.c:40-129.  One iteration is three kernels on the
// library stream, all scalars kept on the device (no host round trip):
//   K1 gb_spmv_kernel<DOT>: ap = A p and the p.ap partials
//   K2 gb_cg_update_r:      alpha = dr / p.ap; r -= alpha ap; r.r partials
//   K3 gb_cg_update_xp:     beta = r.r / dr, convergence test;
//                           ps = alpha p; x += ps; p = r + (beta/alpha) ps
// which is the reference's scale-then-add order (src/cgd.c:92-105) with
// the same separately rounded products and sums (-ffp-contract=off); only
// the order of the dot-product sums differs.  x += ps sits in K3, which
// reads p anyway (one vector read less than in K2; x does not feed r).
// K2 and K3 give each workgroup one contiguous chunk of rows; each
// workgroup adds the previous kernel's partials itself (the same values in
// the same order in every workgroup, so every workgroup gets the same
// scalar) while the loads of its chunk are in flight.
// K2 and K3 read the device `done` flag and return when the solve has
// stopped, so the host can enqueue iterations in batches (or replay them
// from a hipGraph) and still stop exactly where the reference stops.
// `done` is written only by the state's set-up and by K2's workgroup 0: K3
// records its stop in `status`, which every K3 workgroup computes for
// itself, so all of them still add their share of x; the next K2 turns a
// nonzero status into `done`.
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "gb_matrix.h"

#define GB_ELEM_GRID_MAX 2048u
#define GB_CG_NGRAPH 7  // captured batches of 1, 2, 4, ..., 64 iterations

struct gbd_cg {
  gbd_matrix *m;
  uint32_t n;
  double *r, *p, *ap;
  double *p2;         // one-launch runs: the other buffer of p
  uint64_t *slots;    // one-launch runs: the exchanges' slots
  double *b0;         // one-launch runs with x in the place of b: a copy of b
  double *partials;   // SpMV p.Ap partials (one per SpMV workgroup)
  double *partials2;  // r.r partials (one per elementwise workgroup)
  uint32_t npartials;
  gbd_cg_state *st;
  gbd_cg_state *h_st;  // pinned
  double *trace;
  uint32_t trace_cap;
  double *h_trace;     // pinned, trace_cap entries
  const double *b;
  double *x;
  uint32_t grid_elem;  // workgroups of the set-up kernel
  uint32_t grid_one;   // one-launch runs: workgroups of gb_cg_persist; else 0
  uint32_t rows_one;   // and rows per workgroup
  uint32_t spins;      // and reads of a slot before a wait is given up
  uint32_t grid_vec;   // workgroups of the r and x/p updates
  uint32_t chunk;      // rows per workgroup of the r and x/p updates
  hipGraph_t graph[GB_CG_NGRAPH];       // graph[i]: 2^i iterations
  hipGraphExec_t gexec[GB_CG_NGRAPH];
  double *graph_x;                      // x the graphs were captured with
  bool noalloc;  // the workspace in `scratch`: single launches, no graphs
};

// Fixed-order sum of n partials, computed identically by every workgroup
// that calls it and returned to all of its threads.
__device__ __forceinline__ double gb_sum_partials(const double *partials,
                                                  uint32_t n, double *red) {
  // all loads of a chunk issued before the adds: one memory round trip per
  // 2048 partials instead of one per 256
  double s = 0.0;
  for (uint32_t base = 0; base < n; base += GB_BLOCK * 8) {
    double v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      uint32_t i = base + j * GB_BLOCK + threadIdx.x;
      v[j] = i < n ? partials[i] : 0.0;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) s += v[j];
  }
  s = gb_wave_sum(s);
  const int lane = threadIdx.x & (GB_WAVE - 1);
  const int wave = threadIdx.x / GB_WAVE;
  if (lane == 0) red[wave] = s;
  __syncthreads();
  double t = red[0];
#pragma unroll
  for (int w = 1; w < GB_WAVES_PER_BLOCK; ++w) t += red[w];
  __syncthreads();
  return t;
}

// src/cgd.c:81-85: x = 0; r = b; p = r; partial sums of r.r
__global__ void __launch_bounds__(GB_BLOCK)
gb_cg_init(const double *__restrict__ b, double *__restrict__ x,
           double *__restrict__ r, double *__restrict__ p, uint32_t n,
           double *__restrict__ partials) {
  __shared__ double red[GB_WAVES_PER_BLOCK];
  double d = 0.0;
  for (uint32_t i = blockIdx.x * GB_BLOCK + threadIdx.x; i < n;
       i += gridDim.x * GB_BLOCK) {
    double v = b[i];
    x[i] = 0.0;
    r[i] = v;
    p[i] = v;
    d += v * v;
  }
  double bs = gb_block_sum(d, red);
  if (threadIdx.x == 0) partials[blockIdx.x] = bs;
}

// dr = r.r, ||b||, the absolute threshold; one workgroup
__global__ void __launch_bounds__(GB_BLOCK)
gb_cg_init_state(const double *__restrict__ partials, uint32_t np,
                 gbd_cg_state *st, double tol, int rel,
                 unsigned long long maxiter) {
  __shared__ double red[GB_WAVES_PER_BLOCK];
  double s = gb_sum_partials(partials, np, red);
  if (threadIdx.x == 0) {
    st->dr = s;
    st->dr_prev = s;
    st->rnorm0 = sqrt(s);
    st->rnorm = st->rnorm0;
    st->tol = rel ? tol * st->rnorm0 : tol;
    st->pap = 0.0;
    st->alpha = 0.0;
    st->beta = 0.0;
    st->iter = 0;
    st->iter_next = 0;
    st->maxiter = maxiter;
    st->status = 0;
    st->done = 0;
    st->waited = 0;
    if (s == 0.0) {  // b == 0: x = 0 is the solution
      st->done = 1;
      st->status = 1;
    } else if (!isfinite(s)) {
      st->done = 1;
      st->status = 3;
    }
  }
}

// src/cgd.c:90, 96-97: alpha = dr / p.Ap; r -= alpha Ap; partial sums of
// r.r.  Each workgroup owns one contiguous chunk of rows and first issues
// the loads of its r and Ap values, then adds the SpMV's p.Ap partials
// itself -- every workgroup the same values in the same fixed order, so
// all of them get the same alpha and no separate reduction launch is
// needed -- while those loads are in flight.  Workgroup 0 records alpha
// and turns a stop recorded by the previous iteration's x/p update into
// `done`.
// Launch shape of K2 and K3: GB_CGV_THREADS threads, each with GB_CGV_U
// rows per pass, at most one workgroup per CU.  On the 160^3 Laplacian
// (n = 4,096,000) every workgroup then covers its 16,000 rows in one pass,
// with all of its loads issued at once.
#define GB_CGV_THREADS 512
#define GB_CGV_GRID 256u
// rows per thread and pass at most.  Smaller systems take the kernel built
// for the rows they have (U), and for the SpMV partials per thread (R: at
// most 32 loads in one round): the sums' order is the same for every U and R.
// A kernel built for 32 rows a thread spends about 2 us on the 31 absent ones:
// an iteration took 16.2 us on the 256^2 Laplacian, and takes 12.0 us.
#define GB_CGV_U 32

// Fixed-order sum of n partials by a workgroup of T threads: each thread
// issues R loads before adding (one memory round trip per T R partials);
// the result is returned to every thread.
template <int T, int R>
__device__ __forceinline__ double gb_cgv_sum(const double *__restrict__ part,
                                             uint32_t n, double *red) {
  double s = 0.0;
  for (uint32_t base = 0; base < n; base += T * R) {
    double v[R];
#pragma unroll
    for (int j = 0; j < R; ++j) {
      uint32_t i = base + j * T + threadIdx.x;
      v[j] = i < n ? part[i] : 0.0;
    }
#pragma unroll
    for (int j = 0; j < R; ++j) s += v[j];
  }
  s = gb_wave_sum(s);
  if ((threadIdx.x & (GB_WAVE - 1)) == 0) red[threadIdx.x / GB_WAVE] = s;
  __syncthreads();
  double t = red[0];
#pragma unroll
  for (int w = 1; w < T / GB_WAVE; ++w) t += red[w];
  __syncthreads();
  return t;
}

// Sum of one value per thread over a workgroup of T threads (wave
// butterflies, then the wave totals in wave order); valid on thread 0.
template <int T>
__device__ __forceinline__ double gb_cgv_block_sum(double v, double *red) {
  v = gb_wave_sum(v);
  if ((threadIdx.x & (GB_WAVE - 1)) == 0) red[threadIdx.x / GB_WAVE] = v;
  __syncthreads();
  double t = 0.0;
  if (threadIdx.x == 0) {
    t = red[0];
#pragma unroll
    for (int w = 1; w < T / GB_WAVE; ++w) t += red[w];
  }
  return t;
}

template <int T, int U, int R>
__global__ void __launch_bounds__(T)
gb_cg_update_r(double *__restrict__ r, const double *__restrict__ ap, uint32_t n,
               uint32_t chunk, const double *__restrict__ pap_partials, uint32_t npap,
               double *__restrict__ partials, gbd_cg_state *st) {
  __shared__ double red[T / GB_WAVE];
  __shared__ int32_t s_stop, s_bad;
  __shared__ double s_alpha;
  const uint32_t tid = threadIdx.x;
  const uint32_t i0 = blockIdx.x * chunk;  // < n: the grid is ceil(n / chunk)
  const uint32_t len = n - i0 < chunk ? n - i0 : chunk;
  double rv[U], av[U];
#pragma unroll
  for (int j = 0; j < U; ++j) {
    const uint32_t o = j * T + tid;
    if (o < len) {
      const uint32_t i = i0 + o;
      rv[j] = r[i];
      av[j] = ap[i];
    }
  }
  if (tid == 0) {
    // a stop recorded by the previous iteration's x/p update becomes `done`
    // (workgroups that read `done` while workgroup 0 sets it see the
    // nonzero status as well)
    const int32_t dn = *(volatile int32_t *)&st->done;
    const int32_t stop = dn || *(volatile int32_t *)&st->status;
    if (stop && !dn && blockIdx.x == 0) st->done = 1;
    s_stop = stop;
  }
  const double pap = gb_cgv_sum<T, R>(pap_partials, npap, red);  // barriers inside
  if (s_stop) return;
  if (tid == 0) {
    const double dr = st->dr;
    const double alpha = dr / pap;
    const bool bad = !(pap != 0.0) || !isfinite(alpha);
    if (blockIdx.x == 0) {
      st->pap = pap;
      st->alpha = alpha;
      if (bad) {
        st->done = 1;
        st->status = 3;
      } else {
        st->dr_prev = dr;
        st->iter_next = st->iter + 1;
      }
    }
    s_alpha = bad ? 0.0 : alpha;
    s_bad = bad;
  }
  __syncthreads();
  if (s_bad) return;
  const double alpha = s_alpha;
  double d = 0.0;
  for (uint32_t done = 0;;) {
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const uint32_t o = done + j * T + tid;
      if (o < len) {
        const uint32_t i = i0 + o;
        const double aps = alpha * av[j];
        const double rn = rv[j] - aps;
        r[i] = rn;
        d += rn * rn;
      }
    }
    if (len - done <= U * T) break;
    done += U * T;
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const uint32_t o = done + j * T + tid;
      if (o < len) {
        const uint32_t i = i0 + o;
        rv[j] = r[i];
        av[j] = ap[i];
      }
    }
  }
  const double bs = gb_cgv_block_sum<T>(d, red);
  if (tid == 0) partials[blockIdx.x] = bs;
}

// src/cgd.c:92-94, 100-119: beta = r.r / dr; stop when sqrt(r.r) <= tol or
// at the iteration cap; ps = alpha p; x += ps; unless stopping,
// p = nr + (beta/alpha) ps.  The workgroup's x, p and r values are loaded
// first; the r.r partials of the r update are added (the same order in
// every workgroup) while they are in flight.
template <int T, int U>
__global__ void __launch_bounds__(T)
gb_cg_update_xp(double *__restrict__ x, const double *__restrict__ r,
                double *__restrict__ p, uint32_t n, uint32_t chunk,
                const double *__restrict__ dnr_partials, uint32_t ndnr,
                gbd_cg_state *st, double *__restrict__ trace, uint32_t trace_cap) {
  __shared__ double red[T / GB_WAVE];
  __shared__ int32_t s_done;
  const uint32_t tid = threadIdx.x;
  const uint32_t i0 = blockIdx.x * chunk;  // < n: the grid is ceil(n / chunk)
  const uint32_t len = n - i0 < chunk ? n - i0 : chunk;
  double xv[U], pv[U], rv[U];
#pragma unroll
  for (int j = 0; j < U; ++j) {
    const uint32_t o = j * T + tid;
    if (o < len) {
      const uint32_t i = i0 + o;
      xv[j] = x[i];
      pv[j] = p[i];
      rv[j] = r[i];
    }
  }
  // `done` is written only by the r update and the set-up, never during
  // this kernel
  if (tid == 0) s_done = *(volatile int32_t *)&st->done;
  const double dnr = gb_cgv_sum<T, 1>(dnr_partials, ndnr, red);  // barriers inside
  if (s_done) return;
  const double alpha = st->alpha;
  const double beta = dnr / st->dr_prev;
  const double rnorm = sqrt(dnr);
  const unsigned long long it1 = st->iter_next;
  int status = 0;
  if (rnorm <= st->tol) status = 1;
  else if (!isfinite(dnr)) status = 3;
  else if (st->maxiter && it1 >= st->maxiter) status = 2;
  if (blockIdx.x == 0 && tid == 0) {
    st->beta = beta;
    st->dr = dnr;
    st->rnorm = rnorm;
    if (trace_cap) trace[(it1 - 1) % trace_cap] = rnorm;
    st->iter = it1;
    // not `done`: the other workgroups of this launch may not have read it
    if (status) st->status = status;
  }
  const double boa = beta / alpha;
  for (uint32_t done = 0;;) {
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const uint32_t o = done + j * T + tid;
      if (o < len) {
        const uint32_t i = i0 + o;
        const double ps = alpha * pv[j];
        x[i] = xv[j] + ps;
        if (!status) {
          const double t = ps * boa;
          p[i] = rv[j] + t;
        }
      }
    }
    if (len - done <= U * T) break;
    done += U * T;
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const uint32_t o = done + j * T + tid;
      if (o < len) {
        const uint32_t i = i0 + o;
        xv[j] = x[i];
        pv[j] = p[i];
        rv[j] = r[i];
      }
    }
  }
}

// A whole run of iterations in one launch, for systems small enough that the
// matrix fits the workgroups' LDS (one workgroup per CU).  Workgroup w owns a
// range of rows: their entries in LDS, their x, r, p and Ap in registers, one
// thread per row.  What workgroups tell each other goes through memory with
// relaxed agent-scope accesses, which no L1 or other XCD's L2 holds back:
//
//  - a sum over all rows: each workgroup stores its partial (after its other
//    stores have completed) to a slot of its own, and every workgroup reads
//    all slots until none holds the empty mark, and adds them in order.  The
//    same exchange orders the data: whoever has read all partials may read
//    what their owners stored before them.  Three rounds of slots take
//    turns; an owner empties its slot of the round before once it has
//    passed a round (all have then read it).
//  - p: the products of an iteration need the new p of other workgroups'
//    rows, p = r + (beta/alpha) (alpha p).  r was stored before the r.r
//    exchange and the old p an iteration earlier, so each workgroup forms
//    the new p of the columns it needs by itself, with the owner's operations
//    and so the same bits: two exchanges an iteration, p.Ap and r.r.
//
// The sums of each row and the updates are those of gb_cg_update_r and
// gb_cg_update_xp; the dot products are grouped by thread and workgroup in
// this kernel's own fixed way.
//
// The grid is at most the CUs, so the workgroups run side by side.  A workgroup
// whose wait does not end within `spins` reads sets the state's `waited` and
// leaves, without its rows of x; the others then run out of time in a later
// exchange, or, if this was the last, end the solve.  So `waited` is a word
// that only the set-up clears and no other end of a run touches, and the host
// looks at it before all else: the solve starts again on the other kernels,
// and the matrix stays with them until its plan is built anew.
// Workgroups may still be starting when it is set, and one thread decides for
// each of them whether it runs.
//
// Bound: the latency of two exchanges (1.4 us for 16 workgroups to 2.5 us for
// 256, in a kernel of exchanges alone) and of the gathers.  Per iteration,
// with the host's part, against three kernels replayed from a graph: 5.1 and
// 15.3 us on the 64^2 Laplacian, 7.6 and 16.2 us at 256^2, 10.7 and 17.9 us at
// 400^2, 16.5 and 22.1 us at 600^2, 17.5 and 22.4 us at 70^3 (those kernels
// built for small systems, below: 11.2, 12.0, 14.0, 18.5 and 18.8 us).  With
// 1024 threads a workgroup 256^2 takes 8.0 us, with 128 workgroups 8.8 us,
// with 32 workgroups 8.8 us.  Tried instead, and slower at every size above
// 65,000 rows: two kernels an iteration, the x/p update in the SpMV's (11.1 us
// at 256^2, 22.1 us at 600^2, 43 us at 100^3).
#define GB_CGP_THREADS 512
#define GB_CGP_ENTRIES 12544u  // entries in a workgroup's LDS (147 KB)
#define GB_CGP_GRID 256u
#define GB_CGP_ROWS 4          // rows per thread at most
#define GB_CGP_WGS 64u         // workgroups, while the rows fit them
#define GB_CGP_SPINS (1u << 20)  // 0.16 s, paid once: the matrix takes the others then
static_assert(GB_CGP_GRID <= GB_CGP_THREADS, "one slot per thread");
#define GB_CGP_PAD 16          // slots a cache line apart
#define GB_CGP_SLOT_BYTES (3ull * GB_CGP_GRID * GB_CGP_PAD * 8)
#define GB_CGP_EMPTY 0x7ff8dead00000001ull

__device__ __forceinline__ double gb_cgp_load(const double *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void gb_cgp_store(double *p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct gb_cgp_lds {
  double val[GB_CGP_ENTRIES];
  uint32_t col[GB_CGP_ENTRIES];
  double part[GB_CGP_GRID];
  double red[GB_CGP_THREADS / GB_WAVE];
  uint32_t stop;  // no run, or a wait given up
};

// the sum of every workgroup's d, in a fixed order, on every thread; round
// counts the exchanges of the launch.  False when a wait ran out.  (In exchange
// `lost` the last workgroup's does, whatever it reads: GB_FAULT_CG_WAIT.)
__device__ __forceinline__ bool gb_cgp_sum(double d, uint64_t *slots, uint32_t round,
                                           uint32_t spins, uint32_t lost, gb_cgp_lds &L,
                                           double *sum) {
  const uint32_t tid = threadIdx.x, W = gridDim.x;
  d = gb_wave_sum(d);
  if ((tid & (GB_WAVE - 1)) == 0) L.red[tid / GB_WAVE] = d;
  // this wavefront's stores have completed before any partial is out
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  uint64_t *mine = slots + (size_t)(round % 3) * GB_CGP_GRID * GB_CGP_PAD;
  if (tid == 0 && W > 1) {
    double t = L.red[0];
#pragma unroll
    for (int w = 1; w < GB_CGP_THREADS / GB_WAVE; ++w) t += L.red[w];
    uint64_t bits = (uint64_t)__double_as_longlong(t);
    if (!(t == t)) bits = 0x7ff8000000000000ull;  // any NaN, and not the mark
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __hip_atomic_store(&mine[blockIdx.x * GB_CGP_PAD], bits, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  }
  if (W == 1) {  // the workgroup's own partials are all
    double t = L.red[0];
#pragma unroll
    for (int w = 1; w < GB_CGP_THREADS / GB_WAVE; ++w) t += L.red[w];
    __syncthreads();  // red is used by the next sum
    *sum = t;
    return true;
  }
  if (tid < W) {
    uint64_t v;
    uint32_t n = 0;
    while ((v = __hip_atomic_load(&mine[tid * GB_CGP_PAD], __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT)) == GB_CGP_EMPTY) {
      if (++n > spins) {
        L.stop = 1;
        break;
      }
    }
    if (round == lost && blockIdx.x == W - 1) L.stop = 1;
    L.part[tid] = __longlong_as_double((long long)v);
  }
  __syncthreads();
  if (L.stop) return false;
  if (tid == 0)  // the round before: everyone has read it
    __hip_atomic_store(&slots[((size_t)((round + 2) % 3) * GB_CGP_GRID + blockIdx.x) *
                              GB_CGP_PAD],
                       GB_CGP_EMPTY, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  double t = 0.0;
  for (uint32_t i = tid & (GB_WAVE - 1); i < W; i += GB_WAVE) t += L.part[i];
  *sum = gb_wave_sum(t);
  return true;
}

__global__ void __launch_bounds__(GB_BLOCK)
gb_cgp_empty(uint64_t *__restrict__ slots) {
  for (uint32_t i = threadIdx.x; i < 3 * GB_CGP_GRID; i += GB_BLOCK)
    slots[(size_t)i * GB_CGP_PAD] = GB_CGP_EMPTY;
}

// most[q]: the most entries that a range of rows[q] rows has, or 0 for none
#define GB_CGP_TRIES 3
struct gb_cgp_tries {
  uint32_t rows[GB_CGP_TRIES];
};
__global__ void __launch_bounds__(GB_BLOCK)
gb_cgp_most(const uint32_t *__restrict__ rowptr, uint32_t n, gb_cgp_tries t,
            uint32_t *__restrict__ most) {
  __shared__ uint32_t m;
  if (threadIdx.x == 0) m = 0;
  __syncthreads();
  const uint32_t rows = t.rows[blockIdx.x];
  for (uint64_t a = (uint64_t)threadIdx.x * rows; rows && a < n; a += (uint64_t)GB_BLOCK * rows)
    atomicMax(&m, rowptr[n - a < rows ? n : a + rows] - rowptr[a]);
  __syncthreads();
  if (threadIdx.x == 0) most[blockIdx.x] = m;
}

// k iterations (fewer when the solve stops); p0 holds p before and after,
// p1 is the other buffer
template <int R>
__global__ void __launch_bounds__(GB_CGP_THREADS)
gb_cg_persist(const uint32_t *__restrict__ rowptr, const uint32_t *__restrict__ rowind,
              const double *__restrict__ val, uint32_t n, uint32_t rows, double *x, double *r,
              double *p0, double *p1, uint64_t *slots, gbd_cg_state *st, double *trace,
              uint32_t trace_cap, uint32_t k, uint32_t spins, uint32_t lost) {
  constexpr uint32_t T = GB_CGP_THREADS;
  constexpr uint32_t U = 8;  // entries of a row whose gathers are in flight
  __shared__ gb_cgp_lds L;
  const uint32_t tid = threadIdx.x;
  if (tid == 0)
    L.stop = *(volatile int32_t *)&st->done | *(volatile int32_t *)&st->status |
             __hip_atomic_load(&st->waited, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (L.stop) return;  // the whole workgroup: set again only past the next barrier
  const uint32_t row0 = blockIdx.x * rows;
  const uint32_t end = n - row0 < rows ? n : row0 + rows;
  const uint32_t k0 = rowptr[row0], k1 = rowptr[end];
  for (uint32_t e = tid; e < k1 - k0; e += T) {
    L.col[e] = rowind[k0 + e];
    L.val[e] = val[k0 + e];
  }
  uint32_t e0[R], e1[R];
  double xo[R], ro[R], po[R], ao[R];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const uint32_t i = row0 + q * T + tid;
    e0[q] = e1[q] = 0;
    xo[q] = ro[q] = po[q] = ao[q] = 0.0;
    if (i < end) {
      e0[q] = rowptr[i] - k0;
      e1[q] = rowptr[i + 1] - k0;
      xo[q] = x[i];
      ro[q] = r[i];
      po[q] = p0[i];
    }
  }
  double dr = st->dr, dr_prev = st->dr_prev, rnorm = st->rnorm, pap = st->pap;
  double alpha = st->alpha, beta = st->beta, boa = 0.0;
  const double tol = st->tol;
  unsigned long long iter = st->iter;
  const unsigned long long maxiter = st->maxiter;
  int status = 0;
  uint32_t round = 0;
  double *pold = p0, *pnew = p1;
  uint32_t ulen = 0;  // entries of the wavefront's longest row
#pragma unroll
  for (int q = 0; q < R; ++q) ulen = max(ulen, e1[q] - e0[q]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) ulen = max(ulen, (uint32_t)__shfl_xor((int)ulen, o, GB_WAVE));
  ulen = (uint32_t)__builtin_amdgcn_readfirstlane((int)ulen);
  __syncthreads();
  for (uint32_t it = 0; it < k && !status; ++it) {
    // Ap of the new p (the first iteration's p is complete)
    double d = 0.0;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const uint32_t i = row0 + q * T + tid;
      if (it && i < end) {
        const double ps = alpha * po[q];
        const double t = ps * boa;
        po[q] = ro[q] + t;
        gb_cgp_store(&pnew[i], po[q]);
      }
      double s = 0.0;
      for (uint32_t e = e0[q]; e < e1[q]; e += U) {
        uint32_t c[U];
        double a[U], gp[U], gr[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) c[u] = L.col[min(e + u, e1[q] - 1)];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
          if (u < ulen) {
            gp[u] = gb_cgp_load(&pold[c[u]]);
            if (it) gr[u] = gb_cgp_load(&r[c[u]]);
          }
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) a[u] = L.val[min(e + u, e1[q] - 1)];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
          double pc = gp[u];
          if (it) {
            const double t = (alpha * gp[u]) * boa;
            pc = gr[u] + t;
          }
          if (e + u < e1[q]) s += a[u] * pc;
        }
      }
      ao[q] = s;
      d += po[q] * s;
    }
    if (!gb_cgp_sum(d, slots, round++, spins, lost, L, &pap)) break;
    alpha = dr / pap;
    if (!(pap != 0.0) || !isfinite(alpha)) {
      status = 3;
      break;
    }
    if (it) {  // pnew is the current p now
      double *t = pold;
      pold = pnew;
      pnew = t;
    }
    d = 0.0;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const uint32_t i = row0 + q * T + tid;
      if (i < end) {
        const double aps = alpha * ao[q];
        ro[q] = ro[q] - aps;
        gb_cgp_store(&r[i], ro[q]);
        d += ro[q] * ro[q];
        const double ps = alpha * po[q];
        xo[q] = xo[q] + ps;
      }
    }
    double dnr;
    if (!gb_cgp_sum(d, slots, round++, spins, lost, L, &dnr)) break;
    beta = dnr / dr;
    dr_prev = dr;
    dr = dnr;
    rnorm = sqrt(dnr);
    ++iter;
    if (rnorm <= tol) status = 1;
    else if (!isfinite(dnr)) status = 3;
    else if (maxiter && iter >= maxiter) status = 2;
    boa = beta / alpha;
    if (trace_cap && blockIdx.x == 0 && tid == 0) trace[(iter - 1) % trace_cap] = rnorm;
  }
  if (L.stop) {  // set before a barrier that every thread has passed
    if (tid == 0)
      __hip_atomic_store(&st->waited, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const uint32_t i = row0 + q * T + tid;
    if (i < end) {
      x[i] = xo[q];
      if (!status) {
        const double ps = alpha * po[q];
        const double t = ps * boa;
        p0[i] = ro[q] + t;
      }
    }
  }
  if (blockIdx.x == 0 && tid == 0) {
    st->pap = pap;
    st->alpha = alpha;
    st->beta = beta;
    st->dr = dr;
    st->dr_prev = dr_prev;
    st->rnorm = rnorm;
    st->iter = iter;
    st->iter_next = iter;
    if (status) {
      st->status = status;
      st->done = 1;
    }
  }
}

template <int U, int R>
static void gb_cg_go_r(gbd_cg *cg, uint32_t npap) {
  gb_cg_update_r<GB_CGV_THREADS, U, R><<<cg->grid_vec, GB_CGV_THREADS, 0, gb_stream()>>>(
      cg->r, cg->ap, cg->n, cg->chunk, cg->partials, npap, cg->partials2, cg->st);
}

template <int U>
static void gb_cg_go_r_u(gbd_cg *cg, uint32_t npap) {
  if (npap <= 1 * GB_CGV_THREADS) gb_cg_go_r<U, 1>(cg, npap);
  else if (npap <= 4 * GB_CGV_THREADS) gb_cg_go_r<U, 4>(cg, npap);
  else gb_cg_go_r<U, 32>(cg, npap);
}

// the r update after npap SpMV partials
static void gb_cg_launch_r(gbd_cg *cg, uint32_t npap) {
  const uint32_t rows = gb_div_up(cg->chunk, GB_CGV_THREADS);
  if (rows <= 1) gb_cg_go_r_u<1>(cg, npap);
  else if (rows <= 4) gb_cg_go_r_u<4>(cg, npap);
  else if (rows <= 8) gb_cg_go_r_u<8>(cg, npap);
  else gb_cg_go_r_u<GB_CGV_U>(cg, npap);
}

template <int U>
static void gb_cg_go_xp(gbd_cg *cg) {
  gb_cg_update_xp<GB_CGV_THREADS, U><<<cg->grid_vec, GB_CGV_THREADS, 0, gb_stream()>>>(
      cg->x, cg->r, cg->p, cg->n, cg->chunk, cg->partials2, cg->grid_vec, cg->st,
      cg->trace, cg->trace_cap);
}

static void gb_cg_launch_xp(gbd_cg *cg) {
  const uint32_t rows = gb_div_up(cg->chunk, GB_CGV_THREADS);
  if (rows <= 1) gb_cg_go_xp<1>(cg);
  else if (rows <= 4) gb_cg_go_xp<4>(cg);
  else if (rows <= 8) gb_cg_go_xp<8>(cg);
  else gb_cg_go_xp<GB_CGV_U>(cg);
}

template <int R>
static void gb_cg_go_persist(gbd_cg *cg, uint32_t k, uint32_t lost) {
  const gbd_matrix *m = cg->m;
  gb_cg_persist<R><<<cg->grid_one, GB_CGP_THREADS, 0, gb_stream()>>>(
      m->rowptr, m->rowind, m->val, cg->n, cg->rows_one, cg->x, cg->r, cg->p, cg->p2,
      cg->slots, cg->st, cg->trace, cg->trace_cap, k, cg->spins, lost);
}

static int gb_cg_enqueue_raw(gbd_cg *cg, uint32_t k) {
  if (cg->grid_one) {
    gb_cgp_empty<<<1, GB_BLOCK, 0, gb_stream()>>>(cg->slots);
    GB_LAUNCH_CHECK();
    const uint32_t per = gb_div_up(cg->rows_one, GB_CGP_THREADS);
    const uint32_t lost = cg->grid_one > 1 ? gb_fault_cg_wait() : 0xffffffffu;
    if (per <= 1) gb_cg_go_persist<1>(cg, k, lost);
    else if (per <= 2) gb_cg_go_persist<2>(cg, k, lost);
    else gb_cg_go_persist<GB_CGP_ROWS>(cg, k, lost);
    GB_LAUNCH_CHECK();
    return GOOSEBERRY_SUCCESS;
  }
  for (uint32_t it = 0; it < k; ++it) {
    int rv = gb_spmv_launch(cg->m, cg->p, cg->ap, 1, cg->partials, cg->st);
    if (rv != GOOSEBERRY_SUCCESS) return rv;
    gb_cg_launch_r(cg, gb_spmv_npartials(cg->m));
    GB_LAUNCH_CHECK();
    gb_cg_launch_xp(cg);
    GB_LAUNCH_CHECK();
  }
  return GOOSEBERRY_SUCCESS;
}

static void gb_cg_drop_graph(gbd_cg *cg) {
  for (int i = 0; i < GB_CG_NGRAPH; ++i) {
    if (cg->gexec[i]) (void)hipGraphExecDestroy(cg->gexec[i]);
    if (cg->graph[i]) (void)hipGraphDestroy(cg->graph[i]);
    cg->gexec[i] = nullptr;
    cg->graph[i] = nullptr;
  }
  cg->graph_x = nullptr;
}

extern "C" {

// ------------------------------------------------- allocation-free solves
// The workspace of gbd_cg_scratch solves (r, p, Ap, the two partial arrays
// and the state) lives in this file-scope device array: such a solve makes
// no device allocation.  Each device holds its own copy at its own address,
// looked up once per device with hipGetSymbolAddress; host code uses that
// address, never the array's name.  Every such solve on a device shares the
// array, so solves that overlap on one device would race (the library lock
// serialises the public entry points of one process).  Small systems run in
// one launch here too, so both entry points give the same bits.
#define GB_CG_SCRATCH_BYTES (128ull << 20)
#define GB_CG_SCRATCH_MAXDEV 64
static __device__ __align__(256) unsigned char scratch[GB_CG_SCRATCH_BYTES];
static void *g_scratch_addr[GB_CG_SCRATCH_MAXDEV];
static gbd_cg g_scratch_cg;            // host bookkeeping of the shared workspace
static gbd_cg_state g_scratch_hst;     // its polled state (pageable host memory)

// the array's address on the current device
static int gb_cg_scratch_base(unsigned char **base) {
  int dev = 0;
  GB_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= GB_CG_SCRATCH_MAXDEV) {
    gb_set_error("device %d is beyond the %d devices the scratch table covers", dev,
                 GB_CG_SCRATCH_MAXDEV);
    return GOOSEBERRY_ERROR_INVALIDINPUT;
  }
  if (!g_scratch_addr[dev]) {
    void *a = nullptr;
    GB_HIP(hipGetSymbolAddress(&a, HIP_SYMBOL(scratch)));
    g_scratch_addr[dev] = a;
  }
  *base = (unsigned char *)g_scratch_addr[dev];
  return GOOSEBERRY_SUCCESS;
}

// Whether the solve runs in one launch, and on which workgroups: the fewest
// (the exchanges' time grows with them) whose rows' entries fit their LDS,
// for matrices with short rows only.  Found once per plan, by a kernel that
// counts the entries of the ranges into the scratch array (no solve is using it
// then), and kept with the matrix: every workspace of it takes the same kernels.
static int gb_cg_one_find(gbd_matrix *m) {
  const uint32_t n = m->nrows;
  m->cg_grid = m->cg_rows = 0;
  if (!n || m->nwave || m->nblockrows || m->nsplit || m->nparts || m->xt.ptr || m->cshift)
    return GOOSEBERRY_SUCCESS;
  uint32_t cus = gb_num_cus();
  if (cus > GB_CGP_GRID) cus = GB_CGP_GRID;
  gb_cgp_tries t = {{0, 0, 0}};
  uint32_t W = GB_CGP_WGS, any = 0, most[GB_CGP_TRIES];
  for (int q = 0; q < GB_CGP_TRIES && W <= cus; ++q, W *= 2) {
    // a row per thread, or fewer rows a workgroup when they are long
    uint32_t w = gb_div_up(n, GB_CGP_THREADS);
    const uint32_t we = gb_div_up(m->nnz, GB_CGP_ENTRIES / 8 * 7);
    if (w < we) w = we;
    if (w > W) w = W;
    const uint32_t rows = gb_div_up(gb_div_up(n, w), GB_WAVE) * GB_WAVE;
    if (rows <= GB_CGP_ROWS * GB_CGP_THREADS) any |= t.rows[q] = rows;
  }
  if (!any) return GOOSEBERRY_SUCCESS;
  unsigned char *base = nullptr;
  const int rv = gb_cg_scratch_base(&base);
  if (rv != GOOSEBERRY_SUCCESS) return rv;
  gb_cgp_most<<<GB_CGP_TRIES, GB_BLOCK, 0, gb_stream()>>>(m->rowptr, n, t, (uint32_t *)base);
  GB_LAUNCH_CHECK();
  GB_HIP(gb_fetch(most, base, sizeof(most)));
  for (int q = 0; q < GB_CGP_TRIES; ++q) {
    if (!t.rows[q] || most[q] > GB_CGP_ENTRIES) continue;
    m->cg_grid = gb_div_up(n, t.rows[q]);
    m->cg_rows = t.rows[q];
    break;
  }
  return GOOSEBERRY_SUCCESS;
}

// Launch geometry and partial-array sizes of a solve with m.
static int gb_cg_geometry(gbd_cg *cg, gbd_matrix *m) {
  cg->m = m;
  cg->n = m->nrows;
  uint32_t ge = gb_div_up(cg->n ? cg->n : 1, GB_BLOCK);
  cg->grid_elem = ge > GB_ELEM_GRID_MAX ? GB_ELEM_GRID_MAX : ge;
  // the vector updates: at most one workgroup per CU, each a contiguous
  // chunk of a multiple of 64 rows (aligned wavefront accesses)
  const uint64_t nn = cg->n ? cg->n : 1;
  uint32_t gv = gb_div_up(nn, GB_CGV_THREADS);
  if (gv > GB_CGV_GRID) gv = GB_CGV_GRID;
  cg->chunk = gb_div_up(gb_div_up(nn, gv), GB_WAVE) * GB_WAVE;
  cg->grid_vec = gb_div_up(nn, cg->chunk);
  uint32_t gs = gb_spmv_npartials(m);
  cg->npartials = gs > cg->grid_elem ? gs : cg->grid_elem;
  if (!m->cg_known) {
    const int rv = gb_cg_one_find(m);
    if (rv != GOOSEBERRY_SUCCESS) return rv;
    m->cg_known = true;
  }
  cg->grid_one = m->cg_grid;
  cg->rows_one = m->cg_rows;
  // GOOSEBERRY_CG_SPINS: the tests' way into the end of a wait
  const char *e = getenv("GOOSEBERRY_CG_SPINS");
  cg->spins = e && *e ? (uint32_t)strtoul(e, nullptr, 10) : GB_CGP_SPINS;
  return GOOSEBERRY_SUCCESS;
}

static uint32_t gb_cg_np2(const gbd_cg *cg) {
  return cg->grid_elem > cg->grid_vec ? cg->grid_elem : cg->grid_vec;
}

int gbd_cg_create(gbd_matrix *m, gbd_cg **out) {
  int rv = gb_ensure_init();
  if (rv != GOOSEBERRY_SUCCESS) return rv;
  if (m->nrows != m->ncols) return GOOSEBERRY_ERROR_INVALIDINPUT;
  gbd_cg *cg = (gbd_cg *)calloc(1, sizeof(gbd_cg));
  if (!cg) return GOOSEBERRY_ERROR_NOMEMORY;
  if ((rv = gb_cg_geometry(cg, m)) != GOOSEBERRY_SUCCESS) {
    free(cg);
    return rv;
  }
  size_t nb = (size_t)(cg->n ? cg->n : 1) * sizeof(double);
  hipError_t e = gb_dev_alloc((void **)&cg->r, nb);
  if (e == hipSuccess) e = gb_dev_alloc((void **)&cg->p, nb);
  if (e == hipSuccess) e = gb_dev_alloc((void **)&cg->ap, nb);
  if (e == hipSuccess && cg->grid_one) e = gb_dev_alloc((void **)&cg->p2, nb);
  if (e == hipSuccess && cg->grid_one)
    e = gb_dev_alloc((void **)&cg->slots, GB_CGP_SLOT_BYTES);
  if (e == hipSuccess)
    e = gb_dev_alloc((void **)&cg->partials, (size_t)cg->npartials * sizeof(double));
  if (e == hipSuccess)
    e = gb_dev_alloc((void **)&cg->partials2, (size_t)gb_cg_np2(cg) * sizeof(double));
  if (e == hipSuccess) e = gb_dev_alloc((void **)&cg->st, sizeof(gbd_cg_state));
  if (e == hipSuccess)
    e = hipHostMalloc((void **)&cg->h_st, sizeof(gbd_cg_state), hipHostMallocDefault);
  if (e == hipSuccess) e = hipMemsetAsync(cg->st, 0, sizeof(gbd_cg_state), gb_stream());
  if (e != hipSuccess) {
    gbd_cg_destroy(cg);
    return gb_hip_fail(e, "gbd_cg_create", __FILE__, __LINE__);
  }
  *out = cg;
  return GOOSEBERRY_SUCCESS;
}

void gbd_cg_destroy(gbd_cg *cg) {
  if (!cg || cg->noalloc) return;
  (void)hipStreamSynchronize(gb_stream());
  gb_cg_drop_graph(cg);
  (void)gb_dev_free(cg->r);
  (void)gb_dev_free(cg->p);
  (void)gb_dev_free(cg->ap);
  (void)gb_dev_free(cg->p2);
  (void)gb_dev_free(cg->slots);
  (void)gb_dev_free(cg->b0);
  (void)gb_dev_free(cg->partials);
  (void)gb_dev_free(cg->partials2);
  (void)gb_dev_free(cg->st);
  (void)gb_dev_free(cg->trace);
  if (cg->h_st) (void)hipHostFree(cg->h_st);
  if (cg->h_trace) (void)hipHostFree(cg->h_trace);
  free(cg);
}

int gbd_cg_start(gbd_cg *cg, const double *d_b, double *d_x, double tol,
                 int rel, uint64_t maxiter, uint32_t trace_cap) {
  hipStream_t s = gb_stream();
  if (trace_cap != cg->trace_cap) {
    GB_HIP(hipStreamSynchronize(s));
    gb_cg_drop_graph(cg);
    if (cg->trace) { GB_HIP(gb_dev_free(cg->trace)); cg->trace = nullptr; }
    if (cg->h_trace) { GB_HIP(hipHostFree(cg->h_trace)); cg->h_trace = nullptr; }
    if (trace_cap) {
      GB_HIP(gb_dev_alloc((void **)&cg->trace, (size_t)trace_cap * sizeof(double)));
      GB_HIP(hipHostMalloc((void **)&cg->h_trace, (size_t)trace_cap * sizeof(double),
                           hipHostMallocDefault));
    }
    cg->trace_cap = trace_cap;
  }
  if (cg->x != d_x) gb_cg_drop_graph(cg);
  if (!cg->m->cg_grid) cg->grid_one = 0;  // another workspace of the matrix gave up
  if (cg->grid_one && d_b == d_x) {
    // a run that gives up a wait starts again from b
    const size_t nb = (size_t)(cg->n ? cg->n : 1) * sizeof(double);
    if (!cg->b0) GB_HIP(gb_dev_alloc((void **)&cg->b0, nb));
    GB_HIP(hipMemcpyAsync(cg->b0, d_b, nb, hipMemcpyDeviceToDevice, s));
    d_b = cg->b0;
  }
  cg->b = d_b;
  cg->x = d_x;
  gb_cg_init<<<cg->grid_elem, GB_BLOCK, 0, s>>>(d_b, d_x, cg->r, cg->p, cg->n,
                                                cg->partials2);
  GB_LAUNCH_CHECK();
  gb_cg_init_state<<<1, GB_BLOCK, 0, s>>>(cg->partials2, cg->grid_elem, cg->st,
                                          tol, rel, (unsigned long long)maxiter);
  GB_LAUNCH_CHECK();
  return GOOSEBERRY_SUCCESS;
}

int gbd_cg_enqueue(gbd_cg *cg, uint32_t k) { return gb_cg_enqueue_raw(cg, k); }

// k iterations as replays of captured graphs of 2^i iterations (one graph
// per power of two, captured on first use and kept while x stays the same).
int gbd_cg_enqueue_graph(gbd_cg *cg, uint32_t k) {
  hipStream_t s = gb_stream();
  if (!gb_graphs_enabled() || cg->noalloc || cg->grid_one) return gb_cg_enqueue_raw(cg, k);
  if (cg->graph_x != cg->x) {
    gb_cg_drop_graph(cg);
    cg->graph_x = cg->x;
  }
  for (int i = GB_CG_NGRAPH - 1; i >= 0 && k; --i) {
    const uint32_t len = 1u << i;
    while (k >= len) {
      if (!cg->gexec[i]) {
        GB_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        int rv = gb_cg_enqueue_raw(cg, len);
        hipGraph_t g = nullptr;
        hipError_t e = hipStreamEndCapture(s, &g);
        if (rv != GOOSEBERRY_SUCCESS) {
          if (g) (void)hipGraphDestroy(g);
          return rv;
        }
        GB_HIP(e);
        cg->graph[i] = g;
        GB_HIP(hipGraphInstantiate(&cg->gexec[i], g, nullptr, nullptr, 0));
      }
      GB_HIP(hipGraphLaunch(cg->gexec[i], s));
      k -= len;
    }
  }
  return GOOSEBERRY_SUCCESS;
}

int gbd_cg_poll(gbd_cg *cg, gbd_cg_state *st, double *h_trace) {
  hipStream_t s = gb_stream();
  GB_HIP(hipMemcpyAsync(cg->h_st, cg->st, sizeof(gbd_cg_state),
                        hipMemcpyDeviceToHost, s));
  if (h_trace && cg->trace_cap)
    GB_HIP(hipMemcpyAsync(cg->h_trace, cg->trace,
                          (size_t)cg->trace_cap * sizeof(double),
                          hipMemcpyDeviceToHost, s));
  GB_HIP(hipStreamSynchronize(s));
  *st = *cg->h_st;
  // the last K3 of a stopped solve records its status before any K2 has
  // turned it into `done`
  if (st->status) st->done = 1;
  if (h_trace && cg->trace_cap)
    memcpy(h_trace, cg->h_trace, (size_t)cg->trace_cap * sizeof(double));
  return GOOSEBERRY_SUCCESS;
}

void gbd_matrix_cg_shape(const gbd_matrix *m, uint32_t *workgroups, uint32_t *rows) {
  *workgroups = m->cg_grid;
  *rows = m->cg_rows;
}

int gbd_cg_one_launch(const gbd_cg *cg) { return cg->grid_one != 0; }

void gbd_cg_several_launches(gbd_cg *cg) { cg->grid_one = cg->m->cg_grid = cg->m->cg_rows = 0; }

const double *gbd_cg_b(const gbd_cg *cg) { return cg->b; }

size_t gbd_cg_scratch_max() { return GB_CG_SCRATCH_BYTES; }

int gbd_cg_scratch(gbd_matrix *m, gbd_cg **out) {
  int rv = gb_ensure_init();
  if (rv != GOOSEBERRY_SUCCESS) return rv;
  if (m->nrows != m->ncols) return GOOSEBERRY_ERROR_INVALIDINPUT;
  gbd_cg *cg = &g_scratch_cg;
  memset(cg, 0, sizeof(*cg));
  if ((rv = gb_cg_geometry(cg, m)) != GOOSEBERRY_SUCCESS) return rv;
  auto al = [](uint64_t b) { return (b + 255) & ~(uint64_t)255; };
  const uint64_t nb = al((uint64_t)(cg->n ? cg->n : 1) * sizeof(double));
  const uint64_t o_p = nb, o_ap = 2 * nb, o_p2 = 3 * nb;
  const uint64_t o_b0 = 4 * nb, o_sl = 5 * nb;
  const uint64_t o_pa = cg->grid_one ? o_sl + GB_CGP_SLOT_BYTES : 3 * nb;
  const uint64_t o_pa2 = o_pa + al((uint64_t)cg->npartials * sizeof(double));
  const uint64_t o_st = o_pa2 + al((uint64_t)gb_cg_np2(cg) * sizeof(double));
  const uint64_t need = o_st + al(sizeof(gbd_cg_state));
  if (need > GB_CG_SCRATCH_BYTES) {
    gb_set_error("the allocation-free CG needs %llu bytes of workspace for this matrix "
                 "(%u rows); its device array holds %llu",
                 (unsigned long long)need, m->nrows, (unsigned long long)GB_CG_SCRATCH_BYTES);
    return GOOSEBERRY_ERROR_INVALIDINPUT;
  }
  unsigned char *base = nullptr;
  if ((rv = gb_cg_scratch_base(&base)) != GOOSEBERRY_SUCCESS) return rv;
  cg->r = (double *)base;
  cg->p = (double *)(base + o_p);
  cg->ap = (double *)(base + o_ap);
  if (cg->grid_one) {
    cg->p2 = (double *)(base + o_p2);
    cg->b0 = (double *)(base + o_b0);
    cg->slots = (uint64_t *)(base + o_sl);
  }
  cg->partials = (double *)(base + o_pa);
  cg->partials2 = (double *)(base + o_pa2);
  cg->st = (gbd_cg_state *)(base + o_st);
  cg->h_st = &g_scratch_hst;
  cg->noalloc = true;
  *out = cg;
  return GOOSEBERRY_SUCCESS;
}

}  // extern "C"
