// gb_batch.hip -- many independent CG solves advanced together.
//
// A batch holds up to max_slots systems, each a resident matrix (its own CSR
// and SpMV plan) with its own vectors, partial-sum arrays and state.  One
// device step advances every active system by one step with three launches
// over work lists:
//   K1 gb_b_spmv     (system, SpMV work item): Ap and one p.Ap partial per
//                    item, or in a refresh step the FP64 residual b - A x and
//                    its partials.  A column-split matrix runs over its
//                    slices into partial vectors (FP64 ones in refresh
//                    steps), which K2 adds; its refresh norm is tested in K3.
//                    A matrix with an x-tile plan has no items: its SpMV is a
//                    launch of its own (gb_b_spmv_xt, one partial per row
//                    block) after the list's.
//   K2 gb_b_update   (system, chunk of GB_BCHUNK rows): alpha, or the refreshed
//                    residual norm and the convergence test (every chunk adds
//                    the system's partials in the same order); x/r update
//                    and r.r partials, or the FP32 copy of a refreshed residual
//   K3 gb_b_pupdate  (system, chunk): beta (again from every chunk's own
//                    sum), stopping / refresh decision, p update
// Every sum of a system is taken over that system's own fixed decomposition
// (its SpMV plan, its chunks) in a fixed order, so a system gives the same
// bits alone and in any mix.
//
// Precision per system:
//   FP64  -- the reference's CG (src/cgd.c:40-129) in FP64.
//   MIXED -- FP32 matrix values and inner vectors (d, r, p, Ap), dot
//            products accumulated in FP64, and reliable updates: when the
//            FP32 recurrence residual has dropped by `delta` since the last
//            refresh (or reaches the tolerance), the step folds d into the
//            FP64 solution x and the next step recomputes r = b - A x with
//            the FP64 matrix; the Krylov direction p is kept.  Convergence
//            is only declared on the FP64 residual.
//   MIXED_JACOBI -- MIXED with the inner FP32 solve on the Jacobi-scaled
//            system D^-1/2 A D^-1/2 (D = diag(A)): the inner vectors live in
//            the scaled space (r^ = D^-1/2 r, x = D^-1/2 x^), the FP64
//            refreshes use A itself, and the refresh test compares the
//            scaled recurrence residual with its value at the last refresh.
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "gb_matrix.h"
#include "gb_xtile.h"

#define GB_BCHUNK 2048           // rows per elementwise work item
#define GB_BCHUNK_ITEMS (GB_BCHUNK / GB_BLOCK)
// The SpMV and elementwise launches get one workgroup per entry of their work
// lists, so items are dispatched in list order, as one launch per matrix
// would be.  The lists' allocations are resized when the lists outgrow them or
// shrink below a quarter of them.  Steps are replayed from graphs once the
// lists have stayed the same for GB_B_STABLE steps, and launched one by one
// before (the host keeps up).  So the kernels read nothing but their item
// first, where a graph that outlives the lists has them read the lists'
// lengths, and one dependent load less shows: 13.1 -> 11.6 us an SpMV.
#define GB_B_STABLE 128u
#define GB_BLIST_MIN 1024u
#define GB_B_NGRAPH 7

enum { GB_MODE_CG = 0, GB_MODE_REFRESH = 1 };

// One SpMV plan as the batched kernels read it: the system's own plan, or
// one column slice of a split matrix (its items numbered from `base`).
struct gb_bplan {
  const uint32_t *rowptr, *rowind, *blk, *wave_rows, *block_rows;
  const int16_t *dcol;  // the row blocks' 16-bit column offsets, or null
  const double *val;
  const float *val32;
  uint32_t nstream, nwave, nwaveblocks, nblockrows, nwork, exact, base, pad;
};

struct gb_bsys {
  gb_bplan pl;      // the matrix's plan (refresh steps, and every step when
                    // the matrix is not split)
  const gb_bplan *slices;  // column slices (nsplit of them) for CG steps
  void *ypart;      // nsplit * n partial products (FP32 for MIXED, else FP64)
  uint32_t nsplit, nwork_split;
  uint32_t n, nchunks;
  const double *b;
  double *x;        // solution (FP64 in both precisions)
  double *r, *p, *ap;  // FP64: residual, direction, A p.  MIXED: r = FP64
                       // residual of refresh steps; p, ap unused
  float *d32, *r32, *p32, *ap32;  // MIXED inner vectors
  double *part1;    // one partial per K1 work item
  double *part2;    // nchunks partials of K3
  double *part3;    // nchunks partials of ||b - A x||^2 (split matrices)
  gbd_bstate *st;
  const double *jscale;  // MIXED_JACOBI: D^-1/2, else null
  // an x-tile plan (xt.ptr non-null): the layout (the matrix's xt in FP64, its
  // xt32 in mixed precision) and the FP32 values of the inner solve (plain
  // or Jacobi-scaled)
  gb_xt xt;
  const float *xt_val32;
  int32_t precision;
  int32_t pad;
};

// The SpMV list is cut into segments, one launch each: segment k holds the
// items of column slice k of every split matrix, and segment 0 also the
// items of the matrices that are not split.  Launch boundaries make the GPU
// finish one slice of x before it starts gathering from the next.
struct gbd_batch {
  uint32_t max_slots;
  gb_bsys *d_sys;          // device table
  gb_bsys *h_sys;          // host mirror
  gbd_bstate *d_st;        // device states, one per slot
  gbd_bstate *h_st;        // pinned copy
  uint8_t *used;           // host: slot in use
  void **slot_mem;         // host: per-slot workspace allocation
  gbd_matrix **slot_mat;   // host: the matrix each used slot holds
  uint2 *d_spmv, *d_elem;  // device work lists: (system, item)
  uint4 *d_desc;  // per SpMV list entry: a row block's r0, r1, first entry, entries
  uint32_t cap_spmv, cap_elem;
  uint32_t nseg;                       // SpMV launches per step
  uint32_t seg[GB_SPLIT_MAX + 1];      // their parts of the SpMV list
  uint32_t lds;                        // gb_b_spmv's dynamic LDS (GB_SPMV_FEW_LDS or 0)
  uint32_t grid_elem;                  // the elementwise launches' grid
  uint32_t stable;                     // steps since the launches changed
  uint32_t *h_slice_nwork;             // host: max_slots x GB_SPLIT_MAX
  uint32_t *h_xt;                      // host: the active x-tile systems' slots
  uint32_t *h_xt_grid;                 // and their launch grids
  uint32_t *h_xt_lc;                   // and tile widths
  uint32_t n_xt;
  gb_bplan *d_slices;                  // max_slots x GB_SPLIT_MAX slice plans
  uint2 *h_spmv, *h_elem;              // pinned staging
  double delta;
  hipGraph_t graph[GB_B_NGRAPH];
  hipGraphExec_t gexec[GB_B_NGRAPH];
};

// ---------------------------------------------------------------- helpers

__device__ __forceinline__ double gb_b_sum_chunks(const double *part, uint32_t n,
                                                  double *red) {
  // same code and order in every workgroup of K2 and K3 and in the init reduction
  double s = 0.0;
#pragma unroll 1
  for (uint32_t base = 0; base < n; base += GB_BLOCK * 4) {
    double v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t i = base + j * GB_BLOCK + threadIdx.x;
      v[j] = i < n ? part[i] : 0.0;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) s += v[j];
  }
  s = gb_wave_sum(s);
  const int lane = threadIdx.x & (GB_WAVE - 1), wave = threadIdx.x / GB_WAVE;
  if (lane == 0) red[wave] = s;
  __syncthreads();
  double t = red[0];
#pragma unroll
  for (int w = 1; w < GB_WAVES_PER_BLOCK; ++w) t += red[w];
  __syncthreads();
  return t;
}

// One SpMV work item of system s (same bins and orders as gb_spmv_kernel).
// EPI 0: y = A x, dot += x[row] * y   (CG step; T = value/vector type)
// EPI 1: out = b - A x in FP64, dot += out^2   (refresh step; T = double)
// A row block's rows and entries come from its descriptor (d), filled when
// the work list is built, so the block's loads start without waiting on the
// plan's block table and row pointers.
template <typename T, int EPI>
__device__ __forceinline__ double gb_b_spmv_item(const gb_bplan &S, uint32_t w,
                                                 const T *__restrict__ val,
                                                 const T *__restrict__ x,
                                                 T *__restrict__ y,
                                                 const double *__restrict__ b,
                                                 T *prod, T *tred, const uint4 d) {
  const uint32_t tid = threadIdx.x;
  const uint32_t lane = tid & (GB_WAVE - 1), wave = tid / GB_WAVE;
  const uint32_t *__restrict__ rowptr = S.rowptr;
  const uint32_t *__restrict__ rowind = S.rowind;
  double dotp = 0.0;
  if (w < S.nstream) {
    const uint32_t r0 = d.x, r1 = d.y;
    const uint32_t k0 = d.z;
    const uint32_t cnt = d.w;
    const uint32_t ra = r0 + tid, rb = r0 + tid + GB_BLOCK;
    uint32_t pa0 = 0, pa1 = 0, pb0 = 0, pb1 = 0;
    T xa = 0, xb = 0;
    double ba = 0, bb = 0;
    if (ra < r1) {
      pa0 = rowptr[ra]; pa1 = rowptr[ra + 1];
      if (EPI == 0) xa = x[ra]; else ba = b[ra];
    }
    if (rb < r1) {
      pb0 = rowptr[rb]; pb1 = rowptr[rb + 1];
      if (EPI == 0) xb = x[rb]; else bb = b[rb];
    }
    if (cnt > 0) {
      const uint32_t klast = k0 + cnt - 1;
      // the matrix's plan decides between 16-bit offsets from r0 (plain
      // loads; FP32 values plain too) and 32-bit indices, as in
      // gb_spmv_kernel; the offsets are added at the gathers
      const int16_t *__restrict__ dcol = S.dcol;
      uint32_t c[GB_STREAM_ITERS];
      T v[GB_STREAM_ITERS], xv[GB_STREAM_ITERS];
      if (dcol) {
#pragma unroll
        for (int i = 0; i < GB_STREAM_ITERS; ++i) {
          if (i * GB_BLOCK < cnt) {
            uint32_t k = min(k0 + i * GB_BLOCK + tid, klast);
            c[i] = (uint32_t)(int32_t)dcol[k];
            if (sizeof(T) == 4) v[i] = val[k];
            else v[i] = __builtin_nontemporal_load(&val[k]);
          }
        }
      } else {
#pragma unroll
        for (int i = 0; i < GB_STREAM_ITERS; ++i) {
          if (i * GB_BLOCK < cnt) {
            uint32_t k = min(k0 + i * GB_BLOCK + tid, klast);
            c[i] = __builtin_nontemporal_load(&rowind[k]);
            v[i] = __builtin_nontemporal_load(&val[k]);
          }
        }
      }
      const T *xg = dcol ? x + r0 : x;
#pragma unroll
      for (int i = 0; i < GB_STREAM_ITERS; ++i)
        if (i * GB_BLOCK < cnt)
          xv[i] = xg[dcol ? (int64_t)(int32_t)c[i] : (int64_t)c[i]];
#pragma unroll
      for (int i = 0; i < GB_STREAM_ITERS; ++i) {
        uint32_t e = i * GB_BLOCK + tid;
        if (i * GB_BLOCK < cnt && e < cnt) prod[e] = v[i] * xv[i];
      }
    }
    __syncthreads();
    if (ra < r1) {
      T s = 0;
      for (uint32_t k = pa0 - k0; k < pa1 - k0; ++k) s += prod[k];
      if (EPI == 0) { y[ra] = s; dotp += (double)xa * (double)s; }
      else { double o = ba - (double)s; ((double *)y)[ra] = o; dotp += o * o; }
    }
    if (rb < r1) {
      T s = 0;
      for (uint32_t k = pb0 - k0; k < pb1 - k0; ++k) s += prod[k];
      if (EPI == 0) { y[rb] = s; dotp += (double)xb * (double)s; }
      else { double o = bb - (double)s; ((double *)y)[rb] = o; dotp += o * o; }
    }
    __syncthreads();
  } else if (w < S.nstream + S.nwaveblocks) {
    const uint32_t wid = (w - S.nstream) * GB_WAVES_PER_BLOCK + wave;
    if (wid < S.nwave) {
      const uint32_t row = S.wave_rows[wid];
      const uint32_t k0 = rowptr[row], k1 = rowptr[row + 1];
      T s = 0;
      if (S.exact) {
        for (uint32_t base = k0; base < k1; base += GB_WAVE) {
          const uint32_t k = base + lane;
          T pr = 0;
          if (k < k1) pr = val[k] * x[rowind[k]];
          const uint32_t cn = min((uint32_t)GB_WAVE, k1 - base);
          for (uint32_t j = 0; j < cn; ++j) s += gb_readlane(pr, j);
        }
      } else {
        s = gb_wave_sum(gb_row_lane_sum<T, GB_WAVE>(rowind, val, x, k0, k1, lane));
      }
      if (lane == 0) {
        if (EPI == 0) { y[row] = s; dotp += (double)x[row] * (double)s; }
        else { double o = b[row] - (double)s; ((double *)y)[row] = o; dotp += o * o; }
      }
    }
  } else {
    const uint32_t row = S.block_rows[w - S.nstream - S.nwaveblocks];
    const uint32_t k0 = rowptr[row], k1 = rowptr[row + 1];
    T s = 0;
    if (S.exact) {
      for (uint32_t base = k0; base < k1; base += GB_STREAM_LDS) {
        const uint32_t cn = min((uint32_t)GB_STREAM_LDS, k1 - base);
        for (uint32_t e = tid; e < cn; e += GB_BLOCK)
          prod[e] = val[base + e] * x[rowind[base + e]];
        __syncthreads();
        if (tid == 0)
          for (uint32_t e = 0; e < cn; ++e) s += prod[e];
        __syncthreads();
      }
    } else {
      s = gb_wave_sum(gb_row_lane_sum<T, GB_BLOCK>(rowind, val, x, k0, k1, tid));
      if (lane == 0) tred[wave] = s;
      __syncthreads();
      if (tid == 0) {
        T t = tred[0];
#pragma unroll
        for (int q = 1; q < GB_WAVES_PER_BLOCK; ++q) t += tred[q];
        s = t;
      }
      __syncthreads();
    }
    if (tid == 0) {
      if (EPI == 0) { y[row] = s; dotp += (double)x[row] * (double)s; }
      else { double o = b[row] - (double)s; ((double *)y)[row] = o; dotp += o * o; }
    }
  }
  return dotp;
}

// ----------------------------------------------------------------- kernels

// The descriptors of the SpMV list entries [a, b) of segment seg: for a
// row block (item below its plan's nstream), its first and last-plus-one
// rows, its first entry and its entry count.
__global__ void __launch_bounds__(GB_BLOCK)
gb_b_describe(const gb_bsys *__restrict__ sys, const uint2 *__restrict__ items,
              uint32_t a, uint32_t b, uint32_t seg, const gb_bplan *__restrict__ slice_tab,
              uint4 *__restrict__ desc) {
  for (uint32_t it = a + blockIdx.x * GB_BLOCK + threadIdx.x; it < b;
       it += gridDim.x * GB_BLOCK) {
    const uint32_t s = items[it].x, lw = items[it].y;
    const gb_bsys &S = sys[s];
    const gb_bplan &L = S.nsplit ? slice_tab[(size_t)s * GB_SPLIT_MAX + seg] : S.pl;
    uint4 d = make_uint4(0u, 0u, 0u, 0u);
    if (lw < L.nstream) {
      d.x = L.blk[2 * lw];
      d.y = L.blk[2 * lw + 1];
      d.z = L.rowptr[d.x];
      d.w = L.rowptr[d.y] - d.z;
    }
    desc[it] = d;
  }
}

// One workgroup per list entry (58 VGPRs: eight wavefronts per SIMD; fewer
// for scattered columns, GB_SPMV_FEW_LDS: 16 random systems of 4,096 to 2^20
// rows in mixed precision 14.2 -> 12.7 ms).  512 threads instead, half the
// loads and rows a thread, took the same time.
__global__ void __launch_bounds__(GB_BLOCK)
gb_b_spmv(const gb_bsys *__restrict__ sys, const uint2 *__restrict__ items,
          const uint4 *__restrict__ desc, uint32_t seg,
          const gbd_bstate *__restrict__ states, const gb_bplan *__restrict__ slice_tab) {
  __shared__ double prodd[GB_STREAM_LDS];
  __shared__ double tredd[GB_WAVES_PER_BLOCK];
  __shared__ double red[GB_WAVES_PER_BLOCK];
  const uint2 item = items[blockIdx.x];  // the segment's list, one item each
  const uint32_t s = item.x, lw = item.y;
  const uint4 d = desc[blockIdx.x];
  // the system, its state and its slice plan are addressed from the slot
  // alone, so their loads go out together
  const gb_bsys &S = sys[s];
  const gbd_bstate *st = states + s;
  if (st->done) return;  // not written during this kernel: uniform
  const int mode = st->mode_next;
  double dotp;
  uint32_t w = lw;  // the item's partial slot
  if (S.nsplit) {
    // a column-split matrix runs every step over its slices, slice r in
    // launch r, each into its partial vector: CG steps in the system's
    // precision, refresh steps A x in FP64 (the update kernel adds them)
    const uint32_t r = seg;
    const gb_bplan &L = slice_tab[(size_t)s * GB_SPLIT_MAX + r];
    w = L.base + lw;
    if (mode == GB_MODE_REFRESH) {
      double *yp = (double *)S.ypart + (size_t)r * S.n;
      dotp = gb_b_spmv_item<double, 0>(L, lw, L.val, S.x, yp, nullptr, prodd, tredd, d);
    } else if (S.precision != GOOSEBERRY_PRECISION_FP64) {
      float *yp = (float *)S.ypart + (size_t)r * S.n;
      dotp = gb_b_spmv_item<float, 0>(L, lw, L.val32, S.p32, yp, nullptr,
                                      (float *)prodd, (float *)tredd, d);
    } else {
      double *yp = (double *)S.ypart + (size_t)r * S.n;
      dotp = gb_b_spmv_item<double, 0>(L, lw, L.val, S.p, yp, nullptr, prodd, tredd, d);
    }
  } else if (mode == GB_MODE_REFRESH) {
    dotp = gb_b_spmv_item<double, 1>(S.pl, w, S.pl.val, S.x, S.r, S.b, prodd, tredd, d);
  } else if (S.precision != GOOSEBERRY_PRECISION_FP64) {
    dotp = gb_b_spmv_item<float, 0>(S.pl, w, S.pl.val32, S.p32, S.ap32, nullptr,
                                    (float *)prodd, (float *)tredd, d);
  } else {
    dotp = gb_b_spmv_item<double, 0>(S.pl, w, S.pl.val, S.p, S.ap, nullptr, prodd, tredd, d);
  }
  // one partial per work item
  const double bs = gb_block_sum(dotp, red);
  if (threadIdx.x == 0) S.part1[w] = bs;
}

// The SpMV of a system on an x-tile plan (grid = its row blocks): Ap and
// the p.Ap partials of a CG step in the system's precision, or in a
// refresh step the FP64 residual b - A x and its squared-norm partials;
// one partial per row block
// (WIDE: doubled tiles, which only FP64 systems have)
template <bool WIDE>
__global__ void __launch_bounds__(GB_XT_THREADS)
gb_b_spmv_xt(const gb_bsys *__restrict__ sys, uint32_t slot,
             const gbd_bstate *__restrict__ states) {
  __shared__ gb_xt_lds_t<WIDE> L;
  const gb_bsys &S = sys[slot];
  const gbd_bstate *st = states + slot;
  if (st->done) return;  // not written during this kernel: uniform
  if constexpr (!WIDE) {
    if (st->mode_next == GB_MODE_REFRESH) {
      gb_xt_spmv<double, GB_XT_RESID>(S.xt.ptr, S.xt.idx, S.xt.val, S.x, S.r, 1, S.b, S.part1,
                                      S.xt.rb, S.n, S.xt.T, S.xt.lc, L);
      return;
    }
    if (S.precision != GOOSEBERRY_PRECISION_FP64) {
      gb_xt_spmv<float, GB_XT_DOT>(S.xt.ptr, S.xt.idx, S.xt_val32, S.p32, S.ap32, 1, nullptr,
                                   S.part1, S.xt.rb, S.n, S.xt.T, S.xt.lc, L);
      return;
    }
  }
  gb_xt_spmv<double, GB_XT_DOT>(S.xt.ptr, S.xt.idx, S.xt.val, S.p, S.ap, 1, nullptr, S.part1,
                                S.xt.rb, S.n, S.xt.T, S.xt.lc, L);
}

// A thread's GB_BCHUNK_ITEMS rows of a whole chunk of an internal vector
// (256-byte aligned), as 16-byte words: word j of thread t is the chunk's
// word j GB_BLOCK + t, so consecutive lanes hold consecutive words.
template <typename T>
__device__ __forceinline__ uint32_t gb_b_row(uint32_t i0, int j, int q) {
  constexpr int N = 16 / sizeof(T);
  return i0 + (j * GB_BLOCK + threadIdx.x) * N + q;
}
template <typename T>
__device__ __forceinline__ void gb_b_ld(const T *__restrict__ v, uint32_t i0, T *o) {
  constexpr int N = 16 / sizeof(T);
  struct alignas(16) word { T e[N]; };
#pragma unroll
  for (int j = 0; j < GB_BCHUNK_ITEMS / N; ++j) {
    const word w = *(const word *)(v + gb_b_row<T>(i0, j, 0));
#pragma unroll
    for (int q = 0; q < N; ++q) o[j * N + q] = w.e[q];
  }
}
template <typename T>
__device__ __forceinline__ void gb_b_st(T *__restrict__ v, uint32_t i0, const T *o) {
  constexpr int N = 16 / sizeof(T);
  struct alignas(16) word { T e[N]; };
#pragma unroll
  for (int j = 0; j < GB_BCHUNK_ITEMS / N; ++j) {
    word w;
#pragma unroll
    for (int q = 0; q < N; ++q) w.e[q] = o[j * N + q];
    *(word *)(v + gb_b_row<T>(i0, j, 0)) = w;
  }
}

// The step's scalars and the x/r updates, one workgroup per chunk of rows,
// eight rows a thread.  Each workgroup issues the loads of its
// chunk, adds the system's SpMV partials itself (every one the same values in
// the same order, so the same alpha) while they are in flight, and updates its
// rows; chunk 0 records the scalars.  In a refresh step the sum is
// ||b - A x||^2 and every workgroup draws the same conclusion from it.
// (`done` may be set by chunk 0 while others start: they would decide to skip
// their rows as well.)  A system's last chunk, split systems and refresh steps
// go row by row.
//
// Bound: latency, on small systems: a launch, the dependent loads from the
// list to the vectors, and fetching the code itself, which every launch runs
// once.  48 Laplacians, per step: a reduction launch 4.2 us, the r update 10.0
// and the p update 7.9 us with eight rows' loads one after another; with those
// unrolled row by row 30 us in the update (128 registers, and code); as they
// are, with the reduction inside, 6.4 and 6.5 us.
__global__ void __launch_bounds__(GB_BLOCK)
gb_b_update(const gb_bsys *__restrict__ sys, const uint2 *__restrict__ items,
            gbd_bstate *states) {
  __shared__ double red[GB_WAVES_PER_BLOCK];
  __shared__ int32_t s_done;
  constexpr int J = GB_BCHUNK_ITEMS;
  const uint2 item = items[blockIdx.x];
  const uint32_t c = item.y;
  const gb_bsys &S = sys[item.x];
  gbd_bstate *st = states + item.x;
  const uint32_t n = S.n, nsplit = S.nsplit;
  const uint32_t i0 = c * GB_BCHUNK;
  const bool inside = n - i0 >= GB_BCHUNK;
  const uint32_t i1 = inside ? i0 + GB_BCHUNK : n;
  const bool mixed = S.precision != GOOSEBERRY_PRECISION_FP64;
  const int mode = st->mode_next;  // only gb_b_pupdate changes it
  const bool whole = mode == GB_MODE_CG && !nsplit && inside;
  if (threadIdx.x == 0) s_done = *(volatile int32_t *)&st->done;
  float rf[J], af[J];
  double rd[J], ad[J], pd[J], xd[J];
  if (whole) {
    if (mixed) {
      gb_b_ld(S.r32, i0, rf);
      gb_b_ld(S.ap32, i0, af);
    } else {
      gb_b_ld(S.r, i0, rd);
      gb_b_ld(S.ap, i0, ad);
      gb_b_ld(S.p, i0, pd);
      const double *const x = S.x;  // the caller's: aligned to 8 bytes
#pragma unroll
      for (int j = 0; j < J; ++j) xd[j] = x[gb_b_row<double>(i0, j / 2, j % 2)];
    }
  }
  const bool first = c == 0 && threadIdx.x == 0;
  double alpha = 0.0;
  if (nsplit && mode == GB_MODE_REFRESH) {
    // A x is still in slices: b - A x is formed below and its norm tested by
    // the p-update kernel
    __syncthreads();
    if (s_done) return;
    if (first) st->mode = mode;
  } else {
    // one partial per SpMV work item (per row block on an x-tile plan)
    const uint32_t np = S.xt.ptr ? S.xt.W : nsplit ? S.nwork_split : S.pl.nwork;
    const double t = gb_b_sum_chunks(S.part1, np, red);  // barriers inside
    if (s_done) return;
    int status = 0;
    if (mode == GB_MODE_REFRESH) {
      const double rn = sqrt(t);  // ||b - A x|| in FP64
      if (rn <= st->tol) status = 1;
      else if (!isfinite(rn)) status = 3;
      else if (st->final_refresh) status = 2;
      if (first) {
        st->mode = mode;
        st->nrefine += 1;
        st->rnorm64 = rn;
        st->rnorm_ref = rn;
      }
    } else {
      const double dr = st->dr;
      alpha = dr / t;
      if (!(t != 0.0) || !isfinite(alpha)) status = 3;
      if (first) {
        st->mode = mode;
        st->pap = t;
        st->alpha = alpha;
        if (!status) {
          st->dr_prev = dr;
          st->iter_next = st->iter + 1;
        }
      }
    }
    if (status) {
      if (first) {
        st->done = 1;
        st->status = status;
      }
      return;
    }
  }
  double d = 0.0;
  if (whole && mixed) {
    // d += a p is done by gb_b_pupdate, which reads p anyway
    const float a = (float)alpha;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      rf[j] = rf[j] - a * af[j];
      d += (double)rf[j] * (double)rf[j];
    }
    gb_b_st(S.r32, i0, rf);
  } else if (whole) {
    // src/cgd.c:92-100
    double *const x = S.x;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const double ps = alpha * pd[j];
      const uint32_t i = gb_b_row<double>(i0, j / 2, j % 2);
      x[i] = xd[j] + ps;
      const double aps = alpha * ad[j];
      rd[j] = rd[j] - aps;
      d += rd[j] * rd[j];
    }
    gb_b_st(S.r, i0, rd);
  } else if (mixed && mode == GB_MODE_REFRESH) {
    // r32 = (float) r64 from the refresh SpMV (for a split matrix r64 =
    // b - A x from the slices' FP64 partials, and its squared norm goes to
    // part3); d = 0 was set when x was updated
    const double *const yp = (const double *)S.ypart;
    double d64 = 0.0;
#pragma unroll 1
    for (uint32_t i = i0 + threadIdx.x; i < i1; i += GB_BLOCK) {
      double rr;
      if (nsplit) {
        double ax = yp[i];
        for (uint32_t r = 1; r < nsplit; ++r) ax += yp[(size_t)r * n + i];
        rr = S.b[i] - ax;
        S.r[i] = rr;
        d64 += rr * rr;
      } else {
        rr = S.r[i];
      }
      const float v = S.jscale ? (float)(S.jscale[i] * rr) : (float)rr;
      S.r32[i] = v;
      d += (double)v * (double)v;
    }
    if (nsplit) {
      const double b64 = gb_block_sum(d64, red);
      if (threadIdx.x == 0) S.part3[c] = b64;
      __syncthreads();
    }
  } else if (mixed) {
    const float a = (float)alpha;
    const float *const yp = (const float *)S.ypart;
#pragma unroll 1
    for (uint32_t i = i0 + threadIdx.x; i < i1; i += GB_BLOCK) {
      float ap;
      if (nsplit) {  // slice partials added in slice order
        ap = yp[i];
        for (uint32_t r = 1; r < nsplit; ++r) ap += yp[(size_t)r * n + i];
      } else {
        ap = S.ap32[i];
      }
      const float rn = S.r32[i] - a * ap;
      S.r32[i] = rn;
      d += (double)rn * (double)rn;
    }
  } else {
    const double *const yp = (const double *)S.ypart;
#pragma unroll 1
    for (uint32_t i = i0 + threadIdx.x; i < i1; i += GB_BLOCK) {
      double ap;
      if (nsplit) {
        ap = yp[i];
        for (uint32_t r = 1; r < nsplit; ++r) ap += yp[(size_t)r * n + i];
      } else {
        ap = S.ap[i];
      }
      const double ps = alpha * S.p[i];
      S.x[i] = S.x[i] + ps;
      const double aps = alpha * ap;
      const double rn = S.r[i] - aps;
      S.r[i] = rn;
      d += rn * rn;
    }
  }
  const double bs = gb_block_sum(d, red);
  if (threadIdx.x == 0) S.part2[c] = bs;
}

// beta, the stopping and refresh decisions and the p update; rows and loads as
// in gb_b_update.
__global__ void __launch_bounds__(GB_BLOCK)
gb_b_pupdate(const gb_bsys *__restrict__ sys, const uint2 *__restrict__ items,
             gbd_bstate *states, double delta) {
  __shared__ double red[GB_WAVES_PER_BLOCK];
  __shared__ int32_t s_done;
  constexpr int J = GB_BCHUNK_ITEMS;
  const uint2 item = items[blockIdx.x];
  const uint32_t c = item.y;
  const gb_bsys &S = sys[item.x];
  gbd_bstate *st = states + item.x;
  const uint32_t n = S.n, i0 = c * GB_BCHUNK;
  const bool mixed = S.precision != GOOSEBERRY_PRECISION_FP64;
  const bool whole = n - i0 >= GB_BCHUNK;
  const uint32_t i1 = whole ? i0 + GB_BCHUNK : n;
  // workgroup 0 of a system may set done during this kernel: decide once
  if (threadIdx.x == 0) s_done = *(volatile int32_t *)&st->done;
  const int mode = st->mode;
  float pf[J], df[J], rf[J];
  double pd[J], rd[J];
  if (whole && mode == GB_MODE_CG) {
    if (mixed) {
      gb_b_ld(S.p32, i0, pf);
      gb_b_ld(S.d32, i0, df);
      gb_b_ld(S.r32, i0, rf);
    } else {
      gb_b_ld(S.p, i0, pd);
      gb_b_ld(S.r, i0, rd);
    }
  }
  const double dnr = gb_b_sum_chunks(S.part2, S.nchunks, red);  // barriers inside
  if (s_done) return;
  if (mode == GB_MODE_REFRESH) {
    // MIXED only: restart the FP32 recurrence from the FP64 residual,
    // keep the direction p.  A split matrix's FP64 residual norm is
    // tested here (the update kernel tests the others').
    if (S.nsplit) {
      const double t = gb_b_sum_chunks(S.part3, S.nchunks, red);
      if (c == 0 && threadIdx.x == 0) {
        const double rn = sqrt(t);
        st->nrefine += 1;
        st->rnorm64 = rn;
        st->rnorm_ref = rn;
        if (rn <= st->tol) {
          st->done = 1;
          st->status = 1;
        } else if (!isfinite(rn)) {
          st->done = 1;
          st->status = 3;
        } else if (st->final_refresh) {
          st->done = 1;
          st->status = 2;
        }
      }
    }
    if (c == 0 && threadIdx.x == 0) {
      st->dr = dnr;
      st->rnorm = sqrt(dnr);
      st->inner = 0;
      st->mode_next = GB_MODE_CG;
      // the refresh test of a scaled system compares scaled residuals
      if (S.jscale) st->rnorm_ref = st->rnorm;
    }
    return;
  }
  // src/cgd.c:100-119 (and its FP32-inner counterpart)
  const double alpha = st->alpha;
  const double beta = dnr / st->dr_prev;
  const double rnorm = sqrt(dnr);
  const unsigned long long it1 = st->iter_next;
  const bool cap = st->maxiter && it1 >= st->maxiter;
  int status = 0;        // FP64: stop here
  bool refresh = false;  // MIXED: fold d into x, FP64 residual next step
  if (mixed) {
    if (!isfinite(dnr)) status = 3;
    // refresh after a drop by delta, or once the recurrence residual
    // predicts convergence (for a scaled system: it has dropped by
    // tol / ||b - A x|| since the last refresh)
    else if (rnorm <= delta * st->rnorm_ref || cap ||
             (S.jscale ? rnorm * st->rnorm64 <= st->tol * st->rnorm_ref
                       : rnorm <= st->tol))
      refresh = true;
  } else {
    if (rnorm <= st->tol) status = 1;
    else if (!isfinite(dnr)) status = 3;
    else if (cap) status = 2;
  }
  if (c == 0 && threadIdx.x == 0) {
    st->beta = beta;
    st->dr = dnr;
    st->rnorm = rnorm;
    st->iter = it1;
    st->inner += 1;
    if (status) {
      st->status = status;
      st->done = 1;
    }
    if (refresh) {
      st->mode_next = GB_MODE_REFRESH;
      if (cap) st->final_refresh = 1;
    }
  }
  if (status) return;
  if (mixed) {
    // this step's d += a p (the same float products and sums as beside
    // the r update, where it was one more read of p), then p = r + beta p.
    // A mixed system's CG step sets `done` above only on a non-finite
    // residual, after which x never takes d: a workgroup that sees that
    // flag early and skips its rows changes no result.
    const float a = (float)alpha;
    const float boa = (float)beta;
    if (whole && !refresh) {
#pragma unroll
      for (int j = 0; j < J; ++j) {
        df[j] = df[j] + a * pf[j];
        pf[j] = rf[j] + boa * pf[j];
      }
      gb_b_st(S.d32, i0, df);
      gb_b_st(S.p32, i0, pf);
    } else {
#pragma unroll 1
      for (uint32_t i = i0 + threadIdx.x; i < i1; i += GB_BLOCK) {
        const float pv = S.p32[i];
        const float dn = S.d32[i] + a * pv;
        S.p32[i] = S.r32[i] + boa * pv;
        if (refresh) {
          // the FP64 solution update
          S.x[i] = S.x[i] + (S.jscale ? S.jscale[i] * (double)dn : (double)dn);
          S.d32[i] = 0.0f;
        } else {
          S.d32[i] = dn;
        }
      }
    }
  } else {
    const double boa = beta / alpha;
    if (whole) {
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const double ps = alpha * pd[j];
        const double t = ps * boa;
        pd[j] = rd[j] + t;
      }
      gb_b_st(S.p, i0, pd);
    } else {
#pragma unroll 1
      for (uint32_t i = i0 + threadIdx.x; i < i1; i += GB_BLOCK) {
        const double ps = alpha * S.p[i];
        const double t = ps * boa;
        S.p[i] = S.r[i] + t;
      }
    }
  }
}

// Start of one system (not part of the step graph): x = 0, r = b, p = r
// (FP64) or r32 = p32 = (float) b, d = 0 (MIXED); chunk partials of b.b
// (part2) and of r32.r32 (part1, MIXED).
__global__ void __launch_bounds__(GB_BLOCK)
gb_b_init(const gb_bsys *__restrict__ sys, uint32_t slot) {
  __shared__ double red[GB_WAVES_PER_BLOCK];
  const gb_bsys &S = sys[slot];
  for (uint32_t c = blockIdx.x; c < S.nchunks; c += gridDim.x) {
    const uint32_t i0 = c * GB_BCHUNK;
    double d = 0.0, f = 0.0;
    for (int j = 0; j < GB_BCHUNK_ITEMS; ++j) {
      uint32_t i = i0 + j * GB_BLOCK + threadIdx.x;
      if (i < S.n) {
        double v = S.b[i];
        S.x[i] = 0.0;
        d += v * v;
        if (S.precision != GOOSEBERRY_PRECISION_FP64) {
          float vf = S.jscale ? (float)(S.jscale[i] * v) : (float)v;
          S.r32[i] = vf;
          S.p32[i] = vf;
          S.d32[i] = 0.0f;
          f += (double)vf * (double)vf;
        } else {
          S.r[i] = v;
          S.p[i] = v;
        }
      }
    }
    double bs = gb_block_sum(d, red);
    __syncthreads();
    double fs = gb_block_sum(f, red);
    if (threadIdx.x == 0) {
      S.part2[c] = bs;
      S.part1[c] = fs;
    }
    __syncthreads();
  }
}

__global__ void __launch_bounds__(GB_BLOCK)
gb_b_init_state(const gb_bsys *__restrict__ sys, uint32_t slot, double tol,
                int rel, unsigned long long maxiter) {
  __shared__ double red[GB_WAVES_PER_BLOCK];
  const gb_bsys &S = sys[slot];
  const double bb = gb_b_sum_chunks(S.part2, S.nchunks, red);
  const double ff = gb_b_sum_chunks(S.part1, S.nchunks, red);
  if (threadIdx.x == 0) {
    gbd_bstate *st = S.st;
    uint32_t *words = (uint32_t *)st;
    for (uint32_t i = 0; i < sizeof(gbd_bstate) / 4; ++i) words[i] = 0u;
    st->rnorm0 = sqrt(bb);
    st->tol = rel ? tol * st->rnorm0 : tol;
    st->maxiter = maxiter;
    st->precision = S.precision;
    st->mode = GB_MODE_CG;
    st->mode_next = GB_MODE_CG;
    if (S.precision != GOOSEBERRY_PRECISION_FP64) {
      st->dr = ff;
      st->rnorm = sqrt(ff);
      st->rnorm64 = st->rnorm0;
      st->rnorm_ref = S.jscale ? st->rnorm : st->rnorm0;
    } else {
      st->dr = bb;
      st->rnorm = st->rnorm0;
    }
    if (bb == 0.0) {
      st->done = 1;
      st->status = 1;
    } else if (!isfinite(bb)) {
      st->done = 1;
      st->status = 3;
    }
  }
}

// ------------------------------------------------------------------ host

static void gb_b_drop_graphs(gbd_batch *B) {
  B->stable = 0;
  for (int i = 0; i < GB_B_NGRAPH; ++i) {
    if (B->gexec[i]) (void)hipGraphExecDestroy(B->gexec[i]);
    if (B->graph[i]) (void)hipGraphDestroy(B->graph[i]);
    B->gexec[i] = nullptr;
    B->graph[i] = nullptr;
  }
}

static int gb_b_enqueue_raw(gbd_batch *B, uint32_t k) {
  hipStream_t s = gb_stream();
  for (uint32_t i = 0; i < k; ++i) {
    for (uint32_t g = 0; g < B->nseg; ++g) {
      const uint32_t a = B->seg[g], grid = B->seg[g + 1] - a;
      if (!grid) continue;  // only x-tile systems
      gb_b_spmv<<<grid, GB_BLOCK, B->lds, s>>>(B->d_sys, B->d_spmv + a, B->d_desc + a, g,
                                               B->d_st, B->d_slices);
      GB_LAUNCH_CHECK();
    }
    if (!B->grid_elem) continue;
    for (uint32_t j = 0; j < B->n_xt; ++j) {
      auto *k = gb_xt_is_wide(B->h_xt_lc[j]) ? gb_b_spmv_xt<true>
                                                          : gb_b_spmv_xt<false>;
      k<<<B->h_xt_grid[j], GB_XT_THREADS, 0, s>>>(B->d_sys, B->h_xt[j], B->d_st);
      GB_LAUNCH_CHECK();
    }
    gb_b_update<<<B->grid_elem, GB_BLOCK, 0, s>>>(B->d_sys, B->d_elem, B->d_st);
    GB_LAUNCH_CHECK();
    gb_b_pupdate<<<B->grid_elem, GB_BLOCK, 0, s>>>(B->d_sys, B->d_elem, B->d_st,
                                                      B->delta);
    GB_LAUNCH_CHECK();
  }
  return GOOSEBERRY_SUCCESS;
}

static uint32_t gb_b_nchunks(uint32_t n) { return (n + GB_BCHUNK - 1) / GB_BCHUNK; }

// Workspace of one system: byte offsets of its buffers inside one
// allocation (each 256-byte aligned); the same function sizes and carves it.
struct gb_b_layout {
  size_t part1, part2, part3, r, p, ap, d32, r32, p32, ap32, ypart, slices, total;
};

// SpMV items of the matrix's column slices (0 when it is not split)
static uint32_t gb_b_nwork_split(const gbd_matrix *m) {
  uint32_t t = 0;
  for (uint32_t r = 0; r < m->nsplit; ++r) t += gb_spmv_nwork(m->split[r]);
  return t;
}

static gb_b_layout gb_b_plan_layout(const gbd_matrix *m, int precision) {
  const size_t n = m->nrows ? m->nrows : 1;
  size_t nwork = m->nsplit ? gb_b_nwork_split(m) : gb_spmv_nwork(m);
  // (both x-tile layouts have the same number of row blocks)
  if (m->xt.ptr && m->xt.W > nwork) nwork = m->xt.W;
  const size_t nch = gb_b_nchunks(m->nrows);
  const size_t np1 = (nwork > nch ? nwork : nch) + 1;
  const size_t np2 = nch + 1;
  gb_b_layout L;
  memset(&L, 0xff, sizeof(L));
  size_t off = 0;
  auto take = [&](size_t nb) {
    size_t o = off;
    off += (nb + 255) & ~(size_t)255;
    return o;
  };
  L.part1 = take(np1 * 8);
  L.part2 = take(np2 * 8);
  L.r = take(n * 8);
  if (precision != GOOSEBERRY_PRECISION_FP64) {
    L.d32 = take(n * 4);
    L.r32 = take(n * 4);
    L.p32 = take(n * 4);
    L.ap32 = take(n * 4);
  } else {
    L.p = take(n * 8);
    L.ap = take(n * 8);
  }
  if (m->nsplit) {
    // FP64-sized: the refresh steps of a mixed system use it in FP64
    L.ypart = take((size_t)m->nsplit * n * 8);
    L.slices = take((size_t)m->nsplit * sizeof(gb_bplan));
    L.part3 = take((nch + 1) * 8);
  }
  L.total = off;
  return L;
}

static gb_bplan gb_b_plan_of(const gbd_matrix *m, uint32_t base, bool jacobi) {
  gb_bplan P;
  memset(&P, 0, sizeof(P));
  P.rowptr = m->rowptr;
  P.rowind = m->rowind;
  P.dcol = m->dcol;
  P.blk = m->blk;
  P.wave_rows = gb_wave_rows(m);
  P.block_rows = gb_block_rows(m);
  P.val = m->val;
  P.val32 = jacobi ? m->val32j : m->val32;
  P.nstream = m->nstream;
  P.nwave = m->nwave;
  P.nwaveblocks = gb_spmv_nwaveblocks(m);
  P.nblockrows = m->nblockrows;
  P.nwork = gb_spmv_nwork(m);
  P.exact = m->params.exact;
  P.base = base;
  return P;
}

extern "C" {

size_t gbd_batch_workspace_bytes(const gbd_matrix *m, int precision) {
  return gb_b_plan_layout(m, precision).total;
}

int gbd_batch_create(uint32_t max_slots, double delta, gbd_batch **out) {
  int rv = gb_ensure_init();
  if (rv != GOOSEBERRY_SUCCESS) return rv;
  if (max_slots == 0) return GOOSEBERRY_ERROR_INVALIDINPUT;
  gbd_batch *B = (gbd_batch *)calloc(1, sizeof(gbd_batch));
  if (!B) return GOOSEBERRY_ERROR_NOMEMORY;
  B->max_slots = max_slots;
  B->delta = delta > 0 && delta < 1 ? delta : 0.05;
  B->used = (uint8_t *)calloc(max_slots, 1);
  B->slot_mem = (void **)calloc(max_slots, sizeof(void *));
  B->slot_mat = (gbd_matrix **)calloc(max_slots, sizeof(gbd_matrix *));
  B->h_slice_nwork = (uint32_t *)calloc((size_t)max_slots * GB_SPLIT_MAX, sizeof(uint32_t));
  B->h_xt = (uint32_t *)calloc(max_slots, sizeof(uint32_t));
  B->h_xt_grid = (uint32_t *)calloc(max_slots, sizeof(uint32_t));
  B->h_xt_lc = (uint32_t *)calloc(max_slots, sizeof(uint32_t));
  B->h_sys = (gb_bsys *)calloc(max_slots, sizeof(gb_bsys));
  hipError_t e = gb_dev_alloc((void **)&B->d_sys, max_slots * sizeof(gb_bsys));
  if (e == hipSuccess) e = gb_dev_alloc((void **)&B->d_st, max_slots * sizeof(gbd_bstate));
  if (e == hipSuccess)
    e = hipHostMalloc((void **)&B->h_st, max_slots * sizeof(gbd_bstate), hipHostMallocDefault);
  if (e == hipSuccess)
    e = gb_dev_alloc((void **)&B->d_slices, (size_t)max_slots * GB_SPLIT_MAX * sizeof(gb_bplan));
  if (e == hipSuccess)
    e = hipMemsetAsync(B->d_st, 0, max_slots * sizeof(gbd_bstate), gb_stream());
  if (e == hipSuccess)
    e = hipMemsetAsync(B->d_sys, 0, max_slots * sizeof(gb_bsys), gb_stream());
  if (e != hipSuccess || !B->used || !B->slot_mem || !B->slot_mat || !B->h_sys ||
      !B->h_slice_nwork || !B->h_xt || !B->h_xt_grid || !B->h_xt_lc) {
    gbd_batch_destroy(B);
    return e != hipSuccess ? gb_hip_fail(e, "gbd_batch_create", __FILE__, __LINE__)
                           : GOOSEBERRY_ERROR_NOMEMORY;
  }
  *out = B;
  return GOOSEBERRY_SUCCESS;
}

void gbd_batch_destroy(gbd_batch *B) {
  if (!B) return;
  (void)hipStreamSynchronize(gb_stream());
  gb_b_drop_graphs(B);
  if (B->slot_mem)
    for (uint32_t i = 0; i < B->max_slots; ++i) (void)gb_dev_free(B->slot_mem[i]);
  if (B->slot_mat && B->used)
    for (uint32_t i = 0; i < B->max_slots; ++i)
      if (B->used[i] && B->slot_mat[i]) B->slot_mat[i]->holders--;
  (void)gb_dev_free(B->d_sys);
  (void)gb_dev_free(B->d_st);
  (void)gb_dev_free(B->d_slices);
  (void)gb_dev_free(B->d_spmv);
  (void)gb_dev_free(B->d_desc);
  (void)gb_dev_free(B->d_elem);
  if (B->h_st) (void)hipHostFree(B->h_st);
  if (B->h_spmv) (void)hipHostFree(B->h_spmv);
  if (B->h_elem) (void)hipHostFree(B->h_elem);
  free(B->used);
  free(B->slot_mem);
  free(B->slot_mat);
  free(B->h_slice_nwork);
  free(B->h_xt);
  free(B->h_xt_grid);
  free(B->h_xt_lc);
  free(B->h_sys);
  free(B);
}

int gbd_batch_add(gbd_batch *B, const gbd_matrix *m, const double *d_b,
                  double *d_x, double tol, int rel, uint64_t maxiter,
                  int precision, uint32_t *slot_out) {
  if (m->nrows != m->ncols) return GOOSEBERRY_ERROR_INVALIDINPUT;
  if (m->nparts) {
    gb_set_error("batched solves of a matrix held as row parts (64-bit row pointers) are "
                 "not supported");
    return GOOSEBERRY_ERROR_UNIMPLEMENTED;
  }
  if (precision != GOOSEBERRY_PRECISION_FP64 &&
      precision != GOOSEBERRY_PRECISION_MIXED &&
      precision != GOOSEBERRY_PRECISION_MIXED_JACOBI)
    return GOOSEBERRY_ERROR_INVALIDINPUT;
  const bool jac = precision == GOOSEBERRY_PRECISION_MIXED_JACOBI;
  if (precision == GOOSEBERRY_PRECISION_MIXED && !m->val32)
    return GOOSEBERRY_ERROR_INVALIDINPUT;
  if (jac && (!m->val32j || !m->jscale || (m->nsplit && !m->sval32j)))
    return GOOSEBERRY_ERROR_INVALIDINPUT;
  // an x-tile plan: the layout's copy of the inner solve's FP32 values
  if (m->xt.ptr && precision != GOOSEBERRY_PRECISION_FP64 &&
      !(jac ? m->xt_val32j : m->xt_val32))
    return GOOSEBERRY_ERROR_INVALIDINPUT;
  uint32_t slot = 0;
  while (slot < B->max_slots && B->used[slot]) ++slot;
  if (slot == B->max_slots) return GOOSEBERRY_ERROR_NOMEMORY;
  if (precision == GOOSEBERRY_PRECISION_MIXED && m->nsplit && !m->sval32)
    return GOOSEBERRY_ERROR_INVALIDINPUT;
  const uint32_t nch = gb_b_nchunks(m->nrows);
  const gb_b_layout L = gb_b_plan_layout(m, precision);
  uint8_t *mem = nullptr;
  GB_HIP(gb_dev_alloc((void **)&mem, L.total));
  gb_bsys S;
  memset(&S, 0, sizeof(S));
  S.pl = gb_b_plan_of(m, 0, jac);
  S.jscale = jac ? m->jscale : nullptr;
  S.n = m->nrows;
  S.nchunks = nch;
  S.nsplit = m->nsplit;
  S.nwork_split = gb_b_nwork_split(m);
  S.b = d_b;
  S.x = d_x;
  S.part1 = (double *)(mem + L.part1);
  S.part2 = (double *)(mem + L.part2);
  S.r = (double *)(mem + L.r);
  if (precision != GOOSEBERRY_PRECISION_FP64) {
    S.d32 = (float *)(mem + L.d32);
    S.r32 = (float *)(mem + L.r32);
    S.p32 = (float *)(mem + L.p32);
    S.ap32 = (float *)(mem + L.ap32);
  } else {
    S.p = (double *)(mem + L.p);
    S.ap = (double *)(mem + L.ap);
  }
  S.st = B->d_st + slot;
  S.precision = precision;
  if (m->xt.ptr) {
    S.xt = precision == GOOSEBERRY_PRECISION_FP64 ? m->xt : m->xt32;
    S.xt_val32 = jac ? m->xt_val32j : m->xt_val32;
  }
  hipStream_t s = gb_stream();
  gb_bplan *hsl = nullptr;
  if (m->nsplit) {
    // the slices' plans, their items numbered after the matrix's own
    S.ypart = mem + L.ypart;
    S.slices = (const gb_bplan *)(mem + L.slices);
    S.part3 = (double *)(mem + L.part3);
    hsl = (gb_bplan *)calloc(m->nsplit, sizeof(gb_bplan));
    if (!hsl) {
      (void)gb_dev_free(mem);
      return GOOSEBERRY_ERROR_NOMEMORY;
    }
    uint32_t base = 0;
    for (uint32_t r = 0; r < m->nsplit; ++r) {
      hsl[r] = gb_b_plan_of(m->split[r], base, jac);
      base += hsl[r].nwork;
      B->h_slice_nwork[(size_t)slot * GB_SPLIT_MAX + r] = hsl[r].nwork;
    }
    hipError_t e = hipMemcpyAsync(mem + L.slices, hsl, m->nsplit * sizeof(gb_bplan),
                                  hipMemcpyHostToDevice, s);
    if (e == hipSuccess)
      e = hipMemcpyAsync(B->d_slices + (size_t)slot * GB_SPLIT_MAX, hsl,
                         m->nsplit * sizeof(gb_bplan), hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    free(hsl);
    if (e != hipSuccess) {
      (void)gb_dev_free(mem);
      return gb_hip_fail(e, "gbd_batch_add slices", __FILE__, __LINE__);
    }
  }
  B->h_sys[slot] = S;
  GB_HIP(hipMemcpyAsync(B->d_sys + slot, &B->h_sys[slot], sizeof(gb_bsys),
                        hipMemcpyHostToDevice, s));
  uint32_t g = nch > 1024 ? 1024 : (nch ? nch : 1);
  gb_b_init<<<g, GB_BLOCK, 0, s>>>(B->d_sys, slot);
  GB_LAUNCH_CHECK();
  gb_b_init_state<<<1, GB_BLOCK, 0, s>>>(B->d_sys, slot, tol, rel,
                                         (unsigned long long)maxiter);
  GB_LAUNCH_CHECK();
  // the staging copy of h_sys[slot] must not change before the copy runs
  GB_HIP(hipStreamSynchronize(s));
  B->used[slot] = 1;
  B->slot_mem[slot] = mem;
  // the slot's descriptor holds the plan's arrays: no replan or free of the
  // matrix until the slot is removed
  B->slot_mat[slot] = const_cast<gbd_matrix *>(m);
  B->slot_mat[slot]->holders++;
  *slot_out = slot;
  return GOOSEBERRY_SUCCESS;
}

int gbd_batch_remove(gbd_batch *B, uint32_t slot) {
  if (slot >= B->max_slots || !B->used[slot]) return GOOSEBERRY_ERROR_INVALIDINPUT;
  // ordered after the steps already queued that still read the workspace
  GB_HIP(gb_dev_free(B->slot_mem[slot]));
  B->slot_mem[slot] = nullptr;
  B->used[slot] = 0;
  if (B->slot_mat[slot]) B->slot_mat[slot]->holders--;
  B->slot_mat[slot] = nullptr;
  return GOOSEBERRY_SUCCESS;
}

// Rebuild the work lists from the active slots (active[i] != 0 and in use).
int gbd_batch_commit(gbd_batch *B, const uint8_t *active) {
  hipStream_t s = gb_stream();
  uint64_t ns = 0, ne = 0;
  for (uint32_t i = 0; i < B->max_slots; ++i) {
    if (!B->used[i] || (active && !active[i])) continue;
    if (!B->h_sys[i].xt.ptr)
      ns += B->h_sys[i].nsplit ? B->h_sys[i].nwork_split : B->h_sys[i].pl.nwork;
    ne += B->h_sys[i].nchunks;
  }
  if (ns > 0xffffffffull || ne > 0xffffffffull) return GOOSEBERRY_ERROR_INVALIDINPUT;
  GB_HIP(hipStreamSynchronize(s));  // staging buffers are reused
  auto resize = [](uint64_t need, uint32_t cap) {
    return need > cap || (cap > 4 * GB_BLIST_MIN && need < cap / 4);
  };
  if (resize(ns, B->cap_spmv) || !B->d_spmv) {
    uint32_t cap = (uint32_t)(ns + ns / 2 + GB_BLIST_MIN);
    if (B->d_spmv) GB_HIP(gb_dev_free(B->d_spmv));
    if (B->d_desc) GB_HIP(gb_dev_free(B->d_desc));
    if (B->h_spmv) GB_HIP(hipHostFree(B->h_spmv));
    GB_HIP(gb_dev_alloc((void **)&B->d_spmv, (size_t)cap * 8));
    GB_HIP(gb_dev_alloc((void **)&B->d_desc, (size_t)cap * sizeof(uint4)));
    GB_HIP(hipHostMalloc((void **)&B->h_spmv, (size_t)cap * 8, hipHostMallocDefault));
    B->cap_spmv = cap;
    gb_b_drop_graphs(B);  // the graphs hold the old list pointer
  }
  if (resize(ne, B->cap_elem) || !B->d_elem) {
    uint32_t cap = (uint32_t)(ne + ne / 2 + GB_BLIST_MIN);
    if (B->d_elem) GB_HIP(gb_dev_free(B->d_elem));
    if (B->h_elem) GB_HIP(hipHostFree(B->h_elem));
    GB_HIP(gb_dev_alloc((void **)&B->d_elem, (size_t)cap * 8));
    GB_HIP(hipHostMalloc((void **)&B->h_elem, (size_t)cap * 8, hipHostMallocDefault));
    B->cap_elem = cap;
    gb_b_drop_graphs(B);
  }
  // SpMV segments: slice k of every split matrix in segment k, the other
  // matrices in segment 0
  uint32_t nseg = 1;
  uint64_t cnt[GB_SPLIT_MAX] = {0};
  uint64_t scattered = 0, blocks = 0;  // items of row blocks of scattered columns, all items
  for (uint32_t i = 0; i < B->max_slots; ++i) {
    if (!B->used[i] || (active && !active[i])) continue;
    const gb_bsys &S = B->h_sys[i];
    if (S.xt.ptr) continue;  // launched on its own
    if (!S.nsplit) {
      scattered += B->slot_mat[i]->scattered && !S.pl.dcol ? S.pl.nstream : 0;
      blocks += S.pl.nwork;
    }
    if (S.nsplit) {
      if (S.nsplit > nseg) nseg = S.nsplit;
      for (uint32_t r = 0; r < S.nsplit; ++r)
        cnt[r] += B->h_slice_nwork[(size_t)i * GB_SPLIT_MAX + r];
    } else {
      cnt[0] += S.pl.nwork;
    }
  }
  // few workgroups per CU where that suits nearly all items (see the constant)
  const uint32_t lds = blocks && scattered * 10 >= blocks * 9 && nseg == 1 ? GB_SPMV_FEW_LDS : 0;
  bool regrid = nseg != B->nseg || ne != B->grid_elem || lds != B->lds;
  uint64_t a = 0, c = 0;
  for (uint32_t g = 0; g < nseg; ++g) {
    regrid = regrid || B->seg[g] != a || B->seg[g + 1] != a + cnt[g];
    B->seg[g] = (uint32_t)a;
    for (uint32_t i = 0; i < B->max_slots; ++i) {
      if (!B->used[i] || (active && !active[i])) continue;
      const gb_bsys &S = B->h_sys[i];
      uint32_t nw = 0;
      if (S.xt.ptr) nw = 0;
      else if (S.nsplit) nw = g < S.nsplit ? B->h_slice_nwork[(size_t)i * GB_SPLIT_MAX + g] : 0;
      else if (g == 0) nw = S.pl.nwork;
      for (uint32_t w = 0; w < nw; ++w) B->h_spmv[a++] = make_uint2(i, w);
    }
    B->seg[g + 1] = (uint32_t)a;
  }
  if (regrid) {
    B->grid_elem = (uint32_t)ne;
    B->nseg = nseg;
    B->lds = lds;
    gb_b_drop_graphs(B);  // the graphs hold the launch grids
  }
  // the x-tile systems' launches (the graphs hold them)
  uint32_t nx = 0;
  bool xchanged = false;
  for (uint32_t i = 0; i < B->max_slots; ++i) {
    if (!B->used[i] || (active && !active[i]) || !B->h_sys[i].xt.ptr) continue;
    xchanged = xchanged || nx >= B->n_xt || B->h_xt[nx] != i ||
               B->h_xt_grid[nx] != B->h_sys[i].xt.W || B->h_xt_lc[nx] != B->h_sys[i].xt.lc;
    B->h_xt[nx] = i;
    B->h_xt_grid[nx] = B->h_sys[i].xt.W;
    B->h_xt_lc[nx] = B->h_sys[i].xt.lc;
    ++nx;
  }
  if (xchanged || nx != B->n_xt) {
    B->n_xt = nx;
    gb_b_drop_graphs(B);
  }
  for (uint32_t i = 0; i < B->max_slots; ++i) {
    if (!B->used[i] || (active && !active[i])) continue;
    for (uint32_t k = 0; k < B->h_sys[i].nchunks; ++k) {
      B->h_elem[c++] = make_uint2(i, k);
    }
  }
  if (ns) {
    GB_HIP(hipMemcpyAsync(B->d_spmv, B->h_spmv, ns * 8, hipMemcpyHostToDevice, s));
    for (uint32_t g = 0; g < nseg; ++g) {
      const uint32_t a0 = B->seg[g], a1 = B->seg[g + 1];
      if (a1 > a0) {
        uint32_t gr = gb_div_up(a1 - a0, GB_BLOCK);
        if (gr > 4096u) gr = 4096u;
        gb_b_describe<<<gr, GB_BLOCK, 0, s>>>(B->d_sys, B->d_spmv, a0, a1, g, B->d_slices,
                                              B->d_desc);
        GB_LAUNCH_CHECK();
      }
    }
  }
  if (ne) GB_HIP(hipMemcpyAsync(B->d_elem, B->h_elem, ne * 8, hipMemcpyHostToDevice, s));
  return GOOSEBERRY_SUCCESS;
}

// k steps, replayed from graphs of 2^i steps captured on first use once the
// launches have stayed the same.
int gbd_batch_step(gbd_batch *B, uint32_t k) {
  hipStream_t s = gb_stream();
  if (!B->d_spmv || !B->d_elem) return GOOSEBERRY_ERROR_INVALIDINPUT;
  if (!gb_graphs_enabled()) return gb_b_enqueue_raw(B, k);
  if (B->stable < GB_B_STABLE) {
    B->stable += k;
    return gb_b_enqueue_raw(B, k);
  }
  for (int i = GB_B_NGRAPH - 1; i >= 0 && k; --i) {
    const uint32_t len = 1u << i;
    while (k >= len) {
      if (!B->gexec[i]) {
        GB_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        int rv = gb_b_enqueue_raw(B, len);
        hipGraph_t g = nullptr;
        hipError_t e = hipStreamEndCapture(s, &g);
        if (rv != GOOSEBERRY_SUCCESS) {
          if (g) (void)hipGraphDestroy(g);
          return rv;
        }
        GB_HIP(e);
        B->graph[i] = g;
        GB_HIP(hipGraphInstantiate(&B->gexec[i], g, nullptr, nullptr, 0));
      }
      GB_HIP(hipGraphLaunch(B->gexec[i], s));
      k -= len;
    }
  }
  return GOOSEBERRY_SUCCESS;
}

int gbd_batch_poll(gbd_batch *B, gbd_bstate *states) {
  hipStream_t s = gb_stream();
  GB_HIP(hipMemcpyAsync(B->h_st, B->d_st, (size_t)B->max_slots * sizeof(gbd_bstate),
                        hipMemcpyDeviceToHost, s));
  GB_HIP(hipStreamSynchronize(s));
  memcpy(states, B->h_st, (size_t)B->max_slots * sizeof(gbd_bstate));
  return GOOSEBERRY_SUCCESS;
}

int gbd_batch_slot_used(const gbd_batch *B, uint32_t slot) {
  return slot < B->max_slots && B->used[slot];
}

}  // extern "C"
