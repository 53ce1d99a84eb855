// gb_matrix.h -- the device-resident CSR matrix and its SpMV plan.
#ifndef GB_MATRIX_H
#define GB_MATRIX_H

#include "gb_common.h"

// LDS staging buffer of one row block, in values.  window + short_max must
// not exceed it.
#define GB_STREAM_LDS 2304
#define GB_STREAM_ITERS (GB_STREAM_LDS / GB_BLOCK)

// An x-tile layout (C = 2^lc columns a tile): the entries grouped by (block
// of rows [rb[b], rb[b + 1]), tile), each group in CSR order; entry j of the
// layout is idx[j] = (row in block << lc) | (column in tile) with value
// val[j], group g = b T + t holding [ptr[g], ptr[g + 1])
struct gb_xt {
  uint32_t *rb;   // W + 1
  uint32_t *ptr;  // W T + 1; null without x tiles
  uint32_t *idx;  // nnz
  double *val;    // nnz
  uint32_t W, T, lc;
};

struct gbd_matrix {
  uint32_t nrows, ncols;
  uint64_t nnz;
  uint32_t *rowptr;   // nrows + 1
  uint32_t *rowind;   // nnz
  double *val;        // nnz
  float *val32;       // nnz, made on request (mixed precision)
  float *val32j;      // nnz, made on request: FP32 values of the Jacobi-scaled
                      // matrix D^-1/2 A D^-1/2 (D = diag(A))
  double *jscale;     // nrows, with val32j: D^-1/2
  gbd_plan_params params;
  // plan
  uint32_t nstream;     // LDS-staged row blocks
  uint32_t *blk;        // 2 * nstream: [row start, row end) per block
  uint4 *bdesc;         // nstream: a block's first row, end row, first entry
                        // and entry count, read by the SpMV in one load
  uint32_t nwave;       // rows processed one wavefront per row
  uint32_t nblockrows;  // rows processed one workgroup per row
  uint32_t *rowbins;    // stable bin permutation: short | wave | block rows
                        // (null when all rows are short)
  int16_t *dcol;        // nnz or null: row-block entries' column - (block's
                        // first row + cshift) (valid only in the row blocks)
  uint32_t cshift;      // 0, or a row part's first row in the whole matrix
                        // (its diagonal's column offset)
  // value-indexed plan (plan wide_values = 0, at most GB_VDICT_MAX distinct
  // values, no column split): each entry's value as an 8-bit index into a
  // table of the distinct values, read instead of val / val32 (vtab32 =
  // the FP32 roundings of vtab)
  uint8_t *vidx;        // nnz or null
  double *vtab;         // GB_VDICT_MAX
  float *vtab32;        // GB_VDICT_MAX, with val32
  uint32_t nvals;
  uint32_t pipe_grid;   // > 0: the SpMV runs the persistent pipelined
                        // row-block kernel on this many workgroups
  // x tiles (params.xtile = C): xt is what FP64 products read.  FP32 products
  // and the FP64 residuals of mixed solves read xt32, made with the FP32
  // values: tiles of C columns and blocks of equal rows always (its arrays
  // are xt's own where that has them too).  See gb_xtile_layout.
  gb_xt xt, xt32;
  float *xt_val32;      // nnz, with val32: its values in xt32's order
  float *xt_val32j;     // nnz, with val32j: its values in xt32's order
  uint64_t hist[33];
  // column split (params.csplit = P > 1): P views, view r holding the
  // entries of columns [r W, (r + 1) W), W = ceil(ncols / P), in row order;
  // the views share the arrays below (row pointers of view r start at
  // srowptr + r * nrows) and own only their plans
  uint32_t nsplit;
  gbd_matrix **split;
  uint32_t *srowptr;  // P * nrows + 1
  uint32_t *srowind;  // nnz
  double *sval;       // nnz
  float *sval32;      // nnz, with val32
  float *sval32j;     // nnz, with val32j
  double *ypart;      // P * nrows partial results (FP64, or FP32 in place)
  bool view;          // rowptr/rowind/val belong to a parent matrix
  // row parts (more entries than one part may hold, GB_PART_NNZ by
  // default): part q is rows [prow[q], prow[q + 1]) as a view whose 32-bit
  // row pointers (prowptr + prow[q] + q) count from its first entry
  // pbase[q], with a plan of its own; the parent keeps the 64-bit row
  // pointers and owns the indices and values (rowptr is null)
  bool part;          // this view is a row part (it owns its plan arrays)
  uint32_t nparts;
  gbd_matrix **parts;
  uint32_t *prow;     // host, nparts + 1
  uint64_t *pbase;    // host, nparts + 1
  uint32_t *prowptr;  // nrows + nparts
  uint64_t *rowptr64; // nrows + 1
  bool scattered;       // the short rows' columns jump from row to row
  // CG in one launch (gb_cg.hip): what the plan's first solve found
  bool cg_known;
  uint32_t cg_grid;     // workgroups, or 0: several launches an iteration
  uint32_t cg_rows;     // and rows per workgroup
  uint32_t holders;   // batch slots holding pointers into the plan: while
                      // nonzero the plan must not be rebuilt or freed
};

// the plan's wave rows and block rows
static inline const uint32_t *gb_wave_rows(const gbd_matrix *m) {
  return m->rowbins ? m->rowbins + (m->nrows - m->nwave - m->nblockrows) : nullptr;
}
static inline const uint32_t *gb_block_rows(const gbd_matrix *m) {
  return m->rowbins ? m->rowbins + (m->nrows - m->nblockrows) : nullptr;
}

#define GB_SPLIT_MAX 64
// columns of x an x-tile plan stages in LDS at most
#define GB_XT_CMAX 8192
// entries per row part of a matrix with 64-bit row pointers: every entry
// offset inside a part, and every offset a kernel forms past a part's last
// entry, stays below 2^32
#define GB_PART_NNZ (1ull << 31)
#define GB_VDICT_MAX 256

// One matrix entry's value: val[k], or vtab[vidx[k]] on a value-indexed
// plan (VD).  Plain FP64 values are streamed with non-temporal loads.
template <typename T, bool VD>
__device__ __forceinline__ T gb_ld_val(const T *__restrict__ val,
                                       const uint8_t *__restrict__ vidx,
                                       const T *__restrict__ vtab, uint32_t k) {
  if (VD) return vtab[vidx[k]];
  return __builtin_nontemporal_load(&val[k]);
}

// workgroups of the split sum (fixed, so the partial count is known)
static inline uint32_t gb_split_sum_grid(const gbd_matrix *m) {
  uint32_t g = (m->nrows + GB_BLOCK - 1) / GB_BLOCK;
  return g > 1024u ? 1024u : (g ? g : 1u);
}

// One lane's share of a row: the products val[k] * x[rowind[k]] for
// k = k0 + lane, k0 + lane + STRIDE, ... added in k order from +0.0.  Four
// strides of index and value loads, then their four gathers, are issued
// before the products are added, so a lane keeps four gathers in flight;
// the additions are those of the plain strided loop, in the same order.
template <typename T, uint32_t STRIDE, bool VD = false>
__device__ __forceinline__ T gb_row_lane_sum(const uint32_t *__restrict__ rowind,
                                             const T *__restrict__ val,
                                             const T *__restrict__ x, uint32_t k0,
                                             uint32_t k1, uint32_t lane,
                                             const uint8_t *__restrict__ vidx = nullptr,
                                             const T *__restrict__ vtab = nullptr) {
  T s = 0;
  uint32_t k = k0 + lane;
  for (; (uint64_t)k + 3 * STRIDE < k1; k += 4 * STRIDE) {
    const uint32_t c0 = __builtin_nontemporal_load(&rowind[k]);
    const uint32_t c1 = __builtin_nontemporal_load(&rowind[k + STRIDE]);
    const uint32_t c2 = __builtin_nontemporal_load(&rowind[k + 2 * STRIDE]);
    const uint32_t c3 = __builtin_nontemporal_load(&rowind[k + 3 * STRIDE]);
    const T v0 = gb_ld_val<T, VD>(val, vidx, vtab, k);
    const T v1 = gb_ld_val<T, VD>(val, vidx, vtab, k + STRIDE);
    const T v2 = gb_ld_val<T, VD>(val, vidx, vtab, k + 2 * STRIDE);
    const T v3 = gb_ld_val<T, VD>(val, vidx, vtab, k + 3 * STRIDE);
    const T x0 = x[c0], x1 = x[c1], x2 = x[c2], x3 = x[c3];
    s += v0 * x0;
    s += v1 * x1;
    s += v2 * x2;
    s += v3 * x3;
  }
  for (; k < k1; k += STRIDE) {
    const uint32_t c = __builtin_nontemporal_load(&rowind[k]);
    const T v = gb_ld_val<T, VD>(val, vidx, vtab, k);
    s += v * x[c];
  }
  return s;
}

// Launch geometry of one SpMV: stream blocks, then blocks of 4 wave rows,
// then one block per long row.
static inline uint32_t gb_spmv_nwaveblocks(const gbd_matrix *m) {
  return (m->nwave + GB_WAVES_PER_BLOCK - 1) / GB_WAVES_PER_BLOCK;
}
static inline uint32_t gb_spmv_nwork(const gbd_matrix *m) {
  return m->nstream + gb_spmv_nwaveblocks(m) + m->nblockrows;
}
// Row blocks whose columns scatter over x gather best from three workgroups of
// 256 threads per CU: with more, their gathers queue up in the caches.  These
// bytes of LDS, unused, on top of a row-block kernel's own (9 or 18 KB) keep
// it to three.  Taken where the rows' columns jump (gb_plan_classify: half of
// the short rows or more), the plan has no 16-bit offsets and nine of ten work
// items are row blocks.  Random matrices of 29 entries a row, FP32 / FP64 SpMV,
// at 8 and 3 workgroups: 100,000 rows 19.5 -> 18.5 / 21.1 -> 20.3 us, 300,007
// rows 52.9 -> 43.8 / 55.8 -> 49.6 us, 1,048,576 rows 200 -> 173 / 309 -> 306 us,
// in four column slices 216 -> 178 / 212 -> 188.  Wavefront rows (100 entries:
// 136 us at eight, 199 at three) want them all, and so do stencils whose
// offsets do not fit 16 bits (200 x 200 x 100 points 55.4 and 77.7 / 74.4 and
// 90.0 us) or were not asked for (160^3 points 59.2 and 85.1 / 76.5 and 95.6).
#define GB_SPMV_FEW_LDS 34000u
static inline uint32_t gb_spmv_few_lds(const gbd_matrix *m) {
  const bool few = m->scattered && !m->dcol &&
                   (uint64_t)m->nstream * 10 >= (uint64_t)gb_spmv_nwork(m) * 9;
  return few ? GB_SPMV_FEW_LDS : 0;
}
// workgroups of one SpMV launch (the number of p.Ap partials with DOT)
uint32_t gb_spmv_grid(const gbd_matrix *m);

// p.Ap partials written by one SpMV launch with DOT (one per workgroup)
static inline uint32_t gb_spmv_npartials(const gbd_matrix *m) {
  return (m->nsplit || m->nparts || m->xt.ptr) ? gb_split_sum_grid(m) : gb_spmv_grid(m);
}

// Enqueue y = A x; when cg != nullptr also write the per-workgroup partial
// sums of p.Ap (x = p, y = Ap) to partials[gb_spmv_npartials(m)].
int gb_spmv_launch(const gbd_matrix *m, const double *x, double *y,
                   uint32_t ystride, double *partials, const gbd_cg_state *cg);
int gb_spmv_launch_f32(const gbd_matrix *m, const float *x, float *y,
                       double *partials, const gbd_cg_state *cg);

#endif
