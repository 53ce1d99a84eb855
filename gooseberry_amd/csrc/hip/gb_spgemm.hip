// gb_spgemm.hip -- C = A B for sparse A and B (src/blas.c:94-234,609-791),
// bit for bit the reference's row-by-row scan.
//
// The reference walks row i of A entry by entry (j), and for each the row
// arowind[j] of B entry by entry (k): the product x_j * b_k goes to column
// browind[k] of C.  Each C element is the sum of its products in that scan
// order; in the sparse result the columns of a row appear in the order of
// their first product.  A row's products are numbered t = 0, 1, ... in that
// scan order.  Rows take one of three paths:
//
// Short rows (at most 64 products from at most 64 entries of A): a
// wavefront takes up to 16 of them one after another, lane t holding product
// t of the row.  The lanes enter their
// columns in a 128-slot LDS hash table, each slot keeping the mask of lanes
// with its column: a lane with no lower lane in its mask is the head of its
// column, and its sum is its own product followed by the other lanes' in
// the mask, added in lane (= t) order.  The heads in lane order are the
// columns in first-appearance order (a ballot gives each head its rank).
//
// Medium rows (at most 4096 distinct columns, by the lesser of the row's
// products and C's columns): one wavefront per row, 64 products a step
// in t order, the columns found so far in an LDS hash table with each
// column's rank (the order of its first product) and running sum.
//
// Other rows: every product is materialised at its position t (numbered
// over these rows, row-major), then
//   1. stable radix sort of t by column, then by row: (row, col, t) order
//   2. one sequential sum per (row, col) run, in t order
//   3. the runs sorted by their first t (unique, row-major), so each row
//      lists its columns by first appearance.
//
// All paths add a column's products one after another in t order: the
// first product, then += the others (the dense variant starts from +0.0 as
// the reference's zeroed row does, so a lone -0.0 becomes +0.0).  The sparse
// result needs each row's entry count before the rows can be placed: the
// short and medium rows write their entries in first-appearance order to a
// staging area at the row's first product position (where all rows are short,
// a wavefront's rows follow one another there), with their counts; the
// scan of the counts gives the row pointers and a copy puts the staged rows
// in place.  (When the staging area would pass its limit, 8 GiB unless
// GOOSEBERRY_SPGEMM_STAGE_MAX says otherwise, these rows are counted in
// one pass and written in another instead.)
#include <stdlib.h>

#include "gb_common.h"

#define GB_SG_SHORT 64  // products (and A entries) of a short row

// Row classes: short rows, six classes of medium rows by the distinct
// columns their hash table must hold, and the rows of the sort path.  On
// random matrices of 29 entries a row (841 products, 60,000 rows) three
// classes (256, 1024, 4096) took 1.20 ms, these six 0.88 ms: a row in the
// smallest table that fits leaves LDS for more wavefronts.
#define GB_SG_NHASH 6
enum { GB_SG_CSHORT = 0, GB_SG_CHASH = 1, GB_SG_CSORT = GB_SG_CHASH + GB_SG_NHASH,
       GB_SG_NCLASS };
constexpr uint32_t gb_sg_cap[GB_SG_NHASH] = {256, 512, 1024, 1536, 2560, 4096};
constexpr uint32_t gb_sg_slots(uint32_t cap) { return cap * 3 / 2; }
// products and A entries of a medium row at most: one wavefront walks them
// alone, 64 in about half a microsecond, so a longer row would hold up the
// launch for more than half a millisecond
#define GB_SG_HASH_MAXP 65536u

enum { GB_SG_COUNT = 0, GB_SG_FILL = 1, GB_SG_DENSE = 2, GB_SG_STAGE = 3 };
#define GB_SG_STAGE_MAX (8ull << 30)  // bytes of staged short-row entries

// the staging limit: GOOSEBERRY_SPGEMM_STAGE_MAX (bytes; 0 turns staging
// off) when set, read at every product
static uint64_t gb_sg_stage_max() {
  const char *e = getenv("GOOSEBERRY_SPGEMM_STAGE_MAX");
  if (e && *e) {
    char *end = nullptr;
    const unsigned long long v = strtoull(e, &end, 10);
    if (end != e) return v;
  }
  return GB_SG_STAGE_MAX;
}

// products per A entry (the length of the B row it selects) and their total
__global__ void __launch_bounds__(GB_BLOCK)
gb_sg_len(uint64_t annz, const uint32_t *__restrict__ arowind,
          const uint32_t *__restrict__ browptr, uint32_t *__restrict__ len,
          unsigned long long *__restrict__ total) {
  __shared__ unsigned long long lds[GB_WAVES_PER_BLOCK];
  unsigned long long v = 0;
#pragma unroll 4
  for (uint64_t j = (uint64_t)blockIdx.x * GB_BLOCK + threadIdx.x; j < annz;
       j += (uint64_t)gridDim.x * GB_BLOCK) {
    const uint32_t l = arowind[j];
    const uint32_t n = browptr[l + 1] - browptr[l];
    len[j] = n;
    v += n;
  }
  v = gb_block_sum(v, lds);
  if (threadIdx.x == 0) atomicAdd(total, v);
}

// the class of every row and the rows in each class (off = exclusive scan
// of the products per A entry)
__global__ void __launch_bounds__(GB_BLOCK)
gb_sg_classify(uint32_t anrows, uint32_t bncols, const uint32_t *__restrict__ arowptr,
               const uint32_t *__restrict__ off, uint32_t *__restrict__ cls,
               uint32_t *__restrict__ count) {
  __shared__ uint32_t h[GB_SG_NCLASS];
  if (threadIdx.x < GB_SG_NCLASS) h[threadIdx.x] = 0;
  __syncthreads();
  for (uint32_t i = blockIdx.x * GB_BLOCK + threadIdx.x; i < anrows;
       i += gridDim.x * GB_BLOCK) {
    const uint32_t j0 = arowptr[i], j1 = arowptr[i + 1], m = j1 - j0;
    const uint32_t p = off[j1] - off[j0];
    const uint32_t d = p < bncols ? p : bncols;  // distinct columns at most
    uint32_t c;
    if (p <= GB_SG_SHORT && m <= GB_SG_SHORT) c = GB_SG_CSHORT;
    else if (p > GB_SG_HASH_MAXP || m > GB_SG_HASH_MAXP) c = GB_SG_CSORT;
    else {
      c = GB_SG_CSORT;
#pragma unroll
      for (int k = GB_SG_NHASH - 1; k >= 0; --k)
        if (d <= gb_sg_cap[k]) c = GB_SG_CHASH + k;
    }
    cls[i] = c;
    // one count per class and wavefront: by the lanes' masks
    for (uint64_t todo = __ballot(true); todo;) {
      const uint32_t k = (uint32_t)__builtin_amdgcn_readlane((int)c, __builtin_ctzll(todo));
      const uint64_t same = __ballot(c == k);
      if ((threadIdx.x & (GB_WAVE - 1)) == (uint32_t)__builtin_ctzll(same))
        atomicAdd(&h[k], (uint32_t)__popcll(same));
      todo &= ~same;
    }
  }
  __syncthreads();
  if (threadIdx.x < GB_SG_NCLASS && h[threadIdx.x])
    atomicAdd(&count[threadIdx.x], h[threadIdx.x]);
}

#define GB_SG_PER 16       // rows of a wavefront at most (one lane each for their bounds)
#define GB_SG_HASH_BITS 7
#define GB_SG_HASH (1u << GB_SG_HASH_BITS)  // slots per wavefront row (>= 2 x 64)
#define GB_SG_EMPTY 0xffffffffu            // no column reaches 2^32 - 1

// LDS operations of one wavefront complete in order; this keeps the
// compiler from moving them across the step and waits for them
__device__ __forceinline__ void gb_sg_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// a product and the next lane whose product goes to the same column (its own
// lane at the end): a column's products are walked by one 16-byte LDS read and
// four instructions each
struct __align__(16) gb_sg_link {
  double val;
  uint32_t next;
};

// Short rows, `per` consecutive list rows per wavefront (gb_sg_per).  A row is
// a chain of three loads (A's entries, the B rows' bounds, B's entries), so
// the next row's bounds and the one after's entries are loaded while a row's
// products are added.  COUNT: cnt[i] = distinct columns; FILL: the row's
// entries at crowptr[i]; DENSE: the sums into cdense row i; STAGE: cnt[i], and
// the row's entries at its first product position (pbase) with a list (other
// classes' rows are staged between), without one all rows of the wavefront
// one after another from the first one's position on: they have at most as
// many entries as products.  (A row
// to a wavefront, each staged at its own first product: 347 us for 729,000
// rows of 49 products and 25 columns, now 260; the stage's lines half empty,
// 124 us to put them in place, now 85.)
template <int MODE>
__global__ void __launch_bounds__(GB_BLOCK)
gb_sg_wave(uint32_t nlist, uint32_t per, const uint32_t *__restrict__ list,
           const uint32_t *__restrict__ arowptr, const uint32_t *__restrict__ arowind,
           const double *__restrict__ arowval, const uint32_t *__restrict__ browptr,
           const uint32_t *__restrict__ browind, const double *__restrict__ browval,
           const uint32_t *__restrict__ crowptr, uint32_t *__restrict__ cnt,
           uint32_t *__restrict__ crowind, double *__restrict__ crowval,
           double *__restrict__ cdense, uint32_t bncols,
           const uint32_t *__restrict__ pbase) {
  __shared__ uint32_t hkey[GB_WAVES_PER_BLOCK][GB_SG_HASH];
  __shared__ unsigned long long hmask[GB_WAVES_PER_BLOCK][GB_SG_HASH];
  __shared__ gb_sg_link hlink[GB_WAVES_PER_BLOCK][GB_WAVE];
  const uint32_t lane = threadIdx.x & (GB_WAVE - 1);
  const uint64_t w0 = ((uint64_t)blockIdx.x * GB_WAVES_PER_BLOCK + threadIdx.x / GB_WAVE) * per;
  if (w0 >= nlist) return;  // the whole wavefront
  const uint32_t nrow = (uint32_t)__builtin_amdgcn_readfirstlane(
      (int)(nlist - w0 < per ? (uint32_t)(nlist - w0) : per));
  uint32_t *key = hkey[threadIdx.x / GB_WAVE];
  unsigned long long *msk = hmask[threadIdx.x / GB_WAVE];
  gb_sg_link *lnk = hlink[threadIdx.x / GB_WAVE];
  // lane r < nrow: row r's number, A entries, place and entries
  uint32_t ri = 0, rj = 0, rm = 0, ro = 0, rcnt = 0;
  if (lane < nrow) {
    ri = list ? list[w0 + lane] : (uint32_t)w0 + lane;
    rj = arowptr[ri];
    rm = arowptr[ri + 1] - rj;
    if (MODE == GB_SG_FILL) ro = crowptr[ri];
    if (MODE == GB_SG_STAGE) ro = pbase[rj];
  }
  const bool placed = MODE == GB_SG_FILL || list;  // each row at its own place
  uint32_t o = (uint32_t)__builtin_amdgcn_readfirstlane((int)ro);
  // lane a < m: A entry a of a row (its column l, one row ahead), the B row
  // it selects and its value
  uint32_t l = 0, bstart = 0, bend = 0;
  double x = 0.0;
  auto load_a = [&](uint32_t r) {
    const uint32_t j0 = (uint32_t)__builtin_amdgcn_readlane((int)rj, (int)r);
    if (lane < (uint32_t)__builtin_amdgcn_readlane((int)rm, (int)r)) l = arowind[j0 + lane];
  };
  auto load_b = [&](uint32_t r) {
    const uint32_t j0 = (uint32_t)__builtin_amdgcn_readlane((int)rj, (int)r);
    bstart = bend = 0;
    if (lane < (uint32_t)__builtin_amdgcn_readlane((int)rm, (int)r)) {
      bstart = browptr[l];
      bend = browptr[l + 1];
      x = arowval[j0 + lane];
    }
  };
  load_a(0);
  load_b(0);
  if (nrow > 1) load_a(1);
  for (uint32_t r = 0; r < nrow; ++r) {
    const uint32_t m = (uint32_t)__builtin_amdgcn_readlane((int)rm, (int)r);
    const uint32_t blen = bend - bstart;
    const uint32_t incl = gb_wave_scan_incl(blen);
    const uint32_t excl = incl - blen;
    const uint32_t P = (uint32_t)__builtin_amdgcn_readlane((int)incl, GB_WAVE - 1);  // <= 64
    // product t = lane comes from the last A entry a whose products start at
    // or before t (entries selecting empty rows start where the next starts)
    uint32_t a = 0;
    for (uint32_t u = 0; u < m; ++u)
      if ((uint32_t)__builtin_amdgcn_readlane((int)excl, (int)u) <= lane) a = u;
    const uint32_t k0 =
        (uint32_t)__shfl((int)(bstart - excl), (int)a, GB_WAVE);  // mod 2^32
    const double x_a = __shfl(x, (int)a, GB_WAVE);
    const bool live = lane < P;
    uint32_t col = 0xffffffffu;
    double bv = 0.0;
    if (live) {
      const uint32_t k = k0 + lane;
      col = browind[k];
      bv = browval[k];
    }
    if (r + 1 < nrow) load_b(r + 1);
    if (r + 2 < nrow) load_a(r + 2);
    // the row's columns in a small LDS hash table: slot -> column and the
    // mask of lanes holding it; a lane is its column's head when no lower
    // lane is in the mask, and the head adds the other lanes' products in
    // lane (= scan) order, each lane naming the next
    key[lane] = GB_SG_EMPTY;
    key[lane + GB_WAVE] = GB_SG_EMPTY;
    msk[lane] = 0ull;
    msk[lane + GB_WAVE] = 0ull;
    gb_sg_wave_sync();
    uint32_t slot = 0;
    if (live) {
      uint32_t h = (col * 2654435761u) >> (32 - GB_SG_HASH_BITS);
      for (;;) {  // at most 64 columns in 128 slots: a free or equal slot exists
        const uint32_t prev = atomicCAS(&key[h], GB_SG_EMPTY, col);
        if (prev == GB_SG_EMPTY || prev == col) break;
        h = (h + 1) & (GB_SG_HASH - 1);
      }
      slot = h;
      atomicOr(&msk[slot], 1ull << lane);
    }
    gb_sg_wave_sync();
    const unsigned long long mk = live ? msk[slot] : 0ull;
    const bool head = live && (mk & ((1ull << lane) - 1ull)) == 0;
    double sum = 0.0;
    if (MODE != GB_SG_COUNT) {
      const double val = x_a * bv;
      const unsigned long long rest = mk & ~((2ull << lane) - 1ull);  // lanes above this one
      uint32_t next = rest ? (uint32_t)__builtin_ctzll(rest) : lane;
      lnk[lane] = {val, next};
      gb_sg_wave_sync();
      if (head) {
        sum = MODE == GB_SG_DENSE ? 0.0 + val : val;
        for (uint32_t at = lane; next != at;) {
          at = next;
          const gb_sg_link q = lnk[at];
          sum += q.val;
          next = q.next;
        }
      }
    }
    const uint64_t heads = __ballot(head);
    const uint32_t n = (uint32_t)__popcll(heads);
    if (lane == r) rcnt = n;
    if (MODE == GB_SG_FILL || MODE == GB_SG_STAGE) {
      if (placed) o = (uint32_t)__builtin_amdgcn_readlane((int)ro, (int)r);
      if (head) {
        const uint32_t at = o + (uint32_t)__popcll(heads & ((1ull << lane) - 1ull));
        crowind[at] = col;
        crowval[at] = sum;
      }
      o += n;
    }
    if (MODE == GB_SG_DENSE && head)
      cdense[(size_t)(uint32_t)__builtin_amdgcn_readlane((int)ri, (int)r) * bncols + col] = sum;
    gb_sg_wave_sync();
  }
  if ((MODE == GB_SG_COUNT || MODE == GB_SG_STAGE) && lane < nrow) cnt[ri] = rcnt;
}

// One wavefront (and workgroup) per medium row of at most CAP distinct
// columns.  A entries are taken 64 at a time: a scan of their B rows' lengths
// numbers the products, and 64 consecutive products at a time are formed,
// one per lane, the next 64 loaded while these are added.  A lane finds its
// column's slot in the hash table (linear probing, compare-and-swap); new
// columns take ranks in lane order.  When every lane holds a column of its
// own (each lane writes its number into its slot and reads it back), one
// read, add and write of the sums does; otherwise the lowest lane of each
// shared column adds the others' products in lane order.  LDS operations of
// a wavefront complete in order, so the steps' additions to a column keep
// t order.
//
// Bound: a chain of about a dozen dependent LDS operations per 64 products;
// the table's size decides how many wavefronts a CU holds to overlap them,
// hence the classes and the load of two thirds.  The sort path, which took
// these rows before, moves each product through global memory about 20 times:
// a product of random matrices of 29 entries a row (60,000 rows, 50 million
// products) and its first SpMV took 10.6 ms, and take 2.04 ms.
template <uint32_t CAP, uint32_t SLOTS, int MODE>
__global__ void __launch_bounds__(GB_WAVE)
gb_sg_hash(const uint32_t *__restrict__ list, const uint32_t *__restrict__ arowptr,
           const uint32_t *__restrict__ arowind, const double *__restrict__ arowval,
           const uint32_t *__restrict__ browptr, const uint32_t *__restrict__ browind,
           const double *__restrict__ browval, const uint32_t *__restrict__ crowptr,
           uint32_t *__restrict__ cnt, uint32_t *__restrict__ crowind,
           double *__restrict__ crowval, double *__restrict__ cdense, uint32_t bncols,
           const uint32_t *__restrict__ pbase) {
  static_assert(CAP <= 65536 && SLOTS > CAP, "16-bit ranks, and a free slot always");
  __shared__ uint32_t key[SLOTS];
  __shared__ double sum[MODE == GB_SG_COUNT ? 1 : CAP];
  __shared__ double bx[GB_WAVE];      // A entry: its value
  __shared__ uint32_t boff[GB_WAVE];  // A entry: B position of product t, less t
  __shared__ uint32_t mark[GB_WAVE];
  __shared__ uint16_t rnk[SLOTS];
  __shared__ uint8_t tag[SLOTS];
  const uint32_t lane = threadIdx.x;
  const unsigned long long below = (1ull << lane) - 1ull;
  const uint32_t i =
      (uint32_t)__builtin_amdgcn_readfirstlane((int)(list ? list[blockIdx.x] : blockIdx.x));
  const uint32_t j0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)arowptr[i]);
  const uint32_t m = (uint32_t)__builtin_amdgcn_readfirstlane((int)arowptr[i + 1]) - j0;
  uint32_t o = 0;  // the row's place in crowind and crowval
  if (MODE == GB_SG_FILL) o = (uint32_t)__builtin_amdgcn_readfirstlane((int)crowptr[i]);
  if (MODE == GB_SG_STAGE) o = (uint32_t)__builtin_amdgcn_readfirstlane((int)pbase[j0]);
  for (uint32_t q = lane; q < SLOTS; q += GB_WAVE) key[q] = GB_SG_EMPTY;
  uint32_t ndist = 0;
  for (uint32_t jb = 0; jb < m; jb += GB_WAVE) {
    uint32_t bstart = 0, blen = 0;
    double x = 0.0;
    if (jb + lane < m) {
      const uint32_t l = arowind[j0 + jb + lane];
      x = arowval[j0 + jb + lane];
      bstart = browptr[l];
      blen = browptr[l + 1] - bstart;
    }
    const uint32_t incl = gb_wave_scan_incl(blen);
    const uint32_t excl = incl - blen;
    const uint32_t P = (uint32_t)__builtin_amdgcn_readlane((int)incl, GB_WAVE - 1);
    gb_sg_wave_sync();
    boff[lane] = bstart - excl;
    bx[lane] = x;
    uint32_t acarry = 0;  // the A entry of the product before this step's first
    // the column and factors of product t = c0 + lane (loads only)
    auto fetch = [&](uint32_t c0, uint32_t &col, double &xa, double &bv) {
      gb_sg_wave_sync();
      mark[lane] = GB_SG_EMPTY;
      gb_sg_wave_sync();
      if (blen && excl - c0 < GB_WAVE) mark[excl - c0] = lane;
      gb_sg_wave_sync();
      const uint32_t mk = mark[lane];
      const unsigned long long at = __ballot(mk != GB_SG_EMPTY) & (below | (1ull << lane));
      const uint32_t from = (uint32_t)__shfl((int)mk, at ? 63 - __clzll(at) : 0, GB_WAVE);
      const uint32_t a = at ? from : acarry;
      acarry = (uint32_t)__builtin_amdgcn_readlane((int)a, GB_WAVE - 1);
      col = 0;
      xa = bv = 0.0;
      if (c0 + lane < P) {
        const uint32_t k = boff[a] + c0 + lane;
        col = browind[k];
        if (MODE != GB_SG_COUNT) {
          bv = browval[k];
          xa = bx[a];
        }
      }
    };
    uint32_t col = 0, ncol = 0;
    double xa = 0.0, bv = 0.0, nxa = 0.0, nbv = 0.0;
    if (P) fetch(0, ncol, nxa, nbv);
    for (uint32_t c0 = 0; c0 < P; c0 += GB_WAVE) {
      col = ncol;
      xa = nxa;
      bv = nbv;
      if (c0 + GB_WAVE < P) fetch(c0 + GB_WAVE, ncol, nxa, nbv);
      const bool live = c0 + lane < P;
      const double val = xa * bv;
      uint32_t slot = 0;
      bool won = false;
      if (live) {
        uint32_t h = __umulhi(col * 2654435761u, SLOTS);
        for (;;) {  // at most CAP < SLOTS columns: a free or equal slot exists
          const uint32_t prev = atomicCAS(&key[h], GB_SG_EMPTY, col);
          won = prev == GB_SG_EMPTY;
          if (won || prev == col) break;
          if (++h == SLOTS) h = 0;
        }
        slot = h;
        tag[slot] = (uint8_t)lane;
      }
      gb_sg_wave_sync();
      const unsigned long long dup = __ballot(live && tag[slot] != lane);
      unsigned long long newm = __ballot(won);    // lanes whose column is new
      unsigned long long lead = __ballot(live);   // lanes that write their column's sum
      for (unsigned long long todo = dup; todo;) {
        const uint32_t s = (uint32_t)__builtin_amdgcn_readlane((int)slot, __ffsll(todo) - 1);
        const unsigned long long grp = __ballot(live && slot == s);
        const unsigned long long first = grp & (0ull - grp);
        if (newm & grp) newm = (newm & ~grp) | first;
        lead = (lead & ~grp) | first;
        todo &= ~grp;
      }
      const bool isnew = (newm >> lane) & 1ull, leads = (lead >> lane) & 1ull;
      uint32_t r = 0;
      if (isnew) {
        r = ndist + (uint32_t)__popcll(newm & below);
        rnk[slot] = (uint16_t)r;
        if (MODE == GB_SG_FILL || MODE == GB_SG_STAGE) crowind[o + r] = col;
      } else if (leads) {
        r = rnk[slot];
      }
      ndist += (uint32_t)__popcll(newm);
      if (MODE != GB_SG_COUNT) {
        double acc = 0.0;
        if (isnew) acc = MODE == GB_SG_DENSE ? 0.0 + val : val;
        else if (leads) acc = sum[r] + val;
        for (unsigned long long todo = dup; todo;) {
          const uint32_t s = (uint32_t)__builtin_amdgcn_readlane((int)slot, __ffsll(todo) - 1);
          const unsigned long long grp = __ballot(live && slot == s);
          const uint32_t first = (uint32_t)__ffsll(grp) - 1;
          for (unsigned long long rest = grp & (grp - 1ull); rest; rest &= rest - 1ull) {
            const double v = gb_readlane(val, (uint32_t)__ffsll(rest) - 1);
            if (lane == first) acc += v;
          }
          todo &= ~grp;
        }
        if (leads) sum[r] = acc;
      }
      gb_sg_wave_sync();
    }
  }
  gb_sg_wave_sync();
  if ((MODE == GB_SG_COUNT || MODE == GB_SG_STAGE) && lane == 0) cnt[i] = ndist;
  if (MODE == GB_SG_FILL || MODE == GB_SG_STAGE)
    for (uint32_t q = lane; q < ndist; q += GB_WAVE) crowval[o + q] = sum[q];
  if (MODE == GB_SG_DENSE)
    for (uint32_t q = lane; q < SLOTS; q += GB_WAVE)
      if (key[q] != GB_SG_EMPTY) cdense[(size_t)i * bncols + key[q]] = sum[rnk[q]];
}

// the staged medium rows to their places, one wavefront per row
__global__ void __launch_bounds__(GB_BLOCK)
gb_sg_unstage_wave(uint32_t nlist, const uint32_t *__restrict__ list,
                   const uint32_t *__restrict__ arowptr, const uint32_t *__restrict__ pbase,
                   const uint32_t *__restrict__ cnt, const uint32_t *__restrict__ sind,
                   const double *__restrict__ sval, const uint32_t *__restrict__ crowptr,
                   uint32_t *__restrict__ crowind, double *__restrict__ crowval) {
  const uint32_t w = blockIdx.x * GB_WAVES_PER_BLOCK + threadIdx.x / GB_WAVE;
  if (w >= nlist) return;
  const uint32_t i = (uint32_t)__builtin_amdgcn_readfirstlane((int)(list ? list[w] : w));
  const uint32_t c = cnt[i], src = pbase[arowptr[i]], dst = crowptr[i];
  for (uint32_t q = threadIdx.x & (GB_WAVE - 1); q < c; q += GB_WAVE) {
    crowind[dst + q] = sind[src + q];
    crowval[dst + q] = sval[src + q];
  }
}

// the staged short rows to their places, one wavefront per gb_sg_wave
// wavefront of `per` list rows.  Without a list they lie one after another in
// the stage and in C, one copy; else four rows at a time, 16 lanes a row.
__global__ void __launch_bounds__(GB_BLOCK)
gb_sg_unstage(uint32_t nlist, uint32_t per, const uint32_t *__restrict__ list,
              const uint32_t *__restrict__ arowptr, const uint32_t *__restrict__ pbase,
              const uint32_t *__restrict__ cnt, const uint32_t *__restrict__ sind,
              const double *__restrict__ sval, const uint32_t *__restrict__ crowptr,
              uint32_t *__restrict__ crowind, double *__restrict__ crowval) {
  const uint32_t lane = threadIdx.x & (GB_WAVE - 1);
  const uint64_t w0 = ((uint64_t)blockIdx.x * GB_WAVES_PER_BLOCK + threadIdx.x / GB_WAVE) * per;
  if (w0 >= nlist) return;
  const uint32_t nrow = (uint32_t)__builtin_amdgcn_readfirstlane(
      (int)(nlist - w0 < per ? (uint32_t)(nlist - w0) : per));
  if (!list) {
    const uint32_t i0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)w0);
    const size_t from = pbase[arowptr[i0]], to = crowptr[i0];
    const uint32_t n = crowptr[i0 + nrow] - (uint32_t)to;
#pragma unroll 4
    for (uint32_t q = lane; q < n; q += GB_WAVE) {
      crowind[to + q] = sind[from + q];
      crowval[to + q] = sval[from + q];
    }
    return;
  }
  uint32_t c = 0, src = 0, dst = 0;
  if (lane < nrow) {
    const uint32_t i = list[w0 + lane];
    c = cnt[i];
    src = pbase[arowptr[i]];
    dst = crowptr[i];
  }
  for (uint32_t r4 = 0; r4 < nrow; r4 += GB_WAVE / 16u) {
    const uint32_t r = r4 + lane / 16u;  // lanes from nrow on hold no entries
    const uint32_t n = (uint32_t)__shfl((int)c, (int)r, GB_WAVE);
    const size_t from = (uint32_t)__shfl((int)src, (int)r, GB_WAVE);
    const size_t to = (uint32_t)__shfl((int)dst, (int)r, GB_WAVE);
    for (uint32_t q = lane & 15u; q < n; q += 16u) {
      crowind[to + q] = sind[from + q];
      crowval[to + q] = sval[from + q];
    }
  }
}

// the row of A entry j: the last row i with arowptr[i] <= j
__device__ __forceinline__ uint32_t gb_sg_row_of(const uint32_t *arowptr, uint32_t nrows,
                                                 uint32_t j) {
  uint32_t lo = 0, hi = nrows - 1;
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo + 1) / 2;
    if (arowptr[mid] <= j) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// products per A entry of the sort path's rows (0 for other rows)
__global__ void __launch_bounds__(GB_BLOCK)
gb_sg_len_long(uint32_t anrows, uint64_t annz, const uint32_t *__restrict__ arowptr,
               const uint32_t *__restrict__ cls, const uint32_t *__restrict__ len,
               uint32_t *__restrict__ len2) {
  for (uint64_t j = (uint64_t)blockIdx.x * GB_BLOCK + threadIdx.x; j < annz;
       j += (uint64_t)gridDim.x * GB_BLOCK) {
    const uint32_t i = gb_sg_row_of(arowptr, anrows, (uint32_t)j);
    len2[j] = cls[i] == GB_SG_CSORT ? len[j] : 0u;
  }
}

// the products of A entry j (row i, column l) with B row l, at positions
// off[j] .. off[j] + len[j] - 1: their scan order
__global__ void __launch_bounds__(GB_BLOCK)
gb_sg_expand(uint32_t anrows, uint64_t annz, const uint32_t *__restrict__ arowptr,
             const uint32_t *__restrict__ arowind, const double *__restrict__ arowval,
             const uint32_t *__restrict__ browptr, const uint32_t *__restrict__ browind,
             const double *__restrict__ browval, const uint32_t *__restrict__ off,
             const uint32_t *__restrict__ len, uint32_t *__restrict__ erow,
             uint32_t *__restrict__ ecol, double *__restrict__ eval) {
  for (uint64_t j = (uint64_t)blockIdx.x * GB_BLOCK + threadIdx.x; j < annz;
       j += (uint64_t)gridDim.x * GB_BLOCK) {
    const uint32_t nk = len[j];
    if (!nk) continue;
    const uint32_t i = gb_sg_row_of(arowptr, anrows, (uint32_t)j);
    const uint32_t l = arowind[j];
    const double x = arowval[j];
    const uint32_t k0 = browptr[l];
    uint32_t t = off[j];
    for (uint32_t k = k0; k < k0 + nk; ++k, ++t) {
      erow[t] = i;
      ecol[t] = browind[k];
      eval[t] = x * browval[k];
    }
  }
}

__global__ void __launch_bounds__(GB_BLOCK)
gb_sg_gather_u32(uint32_t n, const uint32_t *__restrict__ idx,
                 const uint32_t *__restrict__ in, uint32_t *__restrict__ out) {
  for (uint32_t p = blockIdx.x * GB_BLOCK + threadIdx.x; p < n; p += gridDim.x * GB_BLOCK)
    out[p] = in[idx[p]];
}

// run starts of equal (row, col) in sorted order (ord = t sorted)
__global__ void __launch_bounds__(GB_BLOCK)
gb_sg_runflag(uint32_t n, const uint32_t *__restrict__ ord, const uint32_t *__restrict__ erow,
              const uint32_t *__restrict__ ecol, uint32_t *__restrict__ flag) {
  for (uint32_t p = blockIdx.x * GB_BLOCK + threadIdx.x; p < n; p += gridDim.x * GB_BLOCK) {
    uint32_t f = 1;
    if (p > 0) {
      const uint32_t a = ord[p - 1], b = ord[p];
      f = (erow[a] != erow[b] || ecol[a] != ecol[b]) ? 1u : 0u;
    }
    flag[p] = f;
  }
}

// start position of each run (runstart[run] = p)
__global__ void __launch_bounds__(GB_BLOCK)
gb_sg_runstart(uint32_t n, const uint32_t *__restrict__ flag,
               const uint32_t *__restrict__ rid, uint32_t *__restrict__ runstart) {
  for (uint32_t p = blockIdx.x * GB_BLOCK + threadIdx.x; p < n; p += gridDim.x * GB_BLOCK)
    if (flag[p]) runstart[rid[p]] = p;
}

// one sequential sum per run, in t order; the run's row, column, first t
template <bool DENSE>
__global__ void __launch_bounds__(GB_BLOCK)
gb_sg_runsum(uint32_t nruns, uint32_t n, const uint32_t *__restrict__ runstart,
             const uint32_t *__restrict__ ord, const uint32_t *__restrict__ erow,
             const uint32_t *__restrict__ ecol, const double *__restrict__ eval,
             uint32_t bncols, double *__restrict__ cdense, uint32_t *__restrict__ rrow,
             uint32_t *__restrict__ rcol, uint32_t *__restrict__ rfirst,
             double *__restrict__ rval) {
  for (uint32_t q = blockIdx.x * GB_BLOCK + threadIdx.x; q < nruns; q += gridDim.x * GB_BLOCK) {
    const uint32_t p0 = runstart[q], p1 = q + 1 < nruns ? runstart[q + 1] : n;
    const uint32_t t0 = ord[p0];
    double v;
    if (DENSE) {
      v = 0.0;
      for (uint32_t p = p0; p < p1; ++p) v += eval[ord[p]];
      cdense[(size_t)erow[t0] * bncols + ecol[t0]] = v;
    } else {
      v = eval[t0];
      for (uint32_t p = p0 + 1; p < p1; ++p) v += eval[ord[p]];
      rrow[q] = erow[t0];
      rcol[q] = ecol[t0];
      rfirst[q] = t0;
      rval[q] = v;
    }
  }
}

// runs are in (row, col) order: rbeg[r] = the first run of row r and
// cnt[r] = its number of runs, for every row that has runs (a row's runs
// are contiguous; its last one is found by binary search)
__global__ void __launch_bounds__(GB_BLOCK)
gb_sg_rowruns(uint32_t nruns, const uint32_t *__restrict__ rrow, uint32_t *__restrict__ rbeg,
              uint32_t *__restrict__ cnt) {
  for (uint32_t q = blockIdx.x * GB_BLOCK + threadIdx.x; q < nruns;
       q += gridDim.x * GB_BLOCK) {
    const uint32_t r = rrow[q];
    if (q == 0 || rrow[q - 1] != r) {
      uint32_t lo = q, hi = nruns - 1;
      while (lo < hi) {
        const uint32_t mid = lo + (hi - lo + 1) / 2;
        if (rrow[mid] == r) lo = mid; else hi = mid - 1;
      }
      rbeg[r] = q;
      cnt[r] = lo + 1 - q;
    }
  }
}

// runs in first-appearance order (ordr): run q is entry q - rbeg[r] of its
// row r (the order is row-major, so a row's runs are q = rbeg[r] ..)
__global__ void __launch_bounds__(GB_BLOCK)
gb_sg_out(uint32_t nruns, const uint32_t *__restrict__ ordr, const uint32_t *__restrict__ rrow,
          const uint32_t *__restrict__ rcol, const double *__restrict__ rval,
          const uint32_t *__restrict__ rbeg, const uint32_t *__restrict__ crowptr,
          uint32_t *__restrict__ crowind, double *__restrict__ crowval) {
  for (uint32_t q = blockIdx.x * GB_BLOCK + threadIdx.x; q < nruns; q += gridDim.x * GB_BLOCK) {
    const uint32_t sidx = ordr[q];
    const uint32_t r = rrow[sidx];
    const uint32_t o = crowptr[r] + (q - rbeg[r]);
    crowind[o] = rcol[sidx];
    crowval[o] = rval[sidx];
  }
}

__global__ void __launch_bounds__(GB_BLOCK)
gb_sg_zero(size_t n, double *__restrict__ c) {
  for (size_t i = (size_t)blockIdx.x * GB_BLOCK + threadIdx.x; i < n;
       i += (size_t)gridDim.x * GB_BLOCK)
    c[i] = 0.0;
}

static uint32_t gb_sg_grid(uint64_t n) {
  uint64_t g = (n + GB_BLOCK - 1) / GB_BLOCK;
  if (g > 65536) g = 65536;
  return g ? (uint32_t)g : 1u;
}

// short rows per wavefront: one until the launch fills the GPU's wavefronts
// (8192) twice, then more, so that their loads overlap and the stage is dense.
// The whole square of a 3D stencil of 729,000 rows took 1092 us at one row,
// 863 at 4, 857 at 8, 851 at 16; of 262,000 rows 603, 551, 545 and 549.
static uint32_t gb_sg_per(uint32_t nshort) {
  const uint32_t per = nshort / 16384u;
  return per < 1u ? 1u : (per > GB_SG_PER ? GB_SG_PER : per);
}
static uint32_t gb_sg_short_grid(uint32_t nshort) {
  return gb_div_up(nshort, GB_WAVES_PER_BLOCK * gb_sg_per(nshort));
}

// the medium rows of one class in one mode (dense and the staged or final
// arrays as the short rows' kernel takes them)
template <int MODE>
static hipError_t gb_sg_medium(const uint32_t *count, const uint32_t *list,
                               const uint32_t *arowptr, const uint32_t *arowind,
                               const double *arowval, const uint32_t *browptr,
                               const uint32_t *browind, const double *browval,
                               const uint32_t *crowptr, uint32_t *cnt, uint32_t *crowind,
                               double *crowval, double *cdense, uint32_t bncols,
                               const uint32_t *pbase) {
  uint32_t first = count[GB_SG_CSHORT];
  for (int c = 0; c < GB_SG_NHASH; ++c) {
    const uint32_t n = count[GB_SG_CHASH + c];
    if (!n) continue;
    auto *k = gb_sg_hash<gb_sg_cap[0], gb_sg_slots(gb_sg_cap[0]), MODE>;
    switch (c) {
      case 1: k = gb_sg_hash<gb_sg_cap[1], gb_sg_slots(gb_sg_cap[1]), MODE>; break;
      case 2: k = gb_sg_hash<gb_sg_cap[2], gb_sg_slots(gb_sg_cap[2]), MODE>; break;
      case 3: k = gb_sg_hash<gb_sg_cap[3], gb_sg_slots(gb_sg_cap[3]), MODE>; break;
      case 4: k = gb_sg_hash<gb_sg_cap[4], gb_sg_slots(gb_sg_cap[4]), MODE>; break;
      case 5: k = gb_sg_hash<gb_sg_cap[5], gb_sg_slots(gb_sg_cap[5]), MODE>; break;
    }
    k<<<n, GB_WAVE, 0, gb_stream()>>>(list ? list + first : nullptr, arowptr, arowind, arowval,
                                      browptr, browind, browval, crowptr, cnt, crowind,
                                      crowval, cdense, bncols, pbase);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    first += n;
  }
  return hipSuccess;
}

extern "C" {

int gbd_spgemm(uint32_t anrows, uint32_t ancols, uint32_t bncols,
               const uint32_t *d_arowptr, const uint32_t *d_arowind,
               const double *d_arowval, const uint32_t *d_browptr,
               const uint32_t *d_browind, const double *d_browval,
               double *d_cdense, uint32_t **d_crowptr, uint32_t **d_crowind,
               double **d_crowval, uint32_t *r_cnnz) {
  int rv = gb_ensure_init();
  if (rv != GOOSEBERRY_SUCCESS) return rv;
  const bool dense = d_cdense != nullptr;
  if (!dense && (!d_crowptr || !d_crowind || !d_crowval || !r_cnnz))
    return GOOSEBERRY_ERROR_INVALIDINPUT;
  hipStream_t s = gb_stream();
  uint32_t annz = 0, E = 0, nruns = 0, nshort = 0, nmed = 0, nlong = 0, cnnz = 0;
  uint32_t hcount[GB_SG_NCLASS] = {0};
  uint32_t *len = nullptr, *off = nullptr, *cls = nullptr, *count = nullptr,
           *list = nullptr, *mlist = nullptr, *len2 = nullptr, *off2 = nullptr, *erow = nullptr,
           *ecol = nullptr, *perm1 = nullptr, *row1 = nullptr, *ord = nullptr,
           *flag = nullptr, *rid = nullptr, *runstart = nullptr, *rrow = nullptr,
           *rcol = nullptr, *rfirst = nullptr, *ordr = nullptr, *rbeg = nullptr,
           *cnt = nullptr, *crowptr = nullptr, *crowind = nullptr, *sind = nullptr;
  double *eval = nullptr, *rval = nullptr, *crowval = nullptr, *sval = nullptr;
  unsigned long long e64 = 0, *tot = nullptr;
  bool staged = false, one_class = false;
  hipError_t he = hipSuccess;
#define GB_SG_TRY(call)                                         \
  do {                                                          \
    he = (call);                                                \
    if (he != hipSuccess) {                                     \
      rv = gb_hip_fail(he, #call, __FILE__, __LINE__);          \
      goto done;                                                \
    }                                                           \
  } while (0)
#define GB_SG_RV(call)                                          \
  do {                                                          \
    rv = (call);                                                \
    if (rv != GOOSEBERRY_SUCCESS) goto done;                    \
  } while (0)

  (void)ancols;
  if (dense && (uint64_t)anrows * bncols) {
    gb_sg_zero<<<gb_sg_grid((uint64_t)anrows * bncols), GB_BLOCK, 0, s>>>(
        (size_t)anrows * bncols, d_cdense);
    GB_SG_TRY(hipGetLastError());
  }
  GB_SG_TRY(gb_fetch(&annz, d_arowptr + anrows, 4));
  GB_SG_TRY(gb_dev_alloc((void **)&len, ((size_t)annz + 1) * 4));
  GB_SG_TRY(gb_dev_alloc((void **)&off, ((size_t)annz + 1) * 4));
  // every product position must fit 32 bits: the total in 64 bits first
  GB_SG_TRY(gb_dev_alloc((void **)&tot, 8));
  GB_SG_RV(gbd_zero(tot, 8));
  if (annz) {
    const uint32_t g = gb_sg_grid(annz);
    gb_sg_len<<<g > 1024u ? 1024u : g, GB_BLOCK, 0, s>>>(annz, d_arowind, d_browptr, len, tot);
    GB_SG_TRY(hipGetLastError());
  }
  GB_SG_TRY(gb_fetch(&e64, tot, 8));
  if (e64 > 0xfffffffeull) {
    rv = GOOSEBERRY_ERROR_INVALIDINPUT;
    goto done;
  }
  GB_SG_RV(gbd_scan_u32(len, off, annz, off + annz));
  // row classes, and the rows in class order unless they are all of one
  GB_SG_TRY(gb_dev_alloc((void **)&cls, ((size_t)anrows + 1) * 4));
  GB_SG_TRY(gb_dev_alloc((void **)&count, GB_SG_NCLASS * 4));
  GB_SG_TRY(gb_dev_alloc((void **)&cnt, ((size_t)anrows + 1) * 4));
  GB_SG_RV(gbd_zero(count, GB_SG_NCLASS * 4));
  if (anrows) {
    // few workgroups: each adds its counts to the same words (2,848 of them
    // took 37 us for 729,000 rows)
    const uint32_t g = gb_sg_grid(anrows);
    gb_sg_classify<<<g > 512u ? 512u : g, GB_BLOCK, 0, s>>>(anrows, bncols, d_arowptr, off,
                                                            cls, count);
    GB_SG_TRY(hipGetLastError());
  }
  GB_SG_TRY(gb_fetch(hcount, count, GB_SG_NCLASS * 4));
  nshort = hcount[GB_SG_CSHORT];
  nlong = hcount[GB_SG_CSORT];
  nmed = anrows - nshort - nlong;
  for (int c = 0; c < GB_SG_NCLASS; ++c) one_class |= hcount[c] == anrows;
  if (!one_class) {
    GB_SG_TRY(gb_dev_alloc((void **)&list, (size_t)anrows * 4));
    GB_SG_RV(gbd_countingsort_kv_unchecked(cls, nullptr, 0, GB_SG_NCLASS - 1, anrows, list,
                                           nullptr));
  }
  if (!dense) {
    if (nlong) GB_SG_RV(gbd_zero(cnt, ((size_t)anrows + 1) * 4));
    staged = e64 * 12 <= gb_sg_stage_max();
    if ((nshort || nmed) && staged) {
      GB_SG_TRY(gb_dev_alloc((void **)&sind, (size_t)e64 * 4));
      GB_SG_TRY(gb_dev_alloc((void **)&sval, (size_t)e64 * 8));
    }
    if (nshort && staged) {
      gb_sg_wave<GB_SG_STAGE><<<gb_sg_short_grid(nshort), GB_BLOCK, 0, s>>>(
          nshort, gb_sg_per(nshort), list, d_arowptr, d_arowind, d_arowval, d_browptr,
          d_browind, d_browval, nullptr, cnt, sind, sval, nullptr, 0, off);
      GB_SG_TRY(hipGetLastError());
    } else if (nshort) {
      gb_sg_wave<GB_SG_COUNT><<<gb_sg_short_grid(nshort), GB_BLOCK, 0, s>>>(
          nshort, gb_sg_per(nshort), list, d_arowptr, d_arowind, d_arowval, d_browptr,
          d_browind, d_browval, nullptr, cnt, nullptr, nullptr, nullptr, 0, nullptr);
      GB_SG_TRY(hipGetLastError());
    }
    if (nmed && staged)
      GB_SG_TRY(gb_sg_medium<GB_SG_STAGE>(hcount, list, d_arowptr, d_arowind, d_arowval,
                                          d_browptr, d_browind, d_browval, nullptr, cnt, sind,
                                          sval, nullptr, 0, off));
    else if (nmed)
      GB_SG_TRY(gb_sg_medium<GB_SG_COUNT>(hcount, list, d_arowptr, d_arowind, d_arowval,
                                          d_browptr, d_browind, d_browval, nullptr, cnt,
                                          nullptr, nullptr, nullptr, 0, nullptr));
  } else {
    if (nshort) {
      gb_sg_wave<GB_SG_DENSE><<<gb_sg_short_grid(nshort), GB_BLOCK, 0, s>>>(
          nshort, gb_sg_per(nshort), list, d_arowptr, d_arowind, d_arowval, d_browptr,
          d_browind, d_browval, nullptr, nullptr, nullptr, nullptr, d_cdense, bncols, nullptr);
      GB_SG_TRY(hipGetLastError());
    }
    if (nmed)
      GB_SG_TRY(gb_sg_medium<GB_SG_DENSE>(hcount, list, d_arowptr, d_arowind, d_arowval,
                                          d_browptr, d_browind, d_browval, nullptr, nullptr,
                                          nullptr, nullptr, d_cdense, bncols, nullptr));
  }
  // the sort path's products, numbered over its rows
  if (nlong && annz) {
    GB_SG_TRY(gb_dev_alloc((void **)&len2, ((size_t)annz + 1) * 4));
    GB_SG_TRY(gb_dev_alloc((void **)&off2, ((size_t)annz + 1) * 4));
    gb_sg_len_long<<<gb_sg_grid(annz), GB_BLOCK, 0, s>>>(anrows, annz, d_arowptr, cls, len,
                                                        len2);
    GB_SG_TRY(hipGetLastError());
    GB_SG_RV(gbd_scan_u32(len2, off2, annz, off2 + annz));
    GB_SG_TRY(gb_fetch(&E, off2 + annz, 4));
  }
  if (E) {
    GB_SG_TRY(gb_dev_alloc((void **)&erow, (size_t)E * 4));
    GB_SG_TRY(gb_dev_alloc((void **)&ecol, (size_t)E * 4));
    GB_SG_TRY(gb_dev_alloc((void **)&eval, (size_t)E * 8));
    GB_SG_TRY(gb_dev_alloc((void **)&perm1, (size_t)E * 4));
    GB_SG_TRY(gb_dev_alloc((void **)&row1, (size_t)E * 4));
    GB_SG_TRY(gb_dev_alloc((void **)&ord, (size_t)E * 4));
    GB_SG_TRY(gb_dev_alloc((void **)&flag, (size_t)E * 4));
    GB_SG_TRY(gb_dev_alloc((void **)&rid, ((size_t)E + 1) * 4));
    gb_sg_expand<<<gb_sg_grid(annz), GB_BLOCK, 0, s>>>(
        anrows, annz, d_arowptr, d_arowind, d_arowval, d_browptr, d_browind, d_browval, off2,
        len2, erow, ecol, eval);
    GB_SG_TRY(hipGetLastError());
    // 1. (row, col, t) order: stable by column, then stable by row
    GB_SG_RV(gbd_countingsort_kv_unchecked(ecol, nullptr, 0, bncols ? bncols - 1 : 0, E,
                                           perm1, nullptr));
    gb_sg_gather_u32<<<gb_sg_grid(E), GB_BLOCK, 0, s>>>(E, perm1, erow, row1);
    GB_SG_TRY(hipGetLastError());
    GB_SG_RV(gbd_countingsort_kv_unchecked(row1, perm1, 0, anrows ? anrows - 1 : 0, E, ord,
                                           nullptr));
    // 2. runs of equal (row, col) and their sums
    gb_sg_runflag<<<gb_sg_grid(E), GB_BLOCK, 0, s>>>(E, ord, erow, ecol, flag);
    GB_SG_TRY(hipGetLastError());
    GB_SG_RV(gbd_scan_u32(flag, rid, E, rid + E));
    GB_SG_TRY(gb_fetch(&nruns, rid + E, 4));
    GB_SG_TRY(gb_dev_alloc((void **)&runstart, ((size_t)nruns + 1) * 4));
    gb_sg_runstart<<<gb_sg_grid(E), GB_BLOCK, 0, s>>>(E, flag, rid, runstart);
    GB_SG_TRY(hipGetLastError());
    if (dense) {
      gb_sg_runsum<true><<<gb_sg_grid(nruns), GB_BLOCK, 0, s>>>(
          nruns, E, runstart, ord, erow, ecol, eval, bncols, d_cdense, nullptr, nullptr,
          nullptr, nullptr);
      GB_SG_TRY(hipGetLastError());
    } else {
      GB_SG_TRY(gb_dev_alloc((void **)&rrow, ((size_t)nruns + 1) * 4));
      GB_SG_TRY(gb_dev_alloc((void **)&rcol, ((size_t)nruns + 1) * 4));
      GB_SG_TRY(gb_dev_alloc((void **)&rfirst, ((size_t)nruns + 1) * 4));
      GB_SG_TRY(gb_dev_alloc((void **)&rval, ((size_t)nruns + 1) * 8));
      GB_SG_TRY(gb_dev_alloc((void **)&ordr, ((size_t)nruns + 1) * 4));
      GB_SG_TRY(gb_dev_alloc((void **)&rbeg, ((size_t)anrows + 1) * 4));
      gb_sg_runsum<false><<<gb_sg_grid(nruns), GB_BLOCK, 0, s>>>(
          nruns, E, runstart, ord, erow, ecol, eval, bncols, nullptr, rrow, rcol, rfirst,
          rval);
      GB_SG_TRY(hipGetLastError());
      gb_sg_rowruns<<<gb_sg_grid(nruns), GB_BLOCK, 0, s>>>(nruns, rrow, rbeg, cnt);
      GB_SG_TRY(hipGetLastError());
      // 3. first-appearance order: the first positions are unique and
      // row-major, so sorting by them alone orders the rows too
      GB_SG_RV(gbd_countingsort_kv_unchecked(rfirst, nullptr, 0, E - 1, nruns, ordr,
                                             nullptr));
    }
  }
  if (!dense) {
    GB_SG_TRY(gb_dev_alloc((void **)&crowptr, ((size_t)anrows + 1) * 4));
    GB_SG_RV(gbd_scan_u32(cnt, crowptr, anrows, crowptr + anrows));
    GB_SG_TRY(gb_fetch(&cnnz, crowptr + anrows, 4));
    GB_SG_TRY(gb_dev_alloc((void **)&crowind, ((size_t)cnnz + 1) * 4));
    GB_SG_TRY(gb_dev_alloc((void **)&crowval, ((size_t)cnnz + 1) * 8));
    if (nshort && staged) {
      gb_sg_unstage<<<gb_sg_short_grid(nshort), GB_BLOCK, 0, s>>>(
          nshort, gb_sg_per(nshort), list, d_arowptr, off, cnt, sind, sval, crowptr, crowind,
          crowval);
      GB_SG_TRY(hipGetLastError());
    } else if (nshort) {
      gb_sg_wave<GB_SG_FILL><<<gb_sg_short_grid(nshort), GB_BLOCK, 0, s>>>(
          nshort, gb_sg_per(nshort), list, d_arowptr, d_arowind, d_arowval, d_browptr,
          d_browind, d_browval, crowptr, nullptr, crowind, crowval, nullptr, 0, nullptr);
      GB_SG_TRY(hipGetLastError());
    }
    if (nmed && staged) {
      mlist = list ? list + nshort : nullptr;
      gb_sg_unstage_wave<<<gb_div_up(nmed, GB_WAVES_PER_BLOCK), GB_BLOCK, 0, s>>>(
          nmed, mlist, d_arowptr, off, cnt, sind, sval, crowptr, crowind, crowval);
      GB_SG_TRY(hipGetLastError());
    } else if (nmed) {
      GB_SG_TRY(gb_sg_medium<GB_SG_FILL>(hcount, list, d_arowptr, d_arowind, d_arowval,
                                         d_browptr, d_browind, d_browval, crowptr, nullptr,
                                         crowind, crowval, nullptr, 0, nullptr));
    }
    if (nruns) {
      gb_sg_out<<<gb_sg_grid(nruns), GB_BLOCK, 0, s>>>(nruns, ordr, rrow, rcol, rval, rbeg,
                                                       crowptr, crowind, crowval);
      GB_SG_TRY(hipGetLastError());
    }
    *d_crowptr = crowptr;
    *d_crowind = crowind;
    *d_crowval = crowval;
    *r_cnnz = cnnz;
    crowptr = crowind = nullptr;
    crowval = nullptr;
  }
  GB_SG_TRY(hipStreamSynchronize(s));
  rv = GOOSEBERRY_SUCCESS;
done:
  {
    void *tmp[] = {len, off, cls, count, list, len2, off2, erow, ecol, eval,
                   perm1, row1, ord, flag, rid, runstart, rrow, rcol, rfirst, rval,
                   ordr, rbeg, cnt, crowptr, crowind, crowval, tot, sind, sval};
    for (void *q : tmp) (void)gb_dev_free(q);
  }
  return rv;
#undef GB_SG_TRY
#undef GB_SG_RV
}

}  // extern "C"
