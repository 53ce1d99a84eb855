// gb_ingest.hip -- CSR construction straight into device memory: the .csr
// text reader of src/io.c:369-498 run on the GPU, and the binary CSR
// format's loader.
//
// .csr text: one line per row, "col val col val ...".  A line is the text
// up to '\n' (a final line without one counts); a line whose first byte is
// one of # % ' " / is a comment (src/io.c:63-69, 406-410) and is skipped;
// any other line, blank ones included, is a row.  A row's entries come
// from the reference's loop: strtoull(.., 10) for a column, then strtod
// for a value, repeated while strtod converts something (src/io.c:415-446),
// so rows keep file order (no sort, no merge of repeated columns).
// Columns are shifted by mincol = min(1, smallest column) and ncols =
// maxcol - mincol + 1 (src/io.c:433-435, 464, 478).
//
// On the device:
//   1. newlines and token starts (a byte that is no space after one that is)
//      counted per 4 KiB chunk, scanned, and written down per line: its
//      start and the number of tokens before it
//   2. comment flags per line, scanned: the row of every line
//   3. In plain text every pair of tokens is one entry: entries per row =
//      tokens / 2, row pointers = their scan, and one thread per pair converts
//      it and writes it at its place.  The thread checks that both
//      conversions take their whole token (and a line's odd last one is a
//      column without a value); the reference's loop then makes just these
//      entries of the line.
//   4. If any token failed (or the text holds too many for 32-bit row
//      pointers, or a line of over 8 GiB), the lines are gone through by the reference's loop, one
//      line per lane: a count pass (entries per row and the column range),
//      row pointers, a fill pass.
//   5. A value whose rounding needs more than 19 digits' worth of precision
//      is listed by the conversion and settled afterwards, one thread each, by
//      exact big-integer comparison.
// Every conversion is the C library's (gb_strtod.h), so the arrays are
// bitwise those of the host reader for the same text.
#include <errno.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/stat.h>
#include <unistd.h>

#define GB_HD __host__ __device__
#include "gb_strtod.h"
#include "gb_common.h"
#include "gb_stage.h"

#define GB_IN_CHUNK 4096                       // bytes per workgroup, line split
static_assert(GB_IN_CHUNK == 16 * GB_BLOCK, "one 16-byte word per thread");
#define GB_IN_FIX0 4096                        // initial capacity of the hard list
#define GB_IN_LOOK 256                         // bytes past its chunk that an entry may reach
// (min, max) column pairs that the count pass's wavefronts share, each in a
// cache line of its own (their atomics on one pair would queue up)
#define GB_IN_MM 64
#define GB_IN_MM_STRIDE 32

struct gb_in_fix {
  uint64_t p;    // where strtod starts
  uint64_t end;  // the end of its line
  uint32_t out;  // entry index
  uint32_t pad;
};

__device__ __forceinline__ bool gb_in_is_comment(unsigned c) {
  return c == '#' || c == '%' || c == '\'' || c == '"' || c == '/';
}

// [p, p + 16) of the text as one word; bytes outside [0, len) read as 0.
// txt + p is 16-byte aligned (p may lie before the text's first byte).
__device__ __forceinline__ uint4 gb_in_word(const char *txt, uint64_t len, int64_t p) {
  if (p >= 0 && (uint64_t)p + 16 <= len) return *(const uint4 *)(txt + p);
  uint32_t w[4] = {0, 0, 0, 0};
  for (int i = 0; i < 16; ++i) {
    const int64_t q = p + i;
    if (q >= 0 && (uint64_t)q < len) w[i >> 2] |= (uint32_t)(uint8_t)txt[q] << (8 * (i & 3));
  }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// four flags at the top bits of a word's bytes as four bits
__device__ __forceinline__ uint32_t gb_in_flags4(uint32_t z) {
  return (z >> 7 & 1u) | (z >> 14 & 2u) | (z >> 21 & 4u) | (z >> 28 & 8u);
}
// the top bit of each byte of v that equals c (c repeated in every byte)
__device__ __forceinline__ uint32_t gb_in_eq(uint32_t v, uint32_t c) {
  const uint32_t t = v ^ c;
  return ~(((t & 0x7f7f7f7fu) + 0x7f7f7f7fu) | t | 0x7f7f7f7fu);
}

// of the 16 bytes at p: bit i of *nl set where byte i is a newline, bit i of
// *tok where a token starts (nothing outside [0, len))
template <bool TOK>
__device__ __forceinline__ void gb_in_bits(const char *txt, uint64_t len, int64_t p, uint4 w,
                                           uint32_t *nl, uint32_t *tok) {
  const uint32_t v[4] = {w.x, w.y, w.z, w.w};
  uint32_t n = 0, sp = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    n |= gb_in_flags4(gb_in_eq(v[i], 0x0a0a0a0au)) << (4 * i);
    if (TOK) {  // spaces: 9 to 13, and 32
      const uint32_t x = v[i] & 0x7f7f7f7fu;
      const uint32_t ctl = (x + 0x77777777u) & ~(x + 0x72727272u) & ~v[i];
      sp |= gb_in_flags4((ctl & 0x80808080u) | gb_in_eq(v[i], 0x20202020u)) << (4 * i);
    }
  }
  *nl = n;
  if (!TOK) return;
  if (p < 0 || (uint64_t)p + 16 > len)
    for (int i = 0; i < 16; ++i)
      if (p + i < 0 || (uint64_t)(p + i) >= len) sp |= 1u << i;
  bool before = true;  // a space (or nothing) before byte 0
  if (p > 0 && (uint64_t)p <= len) {
    const unsigned c = (unsigned char)txt[p - 1];
    before = gbt_space(c);
  }
  *tok = ~sp & (sp << 1 | (before ? 1u : 0u)) & 0xffffu;
}

// Chunks of GB_IN_CHUNK bytes are counted from the last 16-byte boundary at
// or before the text, so that each thread reads one aligned 16-byte word of
// its chunk.  (A byte a thread and load took 87 us to count the newlines and
// 141 us to write their positions on 122 MB of text; words take 39 and 46 us,
// the tokens included.)
static uint64_t gb_in_nchunks(const char *txt, uint64_t len) {
  return len ? (len + ((uintptr_t)txt & 15u) + GB_IN_CHUNK - 1) / GB_IN_CHUNK : 0;
}
__device__ __forceinline__ int64_t gb_in_chunk_pos(const char *txt) {
  return (int64_t)((uint64_t)blockIdx.x * GB_IN_CHUNK) - (int64_t)((uintptr_t)txt & 15u);
}

// newlines (and token starts) per chunk
template <bool TOK>
__global__ void __launch_bounds__(GB_BLOCK)
gb_in_nl_count(const char *__restrict__ txt, uint64_t len, uint32_t *__restrict__ cnt,
               uint32_t *__restrict__ tcnt) {
  __shared__ uint32_t lds[GB_WAVES_PER_BLOCK];
  const int64_t p = gb_in_chunk_pos(txt) + 16 * threadIdx.x;
  uint32_t nl = 0, tok = 0;
  gb_in_bits<TOK>(txt, len, p, gb_in_word(txt, len, p), &nl, &tok);
  // at most 4096 of each: one sum for both
  const uint32_t c = gb_block_sum((uint32_t)__popc(nl) | (uint32_t)__popc(tok) << 16, lds);
  if (threadIdx.x == 0) {
    cnt[blockIdx.x] = c & 0xffffu;
    if (TOK) tcnt[blockIdx.x] = c >> 16;
  }
}

// ls[0] = 0, ls[1 + k] = the position after the k-th newline; lt[1 + k] =
// the tokens before it, lt[one past the newlines + 1] all tokens; off and
// toff = the exclusive scans of the chunk counts, their totals after them
template <bool TOK>
__global__ void __launch_bounds__(GB_BLOCK)
gb_in_nl_pos(const char *__restrict__ txt, uint64_t len, const uint32_t *__restrict__ off,
             const uint32_t *__restrict__ toff, uint64_t *__restrict__ ls,
             uint32_t *__restrict__ lt) {
  __shared__ uint32_t lds[GB_WAVES_PER_BLOCK];
  const int64_t p = gb_in_chunk_pos(txt) + 16 * threadIdx.x;
  uint32_t nl = 0, tok = 0, tot;
  gb_in_bits<TOK>(txt, len, p, gb_in_word(txt, len, p), &nl, &tok);
  const uint32_t e =
      gb_block_scan_excl((uint32_t)__popc(nl) | (uint32_t)__popc(tok) << 16, lds, &tot);
  uint32_t k = off[blockIdx.x] + (e & 0xffffu);
  const uint32_t t = TOK ? toff[blockIdx.x] + (e >> 16) : 0u;
  for (; nl; nl &= nl - 1u, ++k) {
    const uint32_t i = (uint32_t)__ffs((int)nl) - 1u;
    ls[1 + k] = (uint64_t)(p + i) + 1;
    if (TOK) lt[1 + k] = t + (uint32_t)__popc(tok & ((1u << i) - 1u));
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    ls[0] = 0;
    if (TOK) {
      lt[0] = 0;
      lt[off[gridDim.x] + 1] = toff[gridDim.x];
    }
  }
}

// line k: [start, end) without its newline and trailing '\r'
__device__ __forceinline__ void gb_in_line(const char *txt, uint64_t len, const uint64_t *ls,
                                           uint32_t nl, uint32_t k, uint64_t *start,
                                           uint64_t *end) {
  const uint64_t a = ls[k];
  uint64_t b = k < nl ? ls[k + 1] - 1 : len;
  while (b > a && txt[b - 1] == '\r') --b;
  *start = a;
  *end = b;
}

// rowof[k] = 1 for a row line, 0 for a comment (scanned in place later)
__global__ void __launch_bounds__(GB_BLOCK)
gb_in_rowflag(const char *__restrict__ txt, uint64_t len, const uint64_t *__restrict__ ls,
              uint32_t nl, uint32_t nlines, uint32_t *__restrict__ rowof) {
  for (uint32_t k = blockIdx.x * GB_BLOCK + threadIdx.x; k < nlines;
       k += gridDim.x * GB_BLOCK) {
    uint64_t a, b;
    gb_in_line(txt, len, ls, nl, k, &a, &b);
    rowof[k] = (b > a && gb_in_is_comment((unsigned char)txt[a])) ? 0u : 1u;
  }
}

__device__ __forceinline__ uint64_t gb_in_shfl64(uint64_t v, uint32_t l) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), l);
  return (uint64_t)hi << 32 | lo;
}

// the reference's entry loop over one line; FILL false counts entries and
// tracks the column range, FILL true writes them from out0.  The text starts
// at position `base` of the whole text.
template <bool FILL>
__device__ __forceinline__ uint32_t gb_in_parse_line(const char *txt, uint64_t a, uint64_t b,
                                                     uint32_t mincol, uint32_t out0,
                                                     uint32_t *rowind, double *rowval,
                                                     uint32_t *mn, uint32_t *mx,
                                                     gb_in_fix *fix, uint32_t fixcap,
                                                     uint32_t *nfix, uint64_t base = 0) {
  uint32_t nent = 0;
  uint64_t sp = a, c = 0;
  double v = 0.0;
  bool hard = false;
  sp = gbt_strtoull(txt, b, sp, 10, &c);
  uint64_t e = gbt_strtod(txt, b, sp, &v, &hard, FILL);
  while (e != sp) {
    const uint32_t col = (uint32_t)c;
    if (FILL) {
      const uint32_t o = out0 + nent;
      rowind[o] = col - mincol;
      rowval[o] = v;
      if (hard) {
        const uint32_t f = atomicAdd(nfix, 1u);
        if (f < fixcap) {
          fix[f].p = base + sp;
          fix[f].end = base + b;
          fix[f].out = o;
        }
      }
    } else {
      *mn = col < *mn ? col : *mn;
      *mx = col > *mx ? col : *mx;
    }
    ++nent;
    sp = e;
    sp = gbt_strtoull(txt, b, sp, 10, &c);
    e = gbt_strtod(txt, b, sp, &v, &hard, FILL);
  }
  return nent;
}

// The general passes over the lines, one wavefront (and workgroup) for 64
// consecutive lines, one line per lane.  The wavefront copies as many of its
// lines as fit into LDS with 16-byte loads, the lanes parse those from LDS,
// and so on; a line longer than the LDS tile is parsed from global memory.
// FILL false (count pass): cnt[row] = entries, and the smallest and largest
// column in one of the GB_IN_MM pairs of minmax.  FILL true: columns and
// values at the row pointers.
template <bool FILL, uint32_t TILE>
__global__ void __launch_bounds__(GB_WAVE)
gb_in_lines(const char *__restrict__ txt, uint64_t len, const uint64_t *__restrict__ ls,
            uint32_t nl, uint32_t nlines, const uint32_t *__restrict__ rowof,
            uint32_t *__restrict__ cnt, uint32_t *__restrict__ minmax,
            const uint32_t *__restrict__ rowptr, uint32_t mincol,
            uint32_t *__restrict__ rowind, double *__restrict__ rowval,
            gb_in_fix *__restrict__ fix, uint32_t fixcap, uint32_t *__restrict__ nfix) {
  __shared__ uint4 tile[TILE / 16];
  const uint32_t lane = threadIdx.x;
  const uint32_t k = blockIdx.x * GB_WAVE + lane;
  const bool have = k < nlines;
  uint64_t a = 0, b = 0;
  uint32_t r = 0, out0 = 0;
  bool row = false;
  if (have) {
    gb_in_line(txt, len, ls, nl, k, &a, &b);
    r = rowof[k];
    row = rowof[k + 1] != r;  // not a comment
    if (FILL && row) out0 = rowptr[r];
  }
  uint32_t mn = 0xffffffffu, mx = 0, nent = 0;
  const uint32_t off = (uint32_t)(uintptr_t)txt & 15u;
  uint64_t todo = __ballot(have);
  while (todo) {
    const uint32_t first = (uint32_t)__builtin_ctzll(todo);
    const uint64_t a0 = gb_in_shfl64(a, first);
    const int64_t base = (int64_t)((a0 + off) & ~15ull) - off;  // 16-byte aligned
    // the lines that end inside the tile: lanes first, first + 1, ...
    const uint64_t fit = __ballot(have && (int64_t)b - base <= (int64_t)TILE) & todo;
    if (!(fit >> first & 1ull)) {  // longer than the tile
      if (lane == first && row)
        nent = gb_in_parse_line<FILL>(txt, a, b, mincol, out0, rowind, rowval, &mn, &mx, fix,
                                      fixcap, nfix);
      todo &= todo - 1ull;
      continue;
    }
    const uint32_t last = 63 - (uint32_t)__builtin_clzll(fit);
    const uint32_t words = (uint32_t)((int64_t)gb_in_shfl64(b, last) - base + 15) / 16;
    for (uint32_t i = lane; i < words; i += GB_WAVE)
      tile[i] = gb_in_word(txt, len, base + 16 * (int64_t)i);
    __syncthreads();
    if (row && (fit >> lane & 1ull))
      nent = gb_in_parse_line<FILL>((const char *)tile, (uint64_t)((int64_t)a - base),
                                    (uint64_t)((int64_t)b - base), mincol, out0, rowind,
                                    rowval, &mn, &mx, fix, fixcap, nfix, (uint64_t)base);
    __syncthreads();
    todo &= ~fit;
  }
  if (!FILL) {
    if (row) cnt[r] = nent;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      mn = min(mn, (uint32_t)__shfl_xor((int)mn, o, GB_WAVE));
      mx = max(mx, (uint32_t)__shfl_xor((int)mx, o, GB_WAVE));
    }
    if (lane == 0) {
      uint32_t *mm = minmax + (blockIdx.x % GB_IN_MM) * GB_IN_MM_STRIDE;
      if (mn != 0xffffffffu) atomicMin(&mm[0], mn);
      if (mx) atomicMax(&mm[1], mx);
    }
  }
}

// plain text: entries per row = half its tokens, and their total.  Token
// numbers count modulo 2^32, which tells the tokens of a line of up to
// GB_IN_LINE_MAX bytes apart.  With ls, lines longer than `most` bytes raise
// the total beyond what the plain pass takes.
#define GB_IN_LINE_MAX ((1ull << 33) - 2)
__global__ void __launch_bounds__(GB_BLOCK)
gb_in_rowcnt(const uint32_t *__restrict__ lt, uint32_t nlines,
             const uint32_t *__restrict__ rowof, uint32_t *__restrict__ cnt,
             unsigned long long *__restrict__ total, const uint64_t *__restrict__ ls, uint32_t nl,
             uint64_t len, uint64_t most) {
  __shared__ unsigned long long lds[GB_WAVES_PER_BLOCK];
  unsigned long long v = 0;
  for (uint32_t k = blockIdx.x * GB_BLOCK + threadIdx.x; k < nlines;
       k += gridDim.x * GB_BLOCK) {
    const uint32_t r = rowof[k];
    if (rowof[k + 1] == r) continue;  // comment
    const uint32_t n = (lt[k + 1] - lt[k]) / 2;
    cnt[r] = n;
    v += n;
    if (ls && (k < nl ? ls[k + 1] : len) - ls[k] > most) v += 1ull << 32;
  }
  v = gb_block_sum(v, lds);
  if (threadIdx.x == 0) atomicAdd(total, v);
}

// the longest line whose tokens the plain pass can number;
// GOOSEBERRY_INGEST_LINE_MAX: the tests' way to the lines' passes
static uint64_t gb_in_line_max() {
  const char *e = getenv("GOOSEBERRY_INGEST_LINE_MAX");
  const uint64_t v = e && *e ? strtoull(e, nullptr, 10) : GB_IN_LINE_MAX;
  return v < GB_IN_LINE_MAX ? v : GB_IN_LINE_MAX;
}

// An entry in the usual form, "column value" with blanks between, at most 9
// digits in the column and 18 in the value: read at s[q ..) with 32-bit
// positions and no special forms.  False for any other entry (then the
// general conversions decide).  Never looks past s[q + 64).
__device__ __forceinline__ bool gb_in_usual(const char *s, uint32_t n, uint32_t q, uint32_t *col,
                                            uint32_t *e0, uint32_t *e1, double *val,
                                            bool *hard) {
  uint32_t a = q, c = 0, d;
  while ((d = (uint32_t)(uint8_t)s[a] - '0') <= 9u && a < q + 9) {
    c = c * 10 + d;
    ++a;
  }
  if (a == q || s[a] != ' ') return false;
  *col = c;
  *e0 = a;
  const uint32_t lim = a + 9;
  do ++a; while (s[a] == ' ' && a < lim);
  const bool neg = s[a] == '-';
  a += neg ? 1 : 0;
  uint64_t w = 0;
  const uint32_t m0 = a, m1 = a + 18;
  while ((d = (uint32_t)(uint8_t)s[a] - '0') <= 9u && a < m1) {
    w = w * 10 + d;
    ++a;
  }
  int32_t e10 = 0;
  uint32_t digits = a - m0;
  if (s[a] == '.') {
    const uint32_t f0 = ++a;
    while ((d = (uint32_t)(uint8_t)s[a] - '0') <= 9u && a < m1) {
      w = w * 10 + d;
      ++a;
    }
    e10 = (int32_t)f0 - (int32_t)a;
    digits += a - f0;
  }
  if (digits == 0) return false;
  if (s[a] == 'e') {
    ++a;
    const bool eneg = s[a] == '-';
    a += eneg || s[a] == '+' ? 1 : 0;
    const uint32_t x0 = a;
    int32_t ex = 0;
    while ((d = (uint32_t)(uint8_t)s[a] - '0') <= 9u && a < x0 + 3) {
      ex = ex * 10 + (int32_t)d;
      ++a;
    }
    if (a == x0) return false;
    e10 += eneg ? -ex : ex;
  }
  if (a >= n || !gbt_space((uint8_t)s[a])) return false;
  *e1 = a;
  *hard = false;
  uint64_t bits = 0;
  if (w) {
    if (e10 == 0 && w <= (1ull << 53)) bits = gbt_u64((double)w);
    else if (!gbt_eisel_lemire(w, e10, &bits)) *hard = true;
  }
  *val = gbt_bits((neg ? 1ull << 63 : 0ull) | bits);
  return true;
}

// Plain text, one workgroup per chunk: the chunk and the bytes after it in
// LDS, its tokens listed (position, and newlines before it in the chunk), and
// one thread per two tokens, the column among which it converts with the
// value that follows.  Columns are written less 1 (the usual mincol).
// *odd is set when a token is not what plain text has: the results are then
// not used.
//
// One thread per line, as the general passes have it, is a chain of byte
// loads as long as the line, and twice: 500,000 lines of 15 entries (122 MB)
// took 2,135 us to count and 1,917 us to fill from global memory, 557 us and
// 814 us from LDS; this pass takes 256 us in place of both (365 us with the
// general conversions alone).  It is bound by instructions: 758 vector and 992
// scalar ones (the loops' masks) for a wavefront's 64 entries.
__global__ void __launch_bounds__(GB_BLOCK)
gb_in_entries(const char *__restrict__ txt, uint64_t len, const uint32_t *__restrict__ off,
              const uint32_t *__restrict__ toff, const uint32_t *__restrict__ lt,
              const uint32_t *__restrict__ rowof, const uint32_t *__restrict__ rowptr,
              uint32_t *__restrict__ rowind, double *__restrict__ rowval,
              uint32_t *__restrict__ minmax, uint32_t *__restrict__ odd,
              gb_in_fix *__restrict__ fix, uint32_t fixcap, uint32_t *__restrict__ nfix) {
  __shared__ uint4 tile[(GB_IN_CHUNK + GB_IN_LOOK) / 16];
  __shared__ uint32_t list[GB_IN_CHUNK / 2 + 1];
  __shared__ uint32_t lds[GB_WAVES_PER_BLOCK];
  __shared__ uint32_t smn, smx;
  const uint32_t tid = threadIdx.x;
  const int64_t p0 = gb_in_chunk_pos(txt), p = p0 + 16 * tid;
  const uint4 w = gb_in_word(txt, len, p);
  tile[tid] = w;
  if (tid < GB_IN_LOOK / 16)
    tile[GB_BLOCK + tid] = gb_in_word(txt, len, p + GB_IN_CHUNK);
  if (tid == 0) {
    smn = 0xffffffffu;
    smx = 0;
  }
  uint32_t nl = 0, tok = 0, tot;
  gb_in_bits<true>(txt, len, p, w, &nl, &tok);
  const uint32_t ex =
      gb_block_scan_excl((uint32_t)__popc(nl) | (uint32_t)__popc(tok) << 16, lds, &tot);
  for (uint32_t j = ex >> 16; tok; tok &= tok - 1u, ++j) {
    const uint32_t i = (uint32_t)__ffs((int)tok) - 1u;
    const uint32_t lines = (ex & 0xffffu) + (uint32_t)__popc(nl & ((1u << i) - 1u));
    list[j] = (16 * tid + i) | lines << 16;
  }
  __syncthreads();
  const uint32_t ntok = tot >> 16;
  const uint32_t k0 = off[blockIdx.x], t0 = toff[blockIdx.x];
  // the text in the tile ends at n; at_end: so does the whole text
  const uint64_t left = (uint64_t)((int64_t)len - p0);
  const bool at_end = left <= GB_IN_CHUNK + GB_IN_LOOK;
  const uint64_t n = at_end ? left : GB_IN_CHUNK + GB_IN_LOOK;
  const char *s = (const char *)tile;
  uint32_t mn = 0xffffffffu, mx = 0;
  bool bad = false;
  for (uint32_t j2 = 2 * tid; j2 < ntok; j2 += 2 * GB_BLOCK) {
    for (uint32_t j = j2; j < j2 + 2 && j < ntok; ++j) {
      const uint32_t e = list[j], k = k0 + (e >> 16);
      const uint32_t first = lt[k], count = lt[k + 1] - first, i = t0 + j - first;
      if (i & 1u) continue;  // a value
      const uint32_t r = rowof[k];
      if (rowof[k + 1] == r) continue;  // comment
      const uint32_t q = e & 0xffffu;
      uint32_t col = 0, u0 = 0, u1 = 0;
      double v = 0.0;
      bool hard = false;
      uint64_t e0, e1;
      if (i + 1 < count && gb_in_usual(s, (uint32_t)n, q, &col, &u0, &u1, &v, &hard)) {
        e0 = u0;
        e1 = u1;
      } else {
        uint64_t c = 0;
        e0 = gbt_strtoull(s, n, q, 10, &c);
        if (e0 == q || (e0 < n ? !gbt_space(gbt_at(s, n, e0)) : !at_end)) {
          bad = true;
          continue;
        }
        if (i + 1 == count) continue;  // a column without a value
        e1 = gbt_strtod(s, n, e0, &v, &hard, true);
        if (e1 == e0 || (e1 < n ? !gbt_space(gbt_at(s, n, e1)) : !at_end)) {
          bad = true;
          continue;
        }
        col = (uint32_t)c;
      }
      const uint32_t o = rowptr[r] + i / 2;
      rowind[o] = col - 1u;
      rowval[o] = v;
      mn = min(mn, col);
      mx = max(mx, col);
      if (hard) {
        const uint32_t f = atomicAdd(nfix, 1u);
        if (f < fixcap) {
          fix[f].p = (uint64_t)(p0 + (int64_t)e0);
          fix[f].end = (uint64_t)(p0 + (int64_t)e1);
          fix[f].out = o;
        }
      }
    }
  }
  if (mn != 0xffffffffu) atomicMin(&smn, mn);
  if (mx) atomicMax(&smx, mx);
  if (__syncthreads_or(bad) && tid == 0) *odd = 1u;
  if (tid == 0) {
    uint32_t *mm = minmax + (blockIdx.x % GB_IN_MM) * GB_IN_MM_STRIDE;
    if (smn != 0xffffffffu) atomicMin(&mm[0], smn);
    if (smx) atomicMax(&mm[1], smx);
  }
}

// 0-based text: the columns were written less 1
__global__ void __launch_bounds__(GB_BLOCK)
gb_in_shift(uint32_t *__restrict__ rowind, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * GB_BLOCK + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * GB_BLOCK)
    rowind[i] += 1u;
}

// the listed values, exactly (one thread each; the big integers live in
// this kernel's private memory only)
__global__ void __launch_bounds__(64)
gb_in_fixup(const char *__restrict__ txt, const gb_in_fix *__restrict__ fix, uint32_t nfix,
            double *__restrict__ rowval) {
  const uint32_t i = blockIdx.x * 64 + threadIdx.x;
  if (i >= nfix) return;
  gbt_big L, R;
  const gb_in_fix f = fix[i];
  rowval[f.out] = gbt_strtod_exact(txt, f.end, f.p, &L, &R);
}

// what a pass over the text counts, read back in one copy
struct gb_in_meta {
  uint32_t minmax[GB_IN_MM * GB_IN_MM_STRIDE];  // column ranges
  unsigned long long total;                     // entries
  uint32_t nfix;                                // listed values
  uint32_t odd;                                 // not plain text
};

__global__ void gb_in_init_meta(gb_in_meta *m) {
  m->minmax[threadIdx.x * GB_IN_MM_STRIDE] = 0xffffffffu;
  m->minmax[threadIdx.x * GB_IN_MM_STRIDE + 1] = 0;
  if (threadIdx.x == 0) {
    m->total = 0;
    m->nfix = 0;
    m->odd = 0;
  }
}

// text bytes a wavefront of gb_in_lines keeps in LDS
static bool gb_in_wide(uint64_t len, uint32_t nlines) {
  return len / nlines > 8192 / GB_WAVE;
}

__global__ void __launch_bounds__(GB_BLOCK)
gb_in_sum64(const uint32_t *__restrict__ a, uint64_t n, unsigned long long *__restrict__ total) {
  __shared__ unsigned long long lds[GB_WAVES_PER_BLOCK];
  unsigned long long v = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * GB_BLOCK + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * GB_BLOCK)
    v += a[i];
  v = gb_block_sum(v, lds);
  if (threadIdx.x == 0) atomicAdd(total, v);
}

// ---- MatrixMarket body (src/io.c:1060-1145): one coordinate per line

// flag[k] = 1 for an entry line (not blank after '\r' stripping, not a
// comment)
__global__ void __launch_bounds__(GB_BLOCK)
gb_mx_flag(const char *__restrict__ txt, uint64_t len, const uint64_t *__restrict__ ls,
           uint32_t nl, uint32_t nlines, uint32_t *__restrict__ flag) {
  for (uint32_t k = blockIdx.x * GB_BLOCK + threadIdx.x; k < nlines;
       k += gridDim.x * GB_BLOCK) {
    uint64_t a, b;
    gb_in_line(txt, len, ls, nl, k, &a, &b);
    flag[k] = (b == a || gb_in_is_comment((unsigned char)txt[a])) ? 0u : 1u;
  }
}

// entry e (= rank of its line): row i, column j (1-based in the file),
// weight w when one converts (a weight the first 19 digits do not settle is
// listed for gb_in_fixup).  bad: 1 when a coordinate does not convert or is
// out of range; nwt counts the entries with a weight
__global__ void __launch_bounds__(GB_BLOCK)
gb_mx_parse(const char *__restrict__ txt, uint64_t len, const uint64_t *__restrict__ ls,
            uint32_t nl, uint32_t nlines, const uint32_t *__restrict__ ent,
            uint32_t nrows, uint32_t ncols, int sym, uint32_t *__restrict__ ei,
            uint32_t *__restrict__ ej, double *__restrict__ ew, uint32_t *__restrict__ bad,
            uint32_t *__restrict__ nwt, gb_in_fix *__restrict__ fix, uint32_t fixcap,
            uint32_t *__restrict__ nfix) {
  __shared__ uint32_t swt;
  if (threadIdx.x == 0) swt = 0;
  __syncthreads();
  uint32_t b_ = 0, wt = 0;
  for (uint32_t k = blockIdx.x * GB_BLOCK + threadIdx.x; k < nlines;
       k += gridDim.x * GB_BLOCK) {
    const uint32_t e = ent[k];
    if (ent[k + 1] == e) continue;
    uint64_t a, b;
    gb_in_line(txt, len, ls, nl, k, &a, &b);
    uint64_t v = 0;
    uint64_t q = gbt_strtoull(txt, b, a, 10, &v);
    if (q == a) { b_ = 1; continue; }
    const uint32_t i = (uint32_t)v - 1u;
    uint64_t q2 = gbt_strtoull(txt, b, q, 10, &v);
    if (q2 == q) { b_ = 1; continue; }
    const uint32_t j = (uint32_t)v - 1u;
    double w = 1.0;
    bool hard = false;
    const uint64_t q3 = gbt_strtod(txt, b, q2, &w, &hard, true);
    if (q3 != q2) {
      ++wt;
      if (hard) {  // settled by gb_in_fixup
        const uint32_t f = atomicAdd(nfix, 1u);
        if (f < fixcap) {
          fix[f].p = q2;
          fix[f].end = b;
          fix[f].out = e;
        }
      }
    } else {
      w = 1.0;
    }
    if (i >= nrows || j >= ncols || (sym && j >= nrows)) b_ = 1;
    ei[e] = i;
    ej[e] = j;
    ew[e] = w;
  }
  if (b_) atomicOr(bad, 1u);
  if (wt) atomicAdd(&swt, wt);
  __syncthreads();
  if (threadIdx.x == 0 && swt) atomicAdd(nwt, swt);
}

// record keys in file order, a symmetric file's mirrored entry first:
// record 2e = (j, i), 2e + 1 = (i, j); otherwise record e = (i, j)
__global__ void __launch_bounds__(GB_BLOCK)
gb_mx_keys(uint32_t nent, int sym, const uint32_t *__restrict__ ei,
           const uint32_t *__restrict__ ej, uint32_t *__restrict__ key) {
  for (uint32_t e = blockIdx.x * GB_BLOCK + threadIdx.x; e < nent; e += gridDim.x * GB_BLOCK) {
    if (sym) {
      key[2 * (uint64_t)e] = ej[e];
      key[2 * (uint64_t)e + 1] = ei[e];
    } else {
      key[e] = ei[e];
    }
  }
}

// CSR entries from the records in row order (ord = stable sort by row)
__global__ void __launch_bounds__(GB_BLOCK)
gb_mx_gather(uint32_t nnz, int sym, int wgts, const uint32_t *__restrict__ ord,
             const uint32_t *__restrict__ ei, const uint32_t *__restrict__ ej,
             const double *__restrict__ ew, uint32_t *__restrict__ rowind,
             double *__restrict__ rowval) {
  for (uint32_t p = blockIdx.x * GB_BLOCK + threadIdx.x; p < nnz; p += gridDim.x * GB_BLOCK) {
    const uint32_t r = ord[p];
    const uint32_t e = sym ? r >> 1 : r;
    const bool mirror = sym && !(r & 1u);
    rowind[p] = mirror ? ei[e] : ej[e];
    rowval[p] = wgts ? ew[e] : 1.0;
  }
}

// src/io.c:401-402,433-435: mincol starts at 1, maxcol at 0
static void gb_in_range(const gb_in_meta &h, uint32_t *mincol, uint32_t *maxcol) {
  *mincol = 1u;
  *maxcol = 0;
  for (uint32_t i = 0; i < GB_IN_MM; ++i) {
    const uint32_t *mm = h.minmax + i * GB_IN_MM_STRIDE;
    if (mm[0] < *mincol) *mincol = mm[0];
    if (mm[1] > *maxcol) *maxcol = mm[1];
  }
}

static uint32_t gb_in_grid(uint64_t n) {
  uint64_t g = (n + GB_BLOCK - 1) / GB_BLOCK;
  if (g > 16384) g = 16384;
  return g ? (uint32_t)g : 1u;
}

static int gb_in_errno(int e) {
  switch (e) {
    case ENOENT: case ENOTDIR: return GOOSEBERRY_ERROR_FILENOTFOUND;
    case EACCES: case EPERM: return GOOSEBERRY_ERROR_PERMISSIONDENIED;
    case EINVAL: case ENAMETOOLONG: return GOOSEBERRY_ERROR_INVALIDINPUT;
    default: return GOOSEBERRY_ERROR_UNKNOWN;
  }
}

// A file range read into a staging buffer: pread by the staging threads,
// each over its own part of the range.
struct gb_in_file_src {
  int fd;
  uint64_t base;  // file offset of the range's first byte
};

static int gb_in_fill_file(void *ctx, uint64_t off, uint64_t len, char *buf) {
  const gb_in_file_src *f = (const gb_in_file_src *)ctx;
  uint64_t done = 0;
  while (done < len) {
    const ssize_t r = pread(f->fd, buf + done, (size_t)(len - done),
                            (off_t)(f->base + off + done));
    if (r < 0 && errno == EINTR) continue;
    if (r <= 0) return GOOSEBERRY_ERROR_READ;  // an error, or the file ended early
    done += (uint64_t)r;
  }
  return GOOSEBERRY_SUCCESS;
}

// bytes [offset, offset + bytes) of an open file into device memory: the
// staging threads read into one pinned buffer while the other one's copy to
// the device runs
static int gb_in_file_to_device(FILE *f, uint64_t offset, uint64_t bytes, char *d_dst) {
  gb_in_file_src src = {fileno(f), offset};
  return gb_stage_htod(d_dst, bytes, gb_in_fill_file, &src);
}

extern "C" {

int gbd_load_file(const char *file, char **d_txt, uint64_t *r_len) {
  int rv = gb_ensure_init();
  if (rv != GOOSEBERRY_SUCCESS) return rv;
  if (!file || !d_txt || !r_len) return GOOSEBERRY_ERROR_INVALIDINPUT;
  FILE *f = fopen(file, "rb");
  if (!f) return gb_in_errno(errno);
  struct stat st;
  if (fstat(fileno(f), &st) != 0) {
    fclose(f);
    return GOOSEBERRY_ERROR_READ;
  }
  const uint64_t len = (uint64_t)st.st_size;
  char *d = nullptr;
  hipError_t he = gb_dev_alloc((void **)&d, len + 16);
  if (he != hipSuccess) {
    fclose(f);
    return gb_hip_fail(he, "gb_dev_alloc", __FILE__, __LINE__);
  }
  rv = gb_in_file_to_device(f, 0, len, d);
  fclose(f);
  if (rv != GOOSEBERRY_SUCCESS) {
    (void)gb_dev_free(d);
    return rv;
  }
  *d_txt = d;
  *r_len = len;
  return GOOSEBERRY_SUCCESS;
}

int gbd_load_file_range(const char *file, uint64_t offset, uint64_t bytes, void *d_dst) {
  int rv = gb_ensure_init();
  if (rv != GOOSEBERRY_SUCCESS) return rv;
  FILE *f = fopen(file, "rb");
  if (!f) return gb_in_errno(errno);
  rv = gb_in_file_to_device(f, offset, bytes, (char *)d_dst);
  fclose(f);
  return rv;
}

int gbd_parse_csr(const char *d_txt, uint64_t len, uint32_t *r_nrows, uint32_t *r_ncols,
                  uint32_t *r_nnz, uint32_t **d_rowptr, uint32_t **d_rowind,
                  double **d_rowval) {
  int rv = gb_ensure_init();
  if (rv != GOOSEBERRY_SUCCESS) return rv;
  hipStream_t s = gb_stream();
  hipError_t he = hipSuccess;
  const uint64_t nchunks = gb_in_nchunks(d_txt, len);
  if (nchunks >= 0xffffffffull) return GOOSEBERRY_ERROR_INVALIDINPUT;
  uint32_t *ccnt = nullptr, *tcnt = nullptr, *lt = nullptr, *rowof = nullptr, *cnt = nullptr,
           *rowptr = nullptr, *rowind = nullptr;
  uint64_t *ls = nullptr;
  double *rowval = nullptr;
  gb_in_fix *fix = nullptr;
  gb_in_meta *meta = nullptr, h;
  uint32_t nl = 0, nlines = 0, nrows = 0, nnz = 0, fixcap = GB_IN_FIX0;
  uint32_t mincol = 1u, maxcol = 0;
  char lastc = '\n';
#define GB_IN_TRY(call)                                         \
  do {                                                          \
    he = (call);                                                \
    if (he != hipSuccess) {                                     \
      rv = gb_hip_fail(he, #call, __FILE__, __LINE__);          \
      goto done;                                                \
    }                                                           \
  } while (0)
#define GB_IN_RV(call)                                          \
  do {                                                          \
    rv = (call);                                                \
    if (rv != GOOSEBERRY_SUCCESS) goto done;                    \
  } while (0)

  // 1. line starts and tokens
  GB_IN_TRY(gb_dev_alloc((void **)&ccnt, (nchunks + 1) * 4));
  GB_IN_TRY(gb_dev_alloc((void **)&tcnt, (nchunks + 1) * 4));
  if (nchunks) {
    gb_in_nl_count<true><<<(uint32_t)nchunks, GB_BLOCK, 0, s>>>(d_txt, len, ccnt, tcnt);
    GB_IN_TRY(hipGetLastError());
    GB_IN_TRY(hipMemcpyAsync(&lastc, d_txt + len - 1, 1, hipMemcpyDeviceToHost, s));
  }
  GB_IN_RV(gbd_scan_u32(ccnt, ccnt, nchunks, ccnt + nchunks));
  GB_IN_RV(gbd_scan_u32(tcnt, tcnt, nchunks, tcnt + nchunks));
  GB_IN_TRY(gb_fetch(&nl, ccnt + nchunks, 4));
  if (nl == 0xffffffffu) {
    rv = GOOSEBERRY_ERROR_INVALIDINPUT;
    goto done;
  }
  // a last line without a newline counts; text ending in one has no
  // line after it
  nlines = nl + (lastc != '\n' ? 1u : 0u);
  GB_IN_TRY(gb_dev_alloc((void **)&ls, ((uint64_t)nl + 2) * 8));
  GB_IN_TRY(gb_dev_alloc((void **)&lt, ((uint64_t)nl + 2) * 4));
  if (nchunks) {
    gb_in_nl_pos<true><<<(uint32_t)nchunks, GB_BLOCK, 0, s>>>(d_txt, len, ccnt, tcnt, ls, lt);
    GB_IN_TRY(hipGetLastError());
  }
  // 2. rows
  GB_IN_TRY(gb_dev_alloc((void **)&rowof, ((uint64_t)nlines + 1) * 4));
  if (nlines) {
    gb_in_rowflag<<<gb_in_grid(nlines), GB_BLOCK, 0, s>>>(d_txt, len, ls, nl, nlines, rowof);
    GB_IN_TRY(hipGetLastError());
  }
  GB_IN_RV(gbd_scan_u32(rowof, rowof, nlines, rowof + nlines));
  GB_IN_TRY(hipMemcpyAsync(&nrows, rowof + nlines, 4, hipMemcpyDeviceToHost, s));
  GB_IN_TRY(gb_dev_alloc((void **)&cnt, ((uint64_t)nlines + 1) * 4));
  GB_IN_TRY(gb_dev_alloc((void **)&meta, sizeof(*meta)));
  // 3. the entries of plain text, or (general) 4. of any text
  for (int general = 0; general < 2; ++general) {
    gb_in_init_meta<<<1, GB_IN_MM, 0, s>>>(meta);
    GB_IN_TRY(hipGetLastError());
    if (nlines && !general) {
      const uint32_t g = gb_in_grid(nlines);
      const uint64_t most = gb_in_line_max();
      gb_in_rowcnt<<<g > 512u ? 512u : g, GB_BLOCK, 0, s>>>(
          lt, nlines, rowof, cnt, &meta->total, len > most ? ls : nullptr, nl, len, most);
      GB_IN_TRY(hipGetLastError());
    } else if (nlines) {
      auto *k = gb_in_wide(len, nlines) ? gb_in_lines<false, 16384> : gb_in_lines<false, 8192>;
      k<<<gb_div_up(nlines, GB_WAVE), GB_WAVE, 0, s>>>(
          d_txt, len, ls, nl, nlines, rowof, cnt, meta->minmax, nullptr, 0, nullptr, nullptr,
          nullptr, 0, nullptr);
      GB_IN_TRY(hipGetLastError());
      if (nrows) {
        const uint32_t g = gb_in_grid(nrows);
        gb_in_sum64<<<g > 512u ? 512u : g, GB_BLOCK, 0, s>>>(cnt, nrows, &meta->total);
        GB_IN_TRY(hipGetLastError());
      }
    }
    GB_IN_TRY(gb_fetch(&h, meta, sizeof(h)));
    if (h.total > 0xffffffffull) {
      if (!general) continue;
      rv = GOOSEBERRY_ERROR_INVALIDINPUT;  // beyond 32-bit row pointers
      goto done;
    }
    nnz = (uint32_t)h.total;
    if (general) gb_in_range(h, &mincol, &maxcol);
    (void)gb_dev_free(rowptr);
    (void)gb_dev_free(rowind);
    (void)gb_dev_free(rowval);
    rowptr = rowind = nullptr;
    rowval = nullptr;
    GB_IN_TRY(gb_dev_alloc((void **)&rowptr, ((uint64_t)nrows + 1) * 4));
    GB_IN_RV(gbd_scan_u32(cnt, rowptr, nrows, rowptr + nrows));
    GB_IN_TRY(gb_dev_alloc((void **)&rowind, ((uint64_t)nnz + 1) * 4));
    GB_IN_TRY(gb_dev_alloc((void **)&rowval, ((uint64_t)nnz + 1) * 8));
    // the fill, again with a larger list if the first one overflowed
    for (int pass = 0; pass < 2; ++pass) {
      if (pass) {
        (void)gb_dev_free(fix);
        fix = nullptr;
        fixcap = h.nfix;
        gb_in_init_meta<<<1, GB_IN_MM, 0, s>>>(meta);
        GB_IN_TRY(hipGetLastError());
      }
      if (!fix) GB_IN_TRY(gb_dev_alloc((void **)&fix, (uint64_t)fixcap * sizeof(gb_in_fix)));
      if (nlines && !general) {
        gb_in_entries<<<(uint32_t)nchunks, GB_BLOCK, 0, s>>>(
            d_txt, len, ccnt, tcnt, lt, rowof, rowptr, rowind, rowval, meta->minmax,
            &meta->odd, fix, fixcap, &meta->nfix);
        GB_IN_TRY(hipGetLastError());
      } else if (nlines) {
        auto *k = gb_in_wide(len, nlines) ? gb_in_lines<true, 16384> : gb_in_lines<true, 8192>;
        k<<<gb_div_up(nlines, GB_WAVE), GB_WAVE, 0, s>>>(
            d_txt, len, ls, nl, nlines, rowof, nullptr, nullptr, rowptr, mincol, rowind,
            rowval, fix, fixcap, &meta->nfix);
        GB_IN_TRY(hipGetLastError());
      }
      GB_IN_TRY(gb_fetch(&h, meta, sizeof(h)));
      if (h.odd || h.nfix <= fixcap) break;
    }
    if (h.odd) continue;  // not plain text
    if (h.nfix > fixcap) {
      rv = GOOSEBERRY_ERROR_UNKNOWN;
      goto done;
    }
    if (!general) {
      gb_in_range(h, &mincol, &maxcol);
      if (mincol == 0 && nnz) {
        gb_in_shift<<<gb_in_grid(nnz), GB_BLOCK, 0, s>>>(rowind, nnz);
        GB_IN_TRY(hipGetLastError());
      }
    }
    if (h.nfix) {
      gb_in_fixup<<<gb_div_up(h.nfix, 64), 64, 0, s>>>(d_txt, fix, h.nfix, rowval);
      GB_IN_TRY(hipGetLastError());
    }
    GB_IN_TRY(hipStreamSynchronize(s));
    *r_nrows = nrows;
    *r_ncols = maxcol - mincol + 1u;
    *r_nnz = nnz;
    *d_rowptr = rowptr;
    *d_rowind = rowind;
    *d_rowval = rowval;
    rowptr = rowind = nullptr;
    rowval = nullptr;
    break;
  }
  rv = GOOSEBERRY_SUCCESS;
done:
  (void)gb_dev_free(ccnt); (void)gb_dev_free(tcnt); (void)gb_dev_free(ls); (void)gb_dev_free(lt);
  (void)gb_dev_free(rowof); (void)gb_dev_free(cnt); (void)gb_dev_free(meta); (void)gb_dev_free(fix);
  (void)gb_dev_free(rowptr); (void)gb_dev_free(rowind); (void)gb_dev_free(rowval);
  return rv;
#undef GB_IN_TRY
#undef GB_IN_RV
}

// The body of a MatrixMarket file (text at d_txt[off, len)): the lines
// after the size line.  nrows, ncols and sym come from the header, parsed
// on the host.  Rows are filled by a stable sort of the entries' records by
// row, a symmetric file's mirrored entry first (src/io.c:1103-1144).
int gbd_parse_mtx_body(const char *d_txt, uint64_t len, uint64_t off, uint32_t nrows,
                       uint32_t ncols, int sym, uint32_t *r_nnz, uint32_t **d_rowptr,
                       uint32_t **d_rowind, double **d_rowval) {
  int rv = gb_ensure_init();
  if (rv != GOOSEBERRY_SUCCESS) return rv;
  if (off > len) return GOOSEBERRY_ERROR_INVALIDINPUT;
  hipStream_t s = gb_stream();
  hipError_t he = hipSuccess;
  const char *txt = d_txt + off;
  const uint64_t blen = len - off;
  const uint64_t nchunks = gb_in_nchunks(txt, blen);
  if (nchunks >= 0xffffffffull) return GOOSEBERRY_ERROR_INVALIDINPUT;
  uint32_t *ccnt = nullptr, *ent = nullptr, *ei = nullptr, *ej = nullptr, *flags = nullptr,
           *key = nullptr, *ord = nullptr, *rowptr = nullptr, *rowind = nullptr,
           *nfix = nullptr;
  uint64_t *ls = nullptr;
  double *ew = nullptr, *rowval = nullptr;
  gb_in_fix *fix = nullptr;
  uint32_t nl = 0, nlines = 0, nent = 0, hflags[3] = {0, 0, 0}, hnfix = 0, fixcap = GB_IN_FIX0;
  uint64_t last = 0, nnz64 = 0;
  uint32_t nnz = 0;
#define GB_MX_TRY(call)                                         \
  do {                                                          \
    he = (call);                                                \
    if (he != hipSuccess) {                                     \
      rv = gb_hip_fail(he, #call, __FILE__, __LINE__);          \
      goto done;                                                \
    }                                                           \
  } while (0)
#define GB_MX_RV(call)                                          \
  do {                                                          \
    rv = (call);                                                \
    if (rv != GOOSEBERRY_SUCCESS) goto done;                    \
  } while (0)
  // lines of the body
  GB_MX_TRY(gb_dev_alloc((void **)&ccnt, (nchunks + 1) * 4));
  if (nchunks) {
    gb_in_nl_count<false><<<(uint32_t)nchunks, GB_BLOCK, 0, s>>>(txt, blen, ccnt, nullptr);
    GB_MX_TRY(hipGetLastError());
  }
  GB_MX_RV(gbd_scan_u32(ccnt, ccnt, nchunks, ccnt + nchunks));
  GB_MX_TRY(gb_fetch(&nl, ccnt + nchunks, 4));
  if (nl == 0xffffffffu) {
    rv = GOOSEBERRY_ERROR_INVALIDINPUT;
    goto done;
  }
  GB_MX_TRY(gb_dev_alloc((void **)&ls, ((uint64_t)nl + 2) * 8));
  if (nchunks) {
    gb_in_nl_pos<false><<<(uint32_t)nchunks, GB_BLOCK, 0, s>>>(txt, blen, ccnt, nullptr, ls,
                                                            nullptr);
    GB_MX_TRY(hipGetLastError());
    GB_MX_TRY(gb_fetch(&last, ls + nl, 8));
  }
  nlines = nl + (blen > last ? 1u : 0u);
  // entry lines and their ranks
  GB_MX_TRY(gb_dev_alloc((void **)&ent, ((uint64_t)nlines + 1) * 4));
  if (nlines) {
    gb_mx_flag<<<gb_in_grid(nlines), GB_BLOCK, 0, s>>>(txt, blen, ls, nl, nlines, ent);
    GB_MX_TRY(hipGetLastError());
  }
  GB_MX_RV(gbd_scan_u32(ent, ent, nlines, ent + nlines));
  GB_MX_TRY(gb_fetch(&nent, ent + nlines, 4));
  nnz64 = (uint64_t)nent * (sym ? 2u : 1u);
  if (nnz64 > 0xffffffffull) {
    rv = GOOSEBERRY_ERROR_INVALIDINPUT;
    goto done;
  }
  nnz = (uint32_t)nnz64;
  GB_MX_TRY(gb_dev_alloc((void **)&ei, ((uint64_t)nent + 1) * 4));
  GB_MX_TRY(gb_dev_alloc((void **)&ej, ((uint64_t)nent + 1) * 4));
  GB_MX_TRY(gb_dev_alloc((void **)&ew, ((uint64_t)nent + 1) * 8));
  GB_MX_TRY(gb_dev_alloc((void **)&flags, 8));
  GB_MX_TRY(gb_dev_alloc((void **)&nfix, 4));
  for (int pass = 0; pass < 2; ++pass) {
    GB_MX_TRY(gb_dev_alloc((void **)&fix, (uint64_t)fixcap * sizeof(gb_in_fix)));
    GB_MX_RV(gbd_zero(flags, 8));
    GB_MX_RV(gbd_zero(nfix, 4));
    if (nlines) {
      gb_mx_parse<<<gb_in_grid(nlines), GB_BLOCK, 0, s>>>(txt, blen, ls, nl, nlines, ent, nrows,
                                                         ncols, sym, ei, ej, ew, flags,
                                                         flags + 1, fix, fixcap, nfix);
      GB_MX_TRY(hipGetLastError());
    }
    GB_MX_TRY(hipMemcpyAsync(hflags, flags, 8, hipMemcpyDeviceToHost, s));
    GB_MX_TRY(gb_fetch(&hnfix, nfix, 4));
    if (hnfix <= fixcap) break;
    (void)gb_dev_free(fix);
    fix = nullptr;
    fixcap = hnfix;
  }
  // a coordinate missing or out of range; weights on some lines only
  if (hflags[0] || (hflags[1] != 0 && hflags[1] != nent) || hnfix > fixcap) {
    rv = GOOSEBERRY_ERROR_INVALIDINPUT;
    goto done;
  }
  if (hnfix) {
    gb_in_fixup<<<gb_div_up(hnfix, 64), 64, 0, s>>>(txt, fix, hnfix, ew);
    GB_MX_TRY(hipGetLastError());
  }
  // rows: a stable sort of the records by row gives the fill order and,
  // through its run starts, the row pointers
  GB_MX_TRY(gb_dev_alloc((void **)&rowptr, ((uint64_t)nrows + 2) * 4));
  GB_MX_TRY(gb_dev_alloc((void **)&rowind, ((uint64_t)nnz + 1) * 4));
  GB_MX_TRY(gb_dev_alloc((void **)&rowval, ((uint64_t)nnz + 1) * 8));
  if (nnz) {
    GB_MX_TRY(gb_dev_alloc((void **)&key, (uint64_t)nnz * 4));
    GB_MX_TRY(gb_dev_alloc((void **)&ord, (uint64_t)nnz * 4));
    gb_mx_keys<<<gb_in_grid(nent), GB_BLOCK, 0, s>>>(nent, sym, ei, ej, key);
    GB_MX_TRY(hipGetLastError());
    GB_MX_RV(gbd_countingsort_kv_unchecked(key, nullptr, 0, nrows - 1, nnz, ord, rowptr));
    gb_mx_gather<<<gb_in_grid(nnz), GB_BLOCK, 0, s>>>(nnz, sym, hflags[1] != 0, ord, ei, ej, ew,
                                                     rowind, rowval);
    GB_MX_TRY(hipGetLastError());
  } else {
    GB_MX_RV(gbd_zero(rowptr, ((uint64_t)nrows + 1) * 4));
  }
  GB_MX_TRY(hipStreamSynchronize(s));
  *r_nnz = nnz;
  *d_rowptr = rowptr;
  *d_rowind = rowind;
  *d_rowval = rowval;
  rowptr = rowind = nullptr;
  rowval = nullptr;
  rv = GOOSEBERRY_SUCCESS;
done:
  (void)gb_dev_free(ccnt); (void)gb_dev_free(ls); (void)gb_dev_free(ent); (void)gb_dev_free(ei); (void)gb_dev_free(ej);
  (void)gb_dev_free(ew); (void)gb_dev_free(flags); (void)gb_dev_free(nfix); (void)gb_dev_free(fix); (void)gb_dev_free(key);
  (void)gb_dev_free(ord); (void)gb_dev_free(rowptr); (void)gb_dev_free(rowind); (void)gb_dev_free(rowval);
  return rv;
#undef GB_MX_TRY
#undef GB_MX_RV
}

}  // extern "C"
