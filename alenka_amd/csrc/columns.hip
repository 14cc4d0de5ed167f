// Column codec and row-wise kernels over the segmented, bit-packed column layout:
// encoding (pfor_compress, compress.cu:411-527, as dense bit-packing), decoding
// (pfor_decompress, compress.cu:180-267), gathers (mygather, cm.cu:3350-3413), expression
// evaluation (select.cu:703-790) and the fused scan: decode + predicate + stream
// compaction (filter_op, cm.cu:3609-3666; filter, filter.cu:133-643).
#include <string.h>

#include <atomic>
#include <mutex>
#include <vector>

#include "aln_internal.h"
#include "vm.h"

namespace aln {

// ---- encoding -----------------------------------------------------------------------------

// Partial minima and maxima of each segment's blocks, then one wave per segment over its
// partials.  HBM-bound: 50M values 313 -> 76 us (one atomic pair per wave on the segment's two
// words, 100,000 of them on 100 addresses, took the rest).
__global__ void __launch_bounds__(256) k_seg_minmax(const int64_t *__restrict__ v, uint64_t nrows,
                                                    uint32_t seg_rows, uint32_t blocks_per_seg,
                                                    int64_t *__restrict__ pmin, int64_t *__restrict__ pmax) {
  __shared__ int64_t smn[4], smx[4];
  const uint32_t seg = blockIdx.x / blocks_per_seg, part = blockIdx.x % blocks_per_seg;
  const uint64_t s0 = (uint64_t)seg * seg_rows;
  const uint64_t s1 = s0 + seg_rows < nrows ? s0 + seg_rows : nrows;
  const uint64_t stride = (uint64_t)blocks_per_seg * 256;
  int64_t lo = INT64_MAX, hi = INT64_MIN;
  uint64_t i = s0 + (uint64_t)part * 256 + threadIdx.x;
  for (; i + 7 * stride < s1; i += 8 * stride) {  // eight loads in flight per thread
    int64_t x[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) x[k] = v[i + k * stride];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      lo = x[k] < lo ? x[k] : lo;
      hi = x[k] > hi ? x[k] : hi;
    }
  }
  for (; i < s1; i += stride) {
    const int64_t x = v[i];
    lo = x < lo ? x : lo;
    hi = x > hi ? x : hi;
  }
  for (int o = 32; o > 0; o >>= 1) {
    int64_t a = __shfl_xor(lo, o, 64), b = __shfl_xor(hi, o, 64);
    lo = a < lo ? a : lo;
    hi = b > hi ? b : hi;
  }
  if (__lane_id() == 0) {
    smn[threadIdx.x / 64] = lo;
    smx[threadIdx.x / 64] = hi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) {
      lo = smn[w] < lo ? smn[w] : lo;
      hi = smx[w] > hi ? smx[w] : hi;
    }
    pmin[blockIdx.x] = lo;
    pmax[blockIdx.x] = hi;
  }
}

__global__ void __launch_bounds__(64) k_seg_minmax_final(const int64_t *__restrict__ pmin,
                                                         const int64_t *__restrict__ pmax, uint32_t blocks_per_seg,
                                                         uint32_t nsegs, int64_t *__restrict__ out) {
  const uint32_t seg = blockIdx.x;
  int64_t lo = INT64_MAX, hi = INT64_MIN;
  for (uint32_t i = threadIdx.x; i < blocks_per_seg; i += 64) {
    const int64_t a = pmin[(uint64_t)seg * blocks_per_seg + i], b = pmax[(uint64_t)seg * blocks_per_seg + i];
    lo = a < lo ? a : lo;
    hi = b > hi ? b : hi;
  }
  for (int o = 32; o > 0; o >>= 1) {
    int64_t a = __shfl_xor(lo, o, 64), b = __shfl_xor(hi, o, 64);
    lo = a < lo ? a : lo;
    hi = b > hi ? b : hi;
  }
  if (threadIdx.x == 0) {
    out[seg] = lo;
    out[nsegs + seg] = hi;
  }
}

// A tile of 2048 rows per block, so that it starts on a word: a thread concatenates the codes of
// 8 consecutive rows in registers and ORs the words they make into LDS (two threads share only
// the words at their ends), and the tile's words are stored as whole lines (50M 24-bit codes
// 137 -> 93 us, 5.9 TB/s; a thread per word read its rows again and divided to find them).
constexpr int PK_ROWS = 8;
constexpr int PK_TILE = 256 * PK_ROWS;
__global__ void __launch_bounds__(256) k_pack(const int64_t *__restrict__ v, uint32_t seg_rows, uint32_t seg0,
                                              const aln_seg *__restrict__ segs, uint32_t *__restrict__ words) {
  __shared__ uint32_t out[PK_TILE / 32 * 64];
  const uint32_t seg = seg0 + blockIdx.y;
  const aln_seg sg = segs[seg];
  const uint64_t t0 = (uint64_t)blockIdx.x * PK_TILE;
  if (sg.bits == 0 || t0 >= sg.nrows) return;
  const uint32_t m = sg.nrows - t0 < PK_TILE ? (uint32_t)(sg.nrows - t0) : PK_TILE;
  const uint32_t nw = (m * sg.bits + 31) / 32;
  const int64_t *sv = v + (uint64_t)seg * seg_rows + t0;
  const uint32_t r0 = threadIdx.x * PK_ROWS;
  int64_t x[PK_ROWS];
  if (r0 + PK_ROWS <= m) {
#pragma unroll
    for (int j = 0; j < PK_ROWS; ++j) x[j] = sv[r0 + j];
  } else {
#pragma unroll
    for (int j = 0; j < PK_ROWS; ++j) x[j] = r0 + j < m ? sv[r0 + j] : sg.base;
  }
  for (uint32_t w = threadIdx.x; w < nw; w += 256) out[w] = 0;
  __syncthreads();
  if (r0 < m) {
    const uint32_t bits = sg.bits, lb = bits < 32 ? bits : 32, hb = bits - lb;
    const uint32_t lmask = lb == 32 ? 0xFFFFFFFFu : (1u << lb) - 1u, hmask = hb == 32 ? 0xFFFFFFFFu : (1u << hb) - 1u;
    uint32_t w = r0 * bits >> 5, fill = r0 * bits & 31;
    uint64_t acc = 0;
    auto put = [&](uint32_t part, uint32_t width) {
      acc |= (uint64_t)part << fill;
      fill += width;
      if (fill >= 32) {
        if (w < nw) atomicOr(&out[w], (uint32_t)acc);
        ++w;
        acc >>= 32;
        fill -= 32;
      }
    };
#pragma unroll
    for (int j = 0; j < PK_ROWS; ++j) {  // rows past the end are code 0
      const uint64_t code = (uint64_t)x[j] - (uint64_t)sg.base;
      put((uint32_t)code & lmask, lb);
      if (hb) put((uint32_t)(code >> 32) & hmask, hb);
    }
    if (fill && w < nw) atomicOr(&out[w], (uint32_t)acc);
  }
  __syncthreads();
  uint32_t *dst = words + sg.word_off + t0 / 32 * sg.bits;
  for (uint32_t w = threadIdx.x; w < nw; w += 256) __builtin_nontemporal_store(out[w], dst + w);
}

// ---- row-wise kernels ---------------------------------------------------------------------

// Rows outside the column (a segment past nsegs, or past a short last segment) read as 0.
//
// Consecutive rows [r0, r0 + n): a block's rows mostly lie in one segment, whose descriptor is then
// scalar and whose codes are unpacked with 32-bit bit positions (HBM-bound: 50M 24-bit codes 260 ->
// 94 us; a descriptor, a division and 64-bit positions per row before).  Eight rows per thread, or one
// where many blocks of 2048 rows would cross segments (1M rows in segments of 1000 rows: 11.2 us a
// call with eight, 9.7 with one).
constexpr uint32_t DEC_SEG_ROWS = 8192;
template <int DEC_ROWS>
__global__ void __launch_bounds__(256) k_decode(const uint32_t *__restrict__ words,
                                                const aln_seg *__restrict__ segs, uint32_t nsegs,
                                                uint32_t seg_rows, uint64_t r0, uint64_t n,
                                                int64_t *__restrict__ out) {
  const uint64_t b0 = (uint64_t)blockIdx.x * (256 * DEC_ROWS);
  const uint32_t m = n - b0 < 256 * DEC_ROWS ? (uint32_t)(n - b0) : 256 * DEC_ROWS;
  const uint64_t seg = (r0 + b0) / seg_rows;
  const uint32_t l0 = (uint32_t)(r0 + b0 - seg * seg_rows);
  out += b0;
  const aln_seg sg = segs[seg < nsegs ? seg : 0];
  if (seg < nsegs && (uint64_t)l0 + m <= sg.nrows) {
    const uint64_t bit = (uint64_t)l0 * sg.bits;
    uint32_t idx[DEC_ROWS];
    uint64_t c[DEC_ROWS];
#pragma unroll
    for (int u = 0; u < DEC_ROWS; ++u) {
      const uint32_t i = threadIdx.x + 256 * u;
      idx[u] = i < m ? i : m - 1;
    }
    unpack_codes<DEC_ROWS>(words + sg.word_off + (bit >> 5), sg.bits, idx, c, (uint32_t)bit & 31);
#pragma unroll
    for (int u = 0; u < DEC_ROWS; ++u)
      if (threadIdx.x + 256 * u < m)
        __builtin_nontemporal_store((int64_t)((uint64_t)sg.base + c[u]), out + threadIdx.x + 256 * u);
    return;
  }
  for (uint32_t i = threadIdx.x; i < m; i += 256) {
    const uint64_t r = r0 + b0 + i, s = r / seg_rows, local = r - s * seg_rows;
    out[i] = (s < nsegs && local < segs[s].nrows) ? decode_row(words, segs[s], local) : 0;
  }
}

// The rows of an expression or a gather: U rows of a thread, 256 apart, each row's segment by a
// product with ceil(2^64 / seg_rows) (seg_mul; 0 for one-row segments).  Selected rows ascend,
// so a wave's rows mostly share a segment: its descriptors are then read once, as scalars
// (price * (100 - disc) of 30M of 60M rows 461 -> 105 us, 240 MB written and 340 MB read).
struct RowArgs {
  ColTable ct;
  uint32_t nsegs, seg_rows;
  uint64_t seg_mul;
  const uint32_t *rows;  // NULL: rows 0 .. n-1
  uint64_t n;
};
template <int U>
struct RowSet {
  uint32_t seg[U], local[U];
  bool in[U];   // the row exists in the first column's segment
  bool same;    // every row of the wave lies in segment seg0 (and exists)
  uint32_t seg0;
};

template <int U>
__device__ __forceinline__ void row_set(const RowArgs &a, uint64_t i0, RowSet<U> &s) {
  uint32_t r[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {  // past the end: the block's first row
    const uint64_t i = i0 + threadIdx.x + 256 * u;
    r[u] = a.rows ? a.rows[i < a.n ? i : i0] : (uint32_t)(i < a.n ? i : i0);
  }
  bool same = true;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    s.seg[u] = a.seg_mul ? (uint32_t)__umul64hi(a.seg_mul, (uint64_t)r[u]) : r[u];
    s.local[u] = r[u] - s.seg[u] * a.seg_rows;
  }
  s.seg0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)s.seg[0]);
  const uint32_t nrows0 = s.seg0 < a.nsegs ? a.ct.segs[0][s.seg0].nrows : 0;
#pragma unroll
  for (int u = 0; u < U; ++u) same = same && s.seg[u] == s.seg0 && s.local[u] < nrows0;
  s.same = __builtin_amdgcn_ballot_w64(!same) == 0;
  if (!s.same) {
#pragma unroll
    for (int u = 0; u < U; ++u) s.in[u] = s.seg[u] < a.nsegs && s.local[u] < a.ct.segs[0][s.seg[u]].nrows;
  }
}

// A column's values of the rows.  P: uint32_t when a segment's bits fit in 32 bits.
template <int U, typename P>
__device__ __forceinline__ void row_values(const RowArgs &a, const RowSet<U> &s, int col, int64_t (&v)[U]) {
  if (s.same) {
    const aln_seg sg = a.ct.segs[col][s.seg0];
    P idx[U];
    uint64_t c[U];
#pragma unroll
    for (int u = 0; u < U; ++u) idx[u] = s.local[u];
    unpack_codes<U>(a.ct.words[col] + sg.word_off, sg.bits, idx, c);
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = (int64_t)((uint64_t)sg.base + c[u]);
  } else {
#pragma unroll
    for (int u = 0; u < U; ++u)
      v[u] = s.in[u] ? decode_row(a.ct.words[col], a.ct.segs[col][s.seg[u]], s.local[u]) : 0;
  }
}

template <int U, typename P>
__global__ void __launch_bounds__(VM_BLOCK) k_eval(RowArgs a, VProg p, int64_t *__restrict__ out) {
  extern __shared__ __align__(16) int64_t vm_stack[];
  const uint64_t i0 = (uint64_t)blockIdx.x * (VM_BLOCK * U);
  RowSet<U> s;
  row_set<U>(a, i0, s);
  int64_t t[U];
  vm_eval<U>(p, [&](int col, int64_t(&v)[U]) { row_values<U, P>(a, s, col, v); }, vm_stack + threadIdx.x, t);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint64_t i = i0 + threadIdx.x + VM_BLOCK * u;
    if (i < a.n) __builtin_nontemporal_store(t[u], out + i);
  }
}

template <int U, typename P>
__global__ void __launch_bounds__(256) k_gather(RowArgs a, int64_t *__restrict__ out) {
  const uint64_t i0 = (uint64_t)blockIdx.x * (256 * U);
  RowSet<U> s;
  row_set<U>(a, i0, s);
  int64_t v[U];
  row_values<U, P>(a, s, 0, v);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint64_t i = i0 + threadIdx.x + 256 * u;
    if (i < a.n) __builtin_nontemporal_store(v[u], out + i);
  }
}

__global__ void __launch_bounds__(256) k_apply_perm(const int64_t *__restrict__ in,
                                                    const uint32_t *__restrict__ perm, uint64_t n,
                                                    int64_t *__restrict__ out) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * 256)
    out[i] = in[perm[i]];
}

// out[i] = table[codes[i]], -1 for a code outside the table.
__global__ void __launch_bounds__(256) k_dict_lookup(const int64_t *__restrict__ codes, uint64_t n,
                                                     const int64_t *__restrict__ table, uint64_t ntable,
                                                     int64_t *__restrict__ out) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256) {
    const int64_t c = codes[i];
    out[i] = (c >= 0 && (uint64_t)c < ntable) ? table[c] : -1;
  }
}

// LIKE on one dictionary entry (the reference's gpu_regex, filter.cu:67-129): '%' matches any
// run, retrying from the character after the last attempt's start on a mismatch; '?' any
// character but '.'; others themselves.  The entry is `len` bytes, NUL-padded, and the
// position counter is shared by all attempts and bounded by len, as in the reference.
__device__ bool like_entry(const char *value, uint32_t len, const char *pattern) {
  bool after_pct = false;
  uint32_t used = 0;
  const char *from = value, *pat = pattern;
  for (;;) {
    const char *s = from, *p = pat;
    int stop = 0;  // 0: the value or the budget ran out, 1: '%' consumed, 2: mismatch
    for (; used < len && *s; ++s, ++p, ++used) {
      if (*p == '%') {
        after_pct = true;
        from = s;
        pat = p;
        while (*++pat == '%') {
        }
        if (!*pat) return true;
        stop = 1;
        break;
      }
      if (*p == '?' ? *s == '.' : *s != *p) {
        stop = 2;
        break;
      }
    }
    if (stop == 1) continue;
    if (stop == 2) {
      if (!after_pct) return false;
      ++from;
      ++used;
      continue;
    }
    while (*p == '%') ++p;
    return !*p;
  }
}

// One thread per entry of a fixed-width dictionary, matched where it lies: the matcher reads
// a value character only while its position counter is below the width, and the counter is
// never behind the character's offset, so no read leaves the entry.  A wave covers 64
// entries, so its two bit-set words are written whole from one ballot.
constexpr uint32_t LIKE_MAX_WIDTH = 256;
__global__ void __launch_bounds__(64) k_like_dict(const char *__restrict__ entries, uint64_t n, uint32_t width,
                                                  const char *__restrict__ pattern, uint32_t *__restrict__ bits) {
  const uint64_t i = (uint64_t)blockIdx.x * 64 + threadIdx.x;
  bool m = false;
  if (i < n) m = like_entry(entries + i * width, width, pattern);
  const uint64_t b = __builtin_amdgcn_ballot_w64(m);
  const uint64_t w = (uint64_t)blockIdx.x * 2;
  if (threadIdx.x == 0) bits[w] = (uint32_t)b;
  if (threadIdx.x == 32) bits[w + 1] = (uint32_t)(b >> 32);
}

// ---- fused scan: decode + predicate + compaction -------------------------------------------
constexpr int SC_BLOCK = VM_BLOCK;  // 256
constexpr int SC_ITEMS = 16;
constexpr int SC_TILE = SC_BLOCK * SC_ITEMS;

// One term of a conjunction the scan's fast path evaluates on column col: lo <= v <= hi, or
// (set != 0) membership of v in the bit set at device address lo over codes 0..hi-1.
struct RangeC {
  int32_t col;
  int32_t set;
  int64_t lo, hi;
};

// What one scan kernel call evaluates, by value (no upload).
struct ScanArgs {
  ColTable ct;
  uint32_t seg_rows, tiles_per_seg;
  const char *modes;
};
// At most one interval per column plus one set test per two instructions.
constexpr int MAX_RANGES_C = ALN_MAX_COLS + ALN_MAX_INSN / 2;
struct RangeSet {
  RangeC r[MAX_RANGES_C];
  int n;
};

// Which of the U rows idx[u] of a segment lie in every term.  An interval over codes narrower
// than 64 bits is compared with the codes themselves.
template <int U>
__device__ __forceinline__ void ranges_pass(const RangeSet &rs, const ColTable &ct, uint32_t seg, uint32_t r0,
                                            const uint32_t (&idx)[U], bool (&pass)[U]) {
  for (int k = 0; k < rs.n; ++k) {
    const RangeC t = rs.r[k];
    const aln_seg sg = ct.segs[t.col][seg];
    uint64_t c[U];
    unpack_codes<U>(ct.words[t.col] + sg.word_off + (uint64_t)(r0 >> 5) * sg.bits, sg.bits, idx, c);
    if (t.set) {
      const uint32_t *bs = reinterpret_cast<const uint32_t *>(t.lo);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t v = (int64_t)((uint64_t)sg.base + c[u]);
        pass[u] = pass[u] && v >= 0 && v < t.hi && ((bs[v >> 5] >> (v & 31)) & 1u);
      }
    } else if (sg.bits == 64) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t v = (int64_t)((uint64_t)sg.base + c[u]);
        pass[u] = pass[u] && v >= t.lo && v <= t.hi;
      }
    } else {
      const uint64_t most = (1ull << sg.bits) - 1;
      const uint64_t clo = t.lo <= sg.base ? 0 : (uint64_t)t.lo - (uint64_t)sg.base;
      uint64_t chi = (uint64_t)t.hi - (uint64_t)sg.base;
      chi = chi < most ? chi : most;
      const bool none = t.hi < sg.base || clo > most;
      if (sg.bits <= 32) {
        const uint32_t lo = (uint32_t)clo, width = (uint32_t)chi - lo;
#pragma unroll
        for (int u = 0; u < U; ++u) pass[u] = pass[u] && !none && (uint32_t)c[u] - lo <= width;
      } else {
#pragma unroll
        for (int u = 0; u < U; ++u) pass[u] = pass[u] && !none && c[u] - clo <= chi - clo;
      }
    }
  }
}

// One tile of SC_TILE rows per block: its passing rows as one bit per row and their number
// (OUT SCAN_MASK), the number alone (SCAN_COUNT), or their global row ids (SCAN_WRITE).  Each
// predicate is decoded and evaluated once, U rows of a thread at a time; the row ids then come
// from the masks (k_scan_expand).  Bound by a chain of latencies per tile, descriptors, column
// loads, then the program's instructions one after another (columns staged in LDS, or fewer or
// more rows at a time, were all slower): 40M rows of (date < d AND disc != 5) OR
// price * (100 - disc) > x took two passes of 1.03 ms each with one row per instruction and the
// predicate evaluated by the count and by the write, 186 + 25 us now; 60M rows of one interval
// 62 + 35 us.
enum { SCAN_MASK = 0, SCAN_COUNT = 1, SCAN_WRITE = 2 };
template <int OUT, int U, typename Pred>
__device__ __forceinline__ void scan_tile(const ScanArgs &a, uint64_t *__restrict__ masks,
                                          uint32_t *__restrict__ counts, const uint64_t *__restrict__ offs,
                                          uint32_t *__restrict__ out, Pred pred) {
  __shared__ uint32_t wc[SC_BLOCK / 64];
  const uint32_t seg = blockIdx.x / a.tiles_per_seg, tile = blockIdx.x % a.tiles_per_seg;
  const uint32_t nrows = a.ct.segs[0][seg].nrows;
  const uint32_t r0 = tile * SC_TILE;
  const char mode = a.modes ? a.modes[seg] : 'R';
  if (r0 >= nrows || mode == 'N') {
    if (OUT != SCAN_WRITE && threadIdx.x == 0) counts[blockIdx.x] = 0;
    return;
  }
  const unsigned lane = __lane_id(), wid = threadIdx.x / 64;
  const uint32_t left = nrows - r0;
  uint64_t run = OUT == SCAN_WRITE ? offs[blockIdx.x] : 0, mine = 0;
  uint32_t total = 0;
#pragma unroll 1
  for (int j0 = 0; j0 < SC_ITEMS; j0 += U) {
    uint32_t idx[U];
    bool pass[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {  // rows past the segment's end read its last row
      const uint32_t i = (uint32_t)(j0 + u) * SC_BLOCK + threadIdx.x;
      idx[u] = i < left ? i : left - 1;
      pass[u] = true;
    }
    if (mode != 'A') pred(seg, r0, idx, pass);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t i = (uint32_t)(j0 + u) * SC_BLOCK + threadIdx.x;
      const uint64_t bal = __builtin_amdgcn_ballot_w64(pass[u] && i < left);
      if (OUT != SCAN_WRITE) {
        total += (uint32_t)__popcll(bal);
        if (OUT == SCAN_MASK && lane == (unsigned)(j0 + u)) mine = bal;
      } else {
        if (lane == 0) wc[wid] = (uint32_t)__popcll(bal);
        __syncthreads();
        uint32_t before = 0, all = 0;
        for (int w = 0; w < SC_BLOCK / 64; ++w) {
          const uint32_t x = wc[w];
          before += w < (int)wid ? x : 0;
          all += x;
        }
        if (bal >> lane & 1) out[run + before + below_count(bal)] = (uint32_t)((uint64_t)seg * a.seg_rows + r0 + i);
        run += all;
        __syncthreads();
      }
    }
  }
  if (OUT != SCAN_WRITE) {
    // mask word 4 * j + wave of the tile: rows j * 256 + wave * 64 .. + 63
    if (OUT == SCAN_MASK && lane < SC_ITEMS)
      masks[(uint64_t)blockIdx.x * (SC_TILE / 64) + lane * (SC_BLOCK / 64) + wid] = mine;
    if (lane == 0) wc[wid] = total;
    __syncthreads();
    if (threadIdx.x == 0) {
      uint32_t s = 0;
      for (int w = 0; w < SC_BLOCK / 64; ++w) s += wc[w];
      counts[blockIdx.x] = s;
    }
  }
}

template <int OUT>
__global__ void __launch_bounds__(SC_BLOCK) k_scan_ranges(ScanArgs a, RangeSet rs, uint64_t *__restrict__ masks,
                                                          uint32_t *__restrict__ counts,
                                                          const uint64_t *__restrict__ offs,
                                                          uint32_t *__restrict__ out) {
  constexpr int U = 8;
  scan_tile<OUT, U>(a, masks, counts, offs, out,
                    [&](uint32_t seg, uint32_t r0, const uint32_t(&idx)[U], bool(&pass)[U]) {
                      ranges_pass<U>(rs, a.ct, seg, r0, idx, pass);
                    });
}

template <int OUT, int U>
__global__ void __launch_bounds__(SC_BLOCK) k_scan_prog(ScanArgs a, VProg p, uint64_t *__restrict__ masks,
                                                        uint32_t *__restrict__ counts,
                                                        const uint64_t *__restrict__ offs,
                                                        uint32_t *__restrict__ out) {
  extern __shared__ __align__(16) int64_t vm_stack[];
  scan_tile<OUT, U>(a, masks, counts, offs, out,
                    [&](uint32_t seg, uint32_t r0, const uint32_t(&idx)[U], bool(&pass)[U]) {
                      auto load = [&](int col, int64_t(&v)[U]) {
                        const aln_seg sg = a.ct.segs[col][seg];
                        uint64_t c[U];
                        unpack_codes<U>(a.ct.words[col] + sg.word_off + (uint64_t)(r0 >> 5) * sg.bits, sg.bits, idx, c);
#pragma unroll
                        for (int u = 0; u < U; ++u) v[u] = (int64_t)((uint64_t)sg.base + c[u]);
                      };
                      int64_t t[U];
                      vm_eval<U>(p, load, vm_stack + threadIdx.x, t);
#pragma unroll
                      for (int u = 0; u < U; ++u) pass[u] = t[u] != 0;
                    });
}

// Row ids of a tile's set mask bits.  Every wave scans the bit counts of the tile's 64 words
// and writes the rows of 16 of them.
__global__ void __launch_bounds__(SC_BLOCK) k_scan_expand(const uint64_t *__restrict__ masks, uint32_t seg_rows,
                                                          uint32_t tiles_per_seg,
                                                          const uint32_t *__restrict__ counts,
                                                          const uint64_t *__restrict__ offs,
                                                          uint32_t *__restrict__ out) {
  if (counts[blockIdx.x] == 0) return;
  const uint32_t seg = blockIdx.x / tiles_per_seg, tile = blockIdx.x % tiles_per_seg;
  const unsigned lane = __lane_id(), wid = threadIdx.x / 64;
  const uint64_t word = masks[(uint64_t)blockIdx.x * (SC_TILE / 64) + lane];
  const uint32_t n = (uint32_t)__popcll(word);
  uint32_t incl = n;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(incl, o, 64);
    if (lane >= (unsigned)o) incl += y;
  }
  const uint32_t first = incl - n;
  uint32_t *dst = out + offs[blockIdx.x];
  const uint32_t row = (uint32_t)((uint64_t)seg * seg_rows + tile * SC_TILE) + lane;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int w = (int)wid * 16 + j;
    const uint64_t m = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(word >> 32), w) << 32 |
                       (uint32_t)__builtin_amdgcn_readlane((int)word, w);
    const uint32_t at = (uint32_t)__builtin_amdgcn_readlane((int)first, w);
    if (m >> lane & 1) dst[at + below_count(m)] = row + 64u * (uint32_t)w;
  }
}

// Recognise a conjunction of "column OP constant" terms (multiplier 1) and code-set tests
// (LIKE) and turn it into one closed interval per column plus the set tests.  Returns false
// when the program has another shape.
static bool as_intervals(const aln_insn *p, int n, RangeC *out, int *nout, bool *empty) {
  *empty = false;
  *nout = 0;
  int64_t lo[ALN_MAX_COLS], hi[ALN_MAX_COLS];
  bool used[ALN_MAX_COLS] = {false};
  RangeC sets[ALN_MAX_INSN / 2];
  int nsets = 0;
  int i = 0;
  int pending = 0;  // predicates on the evaluation stack
  while (i < n) {
    if (p[i].op == ALN_I_AND) {
      if (pending < 2) return false;
      --pending;
      ++i;
      continue;
    }
    if (i + 1 < n && p[i].op == ALN_I_COL && p[i].k == 1 && p[i + 1].op == ALN_I_INSET) {
      if (nsets == ALN_MAX_INSN / 2 || p[i].a < 0 || p[i].a >= ALN_MAX_COLS) return false;
      sets[nsets++] = RangeC{p[i].a, 1, p[i + 1].k, (int64_t)p[i + 1].a};
      ++pending;
      i += 2;
      continue;
    }
    if (i + 2 >= n) return false;
    if (!(p[i].op == ALN_I_COL && p[i].k == 1 && p[i + 1].op == ALN_I_CONST &&
          p[i + 2].op == ALN_I_CMP))
      return false;
    int c = p[i].a;
    if (c < 0 || c >= ALN_MAX_COLS) return false;
    int64_t v = p[i + 1].k, l = INT64_MIN, h = INT64_MAX;
    switch (p[i + 2].a) {
      case 1:
        if (v == INT64_MIN) *empty = true; else h = v - 1;
        break;
      case 2:
        if (v == INT64_MAX) *empty = true; else l = v + 1;
        break;
      case 4: l = h = v; break;
      case 5: h = v; break;
      case 6: l = v; break;
      default: return false;
    }
    if (!used[c]) {
      used[c] = true;
      lo[c] = l;
      hi[c] = h;
    } else {
      lo[c] = l > lo[c] ? l : lo[c];
      hi[c] = h < hi[c] ? h : hi[c];
    }
    ++pending;
    i += 3;
  }
  if (pending != 1) return false;
  int k = 0;
  for (int c = 0; c < ALN_MAX_COLS; ++c)
    if (used[c]) {
      if (lo[c] > hi[c]) *empty = true;
      out[k++] = RangeC{c, 0, lo[c], hi[c]};
    }
  for (int j = 0; j < nsets; ++j) out[k++] = sets[j];
  *nout = k;
  return true;
}

static int fill_cols(const aln_col *cols, int ncols, ColTable *h) {
  ALN_REQUIRE(ncols >= 1 && ncols <= ALN_MAX_COLS, "column count %d outside 1..%d", ncols,
              ALN_MAX_COLS);
  memset(h, 0, sizeof(*h));
  for (int i = 0; i < ncols; ++i) {
    ALN_REQUIRE(cols[i].words || cols[i].nsegs == 0, "column %d has no words", i);
    ALN_REQUIRE(cols[i].segs, "column %d has no segment descriptors", i);
    ALN_REQUIRE(cols[i].nsegs == cols[0].nsegs, "columns differ in segment count");
    h->words[i] = cols[i].words;
    h->segs[i] = cols[i].segs;
  }
  return ALN_OK;
}

static int check_prog(const aln_insn *prog, int nprog) {
  ALN_REQUIRE(prog && nprog >= 1 && nprog <= ALN_MAX_INSN, "program length %d", nprog);
  int depth = 0, mx = 0;
  for (int i = 0; i < nprog; ++i) {
    int op = prog[i].op;
    ALN_REQUIRE(op >= ALN_I_COL && op <= ALN_I_FCMP, "bad instruction %d", op);
    if (op == ALN_I_COL) ALN_REQUIRE(prog[i].a >= 0 && prog[i].a < ALN_MAX_COLS, "bad column %d", prog[i].a);
    if (op == ALN_I_INSET)
      ALN_REQUIRE(prog[i].a >= 0 && (prog[i].a == 0 || prog[i].k != 0), "set test without a bit set");
    if (op == ALN_I_I2F) ALN_REQUIRE((prog[i].a == 0 || prog[i].a == 1) && depth > prog[i].a, "bad conversion");
    depth += (op == ALN_I_COL || op == ALN_I_CONST) ? 1 : (op == ALN_I_INSET || op == ALN_I_I2F) ? 0 : -1;
    ALN_REQUIRE(depth >= 1, "program underflows its stack");
    mx = depth > mx ? depth : mx;
  }
  ALN_REQUIRE(depth == 1 && mx <= ALN_MAX_STACK, "program leaves %d values (max depth %d)", depth, mx);
  return ALN_OK;
}

static int row_args(const aln_col *cols, int ncols, uint32_t seg_rows, const uint32_t *rows, uint64_t n, RowArgs *a) {
  ALN_TRY(fill_cols(cols, ncols, &a->ct));
  a->nsegs = cols[0].nsegs;
  a->seg_rows = seg_rows;
  a->seg_mul = seg_rows > 1 ? ~0ull / seg_rows + 1 : 0;
  a->rows = rows;
  a->n = n;
  return ALN_OK;
}
// Segments whose widest code positions fit in 32 bits.
static bool narrow_segments(uint32_t seg_rows) { return seg_rows <= (1u << 26); }

// Four rows per thread while their LDS stack is at most 32 KB (four values below the top),
// else one (up to 15 values, 30 KB).
template <int U>
static int eval_launch_rows(hipStream_t st, const RowArgs &a, const VProg &p, int64_t *out) {
  const uint64_t nb = (a.n + VM_BLOCK * U - 1) / (VM_BLOCK * U);
  ALN_REQUIRE(nb < (1ull << 31), "aln_eval: grid too large");
  const size_t lds = (size_t)p.slots * U * sizeof(int64_t) * VM_BLOCK;
  if (narrow_segments(a.seg_rows))
    hipLaunchKernelGGL((k_eval<U, uint32_t>), dim3((unsigned)nb), dim3(VM_BLOCK), lds, st, a, p, out);
  else
    hipLaunchKernelGGL((k_eval<U, uint64_t>), dim3((unsigned)nb), dim3(VM_BLOCK), lds, st, a, p, out);
  return check_launch("eval");
}
static int eval_launch(hipStream_t st, const RowArgs &a, const VProg &p, int64_t *out) {
  return p.slots <= 4 ? eval_launch_rows<4>(st, a, p, out) : eval_launch_rows<1>(st, a, p, out);
}

static int check_prog_cols(const aln_insn *prog, int nprog, int ncols) {
  for (int i = 0; i < nprog; ++i)
    if (prog[i].op == ALN_I_COL && prog[i].a >= ncols)
      return set_error(ALN_E_ARG, "program reads column %d of %d", prog[i].a, ncols);
  return ALN_OK;
}

// A checked scan: a conjunction of intervals and set tests, or a program of any shape.
struct ScanPlan {
  ScanArgs a;
  bool fast, empty;
  RangeSet rs;
  VProg prog;
};
static int scan_plan(const aln_col *cols, int ncols, uint32_t seg_rows, const aln_insn *prog, int nprog,
                     ScanPlan *s) {
  ALN_TRY(fill_cols(cols, ncols, &s->a.ct));
  ALN_TRY(check_prog(prog, nprog));
  s->a.seg_rows = seg_rows;
  s->a.tiles_per_seg = (seg_rows + SC_TILE - 1) / SC_TILE;
  s->a.modes = nullptr;
  s->rs.n = 0;
  s->empty = false;
  s->fast = as_intervals(prog, nprog, s->rs.r, &s->rs.n, &s->empty);
  if (!s->fast) vm_lower(prog, nprog, &s->prog);
  return ALN_OK;
}

// Eight rows per thread and instruction while their LDS stack leaves five blocks per CU
// (two values below the top, 32 KB), else two (up to 15 values, 60 KB).
template <int OUT>
static int scan_launch(hipStream_t st, const ScanPlan &s, uint32_t nblocks, uint64_t *masks, uint32_t *counts,
                       const uint64_t *offs, uint32_t *out) {
  const size_t row = sizeof(int64_t) * VM_BLOCK;
  if (s.fast)
    hipLaunchKernelGGL(k_scan_ranges<OUT>, dim3(nblocks), dim3(SC_BLOCK), 0, st, s.a, s.rs, masks, counts, offs, out);
  else if (s.prog.slots <= 2)
    hipLaunchKernelGGL((k_scan_prog<OUT, 8>), dim3(nblocks), dim3(SC_BLOCK), 8 * s.prog.slots * row, st, s.a, s.prog,
                       masks, counts, offs, out);
  else
    hipLaunchKernelGGL((k_scan_prog<OUT, 2>), dim3(nblocks), dim3(SC_BLOCK), 2 * s.prog.slots * row, st, s.a, s.prog,
                       masks, counts, offs, out);
  return check_launch(OUT == SCAN_WRITE ? "scan_write" : "scan_count");
}

// Segment of the source row behind each index: r = rows ? rows[idx[i]] : idx[i]; the last
// segment start <= r when starts are given (uneven file segments), else r / seg_rows.
__global__ void __launch_bounds__(256) k_row_segments(const uint32_t *__restrict__ idx, uint64_t n,
                                                      const uint32_t *__restrict__ rows,
                                                      const uint64_t *__restrict__ starts, uint32_t nstarts,
                                                      uint32_t seg_rows, int64_t *__restrict__ out) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256) {
    const uint64_t r = rows ? rows[idx[i]] : idx[i];
    int64_t seg;
    if (starts) {  // upper bound of r in starts[0, nstarts), minus one
      uint32_t lo = 0, hi = nstarts;
      while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (starts[mid] <= r) lo = mid + 1; else hi = mid;
      }
      seg = (int64_t)lo - 1;
    } else {
      seg = (int64_t)(r / seg_rows);
    }
    out[i] = seg;
  }
}

template <int DEC_ROWS>
static int launch_decode_rows(aln_ctx *c, const aln_col *col, uint32_t seg_rows, uint64_t row_begin, uint64_t n,
                              int64_t *d_out) {
  const uint64_t nb = (n + 256 * DEC_ROWS - 1) / (256 * DEC_ROWS);
  ALN_REQUIRE(nb < (1ull << 31), "decode: grid too large");
  hipLaunchKernelGGL(k_decode<DEC_ROWS>, dim3((unsigned)nb), dim3(256), 0, c->stream, col->words, col->segs,
                     col->nsegs, seg_rows, row_begin, n, d_out);
  return check_launch("decode");
}
static int launch_decode(aln_ctx *c, const aln_col *col, uint32_t seg_rows, uint64_t row_begin, uint64_t n,
                         int64_t *d_out) {
  if (seg_rows < DEC_SEG_ROWS && n < (1ull << 38))  // (blocks of 256 rows: the grid's limit)
    return launch_decode_rows<1>(c, col, seg_rows, row_begin, n, d_out);
  return launch_decode_rows<8>(c, col, seg_rows, row_begin, n, d_out);
}

// ---- fixed scratch of the allocation-free scan -----------------------------------------------
// aln_scan_filter_noalloc keeps its temporaries in this array instead of the context's
// workspace: the per-segment zone-map verdicts it uploads, the per-tile counts, their exclusive
// scan and the scan's partial sums and total (a mask bit per row would not fit: it evaluates
// the predicate again to write).  Every byte a call reads is written earlier in the same call,
// so nothing is cleared.  Each GPU holds its own copy for the life of the process; host code
// reaches it only through the address hipGetSymbolAddress returns on that device.
constexpr uint64_t NA_TILES = ALN_SCAN_NOALLOC_MAX_TILES;
constexpr size_t NA_TOTAL = 0;                                            // u64 scan total
constexpr size_t NA_MODES = 4096;                                         // u8 per segment
constexpr size_t NA_COUNTS = NA_MODES + NA_TILES;                         // u32 per tile
constexpr size_t NA_OFFS = NA_COUNTS + 4 * NA_TILES;                      // u64 per tile
constexpr size_t NA_SUMS = NA_OFFS + 8 * NA_TILES;                        // u64 per scan tile
constexpr size_t NA_BYTES = NA_SUMS + 8 * ((NA_TILES + 4095) / 4096 + 32);
static_assert(NA_TILES % 256 == 0, "scratch regions lose their alignment");

static __device__ __align__(256) unsigned char scratch[NA_BYTES];

constexpr int NA_MAX_DEVICES = 64;
static std::mutex g_na_mu;
static std::atomic<char *> g_na_ptr[NA_MAX_DEVICES];

int scan_scratch_attach(int device) {
  ALN_REQUIRE(device >= 0 && device < NA_MAX_DEVICES, "device %d outside 0..%d", device,
              NA_MAX_DEVICES - 1);
  std::lock_guard<std::mutex> lock(g_na_mu);
  if (g_na_ptr[device].load()) return ALN_OK;
  void *p = nullptr;
  hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p) {
    (void)hipGetLastError();
    return set_error(ALN_E_HIP, "hipGetSymbolAddress of the scan scratch on device %d failed: %s", device,
                     hipGetErrorString(e));
  }
  g_na_ptr[device].store(static_cast<char *>(p));
  return ALN_OK;
}

// The scratch address on the context's device, looked up now (with that device current for
// the call) if the context's creation could not.
static int scan_scratch(aln_ctx *c, char **out) {
  ALN_REQUIRE(c->device >= 0 && c->device < NA_MAX_DEVICES, "device %d", c->device);
  char *p = g_na_ptr[c->device].load();
  if (!p) {
    int cur = -1;
    ALN_HIP(hipGetDevice(&cur));
    if (cur != c->device) ALN_HIP(hipSetDevice(c->device));
    int r = scan_scratch_attach(c->device);
    if (cur != c->device) ALN_HIP(hipSetDevice(cur));
    ALN_TRY(r);
    p = g_na_ptr[c->device].load();
  }
  *out = p;
  return ALN_OK;
}

}  // namespace aln

using namespace aln;

extern "C" {

int aln_encode_plan(aln_ctx *c, const int64_t *d_vals, uint64_t nrows, uint32_t seg_rows,
                    uint32_t force_bits, aln_seg *h_segs, uint64_t *h_words) {
  ALN_REQUIRE(c && h_segs && h_words && seg_rows > 0, "aln_encode_plan: bad arguments");
  ALN_REQUIRE(nrows == 0 || d_vals, "aln_encode_plan: no values");
  ALN_REQUIRE(force_bits <= 64, "aln_encode_plan: force_bits %u", force_bits);
  ws_reset(c);
  uint32_t nsegs = (uint32_t)((nrows + seg_rows - 1) / seg_rows);
  *h_words = 0;
  if (nsegs == 0) return ALN_OK;
  const uint32_t bps = (uint32_t)grid_for(seg_rows, 256 * 16, 256);
  int64_t *part, *mm;
  ALN_TRY(ws(c, 2 * (size_t)nsegs, &mm));
  part = mm;  // (one block per segment: its partials are the ranges)
  if (bps > 1) ALN_TRY(ws(c, 2 * (size_t)nsegs * bps, &part));
  {
    ProfScope p(c, "seg_minmax");
    int64_t *pmax = part + (size_t)nsegs * bps;
    hipLaunchKernelGGL(k_seg_minmax, dim3(nsegs * bps), dim3(256), 0, c->stream, d_vals, nrows,
                       seg_rows, bps, part, pmax);
    if (bps > 1)
      hipLaunchKernelGGL(k_seg_minmax_final, dim3(nsegs), dim3(64), 0, c->stream, (const int64_t *)part,
                         (const int64_t *)pmax, bps, nsegs, mm);
  }
  ALN_TRY(check_launch("seg_minmax"));
  std::vector<int64_t> range(2 * (size_t)nsegs);
  ALN_TRY(copy_to_host(c, range.data(), mm, 16 * (size_t)nsegs));
  uint64_t off = 0;
  for (uint32_t s = 0; s < nsegs; ++s) {
    aln_seg &g = h_segs[s];
    uint64_t r0 = (uint64_t)s * seg_rows;
    g.nrows = (uint32_t)((r0 + seg_rows <= nrows) ? seg_rows : nrows - r0);
    g.vmin = range[s];
    g.vmax = range[nsegs + s];
    g.base = g.vmin;
    g.bits = bits_for_range_u((uint64_t)g.vmax - (uint64_t)g.vmin);
    if (force_bits) {
      ALN_REQUIRE(force_bits >= g.bits, "aln_encode_plan: segment %u needs %u bits > %u", s,
                  g.bits, force_bits);
      g.bits = force_bits;
      if (force_bits == 64) g.base = 0;
    }
    g.word_off = off;
    off += ((uint64_t)g.nrows * g.bits + 31) / 32;
  }
  *h_words = off;
  return ALN_OK;
}

int aln_encode_pack(aln_ctx *c, const int64_t *d_vals, uint64_t nrows, uint32_t seg_rows,
                    const aln_seg *h_segs, uint32_t *d_words, aln_seg *d_segs) {
  ALN_REQUIRE(c && h_segs && d_segs && seg_rows > 0, "aln_encode_pack: bad arguments");
  ws_reset(c);
  uint32_t nsegs = (uint32_t)((nrows + seg_rows - 1) / seg_rows);
  if (nsegs == 0) return ALN_OK;
  uint64_t maxw = 0, maxr = 0;
  for (uint32_t s = 0; s < nsegs; ++s) {
    uint64_t r0 = (uint64_t)s * seg_rows;
    uint32_t nr = (uint32_t)((r0 + seg_rows <= nrows) ? seg_rows : nrows - r0);
    ALN_REQUIRE(h_segs[s].nrows == nr && h_segs[s].bits <= 64,
                "aln_encode_pack: descriptor %u does not match the plan", s);
    uint64_t w = ((uint64_t)nr * h_segs[s].bits + 31) / 32;
    maxw = w > maxw ? w : maxw;
    maxr = nr > maxr ? nr : maxr;
  }
  ALN_REQUIRE(maxw == 0 || d_words, "aln_encode_pack: no word buffer");
  ALN_HIP(hipMemcpyAsync(d_segs, h_segs, sizeof(aln_seg) * nsegs, hipMemcpyHostToDevice, c->stream));
  if (maxw) {
    ProfScope p(c, "pack");
    for (uint32_t s0 = 0; s0 < nsegs; s0 += 65535) {
      uint32_t ns = nsegs - s0 < 65535 ? nsegs - s0 : 65535;
      hipLaunchKernelGGL(k_pack, dim3(grid_for(maxr, PK_TILE), ns), dim3(256), 0, c->stream,
                         d_vals, seg_rows, s0, (const aln_seg *)d_segs, d_words);
    }
  }
  ALN_TRY(check_launch("pack"));
  ALN_HIP(hipStreamSynchronize(c->stream));
  return ALN_OK;
}

int aln_plain_col(aln_ctx *c, const int64_t *d_vals, uint64_t nrows, uint32_t seg_rows,
                  int32_t decimals, aln_seg *d_segs, aln_col *out) {
  ALN_REQUIRE(c && d_segs && out && seg_rows > 0, "aln_plain_col: bad arguments");
  uint32_t nsegs = (uint32_t)((nrows + seg_rows - 1) / seg_rows);
  std::vector<aln_seg> h(nsegs);
  for (uint32_t s = 0; s < nsegs; ++s) {
    uint64_t r0 = (uint64_t)s * seg_rows;
    h[s].nrows = (uint32_t)((r0 + seg_rows <= nrows) ? seg_rows : nrows - r0);
    h[s].word_off = 2 * r0;
    h[s].base = 0;
    h[s].bits = 64;
    h[s].vmin = INT64_MIN;
    h[s].vmax = INT64_MAX;
  }
  if (nsegs) ALN_TRY(copy_to_device(c, d_segs, h.data(), sizeof(aln_seg) * nsegs));
  out->words = (const uint32_t *)d_vals;
  out->segs = d_segs;
  out->nsegs = nsegs;
  out->decimals = decimals;
  return ALN_OK;
}

int aln_decode(aln_ctx *c, const aln_col *col, uint32_t seg_rows, uint64_t row_begin,
               uint64_t row_end, int64_t *d_out) {
  ALN_REQUIRE(c && col && seg_rows > 0 && row_end >= row_begin, "aln_decode: bad arguments");
  ALN_REQUIRE(row_end <= (uint64_t)col->nsegs * seg_rows, "aln_decode: rows beyond the column");
  uint64_t n = row_end - row_begin;
  if (!n) return ALN_OK;
  ProfScope p(c, "decode");
  ALN_TRY(launch_decode(c, col, seg_rows, row_begin, n, d_out));
  return ALN_OK;
}

int aln_gather(aln_ctx *c, const aln_col *col, uint32_t seg_rows, const uint32_t *d_rows,
               uint64_t n, int64_t *d_out) {
  ALN_REQUIRE(c && col && seg_rows > 0, "aln_gather: bad arguments");
  if (!n) return ALN_OK;
  ProfScope p(c, "gather");
  if (col->nsegs == 0) return fill_i64(c, d_out, n, 0);
  if (!d_rows && n < (1ull << 32)) return launch_decode(c, col, seg_rows, 0, n, d_out);
  constexpr int U = 4;
  RowArgs a;
  a.ct.words[0] = col->words;
  a.ct.segs[0] = col->segs;
  a.nsegs = col->nsegs;
  a.seg_rows = seg_rows;
  a.seg_mul = seg_rows > 1 ? ~0ull / seg_rows + 1 : 0;
  a.rows = d_rows;
  a.n = n;
  const uint64_t nb = (n + 256 * U - 1) / (256 * U);
  ALN_REQUIRE(nb < (1ull << 31), "aln_gather: grid too large");
  if (narrow_segments(seg_rows))
    hipLaunchKernelGGL((k_gather<U, uint32_t>), dim3((unsigned)nb), dim3(256), 0, c->stream, a, d_out);
  else
    hipLaunchKernelGGL((k_gather<U, uint64_t>), dim3((unsigned)nb), dim3(256), 0, c->stream, a, d_out);
  return check_launch("gather");
}

int aln_eval(aln_ctx *c, const aln_col *cols, int ncols, uint32_t seg_rows,
             const aln_insn *prog, int nprog, const uint32_t *d_rows, uint64_t n,
             int64_t *d_out) {
  ALN_REQUIRE(c && cols && seg_rows > 0, "aln_eval: bad arguments");
  ws_reset(c);
  if (!n) return ALN_OK;
  ALN_TRY(check_prog_cols(prog, nprog, ncols));
  RowArgs a;
  VProg p;
  ALN_TRY(row_args(cols, ncols, seg_rows, d_rows, n, &a));
  ALN_TRY(check_prog(prog, nprog));
  vm_lower(prog, nprog, &p);
  ProfScope ps(c, "eval");
  if (cols[0].nsegs == 0) return fill_i64(c, d_out, n, 0);
  return eval_launch(c->stream, a, p, d_out);
}

int aln_apply_perm(aln_ctx *c, const int64_t *d_in, const uint32_t *d_perm, uint64_t n,
                   int64_t *d_out) {
  ALN_REQUIRE(c && (n == 0 || (d_in && d_perm && d_out)), "aln_apply_perm: bad arguments");
  if (!n) return ALN_OK;
  ProfScope p(c, "apply_perm");
  hipLaunchKernelGGL(k_apply_perm, dim3(grid_for(n, 256, 65536)), dim3(256), 0, c->stream, d_in,
                     d_perm, n, d_out);
  return check_launch("apply_perm");
}

int aln_like_dict(aln_ctx *c, const char *d_entries, uint64_t n, uint32_t width, const char *h_pattern,
                  uint32_t *d_bits) {
  ALN_REQUIRE(c && h_pattern && (n == 0 || (d_entries && d_bits)), "aln_like_dict: bad arguments");
  ALN_REQUIRE(width >= 1 && width <= LIKE_MAX_WIDTH, "aln_like_dict: width %u outside 1..%u", width, LIKE_MAX_WIDTH);
  if (!n) return ALN_OK;
  ALN_REQUIRE(n < (1ull << 37), "aln_like_dict: %llu entries", (unsigned long long)n);
  ws_reset(c);
  const size_t plen = strlen(h_pattern) + 1;
  char *dp;
  ALN_TRY(ws(c, plen, &dp));
  ALN_TRY(copy_to_device(c, dp, h_pattern, plen));
  ProfScope p(c, "like_dict");
  hipLaunchKernelGGL(k_like_dict, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, c->stream, d_entries, n, width,
                     (const char *)dp, d_bits);
  ALN_TRY(check_launch("like_dict"));
  ALN_HIP(hipStreamSynchronize(c->stream));
  return ALN_OK;
}

int aln_dict_lookup(aln_ctx *c, const int64_t *d_codes, uint64_t n, const int64_t *d_table, uint64_t ntable,
                    int64_t *d_out) {
  ALN_REQUIRE(c && (n == 0 || (d_codes && d_out)) && (ntable == 0 || d_table), "aln_dict_lookup: bad arguments");
  if (!n) return ALN_OK;
  ProfScope p(c, "dict_lookup");
  hipLaunchKernelGGL(k_dict_lookup, dim3(grid_for(n, 256, 65536)), dim3(256), 0, c->stream, d_codes, n, d_table,
                     ntable, d_out);
  return check_launch("dict_lookup");
}

int aln_scan_filter(aln_ctx *c, const aln_col *cols, int ncols, uint32_t seg_rows,
                    const aln_insn *prog, int nprog, const char *seg_modes, uint32_t *d_row_ids,
                    uint64_t cap, uint64_t *h_count) {
  ALN_REQUIRE(c && cols && h_count && seg_rows > 0, "aln_scan_filter: bad arguments");
  ws_reset(c);
  ALN_TRY(check_prog_cols(prog, nprog, ncols));
  uint32_t nsegs = cols[0].nsegs;
  ALN_REQUIRE((uint64_t)nsegs * seg_rows <= (1ull << 32), "aln_scan_filter: more than 2^32 rows");
  *h_count = 0;
  if (nsegs == 0) return ALN_OK;
  ScanPlan s;
  ALN_TRY(scan_plan(cols, ncols, seg_rows, prog, nprog, &s));
  if (s.fast && s.empty) return ALN_OK;
  if (seg_modes) {
    char *dmodes;
    ALN_TRY(ws(c, nsegs, &dmodes));
    ALN_HIP(hipMemcpyAsync(dmodes, seg_modes, nsegs, hipMemcpyHostToDevice, c->stream));
    s.a.modes = dmodes;
  }
  const uint64_t nblocks = (uint64_t)nsegs * s.a.tiles_per_seg;
  ALN_REQUIRE(nblocks < (1ull << 31), "aln_scan_filter: grid too large");
  uint32_t *counts;
  uint64_t *offs, *masks;
  ALN_TRY(ws(c, nblocks, &counts));
  ALN_TRY(ws(c, nblocks, &offs));
  ALN_TRY(ws(c, nblocks * (SC_TILE / 64), &masks));
  {
    ProfScope p(c, "scan_count");
    ALN_TRY(scan_launch<SCAN_MASK>(c->stream, s, (uint32_t)nblocks, masks, counts, nullptr, nullptr));
  }
  uint64_t total = 0;
  ALN_TRY(exclusive_scan_u32(c, counts, nblocks, offs, &total));
  *h_count = total;
  if (total > cap) return set_error(ALN_E_CAPACITY, "aln_scan_filter: %llu rows pass, capacity %llu",
                                    (unsigned long long)total, (unsigned long long)cap);
  if (total == 0) return ALN_OK;
  ALN_REQUIRE(d_row_ids, "aln_scan_filter: no output buffer");
  {
    ProfScope p(c, "scan_write");
    hipLaunchKernelGGL(k_scan_expand, dim3((unsigned)nblocks), dim3(SC_BLOCK), 0, c->stream, (const uint64_t *)masks,
                       seg_rows, s.a.tiles_per_seg, (const uint32_t *)counts, (const uint64_t *)offs, d_row_ids);
  }
  ALN_TRY(check_launch("scan_write"));
  return stream_wait(c);
}

int aln_row_segments(aln_ctx *c, const uint32_t *d_idx, uint64_t n, const uint32_t *d_rows,
                     const uint64_t *d_starts, uint32_t nstarts, uint32_t seg_rows, int64_t *d_out) {
  ALN_REQUIRE(c && (n == 0 || (d_idx && d_out)), "aln_row_segments: bad arguments");
  ALN_REQUIRE(d_starts ? nstarts > 0 : seg_rows > 0, "aln_row_segments: no segmentation");
  if (n == 0) return ALN_OK;
  hipLaunchKernelGGL(k_row_segments, dim3(grid_for(n, 256, 65536)), dim3(256), 0, c->stream, d_idx, n, d_rows,
                     d_starts, nstarts, seg_rows, d_out);
  return check_launch("row_segments");
}

int aln_scan_filter_noalloc(aln_ctx *c, const aln_col *cols, int ncols, uint32_t seg_rows,
                            const aln_insn *prog, int nprog, const char *seg_modes,
                            uint32_t *d_row_ids, uint64_t cap, uint64_t *h_count) {
  ALN_REQUIRE(c && cols && h_count && seg_rows > 0, "aln_scan_filter_noalloc: bad arguments");
  ALN_TRY(check_prog_cols(prog, nprog, ncols));
  ScanPlan s;
  ALN_TRY(scan_plan(cols, ncols, seg_rows, prog, nprog, &s));
  const uint32_t nsegs = cols[0].nsegs;
  ALN_REQUIRE((uint64_t)nsegs * seg_rows <= (1ull << 32), "aln_scan_filter_noalloc: more than 2^32 rows");
  *h_count = 0;
  if (nsegs == 0) return ALN_OK;
  const uint64_t nblocks = (uint64_t)nsegs * s.a.tiles_per_seg;
  if (nblocks > NA_TILES)
    return set_error(ALN_E_ARG,
                     "aln_scan_filter_noalloc: %u segments of %u rows are %llu tiles of %d rows; the fixed "
                     "scratch holds %llu tiles (use aln_scan_filter)",
                     nsegs, seg_rows, (unsigned long long)nblocks, SC_TILE, (unsigned long long)NA_TILES);
  if (s.fast && s.empty) return ALN_OK;
  char *base;
  ALN_TRY(scan_scratch(c, &base));
  uint64_t *tot = reinterpret_cast<uint64_t *>(base + NA_TOTAL);
  uint32_t *counts = reinterpret_cast<uint32_t *>(base + NA_COUNTS);
  uint64_t *offs = reinterpret_cast<uint64_t *>(base + NA_OFFS);
  uint64_t *sums = reinterpret_cast<uint64_t *>(base + NA_SUMS);
  if (seg_modes) {
    s.a.modes = base + NA_MODES;
    ALN_HIP(hipMemcpyAsync(base + NA_MODES, seg_modes, nsegs, hipMemcpyHostToDevice, c->stream));
  }
  ALN_TRY(scan_launch<SCAN_COUNT>(c->stream, s, (uint32_t)nblocks, nullptr, counts, nullptr, nullptr));
  ALN_TRY(exclusive_scan_u32_buf(c->stream, counts, nblocks, offs, sums, tot));
  uint64_t total = 0;
  ALN_HIP(hipMemcpyAsync(&total, tot, sizeof(total), hipMemcpyDeviceToHost, c->stream));
  ALN_HIP(hipStreamSynchronize(c->stream));
  *h_count = total;
  if (total > cap)
    return set_error(ALN_E_CAPACITY, "aln_scan_filter_noalloc: %llu rows pass, capacity %llu",
                     (unsigned long long)total, (unsigned long long)cap);
  if (total == 0) return ALN_OK;
  ALN_REQUIRE(d_row_ids, "aln_scan_filter_noalloc: no output buffer");
  ALN_TRY(scan_launch<SCAN_WRITE>(c->stream, s, (uint32_t)nblocks, nullptr, counts, offs, d_row_ids));
  ALN_HIP(hipStreamSynchronize(c->stream));
  return ALN_OK;
}

}  // extern "C"
