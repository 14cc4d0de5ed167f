// LSD radix sort, stable multi-key ORDER BY and top-k.
//
// The reference sorts with one thrust::stable_sort_by_key per key, last key first
// (update_permutation, sorts.cu:17-70; emit_order, operators.cu:1675-1763).  Here each key
// is first mapped to an order-preserving unsigned code of just the bits its range needs
// (v - min, or max - v for DESC); when all codes fit in 64 bits they are concatenated and
// sorted once, otherwise one stable radix sort per key runs from the last key to the first.
//
// Radix sort: 8-bit digits, least significant first, each pass stable.  A first kernel
// counts pass 0's digits per block of 16384 items and finds the bits in which the codes
// differ; a pass whose digit every item shares is skipped.  Each pass scans its per-(digit,
// block) counts in digit-major order, which gives every 4096-item tile the first output
// position of each of its digits, and one kernel scatters: a block reorders its tile by
// digit in LDS (ranks from digit matching through LDS lane masks, in memory order) and
// stores every digit's run at consecutive addresses; each XCD takes a contiguous range of
// tiles, so neighbouring runs meet in one L2.  The passes after the first count their own
// digit from the keys the previous pass wrote.  A permutation sort stores only the key
// bytes the later passes read (8 or 4 per key), and its last pass stores none.  The first
// pass of an ORDER BY computes the codes from the key columns itself.  No kernel waits on
// another workgroup.
#include <string.h>

#include <algorithm>
#include <vector>

#include "aln_internal.h"

namespace aln {

struct KeySet {
  const int64_t *k[ALN_MAX_KEYS];
  int64_t ref[ALN_MAX_KEYS];  // min (ASC) or max (DESC)
  uint32_t shift[ALN_MAX_KEYS];
  int32_t desc[ALN_MAX_KEYS];
  int n;
};

// Composite order-preserving code: key 0 in the most significant bits.
__global__ void k_codes(KeySet ks, const uint32_t *__restrict__ perm, uint64_t n,
                        uint64_t *__restrict__ code, uint32_t *__restrict__ idx) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * 256) {
    uint64_t r = perm ? perm[i] : i;
    uint64_t c = 0;
    for (int k = 0; k < ks.n; ++k) {
      int64_t v = ks.k[k][r];
      uint64_t f = ks.desc[k] ? (uint64_t)ks.ref[k] - (uint64_t)v : (uint64_t)v - (uint64_t)ks.ref[k];
      if (ks.shift[k] < 64) c |= f << ks.shift[k];
    }
    code[i] = c;
    if (idx) idx[i] = (uint32_t)r;
  }
}

__device__ __forceinline__ uint64_t ks_code(const KeySet &ks, uint64_t r) {
  uint64_t c = 0;
  for (int k = 0; k < ks.n; ++k) {
    int64_t v = ks.k[k][r];
    uint64_t f = ks.desc[k] ? (uint64_t)ks.ref[k] - (uint64_t)v : (uint64_t)v - (uint64_t)ks.ref[k];
    if (ks.shift[k] < 64) c |= f << ks.shift[k];
  }
  return c;
}

constexpr int RS_BITS = 8;
constexpr int RS_BINS = 1 << RS_BITS;
constexpr int RS_BLOCK = 512;
constexpr int RS_WAVES = RS_BLOCK / 64;
constexpr int RS_ITEMS = 8;
constexpr int RS_TILE = RS_BLOCK * RS_ITEMS;  // items one scatter block reorders in LDS
constexpr int RS_WAVE_ITEMS = 64 * RS_ITEMS;
constexpr int RS_SUB = 4;
constexpr int RS_SUPER = RS_TILE * RS_SUB;  // items one count block counts
constexpr int RS_MAX_PASSES = 8;
constexpr int RS_SCAN_BLOCK = 256;
constexpr uint32_t RS_XCDS = 8;
// From this size on the host reads which bits vary between the codes and skips the passes
// whose digit every item shares; smaller sorts run every pass without a synchronisation.
constexpr uint64_t RS_SYNC_MIN = 1ull << 20;
static_assert(RS_BINS * 2 == RS_BLOCK, "threads 0..255 own one digit each");
static_assert(RS_SUPER % (RS_BLOCK * 4) == 0, "count loop");

template <int B>
struct KeyWord;
template <>
struct KeyWord<4> {
  typedef uint32_t T;
};
template <>
struct KeyWord<8> {
  typedef uint64_t T;
};

// Bytes a key of `bits` bits is stored in: 4 or 8 (scattered stores of narrower words
// cost as much per item as 4-byte ones).
static inline int key_word(uint32_t bits) { return bits <= 32 ? 4 : 8; }

// The items of one pass.  KI (bytes per stored key) 4, 8: keys and values from arrays;
// KI 0: codes computed from the key columns at row r = vals ? vals[i] : i, with value r.
// No values: the item's number.
struct RsIn {
  const void *keys;
  const uint32_t *vals;
  KeySet ks;
};

template <int KI>
__device__ __forceinline__ uint64_t rs_key(const RsIn &in, uint64_t i) {
  if constexpr (KI == 0) {
    return ks_code(in.ks, in.vals ? in.vals[i] : i);
  } else {
    typedef typename KeyWord<KI>::T T;
    return (uint64_t)__builtin_nontemporal_load(static_cast<const T *>(in.keys) + i);
  }
}
template <int KI>
__device__ __forceinline__ uint32_t rs_val(const RsIn &in, uint64_t i) {
  if (!in.vals) return (uint32_t)i;
  return __builtin_nontemporal_load(in.vals + i);
}

// Codes (and, VALS, values) of the N items i0 + j * stride; items at n and beyond get
// code and value 0.  From key columns, the rows are read first and then each column's N
// values, so the loads of all N items are in flight together.
template <int KI, int N, bool VALS>
__device__ __forceinline__ void rs_load(const RsIn &in, uint64_t n, uint64_t i0, uint32_t stride,
                                        uint64_t *key, uint32_t *val) {
  if constexpr (KI == 0) {
    uint64_t r[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      uint64_t i = i0 + (uint64_t)j * stride;
      r[j] = i < n ? (in.vals ? (uint64_t)__builtin_nontemporal_load(in.vals + i) : i) : 0;
      key[j] = 0;
      if (VALS) val[j] = (uint32_t)r[j];
    }
    for (int k = 0; k < in.ks.n; ++k) {
      const int64_t *col = in.ks.k[k];
      const uint64_t ref = (uint64_t)in.ks.ref[k];
      const uint32_t sh = in.ks.shift[k];
      const bool desc = in.ks.desc[k];
      int64_t v[N];
#pragma unroll
      for (int j = 0; j < N; ++j) v[j] = col[r[j]];
#pragma unroll
      for (int j = 0; j < N; ++j) {
        uint64_t f = desc ? ref - (uint64_t)v[j] : (uint64_t)v[j] - ref;
        if (sh < 64) key[j] |= f << sh;
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      uint64_t i = i0 + (uint64_t)j * stride;
      key[j] = i < n ? rs_key<KI>(in, i) : 0;
      if (VALS) val[j] = i < n ? rs_val<KI>(in, i) : 0;
    }
  }
}

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x) {
  const unsigned lane = __lane_id();
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    uint32_t y = __shfl_up(x, d, 64);
    if (lane >= (unsigned)d) x += y;
  }
  return x;
}

// Digit counts of one pass, block s over items [s * RS_SUPER, +RS_SUPER): cnt[digit *
// nsuper + s] (digit-major, for the scan) and, per tile of the block, the count of each
// digit in the block's earlier tiles: sub[(s * RS_SUB + tile) * 256 + digit].  VARY: also
// ORs code ^ (code of item 0) into *vary, the bits in which the codes differ.
template <int KI, bool VARY>
__global__ void __launch_bounds__(RS_BLOCK) k_rs_count(RsIn in, uint64_t n, uint32_t sh, uint32_t mask,
                                                       uint32_t nsuper, uint32_t *__restrict__ cnt,
                                                       uint16_t *__restrict__ sub,
                                                       unsigned long long *__restrict__ vary) {
  __shared__ uint32_t h[RS_SUB][RS_BINS];
  __shared__ uint64_t wv[RS_WAVES];
  const uint32_t t = threadIdx.x, s = blockIdx.x;
  for (uint32_t i = t; i < RS_SUB * RS_BINS; i += RS_BLOCK) (&h[0][0])[i] = 0;
  __syncthreads();
  const uint64_t lo = (uint64_t)s * RS_SUPER;
  uint64_t v = 0;
  const uint64_t c0 = VARY ? rs_key<KI>(in, 0) : 0;
  for (int r = 0; r < RS_SUPER / (RS_BLOCK * 4); ++r) {
    uint64_t k[4];
    const uint64_t i0 = lo + (uint64_t)r * 4 * RS_BLOCK + t;
    rs_load<KI, 4, false>(in, n, i0, RS_BLOCK, k, nullptr);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      uint64_t i = i0 + (uint64_t)u * RS_BLOCK;
      if (i < n) {
        atomicAdd(&h[(uint32_t)((i - lo) / RS_TILE)][(uint32_t)(k[u] >> sh) & mask], 1u);
        if (VARY) v |= k[u] ^ c0;
      }
    }
  }
  if (VARY) {
    for (int d = 32; d > 0; d >>= 1) v |= __shfl_xor(v, d, 64);
    if (__lane_id() == 0) wv[t / 64] = v;
  }
  __syncthreads();
  if (t < RS_BINS) {
    uint32_t run = 0;
#pragma unroll
    for (int j = 0; j < RS_SUB; ++j) {
      sub[((uint64_t)s * RS_SUB + j) * RS_BINS + t] = (uint16_t)run;
      run += h[j][t];
    }
    cnt[(uint64_t)t * nsuper + s] = run;
  }
  if (VARY && t == 0) {
    uint64_t all = 0;
    for (int w = 0; w < RS_WAVES; ++w) all |= wv[w];
    if (all) atomicOr(vary, (unsigned long long)all);
  }
}

// Exclusive scan of each digit's row of block counts, written transposed for the scatter
// blocks: excl[s * 256 + d]; tot[d] = the row's sum (one block per digit).
__global__ void __launch_bounds__(RS_SCAN_BLOCK) k_rs_rowscan(const uint32_t *__restrict__ cnt, uint32_t nsuper,
                                                              uint32_t *__restrict__ excl,
                                                              uint32_t *__restrict__ tot) {
  __shared__ uint32_t wsum[RS_SCAN_BLOCK / 64];
  const uint32_t d = blockIdx.x, t = threadIdx.x, lane = __lane_id(), wid = t / 64;
  const uint32_t per = (nsuper + RS_SCAN_BLOCK - 1) / RS_SCAN_BLOCK;
  const uint32_t *row = cnt + (uint64_t)d * nsuper;
  const uint32_t b = t * per, e = b + per < nsuper ? b + per : nsuper;
  uint32_t local = 0;
  for (uint32_t i = b; i < e; ++i) local += row[i];
  uint32_t incl = wave_incl_scan(local);
  if (lane == 63) wsum[wid] = incl;
  __syncthreads();
  uint32_t before = incl - local;
  for (uint32_t w = 0; w < wid; ++w) before += wsum[w];
  for (uint32_t i = b; i < e; ++i) {
    uint32_t x = row[i];
    excl[(uint64_t)i * RS_BINS + d] = before;
    before += x;
  }
  if (t == RS_SCAN_BLOCK - 1) tot[d] = before;
}

// One pass: digit = (stored key >> sh) & mask; keys are written as (stored key >> oshift)
// in KO bytes (KO 0: not written).  Tile b of count block s = b / RS_SUB stores digit d
// from position base[d] + excl[s * 256 + d] + sub[b * 256 + d], base[d] = the items of
// the digits below d (an exclusive scan of tot, made by every block).
struct RsPass {
  RsIn in;
  uint64_t n;
  const uint32_t *tot, *excl;
  const uint16_t *sub;
  void *kout;
  uint32_t *vout;
  uint32_t sh, mask, oshift, nsuper;
};

// One tile of RS_TILE items per block (8 waves x 64 lanes x 8 items; wave, then (item,
// lane) order is memory order): LDS lane masks match the digits of each wave row, per-wave
// digit counts place the waves, the tile is reordered by digit in LDS and each digit's run
// is stored at consecutive addresses.
template <int KI, int KO>
__global__ void __launch_bounds__(RS_BLOCK) k_rs_scatter(RsPass a) {
  __shared__ uint64_t sk[RS_TILE];
  __shared__ uint32_t sv[RS_TILE];
  __shared__ uint16_t wc[RS_WAVES][RS_BINS];
  __shared__ uint32_t gdel[RS_BINS];
  __shared__ uint32_t wsum[RS_BINS / 64], bsum[RS_BINS / 64];
  const unsigned t = threadIdx.x, lane = __lane_id(), wid = t / 64;
  // Workgroups go to the 8 XCDs round-robin: give each XCD a contiguous range of tiles, so
  // neighbouring tiles' runs of a digit (adjacent in the output) meet in the same L2.
  const uint32_t q = gridDim.x / RS_XCDS, rm = gridDim.x % RS_XCDS;
  const uint32_t x = blockIdx.x % RS_XCDS;
  const uint32_t tile = x * q + (x < rm ? x : rm) + blockIdx.x / RS_XCDS;
  const uint64_t n = a.n;
  const uint32_t sh = a.sh, mask = a.mask;
  // during ranking, sk holds one 64-bit lane mask per (wave, digit)
  uint64_t *pm = sk;
  static_assert(RS_WAVES * RS_BINS <= RS_TILE, "masks fit in the key buffer");
  for (int w = t; w < RS_WAVES * RS_BINS; w += RS_BLOCK) {
    (&wc[0][0])[w] = 0;
    pm[w] = 0;
  }
  const uint64_t tbase = (uint64_t)tile * RS_TILE;
  const uint64_t base = tbase + (uint64_t)wid * RS_WAVE_ITEMS;
  // this tile's first output position of digit t, read before the items so that its
  // latency overlaps theirs
  uint32_t first = 0, dtot = 0;
  if (t < RS_BINS) {
    first = a.excl[(uint64_t)(tile / RS_SUB) * RS_BINS + t] + a.sub[(uint64_t)tile * RS_BINS + t];
    dtot = a.tot[t];
  }
  uint64_t key[RS_ITEMS];
  uint32_t val[RS_ITEMS], rank[RS_ITEMS];
  rs_load<KI, RS_ITEMS, true>(a.in, n, base + lane, 64, key, val);
  __syncthreads();
  // Lanes of one wave row with equal digits: each lane ORs its bit into the row's mask of
  // its digit and reads the mask back (a wave's LDS operations complete in order); the
  // lowest such lane then advances the digit's count and clears the mask.
#pragma unroll
  for (int j = 0; j < RS_ITEMS; ++j) {
    bool valid = base + (uint64_t)j * 64 + lane < n;
    uint32_t d = (uint32_t)(key[j] >> sh) & mask;
    uint64_t *slot = pm + wid * RS_BINS + d;
    if (valid) __hip_atomic_fetch_or(slot, 1ull << lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    uint64_t peers = valid ? __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) : 0;
    uint32_t before = valid ? wc[wid][d] : 0;
    const uint32_t below = below_count(peers);  // peers in lower lanes
    rank[j] = before + below;
    if (valid && below == 0) {
      wc[wid][d] = (uint16_t)(before + (uint32_t)__popcll(peers));
      __hip_atomic_store(slot, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
  __syncthreads();
  uint32_t cnt = 0, incl = 0, bincl = 0;
  if (t < RS_BINS) {
#pragma unroll
    for (int w = 0; w < RS_WAVES; ++w) {
      uint32_t x = wc[w][t];
      wc[w][t] = (uint16_t)cnt;
      cnt += x;
    }
    incl = wave_incl_scan(cnt);
    bincl = wave_incl_scan(dtot);
    if (lane == 63) {
      wsum[wid] = incl;
      bsum[wid] = bincl;
    }
  }
  __syncthreads();
  if (t < RS_BINS) {
    uint32_t tstart = incl - cnt, dbase = bincl - dtot;
    for (unsigned w = 0; w < wid; ++w) {
      tstart += wsum[w];
      dbase += bsum[w];
    }
#pragma unroll
    for (int w = 0; w < RS_WAVES; ++w) wc[w][t] = (uint16_t)(wc[w][t] + tstart);
    gdel[t] = dbase + first - tstart;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < RS_ITEMS; ++j) {
    if (base + (uint64_t)j * 64 + lane < n) {
      uint32_t d = (uint32_t)(key[j] >> sh) & mask;
      uint32_t pos = wc[wid][d] + rank[j];
      sk[pos] = key[j];
      sv[pos] = val[j];
    }
  }
  __syncthreads();
  const uint32_t nvalid = n - tbase < (uint64_t)RS_TILE ? (uint32_t)(n - tbase) : (uint32_t)RS_TILE;
#pragma unroll
  for (int j = 0; j < RS_ITEMS; ++j) {
    uint32_t i = (uint32_t)j * RS_BLOCK + t;
    if (i < nvalid) {
      uint64_t k = sk[i];
      uint32_t dest = gdel[(uint32_t)(k >> sh) & mask] + i;
      if constexpr (KO != 0) {
        typedef typename KeyWord<KO>::T T;
        static_cast<T *>(a.kout)[dest] = (T)(k >> a.oshift);
      }
      a.vout[dest] = sv[i];
    }
  }
}

// ---- bucket sort after two top-digit passes ------------------------------------------------
// Once two stable passes on the two most significant varying digits have put the rows in
// order of their codes' high part (code >> topshift, "buckets"), each block of k_rs_bins and
// k_rs_local owns the buckets that start in its window of `w` positions and sorts them, with
// their continuation past the window, in LDS; only the permutation is stored.  A bucket that
// does not end within RS_TILE positions of its window sets *overflow (the host then tries
// smaller windows, or sorts by the digit passes alone).
//
// k_rs_bins (below) places the rows by one counting pass; the windows whose rows crowd into few
// bins (many codes with equal bits there) are left to k_rs_local, which makes no assumption:
//
// In the block each code's high part is replaced by its bucket's ordinal, the rows of
// [lo, hi) are packed to LDS positions 0 .. m-1, and three or four stable LDS passes rank
// them by the next two varying digits and then the ordinal.  Rows that still tie on every
// bit above the remaining digits stand in runs of consecutive positions (short for spread
// keys); each row's place in its run is the number of rows of the run with a smaller code,
// or an equal code and an earlier position.  A run longer than RL_RUN makes the block rank
// all remaining digits by LDS passes instead, from the order it has (which keeps equal
// codes in input order, so the result is the same).
constexpr uint32_t RL_W = RS_TILE / 2;  // the smallest window, half of a block's positions
constexpr uint32_t RL_RUN = 32;
// Bits of ctl[0]; ctl[1] counts the windows k_rs_bins left to k_rs_local.  RL_CROWDED: so many of them
// that the windows not begun yet go there at once.
constexpr uint32_t RL_OVERFLOW = 1, RL_REDO = 2, RL_CROWDED = 4;
__device__ __forceinline__ uint32_t rl_peek(const uint32_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Sets a bit once: thousands of atomics on one address take 6 ns each.
__device__ __forceinline__ void rl_set(uint32_t *ctl, uint32_t bit) {
  if (!(rl_peek(ctl) & bit)) atomicOr(ctl, bit);
}

struct RsLocal {
  const uint64_t *keys;
  const uint32_t *vals;
  uint32_t *vout;
  uint8_t *heads;  // may be NULL: 1 where a position's code differs from the one before
  uint32_t *ctl;
  uint8_t *redo;  // per window: left by k_rs_bins to k_rs_local
  uint64_t n;
  uint32_t w;     // window: positions whose buckets a block owns (a multiple of 64)
  uint32_t hish, himask;  // the most significant varying digit
  uint32_t nblk, topshift, nlow;  // nlow >= 2 remaining varying digits:
  uint32_t sh[RS_MAX_PASSES], mask[RS_MAX_PASSES];  // least significant first
};

// The window's rows by one counting pass: RB_BINS bins of (bucket ordinal, next bits of the code),
// about a third of a row each, so a row's place is its bin's first position plus the number of
// rows of the bin with a smaller code or an equal code and an earlier position, mostly none or one
// to compare with (the order in which rows enter a bin does not matter).  A bin of more than
// RL_RUN rows leaves the window to k_rs_local.  Bound by LDS operations, about 9 per row (three
// or four stable digit passes took 40): 64M rows 955 -> 366 us.  The rows stay in registers from
// the load to the placing; LDS holds the bins, then the placed codes with their positions (below
// nextshift a code's bits and 12 bits of position fit 64), then the permutation.
constexpr uint32_t RB_BINS = 8192;  // 16-bit counters, two to a word: as large as sv
constexpr uint32_t RB_RESIDENT = 768;  // three blocks on each of 256 CUs
constexpr uint32_t RB_WIDE = 2 * RB_RESIDENT;
__global__ void __launch_bounds__(RS_BLOCK) __attribute__((amdgpu_waves_per_eu(6, 6))) k_rs_bins(RsLocal a) {
  __shared__ uint64_t sk[RS_TILE];
  __shared__ uint32_t sv[RS_TILE];
  __shared__ uint32_t wlast[RS_WAVES], wfirst[RS_WAVES], wnext[RS_WAVES], wstarts[RS_WAVES], winside[RS_WAVES];
  __shared__ uint32_t wsum[RS_WAVES];
  __shared__ uint32_t s_long, s_state;
  static_assert(RB_BINS == 2 * RS_TILE && RS_TILE == 4096, "bins alias sv; 12 bits of position");
  const unsigned t = threadIdx.x, lane = __lane_id(), wid = t / 64;
  const uint32_t q = a.nblk / RS_XCDS, rm = a.nblk % RS_XCDS, x = blockIdx.x % RS_XCDS;
  const uint32_t win = x * q + min(x, rm) + blockIdx.x / RS_XCDS;
  const uint64_t n = a.n, w0 = (uint64_t)win * a.w;
  // blocks after the first that fill the chip: nothing to do once a bucket has overflowed; once half
  // of the windows were crowded the rest only look for an overflow (64 rows of every code, 16M rows:
  // 1.17 ms by k_rs_local alone, 1.37 with every window tried, 1.28 now)
  uint32_t state = 0;
  if (blockIdx.x >= RB_RESIDENT) {
    if (t == 0) s_state = rl_peek(a.ctl);
    __syncthreads();
    state = s_state;
    if (state & RL_OVERFLOW) return;
  }
  uint64_t key[RS_ITEMS];
  uint32_t val[RS_ITEMS], hi16[RS_ITEMS];
  // positions w0 + i, i = wave * 512 + row * 64 + lane
#pragma unroll
  for (int j = 0; j < RS_ITEMS; ++j) {
    const uint32_t i = wid * RS_WAVE_ITEMS + j * 64 + lane;
    key[j] = w0 + i < n ? __builtin_nontemporal_load(a.keys + w0 + i) : ~0ull;
    val[j] = w0 + i < n && !(state & RL_CROWDED) ? __builtin_nontemporal_load(a.vals + w0 + i) : 0u;
  }
  const uint64_t before = w0 > 0 ? a.keys[w0 - 1] : 0;
  auto top = [&](uint64_t k) { return ((uint32_t)(k >> a.hish) & a.himask) << RS_BITS | ((uint32_t)(k >> a.topshift) & 0xFFu); };
#pragma unroll
  for (int j = 0; j < RS_ITEMS; ++j) {
    hi16[j] = top(key[j]);
    sv[j * RS_BLOCK + t] = 0;  // the bins
  }
  if (lane == 63) wlast[wid] = hi16[RS_ITEMS - 1];
  if (t == 0) s_long = 0;
  __syncthreads();
  // bucket starts, their number before each row
  uint64_t st[RS_ITEMS];
  uint32_t starts = 0, inside = 0, first = 0xFFFFFFFFu, next = 0xFFFFFFFFu;
#pragma unroll
  for (int j = 0; j < RS_ITEMS; ++j) {
    const uint32_t i0 = wid * RS_WAVE_ITEMS + j * 64;
    uint32_t p = __shfl_up(hi16[j], 1, 64);
    const uint32_t edge = j > 0 ? (uint32_t)__builtin_amdgcn_readlane((int)hi16[j > 0 ? j - 1 : 0], 63)
                                : (wid > 0 ? wlast[wid > 0 ? wid - 1 : 0] : top(before));
    if (lane == 0) p = edge;
    st[j] = __builtin_amdgcn_ballot_w64(w0 + i0 + lane < n && (p != hi16[j] || w0 + i0 + lane == 0));
    const uint32_t c = (uint32_t)__popcll(st[j]);
    starts += c;
    if (st[j]) {
      const uint32_t at = i0 + (uint32_t)__builtin_ctzll(st[j]);
      if (i0 < a.w) {
        inside += c;
        first = first < at ? first : at;
      } else {
        next = next < at ? next : at;
      }
    }
  }
  if (lane == 0) {
    wfirst[wid] = first;
    wnext[wid] = next;
    wstarts[wid] = starts;
    winside[wid] = inside;
  }
  __syncthreads();
  uint32_t lo = 0xFFFFFFFFu, hi = 0xFFFFFFFFu, nb = 0, seen = 0;
#pragma unroll
  for (unsigned w = 0; w < RS_WAVES; ++w) {
    lo = min(lo, wfirst[w]);
    hi = min(hi, wnext[w]);
    nb += winside[w];
    seen += w < wid ? wstarts[w] : 0;
  }
  if (lo == 0xFFFFFFFFu) return;  // no bucket starts here (uniform across the block)
  if (hi == 0xFFFFFFFFu) {
    if (w0 + RS_TILE < n) {  // the last bucket runs past the block's capacity
      if (t == 0) rl_set(a.ctl, RL_OVERFLOW);
      return;
    }
    hi = (uint32_t)(n - w0);
  }
  if (state & RL_CROWDED) {
    if (t == 0) a.redo[win] = 1;
    return;
  }
  const uint32_t m = hi - lo;
  // bins: the bucket's ordinal and as many code bits below as leave RB_BINS of them
  const uint32_t nextshift = a.sh[a.nlow - 1] + RS_BITS;
  uint32_t kb = 13 - (nb > 1 ? 32 - (uint32_t)__builtin_clz(nb - 1) : 0u);
  kb = kb < nextshift ? kb : nextshift;
  const uint32_t bsh = nextshift - kb, bmask = (1u << kb) - 1u;
  uint32_t bin[RS_ITEMS], rank[RS_ITEMS];
#pragma unroll
  for (int j = 0; j < RS_ITEMS; ++j) {
    const uint32_t i = wid * RS_WAVE_ITEMS + j * 64 + lane;
    const uint32_t ord = seen + below_count(st[j]) + (uint32_t)(st[j] >> lane & 1) - 1u;
    seen += (uint32_t)__popcll(st[j]);
    bin[j] = ord << kb | ((uint32_t)(key[j] >> bsh) & bmask);
    if (i >= lo && i < hi) {
      const uint32_t s16 = (bin[j] & 1) * 16;
      rank[j] = atomicAdd(&sv[bin[j] >> 1], 1u << s16) >> s16 & 0xFFFFu;
    }
  }
  __syncthreads();
  // first positions of the bins: thread t holds bins 16 t .. 16 t + 15
  {
    uint4 *hb = reinterpret_cast<uint4 *>(sv) + 2 * t;
    uint4 h0 = hb[0], h1 = hb[1];
    uint32_t c[8] = {h0.x, h0.y, h0.z, h0.w, h1.x, h1.y, h1.z, h1.w}, sum = 0;
    bool crowd = false;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t e = c[k] & 0xFFFFu, o = c[k] >> 16;
      crowd = crowd || e > RL_RUN || o > RL_RUN;
      c[k] = sum | (sum + e) << 16;
      sum += e + o;
    }
    const uint32_t incl = wave_incl_scan(sum);
    if (lane == 63) wsum[wid] = incl;
    if (crowd) s_long = 1;
    __syncthreads();
    if (s_long) {
      if (t == 0) {
        a.redo[win] = 1;
        rl_set(a.ctl, RL_REDO);
        if (2 * atomicAdd(a.ctl + 1, 1u) >= blockIdx.x && blockIdx.x >= RB_RESIDENT) rl_set(a.ctl, RL_CROWDED);
      }
      return;
    }
    uint32_t base = incl - sum;
#pragma unroll
    for (unsigned w = 0; w < RS_WAVES; ++w) base += w < wid ? wsum[w] : 0;
    const uint32_t b2 = base | base << 16;
    hb[0] = make_uint4(c[0] + b2, c[1] + b2, c[2] + b2, c[3] + b2);
    hb[1] = make_uint4(c[4] + b2, c[5] + b2, c[6] + b2, c[7] + b2);
  }
  __syncthreads();
  const uint64_t lowmask = (1ull << nextshift) - 1;
#pragma unroll
  for (int j = 0; j < RS_ITEMS; ++j) {
    const uint32_t i = wid * RS_WAVE_ITEMS + j * 64 + lane;
    key[j] = (key[j] & lowmask) << 12 | i;
    if (i >= lo && i < hi) {
      const uint32_t b = bin[j], e = b + 1;
      const uint32_t base = sv[b >> 1] >> ((b & 1) * 16) & 0xFFFFu;
      const uint32_t end = e < RB_BINS ? sv[e >> 1] >> ((e & 1) * 16) & 0xFFFFu : m;
      sk[base + rank[j]] = key[j];
      bin[j] = base;
      rank[j] = end - base;  // rows of the bin
    } else {
      rank[j] = 0;
    }
  }
  __syncthreads();
  uint32_t heads = 0;
#pragma unroll
  for (int j = 0; j < RS_ITEMS; ++j) {
    if (rank[j] == 0) continue;
    uint32_t pos = bin[j];
    bool head = true;
    if (rank[j] > 1) {
      for (uint32_t k = bin[j]; k < bin[j] + rank[j]; ++k) {
        const uint64_t c = sk[k];
        pos += c < key[j];
        head = head && !(c < key[j] && c >> 12 == key[j] >> 12);
      }
    }
    sv[pos] = val[j];
    heads |= (head ? 1u : 0u) << j;
    bin[j] = pos;
  }
  __syncthreads();
  for (uint32_t k = t; k < m; k += RS_BLOCK) a.vout[w0 + lo + k] = sv[k];
  if (a.heads) {
    uint8_t *hb = reinterpret_cast<uint8_t *>(sk);  // the placed codes have been read
#pragma unroll
    for (int j = 0; j < RS_ITEMS; ++j)
      if (rank[j]) hb[bin[j]] = (uint8_t)(heads >> j & 1);
    __syncthreads();
    for (uint32_t k = t; k < m; k += RS_BLOCK) a.heads[w0 + lo + k] = hb[k];
  }
}

// 6 waves per SIMD: three blocks per CU, as many as the LDS holds
__global__ void __launch_bounds__(RS_BLOCK) __attribute__((amdgpu_waves_per_eu(6, 6))) k_rs_local(RsLocal a) {
  __shared__ uint64_t sk[RS_TILE];
  __shared__ uint32_t sv[RS_TILE];
  __shared__ uint16_t wc[RS_WAVES][RS_BINS];
  __shared__ uint32_t wsum[RS_WAVES];
  __shared__ uint32_t s_lo, s_hi, s_long;
  const unsigned t = threadIdx.x, lane = __lane_id(), wid = t / 64;
  // each XCD takes a contiguous range of windows: neighbours share RL_W codes and one L2
  const uint32_t q = a.nblk / RS_XCDS, rm = a.nblk % RS_XCDS, x = blockIdx.x % RS_XCDS;
  const uint32_t win = x * q + min(x, rm) + blockIdx.x / RS_XCDS;
  if (!a.redo[win]) return;
  const uint64_t n = a.n, w0 = (uint64_t)win * a.w;
  uint64_t key[RS_ITEMS];
  uint32_t val[RS_ITEMS], rank[RS_ITEMS];
  if (t == 0) {
    s_lo = 0xFFFFFFFFu;
    s_hi = 0xFFFFFFFFu;
    s_long = 0;
  }
  // the codes and values of positions w0 + i, i = wave * 512 + row * 64 + lane (memory
  // order); the values past the block's rows are mostly its neighbour's, in the same L2
#pragma unroll
  for (int j = 0; j < RS_ITEMS; ++j) {
    const uint32_t i = wid * RS_WAVE_ITEMS + j * 64 + lane;
    key[j] = w0 + i < n ? __builtin_nontemporal_load(a.keys + w0 + i) : ~0ull;
    val[j] = w0 + i < n ? __builtin_nontemporal_load(a.vals + w0 + i) : 0u;
    sk[i] = key[j] >> a.topshift;
  }
  const uint64_t tprev = w0 > 0 ? a.keys[w0 - 1] >> a.topshift : ~0ull;
  __syncthreads();
  // bucket starts: the first in the window (lo) and the first at or past its end (hi)
  bool st[RS_ITEMS];
#pragma unroll
  for (int j = 0; j < RS_ITEMS; ++j) {
    const uint32_t i = wid * RS_WAVE_ITEMS + j * 64 + lane;
    st[j] = w0 + i < n && (w0 + i == 0 || (i == 0 ? tprev : sk[i - 1]) != sk[i]);
    if (st[j]) atomicMin(i < a.w ? &s_lo : &s_hi, i);
  }
  __syncthreads();
  const uint32_t lo = s_lo;
  if (lo == 0xFFFFFFFFu) return;  // no bucket starts here (uniform across the block)
  uint32_t hi = s_hi;
  if (hi == 0xFFFFFFFFu) {
    if (w0 + RS_TILE < n) {  // the last bucket runs past the block's capacity
      if (t == 0) rl_set(a.ctl, RL_OVERFLOW);
      return;
    }
    hi = (uint32_t)(n - w0);
  }
  const uint32_t m = hi - lo;
  // bucket ordinals (starts in (lo, i]) by a scan in memory order
  uint32_t carry = 0;
  uint32_t ord[RS_ITEMS];
#pragma unroll
  for (int j = 0; j < RS_ITEMS; ++j) {
    const uint32_t i = wid * RS_WAVE_ITEMS + j * 64 + lane;
    const uint32_t inc = wave_incl_scan((st[j] && i > lo && i < hi) ? 1u : 0u);
    ord[j] = carry + inc;
    carry += __shfl(inc, 63, 64);
  }
  if (lane == 0) wsum[wid] = carry;
  __syncthreads();  // also: every read of the high parts in sk is done
  uint32_t obase = 0, nb = 1;  // nb: buckets in [lo, hi)
  for (unsigned w = 0; w < RS_WAVES; ++w) {
    if (w < wid) obase += wsum[w];
    nb += wsum[w];
  }
  const uint64_t lowmask = (1ull << a.topshift) - 1;
#pragma unroll
  for (int j = 0; j < RS_ITEMS; ++j) {
    const uint32_t i = wid * RS_WAVE_ITEMS + j * 64 + lane;
    if (i >= lo && i < hi) {
      sk[i - lo] = ((uint64_t)(obase + ord[j]) << a.topshift) | (key[j] & lowmask);
      sv[i - lo] = val[j];
    }
  }
  // from here on a wave holds rows wid * S + j * 64 + lane, j < J: every wave has work
  const uint32_t J = (m + RS_BLOCK - 1) / RS_BLOCK, S = 64 * J;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < RS_ITEMS; ++j) {
    const uint32_t i = wid * S + j * 64 + lane;
    if (j < (int)J) {
      key[j] = i < m ? sk[i] : 0;
      val[j] = i < m ? sv[i] : 0;
    }
  }
  // Stable LDS passes, each on the digit (key >> sh) & mask with ranks in position order:
  // first the two digits above the cut and the ordinal (1 or 2 passes: nb <= RS_TILE), then,
  // only after a long run, every remaining digit and the ordinal again.
  const uint32_t nl = a.nlow, cut = a.sh[nl - 2];
  const uint32_t nord = (nb > 1 ? 1u : 0u) + (nb > RS_BINS ? 1u : 0u), npre = 2 + nord;
  uint32_t npass = npre;
  for (uint32_t ps = 0; ps < npass; ++ps) {
    uint32_t sh, mask;
    if (ps < npre) {
      sh = ps < 2 ? a.sh[nl - 2 + ps] : a.topshift + RS_BITS * (ps - 2);
      mask = ps < 2 ? a.mask[nl - 2 + ps] : 0xFFu;
    } else {
      const uint32_t r = ps - npre;
      sh = r < nl ? a.sh[r] : a.topshift + RS_BITS * (r - nl);
      mask = r < nl ? a.mask[r] : 0xFFu;
    }
    uint64_t *pm = sk;  // lane masks of [wave][digit]
    __syncthreads();    // every read of sk and sv before this pass is done
    for (int w = t; w < RS_WAVES * RS_BINS; w += RS_BLOCK) {
      (&wc[0][0])[w] = 0;
      pm[w] = 0;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < RS_ITEMS; ++j) {
      if (j >= (int)J) break;
      const uint32_t i = wid * S + j * 64 + lane;
      const bool valid = i < m;
      const uint32_t d = (uint32_t)(key[j] >> sh) & mask;
      uint64_t *slot = pm + wid * RS_BINS + d;
      if (valid) __hip_atomic_fetch_or(slot, 1ull << lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      const uint64_t peers = valid ? __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) : 0;
      const uint32_t before = valid ? wc[wid][d] : 0;
      const uint32_t below = below_count(peers);  // peers in lower lanes
      rank[j] = before + below;
      if (valid && below == 0) {
        wc[wid][d] = (uint16_t)(before + (uint32_t)__popcll(peers));
        __hip_atomic_store(slot, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
    __syncthreads();
    uint32_t cnt = 0, incl = 0;
    if (t < RS_BINS) {
#pragma unroll
      for (int w = 0; w < RS_WAVES; ++w) {
        const uint32_t c = wc[w][t];
        wc[w][t] = (uint16_t)cnt;
        cnt += c;
      }
      incl = wave_incl_scan(cnt);
      if (lane == 63) wsum[wid] = incl;
    }
    __syncthreads();
    if (t < RS_BINS) {
      uint32_t tstart = incl - cnt;
#pragma unroll
      for (int w = 0; w < RS_WAVES; ++w) tstart += w < (int)wid ? wsum[w] : 0u;
#pragma unroll
      for (int w = 0; w < RS_WAVES; ++w) wc[w][t] = (uint16_t)(wc[w][t] + tstart);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < RS_ITEMS; ++j) {
      if (j >= (int)J) break;
      const uint32_t i = wid * S + j * 64 + lane;
      if (i < m) {
        const uint32_t pos = wc[wid][(uint32_t)(key[j] >> sh) & mask] + rank[j];
        sk[pos] = key[j];
        sv[pos] = val[j];
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < RS_ITEMS; ++j) {
      if (j >= (int)J) break;
      const uint32_t i = wid * S + j * 64 + lane;
      key[j] = i < m ? sk[i] : 0;
      val[j] = i < m ? sv[i] : 0;
    }
    if (ps + 1 != npre || nl == 2) continue;
    // rows that tie on key >> cut stand in runs; a run longer than RL_RUN holds two rows
    // RL_RUN apart
    bool lng = false;
#pragma unroll
    for (int j = 0; j < RS_ITEMS; ++j) {
      if (j >= (int)J) break;
      const uint32_t i = wid * S + j * 64 + lane;
      lng |= i + RL_RUN < m && (sk[i + RL_RUN] >> cut) == (key[j] >> cut);
    }
    if (lng) s_long = 1;
    __syncthreads();
    if (s_long) npass += nl + nord;
  }
  if (nl == 2 || s_long) {  // the rows are in order
#pragma unroll
    for (int j = 0; j < RS_ITEMS; ++j) {
      if (j >= (int)J) break;
      const uint32_t i = wid * S + j * 64 + lane;
      if (i < m) {
        a.vout[w0 + lo + i] = val[j];
        if (a.heads) a.heads[w0 + lo + i] = i == 0 || sk[i - 1] != key[j];
      }
    }
    return;
  }
  // each row's place in its run: the rows of the run with a smaller code, or an equal code
  // and an earlier position.  Runs of 2 from the neighbours' codes; longer runs (rare for
  // spread keys) by a scan of the run.
  uint32_t slow = 0;
#pragma unroll
  for (int j = 0; j < RS_ITEMS; ++j) {
    if (j >= (int)J) break;
    const uint32_t i = wid * S + j * 64 + lane;
    if (i >= m) continue;
    const uint64_t p = key[j] >> cut;
    const uint64_t km1 = i >= 1 ? sk[i - 1] : 0, kp1 = i + 1 < m ? sk[i + 1] : 0;
    const uint64_t km2 = i >= 2 ? sk[i - 2] : 0, kp2 = i + 2 < m ? sk[i + 2] : 0;
    const bool em1 = i >= 1 && (km1 >> cut) == p, ep1 = i + 1 < m && (kp1 >> cut) == p;
    const bool em2 = em1 && i >= 2 && (km2 >> cut) == p, ep2 = ep1 && i + 2 < m && (kp2 >> cut) == p;
    uint32_t pos = i;
    if ((em1 && ep1) || em2 || ep2) {
      slow |= 1u << j;
      continue;
    }
    if (em1) pos = km1 <= key[j] ? i : i - 1;  // run [i-1, i]
    if (ep1) pos = kp1 < key[j] ? i + 1 : i;   // run [i, i+1]
    a.vout[w0 + lo + pos] = val[j];
    if (a.heads) a.heads[w0 + lo + pos] = !(em1 && km1 == key[j]);
  }
#pragma unroll 1
  for (uint32_t j = 0; j < J; ++j) {
    if (!((slow >> j) & 1)) continue;
    const uint32_t i = wid * S + j * 64 + lane;
    const uint64_t kk = sk[i], p = kk >> cut;
    uint32_t rs = i, re = i + 1;
    while (rs > 0 && (sk[rs - 1] >> cut) == p) --rs;
    while (re < m && (sk[re] >> cut) == p) ++re;
    uint32_t pos = rs;
    bool head = true;
    for (uint32_t k = rs; k < re; ++k) {
      const uint64_t c = sk[k];
      pos += c < kk || (c == kk && k < i);
      head = head && !(c == kk && k < i);
    }
    a.vout[w0 + lo + pos] = sv[i];
    if (a.heads) a.heads[w0 + lo + pos] = head;
  }
}

__global__ void k_rs_vals(const uint32_t *__restrict__ vals, uint64_t n, uint32_t *__restrict__ vout) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256)
    vout[i] = vals ? vals[i] : (uint32_t)i;
}

__global__ void k_copy_pairs(const uint64_t *ks, const uint32_t *vs, uint64_t n, uint64_t *kd,
                             uint32_t *vd) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * 256) {
    kd[i] = ks[i];
    vd[i] = vs[i];
  }
}

template <int KI, int KO>
static void rs_scatter_launch(aln_ctx *c, uint32_t ntiles, const RsPass &a) {
  hipLaunchKernelGGL((k_rs_scatter<KI, KO>), dim3(ntiles), dim3(RS_BLOCK), 0, c->stream, a);
}

static int rs_scatter(aln_ctx *c, int ki, int ko, uint32_t ntiles, const RsPass &a) {
  switch (ki * 16 + ko) {
#define RS_CASE(x, y)                      \
  case x * 16 + y:                         \
    rs_scatter_launch<x, y>(c, ntiles, a); \
    break;
    RS_CASE(0, 0) RS_CASE(0, 4) RS_CASE(0, 8)
    RS_CASE(8, 0) RS_CASE(8, 4) RS_CASE(8, 8)
    RS_CASE(4, 0) RS_CASE(4, 4)
#undef RS_CASE
    default:
      ALN_REQUIRE(false, "radix sort: key widths %d -> %d", ki, ko);
  }
  return check_launch("radix_scatter");
}

template <int KI, bool VARY>
static void rs_count_launch(aln_ctx *c, uint32_t nsuper, const RsIn &in, uint64_t n, uint32_t sh,
                            uint32_t mask, uint32_t *cnt, uint16_t *sub, unsigned long long *vary) {
  hipLaunchKernelGGL((k_rs_count<KI, VARY>), dim3(nsuper), dim3(RS_BLOCK), 0, c->stream, in, n, sh, mask,
                     nsuper, cnt, sub, vary);
}

static int rs_count(aln_ctx *c, int ki, bool vary, uint32_t nsuper, const RsIn &in, uint64_t n,
                    uint32_t sh, uint32_t mask, uint32_t *cnt, uint16_t *sub, unsigned long long *d_vary) {
  switch (ki * 2 + (vary ? 1 : 0)) {
    case 0: rs_count_launch<0, false>(c, nsuper, in, n, sh, mask, cnt, sub, d_vary); break;
    case 1: rs_count_launch<0, true>(c, nsuper, in, n, sh, mask, cnt, sub, d_vary); break;
    case 8: rs_count_launch<4, false>(c, nsuper, in, n, sh, mask, cnt, sub, d_vary); break;
    case 16: rs_count_launch<8, false>(c, nsuper, in, n, sh, mask, cnt, sub, d_vary); break;
    case 17: rs_count_launch<8, true>(c, nsuper, in, n, sh, mask, cnt, sub, d_vary); break;
    default:
      ALN_REQUIRE(false, "radix sort: key width %d", ki);
  }
  return check_launch("radix_count");
}

// The bucket path of rs_sort (see k_rs_local): *done = false when a bucket overflowed.
// kt and vt: two code arrays of 8n bytes and two row arrays of n words.
static int rs_hybrid(aln_ctx *c, const RsIn &in, bool from_keys, uint64_t n, uint32_t bits, const uint32_t *run,
                     uint32_t nrun, uint64_t vary, int counted, uint32_t *cnt, uint32_t *excl, uint32_t *tot,
                     uint16_t *sub, uint64_t *const kt[2], uint32_t *const vt[2], uint32_t *vout, uint8_t *heads,
                     bool *done) {
  *done = false;
  const uint32_t nsuper = (uint32_t)((n + RS_SUPER - 1) / RS_SUPER);
  const uint32_t ntiles = (uint32_t)((n + RS_TILE - 1) / RS_TILE);
  auto pass_mask = [&](uint32_t p) {
    uint32_t pb = bits - RS_BITS * p < RS_BITS ? bits - RS_BITS * p : RS_BITS;
    return (1u << pb) - 1;
  };
  uint32_t *ctl;
  ALN_TRY(ws(c, 2, &ctl));
  // the wide window: room for a bucket of 1.25 x the mean (over the codes that the top two
  // digits' varying bits make) and 256 rows more
  const int top_bits = __builtin_popcountll(vary >> (RS_BITS * run[nrun - 1]) & pass_mask(run[nrun - 1])) +
                       __builtin_popcountll(vary >> (RS_BITS * run[nrun - 2]) & pass_mask(run[nrun - 2]));
  const uint64_t tail = (n >> top_bits) + (n >> top_bits) / 4 + 256;
  // (a sort whose windows are all resident at once gains little by fewer of them, and loses a second
  // try where a bucket does not fit)
  const uint32_t wide = tail < RS_TILE - RL_W && n > (uint64_t)RL_W * RB_WIDE ? (uint32_t)(RS_TILE - tail) & ~63u : RL_W;
  // two passes: the second most significant varying digit, then the most significant
  for (uint32_t r = 0; r < 2; ++r) {
    const uint32_t p = run[nrun - 2 + r];
    RsPass a;
    a.in = in;
    if (r > 0) {
      a.in.keys = kt[0];
      a.in.vals = vt[0];
    }
    a.n = n;
    a.tot = tot;
    a.excl = excl;
    a.sub = sub;
    a.kout = kt[r];
    a.vout = vt[r];
    a.sh = RS_BITS * p;
    a.mask = pass_mask(p);
    a.oshift = 0;
    a.nsuper = nsuper;
    const int ki = r == 0 ? (from_keys ? 0 : 8) : 8;
    if (r > 0 || (int)p != counted) {
      ProfScope ps(c, "radix_count");
      ALN_TRY(rs_count(c, ki, false, nsuper, a.in, n, a.sh, a.mask, cnt, sub, nullptr));
    }
    {
      ProfScope ps(c, "radix_scan");
      hipLaunchKernelGGL(k_rs_rowscan, dim3(RS_BINS), dim3(RS_SCAN_BLOCK), 0, c->stream, cnt, nsuper, excl, tot);
    }
    ALN_TRY(check_launch("radix_scan"));
    {
      ProfScope ps(c, "radix_scatter");
      ALN_TRY(rs_scatter(c, ki, 8, ntiles, a));
    }
  }
  // the permutation goes to vout unless vout is also the input's row list, which the digit
  // passes would read again after an overflow: then to vt[0] (read by the second pass, now
  // free) and copied over on success
  const bool alias = in.vals && in.vals == vout;
  RsLocal l;
  memset(&l, 0, sizeof(l));
  l.keys = kt[1];
  l.vals = vt[1];
  l.vout = alias ? vt[0] : vout;
  l.heads = heads;
  l.ctl = ctl;
  l.n = n;
  l.topshift = RS_BITS * run[nrun - 2];
  l.hish = RS_BITS * run[nrun - 1];
  l.himask = pass_mask(run[nrun - 1]);
  l.nlow = nrun - 2;
  for (uint32_t r = 0; r + 2 < nrun; ++r) {
    l.sh[r] = RS_BITS * run[r];
    l.mask[r] = pass_mask(run[r]);
  }
  uint32_t o = RL_OVERFLOW;
  ALN_TRY(ws(c, (size_t)((n + RL_W - 1) / RL_W) + 4, &l.redo));
  // Windows as wide as leave room for the last bucket (each block reads RS_TILE positions for its
  // window): buckets of spread codes hold the mean and a few deviations more.  If one does
  // not fit, windows of half a tile.
  for (uint32_t w = wide; o & RL_OVERFLOW; w = RL_W) {
    l.w = w;
    l.nblk = (uint32_t)((n + w - 1) / w);
    ALN_TRY(fill_u32(c, ctl, 2, 0));
    ALN_TRY(fill_u32(c, reinterpret_cast<uint32_t *>(l.redo), (l.nblk + 3) / 4, 0));
    {
      ProfScope ps(c, "radix_local");
      hipLaunchKernelGGL(k_rs_bins, dim3(l.nblk), dim3(RS_BLOCK), 0, c->stream, l);
    }
    ALN_TRY(check_launch("radix_bins"));
    ALN_TRY(copy_to_host(c, &o, ctl, 4));
    o &= RL_OVERFLOW | RL_REDO;
    if (w == RL_W) break;
  }
  if (o == RL_REDO) {
    {
      ProfScope ps(c, "radix_local");
      hipLaunchKernelGGL(k_rs_local, dim3(l.nblk), dim3(RS_BLOCK), 0, c->stream, l);
    }
    ALN_TRY(check_launch("radix_local"));
    ALN_TRY(copy_to_host(c, &o, ctl, 4));
    o &= RL_OVERFLOW;
  }
  *done = o == 0;
  if (*done && alias) ALN_HIP(hipMemcpyAsync(vout, vt[0], 4ull * n, hipMemcpyDeviceToDevice, c->stream));
  return ALN_OK;
}

// Rows of a sample of a key column, read back by the host.
constexpr uint64_t RS_SAMPLE = 4096;

// Stable LSD sort of the items of `in` by the low `bits` bits of their codes.  from_keys:
// the codes come from in.ks (first pass), else from the 8-byte array in.keys.  The values
// land in vout (may be in.vals).  kout given: the codes land there, whole (may be in.keys);
// otherwise each pass stores only the key bytes the later passes read.
// heads given: *have_heads tells whether the bucket path filled it (see sort_codes).  guess: bits
// in which the codes are expected to differ (what is counted first depends on it, not the result).
static int rs_sort(aln_ctx *c, RsIn in, bool from_keys, uint64_t n, uint32_t bits, uint64_t *kout,
                   uint32_t *vout, uint8_t *heads = nullptr, bool *have_heads = nullptr, uint64_t guess = ~0ull) {
  if (have_heads) *have_heads = false;
  if (n == 0) return ALN_OK;
  ALN_REQUIRE(bits <= 64, "radix sort: %u key bits", bits);
  ALN_REQUIRE(n < (1ull << 32), "radix sort: more than 2^32 items");
  const bool keys_out = kout != nullptr;
  const uint32_t passes = (bits + RS_BITS - 1) / RS_BITS;
  const uint32_t nsuper = (uint32_t)((n + RS_SUPER - 1) / RS_SUPER);
  const uint32_t ntiles = (uint32_t)((n + RS_TILE - 1) / RS_TILE);
  const uint64_t ncnt = (uint64_t)RS_BINS * nsuper;
  const int ki0 = from_keys ? 0 : 8;
  auto pass_mask = [&](uint32_t p) {
    uint32_t pb = bits - RS_BITS * p < RS_BITS ? bits - RS_BITS * p : RS_BITS;
    return (1u << pb) - 1;
  };
  uint32_t *cnt = nullptr, *excl = nullptr, *tot = nullptr;
  uint16_t *sub = nullptr;
  unsigned long long *d_vary = nullptr;
  if (passes > 0) {
    ALN_TRY(ws(c, ncnt, &cnt));
    ALN_TRY(ws(c, ncnt, &excl));
    ALN_TRY(ws(c, (size_t)RS_BINS, &tot));
    ALN_TRY(ws(c, (size_t)nsuper * RS_SUB * RS_BINS, &sub));
    ALN_TRY(ws(c, 1, &d_vary));
  }
  // the bits in which the codes differ, and the counts of one digit of the input: the first
  // the bucket path sorts by when it may run (the second most significant), else digit 0
  const bool sync = n >= RS_SYNC_MIN;
  const bool bucket = !keys_out && sync && passes >= 4;
  int counted = -1;  // the digit whose counts of the input are in cnt and sub
  if (passes > 0) {
    counted = 0;
    if (bucket) {  // the second most significant digit expected to vary
      int top = -1;
      for (int p = (int)passes - 1; p >= 0; --p)
        if ((guess >> (RS_BITS * p)) & pass_mask(p)) {
          if (top >= 0) {
            counted = p;
            break;
          }
          top = p;
        }
    }
    if (sync) ALN_TRY(fill_u64(c, reinterpret_cast<uint64_t *>(d_vary), 1, 0));
    ProfScope ps(c, "radix_count");
    ALN_TRY(rs_count(c, ki0, sync, nsuper, in, n, RS_BITS * counted, pass_mask(counted), cnt, sub, d_vary));
  }
  uint64_t vary = ~0ull;
  if (sync && passes > 0) ALN_TRY(copy_to_host(c, &vary, d_vary, 8));
  uint32_t run[RS_MAX_PASSES], nrun = 0;
  for (uint32_t p = 0; p < passes; ++p)
    if ((vary >> (RS_BITS * p)) & pass_mask(p)) run[nrun++] = p;
  if (nrun == 0) {  // every code equal: the input order is sorted
    if (from_keys || in.vals != vout) {
      hipLaunchKernelGGL(k_rs_vals, dim3(grid_for(n, 256, 65536)), dim3(256), 0, c->stream, in.vals, n, vout);
      ALN_TRY(check_launch("radix_vals"));
    }
    ALN_REQUIRE(!keys_out || !from_keys, "radix sort: codes of the key columns are not kept");
    if (keys_out && kout != in.keys)
      ALN_HIP(hipMemcpyAsync(kout, in.keys, 8ull * n, hipMemcpyDeviceToDevice, c->stream));
    return ALN_OK;
  }
  const bool alias1 = nrun == 1 && ((in.vals && in.vals == vout) || (keys_out && in.keys == kout));
  void *kt[2] = {nullptr, nullptr};
  uint32_t *vt[2] = {nullptr, nullptr};
  if (nrun > 1 || alias1) {
    ALN_TRY(ws(c, 8 * n, reinterpret_cast<uint8_t **>(&kt[0])));
    ALN_TRY(ws(c, 8 * n, reinterpret_cast<uint8_t **>(&kt[1])));
    ALN_TRY(ws(c, n, &vt[0]));
    ALN_TRY(ws(c, n, &vt[1]));
  }
  // A permutation sort of many rows with at least 4 varying digits: two passes on the two
  // most significant ones, then every bucket sorted on the rest in LDS (k_rs_local); if a
  // bucket is too large for that, the digit passes below run instead, from the start, and
  // count pass 0 again (the bucket path's passes used the count buffers).
  if (bucket && nrun >= 4) {
    bool done = false;
    uint64_t *const kt64[2] = {static_cast<uint64_t *>(kt[0]), static_cast<uint64_t *>(kt[1])};
    ALN_TRY(rs_hybrid(c, in, from_keys, n, bits, run, nrun, vary, counted, cnt, excl, tot, sub, kt64, vt, vout, heads, &done));
    if (have_heads) *have_heads = done && heads;
    if (done) return ALN_OK;
    counted = -1;
  }
  // Bytes each pass reads (ki) and writes (ko) per key: the bytes below the next pass's
  // digit are dropped and the rest is stored in the smallest word that holds it.
  int ki[RS_MAX_PASSES], ko[RS_MAX_PASSES];
  uint32_t qin[RS_MAX_PASSES], qout[RS_MAX_PASSES];
  for (uint32_t r = 0; r < nrun; ++r) {
    qin[r] = r == 0 ? 0 : qout[r - 1];
    ki[r] = r == 0 ? ki0 : ko[r - 1];
    if (keys_out) {
      qout[r] = 0;
      ko[r] = 8;
    } else if (r + 1 < nrun) {
      qout[r] = run[r + 1];
      ko[r] = key_word(bits - RS_BITS * qout[r]);
    } else {
      qout[r] = qin[r];
      ko[r] = 0;
    }
  }
  const void *kprev = nullptr;
  const uint32_t *vprev = nullptr;
  for (uint32_t r = 0; r < nrun; ++r) {
    const uint32_t p = run[r];
    const bool direct = r + 1 == nrun && !alias1;
    RsPass a;
    a.in = in;
    if (r > 0) {
      a.in.keys = kprev;
      a.in.vals = vprev;
    }
    a.n = n;
    a.tot = tot;
    a.excl = excl;
    a.sub = sub;
    a.kout = ko[r] == 0 ? nullptr : direct ? static_cast<void *>(kout) : kt[(nrun - 1 - r) & 1];
    a.vout = direct ? vout : vt[(nrun - 1 - r) & 1];
    a.sh = RS_BITS * (p - qin[r]);
    a.mask = pass_mask(p);
    a.oshift = RS_BITS * (qout[r] - qin[r]);
    a.nsuper = nsuper;
    if (r > 0 || (int)p != counted) {
      ProfScope ps(c, "radix_count");
      ALN_TRY(rs_count(c, ki[r], false, nsuper, a.in, n, a.sh, a.mask, cnt, sub, nullptr));
    }
    {
      ProfScope ps(c, "radix_scan");
      hipLaunchKernelGGL(k_rs_rowscan, dim3(RS_BINS), dim3(RS_SCAN_BLOCK), 0, c->stream, cnt, nsuper, excl, tot);
    }
    ALN_TRY(check_launch("radix_scan"));
    {
      ProfScope ps(c, "radix_scatter");
      ALN_TRY(rs_scatter(c, ki[r], ko[r], ntiles, a));
    }
    kprev = a.kout;
    vprev = a.vout;
  }
  if (alias1) {
    if (keys_out) {
      hipLaunchKernelGGL(k_copy_pairs, dim3(grid_for(n, 256, 65536)), dim3(256), 0, c->stream,
                         static_cast<const uint64_t *>(kprev), vprev, n, kout, vout);
      ALN_TRY(check_launch("radix_copy"));
    } else {
      ALN_HIP(hipMemcpyAsync(vout, vprev, 4ull * n, hipMemcpyDeviceToDevice, c->stream));
    }
  }
  return ALN_OK;
}

int sort_codes(aln_ctx *c, const uint64_t *d_codes, uint64_t n, uint32_t bits, uint32_t *d_perm, uint8_t *d_heads,
               bool *have_heads) {
  RsIn in;
  memset(&in, 0, sizeof(in));
  in.keys = d_codes;
  return rs_sort(c, in, false, n, bits, nullptr, d_perm, d_heads, have_heads);
}

int radix_sort_pairs(aln_ctx *c, uint64_t *d_keys, uint32_t *d_vals, uint64_t n, uint32_t bits) {
  if (n <= 1 || bits == 0) return ALN_OK;
  RsIn in;
  memset(&in, 0, sizeof(in));
  in.keys = d_keys;
  in.vals = d_vals;
  return rs_sort(c, in, false, n, bits, d_keys, d_vals);
}

// Range of every key column.
struct KeyRanges {
  int64_t mn[ALN_MAX_KEYS], mx[ALN_MAX_KEYS];
  uint32_t bits[ALN_MAX_KEYS], total;
};

static int key_ranges(aln_ctx *c, const int64_t *const *keys, int nkeys, uint64_t n, KeyRanges *r) {
  r->total = 0;
  ALN_TRY(minmax_keys(c, keys, nkeys, n, r->mn, r->mx));
  for (int k = 0; k < nkeys; ++k) {
    r->bits[k] = bits_for_range_u((uint64_t)r->mx[k] - (uint64_t)r->mn[k]);
    r->total += r->bits[k];
  }
  return ALN_OK;
}

// The code layout of keys [k0, k1) (k0 most significant).  Returns the total bits.
static uint32_t key_set(const KeyRanges &r, const int64_t *const *keys, const int32_t *desc, int k0,
                        int k1, KeySet *ks) {
  memset(ks, 0, sizeof(*ks));
  uint32_t total = 0;
  for (int k = k0; k < k1; ++k) {
    ks->ref[k - k0] = (desc && desc[k]) ? r.mx[k] : r.mn[k];
    ks->desc[k - k0] = desc ? desc[k] : 0;
    ks->k[k - k0] = keys[k];
    total += r.bits[k];
  }
  ks->n = k1 - k0;
  uint32_t sh = total;
  for (int k = 0; k < ks->n; ++k) {
    sh -= r.bits[k0 + k];
    ks->shift[k] = sh;
  }
  return total;
}

static int sort_with_ranges(aln_ctx *c, const KeyRanges &r, const int64_t *const *keys,
                            const int32_t *desc, int nkeys, uint64_t n, uint32_t *d_perm, uint64_t guess = ~0ull) {
  RsIn in;
  memset(&in, 0, sizeof(in));
  if (r.total <= 64) {  // one sort of the concatenated codes, computed by its first pass
    key_set(r, keys, desc, 0, nkeys, &in.ks);
    return rs_sort(c, in, true, n, r.total, nullptr, d_perm, nullptr, nullptr, guess);
  }
  // LSD over keys, last key first, each sort stable (sorts.cu:17-70); each reads its key at
  // the rows of the permutation so far
  for (int k = nkeys - 1; k >= 0; --k) {
    uint32_t b = key_set(r, keys, desc, k, k + 1, &in.ks);
    in.vals = k == nkeys - 1 ? nullptr : d_perm;
    ALN_TRY(rs_sort(c, in, true, n, b, nullptr, d_perm));
  }
  return ALN_OK;
}

int sort_keys_ranged(aln_ctx *c, const int64_t *const *keys, int nkeys, uint64_t n, const int64_t *mn,
                     const int64_t *mx, uint32_t *d_perm) {
  KeyRanges r;
  r.total = 0;
  for (int k = 0; k < nkeys; ++k) {
    r.mn[k] = mn[k];
    r.mx[k] = mx[k];
    r.bits[k] = bits_for_range_u((uint64_t)mx[k] - (uint64_t)mn[k]);
    r.total += r.bits[k];
  }
  return sort_with_ranges(c, r, keys, nullptr, nkeys, n, d_perm);
}

static int sort_keys_impl(aln_ctx *c, const int64_t *const *keys, const int32_t *desc, int nkeys,
                          uint64_t n, uint32_t *d_perm) {
  ALN_REQUIRE(nkeys >= 1 && nkeys <= ALN_MAX_KEYS, "sort: %d keys", nkeys);
  ALN_REQUIRE(n < (1ull << 32), "sort: more than 2^32 rows");
  if (n == 0) return ALN_OK;
  KeyRanges r;
  bool whole = false;
  uint64_t guess = ~0ull;
  if (nkeys == 1 && n >= RS_SYNC_MIN) {
    // One key: codes over the whole int64 range, no min/max pass; the count pass finds the
    // digits every key shares and those passes are skipped.  Unless values of a narrow range
    // differ in many high bits (they cross zero or another power of two): checked on the
    // first rows, where such keys get the min/max pass and codes of just their range.
    std::vector<int64_t> v(std::min<uint64_t>(n, RS_SAMPLE));
    ALN_TRY(copy_to_host(c, v.data(), keys[0], 8 * v.size()));
    uint64_t vary = 0;
    int64_t lo = v[0], hi = v[0];
    for (int64_t x : v) {
      vary |= (uint64_t)x ^ (uint64_t)v[0];
      lo = std::min(lo, x);
      hi = std::max(hi, x);
    }
    whole = bits_for_range_u(vary) <= bits_for_range_u((uint64_t)hi - (uint64_t)lo) + RS_BITS;
    if (whole && vary) guess = vary;
  }
  if (whole) {
    r.mn[0] = INT64_MIN;
    r.mx[0] = INT64_MAX;
    r.bits[0] = r.total = 64;
  } else {
    ALN_TRY(key_ranges(c, keys, nkeys, n, &r));
  }
  return sort_with_ranges(c, r, keys, desc, nkeys, n, d_perm, guess);
}

// ---- top-k: tile-wise bitonic sort of (code, index), keep the first k of each tile -----
constexpr int TK_BLOCK = 256;
constexpr int TK_TILE = 1024;

__device__ __forceinline__ bool tk_less(uint64_t ca, uint32_t ia, uint64_t cb, uint32_t ib) {
  return ca < cb || (ca == cb && ia < ib);
}

__global__ void __launch_bounds__(TK_BLOCK) k_tile_topk(const uint64_t *__restrict__ code,
                                                        const uint32_t *__restrict__ idx,
                                                        uint64_t n, uint32_t k,
                                                        uint64_t *__restrict__ ocode,
                                                        uint32_t *__restrict__ oidx) {
  __shared__ uint64_t sc[TK_TILE];
  __shared__ uint32_t si[TK_TILE];
  uint64_t base = (uint64_t)blockIdx.x * TK_TILE;
  for (int t = threadIdx.x; t < TK_TILE; t += TK_BLOCK) {
    uint64_t i = base + t;
    sc[t] = i < n ? code[i] : ~0ull;
    si[t] = i < n ? idx[i] : 0xFFFFFFFFu;
  }
  __syncthreads();
  for (int size = 2; size <= TK_TILE; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int t = threadIdx.x; t < TK_TILE / 2; t += TK_BLOCK) {
        int lo = 2 * t - (t & (stride - 1));
        int hi = lo + stride;
        bool up = (lo & size) == 0;
        uint64_t a = sc[lo], b = sc[hi];
        uint32_t ia = si[lo], ib = si[hi];
        bool swap = up ? tk_less(b, ib, a, ia) : tk_less(a, ia, b, ib);
        if (swap) {
          sc[lo] = b;
          sc[hi] = a;
          si[lo] = ib;
          si[hi] = ia;
        }
      }
      __syncthreads();
    }
  }
  uint64_t obase = (uint64_t)blockIdx.x * k;
  for (uint32_t t = threadIdx.x; t < k; t += TK_BLOCK) {
    ocode[obase + t] = sc[t];
    oidx[obase + t] = si[t];
  }
}

int topk_codes(aln_ctx *c, uint64_t *code, uint32_t *idx, uint64_t n, uint32_t k,
               uint32_t *d_out_idx, uint32_t *h_nout) {
  // repeatedly reduce each tile to its k best until one tile remains
  const uint64_t n_real = n;
  while (true) {
    uint64_t nt = (n + TK_TILE - 1) / TK_TILE;
    uint64_t *oc;
    uint32_t *oi;
    ALN_TRY(ws(c, nt * k, &oc));
    ALN_TRY(ws(c, nt * k, &oi));
    {
      ProfScope ps(c, "tile_topk");
      hipLaunchKernelGGL(k_tile_topk, dim3((unsigned)nt), dim3(TK_BLOCK), 0, c->stream, code, idx, n,
                         k, oc, oi);
    }
    ALN_TRY(check_launch("tile_topk"));
    if (nt == 1) {
      uint32_t kk = (uint32_t)(n_real < k ? n_real : k);
      ALN_HIP(hipMemcpyAsync(d_out_idx, oi, 4ull * kk, hipMemcpyDeviceToDevice, c->stream));
      ALN_HIP(hipStreamSynchronize(c->stream));
      *h_nout = kk;
      return ALN_OK;
    }
    code = oc;
    idx = oi;
    n = nt * k;  // padding entries (~0, 0xFFFFFFFF) sort last and are never among the k best
  }
}

// ---- top-k: candidates by a bound on the first key -------------------------------------------
// Sorting every tile (above) reads and compares all rows log^2 times: 1.6 of 2.0 ms for the
// first 100 of 50M rows.  The k-th smallest of the minima of disjoint chunks of rows bounds the
// k-th smallest of all rows, so one pass over the first key (the chunk minima, HBM-bound)
// leaves about k candidates when that key is spread, and all keys are compared only among them:
//   k_tk_min      a wave per chunk of 64 to 1024 rows: its minimum code
//   k_tk_bound    one block: the k-th smallest of (up to 4096 strided groups of) the minima
//   k_tk_collect  the rows within the bound, read again only in chunks that have one
//   k_tk_final    one block sorts up to tf_max candidates by all keys and row number
// With one key, equal codes are ordered by row, so the bound is a (code, chunk) pair and rows
// of the bound's code count only up to its chunk: at most k * ceil(chunks / TK_GROUPS) chunks of
// candidates whatever the values.  With more keys every row that ties on the first is a candidate.
// Candidates too many for k_tk_final go through the tile sort, or, when most rows tie, the keys'
// codes are written out and bounded as one key; more than TK_CAND candidates leave the call to the
// tile sort of all rows, also with one key.
constexpr uint32_t TK_GROUPS = 4096;
constexpr uint32_t TK_CAND = 1u << 20;
constexpr uint64_t TK_ALL = 1ull << 20;
constexpr int TF_BLOCK = 1024;

// Order-preserving unsigned code of a key value over the whole int64 range; of a code (desc
// TK_RAW) itself.
constexpr int TK_RAW = 2;
__device__ __forceinline__ uint64_t tk_code(int64_t v, int desc) {
  if (desc == TK_RAW) return (uint64_t)v;
  const uint64_t c = (uint64_t)v ^ 0x8000000000000000ull;
  return desc ? ~c : c;
}

// Chunk c: rows [c * 64 * U, +64 * U).
template <int U>
__global__ void __launch_bounds__(256) k_tk_min(const int64_t *__restrict__ key, int desc, uint64_t n,
                                                uint32_t nchunks, uint64_t *__restrict__ cmin) {
  const uint32_t c = blockIdx.x * 4 + threadIdx.x / 64;
  if (c >= nchunks) return;
  const uint64_t i0 = (uint64_t)c * (64 * U) + __lane_id();
  uint64_t m = ~0ull;
  int64_t v[U];
  // the last chunk's missing rows repeat its first row
#pragma unroll
  for (int u = 0; u < U; ++u)
    v[u] = __builtin_nontemporal_load(key + (i0 + 64 * u < n ? i0 + 64 * u : (uint64_t)c * (64 * U)));
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint64_t x = tk_code(v[u], desc);
    m = x < m ? x : m;
  }
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t x = __shfl_xor(m, o, 64);
    m = x < m ? x : m;
  }
  if (__lane_id() == 0) cmin[c] = m;
}

// ctl[0], ctl[1] = code and chunk of the k-th smallest group minimum (k <= min(nchunks,
// TK_GROUPS)), ctl[2] = 0 (the candidate count).  Groups are strided so that rows in order
// spread over them.
__global__ void __launch_bounds__(TF_BLOCK) k_tk_bound(const uint64_t *__restrict__ cmin, uint32_t nchunks,
                                                       uint32_t k, uint64_t *__restrict__ ctl) {
  __shared__ uint64_t s[TK_GROUPS];
  __shared__ uint32_t sc[TK_GROUPS];
  for (uint32_t g = threadIdx.x; g < TK_GROUPS; g += TF_BLOCK) {
    uint64_t m = ~0ull;
    uint32_t at = g < nchunks ? g : 0xFFFFFFFFu;
    for (uint32_t c = g; c < nchunks; c += TK_GROUPS)
      if (cmin[c] < m) {
        m = cmin[c];
        at = c;
      }
    s[g] = m;
    sc[g] = at;
  }
  uint32_t p2 = 64;
  while (p2 < nchunks && p2 < TK_GROUPS) p2 <<= 1;
  __syncthreads();
  for (uint32_t size = 2; size <= p2; size <<= 1)
    for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
      for (uint32_t t = threadIdx.x; t < p2 / 2; t += TF_BLOCK) {
        const uint32_t lo = 2 * t - (t & (stride - 1)), hi = lo + stride;
        const uint64_t a = s[lo], b = s[hi];
        const uint32_t ca = sc[lo], cb = sc[hi];
        if ((a > b || (a == b && ca > cb)) == ((lo & size) == 0)) {
          s[lo] = b;
          s[hi] = a;
          sc[lo] = cb;
          sc[hi] = ca;
        }
      }
      __syncthreads();
    }
  if (threadIdx.x == 0) {
    ctl[0] = s[k - 1];
    ctl[1] = sc[k - 1];
    ctl[2] = 0;
  }
}

// by_row: the key is the only one (see above).
template <int U>
__global__ void __launch_bounds__(256) k_tk_collect(const int64_t *__restrict__ key, int desc, uint64_t n,
                                                    uint32_t nchunks, int by_row, const uint64_t *__restrict__ cmin,
                                                    uint64_t *ctl, uint32_t *__restrict__ cand) {
  const uint32_t c = blockIdx.x * 4 + threadIdx.x / 64;
  if (c >= nchunks) return;
  uint64_t bound = ctl[0];
  if (cmin[c] > bound) return;
  if (by_row && c > ctl[1]) {  // past the bound's chunk only smaller codes count
    if (cmin[c] == bound) return;
    --bound;
  }
  const uint64_t i0 = (uint64_t)c * (64 * U) + __lane_id();
  uint64_t in[U];
  uint32_t cnt = 0;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint64_t i = i0 + 64 * u;
    in[u] = __builtin_amdgcn_ballot_w64(i < n && tk_code(key[i < n ? i : 0], desc) <= bound);
    cnt += (uint32_t)__popcll(in[u]);
  }
  unsigned long long pos = 0;
  if (__lane_id() == 0) pos = atomicAdd(reinterpret_cast<unsigned long long *>(ctl + 2), (unsigned long long)cnt);
  pos = __shfl(pos, 0, 64);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (in[u] >> __lane_id() & 1) {
      const uint64_t q = pos + below_count(in[u]);
      if (q < TK_CAND) cand[q] = (uint32_t)(i0 + 64 * u);
    }
    pos += (uint32_t)__popcll(in[u]);
  }
}

// The candidates k_tk_final sorts in LDS (8 bytes per key and 4 for the row each).
static inline uint32_t tf_max(int nkeys) { return nkeys <= 3 ? 2048u : 1024u; }

// The first k of the rows cand[0, m) (cand NULL: rows 0..m-1) by keys and row number, m =
// *count (count NULL: n); nothing when m exceeds `most`.
struct TfArgs {
  const int64_t *k[ALN_MAX_KEYS];
  int32_t desc[ALN_MAX_KEYS];
  int nk;
};
__global__ void __launch_bounds__(TF_BLOCK) k_tk_final(TfArgs a, const uint32_t *__restrict__ cand,
                                                       const uint64_t *__restrict__ count, uint64_t n,
                                                       uint32_t most, uint32_t k, uint32_t *__restrict__ out) {
  extern __shared__ __align__(16) uint64_t tf_lds[];
  const uint64_t m = count ? *count : n;
  if (m > most) return;
  uint32_t p2 = 2;
  while (p2 < m) p2 <<= 1;
  uint64_t *code = tf_lds;  // [key][p2]
  uint32_t *row = reinterpret_cast<uint32_t *>(tf_lds + (size_t)a.nk * p2);
  for (uint32_t i = threadIdx.x; i < p2; i += TF_BLOCK) {
    const uint32_t r = i < m ? (cand ? cand[i] : i) : 0xFFFFFFFFu;  // no row has that number: padding sorts last
    row[i] = r;
    for (int j = 0; j < a.nk; ++j) code[(size_t)j * p2 + i] = i < m ? tk_code(a.k[j][r], a.desc[j]) : ~0ull;
  }
  __syncthreads();
  for (uint32_t size = 2; size <= p2; size <<= 1)
    for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
      for (uint32_t t = threadIdx.x; t < p2 / 2; t += TF_BLOCK) {
        const uint32_t lo = 2 * t - (t & (stride - 1)), hi = lo + stride;
        bool greater = row[lo] > row[hi];
        for (int j = a.nk - 1; j >= 0; --j) {
          const uint64_t x = code[(size_t)j * p2 + lo], y = code[(size_t)j * p2 + hi];
          greater = x > y || (x == y && greater);
        }
        if (greater == ((lo & size) == 0)) {
          const uint32_t r = row[lo];
          row[lo] = row[hi];
          row[hi] = r;
          for (int j = 0; j < a.nk; ++j) {
            const uint64_t x = code[(size_t)j * p2 + lo];
            code[(size_t)j * p2 + lo] = code[(size_t)j * p2 + hi];
            code[(size_t)j * p2 + hi] = x;
          }
        }
      }
      __syncthreads();
    }
  for (uint32_t i = threadIdx.x; i < k && i < m; i += TF_BLOCK) out[i] = row[i];
}

// One key: the candidates' codes; more: their gathered key values.
__global__ void k_tk_gather(const int64_t *__restrict__ key, int desc, const uint32_t *__restrict__ cand, uint64_t m,
                            int64_t *__restrict__ out) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < m; i += (uint64_t)gridDim.x * 256)
    out[i] = (int64_t)tk_code(key[cand[i]], desc);
}

template <int U>
static void tk_candidates(aln_ctx *c, const TfArgs &a, uint64_t n, uint32_t nchunks, uint32_t k, uint64_t *cmin,
                          uint64_t *ctl, uint32_t *cand) {
  const dim3 grid((nchunks + 3) / 4);
  hipLaunchKernelGGL(k_tk_min<U>, grid, dim3(256), 0, c->stream, a.k[0], a.desc[0], n, nchunks, cmin);
  hipLaunchKernelGGL(k_tk_bound, dim3(1), dim3(TF_BLOCK), 0, c->stream, (const uint64_t *)cmin, nchunks, k, ctl);
  hipLaunchKernelGGL(k_tk_collect<U>, grid, dim3(256), 0, c->stream, a.k[0], a.desc[0], n, nchunks,
                     a.nk == 1 ? 1 : 0, (const uint64_t *)cmin, ctl, cand);
}

// The candidate path; *done = false when there are too many candidates (nothing written).
// Taken when the rows make at least k chunks of 64, or fit the final sort as they are.
static int topk_bounded(aln_ctx *c, const TfArgs &a, uint64_t n, uint32_t k, uint32_t *d_out_idx, bool *done) {
  *done = false;
  const uint32_t most = tf_max(a.nk);
  const size_t lds = (size_t)most * (8 * a.nk + 4);
  if (n <= most) {
    hipLaunchKernelGGL(k_tk_final, dim3(1), dim3(TF_BLOCK), lds, c->stream, a, (const uint32_t *)nullptr,
                       (const uint64_t *)nullptr, n, most, k, d_out_idx);
    ALN_TRY(check_launch("topk_final"));
    ALN_HIP(hipStreamSynchronize(c->stream));
    *done = true;
    return ALN_OK;
  }
  if (n < 64ull * k) return ALN_OK;
  // chunks as large as leave 8k of them (the bound is then near the k-th row's key)
  uint32_t u = 16;
  while (u > 1 && n / (64 * u) < 8ull * k) u >>= 1;
  const uint32_t nchunks = (uint32_t)((n + 64 * u - 1) / (64 * u));
  uint64_t *cmin, *ctl;
  uint32_t *cand;
  ALN_TRY(ws(c, nchunks, &cmin));
  ALN_TRY(ws(c, 3, &ctl));
  ALN_TRY(ws(c, (size_t)TK_CAND, &cand));
  {
    ProfScope ps(c, "topk_candidates");
    if (u == 16)
      tk_candidates<16>(c, a, n, nchunks, k, cmin, ctl, cand);
    else if (u == 8)
      tk_candidates<8>(c, a, n, nchunks, k, cmin, ctl, cand);
    else if (u == 4)
      tk_candidates<4>(c, a, n, nchunks, k, cmin, ctl, cand);
    else if (u == 2)
      tk_candidates<2>(c, a, n, nchunks, k, cmin, ctl, cand);
    else
      tk_candidates<1>(c, a, n, nchunks, k, cmin, ctl, cand);
  }
  ALN_TRY(check_launch("topk_candidates"));
  hipLaunchKernelGGL(k_tk_final, dim3(1), dim3(TF_BLOCK), lds, c->stream, a, (const uint32_t *)cand,
                     (const uint64_t *)(ctl + 2), n, most, k, d_out_idx);
  ALN_TRY(check_launch("topk_final"));
  uint64_t m = 0;
  ALN_TRY(copy_to_host(c, &m, ctl + 2, 8));
  if (m <= most) {
    *done = true;
    return ALN_OK;
  }
  if (m > TK_CAND) return ALN_OK;
  // Rows in order leave k chunks of candidates, an eighth of all rows at most: more are ties of
  // the first key, and the codes of all rows spread again where the candidates' tile sort is a
  // gather and ranges of every key and several launches (100,000 rows of 5 first values, first 100:
  // 190 us by the tile sort, 145 by all rows' codes, of one value, first 500, 339 and 165; 2M rows, first
  // 500 504 and 312, but first 100 241 and 247, first 10 207 and 241).
  if (a.nk > 1 && m > n / 8 && 4 * m > 320ull * u * k && (n <= TK_ALL || k >= 256)) return ALN_OK;
  // the tile sort of the candidates' codes
  const unsigned gm = grid_for(m, 256, 65536);
  uint64_t *code;
  uint32_t nout;
  ALN_TRY(ws(c, m, &code));
  if (a.nk == 1) {
    hipLaunchKernelGGL(k_tk_gather, dim3(gm), dim3(256), 0, c->stream, a.k[0], a.desc[0], (const uint32_t *)cand, m,
                       reinterpret_cast<int64_t *>(code));
  } else {
    const int64_t *ck[ALN_MAX_KEYS];
    for (int j = 0; j < a.nk; ++j) {
      int64_t *g;
      ALN_TRY(ws(c, m, &g));
      ck[j] = g;
      hipLaunchKernelGGL(k_tk_gather, dim3(gm), dim3(256), 0, c->stream, a.k[j], TK_RAW, (const uint32_t *)cand, m, g);
    }
    KeyRanges r;
    ALN_TRY(key_ranges(c, ck, a.nk, m, &r));
    if (r.total > 64) return ALN_OK;
    KeySet ks;
    key_set(r, ck, a.desc, 0, a.nk, &ks);
    hipLaunchKernelGGL(k_codes, dim3(gm), dim3(256), 0, c->stream, ks, (const uint32_t *)nullptr, m, code,
                       (uint32_t *)nullptr);
  }
  ALN_TRY(check_launch("topk_codes"));
  ALN_TRY(topk_codes(c, code, cand, m, k, d_out_idx, &nout));
  *done = true;
  return ALN_OK;
}

}  // namespace aln

using namespace aln;

extern "C" {

int aln_radix_sort_pairs(aln_ctx *c, uint64_t *d_keys, uint32_t *d_vals, uint64_t n,
                         uint32_t bits) {
  ALN_REQUIRE(c && (n == 0 || (d_keys && d_vals)), "aln_radix_sort_pairs: bad arguments");
  ws_reset(c);
  ALN_TRY(radix_sort_pairs(c, d_keys, d_vals, n, bits));
  ALN_HIP(hipStreamSynchronize(c->stream));
  return ALN_OK;
}

int aln_sort_keys(aln_ctx *c, const int64_t *const *d_keys, const int32_t *desc, int nkeys,
                  uint64_t n, uint32_t *d_perm) {
  ALN_REQUIRE(c && d_keys && (n == 0 || d_perm), "aln_sort_keys: bad arguments");
  ws_reset(c);
  ALN_TRY(sort_keys_impl(c, d_keys, desc, nkeys, n, d_perm));
  return stream_wait(c);
}

int aln_topk(aln_ctx *c, const int64_t *const *d_keys, const int32_t *desc, int nkeys, uint64_t n,
             uint32_t k, uint32_t *d_out_idx, uint32_t *h_nout) {
  ALN_REQUIRE(c && d_keys && h_nout && nkeys >= 1 && nkeys <= ALN_MAX_KEYS,
              "aln_topk: bad arguments");
  ALN_REQUIRE(n < (1ull << 32), "aln_topk: more than 2^32 rows");
  ws_reset(c);
  *h_nout = 0;
  if (n == 0 || k == 0) return ALN_OK;
  ALN_REQUIRE(d_out_idx, "aln_topk: no output buffer");
  TfArgs a;
  memset(&a, 0, sizeof(a));
  a.nk = nkeys;
  for (int j = 0; j < nkeys; ++j) {
    a.k[j] = d_keys[j];
    a.desc[j] = desc && desc[j] ? 1 : 0;
  }
  bool done = false;
  if (k <= TK_TILE / 2) {
    ALN_TRY(topk_bounded(c, a, n, k, d_out_idx, &done));
    if (done) {
      *h_nout = (uint32_t)(n < k ? n : k);
      return ALN_OK;
    }
    ws_reset(c);
  }
  KeyRanges r;
  ALN_TRY(key_ranges(c, d_keys, nkeys, n, &r));
  if (r.total > 64 || k > TK_TILE / 2) {
    // wide keys or large k: full stable sort, then the prefix (emit_order + LIMIT)
    uint32_t *perm;
    ALN_TRY(ws(c, n, &perm));
    ALN_TRY(sort_with_ranges(c, r, d_keys, desc, nkeys, n, perm));
    uint32_t kk = (uint32_t)(n < k ? n : k);
    ALN_HIP(hipMemcpyAsync(d_out_idx, perm, 4ull * kk, hipMemcpyDeviceToDevice, c->stream));
    ALN_HIP(hipStreamSynchronize(c->stream));
    *h_nout = kk;
    return ALN_OK;
  }
  uint64_t *code;
  uint32_t *idx;
  ALN_TRY(ws(c, n, &code));
  ALN_TRY(ws(c, n, &idx));
  KeySet ks;
  key_set(r, d_keys, desc, 0, nkeys, &ks);
  hipLaunchKernelGGL(k_codes, dim3(grid_for(n, 256, 65536)), dim3(256), 0, c->stream, ks,
                     (const uint32_t *)nullptr, n, code, idx);
  ALN_TRY(check_launch("codes"));
  if (nkeys > 1) {  // too many rows tie on the first key: the codes of all of them as one key
    a.nk = 1;
    a.k[0] = reinterpret_cast<const int64_t *>(code);
    a.desc[0] = TK_RAW;
    ALN_TRY(topk_bounded(c, a, n, k, d_out_idx, &done));
    if (done) {
      *h_nout = (uint32_t)(n < k ? n : k);
      return ALN_OK;
    }
  }
  return topk_codes(c, code, idx, n, k, d_out_idx, h_nout);
}

}  // extern "C"
