// GROUP BY with SUM / COUNT / MIN / MAX, and row hashing.
//
// The reference groups by sorting (order_inplace, operators.cu:367-406), finding run heads
// (CudaSet::GroupBy, cm.cu:910-956) and reducing each run (moderngpu segreduce,
// select.cu:481-684); across segments it merges partial groups by MurmurHash64A of the key
// tuple on the host (add / count_avg, merge.cu:92-496).  Integer sums are exact, so the
// result does not depend on the order rows are added in, and this kernel aggregates in an
// table of accumulators instead:
//   * keys are packed into one 63-bit code (key_i - min_i in bits_i bits, key 0 most
//     significant); codes of at most GB_DENSE_BITS bits index the accumulators directly,
//     wider ones go through an open-addressing table (64-bit CAS, linear probing), first
//     one sized for 2^20 groups and, if more turn up, one of 2n slots;
//   * runs of equal codes in adjacent lanes (clustered input) are pre-reduced with a
//     segmented wave scan, and each block adds its rows into an LDS table first, so hot
//     keys and small group counts aggregate in LDS and reach the global table once per
//     block;
//   * few codes (all accumulators fit in LDS): every block keeps them all, in one copy per
//     lane while they fit, and the blocks' results are added up at the end;
//   * many codes and many rows: the rows are first moved next to the rows of the same part of
//     the code range, and each part is then added up in LDS;
//   * no GROUP BY (or keys that never vary) is one group: a block reduction;
//   * the groups are compacted and put in the reference's output order: ascending key
//     tuple (one segment) or ascending MurmurHash64A(keys, 8*nkeys, seed) (the
//     multi-segment merge order).
// Key tuples wider than 63 bits, and wide codes of which a sample shows many groups, go the
// reference's way: sort, run heads, per-run reduction (groupsort.hip).
#include <string.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "groupby.h"

namespace aln {

constexpr uint64_t GB_EMPTY = ~0ull;
// Packed key codes of at most this many bits (and at most 2n codes) use direct-indexed
// accumulators instead of a hash table.
constexpr uint32_t GB_DENSE_BITS = 26;
// The first hash table holds this many groups (at most half full) before the rows are
// aggregated again in a table of 2n slots.
constexpr uint64_t GB_HASH_START = 1ull << 20;
constexpr uint64_t GB_FIRST_PROBES = 64;
// Rows from which wide codes of many groups may be sorted instead (gb_wide), and from which a sample
// of 8192 rows is taken instead of 2048.
constexpr uint64_t GB_SORT_MIN = 1ull << 17, GB_SORT_LARGE = 1ull << 20;
// Codes that never index accumulators directly, but fit a word.
__host__ __device__ constexpr bool gb_wide_bits(uint32_t bits) { return bits > GB_DENSE_BITS && bits <= 63; }

__global__ void __launch_bounds__(256) k_gb_init(uint64_t *tkey, GbArgs a, uint64_t cap) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < cap;
       i += (uint64_t)gridDim.x * 256) {
    tkey[i] = GB_EMPTY;
    for (int v = 0; v < a.nv; ++v) a.tab[v][i] = agg_identity(a.aggs[v]);
  }
}

// Adjacent lanes with equal codes (clustered input): the last lane of each run gets the
// run's combined values and row count and returns true.  As many combining steps as the wave's
// longest run needs: none for unclustered rows.
__device__ __forceinline__ bool gb_wave_runs(const GbArgs &a, bool valid, uint64_t code, int64_t *val,
                                             uint32_t *cnt) {
  const unsigned lane = __lane_id();
  const uint64_t prev = __shfl_up(code, 1, 64);
  const uint64_t heads = __builtin_amdgcn_ballot_w64(lane == 0 || prev != code);  // valid lanes come first
  const uint64_t live = __builtin_amdgcn_ballot_w64(valid);
  *cnt = 1;
  if (~heads == 0) return valid;
  const uint64_t upto = heads & (lane == 63 ? ~0ull : (2ull << lane) - 1);
  const int below = (int)lane - (63 - __builtin_clzll(upto));
  *cnt = (uint32_t)below + 1;
  for (int o = 1; o < 64; o <<= 1) {
    if (!__builtin_amdgcn_ballot_w64(valid && below >= o)) break;
    for (int v = 0; v < a.nv; ++v) {
      const int64_t vu = __shfl_up(val[v], o, 64);
      if (below >= o) val[v] = agg_combine(a.aggs[v], vu, val[v]);
    }
  }
  return valid && (lane == 63 || !(live >> (lane + 1) & 1) || (heads >> (lane + 1) & 1));
}

__device__ __forceinline__ uint64_t gb_code(const GbArgs &a, uint64_t i) {
  uint64_t code = 0;
  for (int k = 0; k < a.nk; ++k)
    code |= (((uint64_t)a.keys[k][i] - (uint64_t)a.kmin[k]) & a.fmask[k]) << a.shift[k];
  return code;
}

// The global table: DENSE, slot = code (row count in gcnt, when there is no COUNT
// aggregate to tell the groups); otherwise open addressing over tkey
// (cap a power of two) by linear probing.  A new key counts into *ngroups; past glimit
// keys, a probe run past GB_FIRST_PROBES in such a limited table, or a full table,
// *overflow is set (the host retries with a larger table).
template <bool DENSE>
__device__ __forceinline__ void gb_global_add(const GbArgs &a, uint64_t code, const int64_t *val, uint32_t cnt,
                                              uint64_t *tkey, uint64_t cap, uint32_t *gcnt, uint32_t *ngroups,
                                              uint32_t glimit, uint32_t *overflow) {
  uint64_t h;
  if (DENSE) {
    h = code;
    if (gcnt) atomicAdd(&gcnt[h], cnt);
  } else {
    // a first, small table that has overflowed is given up: its rows are aggregated again
    const bool first = glimit != 0xFFFFFFFFu;
    if (first && __hip_atomic_load(overflow, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
    const uint64_t mask = cap - 1, limit = first ? GB_FIRST_PROBES : cap;
    h = murmur64a_u64(code, 0x9747b28cu) & mask;
    uint64_t probes = 0;
    while (true) {
      uint64_t cur = tkey[h];
      if (cur == GB_EMPTY) {
        const unsigned long long old = atomicCAS((unsigned long long *)&tkey[h], (unsigned long long)GB_EMPTY,
                                                 (unsigned long long)code);
        if (old == GB_EMPTY) {
          if (atomicAdd(ngroups, 1u) >= glimit) atomicExch(overflow, 1u);
          cur = code;
        } else {
          cur = old;
        }
      }
      if (cur == code) break;
      h = (h + 1) & mask;
      if (++probes > limit) {
        atomicExch(overflow, 1u);
        return;
      }
    }
  }
  for (int v = 0; v < a.nv; ++v) agg_atomic(a.aggs[v], &a.tab[v][h], val[v]);
}

// Aggregation with a per-block LDS table in front of the global one: the block's rows
// (grid-stride) add into GB_LT LDS slots (a hash of the code, GB_LT_PROBES probes; DENSE with
// at most GB_LT codes: slot = code), so hot keys and small group counts aggregate in LDS;
// rows whose key finds no slot go to the global table at once, and the LDS slots are added
// to it at the end.  LDS (dynamic): keys[GB_LT] u64, counts[GB_LT] u32, accumulators
// [nv][GB_LT] i64.
constexpr int GB_LT = 1024;
constexpr int GB_LT_PROBES = 8;

__host__ __device__ constexpr size_t gb_lds_bytes(int nv) { return (size_t)GB_LT * (8 + 4 + 8 * (size_t)nv); }

template <bool DENSE>
__global__ void __launch_bounds__(256) k_gb_agg(GbArgs a, uint64_t n, uint64_t *tkey, uint64_t cap,
                                                uint32_t *gcnt, uint32_t *ngroups, uint32_t glimit,
                                                uint32_t *overflow) {
  extern __shared__ __align__(16) int64_t gb_lds[];
  uint64_t *lkey = reinterpret_cast<uint64_t *>(gb_lds);
  int64_t *lacc = gb_lds + GB_LT;
  uint32_t *lcnt = reinterpret_cast<uint32_t *>(gb_lds + GB_LT + (size_t)a.nv * GB_LT);
  const bool direct = DENSE && cap <= (uint64_t)GB_LT;
  for (int s = threadIdx.x; s < GB_LT; s += 256) {
    lkey[s] = direct ? (uint64_t)s : GB_EMPTY;
    lcnt[s] = 0;
    for (int v = 0; v < a.nv; ++v) lacc[(size_t)v * GB_LT + s] = agg_identity(a.aggs[v]);
  }
  __syncthreads();
  for (uint64_t i0 = (uint64_t)blockIdx.x * 256; i0 < n; i0 += (uint64_t)gridDim.x * 256) {
    const uint64_t i = i0 + threadIdx.x;
    const bool valid = i < n;
    const uint64_t code = valid ? gb_code(a, i) : 0;
    int64_t val[ALN_MAX_AGGS];
    for (int v = 0; v < a.nv; ++v) {
      val[v] = !valid ? 0 : a.aggs[v] == ALN_AGG_COUNT ? 1 : a.vals[v][i];
      if ((a.aggs[v] == ALN_AGG_FMIN || a.aggs[v] == ALN_AGG_FMAX) && bits_f64(val[v]) != bits_f64(val[v]))
        val[v] = agg_identity(a.aggs[v]);  // NaN takes no part, also at the start of a run
    }
    uint32_t cnt;
    if (!gb_wave_runs(a, valid, code, val, &cnt)) continue;
    int slot = -1;
    if (direct) {
      slot = (int)code;
    } else {
      uint32_t h = (uint32_t)murmur64a_u64(code, 0x85ebca6bu) & (GB_LT - 1);
      for (int p = 0; p < GB_LT_PROBES; ++p) {
        uint64_t k = lkey[h];
        if (k == GB_EMPTY) {
          const unsigned long long old =
              atomicCAS((unsigned long long *)&lkey[h], (unsigned long long)GB_EMPTY, (unsigned long long)code);
          k = old == GB_EMPTY ? code : old;
        }
        if (k == code) {
          slot = (int)h;
          break;
        }
        h = (h + 1) & (GB_LT - 1);
      }
    }
    if (slot >= 0) {
      atomicAdd(&lcnt[slot], cnt);
      for (int v = 0; v < a.nv; ++v) agg_atomic(a.aggs[v], &lacc[(size_t)v * GB_LT + slot], val[v]);
    } else {
      gb_global_add<DENSE>(a, code, val, cnt, tkey, cap, gcnt, ngroups, glimit, overflow);
    }
  }
  __syncthreads();
  for (int s = threadIdx.x; s < GB_LT; s += 256) {
    const uint32_t c = lcnt[s];
    if (c == 0) continue;
    int64_t val[ALN_MAX_AGGS];
    for (int v = 0; v < a.nv; ++v) val[v] = lacc[(size_t)v * GB_LT + s];
    gb_global_add<DENSE>(a, lkey[s], val, c, tkey, cap, gcnt, ngroups, glimit, overflow);
  }
}

// ---- few groups: all accumulators in LDS -----------------------------------------------------
// Every block keeps an accumulator per (aggregate, code), in 2^lr copies spread over the lanes
// (one bank column each: with 64 copies a wave's LDS atomics never meet), so no row touches
// global memory and no wave-wide combination is needed; the blocks' accumulators go to part[]
// and one wave per accumulator adds them up.  60M rows, 8 codes, count + 2 sums + f64 sum, min,
// max: 3.68 ms (a segmented wave scan of every value and one copy) -> 0.53 ms, 6.3 TB/s.
// Bounded by HBM: the keys and values once.  f64 MIN / MAX are kept as int64 keys in the order
// of the doubles (NaN never enters, as in agg_combine).
constexpr int GL_U = 8;  // rows of a thread in flight
constexpr size_t GL_COPIES = 32768;  // copies are made while they fit this
constexpr size_t GL_MOST = 65536;    // one copy fits this
constexpr uint64_t GL_PART = 1ull << 22;  // block results kept, at most (accumulators x blocks)

constexpr uint64_t GL_SAMPLE_MIN = 1ull << 20;  // rows from which a sample's ranges are tried
constexpr uint32_t GL_SAMPLE_BITS = 10;  // and the codes: wider ranges than 1024 values are
                                         // seldom hit in full by a sample of 16384 rows

struct GlArgs {
  GbArgs g;         // g.nv accumulators per code, accumulator `cnt` the row count
  int cnt;
  uint32_t ncodes, lr;
};

__device__ __forceinline__ int64_t gl_identity(int a) { return f64_unorder_key(agg_identity(a)); }

// Combines accumulators (f64 MIN / MAX as keys).
__device__ __forceinline__ int64_t gl_combine(int a, int64_t x, int64_t y) {
  if (a == ALN_AGG_MIN || a == ALN_AGG_FMIN) return x < y ? x : y;
  if (a == ALN_AGG_MAX || a == ALN_AGG_FMAX) return x > y ? x : y;
  return agg_combine(a, x, y);
}

// Adds U values into LDS accumulators acc[at[u]] (ag wave-uniform, not COUNT).
template <int U>
__device__ __forceinline__ void gl_add(int ag, int64_t *acc, const uint32_t (&at)[U], const bool (&in)[U],
                                       const int64_t (&x)[U]) {
#define GL_EACH(cond, stmt)                       \
  _Pragma("unroll") for (int u = 0; u < U; ++u) { \
    int64_t *t = acc + at[u];                     \
    const int64_t y = x[u];                       \
    if (in[u] && (cond)) stmt;                    \
  }                                               \
  break
  switch (ag) {
    case ALN_AGG_SUM: GL_EACH(true, atomicAdd((unsigned long long *)t, (unsigned long long)y));
    case ALN_AGG_MIN: GL_EACH(true, atomicMin((long long *)t, (long long)y));
    case ALN_AGG_MAX: GL_EACH(true, atomicMax((long long *)t, (long long)y));
    case ALN_AGG_FSUM: GL_EACH(true, atomicAdd(reinterpret_cast<double *>(t), bits_f64(y)));
    case ALN_AGG_FMIN: GL_EACH(bits_f64(y) == bits_f64(y), atomicMin((long long *)t, (long long)f64_unorder_key(y)));
    default: GL_EACH(bits_f64(y) == bits_f64(y), atomicMax((long long *)t, (long long)f64_unorder_key(y)));
  }
#undef GL_EACH
}

__global__ void __launch_bounds__(256) k_gl_agg(GlArgs a, uint64_t n, int64_t *__restrict__ part,
                                                uint32_t *__restrict__ bad) {
  extern __shared__ __align__(16) int64_t gl_acc[];
  const uint32_t per = a.ncodes << a.lr;  // one aggregate's accumulators
  for (int v = 0; v < a.g.nv; ++v) {
    const int64_t id = a.g.aggs[v] == ALN_AGG_FMIN || a.g.aggs[v] == ALN_AGG_FMAX ? gl_identity(a.g.aggs[v])
                                                                                 : agg_identity(a.g.aggs[v]);
    for (uint32_t i = threadIdx.x; i < per; i += 256) gl_acc[(size_t)v * per + i] = id;
  }
  __syncthreads();
  const uint32_t copy = threadIdx.x & ((1u << a.lr) - 1u);
  bool outside = false;
  for (uint64_t i0 = (uint64_t)blockIdx.x * (256 * GL_U); i0 < n; i0 += (uint64_t)gridDim.x * (256 * GL_U)) {
    uint32_t at[GL_U];
    bool in[GL_U];
#pragma unroll
    for (int u = 0; u < GL_U; ++u) {
      at[u] = 0;
      in[u] = i0 + threadIdx.x + 256 * u < n;
    }
    for (int k = 0; k < a.g.nk; ++k) {
      const int64_t *__restrict__ key = a.g.keys[k] + i0 + threadIdx.x;
      const uint64_t kmin = (uint64_t)a.g.kmin[k], fmask = a.g.fmask[k];
      const uint32_t sh = a.g.shift[k] + a.lr;
      int64_t x[GL_U];
#pragma unroll
      for (int u = 0; u < GL_U; ++u) x[u] = in[u] ? __builtin_nontemporal_load(key + 256 * u) : (int64_t)kmin;
#pragma unroll
      for (int u = 0; u < GL_U; ++u) {
        const uint64_t d = (uint64_t)x[u] - kmin;
        outside = outside || d > fmask;
        in[u] = in[u] && d <= fmask;
        at[u] |= (uint32_t)(d & fmask) << sh;
      }
    }
    for (int v = 0; v < a.g.nv; ++v) {
      const int ag = a.g.aggs[v];
      int64_t *acc = gl_acc + (size_t)v * per + copy;
      if (ag == ALN_AGG_COUNT) {
#pragma unroll
        for (int u = 0; u < GL_U; ++u)
          if (in[u]) atomicAdd((unsigned long long *)(acc + at[u]), 1ull);
        continue;
      }
      const int64_t *__restrict__ val = a.g.vals[v] + i0 + threadIdx.x;
      int64_t x[GL_U];
#pragma unroll
      for (int u = 0; u < GL_U; ++u) x[u] = in[u] ? __builtin_nontemporal_load(val + 256 * u) : 0;
      gl_add<GL_U>(ag, acc, at, in, x);
    }
  }
  if (outside) *bad = 1;
  __syncthreads();
  const uint32_t nacc = a.ncodes * (uint32_t)a.g.nv;
  for (uint32_t s = threadIdx.x; s < nacc; s += 256) {
    const int ag = a.g.aggs[s / a.ncodes];
    const int64_t *t = gl_acc + ((size_t)s << a.lr);
    int64_t r = t[0];
    for (uint32_t c = 1; c < (1u << a.lr); ++c) r = gl_combine(ag, r, t[c]);
    part[(uint64_t)s * gridDim.x + blockIdx.x] = r;
  }
}

// One wave per accumulator: the blocks' results into the tables (g.tab[v][code]).
__global__ void __launch_bounds__(256) k_gl_sum(GlArgs a, const int64_t *__restrict__ part, uint32_t nb) {
  const uint32_t s = blockIdx.x * 4 + threadIdx.x / 64;
  if (s >= a.ncodes * (uint32_t)a.g.nv) return;
  const int v = (int)(s / a.ncodes), ag = a.g.aggs[v];
  const int64_t *__restrict__ p = part + (uint64_t)s * nb;
  // lanes past the blocks repeat block 0's MIN / MAX, or add nothing
  const bool sum = ag == ALN_AGG_COUNT || ag == ALN_AGG_SUM || ag == ALN_AGG_FSUM;
  int64_t r = __lane_id() < nb ? p[__lane_id()] : sum ? 0 : p[0];
  for (uint32_t b = 64 + __lane_id(); b < nb; b += 64) r = gl_combine(ag, r, p[b]);
  for (int o = 32; o > 0; o >>= 1) r = gl_combine(ag, r, (int64_t)__shfl_xor((long long)r, o, 64));
  if (__lane_id() == 0)
    a.g.tab[v][s - v * a.ncodes] = ag == ALN_AGG_FMIN || ag == ALN_AGG_FMAX ? f64_unorder_key(r) : r;
}

// The groups (codes with rows) in code order into the outputs; the number of groups and whether a
// key lay outside the code range to the host.  Nothing is written when one did or there are more
// groups than cap: the call may start again, from inputs that the outputs may lie over.
__global__ void __launch_bounds__(1024) k_gl_emit(GlArgs a, GbOut o, int nv, uint64_t cap,
                                                  const uint32_t *__restrict__ bad, DevResult r) {
  __shared__ uint32_t wsum[16];
  static_assert(GL_MOST / 8 <= 32 * 1024, "a bit per tile of 1024 codes");
  const uint32_t miss = *bad;
  uint32_t mine = 0, n = 0;  // this thread's codes with rows, a bit per tile; the wave's number of them
  for (uint32_t c0 = 0; c0 < a.ncodes; c0 += 1024) {
    const uint32_t c = c0 + threadIdx.x;
    const bool f = c < a.ncodes && a.g.tab[a.cnt][c] != 0;
    mine |= (f ? 1u : 0u) << (c0 / 1024);
    n += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(f));
  }
  if (__lane_id() == 0) wsum[threadIdx.x / 64] = n;
  __syncthreads();
  uint32_t total = 0;
  for (uint32_t w = 0; w < 16; ++w) total += wsum[w];
  __syncthreads();
  uint64_t base = 0;
  for (uint32_t c0 = 0; c0 < a.ncodes && !miss && total <= cap; c0 += 1024) {
    const uint32_t c = c0 + threadIdx.x;
    const bool f = mine >> (c0 / 1024) & 1;
    const uint64_t bal = __builtin_amdgcn_ballot_w64(f);
    if (__lane_id() == 0) wsum[threadIdx.x / 64] = (uint32_t)__popcll(bal);
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (uint32_t w = 0; w < 16; ++w) {
      before += w < threadIdx.x / 64 ? wsum[w] : 0;
      all += wsum[w];
    }
    const uint64_t pos = base + before + below_count(bal);
    if (f) {
      for (int k = 0; k < a.g.nk; ++k)
        o.keys[k][pos] = (int64_t)((uint64_t)a.g.kmin[k] + ((c >> a.g.shift[k]) & a.g.fmask[k]));
      for (int v = 0; v < nv; ++v) o.vals[v][pos] = a.g.tab[v][c];
    }
    base += all;
    __syncthreads();
  }
  block_stores_done();  // the call returns on the result: every wave's groups are written by then
  if (threadIdx.x == 0) {
    r.dst[0] = total;
    r.dst[1] = miss;
    result_done(r);
  }
}

// What a sample of 1024 J rows, 16 J spread runs of 64 (n >= 1024 J), tells of wide keys.
enum { GW_FOUND, GW_ONCE, GW_MOST, GW_EQUAL, GW_RISING, GW_WORDS };
// By a block of 1024 threads: latency only, so all rows are read at once.  Rows are told apart by
// their tuple's hash; those that start a run of equal tuples are counted in an LDS table of 18-bit
// fingerprints and 14-bit counts, at most half full:
//   FOUND  distinct tuples, ONCE those of one run, MOST the runs of the most frequent one;
//   EQUAL  rows whose tuple is that of the row before (in their 64);
//   RISING how many of the 16 J first rows have a first key not below the one before.
template <int J>
__device__ __forceinline__ void gb_wide_sample(const GbArgs &a, uint64_t n, uint64_t *__restrict__ out) {
  constexpr uint32_t SET = 2048 * J;
  __shared__ uint32_t set[SET];
  __shared__ int64_t first[16 * J];
  __shared__ uint32_t sum[GW_WORDS];
  const uint64_t step = (n - 64) / (16 * J - 1);
  int64_t kv[J][ALN_MAX_KEYS];
#pragma unroll
  for (int k = 0; k < ALN_MAX_KEYS; ++k)
#pragma unroll
    for (int j = 0; j < J; ++j)
      kv[j][k] = k < a.nk ? a.keys[k][step * (16 * j + threadIdx.x / 64) + __lane_id()] : 0;
  for (uint32_t i = threadIdx.x; i < SET; i += 1024) set[i] = 0;
  if (threadIdx.x < GW_WORDS) sum[threadIdx.x] = 0;
  __syncthreads();
  uint32_t w[GW_WORDS] = {0, 0, 0, 0, 0};
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const uint64_t h = murmur64a_tuple(kv[j], a.nk, 0x9747b28cu), above = __shfl_up(h, 1, 64);
    if (__lane_id() == 0) first[16 * j + threadIdx.x / 64] = kv[j][0];
    if (__lane_id() > 0 && above == h) {
      ++w[GW_EQUAL];
      continue;
    }
    const uint32_t f = (uint32_t)(h >> 46) | 1u;
    uint32_t at = (uint32_t)h & (SET - 1);
    while (true) {
      const uint32_t old = atomicCAS(&set[at], 0u, f << 14 | 1u);
      if (old != 0 && old >> 14 == f) atomicAdd(&set[at], 1u);
      if (old == 0 || old >> 14 == f) break;
      at = (at + 1) & (SET - 1);
    }
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < SET; i += 1024) {
    const uint32_t c = set[i] & 0x3FFFu;
    w[GW_FOUND] += c != 0;
    w[GW_ONCE] += c == 1;
    w[GW_MOST] = c > w[GW_MOST] ? c : w[GW_MOST];
  }
  if (threadIdx.x > 0 && threadIdx.x < 16 * J) w[GW_RISING] = first[threadIdx.x] >= first[threadIdx.x - 1];
#pragma unroll
  for (int q = 0; q < GW_WORDS; ++q) {
    for (int o = 32; o > 0; o >>= 1) {
      const uint32_t x = (uint32_t)__shfl_xor((int)w[q], o, 64);
      w[q] = q == GW_MOST ? (x > w[q] ? x : w[q]) : w[q] + x;
    }
    if (__lane_id() == 0) {
      if (q == GW_MOST)
        atomicMax(&sum[q], w[q]);
      else
        atomicAdd(&sum[q], w[q]);
    }
  }
  __syncthreads();
  if (threadIdx.x == 0)
    for (int q = 0; q < GW_WORDS; ++q) out[q] = sum[q];
}

template <int J>
__global__ void __launch_bounds__(1024) k_gb_sample(GbArgs a, uint64_t n, DevResult r) {
  gb_wide_sample<J>(a, n, r.dst);
  if (threadIdx.x == 0) result_done(r);
}

// Smallest and largest key values among 16 spread runs of 1024 rows (n >= 16384), one block; and,
// when these ranges make wide codes already, what gb_wide asks of them (the same wait).
__global__ void __launch_bounds__(1024) k_gl_sample(GbArgs a, uint64_t n, DevResult r) {
  __shared__ int64_t lo[16], hi[16];
  __shared__ uint32_t bits;
  const uint64_t step = (n - 1024) / 15;
  if (threadIdx.x == 0) bits = 0;
  for (int k = 0; k < a.nk; ++k) {
    int64_t x[16], mn = INT64_MAX, mx = INT64_MIN;
#pragma unroll
    for (int j = 0; j < 16; ++j) x[j] = a.keys[k][step * j + threadIdx.x];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      mn = x[j] < mn ? x[j] : mn;
      mx = x[j] > mx ? x[j] : mx;
    }
    for (int d = 32; d > 0; d >>= 1) {
      const int64_t p = __shfl_xor(mn, d, 64), q = __shfl_xor(mx, d, 64);
      mn = p < mn ? p : mn;
      mx = q > mx ? q : mx;
    }
    if (__lane_id() == 0) {
      lo[threadIdx.x / 64] = mn;
      hi[threadIdx.x / 64] = mx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < 16; ++w) {
        mn = lo[w] < mn ? lo[w] : mn;
        mx = hi[w] > mx ? hi[w] : mx;
      }
      r.dst[2 * k] = (uint64_t)mn;
      r.dst[2 * k + 1] = (uint64_t)mx;
      bits += mx == mn ? 0 : 64 - (uint32_t)__builtin_clzll((uint64_t)mx - (uint64_t)mn);
    }
    __syncthreads();
  }
  if (gb_wide_bits(bits)) gb_wide_sample<8>(a, n, r.dst + 2 * ALN_MAX_KEYS);
  if (threadIdx.x == 0) result_done(r);
}

// ---- many codes: partitions of the code range ------------------------------------------------
// Global atomics run at 24 G/s whatever they hit (30M rows into 3.3M groups: 43M of them, 1.8 ms),
// so for many rows the codes are split by (code >> GP_LOW) & (parts - 1) into parts whose
// accumulators fit in LDS, the rows are moved into part order (code and value columns, through
// an LDS reorder of 4096-row tiles so that a part's rows leave in runs), and a block per part
// adds its rows up in LDS and stores the part's table.  The low bits stay out of the choice so
// that the table is written in whole 64-byte sectors; low in the code, they spread the hot keys
// of a skewed column (small codes, mostly) over the parts.  A part of more than `chunk` rows is
// added up by several blocks, which then add into the table with atomics.
// Bounded by the moves: the key twice, each value column read, written and read again (30M rows
// of one key and one value column: count 62, move 163, add up 124 us).
constexpr uint32_t GP_LOW = 3;
constexpr int GP_BLOCK = 512;
constexpr int GP_ITEMS = 8;
constexpr uint32_t GP_TILE = GP_BLOCK * GP_ITEMS;
constexpr uint32_t GP_PARTS_MIN = 64, GP_PARTS_FEW = 256, GP_PARTS_MAX = 2048;
constexpr uint32_t GP_SUB = 8;           // tiles a count block counts
constexpr uint32_t GP_XCDS = 8;
// Fewer rows go through the atomics of k_gb_agg, in one launch instead of five (60000 codes,
// uniform and Zipf: 150000 rows 78 and 92 us against 77 and 98 in parts; 250000 rows 87 and 104
// against 78 and 84; 1M rows 152 and 219 against 85 and 89).
constexpr uint64_t GP_ROWS_MIN = 3ull << 16;
constexpr uint64_t GP_BYTES_MAX = 16ull << 30;  // moved rows
constexpr size_t GP_LDS = 65536, GP_LDS_MAX = 131072;

struct GpArgs {
  GbArgs g;                // accumulators as in GlArgs: the row count is g.aggs[cnt]
  int cnt;
  int ncol;                // distinct value columns
  const int64_t *col[ALN_MAX_AGGS];
  int64_t *moved[ALN_MAX_AGGS];
  int32_t col_of[ALN_MAX_AGGS + 1];
  uint32_t *code;          // moved codes
  uint64_t n;
  uint32_t ntiles, nsub, nsuper, lp, ncodes, chunk;  // nsuper: count blocks, of nsub tiles
  uint32_t *cnts, *excl, *tot;   // [part][count block], [count block][part], [part]
  uint16_t *sub;                 // [tile][part]: the part's rows in the count block's earlier tiles
  uint32_t *start, *work;        // [parts + 1]: first row, first work item of a part
};

__device__ __forceinline__ uint32_t gp_part(uint32_t code, uint32_t lp) { return (code >> GP_LOW) & ((1u << lp) - 1u); }

// The codes of the tile's rows GP_BLOCK * j + thread (past the end: 0).
__device__ __forceinline__ void gp_codes(const GpArgs &a, uint64_t i0, uint32_t (&code)[GP_ITEMS]) {
#pragma unroll
  for (int j = 0; j < GP_ITEMS; ++j) code[j] = 0;
  for (int k = 0; k < a.g.nk; ++k) {
    const int64_t *__restrict__ key = a.g.keys[k];
    int64_t x[GP_ITEMS];
#pragma unroll
    for (int j = 0; j < GP_ITEMS; ++j) {
      const uint64_t i = i0 + threadIdx.x + GP_BLOCK * j;
      x[j] = i < a.n ? __builtin_nontemporal_load(key + i) : a.g.kmin[k];
    }
#pragma unroll
    for (int j = 0; j < GP_ITEMS; ++j)
      code[j] |= (uint32_t)(((uint64_t)x[j] - (uint64_t)a.g.kmin[k]) & a.g.fmask[k]) << a.g.shift[k];
  }
}

// The counters of a tile: GP_PARTS_MAX of them, that many copies per part, spread over the lanes.
__global__ void __launch_bounds__(GP_BLOCK) k_gp_count(GpArgs a) {
  __shared__ uint32_t h[GP_PARTS_MAX];
  constexpr uint32_t PER = GP_PARTS_MAX / GP_BLOCK;
  const uint32_t parts = 1u << a.lp, copies = GP_PARTS_MAX >> a.lp, copy = threadIdx.x & (copies - 1);
  uint32_t run[PER];  // of parts thread, thread + GP_BLOCK, ..
#pragma unroll
  for (uint32_t q = 0; q < PER; ++q) run[q] = 0;
  for (uint32_t s = 0; s < a.nsub; ++s) {
    const uint64_t tile = (uint64_t)blockIdx.x * a.nsub + s, i0 = tile * GP_TILE;
    if (i0 >= a.n) break;
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) h[threadIdx.x + GP_BLOCK * q] = 0;
    uint32_t code[GP_ITEMS];
    gp_codes(a, i0, code);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < GP_ITEMS; ++j)
      if (i0 + threadIdx.x + GP_BLOCK * j < a.n) atomicAdd(&h[gp_part(code[j], a.lp) * copies + copy], 1u);
    __syncthreads();
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) {
      const uint32_t p = threadIdx.x + GP_BLOCK * q;
      if (p >= parts) continue;
      a.sub[tile * parts + p] = (uint16_t)run[q];
      for (uint32_t k = 0; k < copies; ++k) run[q] += h[p * copies + ((k + p) & (copies - 1))];
    }
    __syncthreads();
  }
#pragma unroll
  for (uint32_t q = 0; q < PER; ++q) {
    const uint32_t p = threadIdx.x + GP_BLOCK * q;
    if (p < parts) a.cnts[(uint64_t)p * a.nsuper + blockIdx.x] = run[q];
  }
}

// Block p: exclusive scan of part p's counts.
__global__ void __launch_bounds__(256) k_gp_rows(GpArgs a) {
  __shared__ uint32_t wsum[4];
  const uint32_t p = blockIdx.x, t = threadIdx.x, parts = 1u << a.lp;
  const uint32_t per = (a.nsuper + 255) / 256, b = t * per, e = b + per < a.nsuper ? b + per : a.nsuper;
  const uint32_t *row = a.cnts + (uint64_t)p * a.nsuper;
  uint32_t s = 0;
  for (uint32_t i = b; i < e; ++i) s += row[i];
  uint32_t x = s;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o, 64);
    if (__lane_id() >= (unsigned)o) x += y;
  }
  if (__lane_id() == 63) wsum[t / 64] = x;
  __syncthreads();
  uint32_t before = x - s;
  for (uint32_t w = 0; w < t / 64; ++w) before += wsum[w];
  for (uint32_t i = b; i < e; ++i) {
    a.excl[(uint64_t)i * parts + p] = before;
    before += row[i];
  }
  if (t == 255) a.tot[p] = before;
}

// Exclusive scan of up to GP_PARTS_MAX values held two per thread by 1024 threads.
__device__ __forceinline__ void gp_scan2(uint32_t (&v)[2], uint32_t *wsum, uint32_t *total) {
  const uint32_t s = v[0] + v[1], t = threadIdx.x;
  uint32_t x = s;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o, 64);
    if (__lane_id() >= (unsigned)o) x += y;
  }
  if (__lane_id() == 63) wsum[t / 64] = x;
  __syncthreads();
  uint32_t before = x - s, all = 0;
  for (uint32_t w = 0; w < 16; ++w) {
    before += w < t / 64 ? wsum[w] : 0;
    all += wsum[w];
  }
  __syncthreads();
  v[1] = before + v[0];
  v[0] = before;
  *total = all;
}

// The parts' first rows and first work items.
__global__ void __launch_bounds__(1024) k_gp_base(GpArgs a) {
  __shared__ uint32_t wsum[16];
  const uint32_t parts = 1u << a.lp, p = 2 * threadIdx.x;
  uint32_t v[2], w[2], total;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    v[j] = p + j < parts ? a.tot[p + j] : 0;
    w[j] = (uint32_t)(((uint64_t)v[j] + a.chunk - 1) / a.chunk);
  }
  gp_scan2(v, wsum, &total);
  if (threadIdx.x == 0) a.start[parts] = total;
#pragma unroll
  for (int j = 0; j < 2; ++j)
    if (p + j < parts) a.start[p + j] = v[j];
  gp_scan2(w, wsum, &total);
  if (threadIdx.x == 0) a.work[parts] = total;
#pragma unroll
  for (int j = 0; j < 2; ++j)
    if (p + j < parts) a.work[p + j] = w[j];
}

// Moves a tile's rows into part order.  Within a tile the order of a part's rows is free, so a
// row's place is an LDS counter's old value.  Each XCD takes a contiguous range of tiles, so the
// runs of neighbouring tiles meet in one L2 (a block with tiles and part positions of its own
// kept 64 x 512 open lines per XCD, more than its L2: 265 against 163 us for 30M rows, one key
// and one value column).
__global__ void __launch_bounds__(GP_BLOCK) k_gp_move(GpArgs a) {
  __shared__ int64_t sv[GP_TILE];
  __shared__ uint32_t sc[GP_TILE];
  __shared__ uint32_t h[GP_PARTS_MAX], del[GP_PARTS_MAX];
  uint32_t *wsum = reinterpret_cast<uint32_t *>(sv);  // free until the first column's values
  static_assert(12 * GP_TILE + 8 * GP_PARTS_MAX <= 65536, "two blocks per CU");
  constexpr uint32_t PER = GP_PARTS_MAX / GP_BLOCK;
  const uint32_t parts = 1u << a.lp, t = threadIdx.x;
  const uint32_t copies = GP_PARTS_MAX >> a.lp, copy = t & (copies - 1);
  const uint32_t xq = a.ntiles / GP_XCDS, xr = a.ntiles % GP_XCDS, xcd = blockIdx.x % GP_XCDS;
  const uint32_t tile = xcd * xq + (xcd < xr ? xcd : xr) + blockIdx.x / GP_XCDS;
  const uint64_t i0 = (uint64_t)tile * GP_TILE;
  const uint32_t m = a.n - i0 < GP_TILE ? (uint32_t)(a.n - i0) : GP_TILE;
  uint32_t code[GP_ITEMS], rank[GP_ITEMS], off[PER];
  gp_codes(a, i0, code);
#pragma unroll
  for (uint32_t q = 0; q < PER; ++q) {  // the tile's first positions in parts t, t + GP_BLOCK, ..
    const uint32_t p = t + GP_BLOCK * q;
    off[q] = p < parts ? a.start[p] + a.excl[(uint64_t)(tile / a.nsub) * parts + p] + a.sub[(uint64_t)tile * parts + p]
                       : 0;
    h[t + GP_BLOCK * q] = 0;
  }
  int64_t y[GP_ITEMS];  // the first column's values, on their way while the rows are placed
#pragma unroll
  for (int j = 0; j < GP_ITEMS; ++j)
    y[j] = a.ncol && t + GP_BLOCK * j < m ? __builtin_nontemporal_load(a.col[0] + i0 + t + GP_BLOCK * j) : 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < GP_ITEMS; ++j)
    if (t + GP_BLOCK * j < m) rank[j] = atomicAdd(&h[gp_part(code[j], a.lp) * copies + copy], 1u);
  __syncthreads();
  uint32_t c[PER], s = 0;
#pragma unroll
  for (uint32_t q = 0; q < PER; ++q) {
    c[q] = h[t * PER + q];
    s += c[q];
  }
  uint32_t x = s;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t z = __shfl_up(x, o, 64);
    if (__lane_id() >= (unsigned)o) x += z;
  }
  if (__lane_id() == 63) wsum[t / 64] = x;
  __syncthreads();
  uint32_t before = x - s;
  for (uint32_t w = 0; w < t / 64; ++w) before += wsum[w];
#pragma unroll
  for (uint32_t q = 0; q < PER; ++q) {
    h[t * PER + q] = before;  // the counter's first place in the tile
    before += c[q];
  }
  __syncthreads();
#pragma unroll
  for (uint32_t q = 0; q < PER; ++q) {
    const uint32_t p = t + GP_BLOCK * q;
    if (p < parts) del[p] = off[q] - h[p * copies];
  }
#pragma unroll
  for (int j = 0; j < GP_ITEMS; ++j)
    if (t + GP_BLOCK * j < m) {
      rank[j] += h[gp_part(code[j], a.lp) * copies + copy];
      sc[rank[j]] = code[j];
      if (a.ncol) sv[rank[j]] = y[j];
    }
  __syncthreads();
  uint32_t dest[GP_ITEMS];
#pragma unroll
  for (int j = 0; j < GP_ITEMS; ++j) {
    const uint32_t i = t + GP_BLOCK * j;
    if (i < m) {
      const uint32_t cd = sc[i];
      dest[j] = del[gp_part(cd, a.lp)] + i;
      a.code[dest[j]] = cd;
      if (a.ncol) a.moved[0][dest[j]] = sv[i];
    }
  }
  for (int v = 1; v < a.ncol; ++v) {
#pragma unroll
    for (int j = 0; j < GP_ITEMS; ++j)
      y[j] = t + GP_BLOCK * j < m ? __builtin_nontemporal_load(a.col[v] + i0 + t + GP_BLOCK * j) : 0;
    __syncthreads();  // the last column has left sv
#pragma unroll
    for (int j = 0; j < GP_ITEMS; ++j)
      if (t + GP_BLOCK * j < m) sv[rank[j]] = y[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < GP_ITEMS; ++j)
      if (t + GP_BLOCK * j < m) a.moved[v][dest[j]] = sv[t + GP_BLOCK * j];
  }
}

// Work item b: a chunk of a part's rows, added up in LDS (f64 MIN / MAX as keys, see GlArgs).
__global__ void __launch_bounds__(1024) k_gp_agg(GpArgs a) {
  extern __shared__ __align__(16) int64_t gl_acc[];
  const uint32_t parts = 1u << a.lp, slots = a.ncodes >> a.lp;
  if (blockIdx.x >= a.work[parts]) return;
  uint32_t lo = 0, hi = parts;  // the last part whose first work item is <= this one
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) / 2;
    if (a.work[mid] <= blockIdx.x) lo = mid; else hi = mid;
  }
  const uint32_t p = lo, item = blockIdx.x - a.work[p];
  const uint64_t r0 = (uint64_t)a.start[p] + (uint64_t)item * a.chunk;
  const uint64_t r1 = r0 + a.chunk < a.start[p + 1] ? r0 + a.chunk : a.start[p + 1];
  for (int v = 0; v < a.g.nv; ++v) {
    const int ag = a.g.aggs[v];
    const int64_t id = ag == ALN_AGG_FMIN || ag == ALN_AGG_FMAX ? gl_identity(ag) : agg_identity(ag);
    for (uint32_t i = threadIdx.x; i < slots; i += 1024) gl_acc[(size_t)v * slots + i] = id;
  }
  __syncthreads();
  constexpr int U = 4;
  const uint32_t low = (1u << GP_LOW) - 1u;
  for (uint64_t i0 = r0 + threadIdx.x; i0 < r1; i0 += 1024 * U) {
    uint32_t at[U];
    bool in[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      in[u] = i0 + 1024 * u < r1;
      const uint32_t c = in[u] ? __builtin_nontemporal_load(a.code + i0 + 1024 * u) : 0;
      at[u] = (c >> (GP_LOW + a.lp) << GP_LOW) | (c & low);
    }
    for (int v = 0; v < a.g.nv; ++v) {
      const int ag = a.g.aggs[v];
      int64_t *acc = gl_acc + (size_t)v * slots;
      if (ag == ALN_AGG_COUNT) {
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (in[u]) atomicAdd((unsigned long long *)(acc + at[u]), 1ull);
        continue;
      }
      const int64_t *__restrict__ val = a.moved[a.col_of[v]] + i0;
      int64_t x[U];
#pragma unroll
      for (int u = 0; u < U; ++u) x[u] = in[u] ? val[1024 * u] : 0;
      gl_add<U>(ag, acc, at, in, x);
    }
  }
  __syncthreads();
  const bool whole = a.work[p + 1] - a.work[p] == 1;
  for (int v = 0; v < a.g.nv; ++v) {
    const int ag = a.g.aggs[v];
    for (uint32_t i = threadIdx.x; i < slots; i += 1024) {
      const uint32_t c = ((i >> GP_LOW) << (GP_LOW + a.lp)) | (p << GP_LOW) | (i & low);
      int64_t y = gl_acc[(size_t)v * slots + i];
      if (ag == ALN_AGG_FMIN || ag == ALN_AGG_FMAX) y = f64_unorder_key(y);
      if (whole)
        a.g.tab[v][c] = y;
      else if (gl_acc[(size_t)a.cnt * slots + i] != 0)
        agg_atomic(ag, &a.g.tab[v][c], y);
    }
  }
}

// No key that varies: one group, a reduction.  Block partials part[block][v], each block's
// rows grid-strided, combined in a fixed order so the result does not depend on timing.
__global__ void __launch_bounds__(256) k_gb_reduce(GbArgs a, uint64_t n, int64_t *__restrict__ part) {
  __shared__ int64_t red[4][ALN_MAX_AGGS];
  int64_t acc[ALN_MAX_AGGS];
  for (int v = 0; v < a.nv; ++v) acc[v] = agg_identity(a.aggs[v]);
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256)
    for (int v = 0; v < a.nv; ++v)
      acc[v] = agg_combine(a.aggs[v], acc[v], a.aggs[v] == ALN_AGG_COUNT ? 1 : a.vals[v][i]);
  for (int v = 0; v < a.nv; ++v) {
    for (int o = 32; o > 0; o >>= 1)
      acc[v] = agg_combine(a.aggs[v], acc[v], (int64_t)__shfl_xor((long long)acc[v], o, 64));
    if (__lane_id() == 0) red[threadIdx.x / 64][v] = acc[v];
  }
  __syncthreads();
  if ((int)threadIdx.x < a.nv) {
    const int v = threadIdx.x;
    int64_t r = red[0][v];
    for (int w = 1; w < 4; ++w) r = agg_combine(a.aggs[v], r, red[w][v]);
    part[(uint64_t)blockIdx.x * a.nv + v] = r;
  }
}

__global__ void k_gb_reduce_final(GbArgs a, const int64_t *__restrict__ part, uint32_t nparts, GbOut o) {
  const int t = threadIdx.x;
  if (t < a.nv) {
    int64_t r = part[t];
    for (uint32_t b = 1; b < nparts; ++b) r = agg_combine(a.aggs[t], r, part[(uint64_t)b * a.nv + t]);
    o.vals[t][0] = r;
  }
  if (t < a.nk) o.keys[t][0] = a.kmin[t];
}

__global__ void k_gb_dense_init(GbArgs a, uint64_t ncodes, uint32_t *gcnt) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < ncodes; i += (uint64_t)gridDim.x * 256) {
    if (gcnt) gcnt[i] = 0;
    for (int v = 0; v < a.nv; ++v) a.tab[v][i] = agg_identity(a.aggs[v]);
  }
}

// Occupied codes as one bit each and their number per tile of 1024 codes; then their groups in
// code order straight from the tables: no flag, position or code arrays in between (4.2M codes:
// 75 -> 46 us).
constexpr uint32_t GD_TILE = 1024;
__global__ void __launch_bounds__(256) k_gd_mask(const int64_t *__restrict__ cnt64, const uint32_t *__restrict__ cnt32,
                                                 uint64_t ncodes, uint64_t *__restrict__ masks,
                                                 uint32_t *__restrict__ counts) {
  __shared__ uint32_t wc[4];
  const unsigned lane = __lane_id(), wid = threadIdx.x / 64;
  const uint64_t c0 = (uint64_t)blockIdx.x * GD_TILE + wid * 256 + lane;
  uint32_t total = 0;
  uint64_t mine = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {  // word 4 * wave + j of the tile
    const uint64_t c = c0 + 64 * j;
    const bool f = c < ncodes && (cnt64 ? cnt64[c] != 0 : cnt32[c] != 0);
    const uint64_t bal = __builtin_amdgcn_ballot_w64(f);
    total += (uint32_t)__popcll(bal);
    if (lane == (unsigned)j) mine = bal;
  }
  if (lane < 4) masks[(uint64_t)blockIdx.x * (GD_TILE / 64) + wid * 4 + lane] = mine;
  if (lane == 0) wc[wid] = total;
  __syncthreads();
  if (threadIdx.x == 0) counts[blockIdx.x] = wc[0] + wc[1] + wc[2] + wc[3];
}

// o.keys / o.vals: the groups; or (gcode) their codes and slots.
__global__ void __launch_bounds__(256) k_gd_emit(GbArgs a, GbOut o, const uint64_t *__restrict__ masks,
                                                 const uint64_t *__restrict__ offs, uint64_t *__restrict__ gcode,
                                                 uint32_t *__restrict__ gslot) {
  const unsigned lane = __lane_id(), wid = threadIdx.x / 64;
  const uint64_t word = lane < GD_TILE / 64 ? masks[(uint64_t)blockIdx.x * (GD_TILE / 64) + lane] : 0;
  const uint32_t n = (uint32_t)__popcll(word);
  uint32_t incl = n;
#pragma unroll
  for (uint32_t d = 1; d < GD_TILE / 64; d <<= 1) {
    const uint32_t y = __shfl_up(incl, d, 64);
    if (lane >= d) incl += y;
  }
  const uint32_t first = incl - n;
  const uint64_t base = offs[blockIdx.x];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int w = (int)wid * 4 + j;
    const uint64_t m = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(word >> 32), w) << 32 |
                       (uint32_t)__builtin_amdgcn_readlane((int)word, w);
    const uint64_t pos = base + (uint32_t)__builtin_amdgcn_readlane((int)first, w) + below_count(m);
    if (!(m >> lane & 1)) continue;
    const uint64_t c = (uint64_t)blockIdx.x * GD_TILE + 64 * w + lane;
    if (gcode) {
      gcode[pos] = c;
      gslot[pos] = (uint32_t)c;
      continue;
    }
    for (int k = 0; k < a.nk; ++k)
      o.keys[k][pos] = (int64_t)((uint64_t)a.kmin[k] + ((c >> a.shift[k]) & a.fmask[k]));
    for (int v = 0; v < a.nv; ++v) o.vals[v][pos] = a.tab[v][c];
  }
}

__global__ void k_gb_flags(const uint64_t *tkey, uint64_t cap, uint32_t *flag) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < cap;
       i += (uint64_t)gridDim.x * 256)
    flag[i] = tkey[i] != GB_EMPTY;
}

__global__ void k_gb_compact(const uint64_t *tkey, uint64_t cap, const uint32_t *flag,
                             const uint64_t *pos, uint64_t *gcode, uint32_t *gslot) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < cap;
       i += (uint64_t)gridDim.x * 256)
    if (flag[i]) {
      gcode[pos[i]] = tkey[i];
      gslot[pos[i]] = (uint32_t)i;
    }
}

// Decode group keys from codes, compute the merge-order hash of each group.
__global__ void k_gb_hash(GbArgs a, const uint64_t *gcode, uint64_t g, uint32_t seed,
                          uint64_t *hash) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < g;
       i += (uint64_t)gridDim.x * 256) {
    int64_t kv[ALN_MAX_KEYS];
#pragma unroll
    for (int k = 0; k < ALN_MAX_KEYS; ++k)
      kv[k] = k < a.nk ? (int64_t)((uint64_t)a.kmin[k] + ((gcode[i] >> a.shift[k]) & a.fmask[k])) : 0;
    hash[i] = murmur64a_tuple(kv, a.nk, seed);
  }
}

__global__ void k_gb_emit(GbArgs a, GbOut o, const uint64_t *gcode, const uint32_t *gslot,
                          uint64_t g) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < g;
       i += (uint64_t)gridDim.x * 256) {
    uint32_t s = gslot[i];
    for (int k = 0; k < a.nk; ++k)
      o.keys[k][i] = (int64_t)((uint64_t)a.kmin[k] + ((gcode[i] >> a.shift[k]) & a.fmask[k]));
    for (int v = 0; v < a.nv; ++v) o.vals[v][i] = a.tab[v][s];
  }
}

__global__ void k_gb_gather(const uint64_t *gc, const uint32_t *gs, const uint32_t *gi, uint64_t g,
                            uint64_t *oc, uint32_t *os) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < g;
       i += (uint64_t)gridDim.x * 256) {
    oc[i] = gc[gi[i]];
    os[i] = gs[gi[i]];
  }
}

__global__ void k_hash_rows(GbArgs a, uint64_t n, uint32_t seed, uint64_t *out) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * 256) {
    int64_t kv[ALN_MAX_KEYS];
#pragma unroll
    for (int k = 0; k < ALN_MAX_KEYS; ++k) kv[k] = k < a.nk ? a.keys[k][i] : 0;
    out[i] = murmur64a_tuple(kv, a.nk, seed);
  }
}

__global__ void k_f64_keys(const int64_t *in, uint64_t n, int back, int64_t *out) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256)
    out[i] = back ? f64_unorder_key(in[i]) : f64_order_key(in[i]);
}

// The code layout of keys in [mn, mx]: widths, masks and shifts (key 0 most significant).
// Returns the total bits (shifts are set when they fit 63).
static uint32_t gb_layout(GbArgs &a, const int64_t *mn, const int64_t *mx) {
  uint32_t bits[ALN_MAX_KEYS], total = 0;
  for (int k = 0; k < a.nk; ++k) {
    bits[k] = bits_for_range_u((uint64_t)mx[k] - (uint64_t)mn[k]);
    a.kmin[k] = mn[k];
    a.fmask[k] = bits[k] == 64 ? ~0ull : ((1ull << bits[k]) - 1);
    total += bits[k];
  }
  uint32_t sh = total;
  for (int k = 0; k < a.nk; ++k) {
    sh -= bits[k];
    a.shift[k] = total > 63 ? 0 : sh;
  }
  return total;
}

// The few-groups path for codes of `total` bits, if all accumulators fit in LDS: *taken, and
// *outside when a key lay outside the layout (nothing is valid then, and a and *cnt are as before).  With order KEYS or NONE
// the groups are written out and *done is set; else the tables stand in a.tab (a.tab[*cnt] the
// row counts).
static int gb_few(aln_ctx *c, GbArgs &a, uint64_t n, uint32_t total, int order, const GbOut &o, uint64_t cap,
                  uint64_t *h_ngroups, int *cnt, bool *taken, bool *done, bool *outside) {
  *taken = *done = *outside = false;
  GlArgs l;
  l.g = a;
  l.cnt = -1;
  for (int v = 0; v < a.nv && l.cnt < 0; ++v)
    if (a.aggs[v] == ALN_AGG_COUNT) l.cnt = v;
  if (l.cnt < 0) {
    l.cnt = l.g.nv++;
    l.g.aggs[l.cnt] = ALN_AGG_COUNT;
    l.g.vals[l.cnt] = nullptr;
  }
  if (total > 16) return ALN_OK;
  l.ncodes = 1u << total;
  const uint32_t nacc = l.ncodes * (uint32_t)l.g.nv;
  if ((size_t)nacc * 8 > GL_MOST) return ALN_OK;
  l.lr = 0;
  while (l.lr < 6 && ((size_t)nacc * 16 << l.lr) <= GL_COPIES) ++l.lr;
  const size_t lds = (size_t)nacc * 8 << l.lr;
  *taken = true;
  // as many blocks as the LDS holds on 256 CUs (5 or 2 per CU), fewer for few rows
  uint32_t nb = lds <= GL_COPIES ? 1280 : 512;
  nb = grid_for(n, 256 * GL_U, nb);
  // a block clears and stores its accumulators, so it has at least as many rows (1M rows, 4096
  // codes, two aggregates: 111 us with 488 blocks, 78 with 128)
  const uint64_t most = std::max<uint64_t>(128, n / nacc);
  if (nb > most) nb = (uint32_t)most;
  if ((uint64_t)nb * nacc > GL_PART) nb = (uint32_t)(GL_PART / nacc);
  int64_t *part, *tab;
  uint32_t *bad;
  ALN_TRY(ws(c, (size_t)nb * nacc, &part));
  ALN_TRY(ws(c, nacc, &tab));
  ALN_TRY(ws(c, 1, &bad));
  for (int v = 0; v < l.g.nv; ++v) l.g.tab[v] = tab + (size_t)v * l.ncodes;
  ALN_TRY(fill_u32(c, bad, 1, 0));
  {
    ProfScope p(c, "groupby_insert");
    hipLaunchKernelGGL(k_gl_agg, dim3(nb), dim3(256), lds, c->stream, l, n, part, bad);
    hipLaunchKernelGGL(k_gl_sum, dim3((nacc + 3) / 4), dim3(256), 0, c->stream, l, (const int64_t *)part, nb);
  }
  ALN_TRY(check_launch("gb_lds"));
  if (order != ALN_ORDER_HASH) {
    DevResult r;
    uint64_t h[2];
    ALN_TRY(result_open(c, 2, &r));
    hipLaunchKernelGGL(k_gl_emit, dim3(1), dim3(1024), 0, c->stream, l, o, a.nv, cap, (const uint32_t *)bad, r);
    ALN_TRY(check_launch("gb_lds_emit"));
    ALN_TRY(result_wait(c, r, h, 16));
    *outside = h[1] != 0;
    if (*outside) return ALN_OK;
    *h_ngroups = h[0];
    if (h[0] > cap)
      return set_error(ALN_E_CAPACITY, "aln_groupby: %llu groups, capacity %llu", (unsigned long long)h[0],
                       (unsigned long long)cap);
    *done = true;
    return ALN_OK;
  }
  uint32_t hb = 0;
  ALN_TRY(copy_to_host(c, &hb, bad, 4));
  *outside = hb != 0;
  if (*outside) return ALN_OK;
  for (int v = 0; v < l.g.nv; ++v) a.tab[v] = l.g.tab[v];
  *cnt = l.cnt;
  return ALN_OK;
}

// The route of wide key codes: sorted (by_key: for hash order all the same), or through the table
// with nb blocks; and about how many groups there are.  Rows of groups of 32 rows and more share all
// 64 bits of the hash, which the sort's buckets do not hold, and eight digit passes would follow
// instead of the code's four or five (12M rows of 4000 groups 1.96 ms by hash, 1.47 by key, of
// 250,000 groups 1.53 and 1.63).
struct GbWide {
  bool sort, by_key;
  uint32_t nb;
  double groups;
};

// From a sample (k_gb_sample).  Sorting takes about 97 us per 1M rows whatever the keys.  The table's
// time depends on the rows that miss the blocks' LDS tables: 64-way global atomics, about as dear for
// a few lanes of a wave as for many of them, dearer the larger the table, and on 5 ns for every new
// group (the count of groups is one address).  Codes come in three kinds:
//   sorted   the sample's runs rise and do not return: every run of equal codes is a group;
//   skewed   one code far more frequent than the mean: groups grow as a power of the rows, whose
//            exponent is the share of the sample's codes seen once;
//   even     from the repeats among the sample's runs.
// The constants are fitted to both routes' times over 216 inputs of 140,000 to 40M rows of 50 to
// 4M groups, uniform, Zipf 1.2 to 2.2, one hot key, sorted, and in blocks of 3, 16 and 100 rows
// (sorted / table us, the one taken marked: 1.5M rows of 1500 groups 407 / 391*, of 4000 421* / 459;
// 12M rows of 2500 groups 1460 / 1221*, of 20,000 1368* / 1623, Zipf 1.8 1749 / 842*, 600 groups in
// blocks of 16 rows 1385 / 466*, 1M sorted groups 1395* / 3557; 40M rows 99 % of one key 5109 / 1990*).
static GbWide gb_wide(uint64_t n, bool large, int order, const uint64_t *s) {
  const double rows = large ? 8192 : 2048, pairs = rows - rows / 64, m = (double)n;
  const double starts = pairs - (double)s[GW_EQUAL], heads = rows - (double)s[GW_EQUAL];
  const double found = (double)s[GW_FOUND], once = (double)s[GW_ONCE], runs = m * starts / pairs;
  const bool sorted = s[GW_RISING] == (large ? 127u : 31u) && starts < pairs / 2 && found >= starts;
  const bool skewed = !sorted && (double)s[GW_MOST] > 8 + 4 * heads / found;
  GbWide p;
  double cold = 1;  // share of the runs that miss the LDS tables
  if (sorted) {
    p.groups = runs;
  } else if (skewed) {
    p.groups = found * std::pow(std::max(runs, m / 64) / heads, once / found);
    cold = once / heads;
  } else {  // found = groups * (1 - exp(-heads / groups))
    if (heads - found <= heads / 8) {
      p.groups = heads * heads / 2 / std::max(heads - found, 0.5);
    } else {
      p.groups = found;
      for (int i = 0; i < 60; ++i) p.groups = found / (1 - std::exp(-heads / p.groups));
    }
    p.groups = std::max(1.0, std::min(p.groups, runs));
    cold = std::max(0.0, 1 - 1000 / p.groups);
  }
  p.groups = std::min(p.groups, m);
  // blocks of 8192 rows (a block adds up to 1024 groups of its LDS table to the global one at its
  // end); beyond 1024 of them only where few rows of a block miss that table, or repeat in it
  const bool more = sorted ? starts <= pairs / 512 : skewed == (starts >= pairs / 2);
  p.nb = (uint32_t)std::max<uint64_t>(256, std::min<uint64_t>(more ? 2048 : 1024, n >> 13));
  const double lanes = 64 * (runs / m + 1.0 / 64) * cold, wave = lanes < 1 ? 6 * lanes : 6 + lanes * 58 / 64;
  const double flush = p.nb * std::min(std::min(1000.0, p.groups), std::max(1.0, runs / p.nb));
  const double adds = m / 64 * wave * (skewed ? 1.5 : 1) + flush;
  const double scan = 27e-6 * m + (80e-6 + 20e-6 * std::min(1.0, 3e6 / m)) * adds * (1 + p.groups / 100e3);
  const double fresh = 5e-3 * p.groups;
  const double table = 200 + std::max(scan, fresh) + 0.8 * std::min(scan, fresh);
  // (hash order: the table's groups are sorted by hash anyway, the sorted ones as an extra step)
  p.by_key = order == ALN_ORDER_HASH && 32 * p.groups < m;
  p.sort = p.groups > 0.85 * GB_HASH_START || 270 + (p.by_key ? 70 : 0) + 97e-6 * m <= table;
  return p;
}

// Whether an output (up to m values are written) lies over an input.
static bool gb_in_place(const GbArgs &a, uint64_t n, const GbOut &o, uint64_t m) {
  auto over = [&](const int64_t *in, const int64_t *out) {
    return in && out && (uintptr_t)out < (uintptr_t)(in + n) && (uintptr_t)in < (uintptr_t)(out + m);
  };
  for (int i = 0; i < a.nk + a.nv; ++i) {
    const int64_t *out = i < a.nk ? o.keys[i] : o.vals[i - a.nk];
    for (int k = 0; k < a.nk; ++k)
      if (over(a.keys[k], out)) return true;
    for (int v = 0; v < a.nv; ++v)
      if (a.aggs[v] != ALN_AGG_COUNT && over(a.vals[v], out)) return true;
  }
  return false;
}

// The groups of direct-indexed tables in code order (row counts in gcnt, or, gcnt NULL, in
// a.tab[cv]): written out, or with order HASH their codes and slots.
static int gb_dense_groups(aln_ctx *c, const GbArgs &a, int cv, const uint32_t *gcnt, uint64_t ncodes, int order,
                           const GbOut &o, uint64_t cap, uint64_t *h_ngroups, uint64_t **gcode, uint32_t **gslot) {
  const uint32_t nt = (uint32_t)((ncodes + GD_TILE - 1) / GD_TILE);
  uint64_t *masks, *offs, g = 0;
  uint32_t *counts;
  ALN_TRY(ws(c, (size_t)nt * (GD_TILE / 64), &masks));
  ALN_TRY(ws(c, nt, &offs));
  ALN_TRY(ws(c, nt, &counts));
  hipLaunchKernelGGL(k_gd_mask, dim3(nt), dim3(256), 0, c->stream,
                     gcnt ? (const int64_t *)nullptr : (const int64_t *)a.tab[cv], gcnt, ncodes, masks, counts);
  ALN_TRY(check_launch("gb_mask"));
  ALN_TRY(exclusive_scan_u32(c, counts, nt, offs, &g));
  *h_ngroups = g;
  if (g > cap)
    return set_error(ALN_E_CAPACITY, "aln_groupby: %llu groups, capacity %llu", (unsigned long long)g,
                     (unsigned long long)cap);
  *gcode = nullptr;
  *gslot = nullptr;
  if (order == ALN_ORDER_HASH) {
    ALN_TRY(ws(c, g, gcode));
    ALN_TRY(ws(c, g, gslot));
  }
  ProfScope p(c, "groupby_emit");
  hipLaunchKernelGGL(k_gd_emit, dim3(nt), dim3(256), 0, c->stream, a, o, (const uint64_t *)masks,
                     (const uint64_t *)offs, *gcode, *gslot);
  return check_launch("gb_emit");
}

// The partitioned aggregation into a.tab (direct-indexed, initialised): *taken when the rows
// are enough, the parts' accumulators fit in LDS and the workspace holds the moved rows.
// a.tab[*cnt] gets the row counts.
static int gb_parts(aln_ctx *c, GbArgs &a, uint64_t n, uint32_t total, int *cnt, bool *taken) {
  *taken = false;
  if (n < GP_ROWS_MIN || total < GP_LOW + 6) return ALN_OK;
  GpArgs g;
  memset(&g, 0, sizeof(g));
  g.g = a;
  g.n = n;
  g.ncodes = 1u << total;
  g.cnt = -1;
  for (int v = 0; v < a.nv; ++v) {
    if (a.aggs[v] == ALN_AGG_COUNT) {
      if (g.cnt < 0) g.cnt = v;
      continue;
    }
    int k = 0;
    while (k < g.ncol && g.col[k] != a.vals[v]) ++k;
    if (k == g.ncol) g.col[g.ncol++] = a.vals[v];
    g.col_of[v] = k;
  }
  if (g.cnt < 0) {
    g.cnt = g.g.nv++;
    g.g.aggs[g.cnt] = ALN_AGG_COUNT;
  }
  // as few parts as leave two blocks per CU their accumulators (beyond 512 parts one block), but
  // a block for each CU where the codes allow it (30M rows, 60000 codes: 537 us with 64 parts,
  // 431 with 256)
  const uint64_t bytes = 8ull * g.ncodes * g.g.nv;
  uint32_t parts = GP_PARTS_MIN;
  while (parts < GP_PARTS_FEW && parts < g.ncodes >> GP_LOW) parts *= 2;
  while (parts < 512 && bytes / parts > GP_LDS) parts *= 2;
  while (parts < GP_PARTS_MAX && bytes / parts > GP_LDS_MAX) parts *= 2;
  if (bytes / parts > GP_LDS_MAX || parts > g.ncodes >> GP_LOW) return ALN_OK;
  g.lp = 31 - __builtin_clz(parts);
  if (n * (4 + 8ull * g.ncol) > GP_BYTES_MAX) return ALN_OK;
  g.ntiles = (uint32_t)((n + GP_TILE - 1) / GP_TILE);
  g.nsub = g.ntiles < 256 * GP_SUB ? 1 : GP_SUB;  // (fewer tiles: a block each, to fill the chip)
  g.nsuper = (g.ntiles + g.nsub - 1) / g.nsub;
  // a part of even shares stays whole, the part of a hot key is split among blocks (30M Zipf
  // keys: 507 us with chunks of 2n / parts and at least 32768 rows, 446 now)
  const uint64_t chunk = 5 * n / (4 * parts);
  g.chunk = (uint32_t)(chunk < 8192 ? 8192 : chunk);
  const WsMark mark = ws_mark(c);
  int r = ALN_OK;
  for (int v = 0; v < g.g.nv && r == ALN_OK; ++v) r = ws(c, g.ncodes, &g.g.tab[v]);
  const WsMark kept = ws_mark(c);  // what follows is free again when the tables are written
  if (r == ALN_OK) r = ws(c, n, &g.code);
  for (int k = 0; k < g.ncol && r == ALN_OK; ++k) r = ws(c, n, &g.moved[k]);
  if (r == ALN_OK) r = ws(c, (size_t)parts * g.nsuper, &g.cnts);
  if (r == ALN_OK) r = ws(c, (size_t)parts * g.nsuper, &g.excl);
  if (r == ALN_OK) r = ws(c, (size_t)parts * g.ntiles, &g.sub);
  if (r == ALN_OK) r = ws(c, parts, &g.tot);
  if (r == ALN_OK) r = ws(c, parts + 1, &g.start);
  if (r == ALN_OK) r = ws(c, parts + 1, &g.work);
  if (r == ALN_E_NOMEM) {  // the atomics need less
    ws_rewind(c, mark, true);
    return ALN_OK;
  }
  ALN_TRY(r);
  *taken = true;
  *cnt = g.cnt;
  for (int v = 0; v < g.g.nv; ++v) a.tab[v] = g.g.tab[v];
  const size_t lds = bytes / parts;
  if (lds > 65536)
    ALN_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k_gp_agg), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds));
  hipLaunchKernelGGL(k_gb_dense_init, dim3(grid_for(g.ncodes, 256, 65536)), dim3(256), 0, c->stream, g.g,
                     (uint64_t)g.ncodes, (uint32_t *)nullptr);
  {
    ProfScope p(c, "groupby_move");
    hipLaunchKernelGGL(k_gp_count, dim3(g.nsuper), dim3(GP_BLOCK), 0, c->stream, g);
    hipLaunchKernelGGL(k_gp_rows, dim3(parts), dim3(256), 0, c->stream, g);
    hipLaunchKernelGGL(k_gp_base, dim3(1), dim3(1024), 0, c->stream, g);
    hipLaunchKernelGGL(k_gp_move, dim3(g.ntiles), dim3(GP_BLOCK), 0, c->stream, g);
  }
  {
    ProfScope p(c, "groupby_insert");
    hipLaunchKernelGGL(k_gp_agg, dim3(parts + (uint32_t)(n / g.chunk)), dim3(1024), lds, c->stream, g);
  }
  ws_rewind(c, kept);
  return check_launch("gb_parts");
}

}  // namespace aln

using namespace aln;

extern "C" {

int aln_groupby(aln_ctx *c, const int64_t *const *d_keys, int nkeys, const int64_t *const *d_vals,
                const int32_t *aggs, int nvals, uint64_t n, int order, uint32_t seed,
                int64_t *const *d_out_keys, int64_t *const *d_out_vals, uint64_t cap,
                uint64_t *h_ngroups) {
  ALN_REQUIRE(c && h_ngroups && nkeys >= 0 && nkeys <= ALN_MAX_KEYS && (nkeys == 0 || (d_keys && d_out_keys)),
              "aln_groupby: bad key arguments");
  ALN_REQUIRE(nvals >= 0 && nvals <= ALN_MAX_AGGS && (nvals == 0 || (aggs && d_vals && d_out_vals)),
              "aln_groupby: bad aggregate arguments");
  ALN_REQUIRE(order >= ALN_ORDER_KEYS && order <= ALN_ORDER_NONE, "aln_groupby: order %d", order);
  ALN_REQUIRE(n < (1ull << 32), "aln_groupby: more than 2^32 rows");
  ws_reset(c);
  *h_ngroups = 0;
  if (n == 0) return ALN_OK;
  GbArgs a;
  memset(&a, 0, sizeof(a));
  a.nk = nkeys;
  a.nv = nvals;
  for (int k = 0; k < nkeys; ++k) {
    ALN_REQUIRE(d_keys[k], "aln_groupby: key %d is NULL", k);
    a.keys[k] = d_keys[k];
  }
  for (int v = 0; v < nvals; ++v) {
    ALN_REQUIRE(aggs[v] == ALN_AGG_COUNT || aggs[v] == ALN_AGG_SUM || aggs[v] == ALN_AGG_MIN ||
                    aggs[v] == ALN_AGG_MAX || aggs[v] == ALN_AGG_FSUM || aggs[v] == ALN_AGG_FMIN ||
                    aggs[v] == ALN_AGG_FMAX,
                "aln_groupby: aggregate %d", aggs[v]);
    ALN_REQUIRE(aggs[v] == ALN_AGG_COUNT || d_vals[v], "aln_groupby: value %d is NULL", v);
    a.vals[v] = d_vals[v];
    a.aggs[v] = aggs[v];
  }
  GbOut o;
  memset(&o, 0, sizeof(o));
  for (int k = 0; k < nkeys; ++k) o.keys[k] = d_out_keys[k];
  for (int v = 0; v < nvals; ++v) o.vals[v] = d_out_vals[v];

  // A sample's key ranges stand in for the keys' own when they are those of a few groups: the
  // rows are then checked against them as they are added up (and start again when one lies
  // outside), which saves reading the keys twice (60M rows of two keys: 0.18 of 0.76 ms).
  int64_t mn[ALN_MAX_KEYS], mx[ALN_MAX_KEYS];
  uint32_t total = 0;
  bool lds_taken = false, lds_done = false, outside = false;
  int cnt = -1;
  uint64_t wide[GW_WORDS];
  bool have_wide = false;
  static_assert(GL_SAMPLE_MIN == GB_SORT_LARGE, "one sample for both");
  if (nkeys && n >= GL_SAMPLE_MIN) {
    DevResult r;
    int64_t h[2 * ALN_MAX_KEYS + GW_WORDS];
    ALN_TRY(result_open(c, 2 * ALN_MAX_KEYS + GW_WORDS, &r));
    hipLaunchKernelGGL(k_gl_sample, dim3(1), dim3(1024), 0, c->stream, a, n, r);
    ALN_TRY(check_launch("gb_sample"));
    ALN_TRY(result_wait(c, r, h, sizeof(h)));
    for (int k = 0; k < nkeys; ++k) {
      mn[k] = h[2 * k];
      mx[k] = h[2 * k + 1];
    }
    total = gb_layout(a, mn, mx);
    have_wide = gb_wide_bits(total);
    memcpy(wide, h + 2 * ALN_MAX_KEYS, sizeof(wide));
    if (total > 0 && total <= GL_SAMPLE_BITS)
      ALN_TRY(gb_few(c, a, n, total, order, o, cap, h_ngroups, &cnt, &lds_taken, &lds_done, &outside));
    if (outside) lds_taken = lds_done = false;
  }
  if (!lds_taken) {
    if (nkeys) ALN_TRY(minmax_keys(c, a.keys, nkeys, n, mn, mx));
    total = gb_layout(a, mn, mx);
    if (total > 0)
      ALN_TRY(gb_few(c, a, n, total, order, o, cap, h_ngroups, &cnt, &lds_taken, &lds_done, &outside));
  }
  if (lds_done) return ALN_OK;
  if (total == 0) {
    // no GROUP BY, or keys that never vary: one group, a reduction (reduce, select.cu:549)
    *h_ngroups = 1;
    if (cap < 1) return set_error(ALN_E_CAPACITY, "aln_groupby: 1 group, capacity 0");
    const uint32_t nb = grid_for(n, 256 * 16, 1024);
    int64_t *part;
    ALN_TRY(ws(c, (size_t)nb * (nvals ? nvals : 1), &part));
    if (nvals) {
      ProfScope p(c, "groupby_reduce");
      hipLaunchKernelGGL(k_gb_reduce, dim3(nb), dim3(256), 0, c->stream, a, n, part);
    }
    ALN_TRY(check_launch("gb_reduce"));
    hipLaunchKernelGGL(k_gb_reduce_final, dim3(1), dim3(64), 0, c->stream, a, part, nb, o);
    ALN_TRY(check_launch("gb_reduce_final"));
    return stream_wait(c);
  }
  if (total > 63) return gb_sorted(c, a, n, total, mx, order, false, seed, o, cap, h_ngroups);
  // LDS-cached aggregation kernel: at most 2048 blocks, of at least 4 rows per thread (450,000 rows
  // into 200,000 groups: 119 us in 55 blocks of 32 rows per thread, 50 us)
  const size_t lds = gb_lds_bytes(nvals);
  const uint32_t nb = grid_for(n, 256 * 4, 2048);
  uint32_t nbh = std::min<uint32_t>(nb, 256);  // wide codes of few rows; more: gb_wide
  if (lds > 65536) {
    ALN_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k_gb_agg<true>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    ALN_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k_gb_agg<false>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  }
  uint32_t *ctl;  // [0] overflow, [1] keys inserted
  ALN_TRY(ws(c, 2, &ctl));
  uint64_t g = 0, *gcode;
  uint32_t *gslot;
  const uint64_t ncodes = 1ull << total;
  const bool dense = total <= GB_DENSE_BITS && ncodes <= std::max<uint64_t>(2 * n, (uint64_t)GB_LT);
  if (lds_taken || dense) {
    // direct-indexed accumulators: slot = code, groups come out in key order
    uint32_t *gcnt = nullptr;
    bool parts_taken = false;
    if (!lds_taken) ALN_TRY(gb_parts(c, a, n, total, &cnt, &parts_taken));
    if (!lds_taken && !parts_taken) {
      for (int v = 0; v < nvals && cnt < 0; ++v)  // a COUNT aggregate's table tells the occupied codes
        if (aggs[v] == ALN_AGG_COUNT) cnt = v;
      if (cnt < 0) ALN_TRY(ws(c, ncodes, &gcnt));
      for (int v = 0; v < nvals; ++v) ALN_TRY(ws(c, ncodes, &a.tab[v]));
      hipLaunchKernelGGL(k_gb_dense_init, dim3(grid_for(ncodes, 256, 65536)), dim3(256), 0, c->stream, a, ncodes,
                         gcnt);
      ALN_TRY(check_launch("gb_dense_init"));
      ProfScope p(c, "groupby_insert");
      hipLaunchKernelGGL(k_gb_agg<true>, dim3(nb), dim3(256), lds, c->stream, a, n, (uint64_t *)nullptr, ncodes,
                         gcnt, ctl + 1, 0xFFFFFFFFu, ctl);
      ALN_TRY(check_launch("gb_agg"));
    }
    ALN_TRY(gb_dense_groups(c, a, cnt, gcnt, ncodes, order, o, cap, h_ngroups, &gcode, &gslot));
    g = *h_ngroups;
    if (order != ALN_ORDER_HASH) {
      return stream_wait(c);
    }
  } else {
    // (In place, the table: it has read every row before a group is written.)
    if (n >= GB_SORT_MIN && !gb_in_place(a, n, o, std::min(n, cap))) {
      const bool large = n >= GB_SORT_LARGE;
      if (!have_wide) {
        DevResult r;
        ALN_TRY(result_open(c, GW_WORDS, &r));
        if (large)
          hipLaunchKernelGGL(k_gb_sample<8>, dim3(1), dim3(1024), 0, c->stream, a, n, r);
        else
          hipLaunchKernelGGL(k_gb_sample<2>, dim3(1), dim3(1024), 0, c->stream, a, n, r);
        ALN_TRY(check_launch("gb_sample"));
        ALN_TRY(result_wait(c, r, wide, sizeof(wide)));
      }
      const GbWide p = gb_wide(n, large, order, wide);
      nbh = std::min(nb, p.nb);
      if (p.sort) {
        const WsMark mark = ws_mark(c);
        const int rc = gb_sorted(c, a, n, total, mx, order, p.by_key, seed, o, cap, h_ngroups);
        if (rc != ALN_E_NOMEM) return rc;
        ws_rewind(c, mark, true);  // a table of few enough groups needs less (48 to 85 MB for 2^20)
      }
    }
    // open addressing: first a table for up to GB_HASH_START keys (half full at most); more
    // keys than that set the overflow flag and the rows are aggregated again in a table of
    // 2n slots
    const uint64_t full = next_pow2(2 * n < 1024 ? 1024 : 2 * n);
    uint64_t tcap = std::min<uint64_t>(full, next_pow2(2 * std::min<uint64_t>(n, GB_HASH_START) < 1024
                                                           ? 1024
                                                           : 2 * std::min<uint64_t>(n, GB_HASH_START)));
    uint64_t *tkey;
    uint32_t *flag;
    uint64_t *pos;
    while (true) {
      const uint32_t glimit = tcap < full ? (uint32_t)(tcap / 2) : 0xFFFFFFFFu;
      ALN_TRY(ws(c, tcap, &tkey));
      for (int v = 0; v < nvals; ++v) ALN_TRY(ws(c, tcap, &a.tab[v]));
      ALN_TRY(fill_u32(c, ctl, 2, 0));
      hipLaunchKernelGGL(k_gb_init, dim3(grid_for(tcap, 256, 65536)), dim3(256), 0, c->stream, tkey, a, tcap);
      ALN_TRY(check_launch("gb_init"));
      {
        ProfScope p(c, "groupby_insert");
        hipLaunchKernelGGL(k_gb_agg<false>, dim3(nbh), dim3(256), lds, c->stream, a, n, tkey, tcap,
                           (uint32_t *)nullptr, ctl + 1, glimit, ctl);
      }
      ALN_TRY(check_launch("gb_agg"));
      uint32_t hov = 0;
      ALN_TRY(copy_to_host(c, &hov, ctl, sizeof(uint32_t)));
      if (!hov) break;
      if (tcap >= full) return set_error(ALN_E_CAPACITY, "aln_groupby: hash table overflow");
      tcap = full;
    }
    ALN_TRY(ws(c, tcap, &flag));
    ALN_TRY(ws(c, tcap, &pos));
    hipLaunchKernelGGL(k_gb_flags, dim3(grid_for(tcap, 256, 65536)), dim3(256), 0, c->stream, tkey, tcap, flag);
    ALN_TRY(check_launch("gb_flags"));
    ALN_TRY(exclusive_scan_u32(c, flag, tcap, pos, &g));
    *h_ngroups = g;
    if (g > cap)
      return set_error(ALN_E_CAPACITY, "aln_groupby: %llu groups, capacity %llu", (unsigned long long)g,
                       (unsigned long long)cap);
    ALN_TRY(ws(c, g, &gcode));
    ALN_TRY(ws(c, g, &gslot));
    hipLaunchKernelGGL(k_gb_compact, dim3(grid_for(tcap, 256, 65536)), dim3(256), 0, c->stream, tkey, tcap, flag,
                       pos, gcode, gslot);
    ALN_TRY(check_launch("gb_compact"));
    if (order == ALN_ORDER_KEYS) ALN_TRY(radix_sort_pairs(c, gcode, gslot, g, total));
  }
  if (order == ALN_ORDER_HASH) {
    uint64_t *hash;
    ALN_TRY(ws(c, g, &hash));
    hipLaunchKernelGGL(k_gb_hash, dim3(grid_for(g, 256, 65536)), dim3(256), 0, c->stream, a, gcode,
                       g, seed, hash);
    ALN_TRY(check_launch("gb_hash"));
    // sort (hash, group index) then carry the codes along through the index
    uint32_t *gi;
    uint64_t *gcode2;
    uint32_t *gslot2;
    ALN_TRY(ws(c, g, &gi));
    ALN_TRY(ws(c, g, &gcode2));
    ALN_TRY(ws(c, g, &gslot2));
    ALN_TRY(iota_u32(c, gi, g));
    ALN_TRY(radix_sort_pairs(c, hash, gi, g, 64));
    hipLaunchKernelGGL(k_gb_gather, dim3(grid_for(g, 256, 65536)), dim3(256), 0, c->stream, gcode,
                       gslot, gi, g, gcode2, gslot2);
    ALN_TRY(check_launch("gb_gather"));
    gcode = gcode2;
    gslot = gslot2;
  }
  {
    ProfScope p(c, "groupby_emit");
    hipLaunchKernelGGL(k_gb_emit, dim3(grid_for(g, 256, 65536)), dim3(256), 0, c->stream, a, o,
                       gcode, gslot, g);
  }
  ALN_TRY(check_launch("gb_emit"));
  return stream_wait(c);
}

int aln_f64_order_keys(aln_ctx *c, const int64_t *d_in, uint64_t n, int64_t *d_out) {
  ALN_REQUIRE(c && (n == 0 || (d_in && d_out)), "aln_f64_order_keys: bad arguments");
  if (n == 0) return ALN_OK;
  hipLaunchKernelGGL(k_f64_keys, dim3(grid_for(n, 256, 65536)), dim3(256), 0, c->stream, d_in, n, 0, d_out);
  return check_launch("f64_order_keys");
}

int aln_f64_unorder_keys(aln_ctx *c, const int64_t *d_in, uint64_t n, int64_t *d_out) {
  ALN_REQUIRE(c && (n == 0 || (d_in && d_out)), "aln_f64_unorder_keys: bad arguments");
  if (n == 0) return ALN_OK;
  hipLaunchKernelGGL(k_f64_keys, dim3(grid_for(n, 256, 65536)), dim3(256), 0, c->stream, d_in, n, 1, d_out);
  return check_launch("f64_unorder_keys");
}

int aln_hash_rows(aln_ctx *c, const int64_t *const *d_keys, int nkeys, uint64_t n, uint32_t seed,
                  uint64_t *d_out) {
  ALN_REQUIRE(c && d_keys && nkeys >= 1 && nkeys <= ALN_MAX_KEYS && (n == 0 || d_out),
              "aln_hash_rows: bad arguments");
  if (n == 0) return ALN_OK;
  GbArgs a;
  memset(&a, 0, sizeof(a));
  a.nk = nkeys;
  for (int k = 0; k < nkeys; ++k) a.keys[k] = d_keys[k];
  hipLaunchKernelGGL(k_hash_rows, dim3(grid_for(n, 256, 65536)), dim3(256), 0, c->stream, a, n, seed,
                     d_out);
  return check_launch("hash_rows");
}

}  // extern "C"
