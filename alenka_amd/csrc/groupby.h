// What the GROUP BY paths share: the call's keys, aggregates and outputs, and the aggregates'
// identities and combinations.
#pragma once

#include "aln_internal.h"

namespace aln {

struct GbArgs {
  const int64_t *keys[ALN_MAX_KEYS];
  int64_t kmin[ALN_MAX_KEYS];
  uint32_t shift[ALN_MAX_KEYS];
  uint64_t fmask[ALN_MAX_KEYS];
  // one more than a call can ask for: the few-groups path counts rows by itself
  const int64_t *vals[ALN_MAX_AGGS + 1];
  int32_t aggs[ALN_MAX_AGGS + 1];
  int64_t *tab[ALN_MAX_AGGS + 1];
  int nk, nv;
};

__device__ __forceinline__ int64_t agg_combine(int a, int64_t x, int64_t y) {
  if (a == ALN_AGG_MIN) return x < y ? x : y;
  if (a == ALN_AGG_MAX) return x > y ? x : y;
  if (a == ALN_AGG_FSUM) return f64_bits(bits_f64(x) + bits_f64(y));
  if (a == ALN_AGG_FMIN) return bits_f64(y) < bits_f64(x) ? y : x;
  if (a == ALN_AGG_FMAX) return bits_f64(y) > bits_f64(x) ? y : x;
  return (int64_t)((uint64_t)x + (uint64_t)y);  // SUM, COUNT
}

// The starting value of an aggregate's accumulator.
__host__ __device__ __forceinline__ int64_t agg_identity(int a) {
  switch (a) {
    case ALN_AGG_MIN: return INT64_MAX;
    case ALN_AGG_MAX: return INT64_MIN;
    case ALN_AGG_FMIN: return 0x7FF0000000000000ll;                // +inf
    case ALN_AGG_FMAX: return (int64_t)0xFFF0000000000000ull;      // -inf
    default: return 0;                                             // 0, 0.0
  }
}

// Adds x into the accumulator at t.
__device__ __forceinline__ void agg_atomic(int a, int64_t *t, int64_t x) {
  if (a == ALN_AGG_MIN) {
    atomicMin((long long *)t, (long long)x);
  } else if (a == ALN_AGG_MAX) {
    atomicMax((long long *)t, (long long)x);
  } else if (a == ALN_AGG_FSUM) {
    atomicAdd(reinterpret_cast<double *>(t), bits_f64(x));
  } else if (a == ALN_AGG_FMIN || a == ALN_AGG_FMAX) {
    unsigned long long *p = reinterpret_cast<unsigned long long *>(t);
    unsigned long long old = *p, assumed;
    do {
      assumed = old;
      const int64_t nv = agg_combine(a, (int64_t)assumed, x);
      if (nv == (int64_t)assumed) break;
      old = atomicCAS(p, assumed, (unsigned long long)nv);
    } while (old != assumed);
  } else {
    atomicAdd((unsigned long long *)t, (unsigned long long)x);
  }
}

// MurmurHash64A of nk int64 values laid out contiguously (v holds ALN_MAX_KEYS, unrolled so that they
// stay in registers): the merge order of every route.
__device__ __forceinline__ uint64_t murmur64a_tuple(const int64_t *v, int nk, uint32_t seed) {
  const uint64_t m = 0xc6a4a7935bd1e995ULL;
  uint64_t h = (uint64_t)seed ^ ((uint64_t)(8 * nk) * m);
#pragma unroll
  for (int i = 0; i < ALN_MAX_KEYS; ++i) {
    if (i >= nk) break;
    uint64_t k = (uint64_t)v[i];
    k *= m;
    k ^= k >> 47;
    k *= m;
    h ^= k;
    h *= m;
  }
  h ^= h >> 47;
  h *= m;
  h ^= h >> 47;
  return h;
}

struct GbOut {
  int64_t *keys[ALN_MAX_KEYS];
  int64_t *vals[ALN_MAX_AGGS];
};

// Groups by sorting the rows (groupsort.hip): packed codes of `total` bits, or, above 63 bits, key
// tuples.  Writes the groups in the order asked for.
// kmax: the keys' largest values (the smallest are in a).  by_key: for hash order, sort the rows by
// key all the same and then the groups by hash.
int gb_sorted(aln_ctx *c, const GbArgs &a, uint64_t n, uint32_t total, const int64_t *kmax, int order, bool by_key,
              uint32_t seed, const GbOut &o, uint64_t cap, uint64_t *h_ngroups);

}  // namespace aln
