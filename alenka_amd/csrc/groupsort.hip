// GROUP BY by sorting, the reference's own scheme (stable sort, run heads, segmented reduce,
// operators.cu:367-406, cm.cu:910-956, select.cu:481-580), for many groups of wide keys:
//   * the rows' keys and distinct value columns are packed side by side, because what follows
//     reads whole rows in sorted order and a random read costs the same for 8 bytes as for 32
//     (50 G/s): one read per row instead of one per column;
//   * the rows are ordered by one 64-bit code: the packed key code (key order), or the tuple's
//     MurmurHash64A (the multi-segment merge order, merge.cu:138-203, which needs no second sort
//     then; codes of 63 bits of few groups are sorted by key and the groups by hash), or, for key
//     tuples wider than 63 bits in key order, by the keys themselves;
//   * a wave takes 1024 sorted rows, 64 at a time, combines the runs with a segmented scan,
//     carries the open run to the next 64 rows and stores each group when its run ends; only
//     runs that cross waves are combined with atomics.
// Two tuples of one hash would be neighbours with equal codes: the reduction compares their keys,
// and the call starts again in key order with a sort of the groups by hash.
// 12M rows of 12M groups of two sparse keys, three aggregates, hash order: 5.50 -> 0.96 ms
// (two sorts of all rows, a gather per column, atomics per row and value, a permutation per
// output before).
#include <string.h>

#include "groupby.h"

namespace aln {

constexpr int GS_BLOCK = 256;
constexpr uint32_t GS_TILE = 4096;  // rows of a block: 4 waves x 16 words of 64
constexpr int GS_MAX_WORDS = ALN_MAX_KEYS + ALN_MAX_AGGS;

struct GsArgs {
  GbArgs g;
  uint64_t n;
  int nkw;       // key words of a row: the packed code, or the keys
  int ncol;      // distinct value columns
  int stride;    // 8-byte words from packed row to packed row (even)
  bool coded;    // the key word is the packed code
  bool verify;   // equal codes may be different tuples
  const int64_t *col[ALN_MAX_AGGS];
  int32_t col_of[ALN_MAX_AGGS];  // value column of an aggregate, -1 for COUNT
  const int64_t *row;            // the packed rows, or NULL: read from the columns
  const uint64_t *code;          // the code of every row (coded: the key word, when not packed)
  const uint32_t *perm;
  const uint64_t *masks;  // head bits of 64 sorted rows each
  const uint64_t *offs;   // groups that start before a tile
  uint32_t *clash;
};

// The code of every row (NULL: not wanted): the tuple's hash, or the packed key code; and the
// packed rows (NULL: not wanted).
__global__ void __launch_bounds__(GS_BLOCK) k_gs_pack(GsArgs a, int hashed, uint32_t seed, uint64_t *__restrict__ code,
                                                      int64_t *__restrict__ row) {
  const uint64_t i = (uint64_t)blockIdx.x * GS_BLOCK + threadIdx.x;
  if (i >= a.n) return;
  int64_t kv[ALN_MAX_KEYS];
  uint64_t packed = 0;
#pragma unroll
  for (int k = 0; k < ALN_MAX_KEYS; ++k) {
    kv[k] = k < a.g.nk ? __builtin_nontemporal_load(a.g.keys[k] + i) : 0;
    if (k < a.g.nk) packed |= (((uint64_t)kv[k] - (uint64_t)a.g.kmin[k]) & a.g.fmask[k]) << a.g.shift[k];
  }
  if (code) code[i] = hashed ? murmur64a_tuple(kv, a.g.nk, seed) : packed;
  if (!row) return;
  int64_t w[GS_MAX_WORDS];
#pragma unroll
  for (int j = 0; j < GS_MAX_WORDS; ++j) w[j] = 0;
  if (a.coded) {
    w[0] = (int64_t)packed;
  } else {
#pragma unroll
    for (int k = 0; k < ALN_MAX_KEYS; ++k) w[k] = kv[k];
  }
#pragma unroll
  for (int j = 1; j < GS_MAX_WORDS; ++j)
    if (j >= a.nkw && j < a.nkw + a.ncol) w[j] = __builtin_nontemporal_load(a.col[j - a.nkw] + i);
  int64_t *dst = row + i * a.stride;
#pragma unroll
  for (int j = 0; j < GS_MAX_WORDS; j += 2)
    if (j < a.stride) *reinterpret_cast<longlong2 *>(dst + j) = make_longlong2(w[j], w[j + 1]);
}

// Key word k of a row.
__device__ __forceinline__ int64_t gs_key_word(const GsArgs &a, uint32_t r, int k) {
  if (a.row) return a.row[(uint64_t)r * a.stride + k];
  return a.coded ? (int64_t)a.code[r] : a.g.keys[k][r];
}

// Head flags of sorted rows from their key words (sorts that do not give them).
__global__ void __launch_bounds__(GS_BLOCK) k_gs_heads(GsArgs a, const uint64_t *__restrict__ code,
                                                       uint8_t *__restrict__ heads) {
  const uint64_t i = (uint64_t)blockIdx.x * GS_BLOCK + threadIdx.x;
  if (i >= a.n) return;
  const uint32_t r = a.perm[i], p = a.perm[i ? i - 1 : 0];
  bool h = i == 0;
  if (code) {
    h = h || code[r] != code[p];
  } else {
    for (int k = 0; k < a.nkw; ++k) h = h || gs_key_word(a, r, k) != gs_key_word(a, p, k);
  }
  heads[i] = h;
}

// Head bits of each 64 rows and their number per tile.
__global__ void __launch_bounds__(GS_BLOCK) k_gs_mask(const uint8_t *__restrict__ heads, uint64_t n,
                                                      uint64_t *__restrict__ masks, uint32_t *__restrict__ counts) {
  __shared__ uint32_t wc[4];
  const unsigned lane = __lane_id(), wid = threadIdx.x / 64;
  const uint64_t i0 = (uint64_t)blockIdx.x * GS_TILE + wid * 1024 + lane;
  uint8_t h[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) h[j] = i0 + 64 * j < n ? heads[i0 + 64 * j] : 0;
  uint64_t mine = 0;
  uint32_t total = 0;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const uint64_t b = __builtin_amdgcn_ballot_w64(h[j] != 0);
    total += (uint32_t)__popcll(b);
    if (lane == (unsigned)j) mine = b;
  }
  if (lane < 16) masks[(uint64_t)blockIdx.x * (GS_TILE / 64) + wid * 16 + lane] = mine;
  if (lane == 0) wc[wid] = total;
  __syncthreads();
  if (threadIdx.x == 0) counts[blockIdx.x] = wc[0] + wc[1] + wc[2] + wc[3];
}

// Groups whose run crosses into a wave's rows: combined with atomics, so their outputs start
// from the identity (one thread per 1024 rows; a run over several waves is set several times,
// to the same value).
__global__ void __launch_bounds__(64) k_gs_open(GsArgs a, GbOut o) {
  const uint64_t chunk = (uint64_t)blockIdx.x * 64 + threadIdx.x;
  if (chunk * 1024 >= a.n || (a.masks[chunk * 16] & 1)) return;
  uint64_t g = a.offs[chunk / 4];
  for (uint64_t w = chunk / 4 * 64; w < chunk * 16; ++w) g += (uint64_t)__popcll(a.masks[w]);
  for (int v = 0; v < a.g.nv; ++v) o.vals[v][g - 1] = agg_identity(a.g.aggs[v]);
}

// The runs of 1024 sorted rows per wave.  WP: 16-byte words of a packed row (0: read from the
// columns).
template <int WP>
__global__ void __launch_bounds__(GS_BLOCK) k_gs_reduce(GsArgs a, GbOut o) {
  constexpr int W = WP ? 2 * WP : GS_MAX_WORDS;
  constexpr int U = WP && WP <= 2 ? 4 : WP && WP <= 4 ? 2 : 1;  // words of 64 rows in flight
  __shared__ int64_t carry_lds[GS_BLOCK / 64][ALN_MAX_AGGS];
  const unsigned lane = __lane_id(), wid = threadIdx.x / 64;
  // the open run's values between two words: written by lane 63, read by the lanes of its run
  // (volatile: no lane's own view of them is kept in registers)
  volatile int64_t *carry = carry_lds[wid];
  const uint64_t chunk = (uint64_t)blockIdx.x * 4 + wid, i0 = chunk * 1024;
  if (i0 >= a.n) return;
  const uint64_t word = a.masks[(uint64_t)blockIdx.x * (GS_TILE / 64) + lane];
  uint32_t pc = (uint32_t)__popcll(word);
  const uint32_t own = pc;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(pc, d, 64);
    if (lane >= (unsigned)d) pc += y;
  }
  pc -= own;  // groups of the tile that start before the lane's word
  const uint64_t gtile = a.offs[blockIdx.x];
  const uint64_t gfirst = gtile + (uint32_t)__builtin_amdgcn_readlane((int)pc, (int)wid * 16);
  // does the row after the wave's last start a group?
  const uint64_t iend = i0 + 1024;
  const bool next_head = iend >= a.n || (a.masks[iend / 64] & 1);
  int64_t prev_key[ALN_MAX_KEYS] = {0, 0, 0, 0};  // key words of the row before (verify)
  if (a.verify && i0 > 0) {
    const uint32_t r = a.perm[i0 - 1];
#pragma unroll
    for (int k = 0; k < ALN_MAX_KEYS; ++k)
      if (k < a.nkw) prev_key[k] = gs_key_word(a, r, k);
  }
  bool clash = false;
#pragma unroll 1
  for (int s = 0; s < 16; s += U) {
    if (i0 + 64 * s >= a.n) break;
    int64_t x[U][W];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint64_t i = i0 + 64 * (s + u) + lane;
      const uint32_t r = a.perm[i < a.n ? i : a.n - 1];
      if constexpr (WP != 0) {
        const longlong2 *p = reinterpret_cast<const longlong2 *>(a.row + (uint64_t)r * (2 * WP));
#pragma unroll
        for (int w = 0; w < WP; ++w) {
          const longlong2 q = p[w];
          x[u][2 * w] = q.x;
          x[u][2 * w + 1] = q.y;
        }
      } else {
#pragma unroll
        for (int w = 0; w < W; ++w) {
          x[u][w] = 0;
          if (w < a.nkw)
            x[u][w] = a.coded ? (int64_t)a.code[r] : a.g.keys[w < ALN_MAX_KEYS ? w : 0][r];
          else if (w < a.nkw + a.ncol)
            x[u][w] = a.col[w - a.nkw][r];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int w64 = (int)wid * 16 + s + u;
      const uint64_t i = i0 + 64 * (s + u) + lane;
      if (i0 + 64 * (s + u) >= a.n) break;
      const bool in = i < a.n;
      const uint64_t m = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(word >> 32), w64) << 32 |
                         (uint32_t)__builtin_amdgcn_readlane((int)word, w64);
      const uint64_t gword = gtile + (uint32_t)__builtin_amdgcn_readlane((int)pc, w64);
      const bool head = m >> lane & 1;
      const uint64_t upto = m & (lane == 63 ? ~0ull : (2ull << lane) - 1);  // heads at or below the lane
      const uint64_t gi = gword + (uint64_t)__popcll(upto) - 1;
      const int start = upto ? 63 - __builtin_clzll(upto) : -1;  // -1: the run came from before
      const int below = (int)lane - (start < 0 ? 0 : start);     // lanes of the run below this one
      // the last lane of a run in this word; at lane 63 (or the last row) the run goes on unless
      // the next row is a head
      bool next;
      if (s + u < 15)
        next = w64 < 63 && (__builtin_amdgcn_readlane((int)word, w64 < 63 ? w64 + 1 : 63) & 1);
      else
        next = next_head;
      const bool last_row = i + 1 >= a.n;
      const bool ends = in && (last_row || (lane == 63 ? next : (m >> (lane + 1) & 1) != 0));
      const bool leaves = in && lane == 63 && s + u == 15 && !ends;  // open at the wave's end
      const bool open = gi + 1 == gfirst;                            // began before the wave's rows
      const uint64_t longest = __builtin_amdgcn_ballot_w64(below > 0);
      if (head && in) {
        if (a.coded) {
          const uint64_t c = (uint64_t)x[u][0];
          for (int k = 0; k < a.g.nk; ++k)
            o.keys[k][gi] = (int64_t)((uint64_t)a.g.kmin[k] + ((c >> a.g.shift[k]) & a.g.fmask[k]));
        } else {
#pragma unroll
          for (int k = 0; k < ALN_MAX_KEYS; ++k)
            if (k < a.g.nk && k < W) o.keys[k][gi] = x[u][k];
        }
      }
      if (a.verify) {
#pragma unroll
        for (int k = 0; k < ALN_MAX_KEYS; ++k) {
          if (k >= a.nkw || k >= W) break;
          int64_t p = __shfl_up((long long)x[u][k], 1, 64);
          if (lane == 0) p = prev_key[k];
          clash = clash || (in && !head && p != x[u][k]);
          prev_key[k] = __shfl((long long)x[u][k], 63, 64);
        }
      }
      // one aggregate of the word's rows: y = the lane's value
      auto reduce = [&](int v, int64_t y) {
        const int ag = a.g.aggs[v];
        if ((ag == ALN_AGG_FMIN || ag == ALN_AGG_FMAX) && bits_f64(y) != bits_f64(y)) y = agg_identity(ag);
        if (longest) {
#pragma unroll
          for (int d = 1; d < 64; d <<= 1) {
            if (!__builtin_amdgcn_ballot_w64(below >= d)) break;
            const int64_t z = __shfl_up((long long)y, d, 64);
            if (below >= d) y = agg_combine(ag, z, y);
          }
        }
        if (start < 0 && s + u > 0) y = agg_combine(ag, carry[v], y);
        if (ends || leaves) {
          if (open || leaves)
            agg_atomic(ag, &o.vals[v][gi], y);
          else
            o.vals[v][gi] = y;
        }
        if (lane == 63) carry[v] = y;
      };
      for (int v = 0; v < a.g.nv; ++v)
        if (a.col_of[v] < 0) reduce(v, in ? 1 : 0);
#pragma unroll
      for (int w = 1; w < W; ++w) {
        if (w < a.nkw || w >= a.nkw + a.ncol) continue;
        for (int v = 0; v < a.g.nv; ++v)
          if (a.col_of[v] == w - a.nkw) reduce(v, x[u][w]);
      }
    }
  }
  if (clash) *a.clash = 1;
}

// The groups in the order of their tuples' hashes (after a clash).
__global__ void __launch_bounds__(GS_BLOCK) k_gs_group_hash(GbOut o, int nk, uint64_t g, uint32_t seed,
                                                            uint64_t *__restrict__ hash) {
  const uint64_t i = (uint64_t)blockIdx.x * GS_BLOCK + threadIdx.x;
  if (i >= g) return;
  int64_t kv[ALN_MAX_KEYS];
#pragma unroll
  for (int k = 0; k < ALN_MAX_KEYS; ++k) kv[k] = k < nk ? o.keys[k][i] : 0;
  hash[i] = murmur64a_tuple(kv, nk, seed);
}
__global__ void __launch_bounds__(GS_BLOCK) k_gs_permute(const int64_t *__restrict__ in,
                                                         const uint32_t *__restrict__ perm, uint64_t n,
                                                         int64_t *__restrict__ out) {
  const uint64_t i = (uint64_t)blockIdx.x * GS_BLOCK + threadIdx.x;
  if (i < n) out[i] = in[perm[i]];
}

static int gs_by_hash(aln_ctx *c, const GbArgs &a, const GbOut &o, uint64_t g, uint32_t seed) {
  if (g < 2) return ALN_OK;
  uint64_t *hash;
  uint32_t *idx;
  int64_t *tmp;
  bool heads;
  ALN_TRY(ws(c, g, &hash));
  ALN_TRY(ws(c, g, &idx));
  ALN_TRY(ws(c, g, &tmp));
  const dim3 grid(grid_for(g, GS_BLOCK));
  hipLaunchKernelGGL(k_gs_group_hash, grid, dim3(GS_BLOCK), 0, c->stream, o, a.nk, g, seed, hash);
  ALN_TRY(check_launch("gb_group_hash"));
  ALN_TRY(sort_codes(c, hash, g, 64, idx, nullptr, &heads));
  for (int q = 0; q < a.nk + a.nv; ++q) {
    int64_t *col = q < a.nk ? o.keys[q] : o.vals[q - a.nk];
    hipLaunchKernelGGL(k_gs_permute, grid, dim3(GS_BLOCK), 0, c->stream, (const int64_t *)col, (const uint32_t *)idx, g,
                       tmp);
    ALN_TRY(check_launch("gb_permute"));
    ALN_HIP(hipMemcpyAsync(col, tmp, 8 * g, hipMemcpyDeviceToDevice, c->stream));
  }
  return ALN_OK;
}

// One sort and reduction.  hashed: by the tuples' hashes (*clash: two tuples share one, and the
// outputs are void); else in key order.  pack: with packed rows.
static int gs_run(aln_ctx *c, const GbArgs &g, uint64_t n, uint32_t total, const int64_t *kmax, bool hashed,
                  bool pack, uint32_t seed, const GbOut &o, uint64_t cap, uint64_t *h_ngroups, bool *clash) {
  *clash = false;
  GsArgs a;
  memset(&a, 0, sizeof(a));
  a.g = g;
  a.n = n;
  a.coded = total <= 63;
  a.verify = hashed;
  a.nkw = a.coded ? 1 : g.nk;
  for (int v = 0; v < g.nv; ++v) {
    a.col_of[v] = -1;
    if (g.aggs[v] == ALN_AGG_COUNT) continue;
    int k = 0;
    while (k < a.ncol && a.col[k] != g.vals[v]) ++k;
    if (k == a.ncol) a.col[a.ncol++] = g.vals[v];
    a.col_of[v] = k;
  }
  a.stride = (a.nkw + a.ncol + 1) & ~1;
  // codes, packed rows, order
  const bool coded_sort = hashed || a.coded;
  uint64_t *code = nullptr;
  int64_t *row = nullptr;
  uint32_t *perm;
  uint8_t *heads;
  if (coded_sort || a.coded) ALN_TRY(ws(c, n, &code));
  ALN_TRY(ws(c, n, &perm));
  ALN_TRY(ws(c, n, &heads));
  if (pack) ALN_TRY(ws(c, n * a.stride, &row));
  const dim3 rows(grid_for(n, GS_BLOCK));
  if (code || row) {
    ProfScope p(c, "groupby_pack");
    hipLaunchKernelGGL(k_gs_pack, rows, dim3(GS_BLOCK), 0, c->stream, a, hashed ? 1 : 0, seed, code, row);
  }
  ALN_TRY(check_launch("gb_pack"));
  bool have_heads = false;
  if (coded_sort)
    ALN_TRY(sort_codes(c, code, n, hashed ? 64 : total, perm, heads, &have_heads));
  else
    ALN_TRY(sort_keys_ranged(c, g.keys, g.nk, n, g.kmin, kmax, perm));
  a.row = row;
  a.code = code;
  a.perm = perm;
  if (!have_heads) {
    hipLaunchKernelGGL(k_gs_heads, rows, dim3(GS_BLOCK), 0, c->stream, a,
                       coded_sort ? (const uint64_t *)code : (const uint64_t *)nullptr, heads);
    ALN_TRY(check_launch("gb_heads"));
  }
  if (!row && a.coded && hashed) {  // the key words are read from the codes: the packed ones now
    hipLaunchKernelGGL(k_gs_pack, rows, dim3(GS_BLOCK), 0, c->stream, a, 0, seed, code, (int64_t *)nullptr);
    ALN_TRY(check_launch("gb_pack"));
  }
  const uint64_t nt = (n + GS_TILE - 1) / GS_TILE;
  uint64_t *masks, *offs, ng = 0;
  uint32_t *counts, *flag;
  ALN_TRY(ws(c, nt * (GS_TILE / 64) + 1, &masks));
  ALN_TRY(ws(c, nt, &offs));
  ALN_TRY(ws(c, nt, &counts));
  ALN_TRY(ws(c, 1, &flag));
  ALN_TRY(fill_u32(c, flag, 1, 0));
  hipLaunchKernelGGL(k_gs_mask, dim3((unsigned)nt), dim3(GS_BLOCK), 0, c->stream, (const uint8_t *)heads, n, masks,
                     counts);
  ALN_TRY(check_launch("gb_mask"));
  ALN_TRY(exclusive_scan_u32(c, counts, nt, offs, &ng));
  *h_ngroups = ng;
  if (ng > cap && !hashed)
    return set_error(ALN_E_CAPACITY, "aln_groupby: %llu groups, capacity %llu", (unsigned long long)ng,
                     (unsigned long long)cap);
  if (ng > cap) {
    *clash = true;  // tuples of one hash count once here: the number needed, in key order
    return ALN_OK;
  }
  a.masks = masks;
  a.offs = offs;
  a.clash = flag;
  hipLaunchKernelGGL(k_gs_open, dim3((unsigned)((n + 65535) / 65536)), dim3(64), 0, c->stream, a, o);
  ALN_TRY(check_launch("gb_open"));
  {
    ProfScope p(c, "groupby_sorted_agg");
    const dim3 grid((unsigned)nt);
#define GS_CASE(wp)                                                                            \
  case wp:                                                                                     \
    hipLaunchKernelGGL(k_gs_reduce<wp>, grid, dim3(GS_BLOCK), 0, c->stream, a, o);             \
    break
    switch (row ? a.stride / 2 : 0) {
      GS_CASE(1);
      GS_CASE(2);
      GS_CASE(3);
      GS_CASE(4);
      GS_CASE(5);
      GS_CASE(6);
      default:
        hipLaunchKernelGGL(k_gs_reduce<0>, grid, dim3(GS_BLOCK), 0, c->stream, a, o);
    }
#undef GS_CASE
  }
  ALN_TRY(check_launch("gb_sorted_agg"));
  if (hashed) {
    uint32_t h = 0;
    ALN_TRY(copy_to_host(c, &h, flag, 4));
    *clash = h != 0;
  }
  return ALN_OK;
}

// gs_run with packed rows where the workspace holds them beside the sort's buffers (53 bytes a row
// for one value column), else without (37).
static int gs_fit(aln_ctx *c, const GbArgs &a, uint64_t n, uint32_t total, const int64_t *kmax, bool hashed,
                  uint32_t seed, const GbOut &o, uint64_t cap, uint64_t *h_ngroups, bool *clash) {
  const WsMark mark = ws_mark(c);
  const int r = gs_run(c, a, n, total, kmax, hashed, true, seed, o, cap, h_ngroups, clash);
  if (r != ALN_E_NOMEM) return r;
  ws_rewind(c, mark, true);
  return gs_run(c, a, n, total, kmax, hashed, false, seed, o, cap, h_ngroups, clash);
}

int gb_sorted(aln_ctx *c, const GbArgs &a, uint64_t n, uint32_t total, const int64_t *kmax, int order, bool by_key,
              uint32_t seed, const GbOut &o, uint64_t cap, uint64_t *h_ngroups) {
  bool clash = false;
  const WsMark mark = ws_mark(c);
  if (order == ALN_ORDER_HASH && !by_key) {
    ALN_TRY(gs_fit(c, a, n, total, kmax, true, seed, o, cap, h_ngroups, &clash));
    if (!clash) {
      return stream_wait(c);
    }
    ws_rewind(c, mark);
  }
  ALN_TRY(gs_fit(c, a, n, total, kmax, false, seed, o, cap, h_ngroups, &clash));
  if (order == ALN_ORDER_HASH) {
    ws_rewind(c, mark);  // the groups are in the outputs
    ALN_TRY(gs_by_hash(c, a, o, *h_ngroups, seed));
  }
  return stream_wait(c);
}

}  // namespace aln
