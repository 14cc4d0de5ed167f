// Device interpreter of compiled RPN programs (aln_insn) and the unpacking of column codes for
// the kernels that run over rows.
#pragma once

#include <string.h>

#include "aln_internal.h"

namespace aln {

constexpr int VM_BLOCK = 256;

struct ColTable {
  const uint32_t *words[ALN_MAX_COLS];
  const aln_seg *segs[ALN_MAX_COLS];
};

__device__ __forceinline__ int64_t vm_div(int64_t l, int64_t r) {
  if (r == 0) return 0;
  if (l == INT64_MIN && r == -1) return INT64_MIN;
  return l / r;
}

// The program as the row kernels run it: U rows per thread and instruction, so that fetching
// and dispatching an instruction (uniform: scalar loads and branches) is paid once per U rows;
// the top of the stack in registers, only the values below it in LDS; and a constant or a
// column that is the right operand taken by the operation itself (five of the nine pushes of
// (date < d AND disc != 5) OR price * (100 - disc) > x need no stack).  Passed by value, so it
// reaches the kernel with the launch.
enum {
  V_COL = 1,   // push column a * k
  V_CONST = 2, // push k
  V_IMM = 3,   // top = top op k
  V_COLOP = 4, // top = top op (column a * k)
  V_STK = 5,   // top = (value below) op top
  V_INSET = 6, // as ALN_I_INSET
  V_I2F = 7    // as ALN_I_I2F
};
struct VInsn {
  uint8_t kind, op, cmp;  // op: the ALN_I_* operation of V_IMM, V_COLOP, V_STK; cmp: its comparison
  uint8_t spill;          // a push that moves the old top to LDS
  int32_t a;
  int64_t k;
  uint64_t m;  // V_IMM ALN_I_DIV: ceil(2^64 / k) for k in [2, 2^32), else 0
};
struct VProg {
  VInsn ins[ALN_MAX_INSN];
  int n;
  int slots;  // values below the top at the deepest point
};

// Lowers a checked program.
inline void vm_lower(const aln_insn *p, int n, VProg *out) {
  memset(out, 0, sizeof(*out));
  int depth = 0;
  auto binary = [](int op) { return op != ALN_I_COL && op != ALN_I_CONST && op != ALN_I_INSET && op != ALN_I_I2F; };
  for (int i = 0; i < n; ++i) {
    VInsn &v = out->ins[out->n++];
    if (p[i].op == ALN_I_COL || p[i].op == ALN_I_CONST) {
      const bool col = p[i].op == ALN_I_COL;
      v.a = col ? p[i].a : 0;
      v.k = p[i].k;
      if (depth >= 1 && i + 1 < n && binary(p[i + 1].op)) {
        v.kind = col ? V_COLOP : V_IMM;
        v.op = (uint8_t)p[i + 1].op;
        v.cmp = (uint8_t)p[i + 1].a;
        if (!col && v.op == ALN_I_DIV && v.k >= 2 && v.k < (1ll << 32)) v.m = ~0ull / (uint64_t)v.k + 1;
        ++i;
      } else {
        v.kind = col ? V_COL : V_CONST;
        v.spill = depth >= 1;
        ++depth;
        if (depth - 1 > out->slots) out->slots = depth - 1;
      }
    } else if (p[i].op == ALN_I_INSET || p[i].op == ALN_I_I2F) {
      v.kind = p[i].op == ALN_I_INSET ? V_INSET : V_I2F;
      v.a = p[i].a;
      v.k = p[i].k;
    } else {
      v.kind = V_STK;
      v.op = (uint8_t)p[i].op;
      v.cmp = (uint8_t)p[i].a;
      --depth;
    }
  }
}

// o[u] = l[u] op r(u), the operation wave-uniform.
template <int U, typename R>
__device__ __forceinline__ void vm_binary(int op, int cmp, const int64_t (&l)[U], R r, int64_t (&o)[U]) {
#define VM_EACH(expr)                  \
  _Pragma("unroll") for (int u = 0; u < U; ++u) { \
    const int64_t x = l[u], y = r(u);  \
    o[u] = (expr);                     \
  }                                    \
  break
  switch (op) {
    case ALN_I_ADD: VM_EACH((int64_t)((uint64_t)x + (uint64_t)y));
    case ALN_I_SUB: VM_EACH((int64_t)((uint64_t)x - (uint64_t)y));
    case ALN_I_MUL: VM_EACH(wmul(x, y));
    case ALN_I_DIV: VM_EACH(vm_div(x, y));
    case ALN_I_AND: VM_EACH((x != 0) && (y != 0));
    case ALN_I_OR: VM_EACH((x != 0) || (y != 0));
    case ALN_I_CMP:
      switch (cmp) {
        case 1: VM_EACH(x < y);
        case 2: VM_EACH(x > y);
        case 3: VM_EACH(x != y);
        case 4: VM_EACH(x == y);
        case 5: VM_EACH(x <= y);
        case 6: VM_EACH(x >= y);
        default: VM_EACH(0);
      }
      break;
    case ALN_I_FADD: VM_EACH(f64_bits(bits_f64(x) + bits_f64(y)));
    case ALN_I_FSUB: VM_EACH(f64_bits(bits_f64(x) - bits_f64(y)));
    case ALN_I_FMUL: VM_EACH(f64_bits(bits_f64(x) * bits_f64(y)));
    case ALN_I_FDIV: VM_EACH(f64_bits(bits_f64(x) / bits_f64(y)));
    default: VM_EACH(fcmp_code(cmp, bits_f64(x), bits_f64(y)));
  }
#undef VM_EACH
}

// Runs the program on U rows per thread; load(col, v) gives a column's values of them.  stk:
// this thread's entry of an LDS array of p.slots * U rows of VM_BLOCK values.
template <int U, typename Load>
__device__ __forceinline__ void vm_eval(const VProg &p, Load load, int64_t *stk, int64_t (&t)[U]) {
  int sp = 0;  // rows of the LDS stack in use
  VInsn next = p.ins[0];
  for (int i = 0; i < p.n; ++i) {
    const VInsn in = next;  // the one after it is fetched while this one runs
    next = p.ins[i + 1 < p.n ? i + 1 : i];
    switch (in.kind) {
      case V_COL:
      case V_CONST: {
        if (in.spill) {
#pragma unroll
          for (int u = 0; u < U; ++u) stk[(sp + u) * VM_BLOCK] = t[u];
          sp += U;
        }
        if (in.kind == V_CONST) {
#pragma unroll
          for (int u = 0; u < U; ++u) t[u] = in.k;
        } else {
          load(in.a, t);
          if (in.k != 1) {
#pragma unroll
            for (int u = 0; u < U; ++u) t[u] = wmul(t[u], in.k);
          }
        }
        break;
      }
      case V_IMM: {
        const int64_t k = in.k;
        if (in.m) {  // division by a small constant: one 64x32-bit product for 32-bit values
#pragma unroll
          for (int u = 0; u < U; ++u)
            t[u] = ((uint64_t)t[u] >> 32) == 0 ? (int64_t)__umul64hi(in.m, (uint64_t)t[u]) : vm_div(t[u], k);
        } else {
          vm_binary<U>(in.op, in.cmp, t, [k](int) { return k; }, t);
        }
        break;
      }
      case V_COLOP: {
        int64_t v[U];
        load(in.a, v);
        if (in.k != 1) {
#pragma unroll
          for (int u = 0; u < U; ++u) v[u] = wmul(v[u], in.k);
        }
        vm_binary<U>(in.op, in.cmp, t, [&v](int u) { return v[u]; }, t);
        break;
      }
      case V_STK: {
        sp -= U;
        int64_t l[U], r[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          l[u] = stk[(sp + u) * VM_BLOCK];
          r[u] = t[u];
        }
        vm_binary<U>(in.op, in.cmp, l, [&r](int u) { return r[u]; }, t);
        break;
      }
      case V_INSET: {
        const uint32_t *set = reinterpret_cast<const uint32_t *>(in.k);
#pragma unroll
        for (int u = 0; u < U; ++u) t[u] = (t[u] >= 0 && t[u] < in.a) ? (set[t[u] >> 5] >> (t[u] & 31)) & 1u : 0;
        break;
      }
      default:  // V_I2F
        if (in.a == 0) {
#pragma unroll
          for (int u = 0; u < U; ++u) t[u] = f64_bits((double)t[u]);
        } else {
#pragma unroll
          for (int u = 0; u < U; ++u) stk[(sp - U + u) * VM_BLOCK] = f64_bits((double)stk[(sp - U + u) * VM_BLOCK]);
        }
    }
  }
}

// Codes of U rows idx[u] of packed `bits`-wide codes, the first `first` (< 32) bits into w
// (w, bits and first wave-uniform; first 0 when bits is 64).  Only words that hold a code are
// read, so a column's last row never touches the next word.  P: a type that first + idx * bits
// fits in.
template <int U, typename P>
__device__ __forceinline__ void unpack_codes(const uint32_t *__restrict__ w, uint32_t bits, const P (&idx)[U],
                                             uint64_t (&c)[U], uint32_t first = 0) {
  if (bits == 0) {
#pragma unroll
    for (int u = 0; u < U; ++u) c[u] = 0;
  } else if (bits <= 32) {
    const uint32_t mask = bits == 32 ? 0xFFFFFFFFu : (1u << bits) - 1u;
    uint32_t lo[U], hi[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const P pos = idx[u] * bits + first;
      const uint32_t *q = w + (pos >> 5);
      lo[u] = q[0];
      hi[u] = q[((uint32_t)pos & 31) + bits > 32 ? 1 : 0];
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      c[u] = __builtin_amdgcn_alignbit(hi[u], lo[u], (uint32_t)(idx[u] * bits + first) & 31) & mask;
  } else if (bits == 64) {
#pragma unroll
    for (int u = 0; u < U; ++u) __builtin_memcpy(&c[u], w + 2 * idx[u], 8);
  } else {
    const uint64_t mask = (1ull << bits) - 1;
    uint32_t a[U], b[U], d[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const P pos = idx[u] * bits + first;
      const uint32_t *q = w + (pos >> 5);
      a[u] = q[0];
      b[u] = q[1];
      d[u] = q[((uint32_t)pos & 31) + bits > 64 ? 2 : 1];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t s = (uint32_t)(idx[u] * bits + first) & 31;
      const uint32_t lo = __builtin_amdgcn_alignbit(b[u], a[u], s), hi = __builtin_amdgcn_alignbit(d[u], b[u], s);
      c[u] = ((uint64_t)hi << 32 | lo) & mask;
    }
  }
}

}  // namespace aln
