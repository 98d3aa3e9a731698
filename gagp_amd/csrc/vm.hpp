// Device bytecode VM: one wavefront (64 lanes) per program, one case per lane
// per tile. The instruction stream is wave-uniform: straight-line programs run
// ip in lockstep; programs with jumps use min-ip scheduling (each step runs the
// smallest pending ip, for the lanes that are at it), so every fetched
// instruction and its static stack height are scalar values. The operand
// stack lives in LDS, slot-major, one 8-byte payload and one tag byte per
// lane and slot, so every stack access is conflict-free.
//
// Instruction semantics restate cpp/src/runtime/cpu/execute_bytecode_cpu.cpp:
// 194-614 (fuel charged and checked first, the first error ends the case)
// and the scalar builtins of cpp/src/runtime/cpu/builtins_cpu.cpp:130-217,
// 340-375,493-500.
#pragma once
#include "core.hpp"
#include "phase.hpp"
#include "steps.hpp"

namespace gagp_amd {

struct ProgView {
  GAS const Ins* code;
  GAS const Val* pool;
  int len;
  int n_locals;
  int has_jumps;
  int fast;      // certified for vm_fast (phase.hpp fast_operation)
  int n_pool;    // constant-pool entries
  int result_tag;  // static result type of a fast program
};

struct CaseData {
  GAS const std::int64_t* in_val;  // [n_inputs][C]
  GAS const std::uint8_t* in_tag;  // [n_inputs][C] (TAG_INVALID: unbound)
  GAS const std::uint8_t* in_b;    // [n_inputs][C]
  GAS const std::int64_t* exp_val; // [C]
  GAS const std::uint8_t* exp_tag; // [C]
  GAS const std::uint8_t* exp_b;   // [C]
  GAS const std::int64_t* arena;   // IntList elements
  GAS const int* order;            // [C] a permutation of the cases (visiting order of the looping path)
  int C, n_inputs;
};

// Per-wave LDS stack, slot-major: payload[slot*64 + lane], tag[...], flag[...].
// Slots [slots, slots + temps) hold the hidden locals after the evaluator
// inputs (local index n_inputs + k in slot slots + k).
struct WaveStack {
  std::int64_t* v;
  std::uint8_t* t;
  std::uint8_t* b;
  int slots;
  int temps;
  // The last `shadow` hidden slots shadow the evaluator inputs of programs
  // that store into them (statement targets): a store lands there and later
  // loads of that input read it; 0 when inputs are read-only.
  int shadow;
};

// Smallest value of x over the wave for 0 <= x < 2^kBits, by a bitwise
// search with ballots (scalar compares, no LDS round trips): bit b of the
// minimum is 0 iff some lane lies in [m, m + 2^b - 1] for the bits m above it.
#if defined(__HIPCC__)
template <int kBits>
__device__ inline int wave_min_bits(int x) {
  int m = 0;
#pragma unroll
  for (int b = kBits - 1; b >= 0; --b)
    if (__ballot(x <= (m | ((1 << b) - 1))) == 0) m |= 1 << b;
  return m;
}
#endif

GHD inline double fbits(std::int64_t i) { union { std::int64_t i; double f; } u{i}; return u.f; }

struct LaneResult {
  std::int64_t v;
  std::uint8_t t, b;
  int err;
  int fuel_used;  // charged fuel (instructions executed under the unit schedule)
};

#if defined(__HIPCC__)
// Runs `p` for case `c` on this lane (active = lane has a case). Returns the
// result or error of the case.
__device__ inline LaneResult vm_run(const ProgView& p, const CaseData& cd, int c, bool active, int fuel0, WaveStack& st,
                                    int lane) {
  LaneResult r{0, TAG_INVALID, 0, active ? ERR_NONE : ERR_VALUE, 0};
  bool done = !active;
  int fuel = fuel0;
  int ip = 0;
  int uncharged = 0;
  // Every iteration runs at least one live lane's instruction, which charges
  // fuel or counts toward the zero-cost cycle limit; this bound is never
  // reached by a correct schedule and ends the wave with ValueError otherwise.
  const long long iteration_limit = 64LL * ((long long)fuel0 + 2LL * p.len + 2) + 64;
  long long iterations = 0;
  for (int k = 0; k < st.temps; ++k) st.t[(st.slots + k) * 64 + lane] = TAG_INVALID;  // unassigned
  for (;;) {
    // Converged live lanes (always so in straight-line code) share their ip:
    // take it from the first live lane (finished lanes keep a stale ip);
    // otherwise take the smallest one (ip <= len < 8191, the code capacity).
    const unsigned long long live = __ballot(!done);
    if (live == 0) break;
    int at = __builtin_amdgcn_readlane(ip, __ffsll((long long)live) - 1);
    if (p.has_jumps && __ballot(!done && ip != at) != 0)
      at = __builtin_amdgcn_readfirstlane(wave_min_bits<13>(done ? 8191 : (ip < 8191 ? ip : 8190)));
    if (++iterations > iteration_limit) {
      if (!done) { r.err = ERR_VALUE; done = true; }
      break;
    }
    at = __builtin_amdgcn_readfirstlane(at);  // uniform: keeps the fetch scalar
    const bool mine = !done && ip == at;
    if (at >= p.len) {  // ran off the end without RETURN
      if (mine) { r.err = ERR_VALUE; done = true; }
      continue;
    }
    const Ins ins = p.code[at];
    const int sp = ins.sp;
    if (mine) {
      const int cost = ins.fuel;
      if (fuel < cost) { r.err = ERR_TIMEOUT; done = true; }
      else {
        fuel -= cost;
        if (cost) uncharged = 0;
        else if (++uncharged > p.len) { r.err = ERR_VALUE; done = true; }
      }
    }
    if (!mine || done) continue;
    ++ip;
    switch (ins.op) {
      case OP_PUSH_CONST: {
        const Val v = p.pool[ins.a];
        st.v[(sp) * 64 + lane] = v.i; st.t[(sp) * 64 + lane] = v.tag; st.b[(sp) * 64 + lane] = v.b;
        break;
      }
      case OP_LOAD: {
        if (ins.a >= cd.n_inputs) {  // a hidden local
          const int k = ins.a - cd.n_inputs;
          const int at_t = (st.slots + k) * 64 + lane;
          if (k >= st.temps - st.shadow || st.t[at_t] == TAG_INVALID) { r.err = ERR_NAME; done = true; break; }
          st.v[(sp) * 64 + lane] = st.v[at_t]; st.t[(sp) * 64 + lane] = st.t[at_t]; st.b[(sp) * 64 + lane] = st.b[at_t];
          break;
        }
        if (ins.a < st.shadow) {  // a stored input reads its shadow
          const int at_s = (st.slots + st.temps - st.shadow + ins.a) * 64 + lane;
          if (st.t[at_s] != TAG_INVALID) {
            st.v[(sp) * 64 + lane] = st.v[at_s]; st.t[(sp) * 64 + lane] = st.t[at_s]; st.b[(sp) * 64 + lane] = st.b[at_s];
            break;
          }
        }
        const std::size_t at_in = std::size_t(ins.a) * cd.C + c;
        const std::uint8_t tag = cd.in_tag[at_in];
        if (tag == TAG_INVALID) { r.err = ERR_NAME; done = true; break; }
        st.v[(sp) * 64 + lane] = cd.in_val[at_in]; st.t[(sp) * 64 + lane] = tag; st.b[(sp) * 64 + lane] = cd.in_b[at_in];
        break;
      }
      case OP_STORE: {  // a hidden local, or an input's shadow
        const int k = ins.a < cd.n_inputs ? st.temps - st.shadow + ins.a : ins.a - cd.n_inputs;
        if (ins.a < 0 || (ins.a < cd.n_inputs ? ins.a >= st.shadow : k >= st.temps - st.shadow)) {
          r.err = ERR_VALUE; done = true; break;
        }
        const int at_t = (st.slots + k) * 64 + lane;
        st.v[at_t] = st.v[(sp - 1) * 64 + lane]; st.t[at_t] = st.t[(sp - 1) * 64 + lane]; st.b[at_t] = st.b[(sp - 1) * 64 + lane];
        break;
      }
      case OP_CHECK_INT:
        if (st.t[(sp - 1) * 64 + lane] != TAG_INT) { r.err = ERR_TYPE; done = true; }
        break;
      case OP_CHECK_LIST: {
        const std::uint8_t t = st.t[(sp - 1) * 64 + lane];
        if (t != TAG_INT_LIST && t != TAG_FLOAT_LIST && t != TAG_STRING_LIST) { r.err = ERR_TYPE; done = true; }
        break;
      }
      case OP_NEG: {
        const std::uint8_t t = st.t[(sp - 1) * 64 + lane];
        if (t == TAG_INT) st.v[(sp - 1) * 64 + lane] = wrap_neg(st.v[(sp - 1) * 64 + lane]);
        else if (t == TAG_FLOAT) {
          union { std::int64_t i; double f; } u{st.v[(sp - 1) * 64 + lane]};
          st.v[(sp - 1) * 64 + lane] = val_float(canon32(-u.f)).i;
        } else { r.err = ERR_TYPE; done = true; }
        break;
      }
      case OP_NOT:
        if (st.t[(sp - 1) * 64 + lane] != TAG_BOOL) { r.err = ERR_TYPE; done = true; }
        else st.b[(sp - 1) * 64 + lane] = !st.b[(sp - 1) * 64 + lane];
        break;
      case OP_ADD: case OP_SUB: case OP_MUL: case OP_DIV: case OP_MOD: {
        const std::uint8_t ta = st.t[(sp - 2) * 64 + lane], tb = st.t[(sp - 1) * 64 + lane];
        const std::int64_t a = st.v[(sp - 2) * 64 + lane], b = st.v[(sp - 1) * 64 + lane];
        if (ta == TAG_INT && tb == TAG_INT) {
          if ((ins.op == OP_DIV || ins.op == OP_MOD) && b == 0) { r.err = ERR_ZERO_DIV; done = true; break; }
          std::int64_t out;
          if (ins.op == OP_ADD) out = wrap_add(a, b);
          else if (ins.op == OP_SUB) out = wrap_sub(a, b);
          else if (ins.op == OP_MUL) out = wrap_mul(a, b);
          else if (ins.op == OP_MOD) out = py_mod(a, b);
          else {
            st.v[(sp - 2) * 64 + lane] = val_float(canon32(double(a) / double(b))).i;
            st.t[(sp - 2) * 64 + lane] = TAG_FLOAT;
            break;
          }
          st.v[(sp - 2) * 64 + lane] = out;
        } else if (ta == TAG_FLOAT && tb == TAG_FLOAT) {
          union { std::int64_t i; double f; } x{a}, y{b};
          if ((ins.op == OP_DIV || ins.op == OP_MOD) && y.f == 0.0) { r.err = ERR_ZERO_DIV; done = true; break; }
          double out;
          if (ins.op == OP_ADD) out = x.f + y.f;
          else if (ins.op == OP_SUB) out = x.f - y.f;
          else if (ins.op == OP_MUL) out = x.f * y.f;
          else if (ins.op == OP_DIV) out = x.f / y.f;
          else {
            double m = fmod(x.f, y.f);
            if (m == 0.0) m = copysign(0.0, y.f);
            else if (signbit(m) != signbit(y.f)) m += y.f;
            out = m;
          }
          st.v[(sp - 2) * 64 + lane] = val_float(canon32(out)).i;
        } else { r.err = ERR_TYPE; done = true; }
        break;
      }
      case OP_LT: case OP_LE: case OP_GT: case OP_GE: case OP_EQ: case OP_NE: {
        const std::uint8_t ta = st.t[(sp - 2) * 64 + lane], tb = st.t[(sp - 1) * 64 + lane];
        const std::int64_t a = st.v[(sp - 2) * 64 + lane], b = st.v[(sp - 1) * 64 + lane];
        bool out = false;
        if (ins.op == OP_EQ || ins.op == OP_NE) {
          if (ta != tb) { r.err = ERR_TYPE; done = true; break; }
          bool eq;
          if (ta == TAG_BOOL) eq = st.b[(sp - 2) * 64 + lane] == st.b[(sp - 1) * 64 + lane];
          else if (ta == TAG_FLOAT) { union { std::int64_t i; double f; } x{a}, y{b}; eq = x.f == y.f; }
          else if (ta == TAG_INT || ta == TAG_CHAR || ta == TAG_STRING || ta == TAG_INT_LIST || ta == TAG_FLOAT_LIST ||
                   ta == TAG_STRING_LIST) eq = a == b;
          else { r.err = ERR_TYPE; done = true; break; }
          out = ins.op == OP_EQ ? eq : !eq;
        } else if (ta == TAG_INT && tb == TAG_INT) {
          out = ins.op == OP_LT ? a < b : ins.op == OP_LE ? a <= b : ins.op == OP_GT ? a > b : a >= b;
        } else if (ta == TAG_FLOAT && tb == TAG_FLOAT) {
          union { std::int64_t i; double f; } x{a}, y{b};
          out = ins.op == OP_LT ? x.f < y.f : ins.op == OP_LE ? x.f <= y.f : ins.op == OP_GT ? x.f > y.f : x.f >= y.f;
        } else { r.err = ERR_TYPE; done = true; break; }
        st.v[(sp - 2) * 64 + lane] = 0; st.t[(sp - 2) * 64 + lane] = TAG_BOOL; st.b[(sp - 2) * 64 + lane] = out;
        break;
      }
      case OP_JMP:
        ip = ins.a;
        break;
      case OP_JMP_IF_FALSE: case OP_JMP_IF_TRUE: {
        if (st.t[(sp - 1) * 64 + lane] != TAG_BOOL) { r.err = ERR_TYPE; done = true; break; }
        const bool cond = st.b[(sp - 1) * 64 + lane] != 0;
        if ((ins.op == OP_JMP_IF_FALSE && !cond) || (ins.op == OP_JMP_IF_TRUE && cond)) ip = ins.a;
        break;
      }
      case OP_RETURN:
        r.v = st.v[(sp - 1) * 64 + lane]; r.t = st.t[(sp - 1) * 64 + lane]; r.b = st.b[(sp - 1) * 64 + lane];
        done = true;
        break;
      case OP_CALL_BUILTIN: {
        const int argc = ins.argc, base = sp - argc;
        std::int64_t out = 0;
        std::uint8_t out_t = TAG_INT, out_b = 0;
        const auto ti = [&](int k) { return st.t[(base + k) * 64 + lane]; };
        const auto vi = [&](int k) { return st.v[(base + k) * 64 + lane]; };
        switch (ins.a) {
          case B_ABS:
            if (argc != 1 || !is_numeric(ti(0))) { r.err = ERR_TYPE; break; }
            if (ti(0) == TAG_FLOAT) {
              const double x = fbits(vi(0));
              out = val_float(canon32(x < 0 ? -x : x)).i;
              out_t = TAG_FLOAT;
            } else out = vi(0) < 0 ? wrap_neg(vi(0)) : vi(0);
            break;
          case B_MIN: case B_MAX:
            if (argc != 2 || !is_numeric(ti(0)) || ti(0) != ti(1)) { r.err = ERR_TYPE; break; }
            if (ti(0) == TAG_FLOAT) {
              const double a = fbits(vi(0)), b = fbits(vi(1));
              out = val_float(canon32(ins.a == B_MIN ? (a <= b ? a : b) : (a >= b ? a : b))).i;
              out_t = TAG_FLOAT;
            } else out = ins.a == B_MIN ? (vi(0) < vi(1) ? vi(0) : vi(1)) : (vi(0) > vi(1) ? vi(0) : vi(1));
            break;
          case B_CLIP: {
            if (argc != 3 || !is_numeric(ti(0)) || ti(0) != ti(1) || ti(0) != ti(2)) { r.err = ERR_TYPE; break; }
            if (ti(0) == TAG_FLOAT) {
              const double x = fbits(vi(0)), lo = fbits(vi(1)), hi = fbits(vi(2));
              const double m = x > lo ? x : lo;  // min(max(x, lo), hi)
              out = val_float(canon32(m < hi ? m : hi)).i;
              out_t = TAG_FLOAT;
              break;
            }
            const std::int64_t m = vi(0) > vi(1) ? vi(0) : vi(1);
            out = m < vi(2) ? m : vi(2);
            break;
          }
          case B_IDIV0: case B_IMOD0: case B_TRUNC_DIV0: case B_TRUNC_MOD0: {
            if (argc != 2 || ti(0) != TAG_INT || ti(1) != TAG_INT) { r.err = ERR_TYPE; break; }
            const std::int64_t a = vi(0), b = vi(1);
            if (b == 0) out = 0;
            else if (ins.a == B_TRUNC_DIV0) out = trunc_div0(a, b);
            else if (ins.a == B_TRUNC_MOD0) out = trunc_mod0(a, b);
            else if (ins.a == B_IDIV0) out = wrap_div(a, b);
            else out = py_mod(a, b);
            break;
          }
          case B_LEN: {
            const std::uint8_t t = ti(0);
            if (argc != 1 || !(t == TAG_INT_LIST || t == TAG_FLOAT_LIST || t == TAG_STRING_LIST)) { r.err = ERR_TYPE; break; }
            out = std::int64_t(std::uint64_t(vi(0)) & 0xffff);
            break;
          }
          case B_INDEX: case B_INDEX_NONNEG: case B_INDEX_CLAMPED: {
            if (argc != 2 || ti(0) != TAG_INT_LIST || ti(1) != TAG_INT) { r.err = ERR_TYPE; break; }
            const std::int64_t n = std::int64_t(std::uint64_t(vi(0)) & 0xffff);
            const std::uint64_t off = std::uint64_t(vi(0)) >> 16;
            std::int64_t j = vi(1);
            if (ins.a == B_INDEX_CLAMPED) {
              if (n == 0) { out = 0; break; }
              j = j < 0 ? 0 : (j >= n ? n - 1 : j);
            } else {
              if (ins.a == B_INDEX_NONNEG && j < 0) { r.err = ERR_VALUE; break; }
              if (j < 0) j += n;
              if (j < 0 || j >= n) { r.err = ERR_VALUE; break; }
            }
            out = cd.arena[off + std::uint64_t(j)];
            break;
          }
          case B_IS_INT:
            if (argc != 1) { r.err = ERR_TYPE; break; }
            out_t = TAG_BOOL;
            out_b = ti(0) == TAG_INT;
            break;
          default: r.err = ERR_NAME; break;
        }
        if (r.err != ERR_NONE) { done = true; break; }
        st.v[(base) * 64 + lane] = out; st.t[(base) * 64 + lane] = out_t; st.b[(base) * 64 + lane] = out_b;
        break;
      }
      default:
        r.err = ERR_VALUE; done = true;
        break;
    }
  }
  r.fuel_used = fuel0 - fuel;
  return r;
}

// Truncating quotient and remainder of x by y (y neither 0 nor -1) for the
// active lanes. Where every operand fits 32 bits the quotient comes from one
// refined double reciprocal: |x| / |y| is below 2^32 and the reciprocal is
// good to 2^-44, so the floor is the quotient or one off, the fused remainder
// is exact and one correction either way settles it.
__device__ inline void divide_trunc(std::int64_t x, std::int64_t y, std::int64_t& q, std::int64_t& rem) {
  const bool wide = x != std::int64_t(int(x)) || y != std::int64_t(int(y));
  if (__ballot(wide) == 0) {
    const double a = __builtin_fabs(double(int(x))), b = __builtin_fabs(double(int(y)));
    double r = __builtin_amdgcn_rcp(b);
    r = __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);
    double f = __builtin_floor(a * r), m = __builtin_fma(-f, b, a);
    const bool under = m < 0;
    f = under ? f - 1 : f;
    m = under ? m + b : m;
    const bool over = m >= b;
    f = over ? f + 1 : f;
    m = over ? m - b : m;
    const std::int64_t uq = std::int64_t(unsigned(f)), ur = std::int64_t(unsigned(m));
    q = (x < 0) != (y < 0) ? -uq : uq;
    rem = x < 0 ? -ur : ur;
    return;
  }
  q = x / y;
  rem = x - q * y;
}
// MOD and the protected divisions on untagged operands (MOD by zero: 0).
__device__ inline std::int64_t step_divide(int op, std::int64_t x, std::int64_t y) {
  const std::int64_t safe = (y == 0 || y == -1) ? 1 : y;
  std::int64_t q, rem;
  divide_trunc(x, safe, q, rem);
  if (y == -1) { q = wrap_neg(x); rem = 0; }
  const std::int64_t floor_mod = (rem != 0 && ((rem < 0) != (y < 0))) ? rem + y : rem;  // Python %
  if (op == SO_MOD || op == SO_IMOD0) return y == 0 ? 0 : floor_mod;                              // py_mod
  if (op == SO_IDIV0) return y == 0 ? 0 : q;                                                       // wrap_div
  const bool none = y == 0 || (x == INT64_MIN && y == -1);
  return none ? 0 : op == SO_TDIV0 ? q : rem;                                                      // trunc_div0, trunc_mod0
}

// ---- typed straight-line path ----
// A certified program (no jumps, every value statically Int or Bool, integer
// builtins only) needs no run-time tags: values are int64 (Bool as 0/1), the
// stack is a register array indexed by the instruction's static height (the
// index is uniform, so the compiler addresses the array with indexed register
// moves), and every live lane executes the same instruction. Instruction j is
// held by lane j % 64 of register group j / 64 and read with readlane; so are
// the constants. Fuel is charged uniformly: a timeout ends every live lane at
// the same instruction, as the per-lane charge of vm_run would.
struct FastProgram {
  int w0[2], w1[2];  // instruction: op | argc << 8 | sp << 16 | fuel << 24, operand
  int c0[2], c1[2];  // constant payload, low and high words
  int len;
};
__device__ inline FastProgram fast_load(const ProgView& p, int lane) {
  FastProgram f;
  f.len = p.len;
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const int j = g * 64 + lane;
    int w0 = 0, w1 = 0;
    if (j < p.len) {
      const Ins ins = p.code[j];
      w0 = int(ins.op) | int(ins.argc) << 8 | int(ins.sp) << 16 | int(unsigned(ins.fuel) << 24);
      w1 = ins.a;
    }
    std::int64_t v = 0;
    if (j < p.n_pool) {
      const Val x = p.pool[j];
      v = x.tag == TAG_BOOL ? std::int64_t(x.b != 0) : x.i;
    }
    f.w0[g] = w0;
    f.w1[g] = w1;
    f.c0[g] = int(std::uint32_t(std::uint64_t(v)));
    f.c1[g] = int(std::uint32_t(std::uint64_t(v) >> 32));
  }
  return f;
}
__device__ inline int fast_pick(const int (&v)[2], int k) {
  const int lo = __builtin_amdgcn_readlane(v[0], k & 63), hi = __builtin_amdgcn_readlane(v[1], k & 63);
  return k < 64 ? lo : hi;
}
// Inputs of this lane's case: payloads (Bool as 0/1) and the bound mask.
// (Separate fields and a uniform select keep them in registers; an array
// indexed by the operand would live in scratch.)
static_assert(kFastInputs == 4, "four input registers");
struct FastInputs {
  std::int64_t v0, v1, v2, v3;
  unsigned bound;
  __device__ std::int64_t pick(int k) const { return k == 0 ? v0 : k == 1 ? v1 : k == 2 ? v2 : v3; }
};
__device__ inline FastInputs fast_inputs(const CaseData& cd, int n_inputs, int c, bool active) {
  FastInputs in{0, 0, 0, 0, 0};
  std::int64_t v[kFastInputs];
#pragma unroll
  for (int k = 0; k < kFastInputs; ++k) {
    v[k] = 0;
    if (k < n_inputs && k < cd.n_inputs && active) {
      const std::size_t at = std::size_t(k) * cd.C + c;
      const std::uint8_t tag = cd.in_tag[at];
      if (tag != TAG_INVALID) in.bound |= 1u << k;
      v[k] = tag == TAG_BOOL ? std::int64_t(cd.in_b[at] != 0) : cd.in_val[at];
    }
  }
  in.v0 = v[0];
  in.v1 = v[1];
  in.v2 = v[2];
  in.v3 = v[3];
  return in;
}
// The top of the stack is a register of its own, and the array is written by
// one statement of the loop (the top it spills when a value is pushed): with a
// write in every operation the compiler merged the whole array, 32 registers,
// at the end of each. The loop is one nest of two-way uniform branches with a
// single exit, and of a lane that fails it keeps one word: what was merged per
// lane was copied on every path. Bound by instruction issue. Per launch, before
// and after: 1670 programs of the quintic grammar on 256 cases 63 and 35 us, 64
// mixed searches 371 and 225, 360 polynomials on 21 cases 21 and 14, a caller's
// 4001 programs on 777 cases 0.52 and 0.28 ms; with the copies of the failure record 47, 287,
// 17 and 0.34.
__device__ inline LaneResult vm_fast(const FastProgram& f, const FastInputs& in, bool active, int fuel0, int result_tag) {
  enum Outcome : int { RUNS, RETURNED, TIMED_OUT, ENDED, NO_NAME };
  LaneResult r{0, TAG_INVALID, 0, active ? ERR_NONE : ERR_VALUE, 0};
  std::int64_t s[kFastStack];  // the elements below the top
#pragma unroll
  for (int k = 0; k < kFastStack; ++k) s[k] = 0;
  const std::int64_t inputs[kFastInputs] = {in.v0, in.v1, in.v2, in.v3};
  std::int64_t top = 0;
  unsigned bound = 0;  // inputs bound on every lane
#pragma unroll
  for (int k = 0; k < kFastInputs; ++k) bound |= __ballot(active && !(in.bound >> k & 1u)) == 0 ? 1u << k : 0u;
  int fuel = fuel0, ip = 0, outcome = RUNS;
  int failed = 0;  // the lane's failing instruction: 2 * its index + 2, and 1 for a division by zero
  while (outcome == RUNS) {
    const int w = fast_pick(f.w0, ip), a = fast_pick(f.w1, ip);
    const int op = w & 0xff, sp = (w >> 16) & 0xff, cost = int(unsigned(w) >> 24);
    if (ip >= f.len) {
      outcome = ENDED;
    } else if (fuel < cost) {
      outcome = TIMED_OUT;
    } else {
      fuel -= cost;
      ++ip;
      if (op <= OP_LOAD) {
        // Heights are certified within the stack; the mask keeps every index in range.
        s[(sp - 1) & (kFastStack - 1)] = top;
        if (op == OP_PUSH_CONST) {
          const std::uint32_t lo = std::uint32_t(fast_pick(f.c0, a)), hi = std::uint32_t(fast_pick(f.c1, a));
          top = std::int64_t(std::uint64_t(hi) << 32 | lo);
        } else {
          if ((bound >> (a & 31) & 1u) == 0) failed = failed == 0 && !((in.bound >> (a & 31)) & 1u) ? 2 * ip : failed;
          top = inputs[a & (kFastInputs - 1)];
        }
      } else if (op >= OP_ADD && op <= OP_NE && op != OP_MOD) {
        const std::int64_t x = s[(sp - 2) & (kFastStack - 1)], y = top;
        if (op == OP_ADD) {
          top = wrap_add(x, y);
        } else if (op == OP_SUB) {
          top = wrap_sub(x, y);
        } else if (op == OP_MUL) {
          top = wrap_mul(x, y);
        } else if (op != OP_DIV) {
          const bool less = x < y, equal = x == y;
          top = op == OP_LT ? less : op == OP_LE ? less || equal : op == OP_GT ? !(less || equal) : op == OP_GE ? !less
                : op == OP_EQ ? equal : !equal;
        } else {
          outcome = ENDED;
        }
      } else if (op == OP_RETURN) {
        outcome = RETURNED;
      } else if (op == OP_NEG) {
        top = wrap_neg(top);
      } else if (op == OP_NOT) {
        top = top == 0;
      } else if (op == OP_CALL_BUILTIN || op == OP_MOD) {
        const std::int64_t x = s[(sp - 2) & (kFastStack - 1)], y = top;
        // MOD and the protected divisions share one division.
        const int divide = op == OP_MOD ? int(SO_MOD) : a == B_IDIV0 ? int(SO_IDIV0) : a == B_IMOD0 ? int(SO_IMOD0)
                           : a == B_TRUNC_DIV0 ? int(SO_TDIV0) : a == B_TRUNC_MOD0 ? int(SO_TMOD0) : int(SO_NONE);
        if (divide != SO_NONE) {
          if (divide == SO_MOD) failed = failed == 0 && y == 0 ? 2 * ip + 1 : failed;
          top = step_divide(divide, x, y);
        } else if (a == B_ABS) {
          top = y < 0 ? wrap_neg(y) : y;
        } else if (a == B_MIN) {
          top = x < y ? x : y;
        } else if (a == B_MAX) {
          top = x > y ? x : y;
        } else if (a == B_CLIP) {
          const std::int64_t v = s[(sp - 3) & (kFastStack - 1)], m = v > x ? v : x;
          top = m < y ? m : y;
        } else {
          outcome = NO_NAME;
        }
      } else if (op != OP_CHECK_INT) {
        outcome = ENDED;
      }
    }
  }
  if (!active) return r;
  r.fuel_used = fuel0 - fuel;
  if (outcome == RETURNED) {
    if (result_tag == TAG_BOOL) { r.t = TAG_BOOL; r.b = top != 0; r.v = 0; }
    else { r.t = TAG_INT; r.v = top; }
  } else {
    r.err = outcome == TIMED_OUT ? ERR_TIMEOUT : outcome == NO_NAME ? ERR_NAME : ERR_VALUE;
  }
  if (__ballot(failed != 0)) {
    // The charge up to the failing instruction.
    int used = 0;
    for (int k = 0; k < ip; ++k) {
      used += int(unsigned(fast_pick(f.w0, k)) >> 24);
      if (failed >> 1 == k + 1) {
        r = LaneResult{0, TAG_INVALID, 0, failed & 1 ? ERR_ZERO_DIV : ERR_NAME, 0};
        r.fuel_used = used;
      }
    }
  }
  return r;
}

// ---- typed looping path ----
// A program certified like the straight-line path but with jumps, hidden
// locals or IntList views (phase.hpp loop_operation): values are untagged
// int64 (Bool as 0/1, an IntList as its view payload). It runs as decoded
// steps (steps.hpp): the top of the operand stack is a register, and inputs,
// hidden locals and the elements below the top are 8-byte LDS slots per lane
// (slot-major, conflict-free). Step j sits in lane j % 64 of register group
// j / 64 and is read with readlane, so a fetch costs no memory round trip.
//
// Lanes follow their own branches. The lanes at the smallest step index run
// together as a group: inside a run the step index, the decoded fields and the
// fuel charged are scalar, and fuel is checked against the group's smallest
// balance by one scalar compare. A run ends where the group's lanes part, a
// lane finishes, or the group reaches the step at which other lanes wait; only
// there are the per-lane indexes and balances written and the next group
// chosen. Every lane computes; the group's mask selects what it keeps (the top,
// a list element) and where it stores (its slot, else a spare one). Under the
// mask as execution mask the steps would be read from registers whose other
// lanes the compiler may drop in any copy or spill it makes there, which only
// chance kept it from. Stores under the mask cost k_eval_loop more branches: 468
// and 436 us on 4096 list programs x 200 cases, 511 and 479 on 1500 statement
// programs x 130.
// Interpreting the bytecode itself, predicated and one instruction (or fixed
// sequence) at a time, issued about 31 vector and 40 scalar instructions per
// step and three times the steps; k_eval_loop has the measured times.
struct StepProgram {
  unsigned w0[4], w1[4], c0[4], c1[4];
  int n;
};
__device__ inline void steps_hold(StepProgram& f, int g, const Step& s) {
  f.w0[g] = s.w0;
  f.w1[g] = s.w1;
  f.c0[g] = unsigned(std::uint64_t(s.c));
  f.c1[g] = unsigned(std::uint64_t(s.c) >> 32);
}
__device__ inline StepProgram steps_load(GAS const Step* steps, int n, int lane) {
  StepProgram f;
  f.n = n;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int j = g * 64 + lane;
    Step s{0, 0, 0};
    if (j < n) {
      s.w0 = steps[j].w0;
      s.w1 = steps[j].w1;
      s.c = steps[j].c;
    }
    steps_hold(f, g, s);
  }
  return f;
}
// Packed steps and the constants they index: two round trips instead of one,
// once per item of 64 cases.
__device__ inline StepProgram steps_load(GAS const std::uint64_t* words, GAS const Val* pool, int n, int lane) {
  StepProgram f;
  f.n = n;
  std::uint64_t word[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) word[g] = g * 64 + lane < n ? words[g * 64 + lane] : 0;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    Step s = unpack_step(word[g]);
    if (step_indexes(s)) {  // never of an absent step: its word names no constant
      GAS const Val* const v = pool + s.c;
      s.c = v->tag == TAG_BOOL ? std::int64_t(v->b != 0) : v->i;
    }
    steps_hold(f, g, s);
  }
  return f;
}
// Word `v` of step k (uniform, below 64 * kGroups).
template <int kGroups>
__device__ inline unsigned step_word(const unsigned (&v)[4], int k) {
  if constexpr (kGroups == 1) return unsigned(__builtin_amdgcn_readlane(int(v[0]), k));
  const int g = k & 63;
  unsigned w = unsigned(__builtin_amdgcn_readlane(int(v[0]), g));
  if (k >= 64) {
    const unsigned w1 = unsigned(__builtin_amdgcn_readlane(int(v[1]), g));
    const unsigned w2 = unsigned(__builtin_amdgcn_readlane(int(v[2]), g)), w3 = unsigned(__builtin_amdgcn_readlane(int(v[3]), g));
    w = k < 128 ? w1 : k < 192 ? w2 : w3;
  }
  return w;
}
// Smallest value over the wave (all lanes active), in the data-parallel
// shifts: row of 16, then across rows; the last lane holds the result.
__device__ inline int wave_min_all(int x) {
  const auto shifted = [&](auto control, auto rows) {
    const int y = __builtin_amdgcn_update_dpp(0x7fffffff, x, decltype(control)::value, decltype(rows)::value, 0xf, false);
    x = y < x ? y : x;
  };
  shifted(std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xf>{});
  shifted(std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xf>{});
  shifted(std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xf>{});
  shifted(std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xf>{});
  shifted(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});
  shifted(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});
  return __builtin_amdgcn_readlane(x, 63);
}
// `slots`: this wave's LDS area of step_slots(n_inputs) slots (slot k of lane
// j at k * 64 + j). kGroups: register groups that hold the program's steps.
// The run loop is one nest of two-way uniform branches with a single exit (no
// switch, break or continue) and no divergent branch: what a lane records when
// it ends is written after the loop, from the event that ended it. In this
// form the compiler keeps the step index, the fields, the balances and the
// event in scalar registers and only the stack's top in vector ones; any
// per-lane record merged inside the loop would be copied on every path of
// every step.
template <int kGroups>
__device__ inline LaneResult vm_steps(const StepProgram& f, const FastInputs& in, int n_inputs, GAS const std::int64_t* arena,
                                      LAS std::int64_t* slots, int lane, bool active, int fuel0, int result_tag) {
  constexpr int kNone = 0x7fffffff, kMost = 12;  // the largest charge of a step
  constexpr unsigned kStepNoSlot = ~0u;
  enum Event : int { EV_NONE, EV_BRANCH, EV_TEST, EV_ZERO_DIV, EV_VALUE, EV_RETURN, EV_FAIL_TYPE, EV_FAIL_VALUE };
  LaneResult r{0, TAG_INVALID, 0, active ? ERR_NONE : ERR_VALUE, 0};
  LAS std::int64_t* const sl = slots + lane;
  for (int k = 0; k < n_inputs; ++k) sl[k * 64] = in.pick(k);
  const int spare = step_slots(n_inputs) - 1;
  bool done = !active;
  std::int64_t top = 0;
  int ip = 0, fuel = fuel0;
  // No live lane has less fuel than `low`. Lanes with an unbound input run
  // step by step, checked before each.
  unsigned bound = in.bound;
  const bool unbound = __ballot(active && (~bound & ((1u << n_inputs) - 1u)) != 0) != 0;
  int low = unbound ? 0 : fuel0;
  for (;;) {
    const unsigned long long live = __ballot(!done);
    if (live == 0) break;
    // The group: the lanes at the smallest index; `stop`: the next one at
    // which lanes wait. Mostly one index, or two.
    int at = __builtin_amdgcn_readlane(ip, __ffsll((long long)live) - 1), stop = f.n;
    const unsigned long long same = __ballot(!done && ip == at);
    if (same != live) {
      const int other = __builtin_amdgcn_readlane(ip, __ffsll((long long)(live & ~same)) - 1);
      if ((same | __ballot(!done && ip == other)) == live) {
        stop = at < other ? other : at;
        at = at < other ? at : other;
      } else {
        at = wave_min_all(done ? kNone : ip);
        stop = wave_min_all(done || ip == at ? kNone : ip);
      }
    }
    // Restated as uniform: values merged where the branches above part are
    // not known to be.
    at = __builtin_amdgcn_readfirstlane(at);
    stop = __builtin_amdgcn_readfirstlane(stop);
    low = __builtin_amdgcn_readfirstlane(low);
    if (at >= f.n) {  // ran off the end without RETURN
      if (!done && ip == at) { r.err = ERR_VALUE; r.fuel_used = fuel0 - fuel; done = true; }
      continue;
    }
    const bool mine = !done && ip == at;
    const auto store = [&](int slot, std::int64_t v) { sl[(mine ? slot : spare) * 64] = v; };
    int budget = low;
    if (low < kMost) {
      // Near exhaustion the group takes one step at a time. Lanes that cannot
      // pay for it end here, their last unit charged inside it (every
      // instruction charges one).
      const unsigned w0 = step_word<kGroups>(f.w0, at), w1 = step_word<kGroups>(f.w1, at);
      const int op = int(w0 & 63u);
      int need = int(w0 >> 24), err = ERR_TIMEOUT, used = fuel0;
      if (op == SO_WALK_TEST || op == SO_RANGE_TEST) {
        const std::int64_t counter = sl[(w1 & 31u) * 64], limit = sl[((w1 >> 5) & 31u) * 64];
        const bool reverse = op == SO_WALK_TEST && (step_word<kGroups>(f.c0, at) >> 24) != 0;
        if (!(reverse ? counter >= limit : counter < limit)) need = 4;
      }
      bool fails = mine && fuel < need;
      if (unbound && op < kStepControl) {
        // Loads of unbound inputs, in order: an exchanged pair's first operand
        // is its second load.
        const unsigned a = w1 & 31u, b = (w1 >> 5) & 31u, loads = w0 >> 14 & 3u;
        const bool x_out = (w0 & kStepX) && a < unsigned(n_inputs) && !(bound >> a & 1u);
        const bool y_out = ((w0 >> 8) & 3u) == 1 && b < unsigned(n_inputs) && !(bound >> b & 1u);
        const int charge = x_out ? (loads == 3 ? 2 : 1) : (loads >= 2 ? 2 : 1);
        if (mine && (x_out || y_out) && fuel >= charge) {
          fails = true;
          err = ERR_NAME;
          used = fuel0 - fuel + charge;
        }
      }
      if (fails) { r.err = err; r.fuel_used = used; done = true; }
      if (__ballot(fails) != 0) continue;
      if (!unbound) {
        // Other lanes may be the ones near exhaustion.
        low = wave_min_all(done ? kNone : fuel);
        budget = wave_min_all(mine ? fuel : kNone);
      }
    }
    budget = __builtin_amdgcn_readfirstlane(budget);
    const unsigned long long group = __ballot(mine);
    int spent = 0, event = EV_NONE, last = at;
    unsigned long long mask = 0;  // the lanes an event names
    unsigned sink_slot = kStepNoSlot;
    do {
      const unsigned w0 = step_word<kGroups>(f.w0, at), w1 = step_word<kGroups>(f.w1, at);
      const int op = int(w0 & 63u), cost = int(w0 >> 24);
      budget -= cost;
      spent += cost;
      const int a = int(w1 & 31u), b = int((w1 >> 5) & 31u), p = int((w1 >> 10) & 31u), target = int(w1 >> 16);
      int next = at + 1;
      if (op < kStepControl) {
        std::int64_t x = top, y = top;
        if (w0 & kStepPush) store(p, top);
        if (w0 & kStepX) x = sl[a * 64];
        const unsigned yk = (w0 >> 8) & 3u, sink = (w0 >> 10) & 7u;
        if (yk == 2) y = std::int64_t(std::uint64_t(step_word<kGroups>(f.c1, at)) << 32 | step_word<kGroups>(f.c0, at));
        else if (yk == 1) y = sl[b * 64];
        unsigned long long holds = 0;
        std::int64_t out = y;
        if (op >= kStepBool) {
          if (op < SO_GT) {
            if (op < SO_LT) holds = op == SO_TEST ? __ballot(x != 0) : __ballot(x == 0);
            else if (op == SO_LT) holds = __ballot(x < y);
            else holds = __ballot(x <= y);
          } else {
            if (op < SO_EQ) {
              if (op == SO_GT) holds = __ballot(x > y);
              else holds = __ballot(x >= y);
            } else {
              if (op == SO_EQ) holds = __ballot(x == y);
              else holds = __ballot(x != y);
            }
          }
          out = std::int64_t((holds >> lane) & 1u);
        } else if (op < SO_MIN) {
          if (op < SO_SUB) {
            if (op == SO_ADD) out = wrap_add(x, y);
          } else {
            if (op == SO_SUB) out = wrap_sub(x, y);
            else out = wrap_mul(x, y);
          }
        } else if (op < SO_INDEX) {
          if (op < SO_MOD) {
            if (op == SO_MIN) out = x < y ? x : y;
            else out = x > y ? x : y;
          } else {
            out = step_divide(op, mine ? x : 0, mine ? y : 1);
            mask = op == SO_MOD ? __ballot(y == 0) & group : 0;
            event = mask != 0 ? EV_ZERO_DIV : EV_NONE;
          }
        } else if (op < SO_NEG) {
          // List indexing, as in vm_run. Only a valid index is read; the
          // rest read the arena's first element (it is never empty).
          const std::int64_t n = std::int64_t(std::uint64_t(x) & 0xffff);
          const bool clamped = op == SO_INDEX_CLAMPED;  // an empty list reads as 0
          const bool negative = op == SO_INDEX_NONNEG && y < 0;
          const std::int64_t inside = y < 0 ? 0 : y >= n ? n - 1 : y, wrapped = y < 0 ? y + n : y;
          const std::int64_t k = clamped ? inside : wrapped;
          const bool ok = mine && !negative && k >= 0 && k < n;
          const std::int64_t v = arena[ok ? (std::uint64_t(x) >> 16) + std::uint64_t(k) : 0];
          out = ok ? v : 0;
          mask = clamped ? 0 : group & ~__ballot(ok);
          event = mask != 0 ? EV_VALUE : EV_NONE;
        } else if (op < SO_LEN) {
          out = op == SO_NEG || x < 0 ? wrap_neg(x) : x;  // NEG, ABS
        } else if (op < SO_CLIP) {
          out = op == SO_LEN ? std::int64_t(std::uint64_t(x) & 0xffff) : 1;
        } else {
          const std::int64_t m = x > y ? x : y;
          out = m < top ? m : top;
        }
        if (sink < SK_IF_FALSE) {
          top = mine ? out : top;
          next = sink == SK_TOP_JUMP ? target : next;
        } else {
          if (sink == SK_STORE) {
            store(target, out);
            sink_slot = unsigned(target);
          } else {
            const unsigned long long jumps = sink == SK_IF_TRUE ? holds & group : group & ~holds;
            mask = jumps;
            event = jumps != 0 && jumps != group ? EV_BRANCH : EV_NONE;
            next = jumps == group ? target : next;
          }
          if (w0 & kStepPop) top = mine ? sl[p * 64] : top;
        }
      } else if (op < SO_WALK_TEST) {
        event = op == SO_JUMP ? EV_NONE : EV_RETURN;
        next = target;
      } else if (op < SO_RANGE_TEST) {
        if (op == SO_WALK_NEXT) {
          store(a, top);
          if (w0 & kStepPop) top = mine ? sl[p * 64] : top;
          const std::int64_t counter = sl[b * 64];
          store(b, wrap_add(counter, step_word<kGroups>(f.c0, at) ? -1 : 1));
          next = target;
        } else {
          // A loop's test: leaving it charges four units. Leaving lanes
          // bind the arena's first element, which nothing reads.
          const unsigned c0 = step_word<kGroups>(f.c0, at);
          const std::int64_t counter = sl[a * 64], limit = sl[b * 64], xs = sl[p * 64], start = sl[((c0 >> 8) & 31u) * 64];
          const bool more = mine && ((c0 >> 24) != 0 ? counter >= limit : counter < limit);
          const unsigned long long stay = __ballot(more);
          // The counter of a staying lane lies in [0, length).
          store(int(c0 & 31u), arena[more ? (std::uint64_t(xs) >> 16) + std::uint64_t(counter) : 0]);
          store(int((c0 >> 16) & 31u), wrap_add(start, counter));
          mask = stay;
          event = stay != 0 && stay != group ? EV_TEST : EV_NONE;
          next = stay == 0 ? target : next;
          const int refund = stay == 0 ? cost - 4 : 0;
          budget += refund;
          spent -= refund;
        }
      } else if (op < SO_FAIL_TYPE) {
        const std::int64_t counter = sl[a * 64];
        if (op == SO_RANGE_NEXT) {
          store(a, wrap_add(counter, 1));
          next = target;
        } else {
          // Leaving lanes keep the variable, and an unset input unset.
          const std::int64_t limit = sl[b * 64], old = sl[p * 64];
          const bool more = mine && counter < limit;
          const unsigned long long stay = __ballot(more);
          store(p, more ? counter : old);
          sink_slot = stay != 0 ? unsigned(p) : kStepNoSlot;
          mask = stay;
          event = stay != 0 && stay != group ? EV_TEST : EV_NONE;
          next = stay == 0 ? target : next;
          const int refund = stay == 0 ? cost - 4 : 0;
          budget += refund;
          spent -= refund;
        }
      } else {
        event = op == SO_FAIL_TYPE ? EV_FAIL_TYPE : EV_FAIL_VALUE;
      }
      last = at;
      at = next;
    } while (event == EV_NONE && at < stop && budget >= kMost);
    // What ended the run.
    const bool named = (mask >> lane) & 1u;
    const unsigned w0 = step_word<kGroups>(f.w0, last), w1 = step_word<kGroups>(f.w1, last);
    const int target = int(w1 >> 16), refund = int(w0 >> 24) - 4;
    if (mine) {
      ip = at;
      if (event == EV_BRANCH) {
        ip = named ? target : at;
      } else if (event == EV_TEST) {
        ip = named ? at : target;
        fuel += named ? 0 : refund;
      } else if (event != EV_NONE) {
        const bool all = event >= EV_RETURN;
        if (all || named) {
          r.fuel_used = fuel0 - (fuel - spent);
          done = true;
          if (event == EV_RETURN) {
            r.t = std::uint8_t(result_tag);
            if (result_tag == TAG_BOOL) r.b = top != 0;
            else r.v = top;
          } else {
            r.err = event == EV_ZERO_DIV ? ERR_ZERO_DIV : event == EV_FAIL_TYPE ? ERR_TYPE : ERR_VALUE;
          }
        }
      }
      if (unbound && sink_slot < unsigned(n_inputs)) bound |= named || event != EV_TEST ? 1u << sink_slot : 0u;
      fuel -= spent;
    }
    // No lane was charged more than the group.
    low -= unbound ? 0 : spent;
  }
  return r;
}
#endif

}  // namespace gagp_amd
