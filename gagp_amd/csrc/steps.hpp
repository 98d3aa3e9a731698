// Decoded steps of the typed looping path (vm_steps in vm.hpp).
//
// A certified looping program is decoded once, when it is lowered, into
// 16-byte steps: one operator with its operands named (the register top, a
// slot or a constant) and what becomes of its result (the top, the top and a
// jump, a branch on it, a slot). An operand load, the operator that takes it
// and the store, jump or branch that follows run as one step, so a program
// executes about one step per operator instead of one per instruction. Only
// instructions of unit fuel with no jump into their middle are joined, and
// nothing after an operator that can fail (MOD, list indexing), so a case
// that runs out of fuel inside a step fails as it would one instruction at a
// time.
//
// Whether an instruction starts a step depends on its neighbours alone, so
// the device decodes with one lane per instruction (decode_steps_w) and the
// host with a loop (decode_steps).
#pragma once
#include "phase.hpp"

// Inlined into their wavefront callers: a call would cost them the call
// frame's registers.
#if defined(__HIPCC__)
#define STEP_FN __host__ __device__ __attribute__((always_inline)) inline
#else
#define STEP_FN inline
#endif

namespace gagp_amd {

enum StepOp : int {
  // integer results
  SO_MOV = 0, SO_ADD, SO_SUB, SO_MUL, SO_MIN, SO_MAX, SO_MOD, SO_IDIV0, SO_IMOD0, SO_TDIV0, SO_TMOD0, SO_INDEX,
  SO_INDEX_NONNEG, SO_INDEX_CLAMPED, SO_NEG, SO_ABS, SO_LEN, SO_ONE, SO_CLIP,
  // Bool results
  SO_TEST, SO_NOT, SO_LT, SO_LE, SO_GT, SO_GE, SO_EQ, SO_NE,
  // control
  SO_JUMP, SO_RETURN, SO_WALK_TEST, SO_WALK_NEXT, SO_RANGE_TEST, SO_RANGE_NEXT, SO_FAIL_TYPE, SO_FAIL_VALUE,
  SO_NONE,
};
constexpr int kStepBool = SO_TEST, kStepControl = SO_JUMP;
// What becomes of a result: it replaces the top; the same, then a jump; a
// branch when it is false or true; a store into a slot.
enum StepSink : int { SK_TOP = 0, SK_TOP_JUMP, SK_IF_FALSE, SK_IF_TRUE, SK_STORE };

// w0: op [5:0], push the top into slot p first [6], x is slot a (else the
// top) [7], y [9:8] (0 the top, 1 slot b, 2 the constant), sink [12:10], the
// top becomes slot p after a sink that consumed it [13], operand loads that
// are instructions of this step [15:14], charged fuel [31:24].
// w1: a [4:0], b [9:5], p [14:10], jump target step or stored slot [31:16].
// c: the constant; for a fixed loop sequence its further slots (a byte each).
struct alignas(16) Step {
  std::uint32_t w0, w1;
  std::int64_t c;
};
static_assert(sizeof(Step) == 16, "a step is one 16-byte load");
constexpr std::uint32_t kStepPush = 1u << 6, kStepX = 1u << 7, kStepPop = 1u << 13;
constexpr int kStepMax = kLoopCode;  // steps of a program: at most one per instruction
// A step in 8 bytes, as a search keeps it where the instructions were: the
// constant by its pool index (or a WALK_NEXT's direction) in w0 [23:16], which
// a step leaves free; a WALK_TEST's three further slots and direction in w0
// [21:6]. Kept beside the code at 16 bytes each, a search of 8192 list programs
// asked for 164 MB instead of 144, and a server refused some it had admitted.
// Reading them takes a second round trip, for the constants: 13 of 450 us of
// k_eval_loop on 4096 list programs x 200 cases.
static_assert(sizeof(Ins) == sizeof(std::uint64_t) && kLoopPool <= 256, "a packed step replaces an instruction");
STEP_FN std::uint64_t pack_step(const Step& s) {
  const unsigned c = unsigned(std::uint64_t(s.c));
  const unsigned more = (s.w0 & 63u) == unsigned(SO_WALK_TEST) ? (c & 31u) << 6 | (c >> 8 & 31u) << 11 | (c >> 16 & 31u) << 16 | (c >> 24 & 1u) << 21
                                                               : (c & 0xffu) << 16;
  return std::uint64_t(s.w1) << 32 | (s.w0 | more);
}
// The step again, a constant still its pool index.
STEP_FN Step unpack_step(std::uint64_t word) {
  const unsigned lo = unsigned(word);
  const bool walk = (lo & 63u) == unsigned(SO_WALK_TEST);
  const unsigned c = walk ? (lo >> 6 & 31u) | (lo >> 11 & 31u) << 8 | (lo >> 16 & 31u) << 16 | (lo >> 21 & 1u) << 24 : lo >> 16 & 0xffu;
  return Step{lo & (walk ? 0xff00003fu : 0xff00ffffu), unsigned(word >> 32), std::int64_t(c)};
}
// Whether an unpacked step's constant is a pool index.
STEP_FN bool step_indexes(const Step& s) { return (s.w0 & 63u) < unsigned(kStepControl) && (s.w0 >> 8 & 3u) == 2; }
STEP_FN std::int64_t pool_payload(const Val& v) { return v.tag == TAG_BOOL ? std::int64_t(v.b != 0) : v.i; }

// Slots of a lane: the evaluator inputs, the hidden locals, the operand stack's
// elements below the register top, and a spare one for what a lane must not keep.
constexpr int kStepStack = kLoopStack - 1;
STEP_FN int step_slots(int n_inputs) { return n_inputs + kLoopLocals + kStepStack + 1; }

// 256 flags, one per instruction.
struct CodeBits {
  std::uint64_t m[4];
  STEP_FN bool at(int i) const {
    if (i < 0 || i >= 256) return false;
    const std::uint64_t w = i < 128 ? (i < 64 ? m[0] : m[1]) : (i < 192 ? m[2] : m[3]);
    return (w >> (i & 63)) & 1u;
  }
  // Sets [i, i + n).
  STEP_FN void set(int i, int n) {
    for (int k = 0; k < 4; ++k) {
      const int lo = i > 64 * k ? i - 64 * k : 0, hi = i + n < 64 * k + 64 ? i + n - 64 * k : 64;
      if (lo < hi && lo < 64 && hi > 0) m[k] |= (hi - lo >= 64 ? ~0ull : ((1ull << (hi - lo)) - 1)) << lo;
    }
  }
  // Flags set below i.
  STEP_FN int below(int i) const {
    int n = 0;
    for (int k = 0; k < 4; ++k) {
      const int at = i - 64 * k;
      const std::uint64_t w = at >= 64 ? m[k] : at <= 0 ? 0 : m[k] & ((1ull << at) - 1);
#if defined(__HIP_DEVICE_COMPILE__)
      n += __popcll(w);
#else
      n += __builtin_popcountll(w);
#endif
    }
    return n;
  }
};

// The fixed sequences lowering tags (argc of their first instruction): the
// number of instructions, or 0.
STEP_FN int sequence_length(const Ins& x) {
  if (x.op == OP_CALL_BUILTIN || x.op == OP_NEG) return 0;
  switch (x.argc & 0xf0) {
    case kWalkTest: return 12;
    case kWalkNext: return 6;
    case kRangeTest: return 6;
    case kRangeNext: return 5;
    default: return 0;
  }
}
STEP_FN bool jump_op(int op) { return op == OP_JMP || op == OP_JMP_IF_FALSE || op == OP_JMP_IF_TRUE; }

// A program as the decoder sees it. `tagged`: lowered code, whose argc bytes
// carry the sequence tags (and mark the Bool NEG of a failed bound check).
struct StepSource {
  const Ins* code;
  int len;
  const Val* pool;  // null: a step's constant is the pool index
  int n_inputs;
  bool tagged;
  CodeBits target;    // instructions some jump enters
  CodeBits sequence;  // instructions of the fixed sequences
};

STEP_FN Ins step_ins(const StepSource& s, int i) {
  return i >= 0 && i < s.len ? s.code[i] : Ins{255, 0, 0, 0, 0};
}
STEP_FN bool step_leaf(const Ins& x) { return x.op == OP_PUSH_CONST || x.op == OP_LOAD; }
STEP_FN int step_unary(const Ins& x, bool tagged) {
  switch (x.op) {
    case OP_NEG: return tagged && x.argc == 1 ? SO_NONE : SO_NEG;
    case OP_NOT: return SO_NOT;
    case OP_CHECK_INT: return SO_MOV;
    case OP_CALL_BUILTIN: return x.argc != 1 ? SO_NONE : x.a == B_ABS ? SO_ABS : x.a == B_LEN ? SO_LEN : x.a == B_IS_INT ? SO_ONE : SO_NONE;
    default: return SO_NONE;
  }
}
STEP_FN int step_binary(const Ins& x) {
  switch (x.op) {
    case OP_ADD: return SO_ADD;
    case OP_SUB: return SO_SUB;
    case OP_MUL: return SO_MUL;
    case OP_MOD: return SO_MOD;
    case OP_LT: return SO_LT;
    case OP_LE: return SO_LE;
    case OP_GT: return SO_GT;
    case OP_GE: return SO_GE;
    case OP_EQ: return SO_EQ;
    case OP_NE: return SO_NE;
    case OP_CALL_BUILTIN:
      if (x.argc != 2) return SO_NONE;
      switch (x.a) {
        case B_MIN: return SO_MIN;
        case B_MAX: return SO_MAX;
        case B_IDIV0: return SO_IDIV0;
        case B_IMOD0: return SO_IMOD0;
        case B_TRUNC_DIV0: return SO_TDIV0;
        case B_TRUNC_MOD0: return SO_TMOD0;
        case B_INDEX: return SO_INDEX;
        case B_INDEX_NONNEG: return SO_INDEX_NONNEG;
        case B_INDEX_CLAMPED: return SO_INDEX_CLAMPED;
        default: return SO_NONE;
      }
    default: return SO_NONE;
  }
}
// The operator with its operands exchanged, or SO_NONE.
STEP_FN int step_swapped(int op) {
  switch (op) {
    case SO_ADD: case SO_MUL: case SO_MIN: case SO_MAX: case SO_EQ: case SO_NE: return op;
    case SO_LT: return SO_GT;
    case SO_LE: return SO_GE;
    case SO_GT: return SO_LT;
    case SO_GE: return SO_LE;
    default: return SO_NONE;
  }
}
STEP_FN bool step_clip(const Ins& x) { return x.op == OP_CALL_BUILTIN && x.argc == 3 && x.a == B_CLIP; }
// Joinable: unit fuel, not part of a fixed sequence.
STEP_FN bool step_unit(const StepSource& s, const Ins& x, int i) { return x.fuel == 1 && !s.sequence.at(i); }
// Instructions i, i + 1, i + 2 are two operand loads and their operator (one
// of the loads not a constant, and a leading constant only where the operands
// can be exchanged).
STEP_FN bool step_pair(const StepSource& s, const Ins& x, const Ins& y, const Ins& z, int i) {
  if (!step_leaf(x) || !step_leaf(y) || s.target.at(i + 1) || s.target.at(i + 2)) return false;
  const int op = step_binary(z);
  if (op == SO_NONE || !step_unit(s, x, i) || !step_unit(s, y, i + 1) || !step_unit(s, z, i + 2)) return false;
  return x.op == OP_LOAD || (y.op == OP_LOAD && step_swapped(op) != SO_NONE);
}
// Instruction i (`y`) is the operator of the load `x` before it.
STEP_FN bool step_joins(const StepSource& s, const Ins& x, const Ins& y, int i) {
  if (!step_leaf(x) || s.target.at(i) || !step_unit(s, x, i - 1) || !step_unit(s, y, i)) return false;
  return step_binary(y) != SO_NONE || (x.op == OP_LOAD && step_unary(y, s.tagged) != SO_NONE);
}
// Instruction i (`y`) stores, jumps after or branches on the value `x` before it leaves.
STEP_FN bool step_follows(const StepSource& s, const Ins& x, const Ins& y, int i) {
  if (s.target.at(i) || !step_unit(s, x, i - 1) || !step_unit(s, y, i)) return false;
  const int un = step_unary(x, s.tagged), bin = step_binary(x);
  if (bin == SO_MOD || bin == SO_INDEX || bin == SO_INDEX_NONNEG) return false;  // may fail first
  if (y.op == OP_JMP_IF_FALSE || y.op == OP_JMP_IF_TRUE)
    return x.op == OP_LOAD || un == SO_NOT || (bin >= kStepBool && bin < kStepControl);
  return (y.op == OP_JMP || y.op == OP_STORE) && (step_leaf(x) || un != SO_NONE || bin != SO_NONE || step_clip(x));
}
// Whether instruction j starts a step.
STEP_FN bool step_starts(const StepSource& s, int j) {
  const Ins y = step_ins(s, j);
  if (s.sequence.at(j)) return s.tagged && sequence_length(y) != 0;
  const Ins x = step_ins(s, j - 1);
  if (j == 0) return true;
  if (step_joins(s, x, y, j) || step_follows(s, x, y, j)) return false;
  return !(step_leaf(y) && step_pair(s, x, y, step_ins(s, j + 1), j - 1));
}

// The step that starts at instruction j; `starts` flags every start, `n` is
// their number (a jump to the end of the code targets step n).
STEP_FN Step step_at(const StepSource& s, int j, const CodeBits& starts, int n) {
  const Ins i0 = step_ins(s, j), i1 = step_ins(s, j + 1), i2 = step_ins(s, j + 2);
  const int K = s.n_inputs, stack = K + kLoopLocals, sp = i0.sp;
  const auto slot_of = [&](int a) { return unsigned(a < 0 ? 0 : a < K + kLoopLocals ? a : 0); };
  const auto element = [&](int k) { return unsigned(stack + (k < 0 ? 0 : k < kStepStack ? k : kStepStack - 1)); };
  const auto step_of = [&](int t) { return unsigned(t >= s.len ? n : starts.below(t)); };
  const auto constant = [&](const Ins& x) {
    return s.pool ? pool_payload(s.pool[x.a]) : std::int64_t(x.a);
  };
  const auto pack = [](unsigned op, unsigned flags, unsigned y, unsigned sink, unsigned loads, unsigned cost) {
    return op | flags | y << 8 | sink << 10 | loads << 14 | cost << 24;
  };
  Step out{0, 0, 0};
  if (s.sequence.at(j)) {
    const bool reverse = (i0.argc & 3) == 2;
    const unsigned a0 = slot_of(i0.a), b0 = slot_of(i1.a);
    switch (i0.argc & 0xf0) {
      case kWalkTest: {  // counter, bound; list; exit; element, start, index
        out.w0 = pack(SO_WALK_TEST, 0, 0, 0, 0, 12);
        out.w1 = a0 | b0 << 5 | slot_of(step_ins(s, j + 4).a) << 10 | step_of(step_ins(s, j + 3).a) << 16;
        out.c = std::int64_t(slot_of(step_ins(s, j + 7).a) | slot_of(step_ins(s, j + 8).a) << 8 | slot_of(step_ins(s, j + 11).a) << 16 |
                             unsigned(reverse) << 24);
        break;
      }
      case kWalkNext: {  // state, counter; the element below the stored state; head
        out.w0 = pack(SO_WALK_NEXT, sp >= 2 ? kStepPop : 0, 0, 0, 0, 6);
        out.w1 = a0 | b0 << 5 | element(sp - 2) << 10 | step_of(step_ins(s, j + 5).a) << 16;
        out.c = reverse;
        break;
      }
      case kRangeTest: {  // counter, bound; variable; exit
        out.w0 = pack(SO_RANGE_TEST, 0, 0, 0, 0, 6);
        out.w1 = a0 | b0 << 5 | slot_of(step_ins(s, j + 5).a) << 10 | step_of(step_ins(s, j + 3).a) << 16;
        break;
      }
      default: {  // kRangeNext: counter; head
        out.w0 = pack(SO_RANGE_NEXT, 0, 0, 0, 0, 5);
        out.w1 = a0 | step_of(step_ins(s, j + 4).a) << 16;
        break;
      }
    }
    return out;
  }
  int op = SO_NONE, next = j + 1;  // next: the instruction after the value
  unsigned flags = 0, y = 0, loads = 0, a = 0, b = 0, p = 0;
  bool leaves = false;  // the operands are loads: the top is untouched unless the result replaces it
  int left = 0;         // operands on the stack below a consumed top: the new top's element index + 1
  std::int64_t c = 0;
  const auto second = [&](const Ins& x) {
    if (x.op == OP_LOAD) { y = 1; b = slot_of(x.a); }
    else { y = 2; c = constant(x); }
  };
  if (step_leaf(i0)) {
    if (step_pair(s, i0, i1, i2, j)) {
      leaves = true;
      loads = 2;
      op = step_binary(i2);
      if (i0.op == OP_LOAD) { a = slot_of(i0.a); second(i1); }
      else { loads = 3; op = step_swapped(op); a = slot_of(i1.a); second(i0); }
      flags = kStepX;
      next = j + 3;
    } else if (step_joins(s, i0, i1, j + 1)) {
      loads = 1;
      next = j + 2;
      op = step_binary(i1);
      if (op != SO_NONE) { second(i0); left = sp - 1; }
      else {
        leaves = true;
        op = step_unary(i1, s.tagged);
        flags = kStepX;
        a = b = slot_of(i0.a);
        y = op == SO_MOV ? 1 : 0;
      }
    } else {
      leaves = true;
      op = SO_MOV;
      second(i0);
    }
  } else if ((op = step_binary(i0)) != SO_NONE) {
    flags = kStepX;
    a = element(sp - 2);
    left = sp - 2;
  } else if ((op = step_unary(i0, s.tagged)) != SO_NONE) {
    left = sp - 1;
  } else if (step_clip(i0)) {
    op = SO_CLIP;
    flags = kStepX;
    a = element(sp - 3);
    y = 1;
    b = element(sp - 2);
    left = sp - 3;
  }
  if (op != SO_NONE) {
    unsigned sink = SK_TOP, target = 0;
    unsigned cost = 0;
    for (int k = j; k < next; ++k) cost += step_ins(s, k).fuel;
    const Ins f = step_ins(s, next);
    if (next < s.len && step_follows(s, step_ins(s, next - 1), f, next)) {
      cost += f.fuel;
      if (f.op == OP_STORE) { sink = SK_STORE; target = slot_of(f.a); }
      else {
        sink = f.op == OP_JMP ? SK_TOP_JUMP : f.op == OP_JMP_IF_FALSE ? SK_IF_FALSE : SK_IF_TRUE;
        target = step_of(f.a);
        if (sink != SK_TOP_JUMP && op == SO_MOV) { op = SO_TEST; flags |= kStepX; a = b; y = 0; }  // a loaded Bool
      }
    }
    if (sink == SK_TOP || sink == SK_TOP_JUMP) {
      if (leaves && sp > 0) { flags |= kStepPush; p = element(sp - 1); }
    } else if (!leaves && left > 0) {
      flags |= kStepPop;
      p = element(left - 1);
    }
    out.w0 = pack(unsigned(op), flags, y, sink, loads, cost);
    out.w1 = a | b << 5 | p << 10 | target << 16;
    out.c = c;
    return out;
  }
  // A store, jump or return of its own.
  const unsigned cost = i0.fuel, pop = sp >= 2 ? unsigned(kStepPop) : 0u;
  switch (i0.op) {
    case OP_STORE:
      out.w0 = pack(SO_MOV, pop, 0, SK_STORE, 0, cost);
      out.w1 = element(sp - 2) << 10 | slot_of(i0.a) << 16;
      break;
    case OP_JMP_IF_FALSE: case OP_JMP_IF_TRUE:
      out.w0 = pack(SO_TEST, pop, 0, i0.op == OP_JMP_IF_FALSE ? SK_IF_FALSE : SK_IF_TRUE, 0, cost);
      out.w1 = element(sp - 2) << 10 | step_of(i0.a) << 16;
      break;
    case OP_JMP:
      out.w0 = pack(SO_JUMP, 0, 0, 0, 0, cost);
      out.w1 = step_of(i0.a) << 16;
      break;
    case OP_RETURN: out.w0 = pack(SO_RETURN, 0, 0, 0, 0, cost); break;
    case OP_NEG: out.w0 = pack(SO_FAIL_TYPE, 0, 0, 0, 0, cost); break;  // the NEG of a Bool
    default: out.w0 = pack(SO_FAIL_VALUE, 0, 0, 0, 0, cost); break;
  }
  return out;
}

// Host decoding of a certified looping program of at most kLoopCode
// instructions; returns the number of steps written.
inline int decode_steps(const Ins* code, int len, const Val* pool, int n_inputs, bool tagged, Step* out) {
  StepSource s{code, len, pool, n_inputs, tagged, {{0, 0, 0, 0}}, {{0, 0, 0, 0}}};
  for (int i = 0; i < len; ++i) {
    if (jump_op(code[i].op)) s.target.set(code[i].a, 1);
    if (tagged && !s.sequence.at(i) && sequence_length(code[i])) s.sequence.set(i, sequence_length(code[i]));
  }
  CodeBits starts{{0, 0, 0, 0}};
  for (int j = 0; j < len; ++j)
    if (step_starts(s, j)) starts.set(j, 1);
  const int n = starts.below(len);
  for (int j = 0, k = 0; j < len; ++j)
    if (starts.at(j)) out[k++] = step_at(s, j, starts, n);
  return n;
}

#if defined(__HIPCC__)
// Lowered code to packed steps by one wavefront, a lane per instruction.
// `out` may be the code itself: the steps of 64 instructions are stored when
// every lane has them, and replace none that a later one reads.
__device__ __attribute__((always_inline)) inline int decode_steps_w(const Ins* code, int len, int n_inputs, std::uint64_t* out) {
  const int lane = int(threadIdx.x & 63u);
  StepSource s{code, len, nullptr, n_inputs, true, {{0, 0, 0, 0}}, {{0, 0, 0, 0}}};
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    if (64 * g >= len) break;
    const Ins x = step_ins(s, 64 * g + lane);
    const bool in = 64 * g + lane < len;
    for (std::uint64_t m = __ballot(in && jump_op(x.op)); m; m &= m - 1)
      s.target.set(__builtin_amdgcn_readlane(x.a, __ffsll((long long)m) - 1), 1);
    const int length = in ? sequence_length(x) : 0;
    for (std::uint64_t m = __ballot(length != 0); m; m &= m - 1) {
      const int i = __ffsll((long long)m) - 1;
      // A tag inside a sequence is an operand's, never a start.
      if (!s.sequence.at(64 * g + i)) s.sequence.set(64 * g + i, __builtin_amdgcn_readlane(length, i));
    }
  }
  CodeBits starts{{0, 0, 0, 0}};
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    if (64 * g >= len) break;
    const int j = 64 * g + lane;
    starts.m[g] = __ballot(j < len && step_starts(s, j));
  }
  const int n = starts.below(len);
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    if (64 * g >= len) break;
    const int j = 64 * g + lane;
    const bool mine = j < len && starts.at(j);
    const std::uint64_t word = mine ? pack_step(step_at(s, j, starts, n)) : 0;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    __builtin_amdgcn_wave_barrier();
    if (mine) out[starts.below(j)] = word;
  }
  return n;
}
#endif

}  // namespace gagp_amd
