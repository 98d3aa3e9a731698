// Test driver (CPU only): lowers seeded random programs of a task's grammar,
// decodes them into the looping path's steps (steps.hpp), runs the steps one
// case at a time with the rules vm_steps follows, and compares value, error
// and charged fuel of every case with the C oracle VM on the bytecode, at the
// task's fuel and at every small fuel (each instruction of a joined step is
// then the one that runs out).
//
//   step_decoding TASK.json N
//
// Prints one JSON line: cases compared, mismatches, programs, instructions,
// steps, and how many cases ended in each error.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "grammar.hpp"
#include "steps.hpp"
#include "task.hpp"

extern "C" {
// oracle/vm_oracle.c
typedef struct { std::uint8_t op, has_a, has_b, pad; std::int32_t a, b; } OIns;
typedef struct {
  const OIns* code; std::int32_t code_len;
  const std::uint32_t* fuel;
  const gagp_amd::Val* consts; std::int32_t n_consts;
  std::int32_t n_locals;
} OProg;
int orc_run(const OProg* p, const gagp_amd::Val* inputs, const std::uint8_t* set, int n_inputs, const std::int64_t* arena, int fuel,
            gagp_amd::Val* out, int* fuel_left);
}

using namespace gagp_amd;

namespace {
struct Outcome { int err; std::int64_t value; int left; };

// One case through the steps: vm_steps on a group of one lane.
Outcome run_steps(const std::vector<Step>& steps, int n, const Val* inputs, int K, const std::int64_t* arena, int fuel) {
  std::vector<std::int64_t> slot(std::size_t(step_slots(K)), 0x5a5a5a5a5a5a);
  for (int k = 0; k < K; ++k) slot[std::size_t(k)] = inputs[k].tag == TAG_BOOL ? inputs[k].b : inputs[k].i;
  std::int64_t top = 0;
  for (int at = 0;;) {
    if (at >= n) return {ERR_VALUE, 0, fuel};
    const Step s = steps[std::size_t(at)];
    const int op = int(s.w0 & 63u), cost = int(s.w0 >> 24), sink = int((s.w0 >> 10) & 7u);
    const std::size_t a = s.w1 & 31u, b = (s.w1 >> 5) & 31u, p = (s.w1 >> 10) & 31u, target = s.w1 >> 16;
    const std::uint64_t c = std::uint64_t(s.c);
    const bool reverse = op == SO_WALK_TEST && (c >> 24) != 0;
    const bool test = op == SO_WALK_TEST || op == SO_RANGE_TEST;
    const bool more = test && (reverse ? slot.at(a) >= slot.at(b) : slot.at(a) < slot.at(b));
    const int need = test && !more ? 4 : cost;
    if (fuel < need) return {ERR_TIMEOUT, 0, 0};  // every instruction charges one
    fuel -= need;
    std::size_t next = std::size_t(at) + 1;
    if (op < kStepControl) {
      std::int64_t x = top, y = top, out = 0;
      if (s.w0 & kStepPush) slot.at(p) = top;
      if (s.w0 & kStepX) x = slot.at(a);
      const int yk = int((s.w0 >> 8) & 3u);
      if (yk == 1) y = slot.at(b);
      else if (yk == 2) y = s.c;
      const std::int64_t len = std::int64_t(std::uint64_t(x) & 0xffff), off = std::int64_t(std::uint64_t(x) >> 16);
      switch (op) {
        case SO_MOV: out = y; break;
        case SO_ADD: out = wrap_add(x, y); break;
        case SO_SUB: out = wrap_sub(x, y); break;
        case SO_MUL: out = wrap_mul(x, y); break;
        case SO_MIN: out = std::min(x, y); break;
        case SO_MAX: out = std::max(x, y); break;
        case SO_MOD: if (y == 0) return {ERR_ZERO_DIV, 0, fuel}; out = py_mod(x, y); break;
        case SO_IDIV0: out = y == 0 ? 0 : wrap_div(x, y); break;
        case SO_IMOD0: out = y == 0 ? 0 : py_mod(x, y); break;
        case SO_TDIV0: out = trunc_div0(x, y); break;
        case SO_TMOD0: out = trunc_mod0(x, y); break;
        case SO_INDEX: case SO_INDEX_NONNEG: {
          const std::int64_t k = y < 0 && op == SO_INDEX ? y + len : y;
          if (k < 0 || k >= len) return {ERR_VALUE, 0, fuel};
          out = arena[off + k];
          break;
        }
        case SO_INDEX_CLAMPED: out = len == 0 ? 0 : arena[off + std::min(std::max<std::int64_t>(y, 0), len - 1)]; break;
        case SO_NEG: out = wrap_neg(x); break;
        case SO_ABS: out = x < 0 ? wrap_neg(x) : x; break;
        case SO_LEN: out = len; break;
        case SO_ONE: out = 1; break;
        case SO_CLIP: out = std::min(std::max(x, y), top); break;
        case SO_TEST: out = x != 0; break;
        case SO_NOT: out = x == 0; break;
        case SO_LT: out = x < y; break;
        case SO_LE: out = x <= y; break;
        case SO_GT: out = x > y; break;
        case SO_GE: out = x >= y; break;
        case SO_EQ: out = x == y; break;
        default: out = x != y; break;
      }
      if (sink < SK_IF_FALSE) {
        top = out;
        if (sink == SK_TOP_JUMP) next = target;
      } else {
        if (sink == SK_STORE) slot.at(target) = out;
        else if ((out != 0) == (sink == SK_IF_TRUE)) next = target;
        if (s.w0 & kStepPop) top = slot.at(p);
      }
    } else if (op == SO_JUMP) {
      next = target;
    } else if (op == SO_RETURN) {
      return {ERR_NONE, top, fuel};
    } else if (op == SO_WALK_TEST) {
      if (more) {
        slot.at(c & 31u) = arena[(std::uint64_t(slot.at(p)) >> 16) + std::uint64_t(slot.at(a))];
        slot.at((c >> 16) & 31u) = wrap_add(slot.at((c >> 8) & 31u), slot.at(a));
      } else next = target;
    } else if (op == SO_WALK_NEXT) {
      slot.at(a) = top;
      if (s.w0 & kStepPop) top = slot.at(p);
      slot.at(b) = wrap_add(slot.at(b), c ? -1 : 1);
      next = target;
    } else if (op == SO_RANGE_TEST) {
      if (more) slot.at(p) = slot.at(a);
      else next = target;
    } else if (op == SO_RANGE_NEXT) {
      slot.at(a) = wrap_add(slot.at(a), 1);
      next = target;
    } else {
      return {op == SO_FAIL_TYPE ? ERR_TYPE : ERR_VALUE, 0, fuel};
    }
    at = int(next);
  }
}
}  // namespace

int main(int argc, char** argv) {
  if (argc != 3) { std::fprintf(stderr, "usage: step_decoding TASK.json N\n"); return 2; }
  const Task task = load_task(argv[1]);
  const int n = std::atoi(argv[2]);
  const Grammar g = load_grammar_file(task.grammar_path);
  const Cases cases = load_cases(task.train_path);
  const Layout layout = whole_program_layout(g);
  const PhaseGrammar ph = compile_phase(g, g.entry, g.max_depth, 7, cases.input_names);
  const PhaseView gv{ph.exprs.data(), int(ph.exprs.size()), ph.prods.data(),  int(ph.prods.size()),  ph.nts.data(),
                     int(ph.nts.size()), ph.domains.data(), int(ph.domains.size()), ph.values.data(), int(ph.values.size()),
                     ph.minimum.data(), ph.depth_count,     ph.logical_count,     ph.site_depth ? 1 : 0, ph.root};
  const int R = std::min<int>(kPhaseCapacity, int(layout.max_variable_nodes)), K = int(cases.input_names.size());
  const bool statement = g.nts[g.entry].cat == Cat::Program;
  std::vector<int> origin(static_cast<std::size_t>(R)), site(static_cast<std::size_t>(R));
  std::vector<Val> cval(static_cast<std::size_t>(R));
  std::vector<Ins> code(std::size_t(32 * R + 72));
  std::vector<Val> pool(std::size_t(8 * R + 16));
  long long compared = 0, mismatches = 0, instructions = 0, total_steps = 0, errors[5] = {0, 0, 0, 0, 0};
  int programs = 0;
  for (int i = 0; i < n; ++i) {
    GenResult gen{ST_INVALID, 0, 0, 0};
    for (int attempt = 0; gen.status != ST_OK && attempt < 64; ++attempt) {
      gen = generate_phase(gv, gv.root, 0, int(layout.slot_max_depth), R, 0x2545f4914f6cdd1dull * std::uint64_t(i + 1) + attempt,
                           origin.data(), cval.data(), site.data(), 2 + i % 6);
      if (gen.status == ST_OK && statement && !locals_defined(gv, CRow{origin.data(), site.data(), cval.data(), gen.nodes, gen.constants}))
        gen.status = ST_INVALID;
    }
    if (gen.status != ST_OK) continue;
    const CRow row{origin.data(), site.data(), cval.data(), gen.nodes, gen.constants};
    const LowerResult lr = lower_phase<true>(gv, row, cases.input_types.data(), K, statement ? kStatementType : int(g.nts[g.entry].type),
                                             code.data(), int(code.size()), pool.data(), int(pool.size()));
    if (lr.status != ST_OK || !lr.loop) continue;
    ++programs;
    std::vector<OIns> oc;
    std::vector<std::uint32_t> fuel;
    bool bool_neg = false;
    for (int k = 0; k < lr.code; ++k) {
      const Ins& x = code[std::size_t(k)];
      const bool has_a = x.op == OP_PUSH_CONST || x.op == OP_LOAD || x.op == OP_STORE || jump_op(x.op) || x.op == OP_CALL_BUILTIN;
      oc.push_back(OIns{x.op, std::uint8_t(has_a), std::uint8_t(x.op == OP_CALL_BUILTIN), 0, x.a, x.argc});
      fuel.push_back(x.fuel);
      bool_neg = bool_neg || (x.op == OP_NEG && x.argc == 1);
    }
    const OProg p{oc.data(), std::int32_t(oc.size()), fuel.data(), pool.data(), lr.constants, lr.locals};
    // Lowered code with its tags, then the same code as a caller's, untagged.
    for (int tagged = 1; tagged >= 0; --tagged) {
      if (!tagged && bool_neg) continue;  // the NEG of a Bool is not certified in a caller's code
      std::vector<Ins> in(code.begin(), code.begin() + lr.code);
      if (!tagged)
        for (auto& x : in)
          if (x.op != OP_CALL_BUILTIN) x.argc = 0;
      std::vector<Step> steps(std::size_t(lr.code) + 1);
      const int ns = decode_steps(in.data(), lr.code, pool.data(), K, tagged != 0, steps.data());
      if (tagged) { instructions += lr.code; total_steps += ns; }
      for (int c = 0; c < cases.n; ++c) {
        // Every small fuel on a few cases, the task's fuel on all.
        const int low = c % 16 == i % 16 ? 120 : 0;
        for (int f = 0; f <= low; ++f) {
          const int budget = f == low ? int(g.fuel) : f + 1;
          Val out{};
          int left = 0;
          const int err = orc_run(&p, &cases.inputs[std::size_t(c) * K], &cases.set[std::size_t(c) * K], K, cases.arena.data(), budget,
                                  &out, &left);
          const Outcome r = run_steps(steps, ns, &cases.inputs[std::size_t(c) * K], K, cases.arena.data(), budget);
          const std::int64_t want = out.tag == TAG_BOOL ? out.b : out.i;
          ++compared;
          mismatches += r.err != err || r.left != left || (err == ERR_NONE && r.value != want);
          if (err != ERR_NONE) ++errors[err];
        }
      }
    }
  }
  std::printf("{\"compared\":%lld,\"mismatches\":%lld,\"programs\":%d,\"instructions\":%lld,\"steps\":%lld,\"errors\":[%lld,%lld,%lld,%lld,%lld]}\n",
              compared, mismatches, programs, instructions, total_steps, errors[0], errors[1], errors[2], errors[3], errors[4]);
  return 0;
}
