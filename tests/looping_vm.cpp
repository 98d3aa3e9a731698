// Test driver (CPU only): the looping path's VM itself (vm_steps in vm.hpp)
// on one lane (tests/one_lane), with cases that leave inputs unset.
//
//   looping_vm TASK.json N
//     lowers and decodes N seeded random programs of the task's grammar, packs
//     and unpacks their steps, runs every train case with every subset of the inputs unset, at the task's
//     fuel and on a few cases at every small fuel, and compares value, error
//     and charged fuel with the C oracle VM on the bytecode.
//   looping_vm division
//     compares the 32-bit quotient path with the host's 64-bit one.
//
// Prints one JSON line.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "grammar.hpp"
#include "task.hpp"
#include "vm.hpp"

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

namespace gagp_amd {
// The wavefront holds step k in lane k % 64 of a register; one lane has them here.
static Step steps_of_lane[kStepMax];
static StepProgram program_of_lane;
static unsigned word_of_lane(const unsigned (&v)[4], int k) {
  const Step& s = steps_of_lane[k];
  return &v == &program_of_lane.w0 ? s.w0 : &v == &program_of_lane.w1 ? s.w1
         : &v == &program_of_lane.c0 ? unsigned(std::uint64_t(s.c)) : unsigned(std::uint64_t(s.c) >> 32);
}
template <> inline unsigned step_word<1>(const unsigned (&v)[4], int k) { return word_of_lane(v, k); }
template <> inline unsigned step_word<4>(const unsigned (&v)[4], int k) { return word_of_lane(v, k); }
}  // namespace gagp_amd

using namespace gagp_amd;

namespace {
int division() {
  std::vector<std::int64_t> edge{0};
  for (int bit = 0; bit < 34; ++bit)
    for (int d = -1; d <= 1; ++d) {
      edge.push_back((std::int64_t(1) << bit) + d);
      edge.push_back(-(std::int64_t(1) << bit) + d);
    }
  for (std::int64_t v : {3LL, 7LL, 10LL, 46340LL, 46341LL, 65537LL, 1000003LL, 1431655765LL, 2147483629LL}) {
    edge.push_back(v);
    edge.push_back(-v);
  }
  edge.push_back(INT64_MAX);
  edge.push_back(INT64_MIN);
  long long compared = 0, mismatches = 0;
  for (double error : {0.0, 0x1p-23, -0x1p-23}) {
    reciprocal_error = error;
    for (std::int64_t x : edge)
      for (std::int64_t y : edge) {
        const std::int64_t want[5] = {y == 0 ? 0 : py_mod(x, y), y == 0 ? 0 : py_mod(x, y), y == 0 ? 0 : wrap_div(x, y), trunc_div0(x, y),
                                      trunc_mod0(x, y)};
        const int ops[5] = {SO_MOD, SO_IMOD0, SO_IDIV0, SO_TDIV0, SO_TMOD0};
        for (int k = 0; k < 5; ++k) {
          ++compared;
          mismatches += step_divide(ops[k], x, y) != want[k];
        }
      }
  }
  std::printf("{\"compared\":%lld,\"mismatches\":%lld}\n", compared, mismatches);
  return 0;
}
}  // namespace

int main(int argc, char** argv) {
  if (argc == 2 && !std::strcmp(argv[1], "division")) return division();
  if (argc != 3) { std::fprintf(stderr, "usage: looping_vm TASK.json N | division\n"); return 2; }
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
  std::vector<std::int64_t> slots(std::size_t(64 * step_slots(K)));
  long long compared = 0, mismatches = 0, errors[5] = {0, 0, 0, 0, 0};
  int programs = 0, repacked = 0;
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
    for (int k = 0; k < lr.code; ++k) {
      const Ins& x = code[std::size_t(k)];
      const bool has_a = x.op == OP_PUSH_CONST || x.op == OP_LOAD || x.op == OP_STORE || jump_op(x.op) || x.op == OP_CALL_BUILTIN;
      oc.push_back(OIns{x.op, std::uint8_t(has_a), std::uint8_t(x.op == OP_CALL_BUILTIN), 0, x.a, x.argc});
      fuel.push_back(x.fuel);
    }
    const OProg p{oc.data(), std::int32_t(oc.size()), fuel.data(), pool.data(), lr.constants, lr.locals};
    // The steps as a search keeps them: packed, the constants by pool index.
    program_of_lane.n = decode_steps(code.data(), lr.code, nullptr, K, true, steps_of_lane);
    for (int k = 0; k < program_of_lane.n; ++k) {
      Step& s = steps_of_lane[k];
      const Step again = unpack_step(pack_step(s));
      repacked += again.w0 != s.w0 || again.w1 != s.w1 || again.c != s.c;
      s = again;
      if (step_indexes(s)) s.c = pool_payload(pool[std::size_t(s.c)]);
    }
    for (int c = 0; c < cases.n; ++c)
      for (unsigned bound = 0; bound < 1u << K; ++bound) {
        std::uint8_t set[kFastInputs] = {};
        FastInputs in{0, 0, 0, 0, bound};
        std::int64_t* const v[kFastInputs] = {&in.v0, &in.v1, &in.v2, &in.v3};
        for (int k = 0; k < K; ++k) {
          const Val& x = cases.inputs[std::size_t(c) * K + k];
          set[k] = bound >> k & 1u;
          if (set[k]) *v[k] = x.tag == TAG_BOOL ? x.b : x.i;
        }
        const int low = c % 16 == i % 16 ? 120 : 0;
        for (int f = 0; f <= low; ++f) {
          const int budget = f == low ? int(g.fuel) : f + 1;
          Val out{};
          int left = 0;
          const int err = orc_run(&p, &cases.inputs[std::size_t(c) * K], set, K, cases.arena.data(), budget, &out, &left);
          std::fill(slots.begin(), slots.end(), 0x5a5a5a5a5a5a);
          const LaneResult r = (program_of_lane.n <= 64 ? vm_steps<1> : vm_steps<4>)(program_of_lane, in, K, cases.arena.data(), slots.data(), 0,
                                                                                     true, budget, lr.result_type);
          const std::int64_t want = out.tag == TAG_BOOL ? out.b : out.i, got = r.t == TAG_BOOL ? r.b : r.v;
          ++compared;
          mismatches += r.err != err || budget - r.fuel_used != left || (err == ERR_NONE && (got != want || r.t != out.tag));
          if (err != ERR_NONE) ++errors[err];
        }
      }
  }
  std::printf("{\"compared\":%lld,\"mismatches\":%lld,\"programs\":%d,\"repacked\":%d,\"errors\":[%lld,%lld,%lld,%lld,%lld]}\n", compared, mismatches, programs,
              repacked, errors[0], errors[1], errors[2], errors[3], errors[4]);
  return 0;
}
