// Test driver (CPU only): lowers seeded random programs of a grammar and says
// how many the lowering sends to the looping path, and whether the grammar is
// known to (leaves_straight_line), as a search asks before it prepares that path.
//
//   looping_grammar TASK.json N
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "grammar.hpp"
#include "phase.hpp"
#include "task.hpp"

using namespace gagp_amd;

int main(int argc, char** argv) {
  if (argc != 3) { std::fprintf(stderr, "usage: looping_grammar TASK.json N\n"); return 2; }
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
  int lowered = 0, looping = 0;
  for (int i = 0; i < n; ++i) {
    const GenResult gen = generate_phase(gv, gv.root, 0, int(layout.slot_max_depth), R, 0x2545f4914f6cdd1dull * std::uint64_t(i + 1),
                                         origin.data(), cval.data(), site.data(), 2 + i % 6);
    if (gen.status != ST_OK) continue;
    const LowerResult r = lower_phase<true>(gv, CRow{origin.data(), site.data(), cval.data(), gen.nodes, gen.constants},
                                            cases.input_types.data(), K, statement ? kStatementType : int(g.nts[g.entry].type), code.data(),
                                            int(code.size()), pool.data(), int(pool.size()));
    lowered += r.status == ST_OK;
    looping += r.status == ST_OK && r.loop;
  }
  std::printf("{\"lowered\":%d,\"looping\":%d,\"leaves\":%d}\n", lowered, looping,
              int(leaves_straight_line(ph, cases.input_types, layout, R, statement)));
  return 0;
}
