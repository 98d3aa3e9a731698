// Device-resident search engine for gfx950 (see engine.hpp).
//
// One steady-state round (cpp/src/evolution/evolve.cpp:331-441 with the owner
// bodies of cpp/src/evolution/repro/gpu/phase_population_cpu.cpp:314-394) is
// the kernel sequence
//   k_record  history row of generation r/per_epoch (best row, fitness vector)
//   k_vary    tournaments, crossover, mutation, compare, completed-result
//             reuse through the member table, lowering, pending lists
//             (wavefront/child); k_lower lowers what it leaves
//   k_eval    the bytecode VMs + canonical reduction (k_eval, k_eval_tiles,
//             k_eval_loop with k_loop_finish)
//   k_place   mt19937_64 inverse-tournament placement (block/search), with
//             k_clear emptying the member table beside it
//   k_commit  placed children overwrite their members; every member is
//             indexed in the next round's table (wavefront/member)
// over every search of a batch (grid.y = search). Nothing returns to the
// host between rounds.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <fstream>
#include <functional>
#include <numeric>
#include <sstream>
#include <stdexcept>

#include "engine.hpp"
#include "parallel.hpp"
#include "population.hpp"
#include "vary_wave.hpp"
#include "vm.hpp"

namespace gagp_amd {

// The runtime keeps a failed call's error until it is asked for: taken here, it
// is not met again by the check after a later launch.
#define HIP_OK(expr)                                                                                 \
  do {                                                                                               \
    const hipError_t e_ = (expr);                                                                    \
    if (e_ != hipSuccess) {                                                                          \
      (void)hipGetLastError();                                                                       \
      throw std::runtime_error(std::string("HIP error: ") + hipGetErrorString(e_) + " at " #expr);   \
    }                                                                                                \
  } while (0)

namespace {

constexpr int kWavesPerBlock = 4;
constexpr std::size_t kLdsLimit = 160 * 1024;  // of a block
constexpr int kScoreCases = 4096;  // largest case count with an LDS score buffer per wavefront
constexpr int kEvalThreads = 64 * kWavesPerBlock;

struct Counters {
  // Evaluated programs and program-cases, runtime errors, timeouts, VM
  // instructions executed (charged fuel), instructions of the evaluated
  // programs and their constant-pool entries; when profiling, the children
  // made, their nodes and constants, the nodes and constants of the parent
  // and donor rows they read, and the instructions and pool entries lowered
  // for them.
  unsigned long long programs, program_cases, errors, timeouts, vm_instructions, code_words, pool_words;
  unsigned long long children, child_nodes, child_consts, parent_nodes, parent_consts, child_code_words, child_pool_words;
};

// Totals of one program's tile groups in the looping kernel (device atomics),
// taken and cleared by k_loop_finish.
struct alignas(16) LoopAcc {
  unsigned long long sum;   // of the integral scores, two's complement
  unsigned long long fuel;  // charged fuel
  unsigned wrong, errors, timeouts, fractional;
};
// Device state of one search. Every pointer is device memory owned by the
// host Search object.

struct DSearch {
  int active;
  int P, B, R, code_cap, pool_cap, stack_slots;
  int rounds, per_epoch;
  int fuel, lanes;
  double penalty;
  Policy policy;
  int pressure, replacement_size;
  double p_mut;
  OpPolicy pol;
  SlotInfo slot;
  int fixed_nodes, grammar_sites, has_wrong, expected_type, n_locals, site_depth;
  std::uint64_t seed;
  PhaseTables g;
  int stage_tables;  // the phase tables fit the reproduction kernel's LDS
  GAS const std::uint8_t* local_types;
  CaseData cd;
  GAS int *cur_origin, *cur_site, *cur_n, *cur_nc;
  GAS Val* cur_cval;
  GAS int *x_origin, *x_site, *x_n, *x_nc;
  GAS Val* x_cval;
  GAS int *t_origin, *t_site;
  GAS Val* t_cval;
  GAS int *s_origin, *s_site;
  GAS Val* s_cval;
  GAS double* fitness;
  GAS unsigned *wrong, *nodes;
  GAS OpStats* stats;
  GAS int* reuse;    // the member whose result the child takes, -1, or -2 until k_lower has lowered the child
  GAS double* c_fit;
  GAS unsigned *c_wrong, *c_nodes;
  GAS Ins* code;     // of a program of the looping path its packed steps, in the same words
  GAS Val* pool;
  GAS int *code_len, *pool_len, *code_jumps;  // code_jumps: flags, and the number of packed steps << 8
  GAS std::uint64_t* child_hash;
  // pending[2B]: children to score, general ones from the front of [0, B),
  // vm_fast ones from its back, vm_steps ones in [B, 2B); n_pending[3] counts each.
  GAS int *pending, *n_pending;
  GAS std::uint64_t* table_key;  // genotype hash | 1, 0 = empty
  GAS int* table;                // a member with that hash
  int table_mask;
  GAS std::uint64_t* mt;      // std::mt19937_64 state after its last twist
  GAS std::uint64_t* mt_left; // tempered words generated and not yet consumed
  GAS int* n_left;
  int place_lds;          // placement keys fit in LDS
  GAS std::uint64_t* member_hash;
  GAS std::uint64_t* round_seed;
  GAS int *round, *best, *placed;
  GAS int *hist_origin, *hist_n, *hist_nc;
  GAS Val* hist_cval;
  GAS double *hist_fit, *hist_all;
  GAS unsigned* hist_wrong;
  GAS Counters* counters;
  GAS int* error;
  GAS unsigned *e_errors, *e_timeouts;  // per evaluated slot
  GAS unsigned long long* e_fuel;
  int profile;  // tally reproduction row sizes too
  int generational, elites;  // generational schedule (B = P, one round per generation) and its elite count
  int early_exit;            // stop at the first generation boundary whose best member has no wrong case
  GAS int* stop;             // generations completed when it stopped early, else 0
  GAS int* elite;            // elite members of the current generation, best first
  int temp_slots;      // hidden-local slots per lane of the general VM (temporaries, grammar locals, input shadows)
  int input_shadow;    // the last input_shadow of them shadow stored inputs (statement input targets), else 0
  int defer;           // programs may leave the straight-line VM: k_lower lowers what lower_row does not
  int walks;           // the grammar has traversals: lowering runs the kWalks instantiations
  int imported;        // the initial population is uploaded, not generated
  // Selection values of a caller-driven round (the owner seam): tournaments
  // compare them alone; null in the engine's own rounds.
  GAS const double* select;
  int general_scores;  // the general evaluation kernel has an LDS score buffer for this search
  GAS double* loop_scores;  // the looping kernel's case scores: C per program slot
  GAS LoopAcc* loop_acc;    // the looping kernel's totals per program slot (zero between evaluations)
  int looping;              // the search has the looping path: its programs' packed steps replace their code
  int stage_cases;     // the typed evaluation kernel stages the case set in LDS
  int typed_tiles;     // typed programs go to k_eval_tiles (more than one 64-case tile, C <= kScoreCases)
};

__device__ inline CRow member_row(const DSearch& d, int m) {
  const std::size_t o = std::size_t(m) * d.R;
  return CRow{d.cur_origin + o, d.cur_site + o, d.cur_cval + o, d.cur_n[m], d.cur_nc[m]};
}
__device__ inline CRow child_row(const DSearch& d, int c) {
  const std::size_t o = std::size_t(c) * d.R;
  return CRow{d.x_origin + o, d.x_site + o, d.x_cval + o, d.x_n[c], d.x_nc[c]};
}
__device__ inline bool search_live(const DSearch& d) { return d.active && *d.round < d.rounds && !*d.error && !*d.stop; }
__device__ inline void raise(const DSearch& d, int code) { atomicCAS(d.error, 0, code); }

// One entry per launched block of a batch kernel: its search, its block
// index within that search's share and the share's size. Batches launch a
// flat grid of exactly the blocks their searches need (no padding to the
// largest search).
struct BlockMap { int search, block, blocks; };

// Wavefronts (rows) per block of the row kernels. Eight share one LDS copy of
// the phase tables: with four, the list grammar's tables (21 KB a block) left
// room for 28 wavefronts per CU where a population of 8192 brings 32, and the
// last eighth of the children started 100 us late.
constexpr int kVaryWaves = 8;

// ---- initial population (phase_population_cpu.cpp:54-113) ----
// One wavefront per member runs the derivation uniformly (as mutation does),
// so members with different retry counts do not diverge within a wavefront.
// kStaged as k_vary.
template <bool kStaged>
__global__ __launch_bounds__(64 * kVaryWaves) void k_init_pop(DSearch* all, const BlockMap* map) {
  const BlockMap bm = map[blockIdx.x];
  const DSearch& d = all[bm.search];
  if (!d.active || d.imported || (d.stage_tables != 0) != kStaged) return;  // uniform per block
  extern __shared__ __attribute__((aligned(16))) unsigned char vary_lds[];
  const PhaseView g = kStaged ? stage_phase_tables<64 * kVaryWaves>(d.g, vary_lds) : view_of(d.g);
  const int m = bm.block * kVaryWaves + wave_index();
  if (m >= d.P) return;
  const int sd = d.site_depth;
  const int ramp = sd < 2 ? sd : 2 + m % (sd - 1);
  const std::size_t o = std::size_t(m) * d.R;
  GenResult gen{ST_INVALID, 0, 0, 0};
  const int room = d.slot.max_variable_nodes < kPhaseCapacity ? d.slot.max_variable_nodes : kPhaseCapacity;
  for (int logical = ramp, attempt = 0; gen.status != ST_OK; ++attempt) {
    if (room <= 0 || room > d.R) { raise(d, 101); return; }
    const std::uint64_t s = splitmix_mix(d.seed ^ splitmix_mix((std::uint64_t(m) * 8 + 0) * 64 + std::uint64_t(attempt)));
    gen = derive_phase_w(g, g.root, 0, d.slot.max_depth, room, s, d.cur_origin + o, d.cur_cval + o, d.cur_site + o, logical);
    // A statement program may read an unassigned local: the next seed is tried.
    if (gen.status == ST_OK && d.slot.statement &&
        !locals_defined_w(g, CRow{d.cur_origin + o, d.cur_site + o, d.cur_cval + o, gen.nodes, gen.constants}))
      gen.status = ST_INVALID;
    if (gen.status != ST_OK && attempt % 4 == 3 && logical < sd) ++logical;
    if (attempt >= 256) { raise(d, 102); return; }
  }
  if (wlane() == 0) {
    d.cur_n[m] = gen.nodes;
    d.cur_nc[m] = gen.constants;
    d.placed[m] = -1;
  }
}

// ---- lowering: one wavefront per row ----
// Records the lowering `r` of a slot, whose code is in the slot or, where
// `kept` is not null, in this wavefront's LDS: a looping program's is decoded
// into the slot, any other stands there. Returns the code flags it stores
// (code_jumps).
__device__ __attribute__((always_inline)) inline int store_lowered(const DSearch& d, int slot, const LowerResult& r,
                                                                   const Ins* kept = nullptr) {
  Ins* const code = d.code + std::size_t(slot) * d.code_cap;
  const bool ok = r.status == ST_OK && r.stack_bound >= 1 && r.stack_bound <= d.stack_slots &&
                   r.locals - d.n_locals <= d.temp_slots - d.input_shadow;
  const bool steps = ok && r.loop && d.looping;
  int n = 0;
  if (steps) {
    if (!kept) wave_fence();  // the code stored above is read across the lanes
    n = decode_steps_w(kept ? kept : code, r.code, d.n_locals, reinterpret_cast<std::uint64_t*>(code));
  } else if (kept) {
    for (int k = wlane(); k < r.code; k += 64) code[k] = kept[k];
  }
  // bit 0: jumps; bit 1: typed straight-line (vm_fast); bit 2: Bool result; bit 3: typed looping (vm_steps, where
  // the search has that path; else the general VM scores the program)
  const int flags = r.jumps | (r.fast ? 2 : 0) | (r.result_type == TAG_BOOL ? 4 : 0) | (steps ? 8 : 0) | n << 8;
  if (wlane() == 0) {
    if (!ok) raise(d, 200 + r.status);
    d.code_len[slot] = ok ? r.code : 0;
    d.pool_len[slot] = ok ? r.constants : 0;
    d.code_jumps[slot] = flags;
  }
  return flags;
}
// The node-by-node lowering of `row`, in memory, into `slot` (`source`: its
// origins and constants, read into registers as they are needed). kWalks: the
// instantiation with traversals (grammars that have them).
template <bool kWalks>
__device__ __attribute__((always_inline)) inline LowerResult lower_into_w(const PhaseView& g, const DSearch& d, const CRow& row, int slot,
                                                                          WaveOrigins& source, WalkStore<kWalks>& ws) {
  return lower_phase_w<kWalks>(g, row, d.local_types, d.n_locals, d.expected_type, d.code + std::size_t(slot) * d.code_cap, d.code_cap,
                               d.pool + std::size_t(slot) * d.pool_cap, d.pool_cap, source, ws);
}
template <bool kWalks>
__global__ __launch_bounds__(64 * kVaryWaves) void k_lower_members(DSearch* all, const BlockMap* map) {
  const BlockMap bm = map[blockIdx.x];
  const DSearch& d = all[bm.search];
  const int m = bm.block * kVaryWaves + wave_index();
  if (!d.active || (d.walks != 0) != kWalks || m >= d.P || *d.error) return;
  __shared__ LaneStore<true> row_lds[kVaryWaves];
  __shared__ WalkStore<kWalks> walk_lds[kVaryWaves];
  LaneStore<true>& store = row_lds[wave_index()];
  const PhaseView g = view_of(d.g);
  const CRow row = member_row(d, m);
  LowerResult lowered;
  WaveGrammar w;
  bool done = false;
  if (d.R <= kWaveRow && wave_grammar(g, w)) {
    const std::size_t o = std::size_t(m) * d.R;
    const WaveRow r = load_row(d.cur_origin + o, d.cur_site + o, d.cur_cval + o, d.R, row.n, row.nc);
    done = (!d.slot.statement || locals_defined_row(g, w, r)) &&
           lower_row<true>(w, r, d.local_types, d.n_locals, d.expected_type, d.code + std::size_t(m) * d.code_cap, d.code_cap,
                           d.pool + std::size_t(m) * d.pool_cap, d.pool_cap, (LAS LaneStore<true>*)&store, lowered);
  }
  if (!done) {
    WaveOrigins source{row};
    lowered = lower_into_w<kWalks>(g, d, row, m, source, walk_lds[wave_index()]);
  }
  if (done) store_lowered(d, m, lowered, store.code);
  else store_lowered(d, m, lowered);
}

// ---- member hash table (parent_fitness_cache.cuh:11-58) ----
// One entry per distinct genotype hash: identical members share a hash, and
// any one of them carries the result a child identical to them reuses (the
// rows are compared in full before a result is reused). Keys are hash | 1,
// 0 marks an empty slot. A round reads the table its previous round's
// commit built (the initialization builds the first); it is cleared while
// the previous round places its children.
__global__ void k_clear(DSearch* all, const BlockMap* map) {
  const BlockMap bm = map[blockIdx.x];
  const DSearch& d = all[bm.search];
  const int i = bm.block * blockDim.x + threadIdx.x;
  if (!d.active || i > d.table_mask) return;
  d.table_key[i] = 0;
}
// Indexes member m under hash h (one thread).
__device__ inline void insert_member(const DSearch& d, int m, std::uint64_t h) {
  const std::uint64_t key = h | 1;
  for (int probe = 0; probe <= d.table_mask; ++probe) {
    const int slot = int((h + std::uint64_t(probe)) & std::uint64_t(d.table_mask));
    const unsigned long long seen = atomicCAS(reinterpret_cast<unsigned long long*>(d.table_key) + slot, 0ull, key);
    if (seen == 0) { d.table[slot] = m; return; }
    if (seen == key) return;  // a member with this hash is indexed
  }
  raise(d, 400);
}
__global__ void k_index(DSearch* all, const BlockMap* map) {
  const BlockMap bm = map[blockIdx.x];
  const DSearch& d = all[bm.search];
  const int m = bm.block * blockDim.x + threadIdx.x;
  if (!search_live(d) || m >= d.P) return;
  insert_member(d, m, d.member_hash[m]);
}
// The member a child identical to it reuses, or -1: the table probe is
// uniform and the row comparison runs across the lanes (rows_equal's test).
__device__ inline int find_member_w(const DSearch& d, const CRow& child, std::uint64_t h) {
  const std::uint64_t key = h | 1;
  for (int probe = 0; probe <= d.table_mask; ++probe) {
    const int slot = int((h + std::uint64_t(probe)) & std::uint64_t(d.table_mask));
    const std::uint64_t k = d.table_key[slot];
    if (k == 0) return -1;
    if (k != key) continue;
    const int m = d.table[slot];
    if (d.member_hash[m] != h) return -1;
    const CRow member = member_row(d, m);
    if (member.n != child.n || member.nc != child.nc) return -1;
    bool mine = false;
    for (int i = wlane(); i < child.n; i += 64) mine = mine || member.origin[i] != child.origin[i];
    for (int i = wlane(); i < child.nc; i += 64) {
      const Val x = member.cval[i], y = child.cval[i];
      mine = mine || x.tag != y.tag || (x.tag == TAG_BOOL ? x.b != y.b : x.i != y.i);
    }
    return __ballot(mine) != 0 ? -1 : m;
  }
  return -1;
}
// find_member_w for a row in registers.
__device__ inline int find_member_row(const DSearch& d, const WaveRow& child, std::uint64_t h) {
  const std::uint64_t key = h | 1;
  for (int probe = 0; probe <= d.table_mask; ++probe) {
    const int slot = int((h + std::uint64_t(probe)) & std::uint64_t(d.table_mask));
    const std::uint64_t k = d.table_key[slot];
    if (k == 0) return -1;
    if (k != key) continue;
    const int m = __builtin_amdgcn_readfirstlane(d.table[slot]);
    const std::size_t o = std::size_t(m) * d.R;
    const std::uint64_t hash = d.member_hash[m];
    const WaveRow member = load_row(d.cur_origin + o, d.cur_site + o, d.cur_cval + o, d.R, d.cur_n[m], d.cur_nc[m]);
    return hash == h && same_rows(child, member) ? m : -1;
  }
  return -1;
}
// The evaluation kernel that scores a program: 1 the typed straight-line
// path, 2 the typed looping path (both with an LDS score buffer, so only
// where the cases fit it), 0 the general VM.
__device__ inline int eval_class(int code_flags, int C) {
  if (C > kScoreCases) return 0;
  return (code_flags & 2) ? 1 : (code_flags & 8) ? 2 : 0;
}
// Pending list of a round: general children from the front of [0, B), the
// straight-line ones from its back, the looping ones in [B, 2B).
__device__ inline int pending_at(int B, int kind, int i) { return kind == 0 ? i : kind == 1 ? B - 1 - i : B + i; }

// Puts a lowered child on its pending list.
__device__ inline void pend_child(const DSearch& d, int c, int flags) {
  if (wlane() != 0) return;
  d.reuse[c] = -1;
  const int k = eval_class(flags, d.cd.C);
  d.pending[pending_at(d.B, k, atomicAdd(d.n_pending + k, 1))] = c;
}

// ---- reproduction: one wavefront per child (phase_operators.cuh:156-265) ----
// kStaged: the block first copies the phase tables into LDS (searches whose
// tables fit); otherwise the operators read them from global memory.
// kDefer: rows that lower_row does not lower are left to k_lower (searches
// whose programs may jump; those that may not have straight-line code, which
// the small lowering here covers). The node-by-node lowering of a traversal is
// 75-100 us of dependent steps, and its registers in this kernel cost one more
// wavefront per SIMD: 8192 children of a list grammar took 352 us with it, and
// take 150 plus 8 for the launch that finds nothing to lower. With kDefer at
// most 80 vector registers and not 89, so six wavefronts per SIMD and not five,
// for 8 or 9 values spilled to scratch: 150 us for 153 on those children, 154 for
// 159 on 8192 of a statement grammar. Without, six took 93 us for 91 on 8192
// children of the quintic grammar (9 and, for rows in memory, 28 values spilled),
// so those keep their five.
template <bool kStaged, bool kDefer>
__global__ __launch_bounds__(64 * kVaryWaves) __attribute__((amdgpu_waves_per_eu(kDefer ? 6 : 5))) void k_vary(DSearch* all, const BlockMap* map) {
  const BlockMap bm = map[blockIdx.x];
  const DSearch& d = all[bm.search];
  if (!search_live(d) || (d.stage_tables != 0) != kStaged || (d.defer != 0) != kDefer) return;  // uniform per block
  extern __shared__ __attribute__((aligned(16))) unsigned char vary_lds[];
  const PhaseView g = kStaged ? stage_phase_tables<64 * kVaryWaves>(d.g, vary_lds) : view_of(d.g);
  const int c = bm.block * kVaryWaves + wave_index();
  if (c >= d.B) return;
  const std::uint64_t seed = *d.round_seed;
  const Keys keys = d.select ? Keys{d.select, nullptr, nullptr, 0} : Keys{d.fitness, d.wrong, d.nodes, d.has_wrong};
  const std::size_t o = std::size_t(c) * d.R;
  Row x{d.x_origin + o, d.x_site + o, d.x_cval + o, 0, 0};
  Row tmp{d.t_origin + o, d.t_site + o, d.t_cval + o, 0, 0};
  OpStats st;
  // Elite rows replace the first children after variation; a child's draws
  // depend only on (seed, child), so the elite children skip theirs. An elite
  // child is its source member and reuses its result.
  const int elite = d.generational && c < d.elites ? d.elite[c] : -1;
  __shared__ LaneStore<kDefer> row_lds[kVaryWaves];
  LaneStore<kDefer>& store = row_lds[wave_index()];
  LAS int* const hist = (LAS int*)store.sums;
  WaveGrammar w;
  // Rows of one node per lane stay in registers (vary_wave.hpp); wider rows
  // and grammars are varied in memory.
  const bool in_lanes = d.R <= kWaveRow && wave_grammar(g, w);
  WaveRow child_row;
  std::uint64_t h = 0;
  if (in_lanes) {
    const auto member = [&](int m) {
      const std::size_t at = std::size_t(m) * d.R;
      return load_row(d.cur_origin + at, d.cur_site + at, d.cur_cval + at, d.R, d.cur_n[m], d.cur_nc[m]);
    };
    if (elite >= 0) {
      st = OpStats{elite, 0, 0, 0, 0, 0, 0, elite, -1};
      child_row = member(elite);
    } else {
      st = OpStats{-1, 0, 0, 0, 0, 0, 0, -1, -1};
      WaveDraws draws(seed ^ (0x617089e168ULL + std::uint64_t(c)));
      tournament_rows(keys, d.P, d.pressure, draws, st.parent, st.donor);
      const WaveRow parent = member(st.parent), donor = member(st.donor);
      child_row = parent;
      if (parent.n <= 0) st.error = 1;
      else cross_rows(g, w, d.slot, parent, donor, child_row, draws, d.pol, hist, st);
      mutate_row(g, w, d.slot, child_row, tmp, d.p_mut, seed ^ (0x124ab512bf01ULL + std::uint64_t(c)), d.pol, hist, st);
      if (!st.error) compare_rows(parent, child_row, d.P, st);
    }
    if (!st.error) h = row_hash_row(child_row);
    store_row(child_row, d.x_origin + o, d.x_site + o, d.x_cval + o);
    x.n = child_row.n;
    x.nc = child_row.nc;
  } else {
    if (elite >= 0) {
      copy_row_w(member_row(d, elite), x);
      st = OpStats{elite, 0, 0, 0, 0, 0, 0, elite, -1};
      wave_fence();
    } else {
      crossover_w(g, d.slot, c, [&](int m) { return member_row(d, m); }, x, keys, d.P, d.pressure, seed, d.pol, st);
      wave_fence();
      Row spl{d.s_origin + o, d.s_site + o, d.s_cval + o, 0, 0};
      mutate_w(g, d.slot, c, x, tmp, spl, d.p_mut, seed, d.pol, st);
      wave_fence();
      if (!st.error) compare_w(member_row(d, st.parent), as_const(x), d.P, st);
    }
    if (!st.error) h = row_hash_w(as_const(x));
  }
  const CRow child = as_const(x);
  if (wlane() == 0) {
    d.x_n[c] = x.n;
    d.x_nc[c] = x.nc;
    d.stats[c] = st;
    d.child_hash[c] = h;
    if (st.error) raise(d, 300 + st.error);
  }
  if (st.error) return;
  // A child identical to its parent, or to any member, takes that member's
  // completed result and is neither lowered nor evaluated. Results are
  // fixed before any placement of the round.
  const int r = st.reusable_parent >= 0 ? st.reusable_parent : in_lanes ? find_member_row(d, child_row, h) : find_member_w(d, child, h);
  if (r >= 0) {
    if (wlane() == 0) {
      d.code_len[c] = 0;
      d.pool_len[c] = 0;
      d.reuse[c] = r;
      d.c_fit[c] = d.fitness[r];
      d.c_wrong[c] = d.wrong[r];
      d.c_nodes[c] = d.nodes[r];
    }
    return;
  }
  unsigned n;
  if (!d.grammar_sites) {
    n = unsigned(d.fixed_nodes) + unsigned(child.n);
  } else if (in_lanes) {
    n = unsigned(__popcll(__ballot(child_row.site >= 0)));
  } else {
    unsigned mine = 0;
    for (int i = wlane(); i < child.n; i += 64) mine += child.site[i] >= 0;
    for (int off = 32; off > 0; off >>= 1) mine += __shfl_xor(mine, off, 64);
    n = mine;
  }
  if (wlane() == 0) d.c_nodes[c] = n;
  LowerResult lowered;
  const bool done = in_lanes && lower_row<kDefer>(w, child_row, d.local_types, d.n_locals, d.expected_type, d.code + std::size_t(c) * d.code_cap,
                                          d.code_cap, d.pool + std::size_t(c) * d.pool_cap, d.pool_cap, (LAS LaneStore<kDefer>*)&store, lowered);
  if constexpr (kDefer) {
    if (done) pend_child(d, c, store_lowered(d, c, lowered, store.code));
    else if (wlane() == 0) d.reuse[c] = -2;
    return;
  }
  if (!done) {
    WaveOrigins source{child};
    if (in_lanes) {
      source.tile = source.constants = 0;
      source.tile_origin = child_row.origin;
      source.c0 = child_row.c0;
      source.c1 = child_row.c1;
      source.ct = child_row.ct;
    }
    WalkStore<false> ws;
    lowered = lower_into_w<false>(g, d, child, c, source, ws);
  }
  pend_child(d, c, store_lowered(d, c, lowered));
}
// Lowers the children k_vary left, a wavefront each. The grammar's nodes are
// held in lanes where they fit, else its tables are staged.
template <bool kWalks>
__global__ __launch_bounds__(64 * kVaryWaves) void k_lower(DSearch* all, const BlockMap* map) {
  const BlockMap bm = map[blockIdx.x];
  const DSearch& d = all[bm.search];
  if (!search_live(d) || !d.defer || (d.walks != 0) != kWalks) return;  // uniform per block
  extern __shared__ __attribute__((aligned(16))) unsigned char vary_lds[];
  const PhaseView tables = view_of(d.g);
  WaveGrammar w;
  const bool packed = wave_grammar(tables, w);
  const PhaseView g = packed || !d.stage_tables ? tables : stage_phase_tables<64 * kVaryWaves>(d.g, vary_lds);
  const int c = bm.block * kVaryWaves + wave_index();
  if (c >= d.B || __builtin_amdgcn_readfirstlane(d.reuse[c]) != -2) return;
  __shared__ WalkStore<kWalks> walk_lds[kVaryWaves];
  const CRow row = child_row(d, c);
  WaveOrigins source{row};
  source.packed = packed;
  source.node = w.node;
  source.node2 = w.node2;
  const int flags = store_lowered(d, c, lower_into_w<kWalks>(g, d, row, c, source, walk_lds[wave_index()]));
  pend_child(d, c, flags);
}

// ---- evaluation: one wavefront per program ----
__device__ inline double wave_sum_d(double x) {
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
  return x;
}
__device__ inline unsigned wave_sum_u(unsigned x) {
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
  return x;
}
struct EvalParams {
  CaseData cd;
  int fuel, lanes;
  double penalty;
  Policy policy;
};
struct EvalOut { double fitness; unsigned wrong, errors, timeouts; unsigned long long fuel; };

__device__ inline Val expected_of(const CaseData& cd, int c) {
  Val expected{};
  expected.i = cd.exp_val[c]; expected.tag = cd.exp_tag[c]; expected.b = cd.exp_b[c];
  return expected;
}
__device__ inline double lane_score(const EvalParams& e, const LaneResult& r, const Val& expected, bool& exact) {
  if (r.err != ERR_NONE) { exact = false; return -error_ceiling(e.policy, e.penalty); }
  Val actual{};
  actual.i = r.v; actual.tag = r.t; actual.b = r.b;
  return case_score(actual, expected, e.penalty, e.policy, exact);
}
__device__ inline double lane_score(const EvalParams& e, const LaneResult& r, int c, bool& exact) {
  return lane_score(e, r, expected_of(e.cd, c), exact);
}

// The case set of one search copied into a block's LDS for the typed path:
// per case, each input's payload (Bool as 0/1) and a bound mask, and the
// expected value. Every wavefront of a block scores programs of the same
// search, so the block stages it once.
struct StagedCases {
  LAS std::int64_t* value;      // [n_inputs][C]
  LAS std::uint8_t* bound;      // [C]: bit k = input k bound
  LAS std::int64_t* expected;   // [C] payload
  LAS std::uint8_t* exp_tag;    // [C]
  LAS std::uint8_t* exp_b;      // [C]
  bool on;                      // staged for this block
};
// Input rows the typed path reads: those bound by the program's locals and
// present in the case data, at most kFastInputs.
GHD inline int staged_inputs_of(int n_locals, int n_inputs) {
  return std::min(std::min(n_locals, n_inputs), kFastInputs);
}
GHD inline std::size_t staged_case_bytes(int C, int n_rows) { return std::size_t(C) * (8 * std::size_t(n_rows) + 8 + 3); }
template <int kThreads>
__device__ inline StagedCases stage_cases(const CaseData& cd, int n_locals, unsigned char* lds) {
  const int C = cd.C, n_inputs = staged_inputs_of(n_locals, cd.n_inputs);
  StagedCases sc;
  sc.on = true;
  sc.value = (LAS std::int64_t*)lds;
  sc.expected = sc.value + std::size_t(n_inputs) * C;
  sc.bound = (LAS std::uint8_t*)(sc.expected + C);
  sc.exp_tag = sc.bound + C;
  sc.exp_b = sc.exp_tag + C;
  for (int c = threadIdx.x; c < C; c += kThreads) {
    unsigned mask = 0;
    for (int k = 0; k < n_inputs; ++k) {
      const std::size_t at = std::size_t(k) * C + c;
      const std::uint8_t tag = cd.in_tag[at];
      if (tag != TAG_INVALID) mask |= 1u << k;
      sc.value[at] = tag == TAG_BOOL ? std::int64_t(cd.in_b[at] != 0) : cd.in_val[at];
    }
    sc.bound[c] = std::uint8_t(mask);
    sc.expected[c] = cd.exp_val[c];
    sc.exp_tag[c] = cd.exp_tag[c];
    sc.exp_b[c] = cd.exp_b[c];
  }
  __syncthreads();
  return sc;
}
__device__ inline FastInputs staged_inputs(const StagedCases& sc, int C, int n_inputs, int c, bool active) {
  FastInputs in{0, 0, 0, 0, 0};
  if (!active) return in;
  // Unstaged rows beyond n_inputs are unbound, as in fast_inputs.
  in.bound = sc.bound[c];
  if (n_inputs > 0) in.v0 = sc.value[c];
  if (n_inputs > 1) in.v1 = sc.value[std::size_t(C) + c];
  if (n_inputs > 2) in.v2 = sc.value[2 * std::size_t(C) + c];
  if (n_inputs > 3) in.v3 = sc.value[3 * std::size_t(C) + c];
  return in;
}

// The canonical total of C case scores held in `scores`, computed by one
// wavefront: L logical lanes over contiguous case chunks with 48-bit rounding,
// then 32-lane groups and the total (the legacy metric sums the lane partials
// directly). `sums`: kReplayWords doubles of this wavefront's LDS. 512 logical
// lanes at a time leave their partials there, 33 words a group so that the
// groups' reads fall into different banks, and a lane adds up each group.
// Bound by the chain of rounded additions, now 48 and not 528 for 512 lanes;
// with every addition on all lanes, each behind a shuffle, a program took about
// 30 us and the launch of 540 programs on 600 discounted cases 127 us, now 47.
constexpr int kReplayLanes = 512, kReplayWords = kReplayLanes / 32 * 33;
__device__ inline double canonical_from_scores(const EvalParams& e, int C, const double* scores, int lane, double* sums) {
  const int L = e.lanes;
  double total = 0;
  for (int chunk = 0; chunk < L; chunk += kReplayLanes) {
    const int count = min(kReplayLanes, L - chunk);
    for (int base = 0; base < count; base += 64) {
      const int l = chunk + base + lane, at = base + lane;
      const bool own = l < L;
      const int begin = own ? int((std::int64_t(C) * l) / L) : 0;
      const int end = own ? int((std::int64_t(C) * (l + 1)) / L) : 0;
      double local = 0;
      for (int c = begin; c < end; ++c) local = canon48(local + scores[c]);
      sums[at + at / 32] = local;
    }
    wave_fence();
    if (e.policy.metric == METRIC_LEGACY) {
      for (int k = 0; k < count; ++k) total = canon48(total + sums[k + k / 32]);
    } else {
      const int groups = (count + 31) / 32, mine = min(32, count - 32 * lane);
      double group = 0;
      for (int k = 0; k < mine; ++k) group = canon48(group + sums[33 * lane + k]);
      for (int k = 0; k < groups; ++k) total = canon48(total + rdlane_d(group, k));
    }
    wave_fence();
  }
  return total;
}

// Scores one program over all cases with the canonical reduction
// (fitness_cpu.cpp:97-171: L logical lanes over contiguous case chunks,
// 48-bit rounding after every addition, 32-lane groups then the total).
// When every case score is an integer of magnitude <= 2^36 (and C <= 4096)
// every partial sum is an exact integer below 2^48, the rounding is the
// identity and any summation order gives the canonical total.
// kFast: `pv` is certified for the typed straight-line VM (vm_fast);
// otherwise the general VM runs it with its stack in LDS.
// `scores` (this wavefront's LDS buffer of C doubles, or null) keeps every
// case score of the first pass, so the canonical order is replayed from it
// instead of by running the program again; the fast kernel always has it, and `sums`
// (canonical_from_scores).
template <int kKind>
__device__ EvalOut eval_program(const EvalParams& e, const ProgView& pv, WaveStack& st, double* scores, int lane, double* sums,
                                StagedCases staged = StagedCases{}) {
  static_assert(kKind == 0 || kKind == 1, "the looping path has its own kernel");
  constexpr bool kFast = kKind != 0;  // a typed path: scores in LDS, inputs untagged
  const int C = e.cd.C;
  double isum = 0;
  unsigned w = 0, errs = 0, touts = 0;
  unsigned long long fuel = 0;
  bool integral = C <= 4096;
  FastProgram fp{};
  if (kKind == 1) fp = fast_load(pv, lane);
  const int n_in = staged_inputs_of(pv.n_locals, e.cd.n_inputs);
  const auto typed = [&](const FastInputs& in, bool active) { return vm_fast(fp, in, active, e.fuel, pv.result_tag); };
  const auto run = [&](int c, bool active) {
    if (kFast) return typed(fast_inputs(e.cd, pv.n_locals, c, active), active);
    return vm_run(pv, e.cd, active ? c : 0, active, e.fuel, st, lane);
  };
  for (int tile = 0; tile < C; tile += 64) {
    const int c = tile + lane;
    const bool active = c < C;
    LaneResult r;
    Val expected{};
    if constexpr (kFast) {
      // One call site of the typed VM for both input sources.
      const FastInputs in =
          staged.on ? staged_inputs(staged, C, n_in, c, active) : fast_inputs(e.cd, pv.n_locals, c, active);
      r = typed(in, active);
      if (active) {
        if (staged.on) { expected.i = staged.expected[c]; expected.tag = staged.exp_tag[c]; expected.b = staged.exp_b[c]; }
        else expected = expected_of(e.cd, c);
      }
    } else {
      r = run(c, active);
      if (active) expected = expected_of(e.cd, c);
    }
    if (active) {
      bool exact = false;
      const double s = lane_score(e, r, expected, exact);
      w += !exact;
      errs += r.err != ERR_NONE;
      touts += r.err == ERR_TIMEOUT;
      fuel += unsigned(r.fuel_used);
      integral = integral && s == double(std::int64_t(s)) && s >= -68719476736.0 && s <= 68719476736.0;
      isum += s;
      if (scores) scores[c] = s;
    }
  }
  EvalOut out;
  out.wrong = wave_sum_u(w);
  out.errors = wave_sum_u(errs);
  out.timeouts = wave_sum_u(touts);
  for (int off = 32; off > 0; off >>= 1) fuel += __shfl_xor(fuel, off, 64);
  out.fuel = fuel;
  if (__ballot(!integral) == 0) {
    out.fitness = wave_sum_d(isum);
    return out;
  }
  // Canonical order: lane j owns logical lanes j, j+64, ... of L.
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");  // scores[] of other lanes
  __builtin_amdgcn_wave_barrier();
  if constexpr (kFast) {
    out.fitness = canonical_from_scores(e, C, scores, lane, sums);
    return out;
  }
  const int L = e.lanes;
  double group_total = 0;
  for (int base = 0; base < L; base += 64) {
    const int l = base + lane;
    const bool own = l < L;
    const int begin = own ? int((std::int64_t(C) * l) / L) : 0;
    const int end = own ? int((std::int64_t(C) * (l + 1)) / L) : 0;
    int longest = end - begin;
    for (int off = 32; off > 0; off >>= 1) { const int y = __shfl_xor(longest, off, 64); longest = y > longest ? y : longest; }
    double local = 0;
    for (int s = 0; s < longest; ++s) {
      const int c = begin + s;
      const bool active = c < end;
      if (scores) {
        if (active) local = canon48(local + scores[c]);
      } else {
        const LaneResult r = run(active ? c : 0, active);
        if (active) {
          bool exact = false;
          local = canon48(local + lane_score(e, r, c, exact));
        }
      }
    }
    // Two 32-lane groups per 64 logical lanes, summed in lane order.
    for (int half = 0; half < 2; ++half) {
      if (base + half * 32 >= L) break;
      double group = 0;
      for (int k = 0; k < 32; ++k) {
        const int src = half * 32 + k;
        const double v = __shfl(local, src, 64);
        if (base + src < L) group = canon48(group + v);
      }
      if (e.policy.metric == METRIC_LEGACY) {
        // Legacy sums every lane partial in order, with no group stage.
        for (int k = 0; k < 32; ++k) {
          const int src = half * 32 + k;
          const double v = __shfl(local, src, 64);
          if (base + src < L) group_total = canon48(group_total + v);
        }
      } else {
        group_total = canon48(group_total + group);
      }
    }
  }
  out.fitness = group_total;
  return out;
}

// Items of the looping kernel: (program, group of `group` consecutive
// 64-case tiles) pairs, one wavefront each; blocks of one wavefront for n
// programs (at most kLoopBlocks, which loop over the rest).
constexpr int kLoopBlocks = 16384;
__host__ __device__ inline int loop_blocks(int C, int n, int group = 1) {
  const int tiles = (C + 63) / 64, groups = (tiles + group - 1) / group;
  return int(std::min<long long>(kLoopBlocks, (long long)n * groups));
}

// The looping path as a tile queue: every block is one wavefront and takes
// (program, tile group) items of its own, so no wavefront waits for another.
// A group is `group` consecutive 64-case tiles of one program, run one after
// another by the wavefront. Items go tile group first: the cases are visited
// by descending list length, so the longest items of all programs start
// first and the launch ends with the shortest.
// Scores go to the program's row of loop_scores (HBM). A program with one
// group is finished by its wavefront; otherwise every group adds its totals
// (whole numbers, so their order is free) to the program's LoopAcc, and
// k_loop_finish, the next launch, takes them: no fence orders the items of one
// program. LDS: step_slots(n_inputs) slots of 64 lanes, independent of the
// case count.
// kGrouped false is the one-tile instantiation (group 1): its loop-carried
// totals fold away.
// Bound by instruction issue of the step loop (scalar decode and branches).
// Four-wavefront blocks of one program held their slots until the longest of
// its tiles ended, and every item paid two device-wide fences and thirteen
// atomics. Measured together with the decoded steps, per launch: population
// 8192 x 200 list cases 3.18 -> 0.68 ms, 64 mixed searches 5.56 -> 1.62 ms,
// population 1500 x 130 cases of statement programs 0.85 -> 0.33 ms.
template <bool kGrouped>
__global__ __launch_bounds__(64) void k_eval_loop(DSearch* all, const BlockMap* map, int mode, int group_arg) {
  const int group = kGrouped ? group_arg : 1;
  const BlockMap bm = map[blockIdx.x];
  const DSearch& d = all[bm.search];
  if (mode == 1 ? !search_live(d) : (!d.active || *d.error)) return;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x;
  const int C = d.cd.C, tiles = (C + 63) / 64, groups = (tiles + group - 1) / group;
  LAS std::int64_t* const slots = (LAS std::int64_t*)smem;
  const EvalParams e{d.cd, d.fuel, d.lanes, d.penalty, d.policy};
  const int count = mode == 1 ? d.n_pending[2] : d.P;
  const long long items = (long long)count * groups;
  for (long long k = bm.block; k < items; k += bm.blocks) {
    const int q0 = int(k / count), i = int(k % count), first = q0 * group, last = min(tiles, first + group);
    const int slot = mode == 1 ? d.pending[pending_at(d.B, 2, i)] : i;
    const int pmode = d.code_jumps[slot];
    if (mode == 0 && eval_class(pmode, C) != 2) continue;  // another kernel scores it (uniform per wavefront)
    const int n_in = staged_inputs_of(d.n_locals, e.cd.n_inputs), result_tag = (pmode & 4) ? TAG_BOOL : TAG_INT;
    const StepProgram sp = steps_load((GAS const std::uint64_t*)(d.code + std::size_t(slot) * d.code_cap),
                                      d.pool + std::size_t(slot) * d.pool_cap, pmode >> 8, lane);
    GAS double* const scores = d.loop_scores + std::size_t(slot) * C;
    long long total = 0;  // exact while no score is fractional
    bool frac = false;
    unsigned tw = 0, te = 0, tt = 0;
    unsigned long long tf = 0;
    const int n_tiles = kGrouped ? last - first : 1;  // first < tiles: one tile when ungrouped
    for (int q = 0; q < n_tiles; ++q) {
      // Cases in the search's visiting order (similar loop lengths per
      // tile); scores are kept by case index, so the totals are unchanged.
      const int at = (first + q) * 64 + lane;
      const bool active = at < C;
      const int c = active ? e.cd.order[at] : 0;
      const FastInputs in = fast_inputs(e.cd, d.n_locals, c, active);
      const LaneResult r = sp.n <= 64 ? vm_steps<1>(sp, in, n_in, e.cd.arena, slots, lane, active, e.fuel, result_tag)
                                      : vm_steps<4>(sp, in, n_in, e.cd.arena, slots, lane, active, e.fuel, result_tag);
      double sc = 0;
      bool exact = true;
      if (active) {
        sc = lane_score(e, r, expected_of(e.cd, c), exact);
        scores[c] = sc;
      }
      // Integral scores below 2^36 in magnitude: every partial sum is exact.
      const bool fractional =
          __ballot(active && !(sc == double(std::int64_t(sc)) && sc >= -68719476736.0 && sc <= 68719476736.0)) != 0;
      const double ws = wave_sum_d(sc);
      frac = frac || fractional;
      if (!frac) total += (long long)ws;
      tw += unsigned(__popcll(__ballot(active && !exact)));
      te += unsigned(__popcll(__ballot(active && r.err != ERR_NONE)));
      tt += unsigned(__popcll(__ballot(active && r.err == ERR_TIMEOUT)));
      tf += wave_sum_u64(active ? unsigned(r.fuel_used) : 0u);
    }
    if (groups > 1) {
      if (lane == 0) {
        GAS LoopAcc* const acc = d.loop_acc + slot;
        if (frac) atomicOr(&acc->fractional, 1u);
        else atomicAdd(&acc->sum, (unsigned long long)total);
        atomicAdd(&acc->fuel, tf);
        if (tw) atomicAdd(&acc->wrong, tw);
        if (te) atomicAdd(&acc->errors, te);
        if (tt) atomicAdd(&acc->timeouts, tt);
      }
      continue;
    }
    wave_fence();  // the canonical replay reads the other lanes' scores
    // The program has ended: its slots hold the replay's partials.
    static_assert((kLoopLocals + kStepStack) * 64 >= kReplayWords, "slots of a program without inputs");
    const double fitness = frac ? canonical_from_scores(e, C, scores, lane, (double*)slots) : double(total);
    if (lane == 0) {
      // Ranking rounds every published fitness to a 40-bit mantissa.
      if (mode == 1) { d.c_fit[slot] = canon40(fitness); d.c_wrong[slot] = tw; }
      else { d.fitness[slot] = canon40(fitness); d.wrong[slot] = tw; }
      d.e_errors[slot] = te;
      d.e_timeouts[slot] = tt;
      d.e_fuel[slot] = tf;
    }
  }
}

// Takes and clears the LoopAcc of every program of more than one tile group:
// 16 lanes per program and four programs per wavefront, the canonical replay
// over the program's scores by the whole wavefront where some tile had a
// non-integral one.
constexpr int kFinishPrograms = 4 * kWavesPerBlock;  // programs per block
__global__ __launch_bounds__(kEvalThreads) void k_loop_finish(DSearch* all, const BlockMap* map, int mode, int group) {
  const BlockMap bm = map[blockIdx.x];
  const DSearch& d = all[bm.search];
  if (mode == 1 ? !search_live(d) : (!d.active || *d.error)) return;
  const int C = d.cd.C, tiles = (C + 63) / 64, groups = (tiles + group - 1) / group;
  if (groups <= 1 || C > kScoreCases) return;
  __shared__ double replay[kWavesPerBlock][kReplayWords];
  const int lane = threadIdx.x % 64, part = lane % 16;
  const EvalParams e{d.cd, d.fuel, d.lanes, d.penalty, d.policy};
  const int count = mode == 1 ? d.n_pending[2] : d.P;
  for (int base = bm.block * kFinishPrograms + 4 * wave_index(); base < count; base += bm.blocks * kFinishPrograms) {
    const int i = base + lane / 16;
    const int slot = i >= count ? -1 : mode == 1 ? d.pending[pending_at(d.B, 2, i)] : i;
    const bool mine = slot >= 0 && (mode == 1 || eval_class(d.code_jumps[slot], C) == 2);
    LoopAcc t{0, 0, 0, 0, 0, 0};
    if (mine && part == 0) {
      GAS LoopAcc* const acc = d.loop_acc + slot;
      t.sum = acc->sum; t.fuel = acc->fuel;
      t.wrong = acc->wrong; t.errors = acc->errors; t.timeouts = acc->timeouts; t.fractional = acc->fractional;
      acc->sum = acc->fuel = 0;
      acc->wrong = acc->errors = acc->timeouts = acc->fractional = 0;
    }
    double fitness = double((long long)t.sum);
    for (unsigned long long m = __ballot(mine && part == 0 && t.fractional); m; m &= m - 1) {
      const int from = wave_first(m);
      const double total = canonical_from_scores(e, C, d.loop_scores + std::size_t(rdlane(slot, from)) * C, lane, replay[wave_index()]);
      if (lane == from) fitness = total;
    }
    if (mine && part == 0) {
      if (mode == 1) { d.c_fit[slot] = canon40(fitness); d.c_wrong[slot] = t.wrong; }
      else { d.fitness[slot] = canon40(fitness); d.wrong[slot] = t.wrong; }
      d.e_errors[slot] = t.errors;
      d.e_timeouts[slot] = t.timeouts;
      d.e_fuel[slot] = t.fuel;
    }
  }
}

// A wavefront's LDS stack of `slots` operand slots followed by `temps`
// hidden-local slots, 10 bytes per lane and slot; the last `shadow` of them
// shadow stored inputs.
__device__ inline WaveStack stack_of(unsigned char* smem, int slots, int temps, int wave, int shadow) {
  const int all = slots + temps;
  unsigned char* base = smem + std::size_t(wave) * all * 64 * 10;
  return WaveStack{reinterpret_cast<std::int64_t*>(base), base + std::size_t(all) * 64 * 8,
                   base + std::size_t(all) * 64 * 9, slots, temps, shadow};
}

// mode 0: score members 0..P-1 (initial population), mode 1: pending
// children. kFast: the programs certified for vm_fast (pending entries from
// the back of the list); otherwise the rest (from the front).
template <int kKind>
__global__ __launch_bounds__(kEvalThreads) void k_eval(DSearch* all, const BlockMap* map, int mode) {
  constexpr bool kFast = kKind != 0;
  const BlockMap bm = map[blockIdx.x];
  const DSearch& d = all[bm.search];
  if (mode == 1 ? !search_live(d) : (!d.active || *d.error)) return;
  if (kFast && d.typed_tiles) return;  // k_eval_tiles scores them
  extern __shared__ unsigned char smem[];
  __shared__ double replay[kFast ? kWavesPerBlock : 1][kFast ? kReplayWords : 1];
  const int wave = wave_index(), lane = threadIdx.x % 64;
  WaveStack st = stack_of(smem, kFast ? 0 : d.stack_slots, kFast ? 0 : d.temp_slots, wave, kFast ? 0 : d.input_shadow);
  // Score buffers follow the stacks of the block's wavefronts.
  double* scores =
      (kFast ? d.cd.C <= kScoreCases : d.general_scores != 0)
          ? reinterpret_cast<double*>(smem + std::size_t(kWavesPerBlock) * (kFast ? 0 : d.stack_slots + d.temp_slots) * 64 * 10) +
                std::size_t(wave) * d.cd.C
          : nullptr;
  const EvalParams e{d.cd, d.fuel, d.lanes, d.penalty, d.policy};
  // The typed kernel stages the case set after the score buffers.
  StagedCases staged{};
  const bool stage = kFast && d.stage_cases;
  if (stage)
    staged = stage_cases<kEvalThreads>(d.cd, d.n_locals,
                                       smem + std::size_t(kWavesPerBlock) * 8 * std::size_t(d.cd.C));
  const int count = mode == 1 ? d.n_pending[kKind] : d.P;
  for (int i = bm.block * kWavesPerBlock + wave; i < count; i += bm.blocks * kWavesPerBlock) {
    const int slot = mode == 1 ? d.pending[pending_at(d.B, kKind, i)] : i;
    const int pmode = d.code_jumps[slot];
    if (mode == 0 && eval_class(pmode, d.cd.C) != kKind) continue;  // another kernel scores it
    const ProgView pv{d.code + std::size_t(slot) * d.code_cap, d.pool + std::size_t(slot) * d.pool_cap, d.code_len[slot],
                      d.n_locals, pmode & 1, (pmode >> 1) & 1, d.pool_len[slot], (pmode & 4) ? TAG_BOOL : TAG_INT};
    const EvalOut r = eval_program<kKind>(e, pv, st, scores, lane, replay[kKind == 0 ? 0 : wave], staged);
    if (lane == 0) {
      // Ranking rounds every published fitness to a 40-bit mantissa.
      if (mode == 1) { d.c_fit[slot] = canon40(r.fitness); d.c_wrong[slot] = r.wrong; }
      else { d.fitness[slot] = canon40(r.fitness); d.wrong[slot] = r.wrong; }
      // Per-program tallies, summed once per launch by k_tally.
      d.e_errors[slot] = r.errors;
      d.e_timeouts[slot] = r.timeouts;
      d.e_fuel[slot] = r.fuel;
    }
  }
}

// The typed straight-line VM with one block per program: the block's four
// wavefronts take the program's 64-case tiles in turn (tile w, w + 4, ...),
// so a program waits for a quarter of the tile chain one wavefront would
// run. Each wavefront reads its tiles' inputs from the case arrays. The
// case scores go to the block's LDS; the totals of the four wavefronts are
// combined in LDS -- exactly, when every score is an integer of magnitude
// <= 2^36 (all partial sums are integers below 2^48) -- and otherwise the
// canonical replay reads the scores, as in eval_program. mode as k_eval.
__global__ __launch_bounds__(kEvalThreads) void k_eval_tiles(DSearch* all, const BlockMap* map, int mode) {
  const BlockMap bm = map[blockIdx.x];
  const DSearch& d = all[bm.search];
  if (mode == 1 ? !search_live(d) : (!d.active || *d.error)) return;
  if (!d.typed_tiles) return;  // uniform per block
  extern __shared__ unsigned char smem[];
  double* const scores = reinterpret_cast<double*>(smem);  // [C]
  __shared__ double part_sum[kWavesPerBlock], replay[kReplayWords];
  __shared__ unsigned part_count[kWavesPerBlock][4];  // wrong, errors, timeouts, integral
  __shared__ unsigned long long part_fuel[kWavesPerBlock];
  const int wave = wave_index(), lane = threadIdx.x % 64;
  const EvalParams e{d.cd, d.fuel, d.lanes, d.penalty, d.policy};
  const int C = d.cd.C;
  const int count = mode == 1 ? d.n_pending[1] : d.P;
  for (int i = bm.block; i < count; i += bm.blocks) {  // one program per block, uniform
    const int slot = mode == 1 ? d.pending[pending_at(d.B, 1, i)] : i;
    const int pmode = d.code_jumps[slot];
    if (mode == 0 && eval_class(pmode, C) != 1) continue;
    const ProgView pv{d.code + std::size_t(slot) * d.code_cap, d.pool + std::size_t(slot) * d.pool_cap, d.code_len[slot],
                      d.n_locals, pmode & 1, (pmode >> 1) & 1, d.pool_len[slot], (pmode & 4) ? TAG_BOOL : TAG_INT};
    const FastProgram fp = fast_load(pv, lane);
    double isum = 0;
    unsigned w = 0, errs = 0, touts = 0;
    unsigned long long fuel = 0;
    bool integral = true;  // C <= kScoreCases <= 4096
    for (int tile = wave * 64; tile < C; tile += kWavesPerBlock * 64) {
      const int c = tile + lane;
      const bool active = c < C;
      const LaneResult r = vm_fast(fp, fast_inputs(e.cd, pv.n_locals, c, active), active, e.fuel, pv.result_tag);
      if (active) {
        bool exact = false;
        const double sc = lane_score(e, r, expected_of(e.cd, c), exact);
        w += !exact;
        errs += r.err != ERR_NONE;
        touts += r.err == ERR_TIMEOUT;
        fuel += unsigned(r.fuel_used);
        integral = integral && sc == double(std::int64_t(sc)) && sc >= -68719476736.0 && sc <= 68719476736.0;
        isum += sc;
        scores[c] = sc;
      }
    }
    const double ws = wave_sum_d(isum);
    const unsigned ww = wave_sum_u(w), we = wave_sum_u(errs), wt = wave_sum_u(touts);
    for (int off = 32; off > 0; off >>= 1) fuel += __shfl_xor(fuel, off, 64);
    const bool wint = __ballot(!integral) == 0;
    if (lane == 0) {
      part_sum[wave] = ws;
      part_count[wave][0] = ww;
      part_count[wave][1] = we;
      part_count[wave][2] = wt;
      part_count[wave][3] = wint;
      part_fuel[wave] = fuel;
    }
    __syncthreads();  // every wavefront's scores and totals
    if (wave == 0) {
      double total = 0;
      unsigned tw = 0, te = 0, tt = 0;
      unsigned long long tf = 0;
      bool all_integral = true;
      for (int k = 0; k < kWavesPerBlock; ++k) {
        total += part_sum[k];
        tw += part_count[k][0];
        te += part_count[k][1];
        tt += part_count[k][2];
        all_integral = all_integral && part_count[k][3] != 0;
        tf += part_fuel[k];
      }
      const double fitness = all_integral ? total : canonical_from_scores(e, C, scores, lane, replay);
      if (lane == 0) {
        // Ranking rounds every published fitness to a 40-bit mantissa.
        if (mode == 1) { d.c_fit[slot] = canon40(fitness); d.c_wrong[slot] = tw; }
        else { d.fitness[slot] = canon40(fitness); d.wrong[slot] = tw; }
        d.e_errors[slot] = te;
        d.e_timeouts[slot] = tt;
        d.e_fuel[slot] = tf;
      }
    }
    __syncthreads();  // before the next program reuses the scores
  }
}

// ---- counters of one evaluation launch and, when profiling, of the
// reproduction that fed it (mode as k_eval) ----
constexpr int kTallyBlocks = 16;  // blocks per search, one atomic per counter each
__global__ __launch_bounds__(256) void k_tally(DSearch* all, int mode) {
  const DSearch& d = all[blockIdx.y];
  if (mode == 1 ? !search_live(d) : (!d.active || *d.error)) return;
  const int front = mode == 1 ? d.n_pending[0] : d.P, back = mode == 1 ? d.n_pending[1] : 0;
  const int count = mode == 1 ? front + back + d.n_pending[2] : d.P;
  const int first = int(blockIdx.x) * 256 + int(threadIdx.x), stride = kTallyBlocks * 256;
  unsigned long long v[11] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int i = first; i < count; i += stride) {
    const int slot = mode != 1        ? i
                     : i < front        ? d.pending[i]
                     : i < front + back ? d.pending[d.B - 1 - (i - front)]
                                        : d.pending[d.B + (i - front - back)];
    v[0] += d.e_errors[slot];
    v[1] += d.e_timeouts[slot];
    v[2] += d.e_fuel[slot];
    v[3] += unsigned(d.code_len[slot]);
    v[9] += unsigned(d.pool_len[slot]);
  }
  if (mode == 1 && d.profile)
    for (int c = first; c < d.B; c += stride) {
      const OpStats st = d.stats[c];
      v[4] += unsigned(d.x_n[c]);
      v[5] += unsigned(d.x_nc[c]);
      if (st.parent >= 0) { v[6] += unsigned(d.cur_n[st.parent]); v[7] += unsigned(d.cur_nc[st.parent]); }
      if (st.crossover_attempted && st.donor >= 0) { v[6] += unsigned(d.cur_n[st.donor]); v[7] += unsigned(d.cur_nc[st.donor]); }
      v[8] += unsigned(d.code_len[c]);
      v[10] += unsigned(d.pool_len[c]);
    }
  __shared__ unsigned long long part[11][256];
  for (int k = 0; k < 11; ++k) part[k][threadIdx.x] = v[k];
  __syncthreads();
  for (int span = 128; span > 0; span >>= 1) {
    if (int(threadIdx.x) < span)
      for (int k = 0; k < 11; ++k) part[k][threadIdx.x] += part[k][threadIdx.x + span];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    Counters* c = d.counters;
    if (blockIdx.x == 0) {
      atomicAdd(&c->programs, (unsigned long long)count);
      atomicAdd(&c->program_cases, (unsigned long long)count * unsigned(d.cd.C));
      if (mode == 1) atomicAdd(&c->children, (unsigned long long)d.B);
    }
    atomicAdd(&c->errors, part[0][0]);
    atomicAdd(&c->timeouts, part[1][0]);
    atomicAdd(&c->vm_instructions, part[2][0]);
    atomicAdd(&c->code_words, part[3][0]);
    atomicAdd(&c->pool_words, part[9][0]);
    if (mode == 1 && d.profile) {
      atomicAdd(&c->child_nodes, part[4][0]);
      atomicAdd(&c->child_consts, part[5][0]);
      atomicAdd(&c->parent_nodes, part[6][0]);
      atomicAdd(&c->parent_consts, part[7][0]);
      atomicAdd(&c->child_code_words, part[8][0]);
      atomicAdd(&c->child_pool_words, part[10][0]);
    }
  }
}

// ---- std::mt19937_64 on the device, generated 312 outputs at a time ----
__device__ inline std::uint64_t mt_temper(std::uint64_t y) {
  y ^= (y >> 29) & 0x5555555555555555ULL;
  y ^= (y << 17) & 0x71D67FFFEDA60000ULL;
  y ^= (y << 37) & 0xFFF7EEE000000000ULL;
  return y ^ (y >> 43);
}
__device__ inline std::uint64_t mt_next_word(std::uint64_t cur, std::uint64_t nxt, std::uint64_t far) {
  const std::uint64_t x = (cur & 0xFFFFFFFF80000000ULL) | (nxt & 0x7FFFFFFFULL);
  return far ^ (x >> 1) ^ ((x & 1ULL) ? 0xB5026F5AA96619E9ULL : 0ULL);
}
// In-place twist by a block of kThreads >= 64 threads: element i < 156 reads
// only old words; 156 <= i < 311 reads the new word i-156; 311 reads new
// words 0 and 155. The thread count is a template constant so the loops do
// not re-read the dispatch packet.
template <int kThreads>
__device__ inline void mt_twist(std::uint64_t* mt) {
  static_assert(kThreads >= 64, "three words per thread at most");
  const int t = threadIdx.x;
  std::uint64_t v[3];
  int n = 0;
  for (int i = t; i < 156; i += kThreads) v[n++] = mt_next_word(mt[i], mt[i + 1], mt[i + 156]);
  __syncthreads();
  n = 0;
  for (int i = t; i < 156; i += kThreads) mt[i] = v[n++];
  __syncthreads();
  n = 0;
  for (int i = 156 + t; i < 311; i += kThreads) v[n++] = mt_next_word(mt[i], mt[i + 1], mt[i - 156]);
  __syncthreads();
  n = 0;
  for (int i = 156 + t; i < 311; i += kThreads) mt[i] = v[n++];
  __syncthreads();
  if (t == 0) mt[311] = mt_next_word(mt[311], mt[0], mt[155]);
  __syncthreads();
}

__global__ __launch_bounds__(256) void k_seed(DSearch* all) {
  const DSearch& d = all[blockIdx.x];
  if (!d.active) return;
  __shared__ std::uint64_t mt[312];
  if (threadIdx.x == 0) {
    mt[0] = d.seed;
    for (int i = 1; i < 312; ++i) mt[i] = 6364136223846793005ULL * (mt[i - 1] ^ (mt[i - 1] >> 62)) + std::uint64_t(i);
  }
  __syncthreads();
  mt_twist<256>(mt);
  for (int i = threadIdx.x; i < 312; i += 256) d.mt[i] = mt[i];
  // Word 0 seeds round 0; words 1..311 wait for the first placement.
  for (int i = 1 + threadIdx.x; i < 312; i += 256) d.mt_left[i - 1] = mt_temper(mt[i]);
  if (threadIdx.x == 0) {
    *d.round_seed = mt_temper(mt[0]);
    *d.n_left = 311;
    *d.round = 0;
  }
}

// Node counts, best member, placements reset (after the initial evaluation).
__global__ void k_init_keys(DSearch* all) {
  const DSearch& d = all[blockIdx.x];
  if (!d.active || *d.error) return;
  for (int m = threadIdx.x; m < d.P; m += blockDim.x) {
    const CRow r = member_row(d, m);
    unsigned n = d.grammar_sites ? 0u : unsigned(d.fixed_nodes);
    if (d.grammar_sites) { for (int i = 0; i < r.n; ++i) n += r.site[i] >= 0; }
    else n += unsigned(r.n);
    d.nodes[m] = n;
    d.member_hash[m] = row_hash(r);
  }
  __syncthreads();
  __shared__ int best[256];
  const Keys keys{d.fitness, d.wrong, d.nodes, d.has_wrong};
  int b = -1;
  for (int m = threadIdx.x; m < d.P; m += blockDim.x)
    if (b < 0 || better(keys, m, b)) b = m;
  best[threadIdx.x] = b;
  __syncthreads();
  if (threadIdx.x == 0) {
    int x = -1;
    for (int t = 0; t < int(blockDim.x); ++t)
      if (best[t] >= 0 && (x < 0 || better(keys, best[t], x))) x = best[t];
    *d.best = x;
  }
}

// ---- history (evolve.cpp:364-372) ----
__global__ void k_record(DSearch* all) {
  const DSearch& d = all[blockIdx.x];
  if (!search_live(d)) return;
  const int r = *d.round;
  if (r % d.per_epoch) return;
  const int gen = r / d.per_epoch;
  const int b = *d.best;
  // Early exit: the state after `gen` generations is exactly that of a run
  // with `gen` generations, whose history has no row `gen`.
  if (d.early_exit && gen > 0 && d.has_wrong && d.wrong[b] == 0) {
    if (threadIdx.x == 0) *d.stop = gen;
    return;
  }
  const CRow row = member_row(d, b);
  const std::size_t o = std::size_t(gen) * d.R;
  for (int i = threadIdx.x; i < row.n; i += blockDim.x) d.hist_origin[o + i] = row.origin[i];
  for (int i = threadIdx.x; i < row.nc; i += blockDim.x) d.hist_cval[o + i] = row.cval[i];
  for (int m = threadIdx.x; m < d.P; m += blockDim.x) d.hist_all[std::size_t(gen) * d.P + m] = d.fitness[m];
  if (threadIdx.x == 0) {
    d.hist_n[gen] = row.n;
    d.hist_nc[gen] = row.nc;
    d.hist_fit[gen] = d.fitness[b];
    d.hist_wrong[gen] = d.wrong[b];
  }
}

// Round, early-stop generation and error of every search of the table.
__global__ void k_status(DSearch* all, int n, int* out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const DSearch& d = all[i];
  out[3 * i + 0] = *d.round;
  out[3 * i + 1] = *d.stop;
  out[3 * i + 2] = *d.error;
}

// ---- placement (evolve.cpp:378-422) ----
// The reference draws victims one group of `replacement_size` words at a
// time: the worst member drawn takes the next child, unless it is the best.
// Here a thread takes one of up to 1024 consecutive groups, and the chunk's
// victims are found as the fixpoint of the sequential rule: given everyone's
// victim, a group compares the members it drew with the keys they hold by its
// turn (the child of the last earlier group that took the member, else the
// member's own). A group depends on earlier ones alone, so every pass settles
// at least the first unsettled group, and an unchanged pass is the sequential
// outcome; most groups share no member with an earlier one, and a chunk takes
// as many passes as its longest chain of such groups. The chunk ends after the
// first group whose child becomes the best (the test against the best and its
// tracking change there) and after the first that places nothing (the children
// shift by one).
// Bound by the passes' chain of LDS reads and barriers in one block a search.
// One wavefront taking the longest prefix of 64 groups without a shared member
// needed a chunk of 1.1 us for every 30 to 60 groups. us a round before and
// after: 47 and 22 for 1024 groups of two draws among 1024 members, 111 and 47
// for 4096, 194 and 85 for 8192; 512 threads take 22, 54 and 100. Of the 47,
// 10 are 26 twists of the generator, 5 the launch and 30 four or five chunks
// of three to four passes. Twisting between the passes' barriers instead took
// 52: the last wavefronts then keep the block waiting.
constexpr int kRing = 4096;          // tempered generator words, a power of two
constexpr int kLeftWords = 1024;     // unconsumed words kept between rounds (at most 311)
constexpr int kPlaceThreads = 1024;  // groups per chunk at most
constexpr int kPlaceBuckets = 2048;  // lists of groups by victim, a power of two
static_assert(kPlaceThreads <= 1024, "a bucket holds a group in 10 bits");
// Dynamic LDS of a placement block: the generator's ring and two states, the
// chunk's child keys (a packed order has 4 bytes in LDS, 8 otherwise), the
// victim lists, then with keys in LDS 12 bytes per member.
constexpr std::size_t place_bytes(bool lds, int members) {
  return 8 * std::size_t(kRing) + 16 * 312 + (lds ? 12 : 16) * std::size_t(kPlaceThreads) + 4 * std::size_t(kPlaceBuckets) +
         4 * std::size_t(kPlaceThreads) + (lds ? 12 * std::size_t(members) : 0);
}

template <bool kLds>
struct PlaceKeys {
  // kLds: fitness and (wrong << 12 | nodes) staged in LDS; otherwise the
  // member arrays in HBM, read past the L1 so every wavefront sees the stores
  // of the previous chunk. Fields are copied out of the search state so that
  // stores to the keys never force it to be re-read.
  GAS double* fitness;
  GAS unsigned* wrong;
  GAS unsigned* nodes;
  int has_wrong;
  double* f;
  unsigned* wn;
  __device__ double fit(int m) const {
    if (kLds) return f[m];
    const unsigned long long bits = __hip_atomic_load((GAS unsigned long long*)(fitness + m), __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT);
    return __longlong_as_double((long long)bits);
  }
  __device__ std::uint64_t order(int m) const {
    if (!has_wrong) return 0;
    if (kLds) return wn[m];
    const unsigned w = __hip_atomic_load(wrong + m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned n = __hip_atomic_load(nodes + m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return std::uint64_t(w) << 32 | n;
  }
  __device__ std::uint64_t pack(unsigned w, unsigned n) const {
    return !has_wrong ? 0 : kLds ? std::uint64_t(w << 12 | n) : std::uint64_t(w) << 32 | n;
  }
  __device__ void store(int m, double fv, unsigned w, unsigned n) const {
    if (kLds) { f[m] = fv; wn[m] = w << 12 | n; }
    fitness[m] = fv;
    wrong[m] = w;
    nodes[m] = n;
  }
};
// `better` (fitness desc, wrong asc, nodes asc, index asc) of two keys.
__device__ inline bool key_better(double fa, std::uint64_t oa, int a, double fb, std::uint64_t ob, int b) {
  if (fa != fb) return fa > fb;
  if (oa != ob) return oa < ob;
  return a < b;
}

template <bool kLds>
__global__ __launch_bounds__(kPlaceThreads) void k_place(DSearch* all) {
  const DSearch& d = all[blockIdx.x];
  if (!search_live(d) || d.generational || d.place_lds != int(kLds)) return;
  extern __shared__ __attribute__((aligned(16))) unsigned char place_smem[];
  std::uint64_t* const ring = reinterpret_cast<std::uint64_t*>(place_smem);
  // Generator state, double-buffered: a twist reads one buffer and writes
  // the other (`cur` is the buffer holding the current state).
  std::uint64_t* const mt = ring + kRing;
  double* const child_f = reinterpret_cast<double*>(mt + 2 * 312);
  using Order = std::conditional_t<kLds, unsigned, std::uint64_t>;
  Order* const child_o = reinterpret_cast<Order*>(child_f + kPlaceThreads);
  // bucket: pass << 10 | last group entered; link: victim << 11 | (next group + 1).
  unsigned* const bucket = reinterpret_cast<unsigned*>(child_o + kPlaceThreads);
  unsigned* const link = bucket + kPlaceBuckets;
  double* const member_f = reinterpret_cast<double*>(link + kPlaceThreads);
  __shared__ int s_cut, s_best, s_kept, s_moved[3];
  __shared__ double s_best_f;
  __shared__ std::uint64_t s_best_o;
  const int t = threadIdx.x, lane = t & 63;
  const int P = d.P, B = d.B, rs = d.replacement_size, has_wrong = d.has_wrong;
  const std::uint64_t P64 = std::uint64_t(P);
  GAS const double* const c_fit = d.c_fit;
  GAS const unsigned* const c_wrong = d.c_wrong;
  GAS const unsigned* const c_nodes = d.c_nodes;
  GAS int* const placed = d.placed;
  const PlaceKeys<kLds> keys{d.fitness, d.wrong, d.nodes, has_wrong, member_f, reinterpret_cast<unsigned*>(member_f + (kLds ? P : 0))};
  // x mod P by a Barrett step: q = mulhi(x, floor((2^64-1)/P)) is
  // floor(x/P) or one less, so one conditional subtraction is exact.
  const std::uint64_t barrett = ~0ull / P64;
  const auto mod_p = [&](std::uint64_t x) {
    std::uint64_t r = x - __umul64hi(x, barrett) * P64;
    return int(r >= P64 ? r - P64 : r);
  };
  // Child keys of this thread's group, loaded a chunk ahead.
  double cf = 0;
  unsigned cw = 0, cn = 0;
  const auto fetch = [&](int c) {
    if (c < B) { cf = c_fit[c]; cw = c_wrong[c]; cn = c_nodes[c]; }
  };
  fetch(t);
  if (kLds) {
    constexpr int kStage = 8;  // loads in flight per thread while staging keys
    for (int m0 = 0; m0 < P; m0 += kPlaceThreads * kStage) {
      double f[kStage];
      unsigned w[kStage], n[kStage];
#pragma unroll
      for (int k = 0; k < kStage; ++k) {
        const int m = m0 + k * kPlaceThreads + t;
        if (m < P) { f[k] = keys.fitness[m]; w[k] = keys.wrong[m]; n[k] = keys.nodes[m]; }
      }
#pragma unroll
      for (int k = 0; k < kStage; ++k) {
        const int m = m0 + k * kPlaceThreads + t;
        if (m < P) { keys.f[m] = f[k]; keys.wn[m] = w[k] << 12 | n[k]; }
      }
    }
  }
  for (int i = t; i < kPlaceBuckets; i += kPlaceThreads) bucket[i] = 0;
  if (t < 3) s_moved[t] = 0;
  int cur = 0;
  for (int i = t; i < 312; i += kPlaceThreads) mt[i] = d.mt[i];
  int head = 0, tail = *d.n_left;
  for (int i = t; i < tail; i += kPlaceThreads) ring[i] = d.mt_left[i];
  __syncthreads();
  // Every thread, uniformly: the next state into the other buffer and its
  // 312 tempered words at the ring's tail. Words 0..155 read only the old
  // state; 156..310 read the new word i-156, and 311 the new words 0 and 155.
  const auto twist = [&] {
    const std::uint64_t* const old = mt + 312 * cur;
    std::uint64_t* const now = mt + 312 * (cur ^ 1);
    const auto put = [&](int i, std::uint64_t w) {
      now[i] = w;
      ring[(tail + i) & (kRing - 1)] = mt_temper(w);
    };
    if (t < 156) put(t, mt_next_word(old[t], old[t + 1], old[t + 156]));
    __syncthreads();
    if (t < 156) put(t + 156, mt_next_word(old[t + 156], t == 155 ? now[0] : old[t + 157], now[t]));
    __syncthreads();
    cur ^= 1;
    tail += 312;
  };
  const int W = min(kPlaceThreads, (kRing - 312) / rs);
  int b = 0, best = *d.best;
  double best_f = keys.fit(best);
  std::uint64_t best_o = keys.order(best);
  unsigned pass = 0;
  int chunk = 0;
  const int chunk_limit = 4 * B + 4096;
  while (b < B) {
    if (++chunk > chunk_limit) {
      if (t == 0) raise(d, 500);
      break;
    }
    const int n = min(W, B - b);
    while (tail - head < n * rs) twist();
    const bool active = t < n;
    const int base = head + t * rs;
    const std::uint64_t co = keys.pack(cw, cn);
    child_f[t] = cf;
    child_o[t] = Order(co);
    if (t == 0) s_cut = n;
    // The first draws and their members' keys stay in registers (named ones:
    // a dynamically indexed array would spill).
    int m0 = 0, m1 = 0, m2 = 0;
    double f0 = 0, f1 = 0, f2 = 0;
    std::uint64_t o0 = 0, o1 = 0, o2 = 0;
    const auto drawn = [&](int k) { return mod_p(ring[(base + k) & (kRing - 1)]); };
    if (active) {
      m0 = drawn(0);
      f0 = keys.fit(m0);
      o0 = keys.order(m0);
      if (rs > 1) { m1 = drawn(1); f1 = keys.fit(m1); o1 = keys.order(m1); }
      if (rs > 2) { m2 = drawn(2); f2 = keys.fit(m2); o2 = keys.order(m2); }
    }
    // The worst member drawn; `settled` reads the lists of the last pass.
    const auto pick = [&](bool settled) {
      int worst = -1;
      double wf = 0;
      std::uint64_t wo = 0;
      const auto consider = [&](int m, double f, std::uint64_t o) {
        if (settled) {
          const unsigned first = bucket[m & (kPlaceBuckets - 1)];
          int found = -1;
          if (first >> 10 == pass)
            for (int j = int(first & 1023u); j >= 0;) {
              const unsigned l = link[j];
              if (int(l >> 11) == m && j < t && j > found) found = j;
              j = int(l & 2047u) - 1;
            }
          if (found >= 0) { f = child_f[found]; o = child_o[found]; }
        }
        if (worst < 0 || key_better(wf, wo, worst, f, o, m)) { worst = m; wf = f; wo = o; }
      };
      consider(m0, f0, o0);
      if (rs > 1) consider(m1, f1, o1);
      if (rs > 2) consider(m2, f2, o2);
      for (int k = 3; k < rs; ++k) {
        const int m = drawn(k);
        consider(m, keys.fit(m), keys.order(m));
      }
      return worst;
    };
    int worst = active ? pick(false) : -1;
    for (int settled = 0; settled <= n; ++settled) {
      ++pass;
      if (active) {
        const unsigned old = atomicExch(&bucket[worst & (kPlaceBuckets - 1)], pass << 10 | unsigned(t));
        link[t] = unsigned(worst) << 11 | (old >> 10 == pass ? (old & 1023u) + 1u : 0u);
      }
      __syncthreads();
      const int now = active ? pick(true) : -1;
      const std::uint64_t moved = __ballot(now != worst);
      worst = now;
      // Three flags in turn: the next is cleared two barriers before its use.
      if (moved && lane == 0) s_moved[pass % 3] = 1;
      if (t == 0) s_moved[(pass + 1) % 3] = 0;
      __syncthreads();
      if (!s_moved[pass % 3]) break;
    }
    // `better` of the child (at the victim's index) against the best member,
    // which is no victim before the chunk's end.
    const bool place = active && worst != best;
    const bool raises = place && key_better(cf, co, worst, best_f, best_o, best);
    const std::uint64_t ends = __ballot(active && (!place || raises));
    if (ends && lane == 0) atomicMin(&s_cut, (t & ~63) + wave_first(ends) + 1);
    __syncthreads();
    const int cut = s_cut;
    if (place && t < cut) {
      // The last group of the chunk that took the member leaves its child there.
      bool last = true;
      for (int j = int(bucket[worst & (kPlaceBuckets - 1)] & 1023u); j >= 0;) {
        const unsigned l = link[j];
        last = last && !(int(l >> 11) == worst && j > t && j < cut);
        j = int(l & 2047u) - 1;
      }
      if (last) {
        keys.store(worst, cf, cw, cn);
        placed[worst] = b + t;
      }
    }
    if (t == cut - 1) {
      s_kept = place ? cut : cut - 1;
      s_best = raises ? worst : best;
      s_best_f = raises ? cf : best_f;
      s_best_o = raises ? co : best_o;
    }
    if (!kLds) __threadfence();
    __syncthreads();
    b += s_kept;
    best = s_best;
    best_f = s_best_f;
    best_o = s_best_o;
    head += cut * rs;
    fetch(b + t);
  }
  while (tail - head < 1) twist();
  const std::uint64_t next_seed = ring[head & (kRing - 1)];
  ++head;
  const int left = tail - head;
  for (int i = t; i < left && i < kLeftWords; i += kPlaceThreads) d.mt_left[i] = ring[(head + i) & (kRing - 1)];
  for (int i = t; i < 312; i += kPlaceThreads) d.mt[i] = mt[312 * cur + i];
  if (t == 0) {
    *d.n_left = left;
    *d.round_seed = next_seed;
    *d.best = best;
    d.n_pending[0] = 0;
    d.n_pending[1] = 0;
    d.n_pending[2] = 0;
    atomicAdd(d.round, 1);
  }
}

// ---- generational schedule (evolve.cpp:253-322; phase_population_cpu.cpp:269-312) ----
// Elites (the top `elites` members by the ranking order, best first; the
// best alone when elitism is 0) and the generation's seed, one generator
// word drawn after the history row as in the reference's loop.
__global__ __launch_bounds__(256) void k_gen_begin(DSearch* all) {
  const DSearch& d = all[blockIdx.x];
  if (!d.generational || !search_live(d)) return;
  const int t = threadIdx.x, P = d.P, want = d.elites > 0 ? d.elites : 1;
  const Keys keys{d.fitness, d.wrong, d.nodes, d.has_wrong};
  __shared__ unsigned taken[16384 / 32];
  __shared__ int cand[256];
  __shared__ std::uint64_t mt[312];
  for (int i = t; i < (P + 31) / 32; i += 256) taken[i] = 0;
  __syncthreads();
  for (int k = 0; k < want; ++k) {
    int b = -1;
    for (int m = t; m < P; m += 256)
      if (!((taken[m >> 5] >> (m & 31)) & 1u) && (b < 0 || better(keys, m, b))) b = m;
    cand[t] = b;
    __syncthreads();
    for (int span = 128; span > 0; span >>= 1) {
      if (t < span && cand[t + span] >= 0 && (cand[t] < 0 || better(keys, cand[t + span], cand[t]))) cand[t] = cand[t + span];
      __syncthreads();
    }
    const int pick = cand[0];
    if (t == 0) {
      if (k < d.elites) d.elite[k] = pick;
      if (k == 0) *d.best = pick;
      taken[pick >> 5] |= 1u << (pick & 31);
    }
    __syncthreads();
  }
  // One word of the run generator: the oldest unconsumed word, refilled by a
  // twist when none is left. Word 0 seeds generation 0 (stored by k_seed).
  if (*d.round == 0) return;
  int left = *d.n_left;
  if (left == 0) {
    for (int i = t; i < 312; i += 256) mt[i] = d.mt[i];
    __syncthreads();
    mt_twist<256>(mt);
    for (int i = t; i < 312; i += 256) { d.mt[i] = mt[i]; d.mt_left[i] = mt_temper(mt[i]); }
    left = 312;
    __syncthreads();
  }
  const std::uint64_t word = d.mt_left[0];
  std::uint64_t keep[4];
  for (int j = 0; j < 4; ++j) {
    const int i = t + 256 * j + 1;
    keep[j] = i < left ? d.mt_left[i] : 0;
  }
  __syncthreads();
  for (int j = 0; j < 4; ++j) {
    const int i = t + 256 * j + 1;
    if (i < left) d.mt_left[i - 1] = keep[j];
  }
  if (t == 0) {
    *d.round_seed = word;
    *d.n_left = left - 1;
  }
}
// Every child becomes the member of its index (keys now; rows in k_commit).
__global__ void k_gen_place(DSearch* all, const BlockMap* map) {
  const BlockMap bm = map[blockIdx.x];
  const DSearch& d = all[bm.search];
  const int m = bm.block * blockDim.x + threadIdx.x;
  if (!d.generational || !search_live(d) || m >= d.P) return;
  d.fitness[m] = d.c_fit[m];
  d.wrong[m] = d.c_wrong[m];
  d.nodes[m] = d.c_nodes[m];
  d.placed[m] = m;
}
__global__ void k_gen_end(DSearch* all) {
  const DSearch& d = all[blockIdx.x];
  if (!d.generational || !search_live(d) || threadIdx.x) return;
  d.n_pending[0] = 0;
  d.n_pending[1] = 0;
  d.n_pending[2] = 0;
  atomicAdd(d.round, 1);
}

// One wavefront per member: a placed child's row is copied across the lanes.
__global__ __launch_bounds__(64 * kVaryWaves) void k_commit(DSearch* all, const BlockMap* map) {
  const BlockMap bm = map[blockIdx.x];
  const DSearch& d = all[bm.search];
  const int m = __builtin_amdgcn_readfirstlane(bm.block * kVaryWaves + wave_index());
  if (!d.active || m >= d.P) return;
  const int c = d.placed[m];
  if (c >= 0) {
    const CRow src = child_row(d, c);
    const std::size_t o = std::size_t(m) * d.R;
    GAS int* const origin = d.cur_origin + o;
    GAS int* const site = d.cur_site + o;
    GAS Val* const cval = d.cur_cval + o;
    for (int i = wlane(); i < src.n; i += 64) { origin[i] = src.origin[i]; site[i] = src.site[i]; }
    for (int i = wlane(); i < src.nc; i += 64) cval[i] = src.cval[i];
  }
  if (wlane() == 0) {
    const std::uint64_t h = c >= 0 ? d.child_hash[c] : d.member_hash[m];
    if (c >= 0) {
      d.cur_n[m] = d.x_n[c];
      d.cur_nc[m] = d.x_nc[c];
      d.member_hash[m] = h;
      d.placed[m] = -1;
    }
    // The next round's member table (cleared during placement).
    if (search_live(d)) insert_member(d, m, h);
  }
}

// ---- evaluation session kernel (external bytecode) ----
struct DProg { GAS const Ins* code; GAS const Val* pool; int len, has_jumps, n_locals, fast, n_pool, result_tag; };
static_assert(sizeof(DProg) == 40, "program table entry size is part of the workspace bound");
__device__ inline ProgView view_of(const DProg& p) {
  return ProgView{p.code, p.pool, p.len, p.n_locals, p.has_jumps, p.fast, p.n_pool, p.result_tag};
}
// kFast: scores the programs certified for vm_fast (LDS: a score buffer of C
// doubles per wavefront); otherwise the rest (LDS: the general stacks).
// Scores a launch's typed straight-line (kFast) or general programs, one
// wavefront each, as block `block` of `blocks`.
template <bool kFast>
__device__ __attribute__((always_inline)) inline void score_programs(int block, int blocks, const DProg* progs, int n, const EvalParams& e,
                                                                     int slots, int temps, int shadow, unsigned char* smem, double* replay,
                                                                     double* fitness, unsigned* wrong, unsigned* counts) {
  const int wave = wave_index(), lane = threadIdx.x % 64;
  WaveStack st = stack_of(smem, kFast ? 0 : slots, kFast ? 0 : temps, wave, kFast ? 0 : shadow);
  double* scores = kFast ? reinterpret_cast<double*>(smem) + std::size_t(wave) * e.cd.C : nullptr;
  for (int i = block * kWavesPerBlock + wave; i < n; i += blocks * kWavesPerBlock) {
    const DProg p = progs[i];
    if (p.fast != int(kFast)) continue;  // 2: score_steps has it
    const EvalOut r = eval_program<kFast ? 1 : 0>(e, view_of(p), st, scores, lane, replay);
    if (lane == 0) {
      fitness[i] = r.fitness;
      wrong[i] = e.policy.metric == METRIC_LEGACY ? 0 : r.wrong;
      counts[3 * i + 0] = unsigned(e.cd.C);
      counts[3 * i + 1] = r.errors;
      counts[3 * i + 2] = r.timeouts;
    }
  }
}
template <bool kFast>
__global__ __launch_bounds__(kEvalThreads) void k_eval_programs(const DProg* progs, int n, EvalParams e, int slots, int temps,
                                                                 int shadow, double* fitness, unsigned* wrong, unsigned* counts) {
  extern __shared__ unsigned char smem[];
  __shared__ double replay[kFast ? kWavesPerBlock : 1][kFast ? kReplayWords : 1];
  score_programs<kFast>(int(blockIdx.x), int(gridDim.x), progs, n, e, slots, temps, shadow, smem, replay[kFast ? wave_index() : 0],
                        fitness, wrong, counts);
}
// A caller's looping programs on the decoded steps (certify_loop): one block
// per program, whose wavefronts take its 64-case tiles in turn in the visiting
// order (longest lists first). Totals are combined in LDS as in k_eval_tiles.
// LDS: step_slots(n_inputs) slots per wavefront, then C scores. Bound by the
// step loop's issue, as k_eval_loop; 512 programs x 200 list cases took
// 6.17 ms on the general VM (tagged values, a few cases' branches predicated
// per instruction) and take 0.45 ms here.
struct StepProg { GAS const Step* steps; int n_steps, index, result_tag; };
struct StepTotals {
  double sum[kWavesPerBlock], replay[kReplayWords];
  unsigned count[kWavesPerBlock][4];  // wrong, errors, timeouts, integral
};
__device__ __attribute__((always_inline)) inline void score_steps(int block, int blocks, const StepProg* progs, int n, const EvalParams& e,
                                                                  unsigned char* smem, StepTotals& part, double* fitness,
                                                                  unsigned* wrong, unsigned* counts) {
  const int waves = int(blockDim.x) / 64, wave = wave_index(), lane = threadIdx.x % 64;
  const int C = e.cd.C, n_in = e.cd.n_inputs, slots = step_slots(n_in);
  LAS std::int64_t* const sl = (LAS std::int64_t*)smem + std::size_t(wave) * slots * 64;
  double* const scores = reinterpret_cast<double*>(smem + std::size_t(waves) * slots * 64 * 8);
  for (int i = block; i < n; i += blocks) {  // one program per block, uniform
    const StepProg p = progs[i];
    const StepProgram sp = steps_load(p.steps, p.n_steps, lane);
    double isum = 0;
    unsigned w = 0, errs = 0, touts = 0;
    bool integral = true;  // C <= kScoreCases <= 4096
    for (int tile = wave * 64; tile < C; tile += waves * 64) {
      const bool active = tile + lane < C;
      const int c = active ? e.cd.order[tile + lane] : 0;
      const FastInputs in = fast_inputs(e.cd, n_in, c, active);
      const LaneResult r = sp.n <= 64 ? vm_steps<1>(sp, in, n_in, e.cd.arena, sl, lane, active, e.fuel, p.result_tag)
                                      : vm_steps<4>(sp, in, n_in, e.cd.arena, sl, lane, active, e.fuel, p.result_tag);
      if (active) {
        bool exact = false;
        const double sc = lane_score(e, r, expected_of(e.cd, c), exact);
        w += !exact;
        errs += r.err != ERR_NONE;
        touts += r.err == ERR_TIMEOUT;
        integral = integral && sc == double(std::int64_t(sc)) && sc >= -68719476736.0 && sc <= 68719476736.0;
        isum += sc;
        scores[c] = sc;
      }
    }
    const double ws = wave_sum_d(isum);
    const unsigned ww = wave_sum_u(w), we = wave_sum_u(errs), wt = wave_sum_u(touts);
    const bool wint = __ballot(!integral) == 0;
    if (lane == 0) {
      part.sum[wave] = ws;
      part.count[wave][0] = ww;
      part.count[wave][1] = we;
      part.count[wave][2] = wt;
      part.count[wave][3] = wint;
    }
    __syncthreads();  // every wavefront's scores and totals
    if (wave == 0) {
      double total = 0;
      unsigned tw = 0, te = 0, tt = 0;
      bool all_integral = true;
      for (int k = 0; k < waves; ++k) {
        total += part.sum[k];
        tw += part.count[k][0];
        te += part.count[k][1];
        tt += part.count[k][2];
        all_integral = all_integral && part.count[k][3] != 0;
      }
      const double f = all_integral ? total : canonical_from_scores(e, C, scores, lane, part.replay);
      if (lane == 0) {
        fitness[p.index] = f;
        wrong[p.index] = e.policy.metric == METRIC_LEGACY ? 0 : tw;
        counts[3 * p.index + 0] = unsigned(C);
        counts[3 * p.index + 1] = te;
        counts[3 * p.index + 2] = tt;
      }
    }
    __syncthreads();  // before the next program reuses the scores
  }
}
__global__ __launch_bounds__(kEvalThreads) void k_eval_steps(const StepProg* progs, int n, EvalParams e, double* fitness,
                                                              unsigned* wrong, unsigned* counts) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ StepTotals part;
  score_steps(int(blockIdx.x), int(gridDim.x), progs, n, e, smem, part, fitness, wrong, counts);
}
// A launch with both kinds of looping program: the first `general` blocks score
// the general VM's, each a chain of its own, and the others run the rest beside
// them. 511 programs on the steps and one whose stack is past the path took
// 6.41 ms one after the other and take 5.92 so; all of them on the general VM
// had taken 6.29.
__global__ __launch_bounds__(kEvalThreads) void k_eval_both(const DProg* progs, int n, int general, const StepProg* step_progs, int loops,
                                                             EvalParams e, int slots, int temps, int shadow, double* fitness,
                                                             unsigned* wrong, unsigned* counts) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ StepTotals part;
  const int block = int(blockIdx.x);
  if (block < general) score_programs<false>(block, general, progs, n, e, slots, temps, shadow, smem, nullptr, fitness, wrong, counts);
  else score_steps(block - general, int(gridDim.x) - general, step_progs, loops, e, smem, part, fitness, wrong, counts);
}
template <bool kFast>
__global__ __launch_bounds__(kEvalThreads) void k_eval_cases(DProg p, CaseData cd, int fuel, int slots, int temps, int shadow,
                                                              Val* values, int* errors) {
  extern __shared__ unsigned char smem[];
  const int wave = wave_index(), lane = threadIdx.x % 64;
  WaveStack st = stack_of(smem, kFast ? 0 : slots, kFast ? 0 : temps, wave, kFast ? 0 : shadow);
  const ProgView pv = view_of(p);
  FastProgram fp{};
  if (kFast) fp = fast_load(pv, lane);
  for (int tile = (blockIdx.x * kWavesPerBlock + wave) * 64; tile < cd.C; tile += gridDim.x * kWavesPerBlock * 64) {
    const int c = tile + lane;
    const bool active = c < cd.C;
    const LaneResult r = kFast ? vm_fast(fp, fast_inputs(cd, pv.n_locals, c, active), active, fuel, pv.result_tag)
                               : vm_run(pv, cd, active ? c : 0, active, fuel, st, lane);
    if (active) {
      Val v{};
      v.i = r.v; v.tag = r.t; v.b = r.b;
      values[c] = v;
      errors[c] = r.err;
    }
  }
}

// Lets a kernel take `bytes` of dynamic LDS. Without it a block has 64 KB in
// all, of which no kernel here declares more than 30 KB beside them.
void allow_lds(const void* kernel, std::size_t bytes) {
  if (bytes > 32 * 1024) HIP_OK(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes)));
}

// ---- device buffers ----
// Bump allocator over device chunks that double in size (1 MiB up to
// 256 MiB): a search's arrays take a handful of hipMalloc calls in all.
// Arrays are 256-byte aligned. A counting arena (`dry`) runs the same chunk
// arithmetic without touching the device, so the footprint of a search is
// known before any of its memory is allocated. The arena owns its chunks:
// it can be moved but not copied, and release() (or destruction) returns
// them to the device.
struct DeviceArena {
  std::vector<void*> blocks;
  std::size_t bytes = 0;     // bytes handed out
  std::size_t reserved = 0;  // bytes of device chunks held (the footprint)
  bool dry = false;
  char* cursor = nullptr;
  std::size_t left = 0, next_chunk = kFirstChunk;
  static constexpr std::size_t kFirstChunk = std::size_t(1) << 20;

  DeviceArena() = default;
  explicit DeviceArena(bool count_only) : dry(count_only) {}
  DeviceArena(const DeviceArena&) = delete;
  DeviceArena& operator=(const DeviceArena&) = delete;
  DeviceArena(DeviceArena&& o) noexcept { take(o); }
  DeviceArena& operator=(DeviceArena&& o) noexcept {
    if (this != &o) {
      release();
      take(o);
    }
    return *this;
  }
  ~DeviceArena() { release(); }

  void release() {
    for (void* p : blocks) (void)hipFree(p);
    blocks.clear();
    bytes = reserved = 0;
    cursor = nullptr;
    left = 0;
    next_chunk = kFirstChunk;
  }
  template <class T>
  GAS T* alloc(std::size_t n) {
    const std::size_t sz = (std::max<std::size_t>(n, 1) * sizeof(T) + 255) & ~std::size_t(255);
    if (sz > left) {
      const std::size_t chunk = std::max(sz, next_chunk);
      void* p = nullptr;
      if (!dry) {
        HIP_OK(hipMalloc(&p, chunk));
        blocks.push_back(p);
      }
      cursor = static_cast<char*>(p);
      left = chunk;
      reserved += chunk;
      next_chunk = std::min(next_chunk * 2, std::size_t(256) << 20);
    }
    void* p = cursor;
    if (!dry) cursor += sz;
    left -= sz;
    bytes += sz;
    return gbl(static_cast<T*>(p));
  }
  template <class T>
  GAS T* upload(const std::vector<T>& v) {
    GAS T* p = alloc<T>(v.size());
    if (!dry && !v.empty()) HIP_OK(hipMemcpy((void*)p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return p;
  }
  // Clears `n` elements (skipped when counting).
  template <class T>
  void zero(GAS T* p, std::size_t n) {
    if (!dry && n) HIP_OK(hipMemset((void*)p, 0, n * sizeof(T)));
  }

 private:
  void take(DeviceArena& o) {
    blocks = std::move(o.blocks);
    bytes = o.bytes;
    reserved = o.reserved;
    dry = o.dry;
    cursor = o.cursor;
    left = o.left;
    next_chunk = o.next_chunk;
    o.blocks.clear();
    o.bytes = o.reserved = 0;
    o.cursor = nullptr;
    o.left = 0;
    o.next_chunk = kFirstChunk;
  }
};

struct DeviceCases {
  CaseData cd{};
  void upload(DeviceArena& a, const Cases& c) {
    const int C = c.n, K = int(c.input_names.size());
    std::vector<std::int64_t> v(std::size_t(K) * C);
    std::vector<std::uint8_t> t(std::size_t(K) * C, TAG_INVALID), b(std::size_t(K) * C, 0);
    for (int i = 0; i < C; ++i)
      for (int k = 0; k < K; ++k) {
        const std::size_t src = std::size_t(i) * K + k, dst = std::size_t(k) * C + i;
        if (!c.set[src]) continue;
        v[dst] = c.inputs[src].i;
        t[dst] = c.inputs[src].tag;
        b[dst] = c.inputs[src].b;
      }
    std::vector<std::int64_t> ev(C);
    std::vector<std::uint8_t> et(C), eb(C);
    for (int i = 0; i < C; ++i) { ev[i] = c.expected[i].i; et[i] = c.expected[i].tag; eb[i] = c.expected[i].b; }
    std::vector<std::int64_t> arena = c.arena;
    if (arena.empty()) arena.push_back(0);
    cd.in_val = a.upload(v);
    cd.in_tag = a.upload(t);
    cd.in_b = a.upload(b);
    cd.exp_val = a.upload(ev);
    cd.exp_tag = a.upload(et);
    cd.exp_b = a.upload(eb);
    cd.arena = a.upload(arena);
    // Visiting order of the looping path: cases by descending total list
    // length (stable), so a tile's lanes run loops of similar length.
    const std::size_t n = std::size_t(C);
    std::vector<int> order(n);
    std::vector<std::int64_t> work(n, 0);
    for (int i = 0; i < C; ++i) {
      order[std::size_t(i)] = i;
      for (int k = 0; k < K; ++k) {
        const std::size_t src = std::size_t(i) * K + k;
        if (c.set[src] && c.inputs[src].tag == TAG_INT_LIST) work[std::size_t(i)] += std::int64_t(std::uint64_t(c.inputs[src].i) & 0xffff);
      }
    }
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return work[std::size_t(x)] > work[std::size_t(y)]; });
    cd.order = a.upload(order);
    cd.C = C;
    cd.n_inputs = K;
  }
};

int next_pow2(int x) { int p = 1; while (p < x) p <<= 1; return p; }

}  // namespace


// ====================== host side ======================

// One admitted search: host documents, tables and the device state it owns.
struct SearchState {
  SearchSpec spec;
  Task task;
  Grammar grammar;
  Cases train;
  SearchConfig cfg;
  Layout layout;
  PhaseGrammar phase;
  int P = 0, B = 0, R = 0, G = 0, rounds = 0, per_epoch = 0;
  int stepped = 0;  // rounds the host has stepped this search (it idles past `rounds`)
  int fuel = 0;
  double penalty = 0;
  bool may_jump = false;   // programs may go to the looping path (leaves_straight_line)
  bool statement = false;  // a Program entry: statement programs with grammar locals
  // The export name table: the names the first initial member uses, in
  // declaration order (the layout prototype of phase_population_cpu.cpp:195),
  // or an imported first program's own table; and the first binder id of an
  // exported program (-1: the generated population's numbering).
  std::vector<std::string> layout_names;
  int binder_base = -1;
  // Rows of an imported initial population, held until they are uploaded.
  ImportedPopulation imported;
  bool has_import = false;
  DeviceArena arena;
  DSearch d{};
  double init_ms = 0;
  bool configured = false, retired = false;

  explicit SearchState(const SearchSpec& s) : spec(s) {
    task = load_task(s.task_path);
    grammar = load_grammar_file(task.grammar_path);
    train = load_cases(task.train_path);
    cfg = default_search_config();
    if (!s.search_path.empty()) {
      std::ifstream in(s.search_path);
      if (!in) throw std::invalid_argument("search config: cannot read " + s.search_path);
      std::ostringstream text;
      text << in.rdbuf();
      apply_search(cfg, json::parse(text.str()));
    }
    if (s.population) cfg.population = *s.population;
    if (s.generations) cfg.generations = *s.generations;
    if (s.seed) cfg.seed = *s.seed;
    if (!cfg.resident) throw Unsupported("native_ast representation (host reproduction)");
    if (cfg.site_depth < 1 && s.init_path.empty())
      throw Unsupported("site_depth 0 (initial population from the native generator)");
    if (cfg.population < 2 || cfg.population > 16384) throw Unsupported("population outside 2..16384");
    if (cfg.elitism < 0 || cfg.elitism >= cfg.population) throw std::invalid_argument("elite_count must be >= 0 and < population_size");
    P = cfg.population;
    B = cfg.schedule == Schedule::Generational ? P : (cfg.batch ? cfg.batch : P);
    if (B > P || P % B) throw std::invalid_argument("search config: steady_state batch must divide the population");
    G = cfg.generations;
    rounds = int((std::int64_t(P) * G) / B);
    per_epoch = P / B;
    penalty = cfg.penalty.value_or(task.case_cap);
    fuel = cfg.fuel.value_or(int(grammar.fuel));
    // Inputs must exactly cover the grammar inputs.
    {
      std::vector<std::string> want;
      for (const auto& in : grammar.inputs) want.push_back(in.name);
      std::sort(want.begin(), want.end());
      if (want != train.input_names) throw std::invalid_argument("every fitness case must supply every compiled grammar input");
      for (std::size_t k = 0; k < train.input_names.size(); ++k)
        for (const auto& in : grammar.inputs)
          if (in.name == train.input_names[k] && in.type != train.input_types[k])
            throw std::invalid_argument("case input type disagrees with the grammar");
    }
    layout = whole_program_layout(grammar);
    phase = compile_phase(grammar, grammar.entry, grammar.max_depth, unsigned(cfg.site_depth), train.input_names);
    R = std::min<int>(kPhaseCapacity, int(layout.max_variable_nodes));
    statement = grammar.nts[grammar.entry].cat == Cat::Program;
    may_jump = leaves_straight_line(phase, train.input_types, layout, R, statement);
    if (!s.init_path.empty()) {
      imported = load_population(s.init_path, grammar, phase, unsigned(cfg.site_depth), R, std::size_t(P));
      has_import = true;
      layout_names = imported.layout_names;
      binder_base = imported.binder_base;
    }
  }

  // Allocates every device array of the search in its arena.
  // One device block of exactly the search's bytes.
  void allocate() {
    DeviceArena count(true);
    (void)build(count);
    arena.next_chunk = count.bytes;
    d = build(arena);
  }
  // Device bytes the search is admitted by: its arrays in chunks doubling from
  // 1 MiB, never less than the one block they are allocated as; computed
  // without allocating.
  std::size_t planned_bytes() const {
    DeviceArena count(true);
    (void)build(count);
    return count.reserved;
  }

  DSearch build(DeviceArena& a) const {
    DSearch x{};
    x.active = 1;
    x.P = P; x.B = B; x.R = R;
    // A traversal lowers to at most 64 instructions and 8 constants of its
    // own besides those of its nodes, and keeps 9 temporaries live.
    const int walks = phase.traversals;
    // A for_range lowers to 23 instructions and 4 constants of its own, and
    // takes at least three nodes (itself, its bound and its body).
    const int loops = statement ? (R + 2) / 3 : 0;
    x.code_cap = 4 * R + 8 + 64 * walks + 23 * loops;
    // The general VM schedules instruction indices below 8191.
    if (x.code_cap > 8190) throw Unsupported("lowered programs longer than 8190 instructions");
    x.pool_cap = 2 * R + 8 + 8 * walks + 4 * loops;
    x.stack_slots = std::min(kMaxStack, 2 * int(layout.slot_max_depth) + 2);
    // Statement programs lower through the hidden-locals instantiation too.
    x.walks = walks > 0 || statement || phase.has_let;
    x.imported = has_import ? 1 : 0;
    x.temp_slots = statement || phase.has_let ? std::min(64 - int(train.input_names.size()), int(hidden_local_bound(grammar)))
                   : walks  ? std::max(0, std::min(64 - int(train.input_names.size()), 9 * std::min(walks, 8)))
                            : 0;
    x.input_shadow = phase.input_writes ? int(train.input_names.size()) : 0;
    x.temp_slots += x.input_shadow;
    x.rounds = rounds; x.per_epoch = per_epoch;
    x.fuel = fuel; x.lanes = 512; x.penalty = penalty; x.policy = task.policy;
    x.pressure = std::clamp(cfg.tournament, 1, P);
    x.replacement_size = cfg.replacement_size;
    x.p_mut = cfg.mutation_probability;
    x.pol = OpPolicy{cfg.counted, cfg.uniform_phase, cfg.crossover_probability, cfg.crossover_attempts, cfg.mutation_max_nodes};
    x.slot = SlotInfo{phase.root, 0, int(layout.slot_max_depth), cfg.site_depth, int(layout.max_variable_nodes), R, statement ? 1 : 0};
    x.fixed_nodes = int(layout.fixed_nodes);
    x.grammar_sites = cfg.grammar_sites;
    x.has_wrong = task.policy.metric != METRIC_LEGACY;
    x.expected_type = statement ? kStatementType : grammar.nts[grammar.entry].type;
    x.n_locals = int(train.input_names.size());
    x.site_depth = cfg.site_depth;
    x.seed = cfg.seed;
    // The phase tables back to back in one block (stage_phase_tables).
    std::vector<unsigned char> tables;
    const auto append = [&](const auto& v) {
      using T = typename std::decay_t<decltype(v)>::value_type;
      const std::size_t at = tables.size();
      tables.resize(at + table_bytes(v.size() * sizeof(T)));
      if (!v.empty()) std::memcpy(tables.data() + at, v.data(), v.size() * sizeof(T));
      return at;
    };
    const std::size_t o_expr = append(phase.exprs), o_prod = append(phase.prods), o_nt = append(phase.nts),
                      o_dom = append(phase.domains), o_val = append(phase.values), o_min = append(phase.minimum);
    GAS unsigned char* const base = a.upload(tables);
    x.g = PhaseTables{(GAS const PExpr*)(base + o_expr), int(phase.exprs.size()), (GAS const PProd*)(base + o_prod),
                      int(phase.prods.size()), (GAS const PNt*)(base + o_nt), int(phase.nts.size()),
                      (GAS const PDomain*)(base + o_dom), int(phase.domains.size()), (GAS const Val*)(base + o_val),
                      int(phase.values.size()), (GAS const unsigned*)(base + o_min), phase.depth_count, phase.logical_count,
                      phase.site_depth ? 1 : 0, phase.root};
    x.local_types = a.upload(train.input_types);
    DeviceCases dc;
    dc.upload(a, train);
    x.cd = dc.cd;
    const std::size_t slots = std::size_t(std::max(P, B));
    if (x.cd.C <= kScoreCases) x.loop_scores = a.alloc<double>(slots * std::size_t(x.cd.C));
    x.looping = x.cd.C <= kScoreCases && may_jump;
    if (x.looping) {
      x.loop_acc = a.alloc<LoopAcc>(slots);
      a.zero(x.loop_acc, slots);
    }
    const std::size_t rows = std::size_t(P) * R, crows = std::size_t(B) * R;
    x.cur_origin = a.alloc<int>(rows); x.cur_site = a.alloc<int>(rows); x.cur_cval = a.alloc<Val>(rows);
    x.cur_n = a.alloc<int>(P); x.cur_nc = a.alloc<int>(P);
    x.x_origin = a.alloc<int>(crows); x.x_site = a.alloc<int>(crows); x.x_cval = a.alloc<Val>(crows);
    x.x_n = a.alloc<int>(B); x.x_nc = a.alloc<int>(B);
    x.t_origin = a.alloc<int>(crows); x.t_site = a.alloc<int>(crows); x.t_cval = a.alloc<Val>(crows);
    x.s_origin = a.alloc<int>(crows); x.s_site = a.alloc<int>(crows); x.s_cval = a.alloc<Val>(crows);
    x.fitness = a.alloc<double>(P); x.wrong = a.alloc<unsigned>(P); x.nodes = a.alloc<unsigned>(P);
    x.stats = a.alloc<OpStats>(B); x.reuse = a.alloc<int>(B);
    x.c_fit = a.alloc<double>(B); x.c_wrong = a.alloc<unsigned>(B); x.c_nodes = a.alloc<unsigned>(B);
    const int code_rows = std::max(P, B);
    x.code = a.alloc<Ins>(std::size_t(code_rows) * x.code_cap);
    x.pool = a.alloc<Val>(std::size_t(code_rows) * x.pool_cap);
    x.code_len = a.alloc<int>(code_rows); x.pool_len = a.alloc<int>(code_rows); x.code_jumps = a.alloc<int>(code_rows);
    x.child_hash = a.alloc<std::uint64_t>(B);
    x.pending = a.alloc<int>(2 * std::size_t(B)); x.n_pending = a.alloc<int>(3);
    const int tsize = next_pow2(2 * P);
    x.table_key = a.alloc<std::uint64_t>(tsize); x.table = a.alloc<int>(tsize); x.table_mask = tsize - 1;
    x.mt = a.alloc<std::uint64_t>(312); x.mt_left = a.alloc<std::uint64_t>(kLeftWords); x.n_left = a.alloc<int>(1);
    x.round_seed = a.alloc<std::uint64_t>(1);
    x.member_hash = a.alloc<std::uint64_t>(P);
    // Placement keys (fitness, wrong << 12 | nodes) in LDS.
    x.place_lds = P <= 8192 && train.n < (1 << 20) && int(layout.fixed_nodes) + R < 4096;
    x.round = a.alloc<int>(1); x.best = a.alloc<int>(1); x.placed = a.alloc<int>(P);
    x.hist_origin = a.alloc<int>(std::size_t(G) * R); x.hist_cval = a.alloc<Val>(std::size_t(G) * R);
    x.hist_n = a.alloc<int>(G); x.hist_nc = a.alloc<int>(G);
    x.hist_fit = a.alloc<double>(G); x.hist_wrong = a.alloc<unsigned>(G);
    x.hist_all = a.alloc<double>(std::size_t(G) * P);
    x.counters = a.alloc<Counters>(1);
    x.generational = cfg.schedule == Schedule::Generational;
    x.elites = x.generational ? cfg.elitism : 0;
    x.elite = a.alloc<int>(x.generational ? std::size_t(P) : 1);  // any elite count below P
    x.early_exit = spec.early_exit ? 1 : 0;
    x.stop = a.alloc<int>(1);
    x.e_errors = a.alloc<unsigned>(code_rows); x.e_timeouts = a.alloc<unsigned>(code_rows);
    x.e_fuel = a.alloc<unsigned long long>(code_rows);
    x.error = a.alloc<int>(1);
    a.zero(x.n_pending, 3);
    a.zero(x.counters, 1);
    a.zero(x.error, 1);
    a.zero(x.round, 1);
    a.zero(x.stop, 1);
    return x;
  }

  template <class T>
  std::vector<T> down(GAS const T* p, std::size_t n) const {
    std::vector<T> v(n);
    if (n) HIP_OK(hipMemcpy(v.data(), (const void*)p, n * sizeof(T), hipMemcpyDeviceToHost));
    return v;
  }
  int device_error() const { return down(d.error, 1)[0]; }
};

struct KernelTimer {
  bool on = false;
  std::map<std::string, double> ms;
  std::vector<std::pair<std::string, std::pair<hipEvent_t, hipEvent_t>>> pending;
  template <class F>
  void time(const char* name, hipStream_t s, F&& launch) {
    if (!on) { launch(); return; }
    hipEvent_t a, b;
    HIP_OK(hipEventCreate(&a));
    HIP_OK(hipEventCreate(&b));
    HIP_OK(hipEventRecord(a, s));
    launch();
    HIP_OK(hipEventRecord(b, s));
    pending.push_back({name, {a, b}});
  }
  void collect() {
    for (auto& p : pending) {
      HIP_OK(hipEventSynchronize(p.second.second));
      float t = 0;
      HIP_OK(hipEventElapsedTime(&t, p.second.first, p.second.second));
      ms[p.first] += t;
      (void)hipEventDestroy(p.second.first);
      (void)hipEventDestroy(p.second.second);
    }
    pending.clear();
  }
};

// ---- evaluation launch autotuner ----
// Launch shapes of the evaluation kernels that leave every result unchanged:
// pending programs per wavefront of the typed straight-line kernel (its
// grid, and so how many blocks stage the case set), and tiles per work item
// of the looping kernel (cases per item = 64 * loop_group).
struct TuneChoice {
  int fast_programs = 1;
  int loop_group = 1;
};
// Choices measured so far in this process, by batch shape.
std::mutex tune_mutex;
std::map<std::string, TuneChoice> tune_cache;

struct Batch::Impl {
  std::vector<std::unique_ptr<SearchState>> searches;  // every search ever added (stable indices)
  std::vector<int> live;                                // searches of the round table, in table order
  bool dirty = true;                                    // table, grids and graph need rebuilding
  int* d_status = nullptr;                              // k_status output, 3 ints per table entry
  std::size_t status_cap = 0;
  DSearch* d_all = nullptr;
  hipStream_t stream = nullptr;
  KernelTimer timer;
  int max_P = 0, max_B = 0, max_slots = 0, max_table = 0, max_rounds = 0;
  std::size_t place_lds_bytes = 0, place_hbm_bytes = 0;  // dynamic LDS of the two placement variants
  double run_ms = 0, init_ms = 0;
  bool graph_ready = false;
  hipGraphExec_t graph_exec = nullptr;
  // Side streams of a round's parallel branches (default priority, like
  // `stream`) and the events that fork them from `stream` and join them
  // back; captured, they become parallel branches of the round graph.
  static constexpr int kSides = 2;
  hipStream_t side[kSides] = {};
  hipEvent_t fork_ev = nullptr, join_ev[kSides] = {};
  ~Impl() {
    if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
    if (d_all) (void)hipFree(d_all);
    if (d_status) (void)hipFree(d_status);
    for (int i = 0; i < kSides; ++i) {
      if (side[i]) (void)hipStreamDestroy(side[i]);
      if (join_ev[i]) (void)hipEventDestroy(join_ev[i]);
    }
    if (fork_ev) (void)hipEventDestroy(fork_ev);
    if (stream) (void)hipStreamDestroy(stream);
  }
  void make_streams() {
    if (!stream) HIP_OK(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    if (fork_ev) return;
    HIP_OK(hipEventCreateWithFlags(&fork_ev, hipEventDisableTiming));
    for (int i = 0; i < kSides; ++i) {
      HIP_OK(hipStreamCreateWithFlags(&side[i], hipStreamNonBlocking));
      HIP_OK(hipEventCreateWithFlags(&join_ev[i], hipEventDisableTiming));
    }
  }
  // Runs parts[0] on `stream` and parts[1..] on side streams forked from it,
  // then joins them: the parts must touch disjoint data. With the kernel
  // timer on, every part runs on `stream` in order, so each launch's events
  // bracket that launch alone.
  void branches(const std::vector<std::function<void(hipStream_t)>>& parts) {
    if (timer.on) {
      for (const auto& part : parts) part(stream);
      return;
    }
    HIP_OK(hipEventRecord(fork_ev, stream));
    for (std::size_t i = 1; i < parts.size(); ++i) HIP_OK(hipStreamWaitEvent(side[i - 1], fork_ev, 0));
    parts[0](stream);
    for (std::size_t i = 1; i < parts.size(); ++i) {
      parts[i](side[i - 1]);
      HIP_OK(hipEventRecord(join_ev[i - 1], side[i - 1]));
      HIP_OK(hipStreamWaitEvent(stream, join_ev[i - 1], 0));
    }
  }
  std::size_t eval_fast_lds = 0, eval_general_lds = 0, eval_tiles_lds = 0;  // dynamic LDS of the evaluation kernels
  std::size_t eval_loop_lds = 0;  // the looping path's slots
  std::size_t vary_lds_bytes = 0;  // phase-table copy of the staged reproduction kernel
  bool vary_global = false;        // some search reproduces from global tables
  bool any_generational = false;

  // Flat grids: every search contributes exactly its own blocks.
  struct Grid { GAS BlockMap* map = nullptr; int blocks = 0; };
  DeviceArena map_arena;
  Grid g_init, g_lower, g_eval_init, g_vary_staged, g_vary_global, g_vary_staged_d, g_vary_global_d, g_lower_c, g_lower_w, g_table, g_member,
      g_eval, g_eval_tiles, g_eval_general, g_eval_loop, g_finish, g_member_w;
  // Evaluation launch shapes of the round (the autotuner's choice, or the
  // fixed default: one program per wavefront, one 64-case tile per item).
  TuneChoice tune;
  int autotune = 1;  // 0 off, 1 above kTuneWork, 2 always
  bool seam = false;  // rounds driven through the owner seam
  bool tuned = false;
  std::string tune_report;  // JSON of the last tuning pass
  bool any_walks(const std::vector<int>& ids) const {
    for (int id : ids)
      if (searches[std::size_t(id)]->d.walks) return true;
    return false;
  }
  // Some grammar can lower to jumps (if/and/or or traversals): the looping
  // evaluation kernel has work.
  bool any_jumps(const std::vector<int>& ids) const {
    for (int id : ids)
      if (searches[std::size_t(id)]->may_jump) return true;
    return false;
  }
  bool loop_kernel = false;  // any_jumps(live)
  template <class Blocks>
  Grid build_grid(DeviceArena& arena, const std::vector<int>& table, Blocks blocks_of) {
    std::vector<BlockMap> v;
    for (std::size_t i = 0; i < table.size(); ++i) {
      const int nb = blocks_of(*searches[std::size_t(table[i])]);
      for (int j = 0; j < nb; ++j) v.push_back(BlockMap{int(i), j, nb});
    }
    Grid g;
    g.blocks = int(v.size());
    if (!v.empty()) g.map = arena.upload(v);
    return g;
  }
  static int up(int x, int k) { return (x + k - 1) / k; }
  void build_round_grids() {
    map_arena.release();
    const auto vary = [&](bool staged, bool defer) {
      return build_grid(map_arena, live, [&](const SearchState& s) {
        return (s.d.stage_tables != 0) == staged && (s.d.defer != 0) == defer ? up(s.B, kVaryWaves) : 0;
      });
    };
    const auto lower = [&](bool walks) {
      return build_grid(map_arena, live, [&](const SearchState& s) {
        return s.d.defer && (s.d.walks != 0) == walks ? up(s.B, kVaryWaves) : 0;
      });
    };
    g_vary_staged = vary(true, false);
    g_vary_global = vary(false, false);
    g_vary_staged_d = vary(true, true);
    g_vary_global_d = vary(false, true);
    g_lower_c = lower(false);
    g_lower_w = lower(true);
    g_table = build_grid(map_arena, live, [&](const SearchState& s) { return up(s.d.table_mask + 1, 256); });
    g_member = build_grid(map_arena, live, [&](const SearchState& s) { return up(s.P, 128); });
    // one wavefront per child / member
    g_member_w = build_grid(map_arena, live, [&](const SearchState& s) { return up(s.P, kVaryWaves); });
    g_eval = typed_grid(map_arena, tune.fast_programs);
    g_eval_tiles = tiles_grid(map_arena, live, false);
    g_eval_general = eval_grid(map_arena, 1);
    g_eval_loop = loop_grid(map_arena, tune.loop_group);
    g_finish = finish_grid(map_arena, live, false);
  }
  // Evaluation grids of the live searches: `per_wave` pending programs per
  // wavefront of the typed and general kernels; `group` tiles per work item
  // of the looping kernel.
  Grid eval_grid(DeviceArena& arena, int per_wave) {
    return build_grid(arena, live, [&](const SearchState& s) { return std::min(4096, up(s.B, kWavesPerBlock * per_wave)); });
  }
  // The typed kernels: k_eval<1> for searches whose cases fit one tile,
  // k_eval_tiles (one block per program) for the rest.
  Grid typed_grid(DeviceArena& arena, int per_wave) {
    return build_grid(arena, live, [&](const SearchState& s) {
      return s.d.typed_tiles ? 0 : std::min(4096, up(s.B, kWavesPerBlock * per_wave));
    });
  }
  Grid tiles_grid(DeviceArena& arena, const std::vector<int>& table, bool members) {
    return build_grid(arena, table, [&](const SearchState& s) { return s.d.typed_tiles ? std::min(4096, members ? s.P : s.B) : 0; });
  }
  Grid finish_grid(DeviceArena& arena, const std::vector<int>& table, bool members) {
    return build_grid(arena, table, [&](const SearchState& s) {
      return s.d.looping && s.d.cd.C > 64 ? up(members ? s.P : s.B, kFinishPrograms) : 0;
    });
  }
  Grid loop_grid(DeviceArena& arena, int group) {
    return build_grid(arena, live, [&](const SearchState& s) { return s.d.looping ? loop_blocks(s.d.cd.C, s.B, group) : 0; });
  }

  // Allocates one search and fixes its kernel variants and LDS needs.
  void configure(SearchState& s) {
    constexpr std::size_t kStageLimit = 64 * 1024;
    s.configured = true;
    s.allocate();
    s.d.profile = timer.on ? 1 : 0;
    s.d.defer = s.may_jump;
    s.d.stage_tables = phase_tables_bytes(s.d.g) <= kStageLimit;
    const std::size_t stacks = std::size_t(kWavesPerBlock) * (s.d.stack_slots + s.d.temp_slots) * 64 * 10;
    const std::size_t score_buf = std::size_t(kWavesPerBlock) * 8 * s.d.cd.C;
    s.d.general_scores = s.d.cd.C <= kScoreCases && stacks + score_buf <= kLdsLimit;
    const std::size_t cases = staged_case_bytes(s.d.cd.C, staged_inputs_of(s.d.n_locals, s.d.cd.n_inputs));
    s.d.stage_cases = s.d.cd.C <= kScoreCases && cases <= 48 * 1024 && score_buf + cases + 16 <= kLdsLimit;
    s.d.typed_tiles = s.d.cd.C > 64 && s.d.cd.C <= kScoreCases;
  }
  // LDS sizes and kernel attributes for a table of searches.
  void size_kernels(const std::vector<int>& table) {
    eval_fast_lds = eval_general_lds = eval_tiles_lds = vary_lds_bytes = place_lds_bytes = place_hbm_bytes = 0;
    eval_loop_lds = 0;
    vary_global = any_generational = false;
    max_P = max_B = max_slots = max_table = 0;
    for (int id : table) {
      const SearchState& x = *searches[std::size_t(id)];
      const std::size_t stacks = std::size_t(kWavesPerBlock) * (x.d.stack_slots + x.d.temp_slots) * 64 * 10;
      const std::size_t score_buf = std::size_t(kWavesPerBlock) * 8 * x.d.cd.C;
      eval_general_lds = std::max(eval_general_lds, stacks + (x.d.general_scores ? score_buf : 0));
      const std::size_t cases = x.d.stage_cases ? staged_case_bytes(x.d.cd.C, staged_inputs_of(x.d.n_locals, x.d.cd.n_inputs)) : 0;
      if (x.d.cd.C <= kScoreCases) {
        if (!x.d.typed_tiles) eval_fast_lds = std::max(eval_fast_lds, score_buf + cases);
        eval_loop_lds = std::max(eval_loop_lds, std::size_t(step_slots(staged_inputs_of(x.d.n_locals, x.d.cd.n_inputs))) * 64 * 8);
      }
      if (x.d.typed_tiles) eval_tiles_lds = std::max(eval_tiles_lds, std::size_t(8) * x.d.cd.C);
      if (x.d.stage_tables) vary_lds_bytes = std::max(vary_lds_bytes, phase_tables_bytes(x.d.g));
      else vary_global = true;
      if (x.d.place_lds) place_lds_bytes = std::max(place_lds_bytes, place_bytes(true, x.P));
      else place_hbm_bytes = place_bytes(false, x.P);
      any_generational = any_generational || x.d.generational;
      max_P = std::max(max_P, x.P);
      max_B = std::max(max_B, x.B);
      max_slots = std::max(max_slots, x.d.stack_slots);
      max_table = std::max(max_table, x.d.table_mask + 1);
    }
    allow_lds(reinterpret_cast<const void*>(&k_init_pop<true>), vary_lds_bytes);
    allow_lds(reinterpret_cast<const void*>(&k_vary<true, false>), vary_lds_bytes);
    allow_lds(reinterpret_cast<const void*>(&k_vary<true, true>), vary_lds_bytes);
    allow_lds(reinterpret_cast<const void*>(&k_lower<false>), vary_lds_bytes);
    allow_lds(reinterpret_cast<const void*>(&k_lower<true>), vary_lds_bytes);
    allow_lds(reinterpret_cast<const void*>(&k_eval<0>), eval_general_lds);
    allow_lds(reinterpret_cast<const void*>(&k_eval<1>), eval_fast_lds);
    allow_lds(reinterpret_cast<const void*>(&k_eval_tiles), eval_tiles_lds);
    allow_lds(reinterpret_cast<const void*>(&k_eval_loop<false>), eval_loop_lds);
    allow_lds(reinterpret_cast<const void*>(&k_eval_loop<true>), eval_loop_lds);
    allow_lds(reinterpret_cast<const void*>(&k_place<true>), place_lds_bytes);
    allow_lds(reinterpret_cast<const void*>(&k_place<false>), place_hbm_bytes);
  }
  // Builds and scores the initial populations of `ids` (not yet in the
  // round table) on the stream, through a table of their own.
  void init_searches(const std::vector<int>& ids) {
    if (ids.empty()) return;
    std::vector<DSearch> host;
    for (int id : ids) host.push_back(searches[std::size_t(id)]->d);
    const int n = int(ids.size());
    DeviceArena tmp;
    GAS DSearch* table = tmp.upload(host);
    DSearch* t = (DSearch*)table;
    size_kernels(ids);
    const Grid gi = build_grid(tmp, ids, [&](const SearchState& x) { return up(x.P, kVaryWaves); });
    const Grid gl = build_grid(tmp, ids, [&](const SearchState& x) { return up(x.P, kVaryWaves); });
    const Grid ge = build_grid(tmp, ids, [&](const SearchState& x) { return std::min(4096, up(x.P, kWavesPerBlock)); });
    // Imported populations: their rows go up in place of k_init_pop's
    // (which skips those searches); the staging vectors live until the
    // stream is synchronized below.
    std::vector<std::vector<int>> up_i;
    std::vector<std::vector<Val>> up_v;
    for (int id : ids) {
      SearchState& x = *searches[std::size_t(id)];
      if (!x.has_import) continue;
      const std::size_t P = std::size_t(x.P), R = std::size_t(x.R);
      if (x.imported.rows.size() != P) throw std::logic_error("imported population size");
      std::vector<int> origin(P * R, 0), site(P * R, -1), n(P), nc(P), placed(P, -1);
      std::vector<Val> cval(P * R, Val{});
      for (std::size_t m = 0; m < P; ++m) {
        const PhaseRow& r = x.imported.rows[m];
        if (r.origin.size() > R || r.cval.size() > R) throw std::logic_error("imported row capacity");
        std::copy(r.origin.begin(), r.origin.end(), origin.begin() + std::ptrdiff_t(m * R));
        std::copy(r.site.begin(), r.site.end(), site.begin() + std::ptrdiff_t(m * R));
        std::copy(r.cval.begin(), r.cval.end(), cval.begin() + std::ptrdiff_t(m * R));
        n[m] = int(r.origin.size());
        nc[m] = int(r.cval.size());
      }
      const auto put = [&](GAS void* to, const void* from, std::size_t bytes) {
        HIP_OK(hipMemcpyAsync((void*)to, from, bytes, hipMemcpyHostToDevice, stream));
      };
      put(x.d.cur_origin, origin.data(), origin.size() * sizeof(int));
      put(x.d.cur_site, site.data(), site.size() * sizeof(int));
      put(x.d.cur_cval, cval.data(), cval.size() * sizeof(Val));
      put(x.d.cur_n, n.data(), n.size() * sizeof(int));
      put(x.d.cur_nc, nc.data(), nc.size() * sizeof(int));
      put(x.d.placed, placed.data(), placed.size() * sizeof(int));
      for (auto* v : {&origin, &site, &n, &nc, &placed}) up_i.push_back(std::move(*v));
      up_v.push_back(std::move(cval));
    }
    timer.time("k_init_pop", stream,
               [&] {
                 if (vary_lds_bytes)
                   hipLaunchKernelGGL(k_init_pop<true>, dim3(gi.blocks), dim3(64 * kVaryWaves), vary_lds_bytes, stream, t, gi.map);
                 if (vary_global) hipLaunchKernelGGL(k_init_pop<false>, dim3(gi.blocks), dim3(64 * kVaryWaves), 0, stream, t, gi.map);
               });
    timer.time("k_lower_members", stream,
               [&] { hipLaunchKernelGGL(k_lower_members<false>, dim3(gl.blocks), dim3(64 * kVaryWaves), 0, stream, t, gl.map); });
    if (any_walks(ids))
      timer.time("k_lower_members_walks", stream,
                 [&] { hipLaunchKernelGGL(k_lower_members<true>, dim3(gl.blocks), dim3(64 * kVaryWaves), 0, stream, t, gl.map); });
    timer.time("k_eval_init", stream,
               [&] { hipLaunchKernelGGL(k_eval<1>, dim3(ge.blocks), dim3(kEvalThreads), eval_fast_lds, stream, t, ge.map, 0); });
    const Grid gt = tiles_grid(tmp, ids, true);
    if (gt.blocks)
      timer.time("k_eval_init_tiles", stream, [&] {
        hipLaunchKernelGGL(k_eval_tiles, dim3(gt.blocks), dim3(kEvalThreads), eval_tiles_lds, stream, t, gt.map, 0);
      });
    if (any_jumps(ids))
      timer.time("k_eval_init_loop", stream, [&] {
        const Grid gp = build_grid(tmp, ids, [&](const SearchState& x) { return x.d.looping ? loop_blocks(x.d.cd.C, x.P) : 0; });
        if (gp.blocks) hipLaunchKernelGGL(k_eval_loop<false>, dim3(gp.blocks), dim3(64), eval_loop_lds, stream, t, gp.map, 0, 1);
        const Grid gf = finish_grid(tmp, ids, true);
        if (gf.blocks) hipLaunchKernelGGL(k_loop_finish, dim3(gf.blocks), dim3(kEvalThreads), 0, stream, t, gf.map, 0, 1);
      });
    timer.time("k_eval_init_general", stream, [&] {
      hipLaunchKernelGGL(k_eval<0>, dim3(ge.blocks), dim3(kEvalThreads), eval_general_lds, stream, t, ge.map, 0);
    });
    timer.time("k_tally_init", stream, [&] { hipLaunchKernelGGL(k_tally, dim3(kTallyBlocks, n), dim3(256), 0, stream, t, 0); });
    timer.time("k_init_keys", stream, [&] { hipLaunchKernelGGL(k_init_keys, dim3(n), dim3(256), 0, stream, t); });
    timer.time("k_seed", stream, [&] { hipLaunchKernelGGL(k_seed, dim3(n), dim3(256), 0, stream, t); });
    // The first round's member table (later rounds' are built by k_commit).
    const Grid gt_clear = build_grid(tmp, ids, [&](const SearchState& x) { return up(x.d.table_mask + 1, 256); });
    const Grid gt_index = build_grid(tmp, ids, [&](const SearchState& x) { return up(x.P, 128); });
    timer.time("k_clear_init", stream, [&] { hipLaunchKernelGGL(k_clear, dim3(gt_clear.blocks), dim3(256), 0, stream, t, gt_clear.map); });
    timer.time("k_index_init", stream, [&] { hipLaunchKernelGGL(k_index, dim3(gt_index.blocks), dim3(128), 0, stream, t, gt_index.map); });
    HIP_OK(hipStreamSynchronize(stream));
    timer.collect();
    for (int id : ids) {
      SearchState& x = *searches[std::size_t(id)];
      if (const int e = x.device_error()) throw std::runtime_error("device initialization error " + std::to_string(e));
      if (x.has_import) {
        x.imported.rows.clear();
        x.imported.rows.shrink_to_fit();
        continue;  // the first imported program's names are the layout's
      }
      const int n0 = x.down(x.d.cur_n, 1)[0];
      x.layout_names = names_used(x.grammar, x.down(x.d.cur_origin, std::size_t(n0)));
    }
  }
  // Round table, grids, kernel sizes and graph for the current live set.
  // Batch shape for the tuning cache: per kernel, log2 buckets of the
  // searches' programs per round and cases, summed over the live searches.
  std::string shape_key() const {
    const auto bucket = [](double x) { return x <= 1 ? 0 : int(std::floor(std::log2(x))); };
    double fast_programs = 0, fast_cases = 0, loop_items = 0, loop_cases = 0;
    int loops = 0;
    for (int id : live) {
      const SearchState& x = *searches[std::size_t(id)];
      fast_programs += x.B;
      fast_cases += double(x.B) * x.d.cd.C;
      if (x.may_jump) {
        loop_items += double(x.B) * ((x.d.cd.C + 63) / 64);
        loop_cases += double(x.B) * x.d.cd.C;
        ++loops;
      }
    }
    std::ostringstream k;
    k << "typed:" << bucket(fast_programs) << "/" << bucket(fast_cases / std::max(1.0, fast_programs)) << " loop:" << loops << "/"
      << bucket(loop_items) << "/" << bucket(loop_cases / std::max(1.0, loop_items * 64) * 64);
    return k.str();
  }
  // Evaluation work of one round (program-cases over the live searches):
  // below kTuneWork, or with fewer than kTuneRounds rounds left to run,
  // the tuning pass would cost more than it can gain, and the fixed shapes
  // run.
  static constexpr double kTuneWork = double(1 << 22);
  static constexpr int kTuneRounds = 128;
  int rounds_left() const {
    int left = 0;
    for (int id : live) left = std::max(left, searches[std::size_t(id)]->rounds - searches[std::size_t(id)]->stepped);
    return left;
  }
  double round_work() const {
    double w = 0;
    for (int id : live) w += double(searches[std::size_t(id)]->B) * searches[std::size_t(id)]->d.cd.C;
    return w;
  }
  // Measures the evaluation kernels over the current round's pending
  // programs under each candidate launch shape and keeps the fastest.
  // Re-running an evaluation kernel over the same pending list rewrites the
  // same results (each program's fitness, wrong count and tallies; k_loop_finish
  // takes the looping kernel's totals after every launch), so tuning changes no
  // search. Call between enqueue_front and
  // enqueue_eval of a round, with the stream idle.
  void tune_launches() {
    const std::string key = shape_key();
    if (autotune == 1 && (round_work() < kTuneWork || rounds_left() < kTuneRounds)) {
      apply_tuning(TuneChoice{});
      std::ostringstream r;
      r << "{\"key\":\"" << key << "\",\"cached\":false,\"skipped\":\"fewer than " << kTuneWork
        << " program-cases per round or " << kTuneRounds << " rounds left\",\"fast_programs\":1,\"loop_group\":1}";
      tune_report = r.str();
      return;
    }
    {
      std::lock_guard<std::mutex> lock(tune_mutex);
      auto it = tune_cache.find(key);
      if (it != tune_cache.end()) {
        apply_tuning(it->second);
        std::ostringstream r;
        r << "{\"key\":\"" << key << "\",\"cached\":true,\"fast_programs\":" << tune.fast_programs
          << ",\"loop_group\":" << tune.loop_group << "}";
        tune_report = r.str();
        return;
      }
    }
    hipEvent_t a, b;
    HIP_OK(hipEventCreate(&a));
    HIP_OK(hipEventCreate(&b));
    // The first candidate of each kernel runs twice (its first launch warms
    // code and caches), every other candidate once.
    int reps = 2;
    // `after`, not timed, follows every launch.
    const auto measure = [&](auto launch, auto after) {
      float best = 1e30f;
      for (int rep = 0; rep < reps; ++rep) {
        HIP_OK(hipEventRecord(a, stream));
        launch();
        HIP_OK(hipEventRecord(b, stream));
        after();
        HIP_OK(hipEventSynchronize(b));
        float ms = 0;
        HIP_OK(hipEventElapsedTime(&ms, a, b));
        best = std::min(best, ms);
      }
      return best;
    };
    std::ostringstream r;
    r << "{\"key\":\"" << key << "\",\"cached\":false";
    TuneChoice choice;
    DeviceArena tmp;
    // A candidate replaces the default only when at least 3% faster; the
    // candidates grow the work per wavefront, so once one is 15% slower
    // than the best the larger ones are not tried.
    const auto pick = [&](const char* name, const std::vector<int>& values, auto time_of) {
      r << ",\"" << name << "_ms\":{";
      int chosen = values[0];
      float chosen_ms = 0;
      for (std::size_t i = 0; i < values.size(); ++i) {
        reps = i == 0 ? 2 : 1;
        const float ms = time_of(values[i]);
        r << (i ? "," : "") << "\"" << values[i] << "\":" << ms;
        if (i == 0) chosen_ms = ms;
        else if (ms < 0.97f * chosen_ms) { chosen = values[i]; chosen_ms = ms; }
        else if (ms > 1.15f * chosen_ms) break;
      }
      r << "}";
      return chosen;
    };
    choice.fast_programs = pick("typed", {1, 2, 4}, [&](int k) {
      tmp.release();
      const Grid g = typed_grid(tmp, k);
      return g.blocks ? measure([&] {
        hipLaunchKernelGGL(k_eval<1>, dim3(g.blocks), dim3(kEvalThreads), eval_fast_lds, stream, d_all, g.map, 1);
      }, [] {}) : 0.f;
    });
    if (loop_kernel) {
      choice.loop_group = pick("loop", {1, 2, 4}, [&](int group) {
        tmp.release();
        const Grid g = loop_grid(tmp, group);
        return g.blocks ? measure([&] {
          if (group == 1)
            hipLaunchKernelGGL(k_eval_loop<false>, dim3(g.blocks), dim3(64), eval_loop_lds, stream, d_all, g.map, 1, 1);
          else
            hipLaunchKernelGGL(k_eval_loop<true>, dim3(g.blocks), dim3(64), eval_loop_lds, stream, d_all, g.map, 1, group);
        }, [&] {
          if (g_finish.blocks) hipLaunchKernelGGL(k_loop_finish, dim3(g_finish.blocks), dim3(kEvalThreads), 0, stream, d_all, g_finish.map, 1, group);
        }) : 0.f;
      });
    }
    HIP_OK(hipGetLastError());
    HIP_OK(hipStreamSynchronize(stream));
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    r << ",\"fast_programs\":" << choice.fast_programs << ",\"loop_group\":" << choice.loop_group << "}";
    tune_report = r.str();
    {
      std::lock_guard<std::mutex> lock(tune_mutex);
      tune_cache[key] = choice;
    }
    apply_tuning(choice);
  }
  // New launch shapes: grids rebuilt, the round graph captured again.
  void apply_tuning(const TuneChoice& c) {
    tune = c;
    tuned = true;
    if (graph_exec) { (void)hipGraphExecDestroy(graph_exec); graph_exec = nullptr; }
    graph_ready = false;
    build_round_grids();
  }

  static constexpr int kCaptureAfter = 8;
  int table_rounds = 0;  // rounds stepped since the round table was formed
  void rebuild() {
    if (graph_exec) { (void)hipGraphExecDestroy(graph_exec); graph_exec = nullptr; }
    graph_ready = false;
    tuned = false;
    table_rounds = 0;
    if (d_all) { (void)hipFree(d_all); d_all = nullptr; }
    max_rounds = 0;
    if (!live.empty()) {
      std::vector<DSearch> host;
      for (int id : live) {
        host.push_back(searches[std::size_t(id)]->d);
        max_rounds = std::max(max_rounds, searches[std::size_t(id)]->rounds);
      }
      HIP_OK(hipMalloc(&d_all, sizeof(DSearch) * host.size()));
      HIP_OK(hipMemcpy(d_all, host.data(), sizeof(DSearch) * host.size(), hipMemcpyHostToDevice));
      size_kernels(live);
      build_round_grids();
      loop_kernel = any_jumps(live);
      if (status_cap < live.size()) {
        if (d_status) (void)hipFree(d_status);
        status_cap = std::max<std::size_t>(64, 2 * live.size());
        HIP_OK(hipMalloc(&d_status, sizeof(int) * 3 * status_cap));
      }
    }
    dirty = false;
  }

  template <class Kernel, class... Args>
  void launch_on(hipStream_t s, const char* name, const Grid& g, Kernel kernel, int threads, std::size_t lds, Args... args) {
    if (g.blocks)
      timer.time(name, s, [&] { hipLaunchKernelGGL(kernel, dim3(g.blocks), dim3(threads), lds, s, d_all, g.map, args...); });
  }
  template <class Kernel, class... Args>
  void launch(const char* name, const Grid& g, Kernel kernel, int threads, std::size_t lds, Args... args) {
    launch_on(stream, name, g, kernel, threads, lds, args...);
  }
  void enqueue_round() {
    enqueue_front();
    enqueue_eval();
    enqueue_back();
  }
  // A round in three parts: reproduction up to the pending lists, the
  // evaluation kernels, then tallies, placement and commit.
  void enqueue_front() {
    const int n = int(live.size());
    // Caller-driven rounds (the owner seam) bring their own elites, seed and
    // history.
    if (any_generational && !seam)
      timer.time("k_gen_begin", stream, [&] { hipLaunchKernelGGL(k_gen_begin, dim3(n), dim3(256), 0, stream, d_all); });
    if (!seam) timer.time("k_record", stream, [&] { hipLaunchKernelGGL(k_record, dim3(n), dim3(256), 0, stream, d_all); });
    // Two independent branches: the searches whose programs may jump, with
    // the lowering that leaves, and the others (disjoint searches).
    branches({[&](hipStream_t s) {
                launch_on(s, "k_vary_deferred", g_vary_staged_d, k_vary<true, true>, 64 * kVaryWaves, vary_lds_bytes);
                launch_on(s, "k_vary_global_deferred", g_vary_global_d, k_vary<false, true>, 64 * kVaryWaves, 0);
                launch_on(s, "k_lower_walks", g_lower_w, k_lower<true>, 64 * kVaryWaves, vary_lds_bytes);
                launch_on(s, "k_lower", g_lower_c, k_lower<false>, 64 * kVaryWaves, vary_lds_bytes);
              },
              [&](hipStream_t s) {
                launch_on(s, "k_vary", g_vary_staged, k_vary<true, false>, 64 * kVaryWaves, vary_lds_bytes);
                launch_on(s, "k_vary_global", g_vary_global, k_vary<false, false>, 64 * kVaryWaves, 0);
              }});
  }
  void enqueue_eval() {
    // The three evaluation kernels score disjoint pending programs.
    branches({[&](hipStream_t s) {
                if (loop_kernel && tune.loop_group == 1)
                  launch_on(s, "k_eval_loop", g_eval_loop, k_eval_loop<false>, 64, eval_loop_lds, 1, 1);
                else if (loop_kernel)
                  launch_on(s, "k_eval_loop", g_eval_loop, k_eval_loop<true>, 64, eval_loop_lds, 1, tune.loop_group);
                if (loop_kernel) launch_on(s, "k_loop_finish", g_finish, k_loop_finish, kEvalThreads, 0, 1, tune.loop_group);
              },
              [&](hipStream_t s) {
                launch_on(s, "k_eval", g_eval, k_eval<1>, kEvalThreads, eval_fast_lds, 1);
                launch_on(s, "k_eval_tiles", g_eval_tiles, k_eval_tiles, kEvalThreads, eval_tiles_lds, 1);
              },
              [&](hipStream_t s) { launch_on(s, "k_eval_general", g_eval_general, k_eval<0>, kEvalThreads, eval_general_lds, 1); }});
  }
  void enqueue_back() {
    const int n = int(live.size());
    timer.time("k_tally", stream, [&] { hipLaunchKernelGGL(k_tally, dim3(kTallyBlocks, n), dim3(256), 0, stream, d_all, 1); });
    // Placement and the clearing of the member table k_commit refills are
    // independent.
    branches({[&](hipStream_t s) {
                if (place_lds_bytes)
                  timer.time("k_place", s, [&] {
                    hipLaunchKernelGGL(k_place<true>, dim3(n), dim3(kPlaceThreads), place_lds_bytes, s, d_all);
                  });
                if (place_hbm_bytes)
                  timer.time("k_place_hbm", s, [&] {
                    hipLaunchKernelGGL(k_place<false>, dim3(n), dim3(kPlaceThreads), place_hbm_bytes, s, d_all);
                  });
              },
              [&](hipStream_t s) { launch_on(s, "k_clear", g_table, k_clear, 256, 0); }});
    if (any_generational) launch("k_gen_place", g_member, k_gen_place, 128, 0);
    launch("k_commit", g_member_w, k_commit, 64 * kVaryWaves, 0);
    if (any_generational) timer.time("k_gen_end", stream, [&] { hipLaunchKernelGGL(k_gen_end, dim3(n), dim3(64), 0, stream, d_all); });
  }
};

Batch::Batch() : impl_(std::make_unique<Impl>()) {}
Batch::~Batch() = default;
std::size_t Batch::size() const { return impl_->searches.size(); }
void Batch::set_profile(bool on) { impl_->timer.on = on; }
void Batch::set_autotune(int mode) {
  if (mode < 0 || mode > 2) throw std::invalid_argument("autotune mode must be 0, 1 or 2");
  impl_->autotune = mode;
  if (!mode && impl_->tuned) impl_->apply_tuning(TuneChoice{});
  impl_->tuned = false;
}
std::string Batch::tuning_report() const { return impl_->tune_report.empty() ? "{}" : impl_->tune_report; }
int Batch::max_rounds() const { return impl_->max_rounds; }
std::size_t Batch::device_bytes() const {
  std::size_t b = 0;
  for (const auto& s : impl_->searches) b += s->arena.reserved;
  return b;
}
std::vector<std::pair<std::string, double>> Batch::kernel_times() const {
  return {impl_->timer.ms.begin(), impl_->timer.ms.end()};
}

int Batch::add(const SearchSpec& spec) {
  auto s = std::make_unique<SearchState>(spec);
  impl_->searches.push_back(std::move(s));
  return int(impl_->searches.size() - 1);
}

void Batch::prepare() {
  auto& I = *impl_;
  const auto t0 = std::chrono::steady_clock::now();
  I.make_streams();
  std::vector<int> fresh;
  for (std::size_t i = 0; i < I.searches.size(); ++i) {
    if (I.searches[i]->configured) continue;
    I.configure(*I.searches[i]);
    fresh.push_back(int(i));
  }
  I.init_searches(fresh);
  I.live.insert(I.live.end(), fresh.begin(), fresh.end());
  I.rebuild();
  I.init_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

std::size_t Batch::planned_footprint(int index) const { return impl_->searches.at(std::size_t(index))->planned_bytes(); }

void Batch::admit(int index) {
  auto& I = *impl_;
  SearchState& s = *I.searches.at(std::size_t(index));
  if (s.configured || s.retired) throw std::invalid_argument("search already admitted");
  I.make_streams();
  try {
    I.configure(s);
    I.init_searches({index});
  } catch (...) {
    // Undo the partial admission: nothing of the search stays on the
    // device, and the round table never saw it.
    (void)hipStreamSynchronize(I.stream);
    s.arena.release();
    s.d.active = 0;
    s.retired = true;
    throw;
  }
  I.live.push_back(index);
  I.dirty = true;
}

std::vector<std::pair<int, std::string>> Batch::admit_many(const std::vector<int>& indices) {
  auto& I = *impl_;
  std::vector<std::pair<int, std::string>> failed;
  std::vector<int> ready;
  I.make_streams();
  const auto undo = [&](SearchState& s) {
    s.arena.release();
    s.d.active = 0;
    s.retired = true;
  };
  for (int index : indices) {
    SearchState& s = *I.searches.at(std::size_t(index));
    if (s.configured || s.retired) throw std::invalid_argument("search already admitted");
    try {
      I.configure(s);  // allocation: a failure here is this search's alone
      ready.push_back(index);
    } catch (const std::exception& e) {
      (void)hipStreamSynchronize(I.stream);
      undo(s);
      failed.push_back({index, e.what()});
    }
  }
  try {
    I.init_searches(ready);  // one launch sequence for all of them
  } catch (const std::exception& e) {
    (void)hipStreamSynchronize(I.stream);
    for (int index : ready) {
      undo(*I.searches[std::size_t(index)]);
      failed.push_back({index, e.what()});
    }
    ready.clear();
  }
  for (int index : ready) I.live.push_back(index);
  if (!ready.empty()) I.dirty = true;
  return failed;
}

void Batch::drop(int index) {
  SearchState& s = *impl_->searches.at(std::size_t(index));
  if (s.configured && !s.retired) throw std::invalid_argument("search is admitted: retire it");
  s.arena.release();
  s.retired = true;
}

void Batch::retire(int index) {
  auto& I = *impl_;
  const auto it = std::find(I.live.begin(), I.live.end(), index);
  if (it == I.live.end()) throw std::invalid_argument("search is not in the batch");
  I.live.erase(it);
  I.dirty = true;
  SearchState& s = *I.searches.at(std::size_t(index));
  s.arena.release();  // the stream is idle between steps: the memory is free to return
  s.d.active = 0;
  s.retired = true;
}

std::vector<Batch::Status> Batch::status() {
  auto& I = *impl_;
  if (I.dirty) I.rebuild();
  std::vector<Status> out;
  if (I.live.empty()) return out;
  const int n = int(I.live.size());
  hipLaunchKernelGGL(k_status, dim3((n + 63) / 64), dim3(64), 0, I.stream, I.d_all, n, I.d_status);
  HIP_OK(hipGetLastError());
  std::vector<int> v(std::size_t(3 * n));
  HIP_OK(hipMemcpyAsync(v.data(), I.d_status, sizeof(int) * v.size(), hipMemcpyDeviceToHost, I.stream));
  HIP_OK(hipStreamSynchronize(I.stream));
  for (int i = 0; i < n; ++i) {
    const SearchState& x = *I.searches[std::size_t(I.live[std::size_t(i)])];
    Status st{I.live[std::size_t(i)], v[std::size_t(3 * i)], v[std::size_t(3 * i + 1)], v[std::size_t(3 * i + 2)], false};
    st.done = st.error != 0 || st.stopped_at != 0 || st.round >= x.rounds;
    out.push_back(st);
  }
  return out;
}

std::size_t Batch::footprint(int index) const { return impl_->searches.at(std::size_t(index))->arena.reserved; }

void Batch::step(int rounds, bool use_graph) {
  auto& I = *impl_;
  if (I.dirty) I.rebuild();
  if (I.live.empty() || rounds <= 0) return;
  // Every live search has been stepped `rounds` more when this returns (the
  // tuning rule below reads the count from before this step).
  struct Stepped {
    Impl& impl;
    int n;
    ~Stepped() {
      for (int id : impl.live) impl.searches[std::size_t(id)]->stepped += n;
    }
  } stepped{I, rounds};
  const auto t0 = std::chrono::steady_clock::now();
  if (I.autotune && !I.tuned) {
    // The first round of a new table: its pending programs are measured
    // under every candidate shape between reproduction and placement.
    I.enqueue_front();
    HIP_OK(hipStreamSynchronize(I.stream));
    I.tune_launches();
    I.enqueue_eval();
    I.enqueue_back();
    HIP_OK(hipStreamSynchronize(I.stream));
    I.timer.collect();
    if (--rounds == 0) {
      I.run_ms += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
      return;
    }
  }
  // A new round table runs on stream launches until it has stepped
  // kCaptureAfter rounds: capturing and instantiating a graph costs more
  // than the launches of a table that changes every few rounds (serving).
  const bool replay = I.graph_ready || I.table_rounds + rounds >= Impl::kCaptureAfter;
  I.table_rounds += rounds;
  if (use_graph && !I.timer.on && replay) {
    if (!I.graph_ready) {
      hipGraph_t graph;
      HIP_OK(hipStreamBeginCapture(I.stream, hipStreamCaptureModeThreadLocal));
      I.enqueue_round();
      HIP_OK(hipStreamEndCapture(I.stream, &graph));
      HIP_OK(hipGraphInstantiate(&I.graph_exec, graph, nullptr, nullptr, 0));
      (void)hipGraphDestroy(graph);
      I.graph_ready = true;
    }
    for (int r = 0; r < rounds; ++r) HIP_OK(hipGraphLaunch(I.graph_exec, I.stream));
    HIP_OK(hipStreamSynchronize(I.stream));
  } else {
    for (int r = 0; r < rounds; ++r) {
      I.enqueue_round();
      if (I.timer.on && (r % 8 == 7)) I.timer.collect();
    }
    HIP_OK(hipStreamSynchronize(I.stream));
    I.timer.collect();
  }
  I.run_ms += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

void Batch::finish() {
  for (int id : impl_->live) {
    if (const int e = impl_->searches[std::size_t(id)]->device_error()) throw std::runtime_error("device search error " + std::to_string(e));
  }
}

void Batch::run(bool use_graph) {
  prepare();
  step(impl_->max_rounds, use_graph);
  finish();
}

std::vector<std::uint64_t> Batch::counters(int index) const {
  const SearchState& s = *impl_->searches.at(std::size_t(index));
  const Counters c = s.down(s.d.counters, 1)[0];
  return {c.programs,     c.program_cases, c.errors,       c.timeouts,      c.vm_instructions,  c.code_words,
          c.pool_words,   c.children,      c.child_nodes,  c.child_consts,  c.parent_nodes,     c.parent_consts,
          c.child_code_words, c.child_pool_words};
}
double Batch::init_ms() const { return impl_->init_ms; }

// ---- the owner seam (caller-driven steady-state rounds) ----
struct Owner::Impl {
  Batch batch;
  SearchState* s = nullptr;
  double* select = nullptr;  // device selection values, P doubles
  bool made = false;         // a batch is made and not yet committed
  bool scored = false;
  bool reproduced = false;   // the members are the children of reproduce()
  std::vector<int> reuse;
  ~Impl() {
    if (select) (void)hipFree(select);
  }
};

Owner::Owner(const SearchSpec& spec) : impl_(std::make_unique<Impl>()) {
  Impl& O = *impl_;
  O.batch.add(spec);
  O.s = O.batch.impl_->searches[0].get();
  O.batch.set_autotune(0);
  O.batch.impl_->seam = true;
  O.batch.prepare();
  HIP_OK(hipMalloc(&O.select, sizeof(double) * std::size_t(O.s->P)));
  O.s->d.select = (GAS const double*)O.select;
  O.batch.impl_->rebuild();  // the round table with the selection array
  if (const int e = O.s->device_error()) throw std::runtime_error("device initialization error " + std::to_string(e));
}
Owner::~Owner() = default;
int Owner::population_size() const { return impl_->s->P; }
int Owner::batch_size() const { return impl_->s->B; }
bool Owner::has_wrong() const { return impl_->s->d.has_wrong != 0; }

namespace {
// {program cases, errors, timeouts, fallbacks, unscored} of evaluated slots.
void slot_counts(const SearchState& s, int n, const std::vector<int>* reuse, std::uint64_t* counts) {
  const std::vector<unsigned> errors = s.down(s.d.e_errors, std::size_t(n)), timeouts = s.down(s.d.e_timeouts, std::size_t(n));
  for (int i = 0; i < n; ++i) {
    std::uint64_t* c = counts + 5 * std::size_t(i);
    const bool scored = !reuse || (*reuse)[std::size_t(i)] < 0;
    c[0] = scored ? std::uint64_t(s.d.cd.C) : 0;
    c[1] = scored ? errors[std::size_t(i)] : 0;
    c[2] = scored ? timeouts[std::size_t(i)] : 0;
    c[3] = 0;
    c[4] = 0;
  }
}
// Node or grammar-site counts of n rows (counts, site rows of stride R).
void row_counts(const SearchState& s, bool grammar_sites, GAS const int* n_rows, GAS const int* sites, int n, unsigned* out) {
  const std::vector<int> len = s.down(n_rows, std::size_t(n));
  if (!grammar_sites) {
    for (int i = 0; i < n; ++i) out[i] = unsigned(s.d.fixed_nodes) + unsigned(len[std::size_t(i)]);
    return;
  }
  const std::vector<int> site = s.down(sites, std::size_t(n) * std::size_t(s.R));
  for (int i = 0; i < n; ++i) {
    unsigned k = 0;
    for (int j = 0; j < len[std::size_t(i)]; ++j) k += site[std::size_t(i) * std::size_t(s.R) + std::size_t(j)] >= 0;
    out[i] = k;
  }
}
}  // namespace

void Owner::evaluate(double* fitness, unsigned* wrong, std::uint64_t* counts) {
  const SearchState& s = *impl_->s;
  const std::vector<double> f = s.down(s.d.fitness, std::size_t(s.P));
  const std::vector<unsigned> w = s.down(s.d.wrong, std::size_t(s.P));
  std::copy(f.begin(), f.end(), fitness);
  std::copy(w.begin(), w.end(), wrong);
  // After reproduce(), member m is child m: reused children were not scored.
  slot_counts(s, s.P, impl_->reproduced ? &impl_->reuse : nullptr, counts);
}

void Owner::reproduce(const double* selection, int pressure, double p_mut, std::uint64_t seed, int elites) {
  Impl& O = *impl_;
  auto& I = *O.batch.impl_;
  SearchState& s = *O.s;
  if (!s.d.generational) throw std::invalid_argument("reproduce() is the generational schedule's; steady-state searches make batches");
  if (pressure < 1 || pressure > s.P) throw std::invalid_argument("tournament pressure outside 1..P");
  if (!(p_mut >= 0 && p_mut <= 1)) throw std::invalid_argument("mutation probability outside [0, 1]");
  if (elites < 0 || elites >= s.P) throw std::invalid_argument("elite count outside 0..P-1");
  for (int m = 0; m < s.P; ++m)
    if (std::isnan(selection[m])) throw std::invalid_argument("selection values must not be NaN");
  if (pressure != s.d.pressure || p_mut != s.d.p_mut || elites != s.d.elites) {
    s.d.pressure = pressure;
    s.d.p_mut = p_mut;
    s.d.elites = elites;
    I.rebuild();
  }
  // Elites: highest selection value, ties to the lowest index.
  std::vector<int> order(std::size_t(s.P));
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return selection[a] > selection[b]; });
  HIP_OK(hipMemcpyAsync((void*)s.d.elite, order.data(), sizeof(int) * std::size_t(elites), hipMemcpyHostToDevice, I.stream));
  HIP_OK(hipMemcpyAsync(O.select, selection, sizeof(double) * std::size_t(s.P), hipMemcpyHostToDevice, I.stream));
  HIP_OK(hipMemcpyAsync((void*)s.d.round_seed, &seed, sizeof(seed), hipMemcpyHostToDevice, I.stream));
  I.enqueue_front();
  I.enqueue_eval();
  I.launch("k_gen_place", I.g_member, k_gen_place, 128, 0);
  I.launch("k_clear", I.g_table, k_clear, 256, 0);
  I.launch("k_commit", I.g_member_w, k_commit, 64 * kVaryWaves, 0);
  const int zero[3] = {0, 0, 0};
  HIP_OK(hipMemcpyAsync((void*)s.d.n_pending, zero, sizeof(zero), hipMemcpyHostToDevice, I.stream));
  HIP_OK(hipStreamSynchronize(I.stream));
  if (const int e = s.device_error()) throw std::runtime_error("device reproduction error " + std::to_string(e));
  O.reuse = s.down(s.d.reuse, std::size_t(s.P));
  O.reproduced = true;
}

void Owner::node_counts(bool grammar_sites, unsigned* out) {
  const SearchState& s = *impl_->s;
  row_counts(s, grammar_sites, s.d.cur_n, s.d.cur_site, s.P, out);
}

void Owner::begin_steady(int batch) {
  if (batch != impl_->s->B)
    throw std::invalid_argument("steady batch " + std::to_string(batch) + " differs from the search configuration's " +
                                std::to_string(impl_->s->B));
}

void Owner::make_batch(const double* selection, int pressure, double p_mut, std::uint64_t seed, int* reuse) {
  Impl& O = *impl_;
  auto& I = *O.batch.impl_;
  SearchState& s = *O.s;
  if (s.d.generational) throw std::invalid_argument("make_batch() is the steady-state schedule's; generational searches reproduce");
  if (O.made) throw std::invalid_argument("the previous batch is not committed");
  if (pressure < 1 || pressure > s.P) throw std::invalid_argument("tournament pressure outside 1..P");
  if (!(p_mut >= 0 && p_mut <= 1)) throw std::invalid_argument("mutation probability outside [0, 1]");
  if (pressure != s.d.pressure || p_mut != s.d.p_mut) {
    s.d.pressure = pressure;
    s.d.p_mut = p_mut;
    I.rebuild();
  }
  HIP_OK(hipMemcpyAsync(O.select, selection, sizeof(double) * std::size_t(s.P), hipMemcpyHostToDevice, I.stream));
  HIP_OK(hipMemcpyAsync((void*)s.d.round_seed, &seed, sizeof(seed), hipMemcpyHostToDevice, I.stream));
  I.enqueue_front();
  HIP_OK(hipStreamSynchronize(I.stream));
  if (const int e = s.device_error()) throw std::runtime_error("device reproduction error " + std::to_string(e));
  O.reuse = s.down(s.d.reuse, std::size_t(s.B));
  std::copy(O.reuse.begin(), O.reuse.end(), reuse);
  O.made = true;
  O.scored = false;
}

void Owner::evaluate_batch(double* fitness, unsigned* wrong, std::uint64_t* counts) {
  Impl& O = *impl_;
  auto& I = *O.batch.impl_;
  const SearchState& s = *O.s;
  if (!O.made || O.scored) throw std::invalid_argument("no batch to evaluate");
  I.enqueue_eval();
  HIP_OK(hipStreamSynchronize(I.stream));
  if (const int e = s.device_error()) throw std::runtime_error("device evaluation error " + std::to_string(e));
  const std::vector<double> f = s.down(s.d.c_fit, std::size_t(s.B));
  const std::vector<unsigned> w = s.down(s.d.c_wrong, std::size_t(s.B));
  std::copy(f.begin(), f.end(), fitness);
  std::copy(w.begin(), w.end(), wrong);
  slot_counts(s, s.B, &O.reuse, counts);
  O.scored = true;
}

void Owner::batch_nodes(bool grammar_sites, unsigned* out) {
  const SearchState& s = *impl_->s;
  if (!impl_->made) throw std::invalid_argument("no batch made");
  row_counts(s, grammar_sites, s.d.x_n, s.d.x_site, s.B, out);
}

void Owner::commit_batch(const int* pairs, int n) {
  Impl& O = *impl_;
  auto& I = *O.batch.impl_;
  const SearchState& s = *O.s;
  if (!O.made || !O.scored) throw std::invalid_argument("commit before the batch is made and evaluated");
  std::vector<int> placed(std::size_t(s.P), -1);
  for (int k = 0; k < n; ++k) {
    const int m = pairs[2 * k], c = pairs[2 * k + 1];
    if (m < 0 || m >= s.P || c < 0 || c >= s.B) throw std::invalid_argument("placement outside the population or batch");
    placed[std::size_t(m)] = c;
  }
  const int zero[3] = {0, 0, 0};
  HIP_OK(hipMemcpyAsync((void*)s.d.placed, placed.data(), sizeof(int) * placed.size(), hipMemcpyHostToDevice, I.stream));
  I.launch("k_clear", I.g_table, k_clear, 256, 0);
  I.launch("k_commit", I.g_member_w, k_commit, 64 * kVaryWaves, 0);
  HIP_OK(hipMemcpyAsync((void*)s.d.n_pending, zero, sizeof(zero), hipMemcpyHostToDevice, I.stream));
  HIP_OK(hipStreamSynchronize(I.stream));
  if (const int e = s.device_error()) throw std::runtime_error("device commit error " + std::to_string(e));
  O.made = O.scored = false;
}

namespace {
Ast export_row(const SearchState& s, const int* origin, const Val* cval, int n, int nc);
}

json::Value Owner::export_member(int member) {
  const SearchState& s = *impl_->s;
  if (member < 0 || member >= s.P) throw std::invalid_argument("member outside the population");
  const std::size_t o = std::size_t(member) * std::size_t(s.R);
  const int n = s.down(s.d.cur_n + member, 1)[0], nc = s.down(s.d.cur_nc + member, 1)[0];
  const std::vector<int> origin = s.down(s.d.cur_origin + o, std::size_t(n));
  const std::vector<Val> cval = s.down(s.d.cur_cval + o, std::size_t(nc));
  return ast_json(export_row(s, origin.data(), cval.data(), n, nc));
}

namespace {
Ast export_row(const SearchState& s, const int* origin, const Val* cval, int n, int nc) {
  return export_whole_program(s.grammar, s.phase, s.layout_names, std::vector<int>(origin, origin + n),
                              std::vector<Val>(cval, cval + nc), s.binder_base);
}

// The run's success criterion on `test`, the held-out cases of a run or the
// split `gagp eval` names, with `fuel` per case (cpp/src/cli/run.cpp:179-239).
json::Value judge(const SearchState& s, const Cases& test, int fuel, const std::vector<int>& origin, const std::vector<Val>& cval) {
  // Lower the best phase exactly as the engine does, then score on the device.
  std::vector<Ins> code(std::size_t(s.d.code_cap));
  std::vector<Val> pool(std::size_t(s.d.pool_cap));
  std::vector<int> sites(origin.size(), -1);
  PhaseView gv{s.phase.exprs.data(), int(s.phase.exprs.size()), s.phase.prods.data(), int(s.phase.prods.size()),
               s.phase.nts.data(), int(s.phase.nts.size()), s.phase.domains.data(), int(s.phase.domains.size()),
               s.phase.values.data(), int(s.phase.values.size()), s.phase.minimum.data(), s.phase.depth_count,
               s.phase.logical_count, s.phase.site_depth ? 1 : 0, s.phase.root};
  const CRow row{origin.data(), sites.data(), cval.data(), int(origin.size()), int(cval.size())};
  std::vector<std::uint8_t> local_types = s.train.input_types;
  if (test.input_names != s.train.input_names) throw std::invalid_argument("test cases must bind the train inputs");
  const LowerResult lr = s.d.walks ? lower_phase<true>(gv, row, local_types.data(), int(local_types.size()), s.d.expected_type,
                                                       code.data(), int(code.size()), pool.data(), int(pool.size()))
                                    : lower_phase<false>(gv, row, local_types.data(), int(local_types.size()), s.d.expected_type,
                                                         code.data(), int(code.size()), pool.data(), int(pool.size()));
  if (lr.status != ST_OK) throw std::runtime_error("lowering of the best program failed");
  ProgramIn p;
  for (int i = 0; i < lr.code; ++i) {
    const Ins& x = code[i];
    const bool a = x.op == OP_PUSH_CONST || x.op == OP_LOAD || x.op == OP_STORE || x.op == OP_JMP || x.op == OP_JMP_IF_FALSE ||
                   x.op == OP_JMP_IF_TRUE || x.op == OP_CALL_BUILTIN;
    p.code.push_back(CodeIn{x.op, a, x.op == OP_CALL_BUILTIN, x.a, x.argc, x.fuel});
  }
  p.consts.assign(pool.begin(), pool.begin() + lr.constants);
  p.n_locals = lr.locals;
  Session session(test, fuel, 512, s.penalty, s.task.policy);
  std::vector<Val> values;
  std::vector<int> errors;
  session.eval_cases(p, values, errors);
  std::size_t correct = 0, errs = 0;
  double loss = 0;
  const bool absolute = s.task.policy.metric == METRIC_ABSOLUTE;
  for (int i = 0; i < test.n; ++i) {
    bool ok = false, error = false;
    double l = absolute ? s.task.case_cap : 1;
    const Val& want = test.expected[i];
    if (errors[i] != ERR_NONE) error = true;
    else if (want.tag == TAG_INT) {
      if (values[i].tag != TAG_INT) error = true;
      else {
        ok = values[i].i == want.i;
        if (absolute) l = std::min(s.task.case_cap, integer_gap(values[i].i, want.i));
      }
    } else if (want.tag == TAG_INT_LIST) {
      error = true;  // list results are outside the engine's values
    } else {
      bool exact = false;
      const Policy exact_policy{METRIC_EXACT, PROX_CAPPED, 0, 0.1, 100};
      (void)case_score(values[i], want, 1, exact_policy, exact);
      ok = exact;
    }
    if (ok) l = 0;
    correct += ok;
    errs += error;
    loss += l;
  }
  const double n = double(test.n);
  json::Value v = json::make_object();
  v.obj["cases"] = json::make_number(n);
  v.obj["correct"] = json::make_number(double(correct));
  v.obj["wrong"] = json::make_number(n - double(correct));
  v.obj["runtime_errors"] = json::make_number(double(errs));
  v.obj["mean_loss"] = json::make_number(loss / n);
  v.obj["solved"] = json::make_bool(correct == std::size_t(test.n));
  return v;
}
}  // namespace

json::Value evaluate_program(const std::string& task_path, const std::string& program_path, const std::string& split) {
  if (split != "train" && split != "test") throw std::invalid_argument("--split must be train or test");
  SearchSpec spec;
  spec.task_path = task_path;
  SearchState s(spec);
  const std::string& cases_path = split == "train" ? s.task.train_path : s.task.test_path;
  if (cases_path.empty()) throw std::invalid_argument("task has no " + split + " split");
  std::ifstream in(program_path, std::ios::binary);
  if (!in) throw std::invalid_argument("cannot read " + program_path);
  std::ostringstream text;
  text << in.rdbuf();
  const json::Value doc = json::parse(text.str());
  // The program must be a member of the task's grammar; its row lowers as
  // the engine lowers a member. Lowering capacities come from the search's
  // shapes, computed without allocating.
  const PhaseRow row = import_row(s.grammar, s.phase, decode_ast(program_of_document(doc)), 0, s.R);
  DeviceArena shapes(true);
  s.d = s.build(shapes);
  json::Value v = judge(s, load_cases(cases_path), int(s.grammar.fuel), row.origin, row.cval);
  v.obj["task"] = json::make_string(s.task.name);
  v.obj["split"] = json::make_string(split);
  return v;
}

void Batch::results(std::vector<SearchResult>& out) {
  int device = 0;
  HIP_OK(hipGetDevice(&device));
  const std::size_t n = size();
  std::vector<SearchResult> made(n);
  std::vector<std::exception_ptr> failed(n);
  parallel_ranges(n, 1, [&](std::size_t begin, std::size_t end) {
    HIP_OK(hipSetDevice(device));  // a new thread's device is the first
    for (std::size_t i = begin; i < end; ++i) {
      try {
        made[i] = result(int(i), false);
      } catch (...) {
        failed[i] = std::current_exception();
        return;
      }
    }
  });
  for (std::size_t i = 0; i < n; ++i) {
    if (failed[i]) std::rethrow_exception(failed[i]);
    out.push_back(std::move(made[i]));
  }
}

SearchResult Batch::result(int index, bool save_all) {
  auto& I = *impl_;
  SearchState& s = *I.searches.at(std::size_t(index));
  const DSearch& d = s.d;
  SearchResult out;
  // A search that stopped early after G generations publishes what a run
  // with G generations publishes.
  const int stopped = s.down(d.stop, 1)[0];
  const int G = stopped ? stopped : s.G;
  SearchConfig published = s.cfg;
  published.generations = G;
  const auto fitness = s.down(d.fitness, std::size_t(s.P));
  const auto wrong = s.down(d.wrong, std::size_t(s.P));
  const auto nodes = s.down(d.nodes, std::size_t(s.P));
  // The front of the strict order over the final keys (for the generational
  // schedule the device's best index predates the last replacement).
  const Keys final_keys{fitness.data(), wrong.data(), nodes.data(), d.has_wrong};
  int best = 0;
  for (int m = 1; m < s.P; ++m)
    if (better(final_keys, m, best)) best = m;
  const auto cur_n = s.down(d.cur_n, std::size_t(s.P));
  const auto cur_nc = s.down(d.cur_nc, std::size_t(s.P));
  const Counters counters = s.down(d.counters, 1)[0];
  out.evaluated_program_cases = counters.program_cases;
  out.evaluated_programs = counters.programs;
  // History rows.
  const auto hn = s.down(d.hist_n, std::size_t(G));
  const auto hnc = s.down(d.hist_nc, std::size_t(G));
  const auto ho = s.down(d.hist_origin, std::size_t(G) * s.R);
  const auto hc = s.down(d.hist_cval, std::size_t(G) * s.R);
  const auto hf = s.down(d.hist_fit, std::size_t(G));
  const auto hw = s.down(d.hist_wrong, std::size_t(G));
  const auto ha = s.down(d.hist_all, std::size_t(G) * s.P);
  const double per_gen_ms = G ? I.run_ms / G : 0;
  json::Value history = json::make_array();
  for (int gen = 0; gen < G; ++gen) {
    const Ast ast = export_row(s, &ho[std::size_t(gen) * s.R], &hc[std::size_t(gen) * s.R], hn[gen], hnc[gen]);
    long double sum = 0;
    for (int m = 0; m < s.P; ++m) sum += ha[std::size_t(gen) * s.P + m];
    json::Value h = json::make_object();
    h.obj["generation"] = json::make_number(gen);
    h.obj["best_fitness"] = json::make_number(hf[gen]);
    h.obj["mean_fitness"] = json::make_number(double(sum / s.P));
    h.obj["best_wrong"] = json::make_number(hw[gen]);
    h.obj["best_nodes"] = json::make_number(double(ast.nodes.size()));
    h.obj["elapsed_ms"] = json::make_number(I.init_ms + per_gen_ms * (gen + 1));
    h.obj["eval_ms"] = json::make_number(per_gen_ms);
    h.obj["repro_ms"] = json::make_number(0);
    history.arr.push_back(h);
    if (save_all) {
      json::Value l = json::make_object();
      l.obj["generation"] = json::make_number(gen);
      l.obj["fitness"] = json::make_number(hf[gen]);
      l.obj["program"] = ast_json(ast);
      out.lineage.push_back(l);
    }
  }
  out.grammar_hash = s.grammar.content_hash;
  // Best member (the strict order's front after the last round).
  const std::vector<int> bo = s.down(d.cur_origin + std::size_t(best) * s.R, std::size_t(cur_n[best]));
  const std::vector<Val> bc = s.down(d.cur_cval + std::size_t(best) * s.R, std::size_t(cur_nc[best]));
  const Ast best_ast = export_whole_program(s.grammar, s.phase, s.layout_names, bo, bc, s.binder_base);
  json::Value bj = json::make_object();
  bj.obj["fitness"] = json::make_number(fitness[best]);
  bj.obj["wrong"] = json::make_number(wrong[best]);
  bj.obj["nodes"] = json::make_number(double(best_ast.nodes.size()));
  bj.obj["text"] = json::make_string(program_text(best_ast));
  bj.obj["program"] = ast_json(best_ast);
  if (save_all) {
    const Keys keys{fitness.data(), wrong.data(), nodes.data(), d.has_wrong};
    std::vector<int> order(std::size_t(s.P));
    std::iota(order.begin(), order.end(), 0);
    std::sort(order.begin(), order.end(), [&](int a, int b) { return better(keys, a, b); });
    const auto all_o = s.down(d.cur_origin, std::size_t(s.P) * s.R);
    const auto all_c = s.down(d.cur_cval, std::size_t(s.P) * s.R);
    for (int m : order)
      out.population.push_back(ast_json(export_row(s, &all_o[std::size_t(m) * s.R], &all_c[std::size_t(m) * s.R], cur_n[m], cur_nc[m])));
  }
  json::Value r = json::make_object();
  r.obj["format"] = json::make_string("gagp-run-v1");
  r.obj["task"] = json::make_string(s.task.name);
  r.obj["engine"] = json::make_string("gpu");
  r.obj["population"] = json::make_number(s.P);
  r.obj["generations"] = json::make_number(G);
  r.obj["seed"] = json::make_string(std::to_string(s.cfg.seed));
  r.obj["train_cases"] = json::make_number(s.train.n);
  r.obj["search"] = effective_search_json(published, s.penalty, s.fuel);
  r.obj["best"] = bj;
  r.obj["history"] = history;
  json::Value tm = json::make_object();
  tm.obj["total"] = json::make_number(I.init_ms + I.run_ms);
  tm.obj["search"] = json::make_number(I.init_ms + I.run_ms);
  tm.obj["initialization"] = json::make_number(I.init_ms);
  r.obj["time_ms"] = tm;
  if (!s.task.test_path.empty()) r.obj["test"] = judge(s, load_cases(s.task.test_path), s.fuel, bo, bc);
  out.result = r;
  out.search_ms = I.init_ms + I.run_ms;
  return out;
}

// ====================== VALU issue-rate probe ======================
// Eight int32 VALU operations per iteration in four independent
// add/xor chains, which no closed form removes; the final test keeps every
// chain live without a store per iteration.
__global__ __launch_bounds__(256) void k_valu_probe(unsigned* out, int iters, unsigned seed) {
  unsigned a = threadIdx.x ^ seed, b = blockIdx.x, c = a + 1u, d = b + 3u, e = a ^ 5u, f = b ^ 7u, g = a + b, h = a - b;
  for (int i = 0; i < iters; ++i) {
    a += b; c += d; e += f; g += h;
    b ^= a; d ^= c; f ^= e; h ^= g;
  }
  if ((a ^ c ^ e ^ g) == 0x9e3779b9u) out[blockIdx.x] = b ^ d ^ f ^ h;
}

float valu_probe_ms(int blocks, int iters) {
  if (blocks <= 0 || iters <= 0) throw std::invalid_argument("probe needs positive blocks and iterations");
  DeviceArena tmp;
  unsigned* out = (unsigned*)tmp.alloc<unsigned>(std::size_t(blocks));
  hipEvent_t a, b;
  HIP_OK(hipEventCreate(&a));
  HIP_OK(hipEventCreate(&b));
  hipLaunchKernelGGL(k_valu_probe, dim3(blocks), dim3(256), 0, nullptr, out, iters, 1u);  // warm
  HIP_OK(hipEventRecord(a, nullptr));
  hipLaunchKernelGGL(k_valu_probe, dim3(blocks), dim3(256), 0, nullptr, out, iters, 2u);
  HIP_OK(hipEventRecord(b, nullptr));
  HIP_OK(hipGetLastError());
  HIP_OK(hipEventSynchronize(b));
  float ms = 0;
  HIP_OK(hipEventElapsedTime(&ms, a, b));
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  return ms;
}

// ====================== evaluation session ======================
namespace {
// Static stack heights of external bytecode (the verifier's stack-shape
// pass, cpp/src/runtime/bytecode_verify.cpp): every instruction gets one
// height; joins must agree; operand/constant/jump domains are checked.
std::vector<Ins> verify_program(const ProgramIn& p, int n_inputs, int& max_stack, bool& jumps, bool* input_stores = nullptr) {
  const int n = int(p.code.size());
  if (n == 0) throw std::invalid_argument("empty program");
  std::vector<int> height(std::size_t(n) + 1, -1);
  std::vector<int> work{0};
  height[0] = 0;
  max_stack = 0;
  jumps = false;
  // A NEG of a constant that is not a number is a guaranteed runtime error
  // (the verifier's abstract types, bytecode_verify.cpp:629-637): nothing
  // falls through it. Only the pushed constant's own path reaches it when no
  // jump targets the NEG.
  std::vector<char> targeted(std::size_t(n) + 1, 0);
  for (int i = 0; i < n; ++i)
    if ((p.code[i].op == OP_JMP || p.code[i].op == OP_JMP_IF_FALSE || p.code[i].op == OP_JMP_IF_TRUE) && p.code[i].has_a && p.code[i].a >= 0 &&
        p.code[i].a <= n)
      targeted[std::size_t(p.code[i].a)] = 1;
  const auto failing_neg = [&](int ip) {
    if (ip == 0 || targeted[std::size_t(ip)] || p.code[ip - 1].op != OP_PUSH_CONST || !p.code[ip - 1].has_a || p.code[ip - 1].a < 0 ||
        p.code[ip - 1].a >= int(p.consts.size()))
      return false;
    const int tag = p.consts[std::size_t(p.code[ip - 1].a)].tag;
    return tag != TAG_INT && tag != TAG_FLOAT;
  };
  const auto flow = [&](int to, int h) {
    if (to < 0 || to > n) throw std::invalid_argument("jump target out of range");
    if (height[to] < 0) { height[to] = h; work.push_back(to); }
    else if (height[to] != h) throw std::invalid_argument("stack heights disagree at a join");
  };
  while (!work.empty()) {
    const int ip = work.back();
    work.pop_back();
    if (ip == n) continue;
    const int h = height[ip];
    const int op = p.code[ip].op;
    int pop = 0, push = 0;
    bool falls = true;
    switch (op) {
      case OP_PUSH_CONST:
        if (!p.code[ip].has_a || p.code[ip].a < 0 || p.code[ip].a >= int(p.consts.size())) throw std::invalid_argument("const index out of range");
        push = 1; break;
      case OP_LOAD:
        if (!p.code[ip].has_a || p.code[ip].a < 0 || p.code[ip].a >= 64) throw std::invalid_argument("local index out of range");
        push = 1; break;
      case OP_STORE:
        if (!p.code[ip].has_a || p.code[ip].a < 0 || p.code[ip].a >= 64) throw std::invalid_argument("local index out of range");
        // A store into an input slot: the evaluators shadow it per execution.
        if (p.code[ip].a < n_inputs && input_stores) *input_stores = true;
        pop = 1; break;
      case OP_NEG: pop = 1; push = 1; falls = !failing_neg(ip); break;
      case OP_NOT: case OP_CHECK_INT: case OP_CHECK_LIST: pop = 1; push = 1; break;
      case OP_ADD: case OP_SUB: case OP_MUL: case OP_DIV: case OP_MOD:
      case OP_LT: case OP_LE: case OP_GT: case OP_GE: case OP_EQ: case OP_NE: pop = 2; push = 1; break;
      case OP_JMP: jumps = true; if (!p.code[ip].has_a) throw std::invalid_argument("jump target missing"); flow(p.code[ip].a, h); falls = false; break;
      case OP_JMP_IF_FALSE: case OP_JMP_IF_TRUE:
        jumps = true;
        if (!p.code[ip].has_a) throw std::invalid_argument("jump target missing");
        if (h < 1) throw std::invalid_argument("stack underflow");
        flow(p.code[ip].a, h - 1);
        pop = 1; break;
      case OP_CALL_BUILTIN:
        if (!p.code[ip].has_b || p.code[ip].b < 0 || p.code[ip].b > 8) throw std::invalid_argument("invalid builtin argc");
        pop = p.code[ip].b; push = 1; break;
      case OP_RETURN: if (h < 1) throw std::invalid_argument("return requires value on stack"); falls = false; break;
      default: throw Unsupported("opcode outside the device VM: " + std::to_string(op));
    }
    if (h < pop) throw std::invalid_argument("stack underflow");
    const int after = h - pop + push;
    max_stack = std::max(max_stack, after);
    if (after > kMaxStack) throw Unsupported("stack deeper than the device VM");
    if (falls) flow(ip + 1, after);
  }
  std::vector<Ins> out(static_cast<std::size_t>(n));
  for (int i = 0; i < n; ++i) {
    const std::uint32_t f = p.code[i].fuel;
    if (f > 255) throw Unsupported("instruction fuel charges above 255");
    const int h = height[i] < 0 ? 0 : height[i];  // unreachable instructions never run
    out[i] = Ins{p.code[i].op, std::uint8_t(p.code[i].b), std::uint8_t(h), std::uint8_t(f), p.code[i].a};
  }
  return out;
}
}  // namespace

// Static tags of straight-line external bytecode: the program is certified
// for vm_fast when every operand tag is known and Int or Bool and every
// instruction is one vm_fast restates with checks that cannot fail (the same
// rules as the lowering's fast_operation). `input_tags[k]` is the one tag
// input k has wherever it is bound (TAG_INVALID when the cases disagree).
struct FastCert { bool fast = false; int result_tag = TAG_INT; };
FastCert certify_fast(const std::vector<Ins>& code, const std::vector<Val>& consts, const std::vector<std::uint8_t>& input_tags,
                      int n_locals, int max_stack, bool jumps, int C) {
  FastCert cert;
  if (jumps || max_stack > kFastStack || code.size() > std::size_t(kFastCode) || consts.size() > std::size_t(kFastPool) ||
      n_locals > kFastInputs || C > kScoreCases)
    return cert;
  std::vector<std::uint8_t> tags;
  for (const Ins& ins : code) {
    const int h = int(tags.size());
    if (ins.sp != h) return cert;
    const std::uint8_t* args = h >= ins.argc ? tags.data() + (h - ins.argc) : nullptr;
    switch (ins.op) {
      case OP_PUSH_CONST: {
        const int t = consts[std::size_t(ins.a)].tag;
        if (!fast_type(t)) return cert;
        tags.push_back(std::uint8_t(t));
        break;
      }
      case OP_LOAD: {
        if (ins.a >= n_locals || ins.a >= int(input_tags.size()) || !fast_type(input_tags[std::size_t(ins.a)])) return cert;
        tags.push_back(input_tags[std::size_t(ins.a)]);
        break;
      }
      case OP_RETURN:
        if (h < 1 || !fast_type(tags.back())) return cert;
        cert.fast = true;
        cert.result_tag = tags.back();
        return cert;
      case OP_CALL_BUILTIN: {
        if (!args || !fast_operation(OP_CALL_BUILTIN, ins.a, ins.argc, args[0], ins.argc > 1 ? args[1] : 0, ins.argc > 2 ? args[2] : 0))
          return cert;
        tags.resize(std::size_t(h - ins.argc));
        tags.push_back(TAG_INT);
        break;
      }
      default: {
        const int arity = ins.op == OP_NEG || ins.op == OP_NOT || ins.op == OP_CHECK_INT ? 1 : 2;
        if (h < arity) return cert;
        const std::uint8_t* a = tags.data() + (h - arity);
        if (!fast_operation(ins.op, 0, arity, a[0], arity > 1 ? a[1] : 0, 0)) return cert;
        const bool compare = ins.op >= OP_LT && ins.op <= OP_NE;
        const std::uint8_t rt = compare ? TAG_BOOL : ins.op == OP_NOT ? TAG_BOOL : TAG_INT;
        tags.resize(std::size_t(h - arity));
        tags.push_back(rt);
        break;
      }
    }
  }
  return cert;  // falls off the end: the general VM reports it
}

// The looping certificate of external bytecode: the program runs on the
// decoded steps when, by the types every path brings, each operand is an Int,
// a Bool or an IntList view that an operation of the looping path takes
// (loop_operation), every hidden local is stored before it is read, all
// returns share one type, every instruction charges one unit and the limits
// of the path hold. A forward data-flow pass over the verified code (whose
// stack heights agree at joins); a local two paths leave with different types
// has none.
struct LoopCert { bool loop = false; int result_tag = TAG_INT; };
LoopCert certify_loop(const std::vector<Ins>& code, const std::vector<Val>& consts, const std::vector<std::uint8_t>& input_tags,
                      int n_locals, int max_stack, bool unit_fuel, int C) {
  LoopCert cert;
  const int n = int(code.size()), K = int(input_tags.size());
  if (!unit_fuel || n > kLoopCode || int(consts.size()) > kLoopPool || max_stack > kLoopStack || K > kFastInputs ||
      n_locals < K || n_locals - K > kLoopLocals || C > kScoreCases)
    return cert;
  struct State { std::uint8_t stack[kLoopStack], local[kFastInputs + kLoopLocals]; };
  std::vector<State> at(std::size_t(n) + 1);
  std::vector<char> seen(std::size_t(n) + 1, 0);
  State first;
  std::fill(std::begin(first.stack), std::end(first.stack), TAG_INVALID);
  std::fill(std::begin(first.local), std::end(first.local), TAG_INVALID);
  for (int k = 0; k < K; ++k) first.local[k] = input_tags[std::size_t(k)];
  std::vector<int> work;
  int returned = TAG_INVALID;
  // Brings `s` (stack height h) to instruction `to`; false when two paths
  // disagree on a stack element's type.
  const auto flow = [&](int to, const State& s, int h) {
    State& d = at[std::size_t(to)];
    if (!seen[std::size_t(to)]) {
      d = s;
      seen[std::size_t(to)] = 1;
      work.push_back(to);
      return true;
    }
    for (int k = 0; k < h; ++k)
      if (d.stack[k] != s.stack[k]) return false;
    bool changed = false;
    for (int k = 0; k < n_locals; ++k)
      if (d.local[k] != s.local[k] && d.local[k] != TAG_INVALID) { d.local[k] = TAG_INVALID; changed = true; }
    if (changed) work.push_back(to);
    return true;
  };
  flow(0, first, 0);
  while (!work.empty()) {
    const int ip = work.back();
    work.pop_back();
    if (ip == n) continue;  // off the end: ValueError on the steps too
    State s = at[std::size_t(ip)];
    const Ins& x = code[std::size_t(ip)];
    const int h = x.sp;
    int after = h;
    bool falls = true;
    switch (x.op) {
      case OP_PUSH_CONST: case OP_LOAD: {
        if (x.op == OP_LOAD && x.a >= n_locals) return cert;
        const std::uint8_t t = x.op == OP_LOAD ? s.local[x.a] : consts[std::size_t(x.a)].tag;
        if (!loop_type(t)) return cert;
        s.stack[h] = t;
        after = h + 1;
        break;
      }
      case OP_STORE:
        if (x.a >= n_locals) return cert;
        s.local[x.a] = s.stack[h - 1];
        after = h - 1;
        break;
      case OP_JMP: if (!flow(x.a, s, h)) return cert; falls = false; break;
      case OP_JMP_IF_FALSE: case OP_JMP_IF_TRUE:
        if (s.stack[h - 1] != TAG_BOOL || !flow(x.a, s, h - 1)) return cert;
        after = h - 1;
        break;
      case OP_RETURN:
        if (!fast_type(s.stack[h - 1]) || (returned != TAG_INVALID && returned != s.stack[h - 1])) return cert;
        returned = s.stack[h - 1];
        falls = false;
        break;
      default: {
        const bool call = x.op == OP_CALL_BUILTIN;
        const int arity = call ? x.argc : x.op == OP_NEG || x.op == OP_NOT || x.op == OP_CHECK_INT ? 1 : 2;
        if (arity < 1 || arity > 3) return cert;
        const std::uint8_t* a = s.stack + (h - arity);
        const bool is_int = call && x.a == B_IS_INT;
        if (is_int ? (arity != 1 || a[0] != TAG_INT)
                   : !loop_operation(x.op, call ? x.a : 0, arity, a[0], arity > 1 ? a[1] : 0, arity > 2 ? a[2] : 0))
          return cert;
        const bool boolean = is_int || x.op == OP_NOT || (x.op >= OP_LT && x.op <= OP_NE);
        s.stack[h - arity] = boolean ? TAG_BOOL : TAG_INT;
        after = h - arity + 1;
        break;
      }
    }
    if (falls && !flow(ip + 1, s, after)) return cert;
  }
  // Unreachable code is unverified: the general VM skips it.
  if (returned == TAG_INVALID || std::count(seen.begin(), seen.end() - 1, 0) != 0) return cert;
  cert.loop = true;
  cert.result_tag = returned;
  return cert;
}

namespace {
// Host packing of one evaluation launch: verified code and pools laid out
// back to back, with each program's offsets and certificate (`fast`: 1 the
// typed straight-line path, 2 the decoded steps, 0 the general VM).
struct PackedPrograms {
  std::vector<Ins> code;
  std::vector<Val> pool;
  std::vector<std::size_t> code_off, pool_off;
  std::vector<int> lens, jumps, locals, fast, pool_n, result;
  std::vector<Step> steps;  // of the looping programs
  std::vector<std::size_t> step_off;
  std::vector<int> step_n, step_index;
  int slots = 1, temps = 0, shadow = 0;
  bool any_fast = false, any_general = false;
};

}  // namespace

struct Session::Impl {
  DeviceArena arena;
  DeviceCases cases;
  std::vector<std::uint8_t> input_tags;
  std::size_t arena_len = 0;
  int fuel, lanes;
  double penalty;
  Policy policy;
  float last_ms = 0;
  // `decode`: certify and decode looping programs for the steps.
  PackedPrograms pack(const std::vector<ProgramIn>& programs, bool decode) const;
  std::vector<DProg> program_table(const PackedPrograms& k, GAS const Ins* code, GAS const Val* pool) const;
  std::vector<StepProg> step_table(const PackedPrograms& k, GAS const Step* steps) const;
  void launch(const PackedPrograms& k, const DProg* progs, const StepProg* step_progs, int n, double* fit, unsigned* wrong,
              unsigned* counts) const;
};

namespace {
// Container values reach the device only as views inside the case arena.
void check_view(const Val& v, std::size_t arena_len) {
  if (v.tag == TAG_INT_LIST) {
    const std::uint64_t u = std::uint64_t(v.i), off = u >> 16, len = u & 0xffff;
    if (off > arena_len || len > arena_len - off) throw std::invalid_argument("IntList view outside the list arena");
  } else if (v.tag == TAG_STRING || v.tag == TAG_FLOAT_LIST || v.tag == TAG_STRING_LIST || v.tag == TAG_CHAR) {
    throw Unsupported("string, char and non-Int list values are outside the device VM");
  } else if (v.tag > TAG_INVALID) {
    throw std::invalid_argument("unknown value tag");
  }
}
}  // namespace

Session::Session(const Cases& c, int fuel, int lanes, double penalty, Policy policy) : impl_(std::make_unique<Impl>()) {
  for (std::size_t i = 0; i < c.inputs.size(); ++i)
    if (c.set.empty() || c.set[i]) check_view(c.inputs[i], c.arena.size());
  for (const auto& v : c.expected) check_view(v, c.arena.size());
  impl_->arena_len = c.arena.size();
  impl_->cases.upload(impl_->arena, c);
  const std::size_t K = c.input_names.size();
  impl_->input_tags.assign(K, TAG_INVALID);
  std::vector<bool> seen(K, false), mixed(K, false);
  for (int i = 0; i < c.n; ++i)
    for (std::size_t k = 0; k < K; ++k) {
      const std::size_t at = std::size_t(i) * K + k;
      if (!c.set.empty() && !c.set[at]) continue;
      const std::uint8_t t = c.inputs[at].tag;
      if (!seen[k]) { seen[k] = true; impl_->input_tags[k] = t; }
      else if (impl_->input_tags[k] != t) mixed[k] = true;
    }
  for (std::size_t k = 0; k < K; ++k)
    if (mixed[k]) impl_->input_tags[k] = TAG_INVALID;
  impl_->fuel = fuel;
  impl_->lanes = lanes;
  impl_->penalty = penalty;
  impl_->policy = policy;
}
Session::~Session() = default;
float Session::last_kernel_ms() const { return impl_->last_ms; }

PackedPrograms Session::Impl::pack(const std::vector<ProgramIn>& programs, bool decode) const {
  const auto& I = *this;
  struct Item {
    std::vector<Ins> code;
    std::vector<Step> steps;
    int max_stack = 0, kind = 0, result = TAG_INVALID;
    bool jumps = false, stores = false;  // stores: into an input
  };
  std::vector<Item> items(programs.size());
  parallel_ranges(items.size(), 512, [&](std::size_t begin, std::size_t end) {
    for (std::size_t i = begin; i < end; ++i) {
      const ProgramIn& p = programs[i];
      Item& x = items[i];
      x.code = verify_program(p, I.cases.cd.n_inputs, x.max_stack, x.jumps, &x.stores);
      for (const auto& v : p.consts) check_view(v, I.arena_len);
      const FastCert cert = certify_fast(x.code, p.consts, I.input_tags, p.n_locals, x.max_stack, x.jumps, I.cases.cd.C);
      x.kind = cert.fast ? 1 : 0;
      x.result = cert.result_tag;
      if (x.kind || !decode) continue;
      const bool unit = std::all_of(x.code.begin(), x.code.end(), [](const Ins& y) { return y.fuel == 1; });
      const LoopCert loop = certify_loop(x.code, p.consts, I.input_tags, p.n_locals, x.max_stack, unit, I.cases.cd.C);
      if (!loop.loop) continue;
      x.kind = 2;
      x.result = loop.result_tag;
      Step steps[kStepMax];
      const int n = decode_steps(x.code.data(), int(x.code.size()), p.consts.data(), I.cases.cd.n_inputs, false, steps);
      x.steps.assign(steps, steps + n);
    }
  });
  PackedPrograms k;
  bool stores = false;  // some program stores into an input
  for (std::size_t i = 0; i < items.size(); ++i) {
    const ProgramIn& p = programs[i];
    const Item& x = items[i];
    k.temps = std::max(k.temps, std::min(64, p.n_locals) - I.cases.cd.n_inputs);
    stores = stores || x.stores;
    if (x.kind == 2) {
      k.step_off.push_back(k.steps.size());
      k.step_n.push_back(int(x.steps.size()));
      k.step_index.push_back(int(i));
      k.steps.insert(k.steps.end(), x.steps.begin(), x.steps.end());
    }
    k.slots = std::max(k.slots, x.max_stack + 1);
    k.fast.push_back(x.kind);
    k.result.push_back(x.result);
    k.pool_n.push_back(int(p.consts.size()));
    k.code_off.push_back(k.code.size());
    k.pool_off.push_back(k.pool.size());
    k.code.insert(k.code.end(), x.code.begin(), x.code.end());
    k.pool.insert(k.pool.end(), p.consts.begin(), p.consts.end());
    k.lens.push_back(int(x.code.size()));
    k.jumps.push_back(x.jumps);
    k.locals.push_back(p.n_locals);
  }
  if (k.pool.empty()) k.pool.push_back(val_invalid());
  k.shadow = stores ? I.cases.cd.n_inputs : 0;
  k.temps += k.shadow;
  k.any_fast = std::count(k.fast.begin(), k.fast.end(), 1) > 0;
  k.any_general = std::count(k.fast.begin(), k.fast.end(), 0) > 0;
  return k;
}

std::vector<DProg> Session::Impl::program_table(const PackedPrograms& k, GAS const Ins* code, GAS const Val* pool) const {
  std::vector<DProg> progs(k.lens.size());
  for (std::size_t i = 0; i < progs.size(); ++i)
    progs[i] = DProg{code + k.code_off[i], pool + k.pool_off[i], k.lens[i], k.jumps[i], k.locals[i], k.fast[i], k.pool_n[i], k.result[i]};
  return progs;
}

std::vector<StepProg> Session::Impl::step_table(const PackedPrograms& k, GAS const Step* steps) const {
  std::vector<StepProg> progs(k.step_n.size());
  for (std::size_t i = 0; i < progs.size(); ++i)
    progs[i] = StepProg{steps + k.step_off[i], k.step_n[i], k.step_index[i], k.result[std::size_t(k.step_index[i])]};
  return progs;
}

// The evaluation kernels over a packed launch on the null stream.
void Session::Impl::launch(const PackedPrograms& k, const DProg* progs, const StepProg* step_progs, int n, double* fit,
                           unsigned* wrong, unsigned* counts) const {
  const auto& I = *this;
  const EvalParams e{I.cases.cd, I.fuel, I.lanes, I.penalty, I.policy};
  const std::size_t lds = std::size_t(kWavesPerBlock) * (k.slots + k.temps) * 64 * 10;
  const std::size_t fast_lds = std::size_t(kWavesPerBlock) * 8 * std::size_t(I.cases.cd.C);
  const int blocks = std::min(4096, (n + kWavesPerBlock - 1) / kWavesPerBlock), loops = int(k.step_n.size());
  const auto step_lds = [&](int waves) {
    return std::size_t(waves) * step_slots(I.cases.cd.n_inputs) * 64 * 8 + 8 * std::size_t(I.cases.cd.C);
  };
  const int step_blocks = std::min(16384, loops), step_waves = std::min(kWavesPerBlock, (I.cases.cd.C + 63) / 64);
  // Both kinds of looping program go in one launch of whole blocks where the
  // general VM's deepest stack leaves LDS for the steps' totals.
  const std::size_t both_lds = std::max(lds, step_lds(kWavesPerBlock));
  const bool both = loops && k.any_general && both_lds + sizeof(StepTotals) <= kLdsLimit;
  if (both) {
    allow_lds(reinterpret_cast<const void*>(&k_eval_both), both_lds);
    hipLaunchKernelGGL(k_eval_both, dim3(blocks + step_blocks), dim3(kEvalThreads), both_lds, nullptr, progs, n, blocks, step_progs, loops, e,
                       k.slots, k.temps, k.shadow, fit, wrong, counts);
  } else if (loops) {
    allow_lds(reinterpret_cast<const void*>(&k_eval_steps), step_lds(step_waves));
    hipLaunchKernelGGL(k_eval_steps, dim3(step_blocks), dim3(64 * step_waves), step_lds(step_waves), nullptr, step_progs, loops, e, fit,
                       wrong, counts);
  }
  if (k.any_fast) {
    allow_lds(reinterpret_cast<const void*>(&k_eval_programs<true>), fast_lds);
    hipLaunchKernelGGL(k_eval_programs<true>, dim3(blocks), dim3(kEvalThreads), fast_lds, nullptr, progs, n, e, k.slots, k.temps,
                       k.shadow, fit, wrong, counts);
  }
  if (k.any_general && !both) {
    allow_lds(reinterpret_cast<const void*>(&k_eval_programs<false>), lds);
    hipLaunchKernelGGL(k_eval_programs<false>, dim3(blocks), dim3(kEvalThreads), lds, nullptr, progs, n, e, k.slots, k.temps,
                       k.shadow, fit, wrong, counts);
  }
  HIP_OK(hipGetLastError());
}

void Session::eval(const std::vector<ProgramIn>& programs, double* fitness, std::uint32_t* wrong, std::uint32_t* counts) {
  auto& I = *impl_;
  const int n = int(programs.size());
  if (!n) return;
  const PackedPrograms k = I.pack(programs, true);
  // One allocation and one copy each way: the launch's inputs back to back,
  // then its results.
  std::size_t bytes = 0;
  const auto place = [&](std::size_t size) {
    const std::size_t at = bytes;
    bytes += (size + 255) & ~std::size_t(255);
    return at;
  };
  const std::size_t o_progs = place(sizeof(DProg) * std::size_t(n)), o_code = place(sizeof(Ins) * k.code.size()),
                    o_pool = place(sizeof(Val) * k.pool.size()), o_steps = place(sizeof(Step) * k.steps.size()),
                    o_loops = place(sizeof(StepProg) * k.step_n.size()), inputs = bytes;
  const std::size_t o_fit = place(sizeof(double) * std::size_t(n)), o_wrong = place(sizeof(unsigned) * std::size_t(n)),
                    o_counts = place(sizeof(unsigned) * 3 * std::size_t(n));
  struct Block {
    unsigned char* p = nullptr;
    ~Block() { (void)hipFree(p); }
  } block;
  HIP_OK(hipMalloc(&block.p, bytes));
  unsigned char* const base = block.p;
  std::vector<unsigned char> staged(std::max(inputs, bytes - inputs));
  const auto put = [&](std::size_t at, const auto& v) {
    if (!v.empty()) std::memcpy(staged.data() + at, static_cast<const void*>(v.data()), v.size() * sizeof(v[0]));
  };
  put(o_progs, I.program_table(k, gbl(reinterpret_cast<const Ins*>(base + o_code)), gbl(reinterpret_cast<const Val*>(base + o_pool))));
  put(o_code, k.code);
  put(o_pool, k.pool);
  put(o_steps, k.steps);
  put(o_loops, I.step_table(k, gbl(reinterpret_cast<const Step*>(base + o_steps))));
  HIP_OK(hipMemcpy(base, staged.data(), inputs, hipMemcpyHostToDevice));
  struct Event {
    hipEvent_t e = nullptr;
    ~Event() { if (e) (void)hipEventDestroy(e); }
  } a, b;
  HIP_OK(hipEventCreate(&a.e));
  HIP_OK(hipEventCreate(&b.e));
  HIP_OK(hipEventRecord(a.e, nullptr));
  I.launch(k, reinterpret_cast<const DProg*>(base + o_progs), reinterpret_cast<const StepProg*>(base + o_loops), n,
           reinterpret_cast<double*>(base + o_fit), reinterpret_cast<unsigned*>(base + o_wrong), reinterpret_cast<unsigned*>(base + o_counts));
  HIP_OK(hipEventRecord(b.e, nullptr));
  HIP_OK(hipMemcpy(staged.data(), base + inputs, bytes - inputs, hipMemcpyDeviceToHost));
  HIP_OK(hipEventSynchronize(b.e));
  HIP_OK(hipEventElapsedTime(&I.last_ms, a.e, b.e));
  const auto take = [&](void* to, std::size_t at, std::size_t size) { std::memcpy(to, staged.data() + (at - inputs), size); };
  take(fitness, o_fit, sizeof(double) * std::size_t(n));
  if (wrong) take(wrong, o_wrong, sizeof(unsigned) * std::size_t(n));
  if (counts) take(counts, o_counts, sizeof(unsigned) * 3 * std::size_t(n));
}

// ---- allocation-free evaluation ----
// A fixed device workspace, one copy per GPU, for callers that cannot
// allocate device memory (code under HIP graph capture, serving loops,
// harnesses that forbid hipMalloc). It holds one launch's program table,
// code, constant pools and per-program results. Every call on a GPU shares
// that GPU's copy: calls that overlap on one GPU race, and the workspace keeps
// the last call's contents (the kernels write every result they report, so
// nothing needs clearing).
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace {
std::mutex scratch_mutex;
std::map<int, unsigned char*> scratch_address;  // device -> its copy of `scratch`

// The current device's copy of the workspace, resolved once per device with
// that device current. Host code uses only this address, never the symbol.
unsigned char* scratch_on_current_device() {
  int device = 0;
  HIP_OK(hipGetDevice(&device));
  std::lock_guard<std::mutex> lock(scratch_mutex);
  auto it = scratch_address.find(device);
  if (it != scratch_address.end()) return it->second;
  void* p = nullptr;
  HIP_OK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  if (!p) throw std::runtime_error("no device address for the evaluation workspace");
  scratch_address[device] = static_cast<unsigned char*>(p);
  return static_cast<unsigned char*>(p);
}

std::size_t align256(std::size_t x) { return (x + 255) & ~std::size_t(255); }
}  // namespace

std::size_t Session::static_bytes(std::size_t n, std::size_t code, std::size_t pool) {
  return align256(n * sizeof(DProg)) + align256(code * sizeof(Ins)) + align256(pool * sizeof(Val)) +
         align256(n * sizeof(double)) + align256(n * sizeof(unsigned)) + align256(3 * n * sizeof(unsigned));
}

void Session::eval_static(const std::vector<ProgramIn>& programs, double* fitness, std::uint32_t* wrong, std::uint32_t* counts) {
  const auto& I = *impl_;
  const int n = int(programs.size());
  if (!n) return;
  // Steps are staged only where they fit beside the documented parts; a
  // launch that fits without them then runs its looping programs on the
  // general VM.
  PackedPrograms k = I.pack(programs, true);
  const std::size_t need = static_bytes(std::size_t(n), k.code.size(), k.pool.size());
  if (!k.steps.empty() && need <= kStaticScratchBytes &&
      need + align256(k.steps.size() * sizeof(Step)) + align256(k.step_n.size() * sizeof(StepProg)) > kStaticScratchBytes)
    k = I.pack(programs, false);
  if (need > kStaticScratchBytes)
    throw std::invalid_argument("programs need " + std::to_string(need) + " bytes of evaluation workspace; the allocation-free "
                                "entry point holds at most " + std::to_string(kStaticScratchBytes));
  unsigned char* base = scratch_on_current_device();
  std::size_t at = 0;
  const auto carve = [&](std::size_t bytes) { unsigned char* p = base + at; at += align256(bytes); return p; };
  auto* dprogs = reinterpret_cast<DProg*>(carve(std::size_t(n) * sizeof(DProg)));
  auto* dcode = reinterpret_cast<Ins*>(carve(k.code.size() * sizeof(Ins)));
  auto* dpool = reinterpret_cast<Val*>(carve(k.pool.size() * sizeof(Val)));
  auto* dfit = reinterpret_cast<double*>(carve(std::size_t(n) * sizeof(double)));
  auto* dwrong = reinterpret_cast<unsigned*>(carve(std::size_t(n) * sizeof(unsigned)));
  auto* dcounts = reinterpret_cast<unsigned*>(carve(std::size_t(3) * n * sizeof(unsigned)));
  const auto progs = I.program_table(k, gbl(static_cast<const Ins*>(dcode)), gbl(static_cast<const Val*>(dpool)));
  StepProg* dloops = nullptr;
  if (!k.steps.empty()) {
    auto* dsteps = reinterpret_cast<Step*>(carve(k.steps.size() * sizeof(Step)));
    dloops = reinterpret_cast<StepProg*>(carve(k.step_n.size() * sizeof(StepProg)));
    const auto loops = I.step_table(k, gbl(static_cast<const Step*>(dsteps)));
    HIP_OK(hipMemcpy(dsteps, k.steps.data(), k.steps.size() * sizeof(Step), hipMemcpyHostToDevice));
    HIP_OK(hipMemcpy(dloops, loops.data(), loops.size() * sizeof(StepProg), hipMemcpyHostToDevice));
  }
  HIP_OK(hipMemcpy(dcode, k.code.data(), k.code.size() * sizeof(Ins), hipMemcpyHostToDevice));
  HIP_OK(hipMemcpy(dpool, k.pool.data(), k.pool.size() * sizeof(Val), hipMemcpyHostToDevice));
  HIP_OK(hipMemcpy(dprogs, progs.data(), progs.size() * sizeof(DProg), hipMemcpyHostToDevice));
  I.launch(k, dprogs, dloops, n, dfit, dwrong, dcounts);
  HIP_OK(hipMemcpy(fitness, dfit, sizeof(double) * n, hipMemcpyDeviceToHost));
  if (wrong) HIP_OK(hipMemcpy(wrong, dwrong, sizeof(unsigned) * n, hipMemcpyDeviceToHost));
  if (counts) HIP_OK(hipMemcpy(counts, dcounts, sizeof(unsigned) * 3 * n, hipMemcpyDeviceToHost));
}

void Session::eval_cases(const ProgramIn& program, std::vector<Val>& values, std::vector<int>& errors) {
  auto& I = *impl_;
  int ms = 0;
  bool j = false;
  bool stores = false;
  const auto ins = verify_program(program, I.cases.cd.n_inputs, ms, j, &stores);
  for (const auto& v : program.consts) check_view(v, I.arena_len);
  const int shadow = stores ? I.cases.cd.n_inputs : 0;
  const int slots = ms + 1, temps = std::max(0, std::min(64, program.n_locals) - I.cases.cd.n_inputs) + shadow;
  DeviceArena tmp;
  std::vector<Val> consts = program.consts;
  if (consts.empty()) consts.push_back(val_invalid());
  const FastCert cert = certify_fast(ins, program.consts, I.input_tags, program.n_locals, ms, j, I.cases.cd.C);
  const DProg p{tmp.upload(ins), tmp.upload(consts), int(ins.size()), j, program.n_locals, cert.fast, int(program.consts.size()),
                cert.result_tag};
  const int C = I.cases.cd.C;
  auto dv = tmp.alloc<Val>(std::size_t(C));
  auto de = tmp.alloc<int>(std::size_t(C));
  const int blocks = std::max(1, std::min(1024, (C + 255) / 256));
  if (cert.fast) {
    hipLaunchKernelGGL(k_eval_cases<true>, dim3(blocks), dim3(kEvalThreads), 0, nullptr, p, I.cases.cd, I.fuel, slots, temps, shadow,
                       dv, de);
  } else {
    const std::size_t lds = std::size_t(kWavesPerBlock) * (slots + temps) * 64 * 10;
    allow_lds(reinterpret_cast<const void*>(&k_eval_cases<false>), lds);
    hipLaunchKernelGGL(k_eval_cases<false>, dim3(blocks), dim3(kEvalThreads), lds, nullptr, p, I.cases.cd, I.fuel, slots, temps, shadow,
                       dv, de);
  }
  HIP_OK(hipGetLastError());
  HIP_OK(hipDeviceSynchronize());
  values.resize(std::size_t(C));
  errors.resize(std::size_t(C));
  HIP_OK(hipMemcpy(values.data(), dv, sizeof(Val) * C, hipMemcpyDeviceToHost));
  HIP_OK(hipMemcpy(errors.data(), de, sizeof(int) * C, hipMemcpyDeviceToHost));
}

}  // namespace gagp_amd
