// Variation of one child by one wavefront with every row in registers.
//
// For rows of at most 64 nodes over a grammar of at most 64 expressions
// (WaveGrammar): node i of a row is lane i, constant k is lane k, and the
// parent, the donor, the generated subtree and the child never leave the
// registers between being read and being stored once. The prefix-order facts
// the operators need -- subtree ends, depths, grammar-invocation depths --
// come from one pass over the row (row_shape) instead of a walk per question,
// and a splice is a handful of lane shuffles. crossover_w, mutate_w and
// compare_w (phase_wave.hpp) are the forms for wider rows and grammars; both
// consume the same draws and give the same child.
//
// What bounds it: the row-by-row form spent 57% of its cycles waiting for
// about 78 global and 85 LDS loads a child, each a dependent round trip. Here
// a child reads its tournament keys, its two rows at once, and its member
// probe; what is left is the chain of the derivation and of the draws. With the
// derivation over lane registers (derive_w), a round of 4096 children of the
// quintic grammar takes 58 us where it took 154, 1024 of a polynomial 41 for 84,
// 8192 of a list grammar 159 for 282, 1500 of a statement grammar 99 for 189.
#pragma once
#include "phase_wave.hpp"

namespace gagp_amd {

constexpr int kWaveRow = 64;
constexpr int kLaneValues = 64;  // pool entries of a program lowered with jumps
// LDS of a wavefront that lowers rows: exchange words and, with jumps, the
// program, which the caller decodes from here or stores in order.
template <bool kJumps> struct LaneStore { int sums[64]; };
template <> struct LaneStore<true> {
  int sums[64];
  Ins code[kLoopCode];
};

// ---- wavefront reductions and scans in the data-parallel shifts (all lanes active) ----
template <int kControl, int kRows>
__device__ inline int lane_shift(int x) { return __builtin_amdgcn_update_dpp(0, x, kControl, kRows, 0xf, false); }
// Inclusive sum over the lanes.
__device__ inline int wave_scan(int x) {
  x += lane_shift<0x111, 0xf>(x);
  x += lane_shift<0x112, 0xf>(x);
  x += lane_shift<0x114, 0xf>(x);
  x += lane_shift<0x118, 0xf>(x);
  x += lane_shift<0x142, 0xa>(x);
  x += lane_shift<0x143, 0xc>(x);
  return x;
}
// Largest of non-negative values, uniform.
__device__ inline int wave_max(int x) {
  const auto up = [&](int y) { x = y > x ? y : x; };
  up(lane_shift<0x111, 0xf>(x));
  up(lane_shift<0x112, 0xf>(x));
  up(lane_shift<0x114, 0xf>(x));
  up(lane_shift<0x118, 0xf>(x));
  up(lane_shift<0x142, 0xa>(x));
  up(lane_shift<0x143, 0xc>(x));
  return rdlane(x, 63);
}
__device__ inline std::uint64_t wave_total(std::uint64_t x) {
  const auto add = [&](auto shift) {
    const unsigned lo = unsigned(shift(int(unsigned(x)))), hi = unsigned(shift(int(unsigned(x >> 32))));
    x += std::uint64_t(hi) << 32 | lo;
  };
  add([](int v) { return lane_shift<0x111, 0xf>(v); });
  add([](int v) { return lane_shift<0x112, 0xf>(v); });
  add([](int v) { return lane_shift<0x114, 0xf>(v); });
  add([](int v) { return lane_shift<0x118, 0xf>(v); });
  add([](int v) { return lane_shift<0x142, 0xa>(v); });
  add([](int v) { return lane_shift<0x143, 0xc>(v); });
  const unsigned lo = unsigned(rdlane(int(unsigned(x)), 63)), hi = unsigned(rdlane(int(unsigned(x >> 32)), 63));
  return std::uint64_t(hi) << 32 | lo;
}
__device__ inline std::uint64_t bits_below(int i) { return i >= 64 ? ~0ull : (1ull << i) - 1ull; }
__device__ inline int lane_of(int v, int lane) { return __shfl(v, lane & 63, 64); }

// Orders LDS accesses of the wavefront's lanes around it: the hardware runs
// them in order, and the compiler, which sees one lane, must not carry a
// value over.
__device__ inline void lanes_meet() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// ---- draws ----
// bounded(n) for 0 < n < 2^20, rejections included: 2^64 mod n from 2^63 mod n.
__device__ inline unsigned bounded_small(WaveDraws& draws, unsigned n) {
  for (;;) {
    const std::uint64_t v = draws.take();
    if (v < n) {
      const unsigned half = mod_small(1ull << 63, n), threshold = 2 * half >= n ? 2 * half - n : 2 * half;
      if (v < threshold) continue;
    }
    return unsigned(__builtin_amdgcn_readfirstlane(int(mod_small(v, n))));
  }
}

// ---- rows ----
struct WaveRow {
  int n = 0, nc = 0;
  int origin = 0, site = -1;           // node `lane`
  unsigned c0 = 0, c1 = 0, ct = 0;     // constant `lane`: payload, tag | flag << 8
};
// A row in memory (row length R <= 64): all its loads at once, the counts with them.
__device__ inline WaveRow load_row(GAS const int* origin, GAS const int* site, GAS const Val* cval, int R, int n, int nc) {
  WaveRow r;
  const int lane = wlane();
  if (lane < R) {
    r.origin = origin[lane];
    r.site = site[lane];
    const std::int64_t v = cval[lane].i;
    r.ct = unsigned(cval[lane].tag) | unsigned(cval[lane].b) << 8;
    r.c0 = unsigned(std::uint64_t(v));
    r.c1 = unsigned(std::uint64_t(v) >> 32);
  }
  r.n = __builtin_amdgcn_readfirstlane(n);
  r.nc = __builtin_amdgcn_readfirstlane(nc);
  if (lane >= r.n) { r.origin = 0; r.site = -1; }
  if (lane >= r.nc) r.ct = TAG_INVALID;
  return r;
}
__device__ inline void store_row(const WaveRow& r, GAS int* origin, GAS int* site, GAS Val* cval) {
  const int lane = wlane();
  if (lane < r.n) { origin[lane] = r.origin; site[lane] = r.site; }
  if (lane < r.nc) {
    Val v{};
    v.i = std::int64_t(std::uint64_t(r.c1) << 32 | r.c0);
    v.tag = std::uint8_t(r.ct);
    v.b = std::uint8_t(r.ct >> 8);
    cval[lane].i = v.i;
    *(GAS std::uint64_t*)(&cval[lane].b) = std::uint64_t(v.b) | std::uint64_t(v.tag) << 8;
  }
}

// The prefix-order facts of a row, per lane i < n: arity; the position after
// its subtree; depth (1 at the root); the site flags and arities of its
// ancestors; and the contract of its variation site (nonterminal | scope << 8;
// -1 when it has none or a fixed one).
struct RowShape {
  int arity, end, depth, inc, above, open, contract;
  std::uint64_t constants, sites;  // nodes that are constants; nodes with an eligible site
  bool ok;                         // well formed
};
// `hist`: 64 LDS words of this wavefront. With q_i = 1 + sum_{k<i} (arity_k - 1)
// the open child slots before node i, the subtree of j ends at the next i > j
// with q_i = q_j - 1 (the count falls by at most one a node), found for all j
// of one q at once; then the ancestors of i are the nodes before i less those
// whose subtrees have ended, two prefix sums.
__device__ inline RowShape row_shape(const WaveGrammar& w, const WaveRow& r, LAS int* hist) {
  RowShape s;
  const int lane = wlane(), n = r.n;
  const bool live = lane < n;
  const unsigned x = unsigned(lane_of(int(w.expr), r.origin));
  const unsigned y = unsigned(lane_of(int(w.expr), r.site & 63));
  const int target = int(y >> 16) & 63;
  const bool fixed = (unsigned(lane_of(int(w.nt), target)) >> 25 & 1u) != 0;
  s.arity = live ? int((x >> 3) & 15u) : 0;
  s.contract = live && r.site >= 0 && !fixed ? target | int((y >> 7) & 15u) << 8 : -1;
  s.sites = __ballot(s.contract >= 0);
  s.constants = __ballot(live && (x & 7u) == unsigned(PK_CONSTANT));
  const int delta = live ? s.arity - 1 : 0;
  const int sum = wave_scan(delta);
  s.open = 1 + sum - delta;
  s.end = n;
  for (std::uint64_t left = __ballot(live); left;) {
    const int v = rdlane(s.open, wave_first(left));
    const std::uint64_t same = __ballot(live && s.open == v), lower = __ballot(live && s.open == v - 1);
    const std::uint64_t after = lower & ~lanes_below() & ~(1ull << lane);
    if (s.open == v) s.end = after ? __ffsll((long long)after) - 1 : n;
    left &= ~same;
  }
  const int flags = live && r.site >= 0 ? 1 : 0;
  const int mine = live ? 1 | flags << 8 | s.arity << 16 : 0;
  hist[lane] = 0;
  lanes_meet();
  if (live && s.end < n) atomicAdd((int*)(hist + s.end), mine);
  lanes_meet();
  const int ended = hist[lane];
  const int up = wave_scan(mine) - mine - wave_scan(ended);
  s.depth = 1 + (up & 255);
  s.inc = (up >> 8) & 255;
  s.above = up >> 16;
  const int closes = 1 + rdlane(sum, 63);
  s.ok = n > 0 && closes == 0 && __ballot(live && (s.open < 1 || s.arity > kMaxArity || (s.arity > 0 && s.depth >= 64))) == 0;
  return s;
}

// choose_site over the nodes of `eligible`.
__device__ inline int choose_site(std::uint64_t eligible, WaveDraws& draws, bool counted) {
  const int count = __popcll(eligible);
  if (count == 0) return -1;
  if (counted) {
    const int rank = int(bounded_small(draws, unsigned(count)));
    return wave_first(__ballot((eligible >> wlane() & 1u) && __popcll(eligible & lanes_below()) == rank));
  }
  int selected = -1;
  unsigned seen = 0;
  for (std::uint64_t m = eligible; m; m &= m - 1)
    if (bounded_small(draws, ++seen) == 0) selected = wave_first(m);
  return selected;
}

// Row `a` with the subtree [dest, end) replaced by [src, src_end) of `b`;
// `ca`, `cb`: their constant nodes. The caller has checked the bounds.
__device__ inline WaveRow splice_rows(const WaveRow& a, std::uint64_t ca, int dest, int end, const WaveRow& b, std::uint64_t cb, int src,
                                      int src_end) {
  WaveRow out;
  const int lane = wlane(), grown = src_end - src, in_end = dest + grown;
  const bool inside = lane >= dest && lane < in_end;
  const int ia = lane < dest ? lane : lane + (end - dest) - grown, ib = lane - dest + src;
  const int ao = lane_of(a.origin, ia), as = lane_of(a.site, ia), bo = lane_of(b.origin, ib), bs = lane_of(b.site, ib);
  out.n = a.n - (end - dest) + grown;
  out.origin = inside ? bo : ao;
  out.site = inside ? bs : as;
  if (lane == dest) out.site = rdlane(a.site, dest);
  if (lane >= out.n) { out.origin = 0; out.site = -1; }
  const int head = __popcll(ca & bits_below(dest)), tail = __popcll(ca & bits_below(end));
  const int first = __popcll(cb & bits_below(src)), in = __popcll(cb & bits_below(src_end)) - first;
  out.nc = head + in + __popcll(ca) - tail;
  const bool middle = lane >= head && lane < head + in;
  const int ka = lane < head ? lane : lane - head - in + tail, kb = lane - head + first;
  const unsigned a0 = unsigned(lane_of(int(a.c0), ka)), a1 = unsigned(lane_of(int(a.c1), ka)), at = unsigned(lane_of(int(a.ct), ka));
  const unsigned b0 = unsigned(lane_of(int(b.c0), kb)), b1 = unsigned(lane_of(int(b.c1), kb)), bt = unsigned(lane_of(int(b.ct), kb));
  out.c0 = middle ? b0 : a0;
  out.c1 = middle ? b1 : a1;
  out.ct = lane < out.nc ? (middle ? bt : at) : unsigned(TAG_INVALID);
  return out;
}

// A row and its grammar's nodes in registers, for the walk shared with the host.
struct RowOrigins {
  int origin;
  unsigned node, node2;
  __device__ int operator()(int i) const { return rdlane(origin, i); }
};
__device__ inline PNode node_of(const RowOrigins& r, const PhaseView&, int origin) { return unpack_node(r.node, r.node2, origin); }
__device__ inline bool locals_defined_row(const PhaseView& g, const WaveGrammar& w, const WaveRow& r) {
  WaveDefFrames frames;
  return locals_defined_with(g, r.n, RowOrigins{r.origin, w.node, w.node2}, frames);
}

// The parent and donor tournaments (tournaments_w) from the first draws.
__device__ inline void tournament_rows(const Keys& k, int population, int pressure, WaveDraws& draws, int& parent, int& donor) {
  const int drawn = 2 * pressure, lane = wlane();
  const bool mine = lane < drawn;
  const std::uint64_t v = std::uint64_t(draws.hi) << 32 | draws.lo;
  if (drawn > 64 || population >= 1 << 20 || __ballot(mine && v < std::uint64_t(population)) != 0) {
    SplitMix random(draws.base);
    tournaments_w(k, population, pressure, random, parent, donor);
    draws = WaveDraws(random.s);
    return;
  }
  const int c = mine ? int(mod_small(v, unsigned(population))) : 0;
  const double f = mine ? k.fitness[c] : 0.0;
  const int wrong = mine && k.has_wrong ? int(k.wrong[c]) : 0, nodes = mine && k.has_wrong ? int(k.nodes[c]) : 0;
  const auto select = [&](int first) {
    int best = rdlane(c, first), bw = rdlane(wrong, first), bn = rdlane(nodes, first);
    double bf = rdlane_d(f, first);
    for (int i = first + 1; i < first + pressure; ++i) {
      const int ci = rdlane(c, i), wi = rdlane(wrong, i), ni = rdlane(nodes, i);
      const double fi = rdlane_d(f, i);
      bool over;
      if (fi != bf) over = fi > bf;
      else if (!k.has_wrong) over = false;
      else if (wi != bw) over = unsigned(wi) < unsigned(bw);
      else if (ni != bn) over = unsigned(ni) < unsigned(bn);
      else over = ci < best;
      if (over) { best = ci; bf = fi; bw = wi; bn = ni; }
    }
    return best;
  };
  parent = select(0);
  donor = select(pressure);
  draws.next = drawn;
}

// crossover_child: the child of `a` (already in `child`) and `b`.
__device__ inline void cross_rows(const PhaseView& g, const WaveGrammar& w, const SlotInfo& s, const WaveRow& a, const WaveRow& b,
                                  WaveRow& child, WaveDraws& draws, const OpPolicy& pol, LAS int* hist, OpStats& st) {
  if (pol.crossover_probability < 1 && draws.unit() >= pol.crossover_probability) return;
  st.crossover_attempted = 1;
  if (pol.uniform_phase) (void)draws.take();  // bounded(1) accepts any draw
  const RowShape sa = row_shape(w, a, hist), sb = row_shape(w, b, hist);
  const int lane = wlane(), total = a.n;
  for (int attempt = 0; attempt < pol.crossover_attempts && !st.crossover; ++attempt) {
    const int dest = choose_site(sa.sites, draws, pol.counted_sites != 0);
    if (dest < 0) break;
    const int contract = rdlane(sa.contract, dest);
    const int src = choose_site(__ballot(sb.contract == contract), draws, pol.counted_sites != 0);
    bool taken = src >= 0;
    if (taken && !(sa.ok && sb.ok)) { st.error = 3; return; }
    const int from = taken ? src : 0, end = rdlane(sa.end, dest), src_end = rdlane(sb.end, from), length = total - (end - dest) + (src_end - from);
    taken = taken && length <= s.max_variable_nodes && length <= s.row_capacity && s.max_depth > 0 && s.max_depth <= 64;
    if (taken) {
      // The kept nodes of `a` and the donor's at their new depths.
      const bool kept = lane < total && (lane < dest || lane >= end), moved = lane >= from && lane < src_end;
      const int deeper = rdlane(sa.depth, dest) - rdlane(sb.depth, from), further = rdlane(sa.inc, dest) - rdlane(sb.inc, from);
      const bool deep = (kept && sa.depth > s.max_depth) || (moved && sb.depth + deeper > s.max_depth);
      const int va = sa.inc + (a.site >= 0 ? 1 : 0), vb = sb.inc + further + (b.site >= 0 ? 1 : 0);
      const bool far = s.logical_depth && ((kept && va > s.logical_depth) || (moved && vb > s.logical_depth));
      taken = __ballot(deep || far) == 0 && __popcll(sa.constants) <= a.nc && __popcll(sb.constants) <= b.nc;
    }
    if (taken) {
      const WaveRow out = splice_rows(a, sa.constants, dest, end, b, sb.constants, from, src_end);
      taken = !s.statement || locals_defined_row(g, w, out);
      if (taken) child = out;
    }
    if (taken) st.crossover = 1;
    else ++st.crossover_rejected;
  }
}

// The derivation's output in registers (at most 64 nodes).
struct RowSink {
  WaveRow row;
  __device__ void node(int at, int origin, int site) {
    const bool mine = wlane() == at;
    row.origin = mine ? origin : row.origin;
    row.site = mine ? site : row.site;
  }
  __device__ void constant(int k, const Val& v) {
    const bool mine = wlane() == k;
    row.c0 = mine ? unsigned(std::uint64_t(v.i)) : row.c0;
    row.c1 = mine ? unsigned(std::uint64_t(v.i) >> 32) : row.c1;
    row.ct = mine ? unsigned(v.tag) | unsigned(v.b) << 8 : row.ct;
  }
  __device__ void finish(int) {}
};

// mutate_child on `x`; `tmp`: the child's memory row for a subtree the
// general derivation makes.
__device__ inline void mutate_row(const PhaseView& g, const WaveGrammar& w, const SlotInfo& s, WaveRow& x, Row& tmp, double probability,
                                  std::uint64_t seed, const OpPolicy& pol, LAS int* hist, OpStats& st) {
  if (st.error) return;
  if (x.n <= 0) { st.error = 4; return; }
  WaveDraws draws(seed);
  if (draws.unit() >= probability) return;
  if (pol.uniform_phase) (void)draws.take();
  const RowShape sx = row_shape(w, x, hist);
  const int dest = choose_site(sx.sites, draws, pol.counted_sites != 0);
  if (dest < 0) return;
  const int end = rdlane(sx.end, dest), depth = rdlane(sx.depth, dest), incoming = s.logical_depth ? rdlane(sx.inc, dest) : 0;
  if (!sx.ok || incoming > s.logical_depth) { st.error = 6; return; }
  const int site = rdlane(x.site, dest), total = x.n, replaced = end - dest;
  const int whole = s.max_variable_nodes - (total - replaced), phase = kPhaseCapacity - (total - replaced);
  const int available = whole < phase ? whole : phase, uncapped = available < kPhaseCapacity ? available : kPhaseCapacity;
  const bool capped = pol.mutation_max_nodes > 0 && pol.mutation_max_nodes < uncapped;
  const int bounded = capped ? pol.mutation_max_nodes : uncapped;
  if (bounded > s.row_capacity) { st.error = 10; return; }
  const std::uint64_t stream = draws.take();
  const int sub_depth = s.max_depth - depth + 1, logical = s.logical_depth - incoming;
  RowSink sink;
  GenResult gen{ST_INVALID, 0, 0, 0};
  if (derive_w(g, w, site_entry(site), site_parent_scope(site), sub_depth, bounded, stream, sink, logical, gen)) {
    sink.row.n = gen.nodes;
    sink.row.nc = gen.constants;
  } else {
    WaveTasks pending;
    gen = generate_phase_with(g, site_entry(site), site_parent_scope(site), sub_depth, bounded, stream, tmp.origin, tmp.cval, tmp.site, logical,
                              pending);
    wave_fence();
    sink.row = load_row(gbl((const int*)tmp.origin), gbl((const int*)tmp.site), gbl((const Val*)tmp.cval), s.row_capacity, gen.nodes, gen.constants);
  }
  if (capped && gen.status == ST_CAPACITY) return;
  if (gen.status != ST_OK) { st.error = 7; return; }
  const WaveRow& sub = sink.row;
  // The subtree keeps the depth and invocation bounds it was derived under.
  if (site < 0 || rdlane(sub.site, 0) < 0 || total - replaced + sub.n > s.row_capacity) { st.error = 8; return; }
  const unsigned kinds = unsigned(lane_of(int(w.expr), sub.origin));
  const std::uint64_t constants = __ballot(wlane() < sub.n && (kinds & 7u) == unsigned(PK_CONSTANT));
  const WaveRow out = splice_rows(x, sx.constants, dest, end, sub, constants, 0, sub.n);
  if (s.statement && !locals_defined_row(g, w, out)) return;
  x = out;
  st.mutation = 1;
}

// Whether two rows are the same genotype (rows_equal).
__device__ inline bool same_rows(const WaveRow& a, const WaveRow& b) {
  const int lane = wlane();
  const unsigned tag = a.ct & 255u;
  const bool same = tag == (b.ct & 255u) && (tag == unsigned(TAG_BOOL) ? (a.ct >> 8) == (b.ct >> 8) : a.c0 == b.c0 && a.c1 == b.c1);
  return a.n == b.n && a.nc == b.nc && __ballot((lane < a.n && a.origin != b.origin) || (lane < a.nc && !same)) == 0;
}

// compare_child.
__device__ inline void compare_rows(const WaveRow& parent, const WaveRow& child, int population, OpStats& st) {
  if (st.parent < 0 || st.parent >= population) { st.error = 9; return; }
  const bool equal = same_rows(parent, child);
  const bool raw = parent.c0 != child.c0 || parent.c1 != child.c1 || parent.ct >> 8 != child.ct >> 8;
  const bool reusable = __ballot(wlane() < child.nc && raw) == 0;
  st.changed = !equal;
  st.reusable_parent = equal && reusable ? st.parent : -1;
}
__device__ inline std::uint64_t row_hash_row(const WaveRow& r) {
  const int lane = wlane();
  std::uint64_t h = 0;
  if (lane < r.n) h += row_hash_node(lane, r.origin);
  if (lane < r.nc) {
    Val v{};
    v.i = std::int64_t(std::uint64_t(r.c1) << 32 | r.c0);
    v.tag = std::uint8_t(r.ct);
    v.b = std::uint8_t(r.ct >> 8);
    h += row_hash_constant(lane, v);
  }
  return wave_total(h) + row_hash_counts(r.n, r.nc);
}

// ---- lowering ----
// lower_phase_with with one lane per node. The code of a program is its nodes'
// pieces in the order its walk completes children: piece k of a node follows
// its child k (the last one ends the node), and its length depends on the
// node's kind alone. Piece positions, pool indices, live temporaries and stack
// heights are then prefix sums over the row less the open ancestors' share,
// and every lane writes its node's instructions. Returns false, with nothing
// of use stored, unless every check of lower_phase_with passes on the types
// the grammar declares; the node-by-node lowering then decides.
// kJumps: all kinds; otherwise constants, inputs and operations only.
// A statement row has been checked for definite assignment. `store`: this
// wavefront's LDS, which alone has the code with kJumps.
// Node by node a child took 1.2 us a node, and 75-100 us with traversals; a
// row takes 3 us here, 6 with jumps. The program stays in LDS for the decoding,
// which read its neighbours' words from global memory in 20 us and takes half.
template <bool kJumps>
__device__ inline bool lower_row(const WaveGrammar& w, const WaveRow& r, GAS const std::uint8_t* local_types, int local_count,
                                 int expected_type, GAS Ins* code, int code_capacity, GAS Val* pool, int pool_capacity,
                                 LAS LaneStore<kJumps>* store, LowerResult& out) {
  const int lane = wlane(), n = r.n;
  LAS int* const sums = store->sums;
  if (n <= 0 || n > 64) return false;
  const bool live = lane < n, statement = kJumps && expected_type == kStatementType;
  const int x = lane_of(int(w.node), r.origin), x2 = lane_of(int(w.node2), r.origin);
  const int kind = live ? x & 31 : int(TK_NIL), opcode = (x >> 5) & 31, operand = x >> 16, type = x2 & 255;
  const unsigned fuel = unsigned(x2 >> 8) & 255u;
  const RowShape s = row_shape(w, r, sums);
  // Sums over a node's ancestors, of values in disjoint bit fields.
  const auto over_ancestors = [&](int mine) {
    lanes_meet();
    sums[lane] = 0;
    lanes_meet();
    if (live && s.end < n) atomicAdd((int*)(sums + s.end), mine);
    lanes_meet();
    const int ended = sums[lane];
    return wave_scan(mine) - mine - wave_scan(ended);
  };
  const bool constant = live && kind == TK_CONSTANT, local = live && kind == TK_LOCAL, operation = live && kind == TK_OPERATION;
  const bool branch = kJumps && live && kind == TK_IF, logic = kJumps && live && (kind == TK_AND || kind == TK_OR);
  const bool walk = kJumps && live && kind == TK_TRAVERSE, bind = kJumps && live && kind == TK_BOUND;
  const bool let = kJumps && live && kind == TK_LET, range = kJumps && live && kind == TK_FOR_RANGE;
  const bool var = kJumps && live && kind == TK_VAR, assign = kJumps && live && kind == TK_ASSIGN, ret = kJumps && live && kind == TK_RETURN;
  const bool program = kJumps && live && kind == TK_PROGRAM, block = kJumps && live && kind == TK_BLOCK, nil = kJumps && live && kind == TK_NIL;
  const bool ranged = walk && s.arity == 6, reverse = opcode == 2;
  // Arities of the kinds.
  bool bad = live && !(operation ? s.arity >= 1 && s.arity <= 3
                                 : walk ? (s.arity == 4 || s.arity == 6) && operand >= 0 && operand + 2 < 16
                                        : s.arity == (branch ? 3 : logic || let || range || block ? 2 : program || assign || ret ? 1 : 0));
  bad = bad || (live && !(constant || local || operation || branch || logic || walk || bind || let || range || var || assign || ret ||
                          program || block || nil));
  if (__ballot(bad) != 0 || !s.ok) return false;
  // The children's positions.
  const int k1 = lane + 1, k2 = lane_of(s.end, k1), k3 = lane_of(s.end, k2);
  const int k4 = kJumps ? lane_of(s.end, k3) : 0, k5 = kJumps ? lane_of(s.end, k4) : 0, k6 = kJumps ? lane_of(s.end, k5) : 0;
  // The parent's lane and the child's number in it.
  int index = 0, px = 0, parent_arity = 0;
  {
    lanes_meet();
    sums[lane] = 0;
    lanes_meet();
    const auto claim = [&](int child, int k) {
      if (live && s.arity > k) sums[child & 63] = lane | k << 8;
    };
    claim(k1, 0);
    claim(k2, 1);
    claim(k3, 2);
    if (kJumps) {
      claim(k4, 3);
      claim(k5, 4);
      claim(k6, 5);
    }
    lanes_meet();
    const int claimed = sums[lane];
    index = claimed >> 8;
    px = lane_of(x, claimed & 63);
    parent_arity = lane_of(s.arity, claimed & 63);
  }
  const int parent_kind = lane == 0 || !live ? -1 : px & 31;
  // Lengths of the piece before this child and of the node's last piece: code
  // words, and pool entries << 16.
  int before = 0, last = 0;
  if (constant) last = 1 | 1 << 16;
  else if (live && !(branch || program || block || nil || let)) last = 1;
  if (kJumps) {
    if (index > 0) {
      if (parent_kind == TK_IF || parent_kind == TK_AND || parent_kind == TK_OR || parent_kind == TK_LET) before = 1;
      if (parent_kind == TK_FOR_RANGE) before = 18 | 4 << 16;
      if (parent_kind == TK_TRAVERSE) {
        const bool six = parent_arity == 6, back = ((px >> 5) & 31) == 2;
        before = index == parent_arity - 1 ? (back ? 17 | 1 << 16 : 15) : index == (six ? 4 : 2) ? (six ? 39 | 4 << 16 : 11 | 1 << 16) : 1;
      }
    }
    if (logic) last = 4 | 1 << 16;
    if (walk) last = 7 | 1 << 16;
    if (range) last = 5;
  }
  const int mine = before + last, ran = wave_scan(mine) - mine;  // before this node, had every one of them ended
  const int total = rdlane(ran + mine, 63), open = over_ancestors(last);
  const int ran_end = lane_of(ran, s.end), start = ran + before - open, at = (s.end < 64 ? ran_end : total) - open - last;
  const int words = (total & 0xffff) + (statement ? 0 : 1), entries = total >> 16;
  // Values below a node: the earlier operands of the operations it is in.
  const int under = parent_kind == TK_OPERATION ? index : 0;
  int base, depth_live = 0;
  if (kJumps) {
    const int body = parent_kind == TK_FOR_RANGE && index == 1 ? 1 : 0;
    const int held = (walk ? 9 : let || range ? 1 : 0) + body;
    const int sum = over_ancestors(under | held << 16);
    base = (sum & 0xffff) + under;
    depth_live = (sum >> 16) + body;
  } else {
    base = over_ancestors(under) + under;
  }
  const int bound = wave_max(live ? (s.arity == 0 && !nil ? base + 1 : walk || range ? base + 2 : logic ? base + 1 : 0) : 0);
  if (words > code_capacity || entries > pool_capacity || (kJumps && (words > kLoopCode || entries > kLaneValues))) return false;

  // Types: each node's, as the grammar declares it or its rule gives it, and
  // the rules checked against the operands' below.
  const int rank = __popcll(s.constants & lanes_below());
  int rule = TAG_INVALID;
  if (opcode == OP_NEG || opcode == OP_CHECK_INT || (opcode >= OP_ADD && opcode <= OP_MUL) || opcode == OP_MOD) rule = TAG_INT;
  if (opcode == OP_NOT || (opcode >= OP_LT && opcode <= OP_NE)) rule = TAG_BOOL;
  const int constant_type = int(unsigned(lane_of(int(r.ct), rank)) & 255u);
  int result = constant ? constant_type : operation && rule != TAG_INVALID ? rule : logic ? int(TAG_BOOL) : nil || range || program || block || assign || ret ? kStatementType : type;
  if (local) result = operand >= 0 && operand < local_count ? int(local_types[operand]) : int(TAG_INVALID);
  // Binders: the innermost traversal body or let around a bound read, by
  // going through them outside in.
  int binder = -1;  // lane | role << 8
  if (kJumps) {
    for (std::uint64_t m = __ballot(walk || let); m; m &= m - 1) {
      const int j = wave_first(m);
      const int jx = rdlane(x, j), arity = rdlane(s.arity, j), first = jx >> 16;
      const int body = rdlane(arity == 6 ? k6 : arity == 4 ? k4 : k2, j), end = rdlane(s.end, j);
      const int kept = (jx & 31) == TK_LET ? rdlane(result, j + 1) : rdlane(type, j);
      const int roles = (jx & 31) == TK_LET ? 1 : 3, role = operand - first;
      if (bind && lane >= body && lane < end && role >= 0 && role < roles) {
        binder = j | role << 8;
        result = roles == 1 || role == 2 ? kept : int(TAG_INT);
      }
    }
    bad = bind && (binder < 0 || operand < 0 || operand >= 16 || (type != TAG_INVALID && type != result));
  }
  const int t1 = lane_of(result, k1), t2 = lane_of(result, k2), t3 = lane_of(result, k3);
  bool fast = true, typed = true;
  if (constant || local || bind || var) {
    bad = bad || result == TAG_INVALID || result == TAG_FALLBACK || (var && result == kStatementType);
    fast = (constant || local) && fast_type(result);
    typed = constant ? fast_type(result) : loop_type(result);
  }
  if (operation) {
    const bool one = opcode == OP_NEG || opcode == OP_CHECK_INT || opcode == OP_NOT, pair = opcode == OP_EQ || opcode == OP_NE;
    const int want = opcode == OP_NOT ? TAG_BOOL : TAG_INT;
    if (rule != TAG_INVALID)
      bad = bad || s.arity != (one ? 1 : 2) || (type != TAG_INVALID && type != rule) ||
            !(pair ? t1 == t2 && fast_type(t1) : t1 == want && (one || t2 == want));
    bad = bad || result == TAG_INVALID || result == TAG_FALLBACK;
    fast = fast_type(result) && fast_operation(opcode, operand, s.arity, t1, t2, t3);
    typed = fast_type(result) && loop_operation(opcode, operand, s.arity, t1, t2, t3);
  }
  int returned = TAG_INVALID;
  if (kJumps) {
    if (branch) bad = bad || t1 != TAG_BOOL || t2 != t3 || t2 != result;
    if (logic) bad = bad || t1 != TAG_BOOL || t2 != TAG_BOOL;
    const int t4 = lane_of(result, k4), t5 = lane_of(result, k5), t6 = lane_of(result, k6);
    if (walk) {
      bad = bad || t1 != TAG_INT_LIST || t2 != TAG_INT ||
            (ranged ? t3 != TAG_INT || t4 != TAG_INT || t5 != type || t6 != type : t3 != type || t4 != type);
    }
    if (program) bad = bad || t1 != kStatementType;
    if (block) bad = bad || t1 != kStatementType || t2 != kStatementType;
    if (assign || ret) bad = bad || t1 != type || t1 == kStatementType;
    if (range) {
      bad = bad || t1 == kStatementType || t2 != kStatementType;
      typed = t1 == TAG_INT;
    }
    if (let) bad = bad || operand < 0 || operand >= 16 || t1 == kStatementType || t2 == kStatementType || t2 != type;
    const std::uint64_t returns = __ballot(ret);
    if (returns) {
      returned = rdlane(type, wave_first(returns));
      if (ret && type != returned) bad = true;
    }
    if (__popcll(__ballot(range)) > 16 || __popcll(__ballot(let)) > 16 || wave_max(depth_live + (walk ? 9 : 0)) > 64) bad = true;
  }
  const int root = rdlane(result, 0);
  if (__ballot(bad) != 0 || __popcll(s.constants) != r.nc || root != expected_type) return false;

  // Slots: temporary k of those live at once is the same one every time it is
  // taken, numbered when it is first taken among the grammar locals' first
  // writes (a temporary first at equal positions: it was taken earlier).
  int locals = local_count, slot = 0, user = 0;
  int temporaries = 0;
  std::uint64_t named = 0;
  if (kJumps) {
    temporaries = wave_max(live ? depth_live + (walk ? 9 : let ? 1 : range ? 2 : 0) : 0);
    const int opens = start & 0xffff, tested = (lane_of(start - before, k2)) & 0xffff;  // a for_range's piece after its bound
    const int written = assign ? at & 0xffff : tested;
    const bool writes = (assign || range) && operand >= 0;
    int temp_slot = lane, name_slot = 0;
    if (__ballot(writes)) {
      constexpr int kNever = 1 << 20;
      lanes_meet();
      sums[lane] = kNever;
      lanes_meet();
      if (walk)
        for (int k = 0; k < 9; ++k) atomicMin((int*)(sums + ((depth_live + k) & 63)), opens);
      if (let || range) atomicMin((int*)(sums + (depth_live & 63)), opens);
      if (range) atomicMin((int*)(sums + ((depth_live + 1) & 63)), tested);
      lanes_meet();
      const int taken = sums[lane];
      lanes_meet();
      sums[lane] = kNever;
      lanes_meet();
      if (writes && operand < 16) atomicMin((int*)(sums + (operand & 15)), written);
      lanes_meet();
      const int first = sums[lane];
      named = __ballot(lane < 16 && first < kNever);
      for (std::uint64_t m = named; m; m &= m - 1) {
        const int v = wave_first(m), when = rdlane(first, v);
        temp_slot += when < taken ? 1 : 0;
        const int below = __popcll(__ballot(lane < temporaries && taken <= when)) + __popcll(__ballot((named >> lane & 1u) && first < when));
        name_slot = lane == v ? below : name_slot;
      }
      if (__ballot((writes && operand >= 16) || (var && !(operand >= 0 && operand < 16 && (named >> (operand & 15) & 1u))))) return false;
    } else if (__ballot(var)) {
      return false;
    }
    locals += temporaries + __popcll(named);
    if (locals > 64) return false;
    if (__ballot((assign || range) && operand < 0 && -1 - operand >= local_count)) return false;
    // The lane's own first temporary, its named local, and a bound read's slot.
    const int at_binder = binder & 63, role = binder >> 8;
    const int bound_live = lane_of(depth_live + (let ? 0 : 6), at_binder) + role;  // element, index and state follow six others
    const int of = bind ? bound_live : depth_live;
    slot = local_count + lane_of(temp_slot, of);
    const int name = lane_of(name_slot, operand);
    user = operand < 0 ? -1 - operand : local_count + name;
    lanes_meet();
    sums[lane] = local_count + temp_slot;  // each temporary's slot
    lanes_meet();
  }

  // ---- the instructions ----
  const auto put = [&](int to, int op, int argc, int sp, unsigned cost, int a) {
    const std::uint64_t word = std::uint64_t(unsigned(op) | unsigned(argc) << 8 | unsigned(sp) << 16 | cost << 24) | std::uint64_t(unsigned(a)) << 32;
    if constexpr (kJumps) *(LAS std::uint64_t*)(store->code + to) = word;
    else *(GAS std::uint64_t*)(code + to) = word;
  };
  const auto put_value = [&](int to, std::uint64_t v, unsigned tag, unsigned flag) {
    pool[to].i = std::int64_t(v);
    *(GAS std::uint64_t*)(&pool[to].b) = std::uint64_t(flag) | std::uint64_t(tag) << 8;
  };
  const int end = at & 0xffff, end_pool = at >> 16;
  if (constant || local || bind || var || operation) {
    const int op = constant ? int(OP_PUSH_CONST) : operation ? opcode : int(OP_LOAD);
    const int argc = operation && opcode == OP_CALL_BUILTIN ? s.arity : 0;
    const int a = constant ? end_pool : local || (operation && opcode == OP_CALL_BUILTIN) ? operand : bind ? slot : var ? user : 0;
    put(end, op, argc, base + (operation ? s.arity : 0), fuel, a);
  }
  {
    const unsigned c0 = unsigned(lane_of(int(r.c0), rank)), c1 = unsigned(lane_of(int(r.c1), rank)), ct = unsigned(lane_of(int(r.ct), rank));
    if (constant) put_value(end_pool, std::uint64_t(c1) << 32 | c0, ct & 255u, ct >> 8 & 255u);
  }
  bool jumps = false;
  if (kJumps) {
    // Where the pieces after the children start.
    const int piece = start - before;
    const int p2 = lane_of(piece, k2), p3 = lane_of(piece, k3), p4 = lane_of(piece, k4), p5 = lane_of(piece, k5), p6 = lane_of(piece, k6);
    jumps = __ballot(branch || logic || walk || range) != 0;
    if (branch) {
      put(p2 & 0xffff, OP_JMP_IF_FALSE, 0, base + 1, fuel, (p3 & 0xffff) + 1);
      put(p3 & 0xffff, OP_JMP, 0, base + (result == kStatementType ? 0 : 1), unsigned(x2 >> 16) & 255u, end);
    }
    if (logic) {
      put(p2 & 0xffff, kind == TK_OR ? OP_JMP_IF_TRUE : OP_JMP_IF_FALSE, 0, base + 1, fuel, end + 3);
      put(end, OP_NOT, 0, base + 1, fuel, 0);
      put(end + 1, OP_NOT, 0, base + 1, fuel, 0);
      put(end + 2, OP_JMP, 0, base + 1, fuel, end + 4);
      put(end + 3, OP_PUSH_CONST, 0, base, fuel, end_pool);
      put_value(end_pool, 0, TAG_BOOL, kind == TK_OR);
    }
    if (let) put(p2 & 0xffff, OP_STORE, 0, base + 1, fuel, slot);
    if (assign) put(end, OP_STORE, 0, base + 1, fuel, user);
    if (ret) put(end, OP_RETURN, 0, base + 1, fuel, 0);
    if (range) {
      const int p = p2 & 0xffff, q = p2 >> 16, count = sums[(depth_live + 1) & 63];
      put(p, OP_STORE, 0, base + 1, 1, slot);
      put(p + 1, OP_LOAD, 0, base, 1, slot);
      put(p + 2, OP_CALL_BUILTIN, 1, base + 1, 1, B_IS_INT);
      put(p + 3, OP_JMP_IF_FALSE, 0, base + 1, 1, p + 8);
      put(p + 4, OP_LOAD, 0, base, 1, slot);
      put(p + 5, OP_PUSH_CONST, 0, base + 1, 1, q);
      put(p + 6, OP_LT, 0, base + 2, 1, 0);
      put(p + 7, OP_JMP_IF_FALSE, 0, base + 1, 1, p + 10);
      put(p + 8, OP_PUSH_CONST, 0, base, 1, q + 1);
      put(p + 9, OP_NEG, 1, base + 1, 1, 0);
      put(p + 10, OP_PUSH_CONST, 0, base, 1, q + 2);
      put(p + 11, OP_STORE, 0, base + 1, 1, count);
      put(p + 12, OP_LOAD, kRangeTest, base, 1, count);
      put(p + 13, OP_LOAD, 0, base + 1, 1, slot);
      put(p + 14, OP_LT, 0, base + 2, 1, 0);
      put(p + 15, OP_JMP_IF_FALSE, 0, base + 1, 1, end + 5);
      put(p + 16, OP_LOAD, 0, base, 1, count);
      put(p + 17, OP_STORE, 0, base + 1, 1, user);
      put(end, OP_LOAD, kRangeNext, base, 1, count);
      put(end + 1, OP_PUSH_CONST, 0, base + 1, 1, q + 3);
      put(end + 2, OP_ADD, 0, base + 2, 1, 0);
      put(end + 3, OP_STORE, 0, base + 1, 1, count);
      put(end + 4, OP_JMP, 0, base, 1, p + 12);
      put_value(q, 0, TAG_INT, 0);
      put_value(q + 1, 0, TAG_BOOL, 1);
      put_value(q + 2, 0, TAG_INT, 0);
      put_value(q + 3, 1, TAG_INT, 0);
    }
    if (walk) {
      const auto temp = [&](int k) { return sums[(depth_live + k) & 63]; };
      const int xs = temp(0), from = temp(1), begin = temp(2), limit = temp(3), length = temp(4), counter = temp(5), element = temp(6),
                number = temp(7), state = temp(8);
      put(p2 & 0xffff, OP_STORE, 0, base + 1, 1, xs);
      if (ranged) {
        put(p3 & 0xffff, OP_STORE, 0, base + 1, 1, from);
        put(p4 & 0xffff, OP_STORE, 0, base + 1, 1, begin);
      }
      const int checks = ranged ? p5 : p3, ready = ranged ? p6 : p4;
      int to = checks & 0xffff, q = checks >> 16;
      put(to++, OP_STORE, 0, base + 1, 1, ranged ? limit : from);
      const auto check = [&](int v) {
        put(to++, OP_LOAD, 0, base, 1, v);
        put(to++, OP_CHECK_INT, 0, base + 1, 1, 0);
        put(to++, OP_STORE, 0, base + 1, 1, v);
      };
      check(from);
      if (ranged) {
        check(begin);
        check(limit);
      }
      put(to++, OP_LOAD, 0, base, 1, xs);
      put(to++, OP_CALL_BUILTIN, 1, base + 1, 1, B_LEN);
      put(to++, OP_STORE, 0, base + 1, 1, length);
      if (ranged) {
        for (int k = 0; k < 2; ++k) {
          const int v = k ? limit : begin;
          put(to, OP_LOAD, 0, base, 1, v);
          put(to + 1, OP_PUSH_CONST, 0, base + 1, 1, q);
          put(to + 2, OP_LT, 0, base + 2, 1, 0);
          put(to + 3, OP_JMP_IF_FALSE, 0, base + 1, 1, to + 7);
          put(to + 4, OP_PUSH_CONST, 0, base, 1, q + 1);
          put(to + 5, OP_STORE, 0, base + 1, 1, v);
          put(to + 6, OP_JMP, 0, base, 1, to + 13);
          put(to + 7, OP_LOAD, 0, base, 1, v);
          put(to + 8, OP_LOAD, 0, base + 1, 1, length);
          put(to + 9, OP_GT, 0, base + 2, 1, 0);
          put(to + 10, OP_JMP_IF_FALSE, 0, base + 1, 1, to + 13);
          put(to + 11, OP_LOAD, 0, base, 1, length);
          put(to + 12, OP_STORE, 0, base + 1, 1, v);
          put_value(q, 0, TAG_INT, 0);
          put_value(q + 1, 0, TAG_INT, 0);
          to += 13;
          q += 2;
        }
      } else {
        put(to++, OP_PUSH_CONST, 0, base, 1, q);
        put(to++, OP_STORE, 0, base + 1, 1, begin);
        put(to++, OP_LOAD, 0, base, 1, length);
        put(to++, OP_STORE, 0, base + 1, 1, limit);
        put_value(q, 0, TAG_INT, 0);
      }
      to = ready & 0xffff;
      put(to++, OP_STORE, 0, base + 1, 1, state);
      put(to++, OP_LOAD, 0, base, 1, reverse ? limit : begin);
      if (reverse) {
        put(to++, OP_PUSH_CONST, 0, base + 1, 1, ready >> 16);
        put(to++, OP_SUB, 0, base + 2, 1, 0);
        put_value(ready >> 16, 1, TAG_INT, 0);
      }
      put(to++, OP_STORE, 0, base + 1, 1, counter);
      const int head = to, way = reverse ? 2 : 1;
      put(head, OP_LOAD, kWalkTest | way, base, 1, counter);
      put(head + 1, OP_LOAD, 0, base + 1, 1, reverse ? begin : limit);
      put(head + 2, reverse ? OP_GE : OP_LT, 0, base + 2, 1, 0);
      put(head + 3, OP_JMP_IF_FALSE, 0, base + 1, 1, end + 6);
      put(head + 4, OP_LOAD, 0, base, 1, xs);
      put(head + 5, OP_LOAD, 0, base + 1, 1, counter);
      put(head + 6, OP_CALL_BUILTIN, 2, base + 2, 1, B_INDEX);
      put(head + 7, OP_STORE, 0, base + 1, 1, element);
      put(head + 8, OP_LOAD, 0, base, 1, from);
      put(head + 9, OP_LOAD, 0, base + 1, 1, counter);
      put(head + 10, OP_ADD, 0, base + 2, 1, 0);
      put(head + 11, OP_STORE, 0, base + 1, 1, number);
      put(end, OP_STORE, kWalkNext | way, base + 1, 1, state);
      put(end + 1, OP_LOAD, 0, base, 1, counter);
      put(end + 2, OP_PUSH_CONST, 0, base + 1, 1, end_pool);
      put(end + 3, reverse ? OP_SUB : OP_ADD, 0, base + 2, 1, 0);
      put(end + 4, OP_STORE, 0, base + 1, 1, counter);
      put(end + 5, OP_JMP, 0, base, 1, head);
      put(end + 6, OP_LOAD, 0, base, 1, state);
      put_value(end_pool, 1, TAG_INT, 0);
    }
  }
  if (!statement && lane == 0) put(words - 1, OP_RETURN, 0, 1, 1, 0);
  lanes_meet();
  const bool straight = __ballot(live && (!fast || branch || logic || walk || bind || let)) == 0 && !statement;
  const bool few = local_count <= kFastInputs;
  const int value = statement ? returned : root;
  out = LowerResult{ST_OK, words, entries, bound, value, jumps, 0, locals, 0};
  out.fast = few && straight && fast_type(root) && bound <= kFastStack && words <= kFastCode && entries <= kFastPool;
  out.loop = few && !out.fast && __ballot(live && !typed) == 0 && fast_type(value) && bound <= kLoopStack && words <= kLoopCode &&
             entries <= kLoopPool && locals - local_count <= kLoopLocals;
  return true;
}

}  // namespace gagp_amd
