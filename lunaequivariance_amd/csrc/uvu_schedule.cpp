// Path specification parsing and launch scheduling for the UVU convolution.
//
// Paths that read the same input block (x_off, d1, channels) form a group, so
// a wave gathers each source row's block once per edge and keeps every output
// block of the group in registers.  Output blocks written by more than one
// group are separated into phases (one launch each) and accumulated, which
// reproduces the reference's summation of aliased outputs
// (src/lunatp/uvu_conv/kernels/utils.py:135-152) without atomics.
#include <algorithm>
#include <map>
#include <tuple>
#include <cstdio>
#include <cstdlib>
#include <sstream>
#include <stdexcept>

#include "uvu_plan.h"

namespace luna {

namespace {

constexpr int kWave = 64;
// Upper bound on live output accumulators per lane for one group.
// Accumulator budget per wave, in 32-bit registers.
constexpr int kAccumulatorRegisters = 64;
// fp64 backward groups holding more seeds than this are split in two.
constexpr int kSplitSeeds = 24;

int read_int(std::istringstream& in, const char* what) {
  long long value;
  if (!(in >> value)) fail(std::string("spec: expected integer for ") + what);
  if (value < -1 || value > (1LL << 31) - 1) fail(std::string("spec: value out of range for ") + what);
  return static_cast<int>(value);
}

double read_real(std::istringstream& in) {
  std::string token;
  if (!(in >> token)) fail("spec: expected coefficient");
  char* end = nullptr;
  double value = std::strtod(token.c_str(), &end);
  if (end == token.c_str() || *end != '\0') fail("spec: bad coefficient '" + token + "'");
  return value;
}

bool ranges_overlap(long a0, long a1, long b0, long b1) { return a0 < b1 && b0 < a1; }

}  // namespace

Spec parse_spec(const std::string& text) {
  std::istringstream in(text);
  std::string magic;
  in >> magic;
  if (magic != "LUNAUVU1" && magic != "LUNAUVU2") fail("spec: missing LUNAUVU1 header");
  Spec s;
  s.dtype_bits = read_int(in, "dtype");
  if (s.dtype_bits != 32 && s.dtype_bits != 64) fail("spec: dtype must be 32 or 64");
  s.in1 = read_int(in, "in1");
  s.in2 = read_int(in, "in2");
  s.out = read_int(in, "out");
  s.wnum = read_int(in, "weight_numel");
  int npaths = read_int(in, "npaths");
  s.l0_dim = read_int(in, "l0_dim");
  // LUNAUVU2 adds a flag: the weight operand is one row shared by every edge.
  if (magic == "LUNAUVU2") s.w_broadcast = read_int(in, "w_broadcast") != 0;
  if (npaths <= 0) fail("spec: UVU convolution needs at least one path");
  for (int p = 0; p < npaths; ++p) {
    Path q;
    q.x_off = read_int(in, "x_off");
    q.y_off = read_int(in, "y_off");
    q.out_off = read_int(in, "out_off");
    q.w_off = read_int(in, "w_off");
    q.w_stride = read_int(in, "w_stride");
    q.channels = read_int(in, "channels");
    q.d1 = read_int(in, "d1");
    q.d2 = read_int(in, "d2");
    q.d3 = read_int(in, "d3");
    q.l0_col = read_int(in, "l0_col");
    int nterms = read_int(in, "nterms");
    if (q.channels <= 0) fail("spec: UVU convolution requires positive channels for every path");
    if (q.d1 <= 0 || q.d2 <= 0 || q.d3 <= 0 || q.w_stride <= 0) fail("spec: bad path dimensions");
    if ((long)q.x_off + (long)q.channels * q.d1 > s.in1 || q.x_off < 0)
      fail("spec: input block outside in1_dim");
    if (q.y_off < 0 || q.y_off + q.d2 > s.in2) fail("spec: edge block outside in2_dim");
    if (q.out_off < 0 || (long)q.out_off + (long)q.channels * q.d3 > s.out)
      fail("spec: output block outside out_dim");
    if (q.w_off < 0 || (long)q.w_off + (long)(q.channels - 1) * q.w_stride >= s.wnum)
      fail("spec: weight block outside weight_numel");
    if (q.l0_col >= 0 && (q.d3 != 1 || q.l0_col + q.channels > s.l0_dim))
      fail("spec: l0 column outside l0_dim");
    for (int t = 0; t < nterms; ++t) {
      Term term;
      term.i = read_int(in, "i");
      term.j = read_int(in, "j");
      term.k = read_int(in, "k");
      term.c = read_real(in);
      if (term.i < 0 || term.i >= q.d1 || term.j < 0 || term.j >= q.d2 || term.k < 0 || term.k >= q.d3)
        fail("spec: coefficient index outside the path's irreps");
      q.terms.push_back(term);
    }
    s.paths.push_back(std::move(q));
  }
  return s;
}

namespace {

// Channels per chunk.  Up to 32 channels would leave half of a wave's lanes
// idle or more, so such chunks are a power of two wide and a wave takes several
// edges at once (at most eight).  Wider blocks keep whole waves: 96 channels as
// three chunks of 32 took 347 us instead of 242 (lmax 2, 40,000 nodes of two
// edges), 202 instead of 190 us (3,000 nodes of 50).
int chunk_width(int channels, bool one_edge) {
  if (channels > 32 || one_edge) return kWave;
  int w = 8;
  while (w < channels) w *= 2;
  return w;
}

// Split the paths sharing one input block into groups whose output blocks fit
// the accumulator budget.  Paths writing the same output block stay together.
std::vector<Group> make_groups(const Spec& spec, int budget, bool one_edge) {
  std::map<std::tuple<int, int, int>, std::vector<int>> by_input;
  std::vector<std::tuple<int, int, int>> key_order;
  for (int p = 0; p < (int)spec.paths.size(); ++p) {
    const Path& q = spec.paths[p];
    auto key = std::make_tuple(q.x_off, q.d1, q.channels);
    if (!by_input.count(key)) key_order.push_back(key);
    by_input[key].push_back(p);
  }
  std::vector<Group> groups;
  for (const auto& key : key_order) {
    const std::vector<int>& members = by_input[key];
    // Output blocks of this input block, in first-use order.
    std::vector<std::pair<int, int>> blocks;
    std::map<std::pair<int, int>, std::vector<int>> block_paths;
    for (int p : members) {
      auto b = std::make_pair(spec.paths[p].out_off, spec.paths[p].d3);
      if (!block_paths.count(b)) blocks.push_back(b);
      block_paths[b].push_back(p);
    }
    // First-fit by decreasing width.
    std::vector<std::pair<int, int>> sorted = blocks;
    std::stable_sort(sorted.begin(), sorted.end(),
                     [](const auto& a, const auto& b) { return a.second > b.second; });
    std::vector<std::pair<int, std::vector<std::pair<int, int>>>> bins;
    for (const auto& b : sorted) {
      bool placed = false;
      for (auto& bin : bins) {
        if (bin.first + b.second <= budget) {
          bin.first += b.second;
          bin.second.push_back(b);
          placed = true;
          break;
        }
      }
      if (!placed) bins.push_back({b.second, {b}});
    }
    for (auto& bin : bins) {
      Group g;
      g.x_off = std::get<0>(key);
      g.d1 = std::get<1>(key);
      g.channels = std::get<2>(key);
      g.cw = chunk_width(g.channels, one_edge);
      g.chunks = (g.channels + g.cw - 1) / g.cw;
      // Keep the original block order inside the bin.
      for (const auto& b : blocks) {
        if (std::find(bin.second.begin(), bin.second.end(), b) == bin.second.end()) continue;
        int index = (int)g.blocks.size();
        g.blocks.push_back({b.first, b.second, false});
        for (int p : block_paths[b]) {
          g.paths.push_back(p);
          g.path_block.push_back(index);
        }
      }
      groups.push_back(std::move(g));
    }
  }
  return groups;
}

// Greedy phase assignment: groups in one phase touch disjoint ranges.
template <typename RangesOf>
int assign_phases(std::vector<Group>& groups, RangesOf ranges_of) {
  std::vector<std::vector<std::pair<long, long>>> phase_ranges;
  for (Group& g : groups) {
    auto mine = ranges_of(g);
    int phase = 0;
    for (;; ++phase) {
      if (phase == (int)phase_ranges.size()) phase_ranges.emplace_back();
      bool clash = false;
      for (const auto& r : mine)
        for (const auto& o : phase_ranges[phase])
          if (ranges_overlap(r.first, r.second, o.first, o.second)) clash = true;
      if (!clash) break;
    }
    g.phase = phase;
    for (const auto& r : mine) phase_ranges[phase].push_back(r);
  }
  return (int)phase_ranges.size();
}

}  // namespace

static bool compute_message_component_major(const Plan& plan) {
  if (const char* e = std::getenv("LUNAEQ_AMD_MSGCM"))
    if (std::atoi(e) == 0) return false;
  for (size_t a = 0; a < plan.bwd_groups.size(); ++a) {
    for (size_t b = a + 1; b < plan.bwd_groups.size(); ++b) {
      const Group& p = plan.bwd_groups[a];
      const Group& q = plan.bwd_groups[b];
      const bool same = p.x_off == q.x_off && p.d1 == q.d1 && p.channels == q.channels;
      if (!same && ranges_overlap(p.x_off, p.x_off + (long)p.channels * p.d1, q.x_off,
                                  q.x_off + (long)q.channels * q.d1))
        return false;
    }
  }
  return true;
}

static int compute_gather_vector_width(const Plan& plan) {
  const Spec& spec = plan.spec;
  int vec = 16 / (spec.dtype_bits / 8);
  const bool cmajor = plan.msg_cmajor;
  bool aligned = spec.in1 % vec == 0;
  for (const Group& g : plan.bwd_groups) {
    const long end = g.x_off + (long)g.channels * g.d1;
    aligned = aligned && g.x_off % vec == 0 && end % vec == 0;
    // Component-major: the values of one vector must share their component.
    if (cmajor) aligned = aligned && g.channels % vec == 0;
  }
  return aligned ? vec : 1;
}

bool message_component_major(const Plan& plan) { return plan.msg_cmajor; }
int gather_vector_width(const Plan& plan) { return plan.gather_vec; }
int gather_columns(const Plan& plan) {
  return std::max(1, std::min(256, (plan.spec.in1 + plan.gather_vec - 1) / plan.gather_vec));
}
int gather_teams(const Plan& plan) {
  const int row = (plan.spec.in1 + plan.gather_vec - 1) / plan.gather_vec;
  return row > 128 || plan.one_edge ? 1 : std::min(16, 256 / gather_columns(plan));
}

void build_schedule(Plan& plan) {
  const Spec& spec = plan.spec;

  // ---- forward ----
  // The forward splits an input block's paths when their accumulators exceed
  // the register budget (halved for fp64, whose values take two registers);
  // the backward keeps one group per input block, because split groups would
  // have to accumulate their gx messages.
  int acc_regs = kAccumulatorRegisters;
  if (const char* e = std::getenv("LUNAEQ_AMD_FACC")) acc_regs = std::max(8, std::atoi(e));
  plan.fwd_groups = make_groups(spec, acc_regs / (spec.dtype_bits / 32), plan.one_edge);
  auto out_ranges = [](const Group& g) {
    std::vector<std::pair<long, long>> r;
    for (const auto& b : g.blocks) r.push_back({b.out_off, b.out_off + (long)g.channels * b.d3});
    return r;
  };
  // Any overlap between blocks of different groups (or overlapping distinct
  // blocks) means outputs are summed: zero-fill and accumulate everywhere.
  std::vector<std::pair<long, long>> all;
  for (const Group& g : plan.fwd_groups)
    for (const auto& r : out_ranges(g)) all.push_back(r);
  bool collision = false;
  for (size_t a = 0; a < all.size(); ++a)
    for (size_t b = a + 1; b < all.size(); ++b)
      if (ranges_overlap(all[a].first, all[a].second, all[b].first, all[b].second)) collision = true;
  std::vector<std::pair<long, long>> merged = all;
  std::sort(merged.begin(), merged.end());
  long covered = 0;
  bool holes = false;
  for (const auto& r : merged) {
    if (r.first > covered) holes = true;
    covered = std::max(covered, r.second);
  }
  if (covered < spec.out) holes = true;
  plan.fwd_needs_zero = collision || holes;
  for (Group& g : plan.fwd_groups)
    for (auto& b : g.blocks) b.accumulate = collision;
  plan.fwd_phases = assign_phases(plan.fwd_groups, out_ranges);
  plan.phase_slots.assign(plan.fwd_phases, 0);
  // Two waves per workgroup: the two 64-channel chunks of a 128-channel group
  // gather adjacent halves of the same x rows together.  (All slots of a node
  // in one workgroup, or the slots of a node on consecutive workgroups, keep
  // every input block's gathers live at once and measured slower.)
  int limit = 2;
  if (const char* e = std::getenv("LUNAEQ_AMD_WG")) limit = std::max(0, std::min(16, std::atoi(e)));
  bool sibling_pairs = true;
  if (const char* e = std::getenv("LUNAEQ_AMD_FWDPAIR")) sibling_pairs = std::atoi(e) != 0;
  for (int phase = 0; phase < plan.fwd_phases; ++phase) {
    std::vector<Group*> members;
    for (Group& g : plan.fwd_groups)
      if (g.phase == phase) members.push_back(&g);
    auto key = [](const Group* g) { return std::make_tuple(g->x_off, g->d1, g->channels); };
    // An input block split over several groups (its accumulators exceed the
    // budget) is gathered by each of them.  Two such sibling groups of two
    // chunks each run as the four waves of one workgroup, so that their
    // gathers of the same x rows arrive together and the second is served by
    // the first's cache lines instead of a second trip to the fabric.
    bool siblings = false, two_chunks = true;
    for (size_t a = 0; a < members.size(); ++a) {
      two_chunks = two_chunks && members[a]->chunks == 2;
      for (size_t b = a + 1; b < members.size(); ++b) siblings = siblings || key(members[a]) == key(members[b]);
    }
    int slot = 0;
    if (sibling_pairs && siblings && two_chunks && limit == 2) {
      std::vector<bool> placed(members.size(), false);
      std::vector<Group*> singles;
      for (size_t a = 0; a < members.size(); ++a) {
        if (placed[a]) continue;
        placed[a] = true;
        size_t b = a + 1;
        while (b < members.size() && (placed[b] || key(members[b]) != key(members[a]))) ++b;
        if (b == members.size()) {
          singles.push_back(members[a]);
          continue;
        }
        placed[b] = true;
        members[a]->slot_base = slot;
        members[b]->slot_base = slot + 2;
        slot += 4;
      }
      for (Group* g : singles) {
        g->slot_base = slot;
        slot += 2;
      }
      slot += slot % 4;  // the last workgroup's idle half, if any
      plan.fwd_block_waves.push_back(4);
    } else {
      for (Group* g : members) {
        g->slot_base = slot;
        slot += g->chunks;
      }
      plan.fwd_block_waves.push_back(std::min(slot, limit));
    }
    plan.phase_slots[phase] = slot;
  }
  // The kernels test slots in group order.
  std::stable_sort(plan.fwd_groups.begin(), plan.fwd_groups.end(), [](const Group& a, const Group& b) {
    return std::make_pair(a.phase, a.slot_base) < std::make_pair(b.phase, b.slot_base);
  });
  for (int s : plan.phase_slots)
    if (s > 65535) fail("too many channel chunks for one launch");

  // ---- backward ----
  plan.bwd_groups = make_groups(spec, kAccumulatorRegisters, plan.one_edge);
  auto in_ranges = [](const Group& g) {
    return std::vector<std::pair<long, long>>{{g.x_off, g.x_off + (long)g.channels * g.d1}};
  };
  std::vector<std::pair<long, long>> xs;
  for (const Group& g : plan.bwd_groups) xs.push_back(in_ranges(g)[0]);
  bool x_collision = false;
  for (size_t a = 0; a < xs.size(); ++a)
    for (size_t b = a + 1; b < xs.size(); ++b)
      if (ranges_overlap(xs[a].first, xs[a].second, xs[b].first, xs[b].second)) x_collision = true;
  std::sort(xs.begin(), xs.end());
  covered = 0;
  bool x_holes = false;
  for (const auto& r : xs) {
    if (r.first > covered) x_holes = true;
    covered = std::max(covered, r.second);
  }
  if (covered < spec.in1) x_holes = true;
  plan.bwd_gx_needs_zero = x_collision || x_holes;
  for (Group& g : plan.bwd_groups) g.gx_accumulate = x_collision;
  int bwd_phases = assign_phases(plan.bwd_groups, in_ranges);
  // fp64 groups with many seeds run as two path subsets (half the seeds in
  // registers per wave, which doubles or triples the waves that fit).
  int split_seeds = spec.dtype_bits == 64 ? kSplitSeeds : 0;
  if (const char* e = std::getenv("LUNAEQ_AMD_BSPLIT")) split_seeds = std::atoi(e);
  bool any_split = false;
  for (Group& g : plan.bwd_groups) {
    int seeds = 0;
    for (const auto& b : g.blocks) seeds += b.d3;
    g.path_subset.assign(g.paths.size(), 0);
    if (split_seeds <= 0 || seeds <= split_seeds || g.paths.size() < 2) continue;
    // Greedy balance of per-edge work: terms plus the seeds each path holds.
    std::vector<int> order(g.paths.size());
    for (size_t n = 0; n < order.size(); ++n) order[n] = (int)n;
    auto cost = [&](int n) {
      const Path& q = spec.paths[g.paths[n]];
      return (long)q.terms.size() + 2L * q.d3 + q.d1 + q.d2;
    };
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return cost(a) > cost(b); });
    long load[2] = {0, 0};
    for (int n : order) {
      const int s = load[1] < load[0] ? 1 : 0;
      g.path_subset[n] = s;
      load[s] += cost(n);
    }
    g.subsets = 2;
    any_split = true;
  }
  // Backward phases reuse Group::phase; slots are numbered per phase (a split
  // group starts on an even slot, so its waves pair up in one workgroup), and
  // gy partial slots are global.
  std::vector<int> slots(bwd_phases, 0);
  for (Group& g : plan.bwd_groups) {
    if (g.subsets > 1 && slots[g.phase] % 2) ++slots[g.phase];
    g.slot_base = slots[g.phase];
    slots[g.phase] += g.chunks * g.subsets;
  }
  plan.bwd_phases = bwd_phases;
  plan.bwd_phase_slots = slots;
  // The backward uses the forward's two waves per workgroup.
  int bwd_limit = limit;
  if (const char* e = std::getenv("LUNAEQ_AMD_BWG")) bwd_limit = std::max(0, std::min(16, std::atoi(e)));
  for (int s : plan.bwd_phase_slots) plan.bwd_block_waves.push_back(any_split ? 2 : std::min(s, bwd_limit));
  // A group whose two chunks are the two waves of one workgroup adds their gy
  // partials through LDS and writes one slot (half the partial traffic).
  bool pair = true;
  if (const char* e = std::getenv("LUNAEQ_AMD_PAIRGY")) pair = std::atoi(e) != 0;
  int parts = 0;
  for (Group& g : plan.bwd_groups) {
    g.pair_partials = pair && g.subsets == 1 && g.chunks == 2 && g.slot_base % 2 == 0 &&
                      plan.bwd_block_waves[g.phase] == 2;
    g.combine_subsets = pair && g.subsets == 2 && plan.bwd_block_waves[g.phase] == 2;
    g.gy_slot_base = parts;
    parts += g.pair_partials ? 1 : g.combine_subsets ? g.chunks : g.chunks * g.subsets;
  }
  plan.gy_parts = parts;
  plan.msg_cmajor = compute_message_component_major(plan);
  plan.gather_vec = compute_gather_vector_width(plan);
  for (int s : slots)
    if (s > 65535) fail("too many channel chunks for one launch");
}

}  // namespace luna
