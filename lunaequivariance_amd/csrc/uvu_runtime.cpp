// C-ABI entry points of the UVU convolution: plan lifetime and launchers.
#include <algorithm>
#include <cstdio>
#include <cstring>
#include <initializer_list>

#include "../../include/lunaeq_amd.h"
#include "uvu_plan.h"

using namespace luna;

namespace {

std::string source_for(const Plan& plan, const std::string& variant) {
  // Variant names: fwd<env><l0>, fws<env><l0> (split over waves),
  // bwd<env><gl0><gw><msg><part>, and row-wise rwf<shared> and
  // rwb<shared><gw><msg><part>, each flag '0' or '1'.
  auto flag = [&](size_t i) { return variant.size() > i && variant[i] == '1'; };
  if (variant.compare(0, 3, "fwd") == 0) return emit_forward(plan, flag(3), flag(4), false);
  if (variant.compare(0, 3, "fws") == 0) return emit_forward(plan, flag(3), flag(4), true);
  if (variant.compare(0, 3, "rwf") == 0) return emit_rows_forward(plan, flag(3));
  if (variant.compare(0, 3, "rwb") == 0) return emit_rows_backward(plan, flag(3), flag(4), flag(5), flag(6));
  return emit_backward(plan, flag(3), flag(4), flag(5), flag(6), flag(7));
}

// Kernel `name` of variant <kind><flags...>; at most five flags.
enum Kind { kFwd, kFws, kBwd, kRwf, kRwb };
template <typename N>
hipFunction_t kernel_of(Plan& plan, Kind kind, std::initializer_list<bool> flags, int which, N name) {
  uint64_t code = (uint64_t)which << 8 | (uint64_t)kind << 5;
  int bit = 0;
  for (bool f : flags) code |= (uint64_t)f << bit++;
  return plan.kernels.function(
      code,
      [&] {
        static const char* const names[] = {"fwd", "fws", "bwd", "rwf", "rwb"};
        std::string v = names[kind];
        for (bool f : flags) v += f ? '1' : '0';
        return v;
      },
      [&](const std::string& v) { return source_for(plan, v); }, name);
}

// Workspace layout: gy/genv partials, then the per-edge gx messages.
size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }
size_t part_bytes(const Plan& p, int64_t num_edges) {
  return align256((size_t)p.gy_parts * (size_t)num_edges * (size_t)(p.spec.in2 + 1) * (p.spec.dtype_bits / 8));
}
size_t msg_bytes(const Plan& p, int64_t num_edges) {
  return align256((size_t)num_edges * (size_t)p.spec.in1 * (p.spec.dtype_bits / 8));
}

// waves == 0: one wave per workgroup on a 1-D grid, slot fastest.
dim3 grid_for(int64_t nodes, int slots, int waves) {
  if (waves == 0) {
    if (nodes * slots > 0x7fffffffLL) fail("launch grid exceeds 2^31 workgroups");
    return dim3((unsigned)(nodes * slots));
  }
  return dim3((unsigned)nodes, (unsigned)((slots + waves - 1) / waves));
}

// Pieces a node's edges are cut into when the graph alone gives few waves:
// doubled (up to 8) until the launch holds `target` waves, while each piece
// keeps at least four iterations of the edge loop (a piece pays for the node's
// seeds or output again).  Targets: 4,096 waves (four per SIMD) for the
// forward, 8,192 for the backward.  150 nodes of 128 channels, lmax 3: forward
// 83 us whole, 46 / 44 / 45 us for targets of 2,048 / 4,096 / 8,192, backward
// 133 us, 107 / 90 / 86 us; 1,000 nodes of 32 channels, lmax 2: forward 31, 31
// and (8,192) 34 us, backward 68, 66, 64 us.
int edge_split(const std::vector<Group>& groups, int phase, int64_t waves, int64_t nodes, int64_t edges, int64_t target) {
  int at_once = 1;
  for (const Group& g : groups)
    if (g.phase == phase) at_once = std::max(at_once, 64 / g.cw);
  int split = 1;
  while (split < 8 && waves * split < target && edges >= nodes * at_once * split * 8) split *= 2;
  return split;
}
constexpr int64_t kForwardWaves = 4096, kBackwardWaves = 8192;

// Workgroups along the rows of a row-wise product: every wave loops over rows,
// with the next row's operands in flight, a shared weight row in registers and,
// in its gradient's kernel (`sum_gw`), the sums over the wave's rows too.  That
// one keeps to 8,192 waves, each of which writes a partial row: 64 channels,
// lmax 2, 50,000 rows, shared weights, forward + backward 341 us, 356 with
// 32,768 waves, 475 with a wave per row.  The others take a wave per row up to 2^20
// (forward 128 us with 8,192 waves, 121 so; a weight row per row: forward 170 and
// 149 us, forward + backward 409 and 388 us).
constexpr int64_t kGradientWaves = 8192, kRowWaves = 1 << 20;
unsigned row_blocks(const std::vector<Group>& groups, int phase, int slots, int64_t rows, bool sum_gw) {
  int at_once = 64;
  for (const Group& g : groups)
    if (g.phase == phase) at_once = std::min(at_once, 64 / g.cw);
  const int64_t waves = sum_gw ? kGradientWaves : kRowWaves;
  return (unsigned)std::max<int64_t>(1, std::min((rows + at_once - 1) / at_once, waves / std::max(slots, 1)));
}
// Partials of the shared weight row's gradient: a row per workgroup of the
// largest launch (zeros where a launch has no rows left).
int64_t row_gw_blocks(const Plan& p, int64_t rows) {
  unsigned n = 1;
  for (int phase = 0; phase < p.bwd_phases; ++phase)
    n = std::max(n, row_blocks(p.bwd_groups, phase, p.bwd_phase_slots[phase], rows, true));
  return n;
}
size_t row_gw_bytes(const Plan& p, int64_t rows) {
  return align256((size_t)row_gw_blocks(p, rows) * (size_t)p.spec.wnum * (p.spec.dtype_bits / 8));
}

void check_sizes(const Plan& plan, int64_t num_nodes, int64_t num_edges) {
  if (num_nodes < 0 || num_edges < 0) fail("negative problem size");
  if (num_nodes > 0x7fffffffLL) fail("graph node count exceeds signed int32 capacity");
  if (plan.edge_index_bits == 32 && num_edges > 0x7fffffffLL)
    fail("a graph of 2^31 or more edges needs a plan with 64-bit edge offsets (luna_uvu_plan_create_ex)");
}

}  // namespace

namespace luna {

// Size of the backward workspace (gy partials, then gx messages).
size_t uvu_bwd_workspace_bytes(const Plan& plan, int64_t num_edges) {
  return part_bytes(plan, num_edges) + msg_bytes(plan, num_edges);
}

void uvu_conv_bwd(Plan& plan, const void* x, const void* y, const void* w, const void* env, const void* g,
                  const void* gl0, const int32_t* src, const void* dst_rowptr, const int32_t* node_order,
                  const void* src_rowptr, const void* edge_ids_by_src, void* gx, void* gy, void* gw,
                  void* genv, void* workspace, size_t workspace_bytes, int64_t num_nodes, int64_t num_edges,
                  LunaStream stream) {
  check_sizes(plan, num_nodes, num_edges);
    if (num_nodes == 0) return;
    if (!x || !g || !dst_rowptr || !node_order || !src_rowptr) fail("luna_uvu_conv_bwd: null tensor");
    if (num_edges > 0 && (!y || !w || !src || !edge_ids_by_src)) fail("luna_uvu_conv_bwd: null edge tensor");
    if (gl0 && plan.spec.l0_dim == 0) gl0 = nullptr;
    if (!env) genv = nullptr;
    if (gw && plan.spec.w_broadcast) fail("luna_uvu_conv_bwd: a broadcast weight row has no per-edge gradient");
    int64_t E = num_edges;
    const bool want_parts = (gy || genv) && E > 0;
    const bool want_msg = gx && E > 0;
    const size_t pbytes = part_bytes(plan, E), mbytes = msg_bytes(plan, E);
    if ((want_parts || want_msg) && (!workspace || workspace_bytes < pbytes + mbytes))
      fail("luna_uvu_conv_bwd: workspace too small");
    void* part = want_parts ? workspace : nullptr;
    void* msg = want_msg ? (void*)((char*)workspace + pbytes) : nullptr;
    auto kernel = [&](int which, const char* name, int phase) {
      return kernel_of(plan, kBwd, {env != nullptr, gl0 != nullptr, gw != nullptr, want_msg, want_parts}, which,
                       [&] { return phase < 0 ? std::string(name) : name + std::to_string(phase); });
    };
    hipStream_t s = (hipStream_t)stream;
    if (want_msg && plan.bwd_gx_needs_zero) {
      int64_t n = E * (int64_t)plan.spec.in1;
      if ((n + 255) / 256 > 0xffffffffLL) fail("luna_uvu_conv_bwd: message fill exceeds the launch grid");
      void* args[] = {&msg, &n};
      launch("uvu_fill", kernel(0, "luna_uvu_fill", -1), dim3((unsigned)((n + 255) / 256)), dim3(256), s,
             args);
    }
    if (E > 0 && (gw || want_parts || want_msg)) {
      for (int phase = 0; phase < plan.bwd_phases; ++phase) {
        hipFunction_t f = kernel(3 + phase, "luna_uvu_bwd_p", phase);
        void* args[] = {&x, &y, &w, &env, &g, &gl0, &src, &dst_rowptr, &node_order, &gw, &msg, &part, &E};
        dim3 grid = grid_for(num_nodes, plan.bwd_phase_slots[phase], plan.bwd_block_waves[phase]);
        grid.z = edge_split(plan.bwd_groups, phase, num_nodes * plan.bwd_phase_slots[phase], num_nodes, E,
                            kBackwardWaves);
        launch("uvu_bwd_p" + std::to_string(phase), f, grid,
               dim3(64 * std::max(plan.bwd_block_waves[phase], 1)), s, args);
      }
    }
    if (want_parts) {
      void* args[] = {&part, &gy, &genv, &E};
      launch("uvu_bwd_reduce", kernel(1, "luna_uvu_bwd_reduce", -1), dim3((unsigned)((E + 255) / 256)),
             dim3(256), s, args);
    }
    if (gx) {
      // With no edges the gather still writes zeros (every source row is empty).
      void* args[] = {&msg, &src_rowptr, &edge_ids_by_src, &gx};
      const int vec = gather_vector_width(plan);
      const int64_t per_block = (int64_t)gather_columns(plan) * vec;
      launch("uvu_bwd_gather", kernel(2, "luna_uvu_bwd_gather", -1),
             dim3((unsigned)num_nodes, (unsigned)((plan.spec.in1 + per_block - 1) / per_block)),
             dim3(gather_columns(plan) * gather_teams(plan)), s, args);
    }
}

}  // namespace luna

extern "C" {

int luna_uvu_plan_create(const char* spec, const char* cache_dir, LunaUvuPlan** out) {
  return luna_uvu_plan_create_ex(spec, cache_dir, 32, out);
}

int luna_uvu_plan_create_ex(const char* spec, const char* cache_dir, int edge_index_bits, LunaUvuPlan** out) {
  return guard_call([&] {
    if (!spec || !out) fail("luna_uvu_plan_create: null argument");
    if (edge_index_bits != 32 && edge_index_bits != 64) fail("luna_uvu_plan_create_ex: edge_index_bits must be 32 or 64");
    auto holder = std::make_unique<LunaUvuPlan>();
    holder->plan.edge_index_bits = edge_index_bits;
    holder->plan.spec = parse_spec(spec);
    holder->plan.kernels.cache_dir = cache_dir ? cache_dir : "";
    holder->plan.kernels.tag = "uvu";
    build_schedule(holder->plan);
    int narrow = 64;
    for (const auto* groups : {&holder->plan.fwd_groups, &holder->plan.bwd_groups})
      for (const Group& g : *groups) narrow = std::min(narrow, g.cw);
    if (narrow < 64) {
      holder->sparse_degree = narrow == 32 ? 3 : 2;
      holder->sparse = std::make_unique<Plan>();
      Plan& one = *holder->sparse;
      one.edge_index_bits = edge_index_bits;
      one.spec = holder->plan.spec;
      one.kernels.cache_dir = holder->plan.kernels.cache_dir;
      one.kernels.tag = "uvu";
      one.one_edge = true;
      build_schedule(one);
      // One workspace size and one plan info hold for both.
      if (one.gy_parts != holder->plan.gy_parts || one.fwd_needs_zero != holder->plan.fwd_needs_zero ||
          one.bwd_gx_needs_zero != holder->plan.bwd_gx_needs_zero)
        holder->sparse.reset();
    }
    *out = holder.release();
  });
}

int luna_uvu_plan_destroy(LunaUvuPlan* plan) {
  return guard_call([&] { delete plan; });
}

int luna_uvu_plan_info(const LunaUvuPlan* plan, LunaUvuPlanInfo* info) {
  return guard_call([&] {
    if (!plan || !info) fail("luna_uvu_plan_info: null argument");
    const Plan& p = plan->plan;
    info->dtype_bits = p.spec.dtype_bits;
    info->in1_dim = p.spec.in1;
    info->in2_dim = p.spec.in2;
    info->out_dim = p.spec.out;
    info->weight_numel = p.spec.wnum;
    info->l0_dim = p.spec.l0_dim;
    info->num_paths = (int32_t)p.spec.paths.size();
    info->fwd_needs_zero = p.fwd_needs_zero;
    info->bwd_gx_needs_zero = p.bwd_gx_needs_zero;
    info->num_fwd_launches = p.fwd_phases;
    info->gy_parts = p.gy_parts;
  });
}

int luna_uvu_plan_precompile(LunaUvuPlan* plan) {
  return guard_call([&] {
    if (!plan) fail("luna_uvu_plan_precompile: null plan");
    for (const char* v : {"fwd00", "bwd00111"})
      plan->plan.kernels.code_for(v, [&] { return source_for(plan->plan, v); });
  });
}

int luna_uvu_plan_precompile_all(LunaUvuPlan* plan) {
  return guard_call([&] {
    if (!plan) fail("luna_uvu_plan_precompile_all: null plan");
    auto compile = [](Plan& p, std::initializer_list<const char*> variants) {
      for (const char* v : variants) p.kernels.code_for(v, [&] { return source_for(p, v); });
    };
    const bool own = !plan->plan.spec.w_broadcast;  // a broadcast weight row has no gradient
    if (own)
      compile(plan->plan, {"fwd00", "bwd00111", "fws00", "rwf0", "rwf1", "rwb0111", "rwb1111"});
    else
      compile(plan->plan, {"fwd00", "bwd00011", "fws00", "rwf1", "rwb1011"});
    if (plan->sparse) compile(*plan->sparse, {"fwd00", own ? "bwd00111" : "bwd00011"});
  });
}

int luna_uvu_conv_fwd(const LunaUvuPlan* cplan, const void* x, const void* y, const void* w,
                      const void* env, const int32_t* src, const void* dst_rowptr,
                      const int32_t* node_order, void* out, void* l0, int64_t num_nodes,
                      int64_t num_edges, LunaStream stream) {
  return guard_call([&] {
    if (!cplan) fail("luna_uvu_conv_fwd: null plan");
    Plan& plan = const_cast<LunaUvuPlan*>(cplan)->of(num_nodes, num_edges);
    check_sizes(plan, num_nodes, num_edges);
    if (num_nodes == 0) return;
    if (!x || !out || !dst_rowptr || !node_order) fail("luna_uvu_conv_fwd: null tensor");
    if (num_edges > 0 && (!y || !w || !src)) fail("luna_uvu_conv_fwd: null edge tensor");
    if (l0 && plan.spec.l0_dim == 0) l0 = nullptr;
    for (int phase = 0; phase < plan.fwd_phases; ++phase) {
      int split = edge_split(plan.fwd_groups, phase, num_nodes * plan.phase_slots[phase], num_nodes, num_edges,
                             kForwardWaves);
      const size_t wave_lds = split_forward_lds(plan, phase) * (plan.spec.dtype_bits / 8);
      while (split > 1 && split * wave_lds > 65536) split /= 2;
      hipFunction_t f = kernel_of(plan, split > 1 ? kFws : kFwd, {env != nullptr, l0 != nullptr}, phase,
                                  [&] { return "luna_uvu_fwd_p" + std::to_string(phase); });
      void* args[] = {&x, &y, &w, &env, &src, &dst_rowptr, &node_order, &out, &l0};
      if (split > 1) {
        launch("uvu_fwd_p" + std::to_string(phase), f, dim3((unsigned)num_nodes, (unsigned)plan.phase_slots[phase]),
               dim3(64 * split), (hipStream_t)stream, args,
               (unsigned)(split * wave_lds));
        continue;
      }
      launch("uvu_fwd_p" + std::to_string(phase), f,
             grid_for(num_nodes, plan.phase_slots[phase], plan.fwd_block_waves[phase]),
             dim3(64 * std::max(plan.fwd_block_waves[phase], 1)), (hipStream_t)stream, args);
    }
  });
}

int luna_uvu_conv_bwd_workspace(const LunaUvuPlan* plan, int64_t num_nodes, int64_t num_edges,
                                size_t* bytes) {
  return guard_call([&] {
    if (!plan || !bytes) fail("luna_uvu_conv_bwd_workspace: null argument");
    if (num_nodes < 0 || num_edges < 0) fail("negative problem size");
    *bytes = uvu_bwd_workspace_bytes(plan->plan, num_edges);
  });
}

int luna_uvu_conv_bwd(const LunaUvuPlan* cplan, const void* x, const void* y, const void* w,
                      const void* env, const void* g, const void* gl0, const int32_t* src,
                      const void* dst_rowptr, const int32_t* node_order, const void* src_rowptr,
                      const void* edge_ids_by_src, void* gx, void* gy, void* gw, void* genv,
                      void* workspace, size_t workspace_bytes, int64_t num_nodes, int64_t num_edges,
                      LunaStream stream) {
  return guard_call([&] {
    if (!cplan) fail("luna_uvu_conv_bwd: null plan");
    uvu_conv_bwd(const_cast<LunaUvuPlan*>(cplan)->of(num_nodes, num_edges), x, y, w, env, g, gl0, src, dst_rowptr,
                 node_order, src_rowptr, edge_ids_by_src, gx, gy, gw, genv, workspace, workspace_bytes, num_nodes,
                 num_edges, stream);
  });
}

int luna_uvu_rows_fwd(const LunaUvuPlan* cplan, const void* x, const void* y, const void* w, int shared_w, void* out,
                      int64_t rows, LunaStream stream) {
  return guard_call([&] {
    if (!cplan) fail("luna_uvu_rows_fwd: null plan");
    Plan& plan = const_cast<LunaUvuPlan*>(cplan)->plan;
    check_sizes(plan, rows, rows);
    if (rows == 0) return;
    if (!x || !y || !w || !out) fail("luna_uvu_rows_fwd: null tensor");
    const bool shared = shared_w || plan.spec.w_broadcast;
    for (int phase = 0; phase < plan.fwd_phases; ++phase) {
      hipFunction_t f = kernel_of(plan, kRwf, {shared}, phase,
                                  [&] { return "luna_uvu_rows_fwd_p" + std::to_string(phase); });
      const int waves = std::max(plan.fwd_block_waves[phase], 1), slots = plan.phase_slots[phase];
      void* args[] = {&x, &y, &w, &out, &rows};
      launch("uvu_rows_fwd", f, dim3(row_blocks(plan.fwd_groups, phase, slots, rows, false), (unsigned)((slots + waves - 1) / waves)),
             dim3(64 * waves), (hipStream_t)stream, args);
    }
  });
}

int luna_uvu_rows_bwd_workspace(const LunaUvuPlan* plan, int shared_w, int64_t rows, size_t* bytes) {
  return guard_call([&] {
    if (!plan || !bytes) fail("luna_uvu_rows_bwd_workspace: null argument");
    check_sizes(plan->plan, rows, rows);
    *bytes = part_bytes(plan->plan, rows) + (shared_w ? row_gw_bytes(plan->plan, rows) : 0);
  });
}

int luna_uvu_rows_bwd(const LunaUvuPlan* cplan, const void* x, const void* y, const void* w, int shared_w, const void* g,
                      void* gx, void* gy, void* gw, void* workspace, size_t workspace_bytes, int64_t rows,
                      LunaStream stream) {
  return guard_call([&] {
    if (!cplan) fail("luna_uvu_rows_bwd: null plan");
    Plan& plan = const_cast<LunaUvuPlan*>(cplan)->plan;
    check_sizes(plan, rows, rows);
    if (rows == 0) {
      if (gw && shared_w) fail("luna_uvu_rows_bwd: the gradient of a shared weight row needs at least one row");
      return;
    }
    if (!x || !y || !w || !g) fail("luna_uvu_rows_bwd: null tensor");
    if (gw && plan.spec.w_broadcast) fail("luna_uvu_rows_bwd: a broadcast weight row has no gradient");
    if (!gx && !gy && !gw) return;
    const bool shared = shared_w || plan.spec.w_broadcast, sum_gw = shared && gw;
    const size_t pbytes = part_bytes(plan, rows);
    if ((gy || sum_gw) && (!workspace || workspace_bytes < pbytes + (sum_gw ? row_gw_bytes(plan, rows) : 0)))
      fail("luna_uvu_rows_bwd: workspace too small");
    void* part = gy ? workspace : nullptr;
    void* gw_out = sum_gw ? (void*)((char*)workspace + pbytes) : gw;
    hipStream_t s = (hipStream_t)stream;
    auto kernel = [&](int which, const char* name, int phase) {
      return kernel_of(plan, kRwb, {shared, gw != nullptr, gx != nullptr, gy != nullptr}, which,
                       [&] { return phase < 0 ? std::string(name) : name + std::to_string(phase); });
    };
    if (gx && plan.bwd_gx_needs_zero) {
      int64_t n = rows * (int64_t)plan.spec.in1;
      if ((n + 255) / 256 > 0xffffffffLL) fail("luna_uvu_rows_bwd: gx fill exceeds the launch grid");
      void* args[] = {&gx, &n};
      launch("uvu_fill", kernel(0, "luna_uvu_fill", -1), dim3((unsigned)((n + 255) / 256)), dim3(256), s, args);
    }
    for (int phase = 0; phase < plan.bwd_phases; ++phase) {
      const int waves = std::max(plan.bwd_block_waves[phase], 1), slots = plan.bwd_phase_slots[phase];
      // With several launches every workgroup row of the partials is written by all of them.
      const unsigned blocks = sum_gw ? (unsigned)row_gw_blocks(plan, rows) : row_blocks(plan.bwd_groups, phase, slots, rows, false);
      void* args[] = {&x, &y, &w, &g, &gw_out, &gx, &part, &rows};
      launch("uvu_rows_bwd", kernel(3 + phase, "luna_uvu_rows_bwd_p", phase),
             dim3(blocks, (unsigned)((slots + waves - 1) / waves)), dim3(64 * waves), s, args);
    }
    if (gy) {
      void* genv = nullptr;
      void* args[] = {&part, &gy, &genv, &rows};
      launch("uvu_bwd_reduce", kernel(1, "luna_uvu_bwd_reduce", -1), dim3((unsigned)((rows + 255) / 256)), dim3(256), s,
             args);
    }
    if (sum_gw) {
      int n = (int)row_gw_blocks(plan, rows);
      void* args[] = {&gw_out, &gw, &n};
      launch("uvu_rows_gw", kernel(2, "luna_uvu_rows_gw", -1), dim3((unsigned)((plan.spec.wnum + 31) / 32)), dim3(1024), s,
             args);
    }
  });
}

}  // extern "C"
