// Internal declarations shared by the UVU convolution planner, emitter and
// runtime.  Not part of the public C-ABI (include/lunaeq_amd.h is).
#pragma once

#include <cstdint>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

#include "common.h"

namespace luna {

// One sparse Clebsch-Gordan entry, already scaled by the path weight.
struct Term {
  int i, j, k;
  double c;
};

// One lowered UVU path: input block x_off (channels x d1), edge block y_off
// (d2 components), output block out_off (channels x d3), weights
// w[e, w_off + u * w_stride].
struct Path {
  int x_off, y_off, out_off, w_off, w_stride, channels, d1, d2, d3, l0_col;
  std::vector<Term> terms;
};

struct Spec {
  int dtype_bits = 32;
  int in1 = 0, in2 = 0, out = 0, wnum = 0, l0_dim = 0;
  bool w_broadcast = false;  // one weight row for every edge (no weight gradient)
  std::vector<Path> paths;
};

// An accumulator block: one output block (out_off, d3) of one group.
struct AccBlock {
  int out_off, d3;
  bool accumulate;  // read-modify-write instead of plain store
};

// Paths sharing one input block (x_off, d1, channels), run by one wave per
// (node, chunk of `cw` channels).  A chunk narrower than 64 channels lets a wave
// take 64 / cw edges at once: lane = edge * cw + channel.
struct Group {
  int x_off, d1, channels, chunks;
  int cw = 64;
  std::vector<int> paths;            // indices into Spec::paths
  std::vector<AccBlock> blocks;      // forward output blocks
  std::vector<int> path_block;       // path -> index in blocks
  int phase = 0;
  int slot_base = 0;                 // first grid.y slot of this group in its phase
  bool gx_accumulate = false;        // backward: gx block shared with another group
  int gy_slot_base = 0;              // backward: first partial slot of this group
  // Backward: the group's two 64-channel chunks run as the two waves of one
  // workgroup and add their gy partials through LDS into one slot.
  bool pair_partials = false;
  // Split group whose two path subsets (the two waves of a workgroup) add
  // their gy partials through LDS into one slot per chunk, columns in place.
  bool combine_subsets = false;
  // Backward: the paths may be split into `subsets` path sets, each run by
  // its own wave (slot = chunk * subsets + subset); the two waves of a split
  // group share a workgroup and sum their gx messages through LDS.
  int subsets = 1;
  std::vector<int> path_subset;      // path -> subset
};

struct Plan {
  Spec spec;
  std::vector<Group> fwd_groups;     // forward groups, each with a phase
  int fwd_phases = 0;
  std::vector<int> phase_slots;      // grid.y per forward phase
  bool fwd_needs_zero = false;
  std::vector<Group> bwd_groups;     // backward groups (one launch)
  int bwd_phases = 0;                // backward launches
  std::vector<int> bwd_phase_slots;  // grid.y per backward launch
  int gy_parts = 0;                  // partial slots for the gy reduction
  bool bwd_gx_needs_zero = false;
  // Waves per workgroup of each launch: the slots (waves) of one node share a
  // workgroup, so they run on one CU and stream the node's contiguous weight
  // rows together; grid = (nodes, ceil(slots / waves)).
  std::vector<int> fwd_block_waves, bwd_block_waves;
  // gx message layout and gather vector width, fixed when the schedule is
  // built: the emitted kernels and the launch geometry both read these.
  bool msg_cmajor = true;
  int gather_vec = 1;
  // Width of the edge-offset graph tables (dst_rowptr, src_rowptr,
  // edge_ids_by_src) the kernels read: 32, or 64 for 2^31 or more edges.
  int edge_index_bits = 32;
  // Narrow blocks one edge at a time too (see LunaUvuPlan::sparse).
  bool one_edge = false;
  ModuleCache kernels;  // emitted modules per variant and device
};

Spec parse_spec(const std::string& text);
// Elements per access of the gx gather: 16-byte vectors when every covered
// input range and the row length are multiples of it, else 1 (Plan::gather_vec).
int gather_vector_width(const Plan& plan);
// The gather's workgroup: vectors of a source row it covers, and the teams of
// threads that share the row's edges where the whole row is narrow (256 threads).
int gather_columns(const Plan& plan);
int gather_teams(const Plan& plan);
// True when the gx messages are stored component-major per input block
// (msg[e, x_off + i * C + u]: every store of a wave is 64 contiguous values)
// instead of in the x layout (msg[e, x_off + u * d1 + i]); the gather kernel
// then permutes back.  Requires the groups' input ranges to be identical or
// disjoint.  LUNAEQ_AMD_MSGCM=0 selects the x layout; read once, when the
// plan's schedule is built (Plan::msg_cmajor).
bool message_component_major(const Plan& plan);
void build_schedule(Plan& plan);

// Emitted HIP source of one kernel module variant.  `split`: a workgroup's waves
// share the edges of one (node, slot) instead of taking a slot each.
std::string emit_forward(const Plan& plan, bool env, bool l0, bool split);
// LDS reals per wave of the split forward.
int split_forward_lds(const Plan& plan, int phase);
std::string emit_backward(const Plan& plan, bool env, bool gl0, bool want_gw, bool want_msg, bool want_part);
// Row-wise products (row b is node, source and edge b); `shared`: one weight row
// for every row, whose gradient is summed (a partial per workgroup, then one sum).
std::string emit_rows_forward(const Plan& plan, bool shared);
std::string emit_rows_backward(const Plan& plan, bool shared, bool want_gw, bool want_msg, bool want_part);

// The first-order backward launches (luna_uvu_conv_bwd without the plan
// check), with the caller's workspace of uvu_bwd_workspace_bytes bytes.
size_t uvu_bwd_workspace_bytes(const Plan& plan, int64_t num_edges);
void uvu_conv_bwd(Plan& plan, const void* x, const void* y, const void* w, const void* env, const void* g,
                  const void* gl0, const int32_t* src, const void* dst_rowptr, const int32_t* node_order,
                  const void* src_rowptr, const void* edge_ids_by_src, void* gx, void* gy, void* gw,
                  void* genv, void* workspace, size_t workspace_bytes, int64_t num_nodes, int64_t num_edges,
                  void* stream);


}  // namespace luna

// The C-ABI's opaque plan handle (include/lunaeq_amd.h).
struct LunaUvuPlan {
  luna::Plan plan;
  // For graphs of few edges per node, where a wave that takes several edges of a
  // node at once finds too few (null where the plan takes one at a time anyway): at
  // most two per node, three where the plan takes two at once.  Forward + backward
  // of 40,000 nodes, lmax 2, at 1 / 2 / 3 edges per node, several at once and one:
  // 8 channels 206 / 224 / 240 and 144 / 196 / 256 us, 16 channels 230 / 254 / 274 and 165 /
  // 221 / 285 us, 32 channels 282 / 308 / 388 and 217 / 281 / 349 us (20,000 nodes of four:
  // 213 and 211 us).
  std::unique_ptr<luna::Plan> sparse;
  int sparse_degree = 2;
  bool few(int64_t nodes, int64_t edges) const { return sparse && edges <= sparse_degree * nodes; }
  luna::Plan& of(int64_t nodes, int64_t edges) { return few(nodes, edges) ? *sparse : plan; }
};
