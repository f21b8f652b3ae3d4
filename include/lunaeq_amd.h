/*
 * C-ABI of the MI355X (gfx950) UVU tensor-product convolution library.
 *
 * The reference binds one pybind11 module per irreps configuration, generated
 * and compiled at prepare time:
 *   - run_uvu_conv_fwd_ordered(x, y, weight, env?, l0?, src, rowptr,
 *       node_order, node_tiers?, out, num_nodes)
 *       (src/lunatp/uvu_conv/kernels/forward.py:1117-1128)
 *   - run_uvu_conv_bwd(x, y, w, go, dst, edge_ids, seg_*..., gx_partial,
 *       gy_partial, gx, gy, gw, nodes, edges, segments, env?, ge_partial?, ge?,
 *       grad_l0?)  (src/lunatp/uvu_conv/kernels/backward.py:505-512)
 *   - the double-backward launcher (double_backward.py:1635-...)
 * Here one shared library holds the launchers; a plan object holds the
 * per-configuration kernels, which the library emits as HIP source from the
 * path specification and compiles for gfx950 with hipRTC (code objects are
 * cached on disk).  The compute entry points allocate no device memory:
 * every buffer, the backward workspaces included, comes from the caller.
 * Only luna_placed_alloc (below) allocates, and only when called: the
 * Python layer uses it to hold one region-placed backward workspace per
 * device outside torch's allocator.  Launches are ordered on the
 * caller's stream.  Every function returns 0 on success or a non-zero error
 * code; luna_last_error() gives the message of the last failure on the
 * calling thread.
 *
 * Data layout (row-major, contiguous, dtype of the plan):
 *   x   [N, in1_dim]      node features, e3nn layout (copy-major irreps)
 *   y   [E, in2_dim]      edge attributes
 *   w   [E, weight_numel] per-edge path weights, w[e, w_off + u*w_stride + v]
 *   env [E] or NULL       per-edge envelope multiplying each message
 *   out [N, out_dim]
 *   l0  [E, l0_dim]       optional scalar-path features (before env)
 * Graph tables: src[E], dst[E] (dst sorted ascending), node_order[N] and
 * source_node_order[N] are int32; the edge offsets dst_rowptr[N+1],
 * src_rowptr[N+1] and edge_ids_by_src[E] are int32, or int64 with a plan of
 * 64-bit edge offsets (luna_uvu_plan_create_ex / luna_uuu_plan_create_ex)
 * for graphs of 2^31 or more edges.  Node counts stay below 2^31.
 */
#ifndef LUNAEQ_AMD_H
#define LUNAEQ_AMD_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct LunaUvuPlan LunaUvuPlan;

/* Opaque stream handle: a hipStream_t (NULL = the null stream). */
typedef void* LunaStream;

/* Static facts about a plan, filled by luna_uvu_plan_info. */
typedef struct LunaUvuPlanInfo {
  int32_t dtype_bits;        /* 32 or 64 */
  int32_t in1_dim, in2_dim, out_dim, weight_numel, l0_dim;
  int32_t num_paths;
  int32_t fwd_needs_zero;    /* out must be zero-filled before luna_uvu_conv_fwd */
  int32_t bwd_gx_needs_zero; /* input blocks overlap: gx messages are accumulated */
  int32_t num_fwd_launches;  /* launches per forward call */
  int32_t gy_parts;          /* partial slots of the edge-attribute gradient */
} LunaUvuPlanInfo;

/* Text of the last error on this thread ("" if none). */
const char* luna_last_error(void);

/* Library version string. */
const char* luna_version(void);

/* Number of visible HIP devices (0 without a GPU); never fails. */
int luna_device_count(void);

/*
 * Build a plan from a path specification (the metadata the reference builds in
 * build_uvu_conv_metadata, src/lunatp/uvu_conv/kernels/utils.py:23-119):
 *
 *   "LUNAUVU1 <dtype_bits> <in1> <in2> <out> <weight_numel> <npaths> <l0_dim>"
 *   then per path:
 *   "<x_off> <y_off> <out_off> <w_off> <w_stride> <channels> <d1> <d2> <d3>
 *    <l0_col or -1> <nterms> (<i> <j> <k> <coefficient>)*nterms"
 *
 * The header "LUNAUVU2 <dtype_bits> <in1> <in2> <out> <weight_numel> <npaths>
 * <l0_dim> <w_broadcast>" is the same with one flag: when w_broadcast is 1 the
 * weight operand w is a single row [1, weight_numel] read by every edge (no
 * per-edge weight traffic; gw must then be NULL in luna_uvu_conv_bwd).  The
 * UVW convolution uses it with a row of ones to aggregate per-node sums of the
 * edge products before its weight contraction.
 * Coefficients already include the path weight.  Kernels are emitted and
 * compiled here (or loaded from the code-object cache in cache_dir, which may
 * be NULL for no cache); loading onto a device is deferred to first launch.
 * replaces: LunaTPUVUConv / configure_uvu_conv / load_forward
 * (src/lunatp/interface.py:353-367, uvu_conv/kernels/utils.py:121-158,
 * uvu_conv/kernels/forward.py:1249-1288).
 */
int luna_uvu_plan_create(const char* spec, const char* cache_dir, LunaUvuPlan** plan);
/*
 * luna_uvu_plan_create with the width of the edge-offset tables its kernels
 * read: edge_index_bits 32 (luna_uvu_plan_create) or 64, for graphs of 2^31
 * or more edges, whose dst_rowptr, src_rowptr and edge_ids_by_src are int64
 * (node ids stay int32).  replaces: configure_indexing / select_indexing with
 * index_bits=64 (src/lunatp/utils/layout.py:441-517) and
 * get_graph_with_int64_offsets (src/lunatp/graph.py:147-170).
 */
int luna_uvu_plan_create_ex(const char* spec, const char* cache_dir, int edge_index_bits, LunaUvuPlan** plan);
int luna_uvu_plan_destroy(LunaUvuPlan* plan);
int luna_uvu_plan_info(const LunaUvuPlan* plan, LunaUvuPlanInfo* info);

/*
 * Compile (or fetch from cache) the forward and backward kernels that every layer runs
 * (no envelope, no scalar features), without touching a device.  Used to warm the
 * code-object cache ahead of time; luna_uvu_plan_precompile_all also compiles the
 * kernels for few nodes and for few edges per node, and the row-wise products'.
 */
int luna_uvu_plan_precompile(LunaUvuPlan* plan);
int luna_uvu_plan_precompile_all(LunaUvuPlan* plan);

/*
 * Forward: out[t] = sum over edges e with dst[e]==t of env[e] * TP(x[src[e]], y[e], w[e]).
 * l0 may be NULL; when given, l0[e, :] receives the per-edge scalar-path
 * contributions before env.
 * replaces: run_uvu_conv_fwd_ordered (src/lunatp/uvu_conv/kernels/forward.py:1117-1128)
 */
int luna_uvu_conv_fwd(const LunaUvuPlan* plan,
                      const void* x, const void* y, const void* w, const void* env,
                      const int32_t* src, const void* dst_rowptr,
                      const int32_t* node_order,
                      void* out, void* l0,
                      int64_t num_nodes, int64_t num_edges, LunaStream stream);

/* Bytes of device workspace luna_uvu_conv_bwd needs for this problem size. */
int luna_uvu_conv_bwd_workspace(const LunaUvuPlan* plan, int64_t num_nodes,
                                int64_t num_edges, size_t* bytes);

/*
 * First-order backward.  g = dL/dout [N, out_dim]; gl0 = dL/dl0 [E, l0_dim] or
 * NULL.  Writes gx [N, in1], gy [E, in2], gw [E, weight_numel] and, when env
 * is given and genv is not NULL, genv [E].  Any of gx/gy/gw may be NULL to skip
 * it.  A destination-owned kernel streams each node's in-edges (dst CSR:
 * src, dst_rowptr, node_order) and writes gw, gy partials and one gx message
 * per edge into the workspace; a second pass sums the messages over each
 * node's out-edges (src CSR: src_rowptr, edge_ids_by_src).  workspace must hold
 * luna_uvu_conv_bwd_workspace bytes.
 * replaces: run_uvu_conv_bwd (src/lunatp/uvu_conv/kernels/backward.py:505-512)
 */
int luna_uvu_conv_bwd(const LunaUvuPlan* plan,
                      const void* x, const void* y, const void* w, const void* env,
                      const void* g, const void* gl0,
                      const int32_t* src, const void* dst_rowptr,
                      const int32_t* node_order,
                      const void* src_rowptr, const void* edge_ids_by_src,
                      void* gx, void* gy, void* gw, void* genv,
                      void* workspace, size_t workspace_bytes,
                      int64_t num_nodes, int64_t num_edges, LunaStream stream);

/*
 * Row-wise product: luna_uvu_conv_fwd with row b as node b, edge b and the
 * source of edge b (no graph tables, no env and l0).  shared_w: w is one row
 * [1, weight_numel] for all rows (always so with a w_broadcast plan).
 * out must be zero-filled where the plan's fwd_needs_zero says so.
 * replaces: the row-wise uvu forward (src/lunatp/interface.py:265-285)
 */
int luna_uvu_rows_fwd(const LunaUvuPlan* plan, const void* x, const void* y, const void* w, int shared_w,
                      void* out, int64_t rows, LunaStream stream);
/* Bytes of device workspace luna_uvu_rows_bwd needs where it writes gy, or gw of a shared row. */
int luna_uvu_rows_bwd_workspace(const LunaUvuPlan* plan, int shared_w, int64_t rows, size_t* bytes);
/*
 * Its first-order backward: gx [rows, in1], gy [rows, in2] and gw [rows,
 * weight_numel], or with shared_w [1, weight_numel] summed over the rows; each
 * may be NULL.  gw must be NULL with a w_broadcast plan.
 */
int luna_uvu_rows_bwd(const LunaUvuPlan* plan, const void* x, const void* y, const void* w, int shared_w,
                      const void* g, void* gx, void* gy, void* gw, void* workspace, size_t workspace_bytes,
                      int64_t rows, LunaStream stream);

/*
 * Device buffer of `bytes` (at least 1 GB) placed outside the HBM region of
 * `avoid` (a device buffer of avoid_bytes >= 2 GB whose contents the probe
 * overwrites; NULL: outside the region the allocator is filling now).
 * Concurrent writes to two buffers run about 25 % faster when the buffers lie
 * in different ~96 GB regions of the device than in one; the backward's
 * message workspace is placed this way against the weight gradient it is
 * written beside.  The regions of a fresh allocation are found by measurement
 * (as in luna_region_overlap); allocations whose overlap with `avoid` exceeds
 * 0.25 are held as spacers, up to max_spacer_bytes and while free memory
 * allows, and released on return.  *moved is 1 when the returned buffer's
 * overlap is at most 0.25, 0 when the search gave up (the least overlapping
 * candidate is returned) or max_spacer_bytes is 0 (an ordinary allocation,
 * nothing probed).  Synchronises `stream`.  Release with luna_placed_free.
 * No counterpart in the reference.
 */
int luna_placed_alloc(size_t bytes, void* avoid, size_t avoid_bytes, size_t max_spacer_bytes,
                      LunaStream stream, void** out, int* moved);
/*
 * *overlap = expected share of write pairs that meet in one HBM region when
 * a and b are written together: fa fb + (1 - fa)(1 - fb), where fa and fb are
 * the shares of up to four 1 GB windows of each buffer (start, thirds, end)
 * found in the region of a's first window by a write probe.  1 for two parts
 * of one region, 0 for buffers in different regions.  a_bytes >= 2 GB,
 * b_bytes >= 1 GB.  Overwrites the first 2 GB of a and the windows of a and
 * b; synchronises `stream`.
 */
int luna_region_overlap(void* a, size_t a_bytes, void* b, size_t b_bytes, LunaStream stream,
                        double* overlap);
int luna_placed_free(void* pointer);

/*
 * Allocation-free first-order backward: luna_uvu_conv_bwd with its workspace
 * taken from a static device array of LUNA_UVU_NOALLOC_SCRATCH_BYTES (64 MiB)
 * that every GPU the library runs on holds until the process ends.  It calls no
 * hipMalloc/hipFree; problems whose workspace (luna_uvu_conv_bwd_workspace)
 * exceeds the array are refused with an error.  The first call on a device
 * looks up the array's device address (and, like every entry point, loads the
 * plan's kernels on first use); make one call before capturing a HIP graph.
 * All calls on one GPU share its array: calls that overlap on one GPU race.
 * No counterpart in the reference: it is for callers that cannot allocate
 * (code under HIP graph capture, serving loops, harnesses that forbid it).
 */
#define LUNA_UVU_NOALLOC_SCRATCH_BYTES (64ull << 20)
size_t luna_uvu_conv_bwd_noalloc_limit(void);
int luna_uvu_conv_bwd_noalloc(const LunaUvuPlan* plan,
                              const void* x, const void* y, const void* w, const void* env,
                              const void* g, const void* gl0,
                              const int32_t* src, const void* dst_rowptr,
                              const int32_t* node_order,
                              const void* src_rowptr, const void* edge_ids_by_src,
                              void* gx, void* gy, void* gw, void* genv,
                              int64_t num_nodes, int64_t num_edges, LunaStream stream);

/* ------------------------------------------------------------------------ */
/* Shared-weight UVW tensor product (fp32, matrix cores).                    */

typedef struct LunaUvwPlan LunaUvwPlan;

/*
 * Build a UVW plan from its path specification (the metadata of
 * build_uvw_metadata, src/lunatp/uvw/kernels/utils.py:100-190):
 *   "LUNAUVW1 32 <in1> <in2> <out> <weight_numel> <npaths>"
 *   then per path:
 *   "<x_off> <y_off> <out_off> <w_off> <mul1> <mul2> <mul3> <d1> <d2> <d3> <nterms> (<i> <j> <k> <c>)*"
 * Weights of a path are laid out [u][v][w] (e3nn).  Coefficients include the
 * path weight.
 * replaces: LunaTPUVW / load of the UVW extension (src/lunatp/interface.py:310-335)
 */
int luna_uvw_plan_create(const char* spec, const char* cache_dir, LunaUvwPlan** plan);
int luna_uvw_plan_destroy(LunaUvwPlan* plan);
/* flags[0..3]: out, gx, gy, gw must be zero-filled by the caller (uncovered ranges). */
int luna_uvw_plan_needs_zero(const LunaUvwPlan* plan, int32_t* flags);
int luna_uvw_plan_precompile(LunaUvwPlan* plan);

/*
 * out[b] = sum over paths of the uvw product of x[b] [in1], y[b] [in2] with the
 * shared weight [weight_numel], for b < rows.
 * replaces: the UVW forward launcher (src/lunatp/uvw/kernels/forward.py:1576-1612)
 */
int luna_uvw_fwd(const LunaUvwPlan* plan, const void* x, const void* y, const void* weight,
                 void* out, int64_t rows, LunaStream stream);

/* Bytes of workspace luna_uvw_bwd needs (weight-gradient partials per 256-row
 * chunk and edge-gradient partials per input block and 32-wide K tile). */
int luna_uvw_bwd_workspace(const LunaUvwPlan* plan, int64_t rows, size_t* bytes);

/*
 * Backward of luna_uvw_fwd for seed g [rows, out]: gx and gy (both or neither)
 * and gw [weight_numel] (NULL to skip).  workspace must hold
 * luna_uvw_bwd_workspace bytes whenever anything is requested.  With rows == 0
 * x, y and g may be NULL; gw is then written as zeros.
 * replaces: the UVW backward launcher (src/lunatp/uvw/interface.py:42-49)
 */
int luna_uvw_bwd(const LunaUvwPlan* plan, const void* x, const void* y, const void* weight,
                 const void* g, void* gx, void* gy, void* gw, void* workspace,
                 size_t workspace_bytes, int64_t rows, LunaStream stream);

/* ------------------------------------------------------------------------ */
/* Shared-weight contraction of the UVW convolution (fp32, fp64 matrix cores). */

typedef struct LunaConPlan LunaConPlan;

/*
 * Per output block o (d3 components, mul3 copies) over the channels c of its
 * paths, c = (path, v, u) and row(c) = w_off + (u * mul2 + v) * mul3:
 *   out[n, out_off + m*d3 + k] = sum_c a[n, a_off + c*d3 + k] weight[row(c) + m]
 * Specification (degrees up to 5):
 *   "LUNACON1 <dtype_bits> <aggregate_dim> <out_dim> <weight_numel> <nblocks>"
 *   then per block "<out_off> <a_off> <d3> <mul3> <npaths> (<w_off> <mul1> <mul2>)*npaths"
 * Columns of out (or a, for the gradient) outside every block are not written.
 * replaces: the per-edge weight contraction of the UVW convolution
 * (src/lunatp/uvw_conv/interface.py:190-245)
 */
int luna_con_plan_create(const char* spec, const char* cache_dir, LunaConPlan** plan);
int luna_con_plan_destroy(LunaConPlan* plan);
int luna_con_plan_precompile(LunaConPlan* plan);
int luna_con_fwd(const LunaConPlan* plan, const void* a, const void* weight, void* out, int64_t rows,
                 LunaStream stream);
/* ga[n, a_off + c*d3 + k] = sum_m g[n, out_off + m*d3 + k] weight[row(c) + m]. */
int luna_con_grad_a(const LunaConPlan* plan, const void* g, const void* weight, void* ga, int64_t rows,
                    LunaStream stream);
/* gw[row(c) + m] = sum_{n,k} a[n, a_off + c*d3 + k] g[n, out_off + m*d3 + k] through
 * partial tiles in `workspace` (luna_con_grad_w_workspace bytes). */
int luna_con_grad_w_workspace(const LunaConPlan* plan, int64_t rows, size_t* bytes);
int luna_con_grad_w(const LunaConPlan* plan, const void* a, const void* g, void* gw, void* workspace,
                    size_t workspace_bytes, int64_t rows, LunaStream stream);

/* ------------------------------------------------------------------------ */
/* UUU (channel-wise) tensor-product convolution.                            */

typedef struct LunaUuuPlan LunaUuuPlan;

/*
 * Build a UUU convolution plan (the metadata of build_uuu_conv_metadata,
 * src/lunatp/uuu_conv/kernels/utils.py:342-364, lowered by build_uuu_metadata,
 * src/lunatp/uuu/kernels/utils.py:250-330):
 *   "LUNAUUU1 <dtype_bits> <in1> <in2> <out> <weight_numel> <npaths> <l0_dim>"
 *   then per path:
 *   "<x_off> <y_off> <out_off> <w_off or -1 if unweighted> <channels> <d1> <d2>
 *    <d3> <l0_col or -1> <nterms> (<i> <j> <k> <coefficient>)*nterms"
 * A path reads x[s, x_off + u*d1 + i], y[e, y_off + u*d2 + j] and
 * w[e, w_off + u] for each channel u < channels and writes
 * out[t, out_off + u*d3 + k].  Coefficients include the path weight.
 * replaces: LunaTPUUUConv / configure_uuu_conv (src/lunatp/interface.py:338-350,
 * src/lunatp/uuu_conv/kernels/utils.py:116-199)
 */
int luna_uuu_plan_create(const char* spec, const char* cache_dir, LunaUuuPlan** plan);
/* luna_uuu_plan_create with 32- or 64-bit edge offsets (as luna_uvu_plan_create_ex). */
int luna_uuu_plan_create_ex(const char* spec, const char* cache_dir, int edge_index_bits, LunaUuuPlan** plan);
int luna_uuu_plan_destroy(LunaUuuPlan* plan);
/* flags[0..3]: out, gx, gy, gw must be zero-filled by the caller (ranges no path covers). */
int luna_uuu_plan_needs_zero(const LunaUuuPlan* plan, int32_t* flags);
int luna_uuu_plan_precompile(LunaUuuPlan* plan);

/*
 * Forward: out[t] = sum over edges e with dst[e]==t of env[e] * msg[e]; l0 (may
 * be NULL) receives the scalar-path messages before env, one column per
 * channel.  Destination-owned over the dst CSR (src, dst_rowptr, node_order).
 * replaces: run_uuu_conv at order 0 (src/lunatp/uuu_conv/kernels/utils.py:87-112,
 * launched by launch_forward, src/lunatp/uuu_conv/kernels/traversal.py:2095)
 */
int luna_uuu_conv_fwd(const LunaUuuPlan* plan, const void* x, const void* y, const void* w,
                      const void* env, const int32_t* src, const void* dst_rowptr,
                      const int32_t* node_order, void* out, void* l0, int64_t num_nodes,
                      int64_t num_edges, LunaStream stream);

/* Bytes of device workspace luna_uuu_conv_bwd needs (env-gradient partials; may be 0). */
int luna_uuu_conv_bwd_workspace(const LunaUuuPlan* plan, int64_t num_nodes, int64_t num_edges,
                                size_t* bytes);

/*
 * First-order backward for the seed g [N, out] (and gl0 [E, l0_dim] or NULL):
 * gx [N, in1], gy [E, in2], gw [E, weight_numel], genv [E] (only with env);
 * any output may be NULL.  Source-owned over the src CSR (src_rowptr,
 * edge_ids_by_src, source_node_order) with dst[E] to find each edge's seed.
 * replaces: run_uuu_conv at order 1 (src/lunatp/uuu_conv/kernels/utils.py:87-112,
 * driven by run, src/lunatp/uuu_conv/kernels/traversal.py:1943-2092)
 */
int luna_uuu_conv_bwd(const LunaUuuPlan* plan, const void* x, const void* y, const void* w,
                      const void* env, const void* g, const void* gl0, const int32_t* dst,
                      const void* src_rowptr, const void* edge_ids_by_src,
                      const int32_t* source_node_order, void* gx, void* gy, void* gw, void* genv,
                      void* workspace, size_t workspace_bytes, int64_t num_nodes, int64_t num_edges,
                      LunaStream stream);

/* ------------------------------------------------------------------------ */
/* Graph tables on the GPU.                                                  */

/*
 * status[0..3] (device int64) <- min index over src and dst, max index, 1 if
 * dst descends anywhere else 0, 0.  index_bits is 32 or 64 (src and dst share
 * it).  The caller reads status back to validate.
 * replaces: graph_bounds of the reference's topology extension
 * (src/lunatp/utils/graph.py:806-837, called from src/lunatp/graph.py:77).
 */
int luna_graph_bounds(const void* src, const void* dst, int index_bits, int64_t num_edges, int64_t* status,
                      LunaStream stream);

/* Bytes of device workspace luna_graph_build needs. */
int luna_graph_workspace(int64_t num_nodes, int64_t num_edges, size_t* bytes);

/*
 * Every table of a validated, dst-sorted graph (int32):
 *   src32, dst32 [E]; dst_rowptr, src_rowptr [N+1]; edge_ids_by_src [E]
 *   (stable by source); edge_ids_by_dst [E]; node_order, source_node_order [N]
 *   (descending degree, ties by node id); node_tiers [3]; seg_rowptr [N+1];
 *   seg_nodes, seg_begin, seg_end, seg_order with room for N + E/32 + 1
 *   segments, of which seg_rowptr[N] are real (the others are unspecified).
 * replaces: make_graph_tables of the reference's topology extension
 * (src/lunatp/utils/graph.py:142-846, called from src/lunatp/graph.py:106).
 */
int luna_graph_build(const void* src, const void* dst, int index_bits, int64_t num_nodes, int64_t num_edges,
                     int32_t* src32, int32_t* dst32, int32_t* dst_rowptr, int32_t* src_rowptr,
                     int32_t* edge_ids_by_src, int32_t* edge_ids_by_dst, int32_t* node_order,
                     int32_t* source_node_order, int32_t* node_tiers, int32_t* seg_rowptr, int32_t* seg_nodes,
                     int32_t* seg_begin, int32_t* seg_end, int32_t* seg_order, void* workspace,
                     size_t workspace_bytes, LunaStream stream);

/*
 * luna_graph_build in steps that let the caller size the second one, all on one
 * workspace of luna_graph_workspace bytes and one stream.
 * luna_graph_scan writes src32, dst32, both edge id lists, the row pointers, seg_rowptr
 * and status[8] = smallest and largest index, dst not sorted, segments, largest in- and
 * out-degree, 0, 0; indices outside [0, num_nodes) or out of order are reported, and the
 * tables are valid only if there are none.
 * luna_graph_finish, for validated indices, writes the node orders, tiers and the
 * `segments` source segments; largest_degree bounds both degrees.
 */
int luna_graph_scan(const void* src, const void* dst, int index_bits, int64_t num_nodes, int64_t num_edges,
                    int32_t* src32, int32_t* dst32, int32_t* dst_rowptr, int32_t* src_rowptr,
                    int32_t* edge_ids_by_src, int32_t* edge_ids_by_dst, int32_t* seg_rowptr, int64_t* status,
                    void* workspace, size_t workspace_bytes, LunaStream stream);
int luna_graph_finish(const int32_t* dst_rowptr, const int32_t* src_rowptr, const int32_t* seg_rowptr,
                      int64_t num_nodes, int64_t num_edges, int64_t largest_degree, int64_t segments,
                      int32_t* node_order, int32_t* source_node_order, int32_t* node_tiers, int32_t* seg_nodes,
                      int32_t* seg_begin, int32_t* seg_end, int32_t* seg_order, void* workspace,
                      size_t workspace_bytes, LunaStream stream);

/* Compile (or load from cache_dir) the graph kernels without touching a device;
 * also sets the cache directory the graph kernels use afterwards. */
int luna_graph_precompile(const char* cache_dir);

/*
 * Measurement hook (no counterpart in the reference): while enabled, every
 * launch is bracketed by HIP events on its stream.  luna_profile_collect waits
 * for the recorded events and writes one line per kernel name,
 * "<name> <launches> <total_ms> <min_ms> <max_ms>", then clears the records.
 */
int luna_profile_enable(int on);
int luna_profile_collect(char* buffer, size_t capacity, size_t* needed);

#ifdef __cplusplus
}
#endif

#endif /* LUNAEQ_AMD_H */
