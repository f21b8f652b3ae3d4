// UUU ("channel-wise") tensor-product convolution on gfx950.
//
// For a path p with C channels (mul_in1 = mul_in2 = mul_out = C) and an edge
// e = (s -> t):
//   msg_p[e, u, k] = a_p[e, u] * sum_{(i,j,k)} c_ijk x[s, xo + u*d1 + i] y[e, yo + u*d2 + j]
//   out[t, oo + u*d3 + k] += env[e] * msg_p[e, u, k]
// with a_p = w[e, wo + u] for weighted paths and 1 otherwise (e3nn's uuu
// connection; src/lunatp/uuu/kernels/utils.py:250-330 lowers the paths and
// src/lunatp/uuu_conv/interface.py:143-240 defines the convolution).
//
// Every operand of one channel u is private to that channel, so one lane owns
// one channel and no value ever crosses lanes except in the sums over edges:
//   forward  (destination-owned): a wave streams the in-edges of node t and
//            keeps out[t] in registers; it gathers x[src] per edge;
//   backward (source-owned): a wave streams the out-edges of node s
//            (edge_ids_by_src), gathers g[dst] per edge, keeps gx[s] in
//            registers and writes gy[e] and gw[e] straight from the lanes.
// The source-owned backward needs no per-edge gx messages and no second
// pass; the reference's backward traverses sources the same way
// (src/lunatp/uuu_conv/interface.py:300-330).
//
// Channel counts below 64 would leave lanes idle, so a wave covers 64 / W
// edges at once with W = the next power of two >= C: lane = sub * W + u, and
// the per-node sums are completed across the sub-groups with lane exchanges.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <map>
#include <memory>
#include <set>
#include <sstream>

#include "../../include/lunaeq_amd.h"
#include "common.h"

namespace luna {
namespace {

struct UTerm {
  int i, j, k;
  double c;
};

struct UPath {
  int x_off, y_off, out_off, w_off, ch, d1, d2, d3, l0_col;
  std::vector<UTerm> terms;
  int xb = -1, yb = -1, ob = -1;  // block ids
};

// A block of one operand: channels x d components starting at off.
struct UBlock {
  int off, d, ch;
};

struct USpec {
  int bits = 32;
  int in1 = 0, in2 = 0, out = 0, wnum = 0, l0 = 0;
  std::vector<UPath> paths;
  std::vector<UBlock> xblocks, yblocks, oblocks;
};

// One wave body: the paths a wave evaluates for one node and channel chunk.
struct UGroup {
  std::vector<int> paths;
  int ch = 0, cw = 64, chunks = 1;
  int phase = 0;                 // backward: launch order among groups sharing edge blocks
  int genv_slot = 0;             // backward: first partial slot of env's gradient
  std::set<int> xbs, ybs, obs;
  std::set<int> gx_accumulate;   // backward: x blocks already written by an earlier phase
  std::set<int> out_accumulate;  // forward: output blocks already written by an earlier launch
};

struct UuuPlan {
  USpec spec;
  std::vector<UGroup> fwd, bwd;
  int bwd_phases = 0;
  int genv_slots = 0;
  bool out_zero = false, gx_zero = false, gy_zero = false, gw_zero = false;
  int edge_index_bits = 32;  // width of src_rowptr / dst_rowptr / edge_ids_by_src
  ModuleCache kernels;
};

// Accumulated register estimates (32-bit registers) per wave body.
constexpr int kForwardBudget = 96;
constexpr int kBackwardBudget = 128;

int read_int(std::istringstream& in, const char* what) {
  long long value;
  if (!(in >> value)) fail(std::string("uuu spec: expected integer for ") + what);
  if (value < -1 || value > (1LL << 31) - 1) fail(std::string("uuu spec: value out of range for ") + what);
  return (int)value;
}

// Block id of [off, off + ch*d) in `blocks`; distinct blocks must not overlap.
int block_id(std::vector<UBlock>& blocks, int off, int d, int ch, const char* what) {
  const long lo = off, hi = off + (long)ch * d;
  for (size_t n = 0; n < blocks.size(); ++n) {
    const UBlock& b = blocks[n];
    if (b.off == off && b.d == d && b.ch == ch) return (int)n;
    if (lo < b.off + (long)b.ch * b.d && b.off < hi)
      fail(std::string("uuu spec: overlapping ") + what + " blocks of different shape");
  }
  blocks.push_back({off, d, ch});
  return (int)blocks.size() - 1;
}

USpec parse(const std::string& text) {
  std::istringstream in(text);
  std::string magic;
  in >> magic;
  if (magic != "LUNAUUU1") fail("uuu spec: missing LUNAUUU1 header");
  USpec s;
  s.bits = read_int(in, "dtype");
  if (s.bits != 32 && s.bits != 64) fail("uuu spec: dtype must be 32 or 64");
  s.in1 = read_int(in, "in1");
  s.in2 = read_int(in, "in2");
  s.out = read_int(in, "out");
  s.wnum = read_int(in, "weight_numel");
  const int npaths = read_int(in, "npaths");
  s.l0 = read_int(in, "l0_dim");
  if (s.in1 < 0 || s.in2 < 0 || s.out < 0 || s.wnum < 0 || s.l0 < 0 || npaths < 0)
    fail("uuu spec: negative dimension");
  for (int n = 0; n < npaths; ++n) {
    UPath p;
    p.x_off = read_int(in, "x_off");
    p.y_off = read_int(in, "y_off");
    p.out_off = read_int(in, "out_off");
    p.w_off = read_int(in, "w_off");
    p.ch = read_int(in, "channels");
    p.d1 = read_int(in, "d1");
    p.d2 = read_int(in, "d2");
    p.d3 = read_int(in, "d3");
    p.l0_col = read_int(in, "l0_col");
    const int nterms = read_int(in, "nterms");
    if (p.ch <= 0) fail("uuu spec: UUU convolution requires positive channels for every path");
    if (p.d1 <= 0 || p.d2 <= 0 || p.d3 <= 0 || nterms < 0) fail("uuu spec: bad path dimensions");
    if (p.x_off < 0 || (long)p.x_off + (long)p.ch * p.d1 > s.in1) fail("uuu spec: input block outside in1_dim");
    if (p.y_off < 0 || (long)p.y_off + (long)p.ch * p.d2 > s.in2) fail("uuu spec: edge block outside in2_dim");
    if (p.out_off < 0 || (long)p.out_off + (long)p.ch * p.d3 > s.out)
      fail("uuu spec: output block outside out_dim");
    if (p.w_off >= 0 && (long)p.w_off + p.ch > s.wnum) fail("uuu spec: weight block outside weight_numel");
    if (p.l0_col >= 0 && (p.d3 != 1 || (long)p.l0_col + p.ch > s.l0)) fail("uuu spec: l0 column outside l0_dim");
    for (int t = 0; t < nterms; ++t) {
      UTerm term;
      term.i = read_int(in, "i");
      term.j = read_int(in, "j");
      term.k = read_int(in, "k");
      std::string token;
      in >> token;
      char* end = nullptr;
      term.c = std::strtod(token.c_str(), &end);
      if (token.empty() || *end) fail("uuu spec: bad coefficient '" + token + "'");
      if (term.i < 0 || term.i >= p.d1 || term.j < 0 || term.j >= p.d2 || term.k < 0 || term.k >= p.d3)
        fail("uuu spec: coefficient index outside the path's irreps");
      p.terms.push_back(term);
    }
    p.xb = block_id(s.xblocks, p.x_off, p.d1, p.ch, "input");
    p.yb = block_id(s.yblocks, p.y_off, p.d2, p.ch, "edge");
    p.ob = block_id(s.oblocks, p.out_off, p.d3, p.ch, "output");
    s.paths.push_back(std::move(p));
  }
  // Weighted paths must own disjoint weight ranges (each writes its gradient).
  std::vector<std::pair<int, int>> ws;
  for (const UPath& p : s.paths)
    if (p.w_off >= 0) ws.push_back({p.w_off, p.w_off + p.ch});
  std::sort(ws.begin(), ws.end());
  for (size_t n = 1; n < ws.size(); ++n)
    if (ws[n].first < ws[n - 1].second) fail("uuu spec: weight ranges of two paths overlap");
  return s;
}

int pow2_at_least(int v) {
  int p = 1;
  while (p < v && p < 64) p *= 2;
  return p;
}

void finish_group(UGroup& g, const USpec& s) {
  g.ch = s.paths[g.paths[0]].ch;
  g.cw = pow2_at_least(g.ch);
  g.chunks = (g.ch + 63) / 64;
  for (int p : g.paths) {
    g.xbs.insert(s.paths[p].xb);
    g.ybs.insert(s.paths[p].yb);
    g.obs.insert(s.paths[p].ob);
  }
}

int cost(const USpec& s, const std::vector<int>& paths, bool backward) {
  std::set<int> xs, ys, os;
  int weights = 0;
  for (int p : paths) {
    xs.insert(s.paths[p].xb);
    ys.insert(s.paths[p].yb);
    os.insert(s.paths[p].ob);
    weights += s.paths[p].w_off >= 0;
  }
  int regs = weights;
  for (int b : xs) regs += s.xblocks[b].d * (backward ? 2 : 1);
  for (int b : ys) regs += s.yblocks[b].d * (backward ? 2 : 1);
  for (int b : os) regs += s.oblocks[b].d;
  return regs * (s.bits / 32);
}

// Forward: the unit is an edge block (every path reading it), so each
// per-edge row of y and w is read by one group only; a unit over the register
// estimate is cut by output block.  Units of one channel count are packed into
// a group while its estimate fits.  The output rows are per node: a group whose
// output block an earlier group (launch) already wrote adds to it.
std::vector<UGroup> forward_groups(const USpec& s) {
  std::vector<std::vector<int>> units;
  for (int b = 0; b < (int)s.yblocks.size(); ++b) {
    std::vector<int> unit;
    for (int p = 0; p < (int)s.paths.size(); ++p)
      if (s.paths[p].yb == b) unit.push_back(p);
    if (unit.empty()) continue;
    if (cost(s, unit, false) <= kForwardBudget) {
      units.push_back(unit);
      continue;
    }
    std::map<int, std::vector<int>> by_out;
    for (int p : unit) by_out[s.paths[p].ob].push_back(p);
    for (const auto& kv : by_out) units.push_back(kv.second);
  }
  std::vector<UGroup> groups;
  std::map<int, int> open;  // channels -> index of the group being filled
  for (const auto& unit : units) {
    const int ch = s.paths[unit[0]].ch;
    auto it = open.find(ch);
    if (it != open.end()) {
      std::vector<int> merged = groups[it->second].paths;
      merged.insert(merged.end(), unit.begin(), unit.end());
      if (cost(s, merged, false) <= kForwardBudget) {
        groups[it->second].paths = merged;
        continue;
      }
    }
    UGroup g;
    g.paths = unit;
    groups.push_back(g);
    open[ch] = (int)groups.size() - 1;
  }
  std::set<int> written;
  for (UGroup& g : groups) {
    std::sort(g.paths.begin(), g.paths.end());
    finish_group(g, s);
    for (int b : g.obs)
      if (written.count(b)) g.out_accumulate.insert(b);
    written.insert(g.obs.begin(), g.obs.end());
  }
  return groups;
}

// Backward: a group owns whole edge blocks (gy of an edge is complete in
// registers and written once) and, when it fits, whole connected sets of input
// and edge blocks (gx complete too).  A connected set over budget is cut by
// edge block into groups of distinct phases; a later phase adds its share of
// gx to what an earlier one wrote.  Cutting by edge block keeps every
// per-edge row (y, w, gy, gw) read or written once; only the per-node rows
// (x, the g[dst] gather, gx) are touched by several phases.
std::vector<UGroup> backward_groups(const USpec& s, int* phases) {
  const int nx = (int)s.xblocks.size();
  std::vector<int> root(nx + s.yblocks.size());
  for (size_t n = 0; n < root.size(); ++n) root[n] = (int)n;
  std::function<int(int)> find = [&](int a) { return root[a] == a ? a : root[a] = find(root[a]); };
  for (const UPath& p : s.paths) root[find(p.xb)] = find(nx + p.yb);
  std::map<int, std::vector<int>> components;  // root -> edge blocks, in order
  std::vector<int> component_order;
  for (int b = 0; b < (int)s.yblocks.size(); ++b) {
    bool used = false;
    for (const UPath& p : s.paths) used |= p.yb == b;
    if (!used) continue;
    const int r = find(nx + b);
    if (!components.count(r)) component_order.push_back(r);
    components[r].push_back(b);
  }
  std::vector<UGroup> groups;
  *phases = 0;
  for (int r : component_order) {
    std::vector<std::vector<int>> parts;  // paths per cut
    std::vector<int> current;
    for (int b : components[r]) {
      std::vector<int> block;
      for (int p = 0; p < (int)s.paths.size(); ++p)
        if (s.paths[p].yb == b) block.push_back(p);
      std::vector<int> merged = current;
      merged.insert(merged.end(), block.begin(), block.end());
      if (!current.empty() && cost(s, merged, true) > kBackwardBudget) {
        parts.push_back(current);
        current = block;
      } else {
        current = merged;
      }
    }
    parts.push_back(current);
    std::set<int> written;
    for (size_t n = 0; n < parts.size(); ++n) {
      UGroup g;
      g.paths = parts[n];
      std::sort(g.paths.begin(), g.paths.end());
      g.phase = (int)n;
      finish_group(g, s);
      for (int b : g.xbs)
        if (written.count(b)) g.gx_accumulate.insert(b);
      written.insert(g.xbs.begin(), g.xbs.end());
      groups.push_back(g);
    }
    *phases = std::max(*phases, (int)parts.size());
  }
  return groups;
}

bool covers(std::vector<std::pair<long, long>> ranges, long total) {
  std::sort(ranges.begin(), ranges.end());
  long at = 0;
  for (const auto& r : ranges) {
    if (r.first > at) return false;
    at = std::max(at, r.second);
  }
  return at >= total;
}

// ---------------------------------------------------------------------------
// Emission
// ---------------------------------------------------------------------------

struct Code {
  std::ostringstream s;
  template <typename... A>
  __attribute__((format(printf, 2, 0))) void line(const char* fmt, A... args) {
    const int size = std::snprintf(nullptr, 0, fmt, args...);
    std::string buffer(size + 1, '\0');
    std::snprintf(&buffer[0], buffer.size(), fmt, args...);
    buffer.resize(size);
    s << buffer << '\n';
  }
};

std::string lit(double c, int bits) {
  char b[48];
  if (bits == 64)
    std::snprintf(b, sizeof(b), "%.17e", c);
  else
    std::snprintf(b, sizeof(b), "%.9ef", (double)(float)c);
  return b;
}

std::string prelude(const USpec& s, int edge_index_bits) {
  std::ostringstream o;
  o << "typedef " << (s.bits == 64 ? "double" : "float") << " real;\n";
  o << "typedef long long i64;\n";
  // Edge offsets: int32, or int64 for graphs of 2^31 or more edges.
  o << "typedef " << (edge_index_bits == 64 ? "long long" : "int") << " eix;\n";
  o << "#define FMA(a, b, c) " << (s.bits == 64 ? "__builtin_fma" : "__builtin_fmaf") << "((a), (b), (c))\n";
  o << "#define IN1 " << s.in1 << "LL\n#define IN2 " << s.in2 << "LL\n#define OUTD " << s.out
    << "LL\n#define WNUM " << s.wnum << "LL\n#define L0DIM " << s.l0 << "LL\n";
  // v[lane ^ M]: DPP for M = 1, 2, xor swizzle within 32 lanes up to 16, a
  // permute through the LDS crossbar for 32.
  o << R"(
template <int M>
__device__ __forceinline__ int lane_xor_bits(int v) {
  if constexpr (M == 1) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true);
  else if constexpr (M == 2) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true);
  else if constexpr (M < 32) return __builtin_amdgcn_ds_swizzle(v, 0x1F | (M << 10));
  else return __builtin_amdgcn_ds_bpermute((int)((threadIdx.x ^ 32u) << 2), v);
}
template <int M>
__device__ __forceinline__ float lane_xor(float v) { return __int_as_float(lane_xor_bits<M>(__float_as_int(v))); }
template <int M>
__device__ __forceinline__ double lane_xor(double v) {
  return __hiloint2double(lane_xor_bits<M>(__double2hiint(v)), lane_xor_bits<M>(__double2loint(v)));
}
)";
  return o.str();
}

// Components of each block a group reads, from its terms.
struct Uses {
  std::set<std::pair<int, int>> x, y, o;  // (block, component)
};

Uses uses_of(const USpec& s, const UGroup& g) {
  Uses u;
  for (int p : g.paths) {
    const UPath& q = s.paths[p];
    for (const UTerm& t : q.terms) {
      u.x.insert({q.xb, t.i});
      u.y.insert({q.yb, t.j});
      u.o.insert({q.ob, t.k});
    }
  }
  return u;
}


// Emits `real name = sum_n a_n * b_n` as one multiply and a chain of FMAs.
void fma_sum(Code& c, const std::string& name, const std::vector<std::pair<std::string, std::string>>& products) {
  if (products.empty()) {
    c.line("        const real %s = 0;", name.c_str());
    return;
  }
  c.line("        real %s = %s * %s;", name.c_str(), products[0].first.c_str(), products[0].second.c_str());
  for (size_t n = 1; n < products.size(); ++n)
    c.line("        %s = FMA(%s, %s, %s);", name.c_str(), products[n].first.c_str(), products[n].second.c_str(),
           name.c_str());
}

std::string sfx(int a, int b) { return std::to_string(a) + "_" + std::to_string(b); }

// Sum of `names` over the lanes whose bit `from`..32 differ (one exchange per bit).
void lane_sum(Code& c, const std::vector<std::string>& names, int from, int to, const char* indent) {
  for (int m = from; m <= to; m *= 2)
    for (const std::string& n : names) c.line("%s%s += lane_xor<%d>(%s);", indent, n.c_str(), m, n.c_str());
}

// Kernel head shared by both directions: workgroup -> (node, chunk); its
// `split` waves take interleaved runs of the node's edges; lane -> (sub, u).
void emit_head(Code& c, const char* order_name, int slots) {
  c.line("  const int item = blockIdx.x;");
  c.line("  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);");
  c.line("  const int lane = threadIdx.x & 63;");
  c.line("  const int slot = item %% %d;", slots);
  c.line("  const int node = %s[item / %d];", order_name, slots);
}

// Sums `names` over the waves of the workgroup through LDS (halving tree);
// wave 0 ends with the totals.  Every wave of the workgroup executes it.
void block_sum(Code& c, const std::vector<std::string>& names) {
  const int n = (int)names.size();
  c.line("    if (split > 1) {");
  c.line("      real* red = reinterpret_cast<real*>(lds);");
  c.line("      for (int h = split >> 1; h > 0; h >>= 1) {");
  c.line("        if (wave >= h && wave < 2 * h) {");
  for (int a = 0; a < n; ++a) c.line("          red[((wave - h) * %d + %d) * 64 + lane] = %s;", n, a, names[a].c_str());
  c.line("        }");
  c.line("        __syncthreads();");
  c.line("        if (wave < h) {");
  for (int a = 0; a < n; ++a) c.line("          %s += red[(wave * %d + %d) * 64 + lane];", names[a].c_str(), n, a);
  c.line("        }");
  c.line("        __syncthreads();");
  c.line("      }");
  c.line("    }");
}

void emit_group_lanes(Code& c, const UGroup& g) {
  int log = 0;
  while ((1 << log) < g.cw) ++log;
  c.line("    const int chunk = slot;");
  c.line("    const int u = chunk * 64 + (lane & %d);", g.cw - 1);
  c.line("    const int sub = lane >> %d;", log);
  c.line("    const bool act = u < %d;", g.ch);
}

// Loop of one wave over its runs of a node's edges, nsub at once; the lane's edge is
// `name` where that lies before `end`.  Positions are 64-bit: as int32 those past
// the end, up to 575 ahead, would wrap to negative ones near 2^31 edges.
void emit_edge_loop(Code& c, int nsub, const char* name) {
  c.line("    for (i64 e0 = (i64)beg + wave * %d; e0 < end; e0 += %d * split) {", nsub, nsub);
  c.line("      const i64 %s = e0 + sub;", name);
}

// t{p}_k = sum_{(i,j,k)} c x_i y_j of path p, as sum_i x_i z_ik.
void emit_t(Code& c, const USpec& s, int p) {
  const UPath& q = s.paths[p];
  std::map<int, std::map<int, std::vector<const UTerm*>>> by_ik;  // i -> k -> terms
  std::set<int> ks;
  for (const UTerm& t : q.terms) {
    by_ik[t.i][t.k].push_back(&t);
    ks.insert(t.k);
  }
  for (int k : ks) c.line("        real t%d_%d = 0;", p, k);
  for (const auto& ik : by_ik)
    for (const auto& kv : ik.second) {
      std::vector<std::pair<std::string, std::string>> products;
      for (const UTerm* t : kv.second) products.push_back({lit(t->c, s.bits), "y" + sfx(q.yb, t->j)});
      const std::string z = "z" + std::to_string(p) + "_" + sfx(ik.first, kv.first);
      fma_sum(c, z, products);
      c.line("        t%d_%d = FMA(x%d_%d, %s, t%d_%d);", p, kv.first, q.xb, ik.first, z.c_str(), p, kv.first);
    }
}

// r{tag}{p}_ij = sum_k c_ijk seed(k), then sx{tag}{p}_i = sum_j y_j r_ij,
// sy{tag}{p}_j = sum_i x_i r_ij and S{tag}{p} = sum_i x_i sx_i as requested.
void emit_r_sums(Code& c, const USpec& s, int p, const std::string& tag, const std::function<std::string(int)>& seed,
                 bool want_sx, bool want_sy, bool want_s) {
  const UPath& q = s.paths[p];
  const std::string P = tag + std::to_string(p);
  std::map<std::pair<int, int>, std::vector<const UTerm*>> by_ij;
  for (const UTerm& t : q.terms) by_ij[{t.i, t.j}].push_back(&t);
  std::map<int, std::vector<std::pair<std::string, std::string>>> rows, cols;
  for (const auto& kv : by_ij) {
    const int i = kv.first.first, j = kv.first.second;
    std::vector<std::pair<std::string, std::string>> products;
    for (const UTerm* t : kv.second) products.push_back({lit(t->c, s.bits), seed(t->k)});
    const std::string r = "r" + P + "_" + sfx(i, j);
    fma_sum(c, r, products);
    rows[i].push_back({"y" + sfx(q.yb, j), r});
    cols[j].push_back({"x" + sfx(q.xb, i), r});
  }
  std::vector<std::pair<std::string, std::string>> total;
  if (want_sx || want_s)
    for (const auto& kv : rows) {
      const std::string name = "sx" + P + "_" + std::to_string(kv.first);
      fma_sum(c, name, kv.second);
      total.push_back({"x" + sfx(q.xb, kv.first), name});
    }
  if (want_sy)
    for (const auto& kv : cols) fma_sum(c, "sy" + P + "_" + std::to_string(kv.first), kv.second);
  if (want_s) fma_sum(c, "S" + P, total);
}

std::string emit_forward(const UuuPlan& plan, bool env, bool l0) {
  const USpec& s = plan.spec;
  Code c;
  c.s << prelude(s, plan.edge_index_bits);
  for (size_t gi = 0; gi < plan.fwd.size(); ++gi) {
    const UGroup& g = plan.fwd[gi];
    const Uses use = uses_of(s, g);
    const int nsub = 64 / g.cw;
    c.line("extern \"C\" __global__ void __launch_bounds__(512) luna_uuu_fwd_g%d(", (int)gi);
    c.line("    const real* __restrict__ x, const real* __restrict__ y, const real* __restrict__ w,");
    c.line("    const real* __restrict__ env, const int* __restrict__ src, const eix* __restrict__ rowptr,");
    c.line("    const int* __restrict__ order, real* __restrict__ out, real* __restrict__ l0, int split) {");
    c.line("  extern __shared__ __align__(16) unsigned char lds[];");
    emit_head(c, "order", g.chunks);
    c.line("  const eix beg = rowptr[node], end = rowptr[node + 1];");
    c.line("  {");
    emit_group_lanes(c, g);
    std::vector<std::string> accs;
    for (int b : g.obs)
      for (int k = 0; k < s.oblocks[b].d; ++k) {
        accs.push_back("o" + std::to_string(b) + "_" + std::to_string(k));
        c.line("    real %s = 0;", accs.back().c_str());
      }
    emit_edge_loop(c, nsub, "e");
    c.line("      if (act && e < end) {");
    c.line("        const i64 sn = src[e];");
    for (int b : g.xbs)
      c.line("        const real* xr%d = x + sn * IN1 + %d + (i64)u * %d;", b, s.xblocks[b].off, s.xblocks[b].d);
    for (int b : g.ybs)
      c.line("        const real* yr%d = y + (i64)e * IN2 + %d + (i64)u * %d;", b, s.yblocks[b].off, s.yblocks[b].d);
    for (const auto& xi : use.x) c.line("        const real x%d_%d = xr%d[%d];", xi.first, xi.second, xi.first, xi.second);
    for (const auto& yj : use.y)
      c.line("        const real y%d_%d = __builtin_nontemporal_load(yr%d + %d);", yj.first, yj.second, yj.first,
             yj.second);
    if (env) c.line("        const real ev = env[e];");
    for (int p : g.paths)
      if (s.paths[p].w_off >= 0)
        c.line("        const real w%d = __builtin_nontemporal_load(w + (i64)e * WNUM + %d + u);", p, s.paths[p].w_off);
    // t_k = sum_i x_i z_ik with z_ik = sum_j c_ijk y_j: one FMA per term and
    // one per (i, k), and nothing lives beyond its path.
    for (int p : g.paths) {
      const UPath& q = s.paths[p];
      if (q.terms.empty()) {
        if (l0 && q.l0_col >= 0) c.line("        l0[(i64)e * L0DIM + %d + u] = 0;", q.l0_col);
        continue;
      }
      emit_t(c, s, p);
      std::set<int> ks;
      for (const UTerm& t : q.terms) ks.insert(t.k);
      std::string scale = q.w_off >= 0 ? "w" + std::to_string(p) : "";
      if (env) scale = scale.empty() ? "ev" : "ev * " + scale;
      if (!scale.empty()) c.line("        const real a%d = %s;", p, scale.c_str());
      for (int k : ks) {
        if (scale.empty())
          c.line("        o%d_%d += t%d_%d;", q.ob, k, p, k);
        else
          c.line("        o%d_%d = FMA(a%d, t%d_%d, o%d_%d);", q.ob, k, p, p, k, q.ob, k);
      }
      if (l0 && q.l0_col >= 0) {
        std::string v = ks.count(0) ? "t" + std::to_string(p) + "_0" : "(real)0";
        if (q.w_off >= 0 && ks.count(0)) v = "w" + std::to_string(p) + " * " + v;
        c.line("        l0[(i64)e * L0DIM + %d + u] = %s;", q.l0_col, v.c_str());
      }
    }
    c.line("      }");
    c.line("    }");
    if (nsub > 1) lane_sum(c, accs, g.cw, 32, "    ");
    block_sum(c, accs);
    c.line("    if (wave == 0 && sub == 0 && act) {");
    c.line("      real* orow = out + (i64)node * OUTD;");
    for (int b : g.obs)
      for (int k = 0; k < s.oblocks[b].d; ++k)
        c.line("      orow[%d + u * %d] %s o%d_%d;", s.oblocks[b].off + k, s.oblocks[b].d,
               g.out_accumulate.count(b) ? "+=" : "=", b, k);
    c.line("    }");
    c.line("  }");
    c.line("}");
  }
  return c.s.str();
}

// Backward groups held to three waves per SIMD (168 registers).  Left alone, the
// compiler hoists every load of the lmax-3 group and takes 251 registers, two
// waves: 64 channels, 2,083 nodes, 109,000 edges, step 804 us, at three waves
// with 8 registers spilled 677 us; 10,000 nodes, 300,000 edges 2,101 and 1,897
// us; 192 channels 2,272 and 2,010 us.  Only where every lane of every chunk has a
// channel: with 8-32 channels (two to eight edges of a wave at once) the step took 10 to
// 20 % longer, with 40, 80 and 96 up to 5, 3 and 9 %, with 128 between 7 %
// less and 2 % more.  Blocks wider than 7 components spill 46 to
// 240 registers at three waves, fp64 groups up to 31: left as they are, like the
// groups whose estimate says that they fit by themselves (lmax 2: 56, 95
// registers, which the hint would raise to 124).
bool three_waves(const USpec& s, const UGroup& g) {
  bool narrow = s.bits == 32 && g.ch % 64 == 0 && cost(s, g.paths, true) > 80;
  for (int b : g.xbs) narrow = narrow && s.xblocks[b].d <= 7;
  for (int b : g.ybs) narrow = narrow && s.yblocks[b].d <= 7;
  for (int b : g.obs) narrow = narrow && s.oblocks[b].d <= 7;
  return narrow;
}

std::string emit_backward(const UuuPlan& plan, bool env, bool gl0, bool want_gx, bool want_gy,
                          bool want_gw, bool want_genv) {
  const USpec& s = plan.spec;
  Code c;
  c.s << prelude(s, plan.edge_index_bits);
  for (size_t gi = 0; gi < plan.bwd.size(); ++gi) {
    const UGroup& g = plan.bwd[gi];
    const Uses use = uses_of(s, g);
    const int nsub = 64 / g.cw;
    c.line("extern \"C\" __global__ void __launch_bounds__(512) %sluna_uuu_bwd_g%d(",
           three_waves(s, g) ? "__attribute__((amdgpu_waves_per_eu(3))) " : "", (int)gi);
    c.line("    const real* __restrict__ x, const real* __restrict__ y, const real* __restrict__ w,");
    c.line("    const real* __restrict__ env, const real* __restrict__ g, const real* __restrict__ gl0,");
    c.line("    const int* __restrict__ dst, const eix* __restrict__ rowptr, const eix* __restrict__ edge_ids,");
    c.line("    const int* __restrict__ order, real* __restrict__ gx, real* gy, real* __restrict__ gw,");
    c.line("    real* __restrict__ part, int split, i64 num_edges) {");
    c.line("  extern __shared__ __align__(16) unsigned char lds[];");
    emit_head(c, "order", g.chunks);
    c.line("  const eix beg = rowptr[node], end = rowptr[node + 1];");
    c.line("  {");
    emit_group_lanes(c, g);
    // The source row's input blocks, once.
    for (const auto& xi : use.x) c.line("    real x%d_%d = 0;", xi.first, xi.second);
    c.line("    if (act) {");
    for (const auto& xi : use.x)
      c.line("      x%d_%d = x[(i64)node * IN1 + %d + (i64)u * %d];", xi.first, xi.second,
             s.xblocks[xi.first].off + xi.second, s.xblocks[xi.first].d);
    c.line("    }");
    std::vector<std::string> gxs;
    if (want_gx)
      for (int b : g.xbs)
        for (int i = 0; i < s.xblocks[b].d; ++i) {
          gxs.push_back("gx" + std::to_string(b) + "_" + std::to_string(i));
          c.line("    real %s = 0;", gxs.back().c_str());
        }
    emit_edge_loop(c, nsub, "pos");
    c.line("      const eix e = pos < end ? edge_ids[pos] : 0;");
    if (want_genv) c.line("      real gev = 0;");
    c.line("      if (act && pos < end) {");
    c.line("        const i64 dn = dst[e];");
    for (const auto& yj : use.y)
      c.line("        const real y%d_%d = __builtin_nontemporal_load(y + (i64)e * IN2 + %d + (i64)u * %d);", yj.first,
             yj.second, s.yblocks[yj.first].off + yj.second, s.yblocks[yj.first].d);
    for (const auto& ok : use.o)
      c.line("        const real g%d_%d = g[dn * OUTD + %d + (i64)u * %d];", ok.first, ok.second,
             s.oblocks[ok.first].off + ok.second, s.oblocks[ok.first].d);
    if (env) c.line("        const real ev = env[e];");
    for (int p : g.paths)
      if (s.paths[p].w_off >= 0 && (want_gx || want_gy || want_genv))
        c.line("        const real w%d = __builtin_nontemporal_load(w + (i64)e * WNUM + %d + u);", p, s.paths[p].w_off);
    if (want_gy)
      for (int b : g.ybs)
        for (int j = 0; j < s.yblocks[b].d; ++j) c.line("        real gy%d_%d = 0;", b, j);
    // Per path, with r_ij = sum_k c_ijk seed_k:
    //   sx_i = sum_j y_j r_ij (gx), sy_j = sum_i x_i r_ij (gy), S = sum_i x_i sx_i (gw).
    // The seed is the raw g and the scale env * w is applied to the sums, except
    // on scalar paths with an l0 seed, whose seed is env * g + gl0.
    for (int p : g.paths) {
      const UPath& q = s.paths[p];
      const std::string P = std::to_string(p);
      if (q.terms.empty()) {
        if (want_gw && q.w_off >= 0)
          c.line("        __builtin_nontemporal_store((real)0, gw + (i64)e * WNUM + %d + u);", q.w_off);
        continue;
      }
      const bool l0path = gl0 && q.l0_col >= 0;
      const std::string w = q.w_off >= 0 ? "w" + P : "";
      auto raw = [&](int k) { return "g" + sfx(q.ob, k); };
      std::string seed0;
      if (l0path) {
        c.line("        const real Gl%d = %s + gl0[(i64)e * L0DIM + %d + u];", p,
               env ? ("ev * " + raw(0)).c_str() : raw(0).c_str(), q.l0_col);
        seed0 = "Gl" + P;
      }
      // Scale of the sums: w * env for raw seeds, w for the l0 seed.
      std::string scale = w;
      if (env && !l0path) scale = scale.empty() ? "ev" : "ev * " + scale;
      if (!scale.empty() && (want_gx || want_gy)) c.line("        const real a%d = %s;", p, scale.c_str());
      const bool need_s = want_gw || (want_genv && !l0path);
      emit_r_sums(c, s, p, "", [&](int k) { return (l0path && k == 0) ? seed0 : raw(k); }, want_gx || need_s,
                  want_gy, need_s);
      auto add = [&](const char* acc, int blk, int idx, const std::string& v) {
        if (scale.empty())
          c.line("        %s%d_%d += %s;", acc, blk, idx, v.c_str());
        else
          c.line("        %s%d_%d = FMA(a%d, %s, %s%d_%d);", acc, blk, idx, p, v.c_str(), acc, blk, idx);
      };
      std::set<int> is, js;
      for (const UTerm& t : q.terms) {
        is.insert(t.i);
        js.insert(t.j);
      }
      if (want_gx)
        for (int i : is) add("gx", q.xb, i, "sx" + P + "_" + std::to_string(i));
      if (want_gy)
        for (int j : js) add("gy", q.yb, j, "sy" + P + "_" + std::to_string(j));
      if (want_gw && q.w_off >= 0) {
        const std::string v = (env && !l0path) ? "ev * S" + P : "S" + P;
        c.line("        __builtin_nontemporal_store(%s, gw + (i64)e * WNUM + %d + u);", v.c_str(), q.w_off);
      }
      if (want_genv) {
        // d out / d env = w * sum_ijk c x_i y_j g_k with the raw seed.
        std::string total = "S" + P;
        if (l0path) {
          emit_r_sums(c, s, p, "0", raw, true, false, true);
          total = "S0" + P;
        }
        if (w.empty())
          c.line("        gev += %s;", total.c_str());
        else
          c.line("        gev = FMA(%s, %s, gev);", w.c_str(), total.c_str());
      }
    }
    if (want_gy)
      for (int b : g.ybs)
        for (int j = 0; j < s.yblocks[b].d; ++j) {
          const long off = s.yblocks[b].off + j;
          c.line("        gy[(i64)e * IN2 + %ld + (i64)u * %d] = gy%d_%d;", off, s.yblocks[b].d, b, j);
        }
    c.line("      }");
    if (want_genv) {
      // Sum over the channels of this sub-group's edge; its first lane writes.
      if (g.cw > 1) lane_sum(c, {"gev"}, 1, g.cw / 2, "      ");
      c.line("      if ((lane & %d) == 0 && pos < end) part[(i64)(%d + chunk) * num_edges + e] = gev;", g.cw - 1,
             g.genv_slot);
    }
    c.line("    }");
    if (want_gx) {
      if (nsub > 1) lane_sum(c, gxs, g.cw, 32, "    ");
      block_sum(c, gxs);
      c.line("    if (wave == 0 && sub == 0 && act) {");
      c.line("      real* xrow = gx + (i64)node * IN1;");
      for (int b : g.xbs)
        for (int i = 0; i < s.xblocks[b].d; ++i)
          c.line("      xrow[%d + u * %d] %s gx%d_%d;", s.xblocks[b].off + i, s.xblocks[b].d,
                 g.gx_accumulate.count(b) ? "+=" : "=", b, i);
      c.line("    }");
    }
    c.line("  }");
    c.line("}");
  }
  // Sum of the env-gradient partial slots.
  c.line("extern \"C\" __global__ void __launch_bounds__(256) luna_uuu_genv_reduce(const real* __restrict__ part,");
  c.line("    real* __restrict__ genv, i64 num_edges) {");
  c.line("  const i64 e = (i64)blockIdx.x * 256 + threadIdx.x;");
  c.line("  if (e >= num_edges) return;");
  c.line("  real acc = 0;");
  c.line("  for (int n = 0; n < %d; ++n) acc += part[(i64)n * num_edges + e];", plan.genv_slots);
  c.line("  genv[e] = acc;");
  c.line("}");
  return c.s.str();
}

std::string source_for(const UuuPlan& plan, const std::string& v) {
  // fwd<env><l0>; bwd<env><gl0><gx><gy><gw><genv>
  auto flag = [&](size_t i) { return v.size() > i && v[i] == '1'; };
  if (v.compare(0, 3, "fwd") == 0) return emit_forward(plan, flag(3), flag(4));
  return emit_backward(plan, flag(3), flag(4), flag(5), flag(6), flag(7), flag(8));
}

void check_sizes(const UuuPlan& plan, int64_t num_nodes, int64_t num_edges) {
  if (num_nodes < 0 || num_edges < 0) fail("negative problem size");
  if (num_nodes > 0x7fffffffLL) fail("graph node count exceeds signed int32 capacity");
  if (plan.edge_index_bits == 32 && num_edges > 0x7fffffffLL)
    fail("a graph of 2^31 or more edges needs a plan with 64-bit edge offsets (luna_uuu_plan_create_ex)");
}

unsigned blocks_for(int64_t items) {
  if (items > 0x7fffffffLL) fail("uuu: launch grid exceeds 2^31 workgroups");
  return (unsigned)items;
}

size_t lds_bytes(int split, int accumulators, int bits) {
  return split > 1 ? (size_t)(split / 2) * accumulators * 64 * (bits / 8) : 0;
}

// Waves per workgroup sharing one node's edges: enough workgroups times waves
// to give every SIMD of the chip about eight waves, at most 8 per node, and
// no more than 64 KiB of LDS for the partial sums.
int split_for(int64_t workgroups, int accumulators, int bits) {
  int split = 1;
  while (split < 8 && workgroups * split < 8192 && lds_bytes(split * 2, accumulators, bits) <= 65536) split *= 2;
  return split;
}

}  // namespace
}  // namespace luna

using namespace luna;

struct LunaUuuPlan {
  UuuPlan plan;
};

extern "C" {

int luna_uuu_plan_create(const char* spec, const char* cache_dir, LunaUuuPlan** out) {
  return luna_uuu_plan_create_ex(spec, cache_dir, 32, out);
}

int luna_uuu_plan_create_ex(const char* spec, const char* cache_dir, int edge_index_bits, LunaUuuPlan** out) {
  return guard_call([&] {
    if (!spec || !out) fail("luna_uuu_plan_create: null argument");
    if (edge_index_bits != 32 && edge_index_bits != 64) fail("luna_uuu_plan_create_ex: edge_index_bits must be 32 or 64");
    auto holder = std::make_unique<LunaUuuPlan>();
    UuuPlan& p = holder->plan;
    p.edge_index_bits = edge_index_bits;
    p.spec = parse(spec);
    p.kernels.cache_dir = cache_dir ? cache_dir : "";
    p.kernels.tag = "uuu";
    const USpec& s = p.spec;
    if (!s.paths.empty()) {
      p.fwd = forward_groups(s);
      p.bwd = backward_groups(s, &p.bwd_phases);
      // Launch order: by phase (a later phase adds to the gy an earlier one wrote).
      std::stable_sort(p.bwd.begin(), p.bwd.end(), [](const UGroup& a, const UGroup& b) { return a.phase < b.phase; });
      for (UGroup& g : p.bwd) {
        g.genv_slot = p.genv_slots;
        p.genv_slots += g.chunks;
      }
    }
    std::vector<std::pair<long, long>> xs, ys, os, ws;
    for (const UPath& q : s.paths) {
      xs.push_back({q.x_off, q.x_off + (long)q.ch * q.d1});
      ys.push_back({q.y_off, q.y_off + (long)q.ch * q.d2});
      os.push_back({q.out_off, q.out_off + (long)q.ch * q.d3});
      if (q.w_off >= 0) ws.push_back({q.w_off, q.w_off + q.ch});
    }
    p.out_zero = !covers(os, s.out);
    p.gx_zero = !covers(xs, s.in1);
    p.gy_zero = !covers(ys, s.in2);
    p.gw_zero = !covers(ws, s.wnum);
    *out = holder.release();
  });
}

int luna_uuu_plan_destroy(LunaUuuPlan* plan) {
  return guard_call([&] { delete plan; });
}

int luna_uuu_plan_needs_zero(const LunaUuuPlan* plan, int32_t* flags) {
  return guard_call([&] {
    if (!plan || !flags) fail("luna_uuu_plan_needs_zero: null argument");
    const UuuPlan& p = plan->plan;
    flags[0] = p.out_zero;
    flags[1] = p.gx_zero;
    flags[2] = p.gy_zero;
    flags[3] = p.gw_zero;
  });
}

int luna_uuu_plan_precompile(LunaUuuPlan* plan) {
  return guard_call([&] {
    if (!plan) fail("luna_uuu_plan_precompile: null plan");
    UuuPlan& p = plan->plan;
    if (p.spec.paths.empty()) return;
    for (const std::string v : {"fwd00", "bwd001110"}) p.kernels.code_for(v, [&] { return source_for(p, v); });
  });
}

int luna_uuu_conv_fwd(const LunaUuuPlan* cplan, const void* x, const void* y, const void* w, const void* env,
                      const int32_t* src, const void* dst_rowptr, const int32_t* node_order, void* out, void* l0,
                      int64_t num_nodes, int64_t num_edges, LunaStream stream) {
  return guard_call([&] {
    if (!cplan) fail("luna_uuu_conv_fwd: null plan");
    UuuPlan& p = const_cast<LunaUuuPlan*>(cplan)->plan;
    check_sizes(p, num_nodes, num_edges);
    if (num_nodes == 0 || p.spec.paths.empty()) return;
    if (!x || !out || !dst_rowptr || !node_order) fail("luna_uuu_conv_fwd: null tensor");
    if (num_edges > 0 && (!y || !src || (p.spec.wnum > 0 && !w))) fail("luna_uuu_conv_fwd: null edge tensor");
    if (l0 && p.spec.l0 == 0) l0 = nullptr;
    auto kernel = [&](size_t gi) {
      return p.kernels.function(
          (uint64_t)gi << 8 | (uint64_t)(env != nullptr) << 1 | (uint64_t)(l0 != nullptr),
          [&] { return std::string("fwd") + (env ? '1' : '0') + (l0 ? '1' : '0'); },
          [&](const std::string& v) { return source_for(p, v); },
          [&] { return "luna_uuu_fwd_g" + std::to_string(gi); });
    };
    for (size_t gi = 0; gi < p.fwd.size(); ++gi) {
      const UGroup& g = p.fwd[gi];
      const int64_t items = num_nodes * g.chunks;
      int accs = 0;
      for (int b : g.obs) accs += p.spec.oblocks[b].d;
      int split = split_for(items, accs, p.spec.bits);
      void* args[] = {&x, &y, &w, &env, &src, &dst_rowptr, &node_order, &out, &l0, &split};
      launch("uuu_fwd", kernel(gi), dim3(blocks_for(items)),
             dim3(64 * split), (hipStream_t)stream, args, (unsigned)lds_bytes(split, accs, p.spec.bits));
    }
  });
}

int luna_uuu_conv_bwd_workspace(const LunaUuuPlan* plan, int64_t num_nodes, int64_t num_edges, size_t* bytes) {
  return guard_call([&] {
    if (!plan || !bytes) fail("luna_uuu_conv_bwd_workspace: null argument");
    check_sizes(plan->plan, num_nodes, num_edges);
    const UuuPlan& p = plan->plan;
    // Partial slots of the env gradient, needed only when several wave bodies share an edge.
    *bytes = p.genv_slots > 1 ? (size_t)p.genv_slots * (size_t)num_edges * (p.spec.bits / 8) : 0;
  });
}

int luna_uuu_conv_bwd(const LunaUuuPlan* cplan, const void* x, const void* y, const void* w, const void* env,
                      const void* g, const void* gl0, const int32_t* dst, const void* src_rowptr,
                      const void* edge_ids_by_src, const int32_t* source_node_order, void* gx, void* gy, void* gw,
                      void* genv, void* workspace, size_t workspace_bytes, int64_t num_nodes, int64_t num_edges,
                      LunaStream stream) {
  return guard_call([&] {
    if (!cplan) fail("luna_uuu_conv_bwd: null plan");
    UuuPlan& p = const_cast<LunaUuuPlan*>(cplan)->plan;
    check_sizes(p, num_nodes, num_edges);
    if (num_nodes == 0 || p.spec.paths.empty()) return;
    if (!x || !g || !src_rowptr || !source_node_order) fail("luna_uuu_conv_bwd: null tensor");
    if (num_edges > 0 && (!y || !dst || !edge_ids_by_src || (p.spec.wnum > 0 && !w)))
      fail("luna_uuu_conv_bwd: null edge tensor");
    if (gl0 && p.spec.l0 == 0) gl0 = nullptr;
    if (!env) genv = nullptr;
    int64_t E = num_edges;
    if (E == 0) gy = gw = genv = nullptr;  // nothing per edge; gx is still written (zeros)
    if (!gx && !gy && !gw && !genv) return;
    void* part = nullptr;
    if (genv) {
      if (p.genv_slots > 1) {
        const size_t need = (size_t)p.genv_slots * (size_t)E * (p.spec.bits / 8);
        if (!workspace || workspace_bytes < need) fail("luna_uuu_conv_bwd: workspace too small");
        part = workspace;
      } else {
        part = genv;
      }
    }
    const hipStream_t s = (hipStream_t)stream;
    const void* const flags[] = {env, gl0, gx, gy, gw, genv};
    uint64_t code = 1 << 7;
    for (int n = 0; n < 6; ++n) code |= (uint64_t)(flags[n] != nullptr) << n;
    auto kernel = [&](size_t gi, const char* name) {
      return p.kernels.function(
          (uint64_t)gi << 8 | code,
          [&] {
            std::string v = "bwd";
            for (const void* f : flags) v += f ? '1' : '0';
            return v;
          },
          [&](const std::string& v) { return source_for(p, v); },
          [&] { return gi == p.bwd.size() ? std::string(name) : name + std::to_string(gi); });
    };
    for (size_t gi = 0; gi < p.bwd.size(); ++gi) {
      const UGroup& grp = p.bwd[gi];
      const int64_t items = num_nodes * grp.chunks;
      int accs = 0;
      if (gx)
        for (int b : grp.xbs) accs += p.spec.xblocks[b].d;
      int split = split_for(items, accs, p.spec.bits);
      void* args[] = {&x, &y, &w, &env, &g, &gl0, &dst, &src_rowptr, &edge_ids_by_src, &source_node_order,
                      &gx, &gy, &gw, &part, &split, &E};
      launch("uuu_bwd", kernel(gi, "luna_uuu_bwd_g"), dim3(blocks_for(items)),
             dim3(64 * split), s, args, (unsigned)lds_bytes(split, accs, p.spec.bits));
    }
    if (genv && p.genv_slots > 1) {
      void* args[] = {&part, &genv, &E};
      launch("uuu_genv_reduce", kernel(p.bwd.size(), "luna_uuu_genv_reduce"), dim3((unsigned)((E + 255) / 256)),
             dim3(256), s, args);
    }
  });
}

}  // extern "C"
