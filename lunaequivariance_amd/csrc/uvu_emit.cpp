// HIP source emitter for the UVU convolution kernels of one path set.
//
// Every Clebsch-Gordan coefficient becomes a literal in straight-line code, so
// a wave holds all partial products and output accumulators of its group in
// VGPRs while edge attributes and graph indices, which are uniform across the
// wave, come through scalar loads.  One lane owns one channel u of a
// 64-channel chunk.  Edge loops are software-pipelined: the gathered source
// row and the weight row of edge e+1 are in flight while edge e is computed.
//
// Forward (dst-owned, as the reference's ordered forward kernel,
// src/lunatp/uvu_conv/kernels/forward.py:398-427):
//   out[t, ob + u*d3 + k] = sum_{e in row t} env[e] * w[e, wo + u*ws]
//                           * sum_{(i,j,k)} c_ijk x[src[e], xb + u*d1 + i] y[e, yb + j]
// Backward (the math of src/lunatp/uvu_conv/kernels/backward.py:183-333, but
// destination-owned so the wide output seed g[t] is read once per node):
//   q_ij = sum_k c_ijk G_k with G = env[e] * g[t] (+ gl0 for scalar paths)
//   gw[e, wo + u*ws] = sum_ij x_i y_j q_ij
//   msg[e, xb + u*d1 + i] = w sum_j y_j q_ij;  gx[s] = sum_{e: src[e]=s} msg[e]
//   gy[e, yb + j] = sum_u w sum_i x_i q_ij      (partials per wave, then reduced)
//   genv[e] = sum_u sum_k w g_k t_k, t_k = sum c x_i y_j
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <set>
#include <sstream>
#include <tuple>

#include "uvu_plan.h"

namespace luna {

namespace {

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
  void raw(const std::string& text) { s << text; }
};

// Emission switches, overridable through LUNAEQ_AMD_EMIT="fpre=1,bpre=2,hoist=1,fwpe=2,bwpe=2".
struct Options {
  int fwd_prefetch = 1;  // edge-loop software pipelining depth (0 none, 1 x/w, 2 all operands)
  int bwd_prefetch = 2;
  int prefetch = 0;      // the level of the kernel being emitted
  int packed_prefetch = 2;  // the level of packed and split forward groups
  int fwd_depth = 1;     // edges in flight with prefetch level 2 (1 or 2)
  int bwd_depth = 1;
  int depth = 1;
  bool fwd_nt_w = true;  // stream the per-edge weights with non-temporal loads
  int bwd_nt_w = -1;     // -1: on for fp32, off for fp64 (measured: fp32 -2.6 %, fp64 +15 %)
  bool nt_w = false;     // the setting of the kernel being emitted
  bool nt_gw = true;     // non-temporal stores of the weight gradient
  int nt_msg = 1;        // non-temporal stores of the gx messages (fp64 config 3: backward
                         // 18.57 -> 18.39 ms in interleaved in-process pairs; fp32 9.29 -> 9.05)
  int y_vgpr = -1;       // copy y into vector registers before use (a scalar
                         // operand makes an fp32 FMA issue 1.45x slower); -1: in
                         // the fp32 forward only (fp64 without the copies:
                         // forward 9.7 -> 8.9 ms, backward unchanged; fp32
                         // backward without them 8.66 -> 8.59 ms, 162 -> 155
                         // VGPRs, interleaved in-process pairs; fp32 forward
                         // the same either way)
  bool hoist = false;    // let the backward hoist edge-invariant q_ij out of the edge loop
  int lds_reduce = -1;   // gy partials summed over the 64 lanes through LDS (1) or by a
                         // butterfly of lane exchanges (0); -1: LDS (fp64 backward
                         // 18.7 -> 17.8 ms; fp32 config 2 8.86 -> 8.77 and 9.27 -> 9.17 ms
                         // in interleaved in-process pairs)
  int hoist_regs = -1;   // registers the backward may spend on q classes computed once
                         // per node instead of per edge (-1: by precision)
  int fwd_local = 0;     // forward in per-path form (no products shared between
                         // paths): fewer registers, more arithmetic; 1 on, 0 off
                         // (fp64 measured 10.5 -> 10.0 ms with it off)
  int fwd_wpe = 0;       // amdgpu_waves_per_eu hint for the forward (0 = none)
  int bwd_wpe = 0;       // same for the backward
  bool nt_out = true;     // forward: non-temporal output stores
  bool out_lds = true;     // forward: output blocks leave through LDS as contiguous stores
  bool gather_nt = true;   // gx gather: non-temporal loads of the messages (read once)
  int gather_unroll = 4;   // gx gather: message rows in flight per thread
};

Options options() {
  Options o;
  const char* text = std::getenv("LUNAEQ_AMD_EMIT");
  if (!text) return o;
  std::string s(text);
  auto value = [&](const char* key, int fallback) {
    std::string k = std::string(key) + "=";
    size_t at = s.find(k);
    return at == std::string::npos ? fallback : std::atoi(s.c_str() + at + k.size());
  };
  o.fwd_prefetch = value("fpre", o.fwd_prefetch);
  o.packed_prefetch = value("ppre", o.packed_prefetch);
  o.fwd_depth = value("fdepth", o.fwd_depth);
  o.bwd_depth = value("bdepth", o.bwd_depth);
  o.fwd_nt_w = value("fntw", o.fwd_nt_w) != 0;
  o.bwd_nt_w = value("bntw", o.bwd_nt_w);
  o.nt_gw = value("ntgw", o.nt_gw) != 0;
  o.nt_msg = value("ntmsg", o.nt_msg);
  o.y_vgpr = value("yv", o.y_vgpr);
  o.fwd_local = value("flocal", o.fwd_local);
  o.bwd_prefetch = value("bpre", o.bwd_prefetch);
  o.hoist = value("hoist", o.hoist) != 0;
  o.hoist_regs = value("hq", o.hoist_regs);
  o.lds_reduce = value("lred", o.lds_reduce);
  o.fwd_wpe = value("fwpe", o.fwd_wpe);
  o.bwd_wpe = value("bwpe", o.bwd_wpe);
  o.out_lds = value("olds", o.out_lds) != 0;
  o.nt_out = value("ntout", o.nt_out) != 0;
  o.gather_nt = value("gnt", o.gather_nt) != 0;
  o.gather_unroll = std::max(1, std::min(16, value("gun", o.gather_unroll)));
  return o;
}

std::string literal(double c, int bits) {
  char buffer[64];
  if (bits == 64) {
    // Wrapped so that each use materialises its constant where it is used (see
    // KC in the prelude).
    std::snprintf(buffer, sizeof(buffer), "%.17e", c);
  } else {
    std::snprintf(buffer, sizeof(buffer), "%.9ef", (double)(float)c);
  }
  return buffer;
}

std::string prelude(const Spec& spec, int edge_index_bits) {
  std::ostringstream s;
  const bool fp64 = spec.dtype_bits == 64;
  s << "typedef " << (fp64 ? "double" : "float") << " real;\n";
  s << "typedef long long i64;\n";
  // Edge offsets (row pointers, edge ids, edge loop counters): int32, or
  // int64 for graphs of 2^31 or more edges.  Node ids stay int32.
  s << "typedef " << (edge_index_bits == 64 ? "long long" : "int") << " eix;\n";
  s << "#define FMA(a, b, c) " << (fp64 ? "__builtin_fma" : "__builtin_fmaf") << "((a), (b), (c))\n";
  s << "#define IN1 " << spec.in1 << "LL\n";
  s << "#define IN2 " << spec.in2 << "LL\n";
  s << "#define OUTD " << spec.out << "LL\n";
  s << "#define WNUM " << spec.wnum << "LL\n";
  // Row stride of the weights read per edge: 0 when one row serves every edge.
  s << "#define WROW " << (spec.w_broadcast ? "0LL" : "WNUM") << "\n";
  s << "#define L0DIM " << spec.l0_dim << "LL\n";
  s << "#define PART_W " << spec.in2 + 1 << "LL\n";
  // Edges are compared by distances: with int32 offsets a position past `end`
  // wraps to a negative one where a graph has almost 2^31 edges.
  s << "__device__ __forceinline__ eix edge_at(eix from, int ahead, eix end) {"
       " return end - from > ahead ? from + ahead : end - 1; }\n";
  if (fp64) {
    // A double literal cannot be an instruction operand: it lives in a scalar
    // register pair.  Left alone, the compiler hoists all of a kernel's
    // coefficients out of the edge loop and spills scalar registers into
    // vector lanes; the opaque copy keeps each one local to its use.
    s << "__device__ __forceinline__ double KC(double v) { asm volatile(\"\" : \"+s\"(v)); return v; }\n";
  }
  // Lane exchange v[lane ^ M]: DPP quad permutes for M = 1, 2, a swizzle for
  // M = 4..16 (within 32 lanes) and a permute through LDS hardware for M = 32.
  s << R"(
template <int M>
__device__ __forceinline__ int xchg_bits(int v) {
  if constexpr (M == 1) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true);
  else if constexpr (M == 2) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true);
  else if constexpr (M < 32) return __builtin_amdgcn_ds_swizzle(v, 0x1F | (M << 10));
  else return __builtin_amdgcn_ds_bpermute((int)((threadIdx.x ^ 32u) << 2), v);
}
template <int M>
__device__ __forceinline__ float xchg(float v) { return __int_as_float(xchg_bits<M>(__float_as_int(v))); }
template <int M>
__device__ __forceinline__ double xchg(double v) {
  return __hiloint2double(xchg_bits<M>(__double2hiint(v)), xchg_bits<M>(__double2loint(v)));
}
)";
  return s.str();
}

// Distinct edge-attribute indices and (i, y) products used by a group.
struct GroupUse {
  std::set<int> ys;                       // absolute y indices
  std::set<std::pair<int, int>> products; // (i, absolute y)
};

GroupUse group_use(const Spec& spec, const Group& g) {
  GroupUse use;
  for (int p : g.paths) {
    const Path& q = spec.paths[p];
    for (const Term& t : q.terms) {
      use.ys.insert(q.y_off + t.j);
      use.products.insert({t.i, q.y_off + t.j});
    }
  }
  return use;
}

// Where one weight row serves every edge, weights and coupling coefficients leave
// the edge loop: a node's edges only meet in the products P_ij = sum_e x_i y_j
// (forward), or meet its seeds in Q_ij = sum_paths w sum_k c_ijk G_k (backward:
// gx messages Q y, gy partials Q^T x), so an edge costs one FMA per product instead of one
// per coefficient, component and product (lmax 3: forward 686 -> 234 FMAs, backward
// 1,233 -> 535 with the lane sums).  64 channels, lmax 3, 2,083 nodes, 109,000 edges,
// where both were bound by those: forward 125 -> 81 us, 69 with the whole next edge
// in flight; backward 198 -> 134 us, now bound by its x gathers and messages
// (0.9 GB, 6.7 TB/s from the caches and to memory).  The sums are kept in
// registers, hence the limit: 120 leave three waves per SIMD (lmax 3 has 112 in
// fp32; fp64 at lmax 3 would have 224 and keeps the per-edge form).
bool folds_weights(const Spec& spec, const GroupUse& use) {
  return spec.w_broadcast && (int)use.products.size() * spec.dtype_bits / 32 <= 120;
}

// Reduce-scatter of `names` over the 64 lanes: log2(P) halving steps leave
// every lane with one value index summed over a subset of lanes, then full
// exchanges finish the sum.  Lane L then holds value index L >> shift, and
// the lanes with (L & low_mask) == 0 write it.
std::string emit_butterfly(Code& c, std::vector<std::string> names, const char* prefix, int* shift,
                           int* low_mask) {
  int count = 1;
  while (count < (int)names.size()) count *= 2;
  while ((int)names.size() < count) names.push_back("(real)0");
  int level = 0, split_bits = 0;
  for (int m = 32; m >= 1; m >>= 1, ++level) {
    if (count == 1) {
      c.line("        %s = %s + xchg<%d>(%s);", names[0].c_str(), names[0].c_str(), m, names[0].c_str());
      continue;
    }
    const int half = count / 2;
    c.line("        const bool %sh%d = (lane & %d) != 0;", prefix, level, m);
    std::vector<std::string> next;
    for (int n = 0; n < half; ++n) {
      std::string name = std::string(prefix) + std::to_string(level) + "_" + std::to_string(n);
      c.line("        real %s = (%sh%d ? %s : %s) + xchg<%d>(%sh%d ? %s : %s);", name.c_str(), prefix, level,
             names[half + n].c_str(), names[n].c_str(), m, prefix, level, names[n].c_str(),
             names[half + n].c_str());
      next.push_back(name);
    }
    names = next;
    count = half;
    ++split_bits;
  }
  *shift = 6 - split_bits;
  *low_mask = (1 << (6 - split_bits)) - 1;
  return names[0];
}

// Odd row pitch of the per-wave LDS transpose of n partial values.
int reduce_pitch(int n) { return n % 2 ? n + 2 : n + 1; }

// The same reduction through LDS: every lane writes its n values as one row
// of a per-wave 64 x n table, then L lanes per column each add 64 / L rows
// and lane exchanges within the L finish the sum (fewer VALU instructions
// than the butterfly's selects, which in fp64 are two per value).  Lane L
// then holds column L >> shift, as with emit_butterfly.
std::string emit_lds_reduce(Code& c, const std::vector<std::string>& names, const char* prefix, int* shift,
                            int* low_mask) {
  const int n = (int)names.size(), pitch = reduce_pitch(n);
  int cols = 1;
  while (cols < n) cols *= 2;
  const int lanes = 64 / cols, rows = 64 / lanes;
  for (int v = 0; v < n; ++v) c.line("        red[lane * %d + %d] = %s;", pitch, v, names[v].c_str());
  c.line("        asm volatile(\"\" ::: \"memory\");");
  c.line("        const int %sc = min(lane / %d, %d), %sp = lane %% %d;", prefix, lanes, n - 1, prefix, lanes);
  c.line("        real %ss = red[%sp * %d + %sc];", prefix, prefix, pitch, prefix);
  for (int r = 1; r < rows; ++r)
    c.line("        %ss += red[(%sp + %d) * %d + %sc];", prefix, prefix, r * lanes, pitch, prefix);
  for (int m = lanes / 2; m >= 1; m /= 2) c.line("        %ss += xchg<%d>(%ss);", prefix, m, prefix);
  int bits = 0;
  while ((1 << bits) < lanes) ++bits;
  *shift = bits;
  *low_mask = lanes - 1;
  return std::string(prefix) + "s";
}

// The reduction for a wave that holds several edges (lane = edge * cw +
// channel): the sums of every edge and column, 64 / (edges * columns) lanes per
// sum, or several rounds where there are more than 64 sums.  Calls
// store(edge-of-wave, column rank, total, condition) per round.
void emit_packed_reduce(Code& c, const std::vector<std::string>& names, const char* prefix, int cw,
                        const std::function<void(const char*, const char*, const char*, const char*)>& store) {
  const int n = (int)names.size(), pitch = reduce_pitch(n), edges = 64 / cw;
  int cols = 1;
  while (cols < n) cols *= 2;
  const int sums = edges * cols, lanes = std::max(1, 64 / sums), rounds = std::max(1, sums / 64);
  const int rows = cw / lanes;
  for (int v = 0; v < n; ++v) c.line("        red[lane * %d + %d] = %s;", pitch, v, names[v].c_str());
  c.line("        asm volatile(\"\" ::: \"memory\");");
  for (int r = 0; r < rounds; ++r) {
    c.line("        {");
    c.line("          const int %so = %d + lane / %d, %se = %so / %d, %sr = %so %% %d, %sp = lane %% %d;", prefix, r * 64,
           lanes, prefix, prefix, cols, prefix, prefix, cols, prefix, lanes);
    c.line("          const int %sb = (%se * %d + %sp) * %d + min(%sr, %d);", prefix, prefix, cw, prefix, pitch, prefix,
           n - 1);
    c.line("          real %ss = red[%sb];", prefix, prefix);
    for (int q = 1; q < rows; ++q) c.line("          %ss += red[%sb + %d];", prefix, prefix, q * lanes * pitch);
    for (int m = lanes / 2; m >= 1; m /= 2) c.line("          %ss += xchg<%d>(%ss);", prefix, m, prefix);
    const std::string e = std::string(prefix) + "e", rank = std::string(prefix) + "r", sum = std::string(prefix) + "s";
    const std::string own = std::string(prefix) + "p == 0 && " + rank + " < " + std::to_string(n);
    store(e.c_str(), rank.c_str(), sum.c_str(), own.c_str());
    c.line("        }");
  }
  c.line("        asm volatile(\"\" ::: \"memory\");");
}

// (i, j) pairs of one path grouped by their coefficient vector over k, equal
// up to a global sign (relative tolerance 1e-12 absorbs last-bit differences
// between equal Clebsch-Gordan values).
struct ClassMember {
  int i, j, sign;
};
struct SignedClass {
  std::vector<std::pair<int, double>> coefficients;  // (k, c) of the representative
  std::vector<ClassMember> members;
};

std::vector<SignedClass> signed_classes(const std::map<std::pair<int, int>, std::vector<const Term*>>& by_ij) {
  std::vector<SignedClass> classes;
  for (const auto& kv : by_ij) {
    std::vector<std::pair<int, double>> vec;
    for (const Term* t : kv.second) vec.push_back({t->k, t->c});
    std::sort(vec.begin(), vec.end());
    int found = -1, sign = 1;
    for (size_t n = 0; n < classes.size() && found < 0; ++n) {
      const auto& ref = classes[n].coefficients;
      if (ref.size() != vec.size()) continue;
      for (int s : {1, -1}) {
        bool same = true;
        for (size_t m = 0; m < vec.size() && same; ++m) {
          const double a = ref[m].second, b = s * vec[m].second;
          same = ref[m].first == vec[m].first && std::abs(a - b) <= 1e-12 * std::max(std::abs(a), std::abs(b));
        }
        if (same) {
          found = (int)n;
          sign = s;
          break;
        }
      }
    }
    if (found < 0) {
      classes.push_back({vec, {}});
      found = (int)classes.size() - 1;
      sign = 1;
    }
    classes[found].members.push_back({kv.first.first, kv.first.second, sign});
  }
  return classes;
}


// Emits the copy of y[yi] into a vector register before its first use.
struct YCopies {
  bool on;
  std::set<int> done;
  void need(Code& c, int yi) {
    if (on && done.insert(yi).second) c.line("      asm(\"\" : \"+v\"(y%d));", yi);
  }
};

// Edge loop shared by the forward and backward groups; `body` emits the work
// of one edge e from x0.., w0.., y0.. and ev.
//
// prefetch 0: operands are loaded where they are used.
// prefetch 1: the x block and the path weights of edge e+1 are requested
//   while edge e computes.
// prefetch 2: also the y row, env and (one further ahead) the source index.
//   Empty asm statements that read the requested values at the end of the
//   iteration make the wait for them land there, after the iteration's
//   stores, instead of at the loop head, where it would also cover the stores
//   just issued (vmcnt counts loads and stores in issue order).
// depth 2 (with prefetch 2): two edges in flight, from two register buffers
//   used alternately by a loop unrolled twice.
//
// Packed groups (cw < 64) take 64 / cw edges per iteration, so the edge, its
// source and its y row differ between the lanes (vector loads); lanes past the
// last edge repeat it with ok == false.  One edge at a time, a block of 32
// channels ran half of its lanes idle and its weight rows as 128-byte requests:
// 1,000 nodes, 52,000 edges, lmax 2, 32 channels, forward 76 -> 31 us (100 MB of
// weights, 3.4 TB/s), backward 81 -> 64 us (4.2 TB/s).  `split`: the workgroup's
// waves take the iterations in turn.  `weights` off: the body uses none per edge.
void emit_edge_loop(Code& c, const Spec& spec, const Group& g, const GroupUse& use, bool env,
                    const Options& opt, const std::vector<std::string>& resident,
                    const std::function<void()>& body, bool split = false, bool weights = true) {
  const int np = weights ? (int)g.paths.size() : 0;
  const int nsub = 64 / g.cw;
  const bool packed = nsub > 1;
  const bool full = opt.prefetch >= 2;
  const char cls = packed ? 'v' : 's';
  auto load_edge = [&](const char* edge, const char* srcv, char b) {
    c.line("      {");
    c.line("        const real* xq = x + (i64)%s * IN1 + (%d + uc * %d);", srcv, g.x_off, g.d1);
    for (int i = 0; i < g.d1; ++i) c.line("        %cx%d = xq[%d];", b, i, i);
    c.line("        const real* wq = w + (i64)%s * WROW;", edge);
    for (int n = 0; n < np; ++n) {
      const Path& q = spec.paths[g.paths[n]];
      if (opt.nt_w)
        c.line("        %cw%d = __builtin_nontemporal_load(wq + %d + uc * %d);", b, n, q.w_off, q.w_stride);
      else
        c.line("        %cw%d = wq[%d + uc * %d];", b, n, q.w_off, q.w_stride);
    }
    if (full) {
      c.line("        const real* yq = y + (i64)%s * IN2;", edge);
      for (int yi : use.ys) c.line("        %cy%d = yq[%d];", b, yi, yi);
      if (env) c.line("        %cev = env[%s];", b, edge);
    }
    c.line("      }");
  };
  auto declare = [&](char b) {
    for (int i = 0; i < g.d1; ++i) c.line("      real %cx%d;", b, i);
    for (int n = 0; n < np; ++n) c.line("      real %cw%d;", b, n);
    if (full) {
      for (int yi : use.ys) c.line("      real %cy%d;", b, yi);
      if (env) c.line("      real %cev;", b);
    }
  };
  auto bind = [&](char b) {
    for (int i = 0; i < g.d1; ++i) c.line("      const real x%d = %cx%d;", i, b, i);
    for (int n = 0; n < np; ++n) c.line("      const real w%d = %cw%d;", n, b, n);
    if (full) {
      for (int yi : use.ys) c.line("      real y%d = %cy%d;", yi, b, yi);
      if (env) c.line("      const real ev = %cev;", b);
    }
  };
  auto waits = [&](char b) {
    for (int i = 0; i < g.d1; ++i) c.line("      asm volatile(\"\" :: \"v\"(%cx%d));", b, i);
    for (int n = 0; n < np; ++n) c.line("      asm volatile(\"\" :: \"v\"(%cw%d));", b, n);
    if (full) {
      for (int yi : use.ys) c.line("      asm volatile(\"\" :: \"%c\"(%cy%d));", cls, b, yi);
      if (env) c.line("      asm volatile(\"\" :: \"%c\"(%cev));", cls, b);
    }
    c.line("      asm volatile(\"\" :: \"%c\"(sn));", cls);
  };
  auto inline_y = [&]() {
    c.line("      const real* yr = y + (i64)e * IN2;");
    for (int yi : use.ys) c.line("      real y%d = yr[%d];", yi, yi);
    if (env) c.line("      const real ev = env[e];");
  };
  auto resident_waits = [&]() {
    for (const auto& name : resident) c.line("      asm volatile(\"\" :: \"v\"(%s));", name.c_str());
  };

  if (packed || split) {
    const std::string step = split ? std::to_string(nsub) + " * split" : std::to_string(nsub);
    const std::string lane_edge = packed ? " + sub" : "", skip = split ? "part * " + std::to_string(nsub) : "0";
    // The lane's edge `ahead` after `edge` (which lies before the end), or the last one.
    auto clamped = [&](const std::string& edge, const std::string& ahead) {
      return "edge_at(" + edge + ", " + ahead + lane_edge + ", end)";
    };
    c.line("    if (end - beg > %s) {", skip.c_str());
    c.line("    const eix first = beg + %s;", skip.c_str());
    declare('n');
    c.line("      int sn = src[%s];", clamped("first", "0").c_str());
    load_edge(clamped("first", "0").c_str(), "sn", 'n');
    c.line("      sn = src[%s];", clamped("first", step).c_str());
    waits('n');
    resident_waits();
    if (packed) c.line("      int it = 0;");
    c.line("      for (eix e0 = first;; e0 += %s%s) {", step.c_str(), packed ? ", ++it" : "");
    c.line("      const eix e = %s;", clamped("e0", "0").c_str());
    if (packed) c.line("      const bool ok = end - e0 > sub;");
    bind('n');
    c.line("      const eix en = %s;", clamped("e0", step).c_str());
    load_edge("en", "sn", 'n');
    c.line("      sn = src[%s];", clamped("e0", "2 * " + step).c_str());
    if (!full) inline_y();
    body();
    waits('n');
    c.line("      if (end - e0 <= %s) break;", step.c_str());
    c.line("      }");
    c.line("    }");
    return;
  }
  if (opt.prefetch == 0) {
    c.line("    {");
    c.line("      for (eix e = beg; e < end; ++e) {");
    c.line("      const int s = src[e];");
    c.line("      const real* xr = x + (i64)s * IN1 + (%d + uc * %d);", g.x_off, g.d1);
    for (int i = 0; i < g.d1; ++i) c.line("      const real x%d = xr[%d];", i, i);
    c.line("      const real* wr = w + (i64)e * WROW;");
    for (int n = 0; n < np; ++n) {
      const Path& q = spec.paths[g.paths[n]];
      c.line("      const real w%d = wr[%d + uc * %d];", n, q.w_off, q.w_stride);
    }
    inline_y();
    body();
    c.line("      }");
    c.line("    }");
    return;
  }
  c.line("    if (beg < end) {");
  declare('n');
  if (!full) {
    c.line("      int sn = src[beg];");
    load_edge("beg", "sn", 'n');
    c.line("      for (eix e = beg; e < end; ++e) {");
    bind('n');
    c.line("      const eix en = e + 1 < end ? e + 1 : e;");
    c.line("      sn = src[en];");
    load_edge("en", "sn", 'n');
    inline_y();
    body();
    c.line("      }");
    c.line("    }");
    return;
  }
  if (opt.depth < 2) {
    c.line("      int sn = src[beg];");
    load_edge("beg", "sn", 'n');
    c.line("      sn = src[beg + 1 < end ? beg + 1 : beg];");
    // Resolve the first edge's operands before the loop too, so that the loop
    // head needs no wait on either incoming path.
    waits('n');
    resident_waits();
    c.line("      for (eix e = beg; e < end; ++e) {");
    bind('n');
    c.line("      const eix en = e + 1 < end ? e + 1 : e;");
    load_edge("en", "sn", 'n');
    c.line("      sn = src[en + 1 < end ? en + 1 : en];");
    body();
    waits('n');
    c.line("      }");
    c.line("    }");
    return;
  }
  // Two edges in flight: buffer n holds edge e (resolved), buffer m edge e+1.
  declare('m');
  c.line("      const eix last = end - 1;");
  c.line("      int sn = src[beg];");
  load_edge("beg", "sn", 'n');
  c.line("      sn = src[beg + 1 < end ? beg + 1 : last];");
  load_edge("(beg + 1 < end ? beg + 1 : last)", "sn", 'm');
  c.line("      sn = src[edge_at(beg, 2, end)];");
  waits('n');
  resident_waits();
  c.line("      for (eix e0 = beg;; e0 += 2) {");
  for (int half = 0; half < 2; ++half) {
    const char cur = half == 0 ? 'n' : 'm', other = half == 0 ? 'm' : 'n';
    if (half == 0)
      c.line("      {");
    else
      c.line("      if (e0 + 1 < end) {");
    c.line("      const eix e = e0 + %d;", half);
    bind(cur);
    // Refill this buffer with edge e+2 and fetch the source index of e+3.
    c.line("      const eix en = edge_at(e, 2, end);");
    load_edge("en", "sn", cur);
    c.line("      sn = src[en + 1 < end ? en + 1 : last];");
    body();
    waits(other);
    c.line("      }");
  }
  c.line("      if (end - e0 <= 2) break;");
  c.line("      }");
  c.line("    }");
}

// Loop over the rows of a row-wise product, where node, edge and source are the
// same row: rows blockIdx.x, + gridDim.x, ... (64 / cw rows at once in a packed
// group, lanes past the last row repeating it with ok == false).  The operands
// of the next row are in flight while the current one is computed; a weight row
// shared by every row is loaded once, before the loop.  `seeds`: also the rows'
// output seeds, loaded where they are used (requested a row ahead they take up to
// twice the registers, at the same time: 183 us either way at 64 channels, lmax 2,
// 50,000 rows).  The last row requests nothing: most waves have one.  Bound by
// memory: that backward moves 0.89 GB (4.9 TB/s), its forward 0.77 GB in 121 us.
void emit_row_loop(Code& c, const Spec& spec, const Group& g, const GroupUse& use, bool shared, bool nt_w, bool seeds,
                   const std::function<void()>& body) {
  const int np = (int)g.paths.size(), nsub = 64 / g.cw;
  const bool packed = nsub > 1;
  struct Operand {
    std::string name, address;
    char cls;
    bool nt;
  };
  std::vector<Operand> ops, direct;
  auto at = [&](const char* base, const char* row, long off, int stride) {
    return std::string(base) + " + rn * " + row + " + (" + std::to_string(off) + " + uc * " + std::to_string(stride) + ")";
  };
  for (int i = 0; i < g.d1; ++i) ops.push_back({"x" + std::to_string(i), at("x", "IN1", g.x_off + i, g.d1), 'v', false});
  for (int n = 0; n < np; ++n) {
    const Path& q = spec.paths[g.paths[n]];
    if (shared)
      c.line("    const real w%d = w[%d + uc * %d];", n, q.w_off, q.w_stride);
    else
      ops.push_back({"w" + std::to_string(n), at("w", "WNUM", q.w_off, q.w_stride), 'v', nt_w});
  }
  if (seeds)
    for (size_t b = 0; b < g.blocks.size(); ++b)
      for (int k = 0; k < g.blocks[b].d3; ++k)
        direct.push_back({"G" + std::to_string(b) + "_" + std::to_string(k),
                       at("g", "OUTD", g.blocks[b].out_off + k, g.blocks[b].d3), 'v', false});
  for (int yi : use.ys)
    ops.push_back({"y" + std::to_string(yi), "y + rn * IN2 + " + std::to_string(yi), packed ? 'v' : 's', false});
  auto load = [&](const std::string& row) {
    c.line("      {");
    const std::string mine = packed ? "(" + row + " + sub)" : row;
    c.line("        const i64 rn = %s < end ? %s : end - 1;", mine.c_str(), mine.c_str());
    for (const auto& o : ops)
      c.line(o.nt ? "        n%s = __builtin_nontemporal_load(%s);" : "        n%s = *(%s);", o.name.c_str(),
             o.address.c_str());
    c.line("      }");
  };
  auto waits = [&]() {
    for (const auto& o : ops) c.line("      asm volatile(\"\" :: \"%c\"(n%s));", o.cls, o.name.c_str());
  };
  c.line("    const i64 end = E, first = (i64)blockIdx.x * %d, step = (i64)gridDim.x * %d;", nsub, nsub);
  c.line("    if (first < end) {");
  for (const auto& o : ops) c.line("      real n%s;", o.name.c_str());
  load("first");
  waits();
  c.line("      int it = 0;");
  c.line("      for (i64 e0 = first;; e0 += step, ++it) {");
  c.line("      const i64 e = %s;", packed ? "e0 + sub < end ? e0 + sub : end - 1" : "e0");
  if (packed) c.line("      const bool ok = e0 + sub < end;");
  for (const auto& o : ops) c.line("      real %s = n%s;", o.name.c_str(), o.name.c_str());
  if (!direct.empty()) {
    c.line("      const i64 rn = e;");
    for (const auto& o : direct) c.line("      const real %s = *(%s);", o.name.c_str(), o.address.c_str());
  }
  c.line("      const bool more = e0 + step < end;");
  c.line("      if (more) {");
  load("e0 + step");
  c.line("      }");
  body();
  c.line("      if (!more) break;");
  waits();
  c.line("      }");
  c.line("    }");
}

// Leaves values `names` (d per lane) of the current rows at dst[row, off + u * d + k]:
// through the per-wave buffer `lds`, so that a wave stores consecutive values.
void emit_row_store(Code& c, const Group& g, const std::vector<std::string>& names, const char* lds, const char* dst,
                    const char* width, int off, bool accumulate) {
  const int d = (int)names.size(), nsub = 64 / g.cw, per = g.cw * d;
  c.line("      {");
  for (int k = 0; k < d; ++k) c.line("        %s[lane * %d + %d] = %s;", lds, d, k, names[k].c_str());
  c.line("        asm volatile(\"\" ::: \"memory\");");
  c.line("        real* const ob = %s + e0 * %s + (%d + c0 * %d);", dst, width, off, d);
  for (int m = 0; m < d; ++m) {
    std::string cond, at = "ob + " + std::to_string(m * 64) + " + lane";
    const std::string idx = std::to_string(m * 64) + " + lane";
    if (nsub > 1) {
      c.line("        const int q%d = (%s) / %d, i%d = (%s) - q%d * %d;", m, idx.c_str(), per, m, idx.c_str(), m, per);
      cond = "if (i" + std::to_string(m) + " < nch * " + std::to_string(d) + " && e0 + q" + std::to_string(m) + " < end) ";
      at = "ob + (i64)q" + std::to_string(m) + " * " + width + " + i" + std::to_string(m);
    } else if (g.channels % 64) {
      cond = "if (" + idx + " < nch * " + std::to_string(d) + ") ";
    }
    if (accumulate)
      c.line("        %s*(%s) += %s[%s];", cond.c_str(), at.c_str(), lds, idx.c_str());
    else
      c.line("        %s__builtin_nontemporal_store(%s[%s], %s);", cond.c_str(), lds, idx.c_str(), at.c_str());
  }
  c.line("        asm volatile(\"\" ::: \"memory\");");
  c.line("      }");
}

// Channel u (uc: clamped to the last) of this lane, and the edge of the wave it
// works on (`sub`) in a packed group.
void emit_lanes(Code& c, const Group& g, int slot_base, int subsets) {
  const std::string chunk = subsets > 1 ? "((slot - " + std::to_string(slot_base) + ") / " + std::to_string(subsets) + ")"
                                        : "(slot - " + std::to_string(slot_base) + ")";
  if (g.cw < 64) {
    c.line("    const int u = %s * %d + lane %% %d;", chunk.c_str(), g.cw, g.cw);
    c.line("    const int sub = lane / %d;", g.cw);
  } else {
    c.line("    const int u = %s * 64 + lane;", chunk.c_str());
  }
  c.line("    const bool active = u < %d;", g.channels);
  c.line("    const int uc = active ? u : %d;", g.channels - 1);
}

// The products of one edge (or row) added to the accumulators A<block>_<k>.
void emit_forward_body(Code& c, const Spec& spec, const Group& g, bool env, bool l0, const Options& opt) {
  const int bits = spec.dtype_bits;
  const int np = (int)g.paths.size();
  const bool packed = g.cw < 64;
  if (packed) c.line("      if (ok) {");
  // l0 columns are summed over the paths (edge copies) sharing them.
  std::map<int, std::vector<int>> l0_cols;
  for (int n = 0; n < np; ++n) {
    const Path& q = spec.paths[g.paths[n]];
    if (l0 && q.l0_col >= 0) l0_cols[q.l0_col].push_back(n);
  }
  for (const auto& col : l0_cols) c.line("      real L%d = 0;", col.first);
  // Paths in edge-block order; each x*y product is formed just before the
  // first path that needs it, which bounds the products alive at once.
  std::vector<int> order(np);
  for (int n = 0; n < np; ++n) order[n] = n;
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
    return spec.paths[g.paths[a]].y_off < spec.paths[g.paths[b]].y_off;
  });
  std::set<std::pair<int, int>> formed;
  YCopies ycopy{opt.y_vgpr < 0 ? spec.dtype_bits == 32 : opt.y_vgpr != 0, {}};
  for (int n : order) {
    const Path& q = spec.paths[g.paths[n]];
    const int b = g.path_block[n];
    if (opt.fwd_local && !(l0 && q.l0_col >= 0)) {
      // Per-path form: u_i = w x_i, then A_k += c (u_i y_j).  Nothing is
      // shared between paths, so no product outlives its path (fewer live
      // registers for about a third more arithmetic).
      c.line("      {");
      std::set<int> is;
      for (const Term& t : q.terms) is.insert(t.i);
      for (int i : is) c.line("        const real u%d = %s * x%d;", i, env ? ("w" + std::to_string(n) + " * ev").c_str() : ("w" + std::to_string(n)).c_str(), i);
      std::map<std::pair<int, int>, std::vector<const Term*>> by_ij;
      for (const Term& t : q.terms) by_ij[{t.i, t.j}].push_back(&t);
      for (const auto& kv : by_ij) {
        ycopy.need(c, q.y_off + kv.first.second);
        c.line("        {");
        c.line("          const real p = u%d * y%d;", kv.first.first, q.y_off + kv.first.second);
        for (const Term* t : kv.second)
          c.line("          A%d_%d = FMA(%s, p, A%d_%d);", b, t->k, literal(t->c, bits).c_str(), b, t->k);
        c.line("        }");
      }
      c.line("      }");
      continue;
    }
    for (const Term& t : q.terms) {
      auto key = std::make_pair(t.i, q.y_off + t.j);
      if (formed.insert(key).second) {
        ycopy.need(c, key.second);
        c.line("      const real p%d_%d = x%d * y%d;", key.first, key.second, key.first, key.second);
      }
    }
    c.line("      {");
    if (env)
      c.line("        const real wv = w%d * ev;", n);
    else
      c.line("        const real wv = w%d;", n);
    std::map<int, std::vector<const Term*>> by_k;
    for (const Term& t : q.terms) by_k[t.k].push_back(&t);
    for (const auto& kv : by_k) {
      const int k = kv.first;
      bool first = true;
      for (const Term* t : kv.second) {
        std::string coef = literal(t->c, bits);
        if (first) {
          c.line("        real t%d = %s * p%d_%d;", k, coef.c_str(), t->i, q.y_off + t->j);
          first = false;
        } else {
          c.line("        t%d = FMA(%s, p%d_%d, t%d);", k, coef.c_str(), t->i, q.y_off + t->j, k);
        }
      }
      c.line("        A%d_%d = FMA(wv, t%d, A%d_%d);", b, k, k, b, k);
    }
    if (l0 && q.l0_col >= 0 && by_k.count(0)) c.line("        L%d = FMA(w%d, t0, L%d);", q.l0_col, n, q.l0_col);
    c.line("      }");
  }
  for (const auto& col : l0_cols)
    c.line("      l0[(i64)e * L0DIM + %d + uc] = L%d;", col.first, col.first);
  if (packed) c.line("      }");
}

// The group's accumulators A<block>_<k> from the node's product sums (folds_weights).
void emit_folded_sums(Code& c, const Spec& spec, const Group& g, const GroupUse& use, bool env, const Options& opt,
                      bool split) {
  const int bits = spec.dtype_bits;
  for (const auto& p : use.products) c.line("    real P%d_%d = 0;", p.first, p.second);
  emit_edge_loop(c, spec, g, use, env, opt, {}, [&] {
    if (g.cw < 64) c.line("      if (ok) {");
    std::set<int> is;
    for (const auto& p : use.products) is.insert(p.first);
    for (int i : is) c.line(env ? "      const real z%d = ev * x%d;" : "      const real z%d = x%d;", i, i);
    YCopies ycopy{opt.y_vgpr < 0 ? bits == 32 : opt.y_vgpr != 0, {}};
    for (const auto& p : use.products) {
      ycopy.need(c, p.second);
      c.line("      P%d_%d = FMA(z%d, y%d, P%d_%d);", p.first, p.second, p.first, p.second, p.first, p.second);
    }
    if (g.cw < 64) c.line("      }");
  }, split, false);
  for (size_t b = 0; b < g.blocks.size(); ++b)
    for (int k = 0; k < g.blocks[b].d3; ++k) c.line("    real A%zu_%d = 0;", b, k);
  for (size_t n = 0; n < g.paths.size(); ++n) {
    const Path& q = spec.paths[g.paths[n]];
    c.line("    {");
    c.line("      const real wv = w[%d + uc * %d];", q.w_off, q.w_stride);
    std::set<int> done;
    for (const Term& t : q.terms) {
      const std::string c0 = literal(t.c, bits);
      if (done.insert(t.k).second)
        c.line("      real t%d = %s * P%d_%d;", t.k, c0.c_str(), t.i, q.y_off + t.j);
      else
        c.line("      t%d = FMA(%s, P%d_%d, t%d);", t.k, c0.c_str(), t.i, q.y_off + t.j, t.k);
    }
    for (int k : done) c.line("      A%d_%d = FMA(wv, t%d, A%d_%d);", g.path_block[n], k, k, g.path_block[n], k);
    c.line("    }");
  }
}

void emit_forward_group(Code& c, const Spec& spec, const Group& g, bool env, bool l0, const Options& opt,
                        bool split) {
  GroupUse use = group_use(spec, g);
  const bool packed = g.cw < 64;
  emit_lanes(c, g, g.slot_base, 1);
  if (!l0 && folds_weights(spec, use)) {
    emit_folded_sums(c, spec, g, use, env, opt, split);
  } else {
    for (size_t b = 0; b < g.blocks.size(); ++b)
      for (int k = 0; k < g.blocks[b].d3; ++k) c.line("    real A%zu_%d = 0;", b, k);
    auto body = [&]() { emit_forward_body(c, spec, g, env, l0, opt); };
    emit_edge_loop(c, spec, g, use, env, opt, {}, body, split);
  }
  if (packed || split) {
    // The sums of a wave's edges, and of the waves sharing the node, meet in
    // LDS: piece q (wave and edge of the wave) holds its cw * d3 values in the
    // order they are stored.
    const char* pieces = split ? "split" : "1";
    c.line("    {");
    c.line("      const int c0 = (slot - %d) * %d;", g.slot_base, g.cw);
    c.line("      const int nch = %d - c0 < %d ? %d - c0 : %d;", g.channels, g.cw, g.channels, g.cw);
    for (size_t b = 0; b < g.blocks.size(); ++b) {
      const AccBlock& blk = g.blocks[b];
      for (int k = 0; k < blk.d3; ++k)
        c.line("      obuf[(%slane) * %d + %d] = A%zu_%d;", split ? "part * 64 + " : "", blk.d3, k, b, k);
      c.line(split ? "      __syncthreads();" : "      __builtin_amdgcn_wave_barrier();");
      c.line("      {");
      c.line("        real* ob = out + (i64)t * OUTD + (%d + c0 * %d);", blk.out_off, blk.d3);
      c.line("        for (int i = %s; i < nch * %d; i += 64%s) {", split ? "(int)threadIdx.x" : "lane", blk.d3,
             split ? " * split" : "");
      c.line("          real v = obuf[i];");
      c.line("          #pragma unroll %d", split ? 2 : 64 / g.cw);
      c.line("          for (int q = 1; q < %s * %d; ++q) v += obuf[q * %d + i];", pieces, 64 / g.cw, g.cw * blk.d3);
      c.line(blk.accumulate ? "          ob[i] += v;" : "          __builtin_nontemporal_store(v, ob + i);");
      c.line("        }");
      c.line("      }");
      c.line(split ? "      __syncthreads();" : "      __builtin_amdgcn_wave_barrier();");
    }
    c.line("    }");
    return;
  }
  if (!opt.out_lds) {
    c.line("    if (active) {");
    for (size_t b = 0; b < g.blocks.size(); ++b) {
      const AccBlock& blk = g.blocks[b];
      c.line("      real* o%zu = out + (i64)t * OUTD + (%d + u * %d);", b, blk.out_off, blk.d3);
      for (int k = 0; k < blk.d3; ++k) {
        if (blk.accumulate)
          c.line("      o%zu[%d] += A%zu_%d;", b, k, b, k);
        else
          c.line("      o%zu[%d] = A%zu_%d;", b, k, b, k);
      }
    }
    c.line("    }");
    return;
  }
  // Output blocks leave through LDS: lane u writes its d3 values at u*d3 + k
  // of a per-wave buffer, then every store instruction writes 64 consecutive
  // values of the chunk's contiguous block region, non-temporally.  Writes
  // mixed into the weight read stream are expensive on HBM (the 1.6 GB output
  // of the 128-channel lmax-3 layer costs about 1.4 ms of its forward); as
  // contiguous non-temporal stores they cost 0.2 ms less than as each lane's
  // d3 values stored directly.
  c.line("    {");
  c.line("      const int c0 = (slot - %d) * 64;", g.slot_base);
  if (g.channels % 64 == 0)
    c.line("      const int nch = 64;");
  else
    c.line("      const int nch = %d - c0 < 64 ? %d - c0 : 64;", g.channels, g.channels);
  for (size_t b = 0; b < g.blocks.size(); ++b) {
    const AccBlock& blk = g.blocks[b];
    for (int k = 0; k < blk.d3; ++k) c.line("      obuf[lane * %d + %d] = A%zu_%d;", blk.d3, k, b, k);
    c.line("      __builtin_amdgcn_wave_barrier();");
    c.line("      {");
    c.line("        real* ob = out + (i64)t * OUTD + (%d + c0 * %d);", blk.out_off, blk.d3);
    for (int m = 0; m < blk.d3; ++m) {
      const std::string idx = std::to_string(m * 64) + " + lane";
      std::string cond = g.channels % 64 == 0 ? std::string("") :
          "if (" + idx + " < nch * " + std::to_string(blk.d3) + ") ";
      if (blk.accumulate)
        c.line("        %sob[%s] += obuf[%s];", cond.c_str(), idx.c_str(), idx.c_str());
      else if (opt.nt_out)
        c.line("        %s__builtin_nontemporal_store(obuf[%s], ob + %s);", cond.c_str(), idx.c_str(), idx.c_str());
      else
        c.line("        %sob[%s] = obuf[%s];", cond.c_str(), idx.c_str(), idx.c_str());
    }
    c.line("      }");
    c.line("      __builtin_amdgcn_wave_barrier();");
  }
  c.line("    }");
}

// First channel of this wave's chunk and the number of channels in it.
void emit_chunk(Code& c, const Group& g, int subsets) {
  c.line("    const int c0 = (slot - %d) / %d * %d;", g.slot_base, subsets, g.cw);
  c.line("    const int nch = %d - c0 < %d ? %d - c0 : %d;", g.channels, g.cw, g.channels, g.cw);
}

void emit_rows_forward_group(Code& c, const Spec& spec, const Group& g, bool shared, const Options& opt) {
  GroupUse use = group_use(spec, g);
  emit_lanes(c, g, g.slot_base, 1);
  emit_chunk(c, g, 1);
  emit_row_loop(c, spec, g, use, shared, opt.fwd_nt_w, false, [&] {
    for (size_t b = 0; b < g.blocks.size(); ++b)
      for (int k = 0; k < g.blocks[b].d3; ++k) c.line("      real A%zu_%d = 0;", b, k);
    emit_forward_body(c, spec, g, false, false, opt);
    for (size_t b = 0; b < g.blocks.size(); ++b) {
      const AccBlock& blk = g.blocks[b];
      std::vector<std::string> names;
      for (int k = 0; k < blk.d3; ++k) names.push_back("A" + std::to_string(b) + "_" + std::to_string(k));
      emit_row_store(c, g, names, "obuf", "out", "OUTD", blk.out_off, blk.accumulate);
    }
  });
}

// Backward, destination-owned: the wave keeps the output seeds g[t] of its
// group in registers and streams the node's in-edges, writing gw and the gy
// partials per edge and the per-edge gx message msg[e, x block]; a second
// kernel sums the messages over each source node's out-edges.
// One wave's share of a backward group: all of its paths, or one subset of
// a split group (`g` is then the subset's view, sub its index).
Group subset_view(const Group& g, int sub);

// What a backward wave streams: a node's edges, or the rows of a row-wise
// product with a weight row each or one shared by all of them.
enum class Rows { none, own, shared };

void emit_backward_wave(Code& c, const Spec& spec, const Group& g, bool env, bool gl0, bool want_gw,
                        bool want_msg, bool want_part, const Options& opt, int sub, bool cmajor,
                        const Group* whole, Rows rows) {
  const int bits = spec.dtype_bits;
  GroupUse use = group_use(spec, g);
  const int np = (int)g.paths.size();
  const bool lds_reduce = opt.lds_reduce != 0;
  const bool packed = g.cw < 64;
  const int nsub = 64 / g.cw;
  emit_lanes(c, g, g.slot_base, g.subsets);
  if (rows != Rows::none) emit_chunk(c, g, g.subsets);
  const bool sum_gw = rows == Rows::shared && want_gw;
  if (sum_gw)
    for (int n = 0; n < np; ++n) c.line("    real GW%d = 0;", n);
  std::vector<std::string> seeds;
  for (size_t b = 0; b < g.blocks.size() && rows == Rows::none; ++b) {
    const AccBlock& blk = g.blocks[b];
    c.line("    const real* g%zu = g + (i64)t * OUTD + (%d + uc * %d);", b, blk.out_off, blk.d3);
    for (int k = 0; k < blk.d3; ++k) {
      c.line("    real G%zu_%d = g%zu[%d];", b, k, b, k);
      seeds.push_back("G" + std::to_string(b) + "_" + std::to_string(k));
    }
  }
  const bool fold = rows == Rows::none && !gl0 && !want_gw && folds_weights(spec, use);
  // Some q classes are computed once per node, before the edge loop, within
  // a register budget: classes of two or more terms first (each saves that
  // many instructions per edge), then single-term ones, cheapest first (a
  // seed all of whose classes are hoisted leaves the loop, so hoisting its
  // only class costs no register).
  std::vector<std::vector<SignedClass>> path_classes(np);
  std::map<std::pair<int, size_t>, std::string> hoisted;  // (path, class) -> register name
  {
    struct Candidate {
      int n;
      size_t cls;
      int terms;
      std::vector<std::string> uses;
    };
    std::vector<Candidate> cands;
    std::map<std::string, int> users;  // seed -> classes reading it
    for (int n = 0; n < np; ++n) {
      const Path& q = spec.paths[g.paths[n]];
      std::map<std::pair<int, int>, std::vector<const Term*>> by_ij;
      for (const Term& t : q.terms) by_ij[{t.i, t.j}].push_back(&t);
      path_classes[n] = signed_classes(by_ij);
      const bool scalar_seed = gl0 && q.l0_col >= 0;
      for (size_t m = 0; m < path_classes[n].size(); ++m) {
        Candidate cd{n, m, (int)path_classes[n][m].coefficients.size(), {}};
        for (const auto& kc : path_classes[n][m].coefficients)
          cd.uses.push_back("G" + std::to_string(g.path_block[n]) + "_" + std::to_string(kc.first));
        for (const auto& u : cd.uses) ++users[u];
        if (!scalar_seed) cands.push_back(cd);
      }
    }
    const int per_value = bits / 32;
    int budget = rows != Rows::none || fold ? -1 : opt.hoist_regs >= 0 ? opt.hoist_regs : 36;
    std::map<std::string, int> left = users;  // classes per seed not yet hoisted
    int extra = 0;                            // registers: hoisted values minus freed seeds
    auto cost = [&](const Candidate& cd) {
      int freed = 0;
      for (const auto& u : cd.uses) freed += left[u] == 1;
      return per_value * (1 - freed);
    };
    auto take = [&](const Candidate& cd) {
      extra += cost(cd);
      for (const auto& u : cd.uses) --left[u];
      hoisted[{cd.n, cd.cls}] = "H" + std::to_string(cd.n) + "_" + std::to_string(cd.cls);
    };
    std::stable_sort(cands.begin(), cands.end(), [](const Candidate& a, const Candidate& b) { return a.terms > b.terms; });
    for (const auto& cd : cands)
      if (cd.terms > 1 && extra + cost(cd) <= budget) take(cd);
    for (bool progress = true; progress;) {
      progress = false;
      const Candidate* best = nullptr;
      for (const auto& cd : cands)
        if (cd.terms == 1 && !hoisted.count({cd.n, cd.cls}) && extra + cost(cd) <= budget &&
            (!best || cost(cd) < cost(*best)))
          best = &cd;
      if (best) {
        take(*best);
        progress = true;
      }
    }
    for (const auto& kv : hoisted) {
      const SignedClass& cls = path_classes[kv.first.first][kv.first.second];
      const int b = g.path_block[kv.first.first];
      std::string expr;
      for (const auto& kc : cls.coefficients) {
        const std::string seed = "G" + std::to_string(b) + "_" + std::to_string(kc.first);
        expr = expr.empty() ? literal(kc.second, bits) + " * " + seed
                            : "FMA(" + literal(kc.second, bits) + ", " + seed + ", " + expr + ")";
      }
      c.line("    real %s = %s;", kv.second.c_str(), expr.c_str());
    }
    // Seeds still read in the loop, and the hoisted values, stay resident.
    std::vector<std::string> resident;
    for (const auto& name : seeds)
      if (left[name] > 0) resident.push_back(name);
    for (const auto& kv : hoisted) resident.push_back(kv.second);
    seeds = resident;
  }
  if (fold) {
    std::set<std::pair<int, int>> begun;
    std::vector<std::string> sums;
    for (int n = 0; n < np; ++n) {
      const Path& q = spec.paths[g.paths[n]];
      c.line("    const real wn%d = w[%d + uc * %d];", n, q.w_off, q.w_stride);
      for (const SignedClass& cls : path_classes[n]) {
        std::string expr;
        for (const auto& kc : cls.coefficients) {
          const std::string seed = "G" + std::to_string(g.path_block[n]) + "_" + std::to_string(kc.first);
          expr = expr.empty() ? literal(kc.second, bits) + " * " + seed
                              : "FMA(" + literal(kc.second, bits) + ", " + seed + ", " + expr + ")";
        }
        for (const auto& m : cls.members) {
          const int yi = q.y_off + m.j;
          const std::string name = "Q" + std::to_string(m.i) + "_" + std::to_string(yi);
          if (begun.insert({m.i, yi}).second) {
            c.line("    real %s = %swn%d * (%s);", name.c_str(), m.sign > 0 ? "" : "-", n, expr.c_str());
            sums.push_back(name);
          } else {
            c.line("    %s = FMA(%swn%d, %s, %s);", name.c_str(), m.sign > 0 ? "" : "-", n, expr.c_str(), name.c_str());
          }
        }
      }
    }
    seeds = sums;
  }
  // Combined subsets: lane c of the first subset's wave adds column c (y
  // index, env last) of both subsets' partials; r0 / r1 are that column's
  // positions in the two subsets' value lists (-1: not there).
  const bool combine = whole && whole->combine_subsets && want_part;
  if (combine && sub == 0 && !packed) {
    for (int s2 = 0; s2 < 2; ++s2) {
      const GroupUse other = group_use(spec, subset_view(*whole, s2));
      std::string chain = "-1";
      int rank = 0;
      std::vector<std::pair<int, int>> ranks;
      for (int yi : other.ys) ranks.push_back({yi, rank++});
      if (env) ranks.push_back({(int)spec.in2, rank});
      for (auto it = ranks.rbegin(); it != ranks.rend(); ++it)
        chain = "lane == " + std::to_string(it->first) + " ? " + std::to_string(it->second) + " : (" + chain + ")";
      c.line("    const int r%d = %s;", s2, chain.c_str());
    }
  }
  // Alternates between the iterations of the loop: the half of a shared LDS buffer.
  const std::string parity = packed || rows != Rows::none ? "it & 1" : "(e - beg) & 1";
  auto body = [&]() {
  if (!opt.hoist && rows == Rows::none && !fold) {
    // Opaque to the optimiser: keeps the edge-invariant q_ij inside the loop
    // instead of holding all of them in registers across it.
    for (const auto& name : seeds) c.line("      asm volatile(\"\" : \"+v\"(%s));", name.c_str());
  }
  YCopies ycopy{opt.y_vgpr > 0, {}};
  for (int i = 0; i < g.d1; ++i) c.line("      real M%d = 0;", i);
  for (int yi : use.ys) c.line("      real GY%d = 0;", yi);
  if (env) c.line("      real GE = 0;");
  // Partial-slot column of each gy (and genv) value: the y indices in order,
  // then env.
  std::map<std::string, int> column;
  for (int yi : use.ys) column["GY" + std::to_string(yi)] = (int)column.size();
  if (env) column["GE"] = (int)column.size();
  // gy (and genv) partials of this wave: reduce `values` over the 64 channels
  // and store them to their columns (consecutive from the first one).
  int flush_id = 0;
  auto flush = [&](const std::vector<std::string>& values) {
    if (!want_part || values.empty()) return;
    const std::string tag = "r" + std::to_string(flush_id++) + "_";
    c.line("      {");
    for (const auto& v : values) c.line("        %s = active ? %s : (real)0;", v.c_str(), v.c_str());
    if (packed) {
      emit_packed_reduce(c, values, tag.c_str(), g.cw,
                         [&](const char* edge, const char* rank, const char* total, const char* own) {
        c.line("          if (%s && end - e0 > %s)", own, edge);
        c.line("            part[((i64)(%d + (slot - %d)) * E + (e0 + %s)) * PART_W + %d + %s] = %s;", g.gy_slot_base,
               g.slot_base, edge, column[values[0]], rank, total);
      });
      c.line("      }");
      return;
    }
    int shift = 0, low = 0;
    std::string total = lds_reduce ? emit_lds_reduce(c, values, tag.c_str(), &shift, &low)
                                   : emit_butterfly(c, values, tag.c_str(), &shift, &low);
    c.line("        const int col = lane >> %d;", shift);
    c.line("        const bool own = (lane & %d) == 0 && col < %zu;", low, values.size());
    if (g.pair_partials) {
      // Chunk 1 hands its sums to chunk 0 (two buffers by edge parity: one
      // barrier per edge orders both uses).
      c.line("        const int par = %s;", parity.c_str());
      c.line("        if (slot - %d == 1) {", g.slot_base);
      c.line("          if (own) gy_share[par][%d + col] = %s;", column[values[0]], total.c_str());
      c.line("          __syncthreads();");
      c.line("        } else {");
      c.line("          __syncthreads();");
      c.line("          if (own)");
      c.line("            part[((i64)%d * E + e) * PART_W + %d + col] = %s + gy_share[par][%d + col];",
             g.gy_slot_base, column[values[0]], total.c_str(), column[values[0]]);
      c.line("        }");
    } else {
      c.line("        if (own)");
      c.line("          part[((i64)(%d + (slot - %d)) * E + e) * PART_W + %d + col] = %s;", g.gy_slot_base,
             g.slot_base, column[values[0]], total.c_str());
    }
    c.line("      }");
  };
  if (packed) c.line("      if (ok) {");
  if (fold) {
    YCopies copies{opt.y_vgpr < 0 ? bits == 32 : opt.y_vgpr != 0, {}};
    std::set<int> is;
    for (const auto& p : use.products) {
      is.insert(p.first);
      copies.need(c, p.second);
      c.line("      M%d = FMA(y%d, Q%d_%d, M%d);", p.first, p.second, p.first, p.second, p.first);
    }
    for (int i : is) {
      if (env) c.line("      GE = FMA(x%d, M%d, GE);", i, i);
      if (env) c.line("      M%d *= ev;", i);
      c.line(env ? "      const real z%d = ev * x%d;" : "      const real z%d = x%d;", i, i);
    }
    for (const auto& p : use.products)
      c.line("      GY%d = FMA(z%d, Q%d_%d, GY%d);", p.second, p.first, p.first, p.second, p.second);
  }
  for (int n = 0; n < np && !fold; ++n) {
    const Path& q = spec.paths[g.paths[n]];
    const int b = g.path_block[n];
    const bool scalar_seed = gl0 && q.l0_col >= 0;
    c.line("      {");
    c.line("        const real wv = w%d;", n);
    if (scalar_seed) c.line("        const real S0 = %sG%d_0 + gl0[(i64)e * L0DIM + %d + uc];",
                            env ? "ev * " : "", b, q.l0_col);
    std::set<int> is, js;
    for (const Term& t : q.terms) {
      is.insert(t.i);
      js.insert(t.j);
    }
    for (int j : js) c.line("        real b%d = 0;", j);
    for (int i : is) c.line("        real a%d = 0;", i);
    // Pairs whose coefficient vectors over k agree up to sign share one q
    // (the signed coefficient classes of src/lunatp/utils/layout.py:110-168).
    const std::vector<SignedClass>& classes = path_classes[n];
    for (size_t m = 0; m < classes.size(); ++m) {
      const SignedClass& cls = classes[m];
      const auto h = hoisted.find({n, m});
      if (h != hoisted.end()) {
        c.line("        const real q%zu = %s;", m, h->second.c_str());
      } else {
        bool first = true;
        for (const auto& kc : cls.coefficients) {
          std::string coef = literal(kc.second, bits);
          std::string seed =
              scalar_seed ? std::string("S0") : "G" + std::to_string(b) + "_" + std::to_string(kc.first);
          if (first) {
            c.line("        real q%zu = %s * %s;", m, coef.c_str(), seed.c_str());
            first = false;
          } else {
            c.line("        q%zu = FMA(%s, %s, q%zu);", m, coef.c_str(), seed.c_str(), m);
          }
        }
      }
      for (const auto& member : cls.members) {
        const int i = member.i, j = member.j;
        const char* sign = member.sign > 0 ? "" : "-";
        c.line("        b%d = FMA(%sx%d, q%zu, b%d);", j, sign, i, m, j);
        ycopy.need(c, q.y_off + j);
        c.line("        a%d = FMA(%sy%d, q%zu, a%d);", i, sign, q.y_off + j, m, i);
      }
    }
    // gw = sum_i x_i a_i  (= sum_ij x_i y_j q_ij)
    bool first = true;
    for (int i : is) {
      if (first) {
        c.line("        real gwv = x%d * a%d;", i, i);
        first = false;
      } else {
        c.line("        gwv = FMA(x%d, a%d, gwv);", i, i);
      }
    }
    if (first) c.line("        real gwv = 0;");
    const bool fold_env = env && !scalar_seed;
    if (env) {
      if (scalar_seed) {
        // genv needs sum_k g_k t_k with the raw node seed: t_0 = sum c x_i y_j.
        bool f2 = true;
        for (const Term& t : q.terms) {
          std::string coef = literal(t.c, bits);
          if (f2) {
            ycopy.need(c, q.y_off + t.j);
            c.line("        real t0 = %s * (x%d * y%d);", coef.c_str(), t.i, q.y_off + t.j);
            f2 = false;
          } else {
            ycopy.need(c, q.y_off + t.j);
            c.line("        t0 = FMA(%s, x%d * y%d, t0);", coef.c_str(), t.i, q.y_off + t.j);
          }
        }
        if (f2) c.line("        real t0 = 0;");
        c.line("        GE = FMA(wv, G%d_0 * t0, GE);", b);
      } else {
        c.line("        GE = FMA(wv, gwv, GE);");
      }
    }
    if (fold_env) {
      c.line("        gwv *= ev;");
      c.line("        const real ws = wv * ev;");
    } else {
      c.line("        const real ws = wv;");
    }
    if (sum_gw) {
      c.line("        GW%d += gwv;", n);
    } else if (want_gw) {
      if (opt.nt_gw)
        c.line("        __builtin_nontemporal_store(gwv, gw + (i64)e * WNUM + %d + uc * %d);", q.w_off, q.w_stride);
      else
        c.line("        gw[(i64)e * WNUM + %d + uc * %d] = gwv;", q.w_off, q.w_stride);
    }
    for (int j : js) c.line("        GY%d = FMA(ws, b%d, GY%d);", q.y_off + j, j, q.y_off + j);
    for (int i : is) c.line("        M%d = FMA(ws, a%d, M%d);", i, i, i);
    c.line("      }");
  }
  if (packed) c.line("      }");
  std::vector<std::string> values;
  for (int yi : use.ys) values.push_back("GY" + std::to_string(yi));
  if (env) values.push_back("GE");
  // gy partials of a combined subset: reduced over the lanes and left in LDS
  // (the second subset's before the barrier, the first's after it, each after
  // its message work so that the message values are dead by then).
  auto reduce_to_lds = [&]() {
    c.line("      {");
    for (const auto& v : values) c.line("        %s = active ? %s : (real)0;", v.c_str(), v.c_str());
    const std::string tag = "s" + std::to_string(sub) + "_";
    if (packed) {
      // Every column at its own place (the y index, env last) of its edge.
      std::string place;
      int rank = 0;
      for (int yi : use.ys) place += "rank == " + std::to_string(rank++) + " ? " + std::to_string(yi) + " : ";
      emit_packed_reduce(c, values, tag.c_str(), g.cw,
                         [&](const char* edge, const char* r, const char* total, const char* own) {
        c.line("          { const int rank = %s;", r);
        c.line("          if (%s) gy_sub[%d][%s][%s * PART_W + (%s%d)] = %s; }", own, sub, parity.c_str(), edge,
               place.c_str(), (int)spec.in2, total);
      });
      c.line("      }");
      return;
    }
    int shift = 0, low = 0;
    std::string total = lds_reduce ? emit_lds_reduce(c, values, tag.c_str(), &shift, &low)
                                   : emit_butterfly(c, values, tag.c_str(), &shift, &low);
    c.line("        const int col = lane >> %d;", shift);
    c.line("        if ((lane & %d) == 0 && col < %zu) gy_sub[%d][%s][col] = %s;", low, values.size(), sub, parity.c_str(),
           total.c_str());
    c.line("      }");
  };
  if ((want_msg || combine) && g.subsets > 1) {
    // The second subset hands its message share to the first through LDS
    // (two buffers by edge parity: one barrier per edge orders both uses).
    c.line("      {");
    c.line("        const int par = %s;", parity.c_str());
    if (sub == 1) {
      if (want_msg)
        for (int i = 0; i < g.d1; ++i) c.line("        msg_share[par][%d][lane] = M%d;", i, i);
      if (combine) reduce_to_lds();
      c.line("        __syncthreads();");
    } else {
      c.line("        __syncthreads();");
      if (want_msg)
        for (int i = 0; i < g.d1; ++i) c.line("        M%d += msg_share[par][%d][lane];", i, i);
    }
    c.line("      }");
  }
  if (want_msg && sub == 0 && rows != Rows::none) {
    // The row's only message is its gx.
    std::vector<std::string> names;
    for (int i = 0; i < g.d1; ++i) names.push_back("M" + std::to_string(i));
    emit_row_store(c, g, names, "red", "msg", "IN1", g.x_off, g.gx_accumulate);
  } else if (want_msg && sub == 0) {
    // Lanes past the last channel repeat channel C-1 exactly, so their stores
    // write identical values; only the cross-lane sums below must mask them.
    // Component-major messages: component i of the 64 channels of a chunk is
    // one contiguous 256-byte run (full-line stores; the x layout, d1 values
    // per lane, made every store a strided partial-line write).
    const int stride = cmajor ? g.channels : 1;
    c.line(packed ? "      if (ok) {" : "      {");
    if (cmajor)
      c.line("        real* mr = msg + (i64)e * IN1 + (%d + uc);", g.x_off);
    else
      c.line("        real* mr = msg + (i64)e * IN1 + (%d + uc * %d);", g.x_off, g.d1);
    for (int i = 0; i < g.d1; ++i) {
      if (g.gx_accumulate)
        c.line("        mr[%d] += M%d;", i * stride, i);
      else if (opt.nt_msg)
        c.line("        __builtin_nontemporal_store(M%d, mr + %d);", i, i * stride);
      else
        c.line("        mr[%d] = M%d;", i * stride, i);
    }
    c.line("      }");
  }
  if (combine && sub == 0 && packed) {
    reduce_to_lds();
    auto present = [&](int s2) {
      std::string mask;
      for (int yi : group_use(spec, subset_view(*whole, s2)).ys) mask += "col == " + std::to_string(yi) + " || ";
      return mask + (env ? "col == " + std::to_string((int)spec.in2) : std::string("false"));
    };
    c.line("      asm volatile(\"\" ::: \"memory\");");
    c.line("      for (int o = lane; o < %d * (int)PART_W; o += 64) {", nsub);
    c.line("        const int par = it & 1, edge = o / (int)PART_W, col = o %% (int)PART_W;");
    c.line("        const bool a = %s, b = %s;", present(0).c_str(), present(1).c_str());
    c.line("        if ((a || b) && end - e0 > edge)");
    c.line("          part[((i64)(%d + (slot - %d) / 2) * E + (e0 + edge)) * PART_W + col] =", whole->gy_slot_base,
           whole->slot_base);
    c.line("              (a ? gy_sub[0][par][o] : (real)0) + (b ? gy_sub[1][par][o] : (real)0);");
    c.line("      }");
  } else if (combine && sub == 0) {
    reduce_to_lds();
    c.line("      {");
    c.line("        const int par = %s;", parity.c_str());
    c.line("        if (r0 >= 0 || r1 >= 0)");
    c.line("          part[((i64)(%d + (slot - %d) / 2) * E + e) * PART_W + lane] =", whole->gy_slot_base,
           whole->slot_base);
    c.line("              (r0 >= 0 ? gy_sub[0][par][r0 < 0 ? 0 : r0] : (real)0) +");
    c.line("              (r1 >= 0 ? gy_sub[1][par][r1 < 0 ? 0 : r1] : (real)0);");
    c.line("      }");
  }
  if (!combine) flush(values);
  };
  if (rows == Rows::none) {
    emit_edge_loop(c, spec, g, use, env, opt, seeds, body, false, !fold);
    return;
  }
  emit_row_loop(c, spec, g, use, rows == Rows::shared, opt.nt_w, true, body);
  if (!sum_gw) return;
  // The gradient of the shared weight row over this workgroup's rows.
  for (int n = 0; n < np; ++n) {
    const Path& q = spec.paths[g.paths[n]];
    for (int m = g.cw; m < 64; m *= 2) c.line("    GW%d += xchg<%d>(GW%d);", n, m, n);
    c.line("    if (active%s) gw[(i64)blockIdx.x * WNUM + %d + u * %d] = GW%d;", packed ? " && sub == 0" : "", q.w_off,
           q.w_stride, n);
  }
}

// The paths of subset `sub` of a split group, as a group of their own.
Group subset_view(const Group& g, int sub) {
  Group view = g;
  view.paths.clear();
  view.path_block.clear();
  view.blocks.clear();
  std::map<int, int> remap;
  for (size_t n = 0; n < g.paths.size(); ++n) {
    if (g.path_subset[n] != sub) continue;
    const int b = g.path_block[n];
    if (!remap.count(b)) {
      remap[b] = (int)view.blocks.size();
      view.blocks.push_back(g.blocks[b]);
    }
    view.paths.push_back(g.paths[n]);
    view.path_block.push_back(remap[b]);
  }
  return view;
}

void emit_backward_group(Code& c, const Spec& spec, const Group& g, bool env, bool gl0, bool want_gw,
                         bool want_msg, bool want_part, const Options& opt, bool cmajor, Rows rows) {
  if (g.subsets == 1) {
    emit_backward_wave(c, spec, g, env, gl0, want_gw, want_msg, want_part, opt, 0, cmajor, nullptr, rows);
    return;
  }
  c.line("    const int sub = (slot - %d) %% %d;", g.slot_base, g.subsets);
  for (int sub = 0; sub < g.subsets; ++sub) {
    c.line("    %sif (sub == %d) {", sub ? "else " : "", sub);
    emit_backward_wave(c, spec, subset_view(g, sub), env, gl0, want_gw, want_msg, want_part, opt, sub, cmajor,
                       &g, rows);
    c.line("    }");
  }
}

std::string kernel_attributes(int wpe) {
  if (wpe <= 0) return "";
  return "__attribute__((amdgpu_waves_per_eu(" + std::to_string(wpe) + "))) ";
}

}  // namespace

int split_forward_lds(const Plan& plan, int phase) {
  int max_d3 = 1;
  for (const Group& g : plan.fwd_groups)
    if (g.phase == phase)
      for (const auto& b : g.blocks) max_d3 = std::max(max_d3, b.d3);
  return 64 * max_d3;
}

std::string emit_forward(const Plan& plan, bool env, bool l0, bool split) {
  const Spec& spec = plan.spec;
  Options opt = options();
  opt.prefetch = opt.fwd_prefetch;
  opt.depth = opt.fwd_depth;
  opt.nt_w = opt.fwd_nt_w && !plan.spec.w_broadcast;
  Code c;
  c.raw(prelude(spec, plan.edge_index_bits));
  for (int phase = 0; phase < plan.fwd_phases; ++phase) {
    const int waves = split ? 1 : plan.fwd_block_waves[phase], slots = plan.phase_slots[phase];
    c.line("extern \"C\" __global__ void __launch_bounds__(%d) %sluna_uvu_fwd_p%d(",
           split ? 512 : 64 * std::max(waves, 1), kernel_attributes(opt.fwd_wpe).c_str(), phase);
    c.line("    const real* __restrict__ x, const real* __restrict__ y, const real* __restrict__ w,");
    c.line("    const real* __restrict__ env, const int* __restrict__ src, const eix* __restrict__ rowptr,");
    c.line("    const int* __restrict__ order, real* __restrict__ out, real* __restrict__ l0) {");
    if (split) {
      c.line("  extern __shared__ __attribute__((aligned(16))) unsigned char obuf_lds[];");
      c.line("  real* const obuf = (real*)obuf_lds;");
    } else {
      const int per = split_forward_lds(plan, phase);
      c.line("  __shared__ __attribute__((aligned(16))) real obuf_lds[%d];", std::max(waves, 1) * per);
      c.line("  real* const obuf = obuf_lds + %s * %d;",
             waves > 0 ? "__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)" : "0", per);
    }
    if (split) {
      c.line("  const int lane = threadIdx.x & 63;");
      c.line("  const int split = blockDim.x >> 6, part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);");
      c.line("  const int slot = blockIdx.y;");
      c.line("  const int t = order[blockIdx.x];");
    } else if (waves == 0) {
      // One wave per workgroup, the slots of a node on consecutive workgroups.
      c.line("  const int lane = threadIdx.x;");
      c.line("  const int t = order[blockIdx.x / %d];", slots);
      // Rotated per node, so that the slots spread evenly over the XCDs
      // (workgroups go to XCDs round-robin).
      c.line("  const int slot = (blockIdx.x + blockIdx.x / %d) %% %d;", slots, slots);
    } else {
      c.line("  const int lane = threadIdx.x & 63;");
      c.line("  const int slot = blockIdx.y * %d + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);", waves);
      c.line("  const int t = order[blockIdx.x];");
    }
    c.line("  const eix beg = rowptr[t];");
    c.line("  const eix end = rowptr[t + 1];");
    bool first = true;
    for (const Group& g : plan.fwd_groups) {
      if (g.phase != phase) continue;
      c.line("  %sif (slot < %d) {", first ? "" : "else ", g.slot_base + g.chunks);
      first = false;
      Options own = opt;
      if (g.cw < 64 || split || (!l0 && folds_weights(spec, group_use(spec, g)))) own.prefetch = opt.packed_prefetch;
      emit_forward_group(c, spec, g, env, l0, own, split);
      c.line("  }");
    }
    c.line("}");
  }
  return c.s.str();
}

static std::string backward_source(const Plan& plan, bool env, bool gl0, bool want_gw, bool want_msg, bool want_part,
                                   Rows rows) {
  const Spec& spec = plan.spec;
  Options opt = options();
  opt.prefetch = opt.bwd_prefetch;
  opt.depth = opt.bwd_depth;
  const int streaming = spec.dtype_bits == 32 ? 1 : 0;
  if (opt.bwd_nt_w < 0) opt.bwd_nt_w = streaming;
  opt.nt_w = opt.bwd_nt_w != 0;
  const bool cmajor = message_component_major(plan);
  Code c;
  c.raw(prelude(spec, plan.edge_index_bits));
  for (int phase = 0; phase < plan.bwd_phases; ++phase) {
    const int waves = plan.bwd_block_waves[phase], slots = plan.bwd_phase_slots[phase];
    c.line("extern \"C\" __global__ void __launch_bounds__(%d) %sluna_uvu_%s_p%d(", 64 * std::max(waves, 1),
           kernel_attributes(opt.bwd_wpe).c_str(), rows == Rows::none ? "bwd" : "rows_bwd", phase);
    c.line("    const real* __restrict__ x, const real* __restrict__ y, const real* __restrict__ w,");
    if (rows == Rows::none) {
      c.line("    const real* __restrict__ env, const real* __restrict__ g, const real* __restrict__ gl0,");
      c.line("    const int* __restrict__ src, const eix* __restrict__ rowptr, const int* __restrict__ order,");
    } else {
      c.line("    const real* __restrict__ g,");
    }
    c.line("    real* __restrict__ gw, real* __restrict__ msg, real* __restrict__ part, i64 E) {");
    int share_d1 = 0;
    for (const Group& g : plan.bwd_groups)
      if (g.phase == phase && g.subsets > 1) share_d1 = std::max(share_d1, g.d1);
    if (share_d1 > 0 && want_msg) c.line("  __shared__ real msg_share[2][%d][64];", share_d1);
    bool pairs = false;
    for (const Group& g : plan.bwd_groups) pairs = pairs || (g.phase == phase && g.pair_partials);
    if (pairs && want_part) c.line("  __shared__ real gy_share[2][PART_W];");
    bool combined = false;
    for (const Group& g : plan.bwd_groups) combined = combined || (g.phase == phase && g.combine_subsets);
    if (combined && want_part) {
      int nsub = 1;
      for (const Group& g : plan.bwd_groups)
        if (g.phase == phase && g.combine_subsets) nsub = std::max(nsub, 64 / g.cw);
      c.line("  __shared__ real gy_sub[2][2][%d * PART_W];", nsub);
    }
    bool packed = false;
    for (const Group& g : plan.bwd_groups) packed = packed || (g.phase == phase && g.cw < 64);
    const bool stores = rows != Rows::none && want_msg;
    if ((want_part && (packed || opt.lds_reduce != 0)) || stores) {
      // Per-wave table of the LDS reduction of the gy partials; rows leave gx
      // through it too.
      int most = 1, widest = 1;
      for (const Group& g : plan.bwd_groups) {
        if (g.phase != phase) continue;
        most = std::max(most, (int)group_use(spec, g).ys.size() + (env ? 1 : 0));
        widest = std::max(widest, g.d1);
      }
      const int pitch = std::max(want_part ? reduce_pitch(most) : 1, stores ? widest : 1);
      c.line("  __shared__ real red_lds[%d];", std::max(waves, 1) * 64 * pitch);
      c.line("  real* const red = red_lds + %s * %d;",
             waves > 0 ? "__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)" : "0", 64 * pitch);
    }
    if (rows != Rows::none) {
      c.line("  const int lane = threadIdx.x & 63;");
      c.line("  const int slot = blockIdx.y * %d + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);", std::max(waves, 1));
    } else if (waves == 0) {
      // One wave per workgroup, the slots of a node on consecutive workgroups.
      c.line("  const int lane = threadIdx.x;");
      c.line("  const int t = order[blockIdx.x / %d];", slots);
      // Rotated per node, so that the slots spread evenly over the XCDs
      // (workgroups go to XCDs round-robin).
      c.line("  const int slot = (blockIdx.x + blockIdx.x / %d) %% %d;", slots, slots);
    } else {
      c.line("  const int lane = threadIdx.x & 63;");
      c.line("  const int t = order[blockIdx.x];");
      c.line("  const int slot = blockIdx.y * %d + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);", waves);
    }
    if (rows == Rows::none) {
    // Few nodes: a grid of more than one layer cuts every node's edges into as
    // many runs (nothing is summed over a node's edges here).
    c.line("  eix beg = rowptr[t], end = rowptr[t + 1];");
    c.line("  if (gridDim.z > 1) {");
    c.line("    const eix n = end - beg, layers = (eix)gridDim.z;");
    c.line("    const eix run = n / layers + (n %% layers != 0), skip = run * (eix)blockIdx.z;");
    c.line("    beg += skip < n ? skip : n;");
    c.line("    if (end - beg > run) end = beg + run;");
    c.line("  }");
    }
    bool first = true;
    for (const Group& g : plan.bwd_groups) {
      if (g.phase != phase) continue;
      // A split group may start after an unused (padding) slot: test both ends.
      c.line("  %sif (slot >= %d && slot < %d) {", first ? "" : "else ", g.slot_base,
             g.slot_base + g.chunks * g.subsets);
      first = false;
      emit_backward_group(c, spec, g, env, gl0, want_gw, want_msg, want_part, opt, cmajor, rows);
      c.line("  }");
    }
    c.line("}");
  }
  // Reduction of the per-wave partials into gy (and genv).  Table: for each
  // output column, the (slot, partial column) pairs that hold a share of it.
  const int pw = spec.in2 + (env ? 1 : 0);
  std::vector<std::vector<std::pair<int, int>>> writers(pw);
  for (const Group& g : plan.bwd_groups) {
    if (g.combine_subsets) {
      // One slot per chunk, columns in place (y index, env last).
      const GroupUse use = group_use(spec, g);
      for (int chunk = 0; chunk < g.chunks; ++chunk) {
        for (int yi : use.ys) writers[yi].push_back({g.gy_slot_base + chunk, yi});
        if (env) writers[spec.in2].push_back({g.gy_slot_base + chunk, (int)spec.in2});
      }
      continue;
    }
    for (int sub = 0; sub < g.subsets; ++sub) {
      GroupUse use = group_use(spec, g.subsets > 1 ? subset_view(g, sub) : g);
      for (int chunk = 0; chunk < g.chunks; ++chunk) {
        if (g.pair_partials && chunk > 0) continue;  // chunk 1's share is in chunk 0's slot
        const int slot = g.gy_slot_base + chunk * g.subsets + sub;
        int col = 0;
        for (int yi : use.ys) writers[yi].push_back({slot, col++});
        if (env) writers[spec.in2].push_back({slot, col});
      }
    }
  }
  // 256 edges per workgroup.  Each partial slot's rows of those edges are one
  // contiguous run (PART_W values per edge): they are copied into LDS with
  // consecutive threads on consecutive addresses, then every thread adds its
  // edge's columns; the gy rows leave through LDS the same way.
  std::map<int, std::vector<std::pair<int, int>>> by_slot;  // slot -> (partial column, output column)
  for (int col = 0; col < pw; ++col)
    for (const auto& sc : writers[col]) by_slot[sc.first].push_back({sc.second, col});
  c.line("extern \"C\" __global__ void __launch_bounds__(256) luna_uvu_bwd_reduce(");
  c.line("    const real* __restrict__ part, real* __restrict__ gy, real* __restrict__ genv, i64 E) {");
  c.line("  __shared__ real tile[256 * PART_W];");
  c.line("  const int t = threadIdx.x;");
  c.line("  const i64 e0 = (i64)blockIdx.x * 256;");
  c.line("  const int n = E - e0 < 256 ? (int)(E - e0) : 256;");
  // When every slot holds every column in place (each group reads every y
  // component), the sum is element-wise over the slots' runs: every thread
  // adds the same element of all slots, with all their loads in flight.
  bool in_place = !by_slot.empty() && pw == (int)spec.in2 + (env ? 1 : 0);
  for (const auto& kv : by_slot) {
    in_place = in_place && (int)kv.second.size() == pw;
    for (const auto& pc : kv.second) in_place = in_place && pc.first == pc.second;
  }
  if (in_place) {
    c.line("  #pragma unroll 4");
    c.line("  for (int i = t; i < n * (int)PART_W; i += 256) {");
    bool first = true;
    for (const auto& kv : by_slot) {
      c.line("    %s part[((i64)%d * E + e0) * PART_W + i];", first ? "real v =" : "v +=", kv.first);
      first = false;
    }
    c.line("    tile[i] = v;");
    c.line("  }");
    c.line("  __syncthreads();");
    c.line("  if (gy) {");
    c.line("    real* dst = gy + e0 * IN2;");
    c.line("    for (int i = t; i < n * (int)IN2; i += 256) dst[i] = tile[(i / IN2) * PART_W + i %% IN2];");
    c.line("  }");
    if (env) c.line("  if (genv && t < n) genv[e0 + t] = tile[t * PART_W + IN2];");
    c.line("}");
  } else {
  for (int col = 0; col < pw; ++col) c.line("  real acc%d = 0;", col);
  // Consecutive slots with the same column map (the chunks of one group) share
  // one loop, so the code size does not grow with the channel count.
  std::vector<std::pair<std::pair<int, int>, const std::vector<std::pair<int, int>>*>> runs;
  for (const auto& kv : by_slot) {
    if (!runs.empty() && runs.back().first.second + 1 == kv.first && *runs.back().second == kv.second)
      runs.back().first.second = kv.first;
    else
      runs.push_back({{kv.first, kv.first}, &kv.second});
  }
  for (const auto& run : runs) {
    c.line("  for (int sl = %d; sl <= %d; ++sl) {", run.first.first, run.first.second);
    c.line("    const real* src = part + ((i64)sl * E + e0) * PART_W;");
    c.line("    for (int i = t; i < n * (int)PART_W; i += 256) tile[i] = src[i];");
    c.line("    __syncthreads();");
    c.line("    if (t < n) {");
    for (const auto& pc : *run.second) c.line("      acc%d += tile[t * PART_W + %d];", pc.second, pc.first);
    c.line("    }");
    c.line("    __syncthreads();");
    c.line("  }");
  }
  c.line("  if (gy) {");
  c.line("    if (t < n) {");
  for (int col = 0; col < spec.in2; ++col) c.line("      tile[t * IN2 + %d] = acc%d;", col, col);
  c.line("    }");
  c.line("    __syncthreads();");
  c.line("    real* dst = gy + e0 * IN2;");
  c.line("    for (int i = t; i < n * (int)IN2; i += 256) dst[i] = tile[i];");
  c.line("  }");
  if (env) c.line("  if (genv && t < n) genv[e0 + t] = acc%d;", spec.in2);
  c.line("}");
  }
  c.line("extern \"C\" __global__ void __launch_bounds__(256) luna_uvu_fill(real* __restrict__ p, i64 n) {");
  c.line("  const i64 i = (i64)blockIdx.x * 256 + threadIdx.x;");
  c.line("  if (i < n) p[i] = 0;");
  c.line("}");
  if (rows != Rows::none) {
    if (rows == Rows::own || !want_gw) return c.s.str();
    // Sum of the workgroups' gradients of the shared weight row: 32 columns and 32
    // teams of threads per workgroup, so that few columns still keep many loads
    // in flight.
    c.line("extern \"C\" __global__ void __launch_bounds__(1024) luna_uvu_rows_gw(");
    c.line("    const real* __restrict__ part, real* __restrict__ gw, int n) {");
    c.line("  __shared__ real share[32][33];");
    c.line("  const int lane = threadIdx.x & 31, team = threadIdx.x >> 5, col = blockIdx.x * 32 + lane;");
    c.line("  real v = 0;");
    c.line("  if (col < WNUM) {");
    c.line("    #pragma unroll 8");
    c.line("    for (int r = team; r < n; r += 32) v += part[(i64)r * WNUM + col];");
    c.line("  }");
    c.line("  share[team][lane] = v;");
    c.line("  __syncthreads();");
    c.line("  for (int h = 16; h; h >>= 1) {");
    c.line("    if (team < h) share[team][lane] += share[team + h][lane];");
    c.line("    __syncthreads();");
    c.line("  }");
    c.line("  if (team == 0 && col < WNUM) gw[col] = share[0][lane];");
    c.line("}");
    return c.s.str();
  }
  // Segment sum of the gx messages over each source node's out-edges.
  std::vector<std::pair<long, long>> ranges;
  for (const Group& g : plan.bwd_groups) ranges.push_back({g.x_off, g.x_off + (long)g.channels * g.d1});
  std::sort(ranges.begin(), ranges.end());
  std::vector<std::pair<long, long>> merged;
  for (const auto& r : ranges) {
    if (!merged.empty() && r.first <= merged.back().second)
      merged.back().second = std::max(merged.back().second, r.second);
    else
      merged.push_back(r);
  }
  // Position in gx of message column col (component-major blocks permute).
  c.line("__device__ __forceinline__ int gx_col(int col) {");
  if (cmajor) {
    std::set<std::tuple<int, int, int>> blocks;
    for (const Group& g : plan.bwd_groups) blocks.insert({g.x_off, g.d1, g.channels});
    for (const auto& b : blocks) {
      const int x0 = std::get<0>(b), d1 = std::get<1>(b), ch = std::get<2>(b);
      if (d1 == 1) continue;
      c.line("  if (col >= %d && col < %d) { const int r = col - %d; return %d + (r %% %d) * %d + r / %d; }", x0,
             x0 + ch * d1, x0, x0, ch, d1, ch);
    }
  }
  c.line("  return col;");
  c.line("}");
  c.line("__device__ __forceinline__ bool covered(int col) {");
  if (merged.size() == 1 && merged[0].first == 0 && merged[0].second == spec.in1) {
    c.line("  return true;");
  } else {
    c.raw("  return false");
    for (const auto& r : merged) c.s << " || (col >= " << r.first << " && col < " << r.second << ")";
    c.raw(";\n");
  }
  c.line("}");
  const int vec = gather_vector_width(plan);
  // Clang vector types (element-wise +, and accepted by the non-temporal builtins).
  const char* vtype = vec == 1 ? "real"
                               : (spec.dtype_bits == 64 ? "double __attribute__((ext_vector_type(2)))"
                                                        : "float __attribute__((ext_vector_type(4)))");
  // A workgroup takes gather_columns() vectors of one source row; narrow rows
  // leave room for several teams of threads, which share the source's edges
  // and add up through LDS.
  const int cols = gather_columns(plan), teams = gather_teams(plan);
  c.line("extern \"C\" __global__ void __launch_bounds__(%d) luna_uvu_bwd_gather(", cols * teams);
  c.line("    const real* __restrict__ msg, const eix* __restrict__ srow, const eix* __restrict__ ebs,");
  c.line("    real* __restrict__ gx) {");
  c.line("  typedef %s vec_t;", vtype);
  c.line("  const int s = blockIdx.x;");
  if (teams > 1) {
    c.line("  __shared__ vec_t share[%d];", cols * (teams - 1));
    c.line("  const int team = threadIdx.x / %d, col = (threadIdx.x - team * %d) * %d;", cols, cols, vec);
  } else {
    c.line("  const int col = (blockIdx.y * %d + threadIdx.x) * %d;", cols, vec);
    c.line("  if (col >= IN1) return;");
  }
  const Options gopt = options();
  const int un = gopt.gather_unroll;
  auto load = [&](const std::string& row) {
    const std::string ptr = "(const vec_t*)(msg + (i64)" + row + " * IN1 + col)";
    return gopt.gather_nt ? "__builtin_nontemporal_load(" + ptr + ")" : "*" + ptr;
  };
  for (int n = 0; n < un; ++n) c.line("  vec_t acc%d = {};", n);
  c.line("  if (covered(col)) {");
  c.line("    const eix beg = srow[s];");
  c.line("    eix left = srow[s + 1] - beg%s;", teams > 1 ? " - team" : "");
  c.line("    const eix* p = ebs + (i64)beg%s;", teams > 1 ? " + team" : "");
  c.line("    for (; left > %d; left -= %d, p += %d) {", (un - 1) * teams, un * teams, un * teams);
  for (int n = 0; n < un; ++n)
    c.line("      acc%d += %s;", n, load("p[" + std::to_string(n * teams) + "]").c_str());
  c.line("    }");
  c.line("    for (; left > 0; left -= %d, p += %d) acc0 += %s;", teams, teams, load("*p").c_str());
  c.line("  }");
  // pairwise sum of the partial accumulators
  for (int width = 1; width < un; width *= 2)
    for (int n = 0; n + width < un; n += 2 * width) c.line("  acc%d += acc%d;", n, n + width);
  if (teams > 1) {
    c.line("  if (team) share[threadIdx.x - %d] = acc0;", cols);
    c.line("  __syncthreads();");
    c.line("  if (team) return;");
    for (int n = 1; n < teams; ++n) c.line("  acc0 += share[threadIdx.x + %d];", (n - 1) * cols);
  }
  if (cmajor && vec > 1) {
    // The values of one vector are consecutive channels of one component:
    // their gx positions are d1 apart.
    c.line("  real* gr = gx + (i64)s * IN1;");
    c.line("  const int g0 = gx_col(col);");
    c.line("  const int step = %d > 1 ? gx_col(col + 1) - g0 : 1;", vec);
    for (int n = 0; n < vec; ++n) c.line("  gr[g0 + %d * step] = acc0[%d];", n, n);
  } else if (cmajor) {
    c.line("  gx[(i64)s * IN1 + gx_col(col)] = acc0;");
  } else {
    c.line("  *(vec_t*)(gx + (i64)s * IN1 + col) = acc0;");
  }
  c.line("}");
  return c.s.str();
}

std::string emit_backward(const Plan& plan, bool env, bool gl0, bool want_gw, bool want_msg, bool want_part) {
  return backward_source(plan, env, gl0, want_gw, want_msg, want_part, Rows::none);
}

std::string emit_rows_backward(const Plan& plan, bool shared, bool want_gw, bool want_msg, bool want_part) {
  return backward_source(plan, false, false, want_gw, want_msg, want_part, shared ? Rows::shared : Rows::own);
}

std::string emit_rows_forward(const Plan& plan, bool shared) {
  const Spec& spec = plan.spec;
  const Options opt = options();
  Code c;
  c.raw(prelude(spec, plan.edge_index_bits));
  for (int phase = 0; phase < plan.fwd_phases; ++phase) {
    const int waves = std::max(plan.fwd_block_waves[phase], 1), per = split_forward_lds(plan, phase);
    c.line("extern \"C\" __global__ void __launch_bounds__(%d) luna_uvu_rows_fwd_p%d(", 64 * waves, phase);
    c.line("    const real* __restrict__ x, const real* __restrict__ y, const real* __restrict__ w,");
    c.line("    real* __restrict__ out, i64 E) {");
    c.line("  __shared__ __attribute__((aligned(16))) real obuf_lds[%d];", waves * per);
    c.line("  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;");
    c.line("  real* const obuf = obuf_lds + wave * %d;", per);
    c.line("  const int slot = blockIdx.y * %d + wave;", waves);
    bool first = true;
    for (const Group& g : plan.fwd_groups) {
      if (g.phase != phase) continue;
      c.line("  %sif (slot < %d) {", first ? "" : "else ", g.slot_base + g.chunks);
      first = false;
      emit_rows_forward_group(c, spec, g, shared, opt);
      c.line("  }");
    }
    c.line("}");
  }
  return c.s.str();
}

}  // namespace luna
