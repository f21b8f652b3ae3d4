// Shared-weight UVW tensor product on CDNA4 matrix cores (fp32).
//
// For a path p (input block l1 with mul1 copies, edge block l2 with mul2
// copies, output block io with mul3 copies) and a batch row b:
//   Z_p[b, k, K=(u,v)] = sum_{(i,j)} c_ijk x[b, xo + u*d1 + i] y[b, yo + v*d2 + j]
//   out[b, oo + w*d3 + k] += sum_K Z_p[b, k, K] W_p[K, w]        (W_p = w[wo + K*mul3 + w])
// (e3nn's uvw connection, src/lunatp/uvw/kernels/forward.py:1082-1465).  The
// sparse CG producer is VALU work on rows staged through LDS; the contraction
// over K is v_mfma_f32_32x32x2f32 with 32 output channels (one tile) or 64
// (two tiles fed by one Z operand) as M and a 32-row tile of b as N.  The
// backward is two more matrix-core passes:
//   dZ_p[b, k, K] = sum_w g[b, oo + w*d3 + k] W_p[K, w]  ->  gx, gy through the CG terms
//   dW_p[K, w]    = sum_{b,k} Z_p[b, k, K] g[b, oo + w*d3 + k]   (per row chunk, then reduced)
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

struct UvwTerm {
  int i, j, k;
  double c;
};

struct UvwPath {
  int x_off, y_off, out_off, w_off, mul1, mul2, mul3, d1, d2, d3;
  std::vector<UvwTerm> terms;
};

struct UvwSpec {
  int dtype_bits = 32;
  int in1 = 0, in2 = 0, out = 0, wnum = 0;
  std::vector<UvwPath> paths;
  // Kernel variants, fixed when the plan is created (launch geometry depends
  // on them), from LUNAEQ_AMD_UVW_VEC (0: no 16-byte row loads),
  // LUNAEQ_AMD_UVW_WIDE (0: 32-channel forward tiles only, 1: 64-channel tiles
  // staged through registers, 2 or unset: 64-channel tiles with LDS copies)
  // and LUNAEQ_AMD_UVW_WDMA (0: weight gradient without LDS copies), for
  // comparisons.
  bool vec = true;
  int wide = 2;
  bool wdma = true;
  // LUNAEQ_AMD_UVW_GPAD: seed-row padding in the gx/gy staging (1: scalar LDS
  // writes, 2: pairs, 4: 16-byte writes).  With rows 32 d3 + 2 floats apart,
  // the B-operand reads of one half-wave (16 rows x two w) fall in 32
  // distinct banks (0.863 -> 0.822 ms against 32 d3 + 4 at config 5).
  int gpad = 2;
  int wpad = 2;  // LUNAEQ_AMD_UVW_WPAD: weight-row padding (2: the A-operand reads conflict-free, as above)
  int bcw = 32;  // LUNAEQ_AMD_UVW_BCW: w per staged chunk of the gx/gy kernel (32, or 16)
  int wrows = 2;  // LUNAEQ_AMD_UVW_WROWS: batch rows per LDS copy of the weight gradient (2, or 4)
  // LUNAEQ_AMD_UVW_BDMA: gx/gy chunks copied by global_load_lds one chunk
  // ahead (1) or staged through registers (0); -1: copied in the kernels
  // whose per-lane state leaves two waves per SIMD, where the freed registers
  // pay (degree-3 layer 1.517 -> 1.457 ms), staged where four fit (config 5:
  // 0.771 against 0.781 ms, the copies' 16-byte pieces cannot be padded
  // against the two-way bank conflicts of the B reads).
  int bdma = -1;
  // LUNAEQ_AMD_UVW_BPF: in the register-staged gx/gy kernel, request the next
  // chunk of a path into registers before the current chunk's matrix work, at
  // three waves per SIMD instead of four (1; 163 VGPRs, no spills at config 5:
  // 0.773 -> 0.757 ms, step 2.12 -> 2.07 ms, three processes each); 0: load
  // each chunk just before it is stored to LDS, four waves per SIMD.
  int bpf = 1;
};

constexpr int kChunkRows = 256;  // default batch rows per wave (and per partial) of the weight gradient
constexpr int kReduceGroups = 16;  // parallel groups of partials in the weight-gradient reduction

int read_int(std::istringstream& in, const char* what) {
  long long value;
  if (!(in >> value)) fail(std::string("uvw spec: expected integer for ") + what);
  if (value < 0 || value > (1LL << 31) - 1) fail(std::string("uvw spec: value out of range for ") + what);
  return (int)value;
}

UvwSpec parse(const std::string& text) {
  std::istringstream in(text);
  std::string magic;
  in >> magic;
  if (magic != "LUNAUVW1") fail("uvw spec: missing LUNAUVW1 header");
  UvwSpec s;
  s.dtype_bits = read_int(in, "dtype");
  if (s.dtype_bits != 32) fail("uvw spec: the matrix-core UVW path is fp32");
  s.in1 = read_int(in, "in1");
  s.in2 = read_int(in, "in2");
  s.out = read_int(in, "out");
  s.wnum = read_int(in, "weight_numel");
  const int npaths = read_int(in, "npaths");
  if (npaths <= 0) fail("uvw spec: no paths");
  for (int n = 0; n < npaths; ++n) {
    UvwPath p;
    p.x_off = read_int(in, "x_off");
    p.y_off = read_int(in, "y_off");
    p.out_off = read_int(in, "out_off");
    p.w_off = read_int(in, "w_off");
    p.mul1 = read_int(in, "mul1");
    p.mul2 = read_int(in, "mul2");
    p.mul3 = read_int(in, "mul3");
    p.d1 = read_int(in, "d1");
    p.d2 = read_int(in, "d2");
    p.d3 = read_int(in, "d3");
    const int nterms = read_int(in, "nterms");
    if (p.mul1 <= 0 || p.mul2 <= 0 || p.mul3 <= 0) fail("uvw spec: positive multiplicities required");
    if ((long)p.x_off + (long)p.mul1 * p.d1 > s.in1) fail("uvw spec: input block outside in1_dim");
    if ((long)p.y_off + (long)p.mul2 * p.d2 > s.in2) fail("uvw spec: edge block outside in2_dim");
    if ((long)p.out_off + (long)p.mul3 * p.d3 > s.out) fail("uvw spec: output block outside out_dim");
    if ((long)p.w_off + (long)p.mul1 * p.mul2 * p.mul3 > s.wnum) fail("uvw spec: weights outside weight_numel");
    if (p.d3 > 16) fail("uvw spec: output degree above 7 is not supported");
    // The backward sums over v inside a lane's runs of four consecutive K = (u, v).
    if (4 % p.mul2 != 0) fail("uvw spec: edge multiplicity must be 1, 2 or 4");
    for (int t = 0; t < nterms; ++t) {
      UvwTerm term;
      term.i = read_int(in, "i");
      term.j = read_int(in, "j");
      term.k = read_int(in, "k");
      std::string token;
      in >> token;
      char* end = nullptr;
      term.c = std::strtod(token.c_str(), &end);
      if (token.empty() || *end) fail("uvw spec: bad coefficient");
      if (term.i >= p.d1 || term.j >= p.d2 || term.k >= p.d3) fail("uvw spec: coefficient index out of range");
      p.terms.push_back(term);
    }
    s.paths.push_back(std::move(p));
  }
  return s;
}

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

std::string flit(double c) {
  char b[48];
  std::snprintf(b, sizeof(b), "%.9ef", (double)(float)c);
  return b;
}

int round_up(int v, int m) { return (v + m - 1) / m * m; }

bool overlap(long a0, long a1, long b0, long b1) { return a0 < b1 && b0 < a1; }

// A launch unit: a set of paths whose results one wave combines in registers.
//   forward:  paths writing one output block (out_off, mul3, d3)
//   backward: paths reading one input block (x_off, mul1, d1) with one mul2
struct Unit {
  std::vector<int> paths;
  long lo = 0, hi = 0;  // element range written (out for forward, gx for backward)
  int phase = 0;
  bool accumulate = false;
  int slot_base = 0;    // backward: first gy partial slot (one per K tile)
};

// Units of each phase write disjoint ranges; when ranges of different units
// overlap at all, every unit accumulates into a zero-filled output.
int assign_phases(std::vector<Unit>& units, bool* collision) {
  *collision = false;
  for (size_t a = 0; a < units.size(); ++a)
    for (size_t b = a + 1; b < units.size(); ++b)
      if (overlap(units[a].lo, units[a].hi, units[b].lo, units[b].hi)) *collision = true;
  std::vector<std::vector<std::pair<long, long>>> taken;
  for (Unit& u : units) {
    u.accumulate = *collision;
    int phase = 0;
    for (;; ++phase) {
      if (phase == (int)taken.size()) taken.emplace_back();
      bool clash = false;
      for (const auto& r : taken[phase]) clash = clash || overlap(u.lo, u.hi, r.first, r.second);
      if (!clash) break;
    }
    u.phase = phase;
    taken[phase].push_back({u.lo, u.hi});
  }
  return (int)taken.size();
}

std::vector<Unit> forward_units(const UvwSpec& s) {
  std::vector<Unit> units;
  for (int p = 0; p < (int)s.paths.size(); ++p) {
    const UvwPath& q = s.paths[p];
    bool found = false;
    for (Unit& u : units) {
      const UvwPath& r = s.paths[u.paths[0]];
      if (r.out_off == q.out_off && r.mul3 == q.mul3 && r.d3 == q.d3) {
        u.paths.push_back(p);
        found = true;
        break;
      }
    }
    if (!found) units.push_back({{p}, q.out_off, q.out_off + (long)q.mul3 * q.d3});
  }
  return units;
}

std::vector<Unit> backward_units(const UvwSpec& s) {
  std::vector<Unit> units;
  for (int p = 0; p < (int)s.paths.size(); ++p) {
    const UvwPath& q = s.paths[p];
    bool found = false;
    for (Unit& u : units) {
      const UvwPath& r = s.paths[u.paths[0]];
      if (r.x_off == q.x_off && r.mul1 == q.mul1 && r.d1 == q.d1 && r.mul2 == q.mul2) {
        u.paths.push_back(p);
        found = true;
        break;
      }
    }
    if (!found) units.push_back({{p}, q.x_off, q.x_off + (long)q.mul1 * q.d1});
  }
  return units;
}

int ktiles(const UvwPath& q) { return (q.mul1 * q.mul2 + 31) / 32; }

constexpr int kStageU = 16;  // channels u per LDS chunk of the forward's x staging

// Forward paths whose x block is staged through LDS (16-byte aligned rows,
// whole chunks of channels, one y copy).
bool staged_path(const UvwSpec& s, const UvwPath& q) {
  return s.vec && q.mul2 == 1 && q.mul1 % kStageU == 0 && q.x_off % 4 == 0 && s.in1 % 4 == 0 &&
         (kStageU * q.d1) % 4 == 0;
}


// Forward units computed 64 output channels per wave (two 32-wide matrix
// tiles fed by one Z operand, so the sparse CG work and the x staging are
// shared by twice the matrix work; weights staged per chunk through LDS).
// Needs every path staged and at most 5 output components (160 accumulators).
bool wide_unit(const UvwSpec& s, const Unit& u) {
  if (s.wide == 0) return false;
  const UvwPath& head = s.paths[u.paths[0]];
  if (head.d3 > 5 || head.mul3 <= 32) return false;
  for (int p : u.paths)
    if (!staged_path(s, s.paths[p])) return false;
  return true;
}

// Wide units whose chunks go straight from HBM into LDS (global_load_lds,
// double-buffered: the next chunk streams in while the current one is used):
// weights need 16-byte aligned rows, and mul1 whole chunks of kDmaU channels.
constexpr int kDmaU = 8;
// Units that do not qualify as wide (more than 5 output components, or at
// most 32 channels) take the same LDS copies with one 32-channel tile per
// wave, up to 9 components (144 accumulators).
int dma_tiles(const UvwSpec& s, const Unit& u) {
  if (s.wide != 2) return 0;
  const UvwPath& head = s.paths[u.paths[0]];
  for (int p : u.paths) {
    const UvwPath& q = s.paths[p];
    if (!staged_path(s, q) || q.mul3 % 4 || q.w_off % 4 || q.mul1 % kDmaU || q.d1 > 7) return 0;
  }
  if (wide_unit(s, u)) return 2;
  return head.d3 <= 9 ? 1 : 0;
}
bool dma_unit(const UvwSpec& s, const Unit& u) { return dma_tiles(s, u) > 0; }

int fwd_tiles(const UvwSpec& s, const Unit& u) {
  const int mul3 = s.paths[u.paths[0]].mul3;
  const int dt = dma_tiles(s, u);
  if (dt) return (mul3 + 32 * dt - 1) / (32 * dt);
  return wide_unit(s, u) ? (mul3 + 63) / 64 : (mul3 + 31) / 32;
}

// Backward paths whose seed rows and weights are staged through LDS in
// chunks of 16 output channels.
bool staged_seeds(const UvwSpec& s, const UvwPath& q) {
  return s.vec && q.mul3 % 16 == 0 && q.out_off % 4 == 0 && s.out % 4 == 0 && q.w_off % 4 == 0;
}

// Sorted distinct (i) and (j) indices of a path's terms.
std::set<int> term_is(const UvwPath& q) {
  std::set<int> r;
  for (const auto& t : q.terms) r.insert(t.i);
  return r;
}
std::set<int> term_js(const UvwPath& q) {
  std::set<int> r;
  for (const auto& t : q.terms) r.insert(t.j);
  return r;
}

// c<i>_<k> = sum_j c_ijk y_j of the lane's row: the coupling matrix of one path between
// x_i and output component k.  Formed once per row, it takes one FMA per (i, k)
// and channel where the terms take two per (i, j, k).
void emit_coupling(Code& c, const UvwPath& q, const std::function<std::string(int)>& y) {
  std::set<std::pair<int, int>> begun;
  for (const auto& t : q.terms) {
    const std::string name = "c" + std::to_string(t.i) + "_" + std::to_string(t.k);
    if (begun.insert({t.i, t.k}).second)
      c.line("        real %s = %s * %s;", name.c_str(), flit(t.c).c_str(), y(t.j).c_str());
    else
      c.line("        %s = FMA(%s, %s, %s);", name.c_str(), flit(t.c).c_str(), y(t.j).c_str(), name.c_str());
  }
}
// Distinct (i, k) of a path's terms.
std::set<std::pair<int, int>> term_iks(const UvwPath& q) {
  std::set<std::pair<int, int>> r;
  for (const auto& t : q.terms) r.insert({t.i, t.k});
  return r;
}

// s_waitcnt immediate that waits until at most n vector-memory operations of
// the wave are outstanding (gfx9 encoding: vmcnt bits 3:0 and 15:14; expcnt
// and lgkmcnt left at their maxima, i.e. not waited for).
int vmcnt_imm(int n) {
  if (n < 0 || n > 63) fail("uvw: vmcnt out of range");
  return 0x0F70 | (n & 15) | ((n >> 4) << 14);
}

const char* kPrelude = R"(
typedef float real;
typedef long long i64;
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) float lreal;
typedef __attribute__((address_space(3))) float4 lfloat4;
typedef __attribute__((address_space(3))) void lvoid;
#define FMA(a, b, c) __builtin_fmaf((a), (b), (c))
// D[i][j] += sum_{k<2} A[i][k] B[k][j]; lane l supplies A[l%32][l/32] and
// B[l/32][l%32]; register r of lane l holds D[8(r/4) + 4(l/32) + r%4][l%32].
__device__ __forceinline__ floatx16 mfma32(float a, float b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
)";

// Common head of every kernel: four independent waves per workgroup.
void emit_head(Code& c) {
  c.line("  const int lane = threadIdx.x & 63, hk = lane >> 5, col = lane & 31;");
  c.line("  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);");
}

// Row block rb and tile (unit or path) ut of a workgroup.  With tf set the
// tile index runs fastest over the grid, so the workgroups of one row block
// run together and the units or paths that read the same rows find them in
// the caches (the weight gradient 0.749 -> 0.692 ms at config 5); without
// it (more row blocks than a grid's y extent) the row block runs fastest.
void emit_grid_order(Code& c) {
  c.line("  const int rb = tf ? blockIdx.y : blockIdx.x, ut = tf ? blockIdx.x : blockIdx.y;");
}

// ---------------------------------------------------------------- forward
// out^T[w, b] = sum_p sum_K W_p[K, w] Z_p[b, K] per output component k, on
// the matrix cores with A = W_p^T (rows w, 32 or 64 output channels per wave), B =
// Z_p (32 batch rows per wave), K = (u, v) two per instruction.  Each lane
// produces its own B operand, Z_p[b0 + col, K = 2s + hk, k] for every k, from
// the x and y rows of its batch row (the sparse CG terms as VALU work).
// One wide unit (see wide_unit): a wave owns 32 batch rows and output channels
// w0 .. w0+63; register r of tile t holds channel w0 + 32t + 8(r/4) + 4hk + r%4
// of batch row b0 + col.
void emit_forward_wide(Code& c, const UvwSpec& s, const Unit& u, int nt) {
  const UvwPath& head = s.paths[u.paths[0]];
  const int d3 = head.d3, mul3 = head.mul3;
  c.line("  if (unit < %d) {", nt);
  c.line("    const int w0 = unit * 64;");
  for (int t = 0; t < 2; ++t)
    for (int k = 0; k < d3; ++k) c.line("    floatx16 acc%d_%d = (floatx16)(0.0f);", t, k);
  for (int p : u.paths) {
    const UvwPath& q = s.paths[p];
    const std::set<int> is = term_is(q), js = term_js(q);
    const int chd = kStageU * q.d1;
    const bool wvec = mul3 % 4 == 0 && q.w_off % 4 == 0;
    c.line("    {");
    c.line("      const real* yr = y + (i64)brow * %d + %d;", s.in2, q.y_off);
    for (int j : js) c.line("      const real y%d = yr[%d];", j, j);
    c.line("      for (int c0 = 0; c0 < %d; c0 += %d) {", q.mul1, kStageU);
    c.line("        {");
    // x rows of the chunk: consecutive lanes on consecutive 16-byte pieces.
    c.line("        const float4* xg = (const float4*)(x + %d + c0 * %d);", q.x_off, q.d1);
    c.line("        #pragma unroll 2");
    c.line("        for (int it = 0; it < %d; ++it) {", (32 * chd / 4 + 63) / 64);
    c.line("          const int idx = it * 64 + lane;");
    if ((32 * chd / 4) % 64) c.line("          if (idx < %d) {", 32 * chd / 4);
    else c.line("          {");
    c.line("          const int r = idx / %d, e = idx - r * %d;", chd / 4, chd / 4);
    c.line("          const int rr = b0 + r < B ? b0 + r : B - 1;");
    c.line("          const float4 v = xg[(i64)rr * %d + e];", s.in1 / 4);
    c.line("          real* dst = &xs[wave][r][e * 4];");
    c.line("          dst[0] = v.x; dst[1] = v.y; dst[2] = v.z; dst[3] = v.w;");
    c.line("          }");
    c.line("        }");
    // Weights W_p[c0 .. c0+15, w0 .. w0+63], zero past mul3.
    if (wvec) {
      c.line("        #pragma unroll");
      c.line("        for (int it = 0; it < %d; ++it) {", kStageU * 16 / 64);
      c.line("          const int idx = it * 64 + lane, kk = idx >> 4, w4 = (idx & 15) * 4;");
      c.line("          float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);");
      c.line("          if (w0 + w4 < %d) v = *(const float4*)(wt + %d + (i64)(c0 + kk) * %d + w0 + w4);", mul3,
             q.w_off, mul3);
      c.line("          *(float4*)&ws[wave][kk][w4] = v;");
      c.line("        }");
    } else {
      c.line("        #pragma unroll");
      c.line("        for (int it = 0; it < %d; ++it) {", kStageU);
      c.line("          const int w = w0 + lane;");
      c.line("          ws[wave][it][lane] = w < %d ? wt[%d + (i64)(c0 + it) * %d + w] : 0.0f;", mul3, q.w_off,
             mul3);
      c.line("        }");
    }
    c.line("        }");
    c.line("        const real* xl = &xs[wave][col][0];");
    c.line("        #pragma unroll 2");
    c.line("        for (int s = 0; s < %d; ++s) {", kStageU / 2);
    c.line("          const int ul = 2 * s + hk;");
    for (int i : is) c.line("          const real x%d = xl[ul * %d + %d];", i, q.d1, i);
    c.line("          const real a0 = ws[wave][ul][col], a1 = ws[wave][ul][32 + col];");
    for (int k = 0; k < d3; ++k) c.line("          real z%d = 0;", k);
    for (const auto& t : q.terms)
      c.line("          z%d = FMA(%s, x%d * y%d, z%d);", t.k, flit(t.c).c_str(), t.i, t.j, t.k);
    for (int k = 0; k < d3; ++k) {
      c.line("          acc0_%d = mfma32(a0, z%d, acc0_%d);", k, k, k);
      c.line("          acc1_%d = mfma32(a1, z%d, acc1_%d);", k, k, k);
    }
    c.line("        }");
    c.line("      }");
    c.line("    }");
  }
  c.line("    if (b0 + col < B) {");
  c.line("      real* orow = out + (i64)(b0 + col) * %d + %d;", s.out, head.out_off);
  c.line("      #pragma unroll");
  c.line("      for (int r = 0; r < 16; ++r) {");
  for (int t = 0; t < 2; ++t) {
    c.line("        {");
    c.line("          const int w = w0 + %d + 8 * (r >> 2) + 4 * hk + (r & 3);", 32 * t);
    c.line("          if (w < %d) {", mul3);
    for (int k = 0; k < d3; ++k)
      c.line("            orow[w * %d + %d] %s acc%d_%d[r];", d3, k, u.accumulate ? "+=" : "=", t, k);
    c.line("          }");
    c.line("        }");
  }
  c.line("      }");
  c.line("    }");
  c.line("    return;");
  c.line("  }");
  c.line("  unit -= %d;", nt);
}

// A dma unit (see dma_unit): as emit_forward_wide, with chunks of kDmaU
// channels copied by global_load_lds straight into one of two LDS buffers per
// wave while the other is used, so the next chunk streams in during the
// current chunk's matrix work.  Lane l of copy instruction i lands 16 bytes at
// buffer float 256 i + 4 l, so the x chunk is laid out piece-major: 4-float
// piece `pc` of the chunk's row `row` sits at float (32 pc + row) * 4, and a
// lane reads its row's pieces with 16-byte LDS reads, consecutive lanes on
// consecutive slots.  The two K halves of an MFMA take channels st and st + 4
// of the chunk, so both halves find x_i at the same place in their pieces.
//
// The unit's body is a function whose four buffers are __restrict__
// arguments: inlined, every copy and every LDS read carries the alias scope of
// its buffer, and the compiler waits before a read only for the copies into
// that buffer (without the scopes it waits for every copy in flight).
constexpr int kLateRegisters = 192;
void emit_dma_unit_body(Code& c, const UvwSpec& s, const Unit& u) {
  const UvwPath& head = s.paths[u.paths[0]];
  const int d3 = head.d3, mul3 = head.mul3, T = dma_tiles(s, u), wq = 8 * T;  // wq: 16-byte pieces per K row
  for (int p : u.paths) {
    const UvwPath& q = s.paths[p];
    const std::set<int> is = term_is(q), js = term_js(q);
    const int d1 = q.d1, nch = q.mul1 / kDmaU;
    c.line("  {");
    c.line("    const real* ys = y + (i64)brow * %d + %d;", s.in2, q.y_off);
    for (int j : js) c.line("    const real y%d = ys[%d];", j, j);
    emit_coupling(c, q, [](int j) { return "y" + std::to_string(j); });
    const std::set<std::pair<int, int>> iks = term_iks(q);
    // Fewer input than output components: contract x with the weights first
    // (2 l1 + 1 matrix steps instead of 2 l3 + 1) and couple the results, where
    // both accumulators leave two waves per SIMD without spills.  Forward calls back
    // to back, 200,000 rows, 64 channels, lmax 2: 583 us without, 583 / 566 / 523 us
    // with up to 96 / 128 / 192 registers of accumulators (256 spill 37); 100,000 rows,
    // lmax 1: 108 -> 89 us; 32 channels, lmax 2: 104 -> 97 us.
    const bool late = d1 < d3 && 16 * T * (d1 + d3) <= kLateRegisters;
    c.line("    const real* xrow = x + (i64)rrow * %d + %d + (lane >> 5) * 4;", s.in1, q.x_off);
    c.line("    const real* wrow = wt + %d + (i64)(lane / %d) * %d + wl;", q.w_off, wq, mul3);
    auto copy = [&](const char* chunk, const char* X, const char* W) {
      for (int i = 0; i < d1; ++i)
        c.line("      __builtin_amdgcn_global_load_lds((const void*)(xrow + (%s) * %d + %d), (lvoid*)(%s + %d), 16, 0, 0);",
               chunk, kDmaU * d1, 8 * i, X, 256 * i);
      for (int i = 0; i < T; ++i)
        c.line("      __builtin_amdgcn_global_load_lds((const void*)(wrow + (i64)((%s) * %d + %d) * %d), "
               "(lvoid*)(%s + %d), 16, 0, 0);",
               chunk, kDmaU, 64 / wq * i, mul3, W, 256 * i);
    };
    // Wait until only `left` copies are in flight (vmcnt counts in issue order).
    // The empty asm with a memory clobber keeps the optimizer from moving LDS
    // reads above the wait (the wait intrinsic itself does not order memory
    // accesses); sched_barrier does the same for the machine scheduler.
    auto wait = [&](int left) {
      c.line("      __builtin_amdgcn_s_waitcnt(%d);", vmcnt_imm(left));
      c.line("      asm volatile(\"\" ::: \"memory\");");
      c.line("      __builtin_amdgcn_sched_barrier(0);");
    };
    auto compute = [&](const char* X, const char* W) {
      c.line("      {");
      c.line("        const lfloat4* xp = (const lfloat4*)%s + hk * %d + col;", X, 32 * d1);
      for (int st = 0; st < kDmaU / 2; ++st) {
        c.line("        {");
        std::set<int> pieces;
        for (int i : is) pieces.insert((st * d1 + i) / 4);
        for (int pc : pieces) c.line("          const float4 q%d = xp[%d];", pc, 32 * pc);
        for (int i : is)
          c.line("          const real x%d = q%d.%c;", i, (st * d1 + i) / 4, "xyzw"[(st * d1 + i) % 4]);
        for (int t = 0; t < T; ++t)
          c.line("          const real a%d = %s[(%d + 4 * hk) * %d + %d + col];", t, W, st, 32 * T, 32 * t);
        if (late) {
          for (int i : is)
            for (int t = 0; t < T; ++t) c.line("          xw[%d][%d] = mfma32(a%d, x%d, xw[%d][%d]);", t, i, t, i, t, i);
          c.line("        }");
          continue;
        }
        for (int k = 0; k < d3; ++k) c.line("          real z%d = 0;", k);
        for (const auto& ik : iks)
          c.line("          z%d = FMA(x%d, c%d_%d, z%d);", ik.second, ik.first, ik.first, ik.second, ik.second);
        for (int k = 0; k < d3; ++k)
          for (int t = 0; t < T; ++t) c.line("          acc[%d][%d] = mfma32(a%d, z%d, acc[%d][%d]);", t, k, t, k, t, k);
        c.line("        }");
      }
      c.line("      }");
    };
    const int ncopy = d1 + T;
    if (late) {
      c.line("    floatx16 xw[%d][%d];", T, d1);
      for (int t = 0; t < T; ++t)
        for (int i = 0; i < d1; ++i) c.line("    xw[%d][%d] = (floatx16)(0.0f);", t, i);
    }
    c.line("    {");
    copy("0", "X0", "W0");
    c.line("    }");
    c.line("    #pragma unroll 1");
    c.line("    for (int c = 0; c < %d; c += 2) {", nch);
    copy("c + 1", "X1", "W1");
    wait(ncopy);
    compute("X0", "W0");
    c.line("      if (c + 2 < %d) {", nch);
    copy("c + 2", "X0", "W0");
    wait(ncopy);
    c.line("      } else {");
    wait(0);
    c.line("      }");
    compute("X1", "W1");
    c.line("    }");
    // The next path's copies refill these buffers: nothing may move them above this
    // path's LDS reads (with two chunks the loop is straight-line code, and the
    // scheduler does not order a copy after earlier reads of its buffer).
    c.line("    asm volatile(\"\" ::: \"memory\");");
    c.line("    __builtin_amdgcn_sched_barrier(0);");
    if (late)
      for (const auto& ik : iks)
        for (int t = 0; t < T; ++t)
          c.line("    acc[%d][%d] += c%d_%d * xw[%d][%d];", t, ik.second, ik.first, ik.second, t, ik.first);
    c.line("  }");
  }
}

// The unit branch inside the phase function: tiles of this unit return true
// after storing; others move `unit` past it.
void emit_forward_dma(Code& c, const UvwSpec& s, const Unit& u, int nt) {
  const UvwPath& head = s.paths[u.paths[0]];
  const int d3 = head.d3, mul3 = head.mul3, T = dma_tiles(s, u), wq = 8 * T;
  c.line("  if (unit < %d) {", nt);
  c.line("    const int w0 = unit * %d;", 32 * T);
  c.line("    floatx16 acc[%d][%d];", T, d3);
  for (int t = 0; t < T; ++t)
    for (int k = 0; k < d3; ++k) c.line("    acc[%d][%d] = (floatx16)(0.0f);", t, k);
  c.line("    const int wl = (w0 + (lane %% %d) * 4 < %d) ? w0 + (lane %% %d) * 4 : %d;", wq, mul3, wq, mul3 - 4);
  emit_dma_unit_body(c, s, u);
  c.line("    if (b0 + col < B) {");
  c.line("      real* orow = out + (i64)(b0 + col) * %d + %d;", s.out, head.out_off);
  c.line("      #pragma unroll");
  c.line("      for (int r = 0; r < 16; ++r) {");
  for (int t = 0; t < T; ++t) {
    c.line("        {");
    c.line("          const int w = w0 + %d + 8 * (r >> 2) + 4 * hk + (r & 3);", 32 * t);
    c.line("          if (w < %d) {", mul3);
    for (int k = 0; k < d3; ++k)
      c.line("            orow[w * %d + %d] %s acc[%d][%d][r];", d3, k, u.accumulate ? "+=" : "=", t, k);
    c.line("          }");
    c.line("        }");
  }
  c.line("      }");
  c.line("    }");
  c.line("    return true;");
  c.line("  }");
  c.line("  unit -= %d;", nt);
}

// Every dma unit of a phase in one function, so the four buffers carry the
// same four alias scopes in all of them (the compiler tracks few scopes).
void emit_forward_dma_phase(Code& c, const UvwSpec& s, const std::vector<Unit>& units, int phase) {
  c.line("__device__ __forceinline__ bool fwd_dma_%d(int unit, const real* __restrict__ x,", phase);
  c.line("    const real* __restrict__ y, const real* __restrict__ wt, real* __restrict__ out, int B, int b0,");
  c.line("    int brow, int hk, int col, int lane, lreal* __restrict__ X0, lreal* __restrict__ X1,");
  c.line("    lreal* __restrict__ W0, lreal* __restrict__ W1) {");
  c.line("  const int rrow = b0 + col < B ? b0 + col : B - 1;");
  for (const Unit& u : units) {
    if (u.phase != phase) continue;
    if (dma_unit(s, u)) {
      emit_forward_dma(c, s, u, fwd_tiles(s, u));
    } else {
      // A tile of another kind of unit: the kernel body computes it.
      c.line("  if (unit < %d) return false;", fwd_tiles(s, u));
      c.line("  unit -= %d;", fwd_tiles(s, u));
    }
  }
  c.line("  return false;");
  c.line("}");
}

std::string emit_forward(const UvwSpec& s, const std::vector<Unit>& units, int phases) {
  Code c;
  c.s << kPrelude;
  for (int phase = 0; phase < phases; ++phase) {
    {
      bool any = false;
      for (const Unit& u : units) any = any || (u.phase == phase && dma_unit(s, u));
      if (any) emit_forward_dma_phase(c, s, units, phase);
    }
    bool wide_phase = false;
    for (const Unit& u : units)
      if (u.phase == phase && wide_unit(s, u)) wide_phase = true;
    // Two waves per SIMD for the wide units' 32 d3 accumulator registers.
    c.line("extern \"C\" __global__ void __launch_bounds__(256) %sluna_uvw_fwd_p%d(",
           wide_phase ? "__attribute__((amdgpu_waves_per_eu(2))) " : "", phase);
    c.line("    const real* __restrict__ x, const real* __restrict__ y, const real* __restrict__ wt,");
    c.line("    real* __restrict__ out, int B, int tf) {");
    emit_head(c);
    emit_grid_order(c);
    int stage_d1 = 0;
    for (const Unit& u : units)
      if (u.phase == phase)
        for (int p : u.paths)
          if (staged_path(s, s.paths[p]) && !dma_unit(s, u)) stage_d1 = std::max(stage_d1, s.paths[p].d1);
    bool any_wide = false;
    for (const Unit& u : units)
      if (u.phase == phase && wide_unit(s, u) && !dma_unit(s, u)) any_wide = true;
    int dma_d1 = 0;
    for (const Unit& u : units)
      if (u.phase == phase && dma_unit(s, u))
        for (int p : u.paths) dma_d1 = std::max(dma_d1, s.paths[p].d1);
    // A workgroup runs one unit, so the staging arrays of the different unit
    // kinds share one LDS allocation: xs (row pitch kStageU*d1 + 1, so the 32
    // rows read at one offset fall in 32 banks) and ws of the register-staged
    // units, xwd (two buffers back to back) of the LDS-copied ones.
    const int xs_floats = stage_d1 ? 4 * 32 * (kStageU * stage_d1 + 1) : 0;
    const int ws_floats = any_wide ? 4 * kStageU * 64 : 0;
    const int xwd_pitch = 32 * kDmaU * dma_d1 + kDmaU * 64;
    const int lds_floats = std::max(round_up(xs_floats, 4) + ws_floats, dma_d1 ? 4 * 2 * xwd_pitch : 0);
    if (lds_floats) c.line("  __shared__ __attribute__((aligned(16))) real lds[%d];", lds_floats);
    if (stage_d1) c.line("  real (*xs)[32][%d] = (real (*)[32][%d])lds;", kStageU * stage_d1 + 1, kStageU * stage_d1 + 1);
    if (any_wide) c.line("  real (*ws)[%d][64] = (real (*)[%d][64])(lds + %d);", kStageU, kStageU, round_up(xs_floats, 4));
    if (dma_d1) c.line("  real (*xwd)[2][%d] = (real (*)[2][%d])lds;", xwd_pitch, xwd_pitch);
    c.line("  const int b0 = (rb * 4 + wave) * 32;");
    c.line("  if (b0 >= B) return;");
    c.line("  const int brow = b0 + col < B ? b0 + col : B - 1;");
    if (dma_d1) {
      const int woff = 32 * kDmaU * dma_d1;
      c.line("  if (fwd_dma_%d(ut, x, y, wt, out, B, b0, brow, hk, col, lane, (lreal*)&xwd[wave][0][0],", phase);
      c.line("      (lreal*)&xwd[wave][1][0], (lreal*)&xwd[wave][0][%d], (lreal*)&xwd[wave][1][%d])) return;", woff, woff);
    }
    c.line("  int unit = ut;");
    for (size_t n = 0; n < units.size(); ++n) {
      const Unit& u = units[n];
      if (u.phase != phase) continue;
      const UvwPath& head = s.paths[u.paths[0]];
      const int d3 = head.d3, mul3 = head.mul3;
      const int nt = fwd_tiles(s, u);
      if (dma_unit(s, u)) {
        c.line("  unit -= %d;", nt);
        continue;
      }
      if (wide_unit(s, u)) {
        emit_forward_wide(c, s, u, nt);
        continue;
      }
      c.line("  if (unit < %d) {", nt);
      c.line("    const int w0 = unit * 32;");
      for (int k = 0; k < d3; ++k) c.line("    floatx16 acc%d = (floatx16)(0.0f);", k);
      c.line("    const bool wok = w0 + col < %d;", mul3);
      for (int p : u.paths) {
        const UvwPath& q = s.paths[p];
        const int K = q.mul1 * q.mul2;
        const std::set<int> is = term_is(q), js = term_js(q);
        c.line("    {");
        c.line("      const real* xr = x + (i64)brow * %d + %d;", s.in1, q.x_off);
        c.line("      const real* yr = y + (i64)brow * %d + %d;", s.in2, q.y_off);
        c.line("      const real* wr = wt + %d + (wok ? w0 + col : 0);", q.w_off);
        if (q.mul2 == 1)
          for (int j : js) c.line("      const real y%d = yr[%d];", j, j);
        const int half = (K + 1) / 2;
        if (staged_path(s, q)) {
          // The x block of the wave's 32 rows goes through LDS in chunks of
          // kStageU channels, read from HBM with consecutive lanes on
          // consecutive addresses (a lane-per-row gather costs one cache
          // line per lane in the address unit); lanes then read their own row.
          const int chd = kStageU * q.d1;
          c.line("      for (int c0 = 0; c0 < %d; c0 += %d) {", q.mul1, kStageU);
          c.line("        const float4* xg = (const float4*)(x + %d + c0 * %d);", q.x_off, q.d1);
          c.line("        #pragma unroll 2");
          c.line("        for (int it = 0; it < %d; ++it) {", 32 * chd / 4 / 64);
          c.line("          const int idx = it * 64 + lane, r = idx / %d, e = idx - r * %d;", chd / 4, chd / 4);
          c.line("          const int rr = b0 + r < B ? b0 + r : B - 1;");
          c.line("          const float4 v = xg[(i64)rr * %d + e];", s.in1 / 4);
          c.line("          real* dst = &xs[wave][r][e * 4];");
          c.line("          dst[0] = v.x; dst[1] = v.y; dst[2] = v.z; dst[3] = v.w;");
          c.line("        }");
          c.line("        const real* xl = &xs[wave][col][0];");
          c.line("        #pragma unroll 4");
          c.line("        for (int s = 0; s < %d; ++s) {", kStageU / 2);
          c.line("          const int ul = 2 * s + hk, kk = c0 + ul;");
          for (int i : is) c.line("          const real x%d = xl[ul * %d + %d];", i, q.d1, i);
          c.line("          const real a = wok ? wr[(i64)kk * %d] : 0.0f;", mul3);
          for (int k = 0; k < d3; ++k) c.line("          real z%d = 0;", k);
          for (const auto& t : q.terms)
            c.line("          z%d = FMA(%s, x%d * y%d, z%d);", t.k, flit(t.c).c_str(), t.i, t.j, t.k);
          for (int k = 0; k < d3; ++k) c.line("          acc%d = mfma32(a, z%d, acc%d);", k, k, k);
          c.line("        }");
          c.line("      }");
          c.line("    }");
          continue;
        }
        c.line("      #pragma unroll 4");
        c.line("      for (int s = 0; s < %d; ++s) {", half);
        // An odd K leaves the last upper-half lane without a pair: its A is
        // zero and its loads use the last valid entry.
        c.line("        const int kk = s + hk * %d;", half);
        c.line("        const bool kok = kk < %d;", K);
        c.line("        const int kc = kok ? kk : %d;", K - 1);
        c.line("        const int u = kc / %d, v = kc %% %d;", q.mul2, q.mul2);
        c.line("        (void)v;");
        for (int i : is) c.line("        const real x%d = xr[u * %d + %d];", i, q.d1, i);
        if (q.mul2 != 1)
          for (int j : js) c.line("        const real y%d = yr[v * %d + %d];", j, q.d2, j);
        c.line("        const real a = (kok && wok) ? wr[(i64)kc * %d] : 0.0f;", mul3);
        for (int k = 0; k < d3; ++k) c.line("        real z%d = 0;", k);
        for (const auto& t : q.terms)
          c.line("        z%d = FMA(%s, x%d * y%d, z%d);", t.k, flit(t.c).c_str(), t.i, t.j, t.k);
        for (int k = 0; k < d3; ++k) c.line("        acc%d = mfma32(a, z%d, acc%d);", k, k, k);
        c.line("      }");
        c.line("    }");
      }
      // Register r: output channel w0 + 8(r/4) + 4hk + r%4 of batch row b0 + col.
      c.line("    if (b0 + col < B) {");
      c.line("      real* orow = out + (i64)(b0 + col) * %d + %d;", s.out, head.out_off);
      c.line("      #pragma unroll");
      c.line("      for (int r = 0; r < 16; ++r) {");
      c.line("        const int w = w0 + 8 * (r >> 2) + 4 * hk + (r & 3);");
      c.line("        if (w < %d) {", mul3);
      for (int k = 0; k < d3; ++k)
        c.line("          orow[w * %d + %d] %s acc%d[r];", d3, k, u.accumulate ? "+=" : "=", k);
      c.line("        }");
      c.line("      }");
      c.line("    }");
      c.line("    return;");
      c.line("  }");
      c.line("  unit -= %d;", nt);
    }
    c.line("}");
  }
  return c.s.str();
}

// ---------------------------------------------------------------- backward: gx, gy
// dZ_p^T[K, b] = sum_w W_p[K, w] g[b, oo + w*d3 + k] on the matrix cores with
// v_mfma_f32_16x16x4f32 (A = W_p, 16 K indices per wave; B = the seed rows of
// 16 batch rows; contraction over w, four per instruction).  Lane l then
// holds dZ for batch row b0 + l%16 and the four consecutive K indices
// 16 kt + 4(l/16) + r, so both contractions with the CG terms stay in the lane:
//   gx[b, u, i] += sum_{v,j,k} c y[b, v, j] dZ[b, k, (u, v)]   (v summed in-lane: mul2 | 4)
//   gy[b, v, j] += sum_{u,i,k} c x[b, u, i] dZ[b, k, (u, v)]   (then summed over the
//                                                             four lane groups of a row,
//                                                             one partial slot per K tile)
// A wave covers one input block (all paths reading it with one mul2) and one
// 16-wide K tile, so its gx entries are complete when it stores them.  The
// 16x16 shape keeps the per-lane state small (4 dZ values per component).
int ktiles16(const UvwPath& q) { return (q.mul1 * q.mul2 + 15) / 16; }

std::string emit_backward_xy(const UvwSpec& s, const std::vector<Unit>& units, int phases) {
  Code c;
  c.s << kPrelude;
  c.s << R"(
typedef float floatx4 __attribute__((ext_vector_type(4)));
// D[i][j] += sum_{k<4} A[i][k] B[k][j]; lane l supplies A[l%16][l/16] and
// B[l/16][l%16]; register r of lane l holds D[4(l/16) + r][l%16].
__device__ __forceinline__ floatx4 mfma16(float a, float b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// 16 bytes per lane from src to LDS at dst + 16 lane (dst uniform).  Issued as
// asm so that the compiler does not wait for these copies before unrelated
// LDS reads (it cannot tell the buffers apart); the kernel waits for them
// itself (vmcnt 0) before the barrier that publishes a chunk.  Extra
// outstanding loads only lengthen the compiler's own in-order vmcnt waits.
// Nothing else in these kernels reads M0.
__device__ __forceinline__ void lds_copy16(const void* src, lvoid* dst) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :: "v"(src), "s"((unsigned)(size_t)dst) : "memory");
}
)";
  for (int phase = 0; phase < phases; ++phase) {
    // Four waves per SIMD when the per-lane state is small (short waves whose
    // staging latency is hidden by occupancy: 1.29 -> 1.09 ms at
    // 64x0e+64x1o+64x2e), else two (without the hint the compiler splits the
    // file into VGPRs and AGPRs and leaves one wave per SIMD: 264 registers at
    // 64x0e+64x1o+64x2e+64x3o, 232 with it, no spills).  The estimate counts x
    // and gx entries (4 K rows of d1), dZ (4 d3) and the gy columns, plus
    // addresses and staging temporaries.
    bool four = true;
    for (const Unit& un : units) {
      if (un.phase != phase) continue;
      const UvwPath& head = s.paths[un.paths[0]];
      int d3 = 0;
      std::set<int> ycols;
      for (int p : un.paths) {
        d3 = std::max(d3, s.paths[p].d3);
        for (int v = 0; v < s.paths[p].mul2; ++v)
          for (int j : term_js(s.paths[p])) ycols.insert(s.paths[p].y_off + v * s.paths[p].d2 + j);
      }
      const int estimate = 8 * head.d1 + 4 * d3 + 2 * (int)ycols.size() + 48;
      if (estimate > 128) four = false;
    }
    int stage_d3 = 0, cw = s.bcw;  // w per staged chunk
    bool dma = s.bdma < 0 ? !four : s.bdma != 0;
    for (const Unit& u : units)
      if (u.phase == phase)
        for (int p : u.paths)
          if (staged_seeds(s, s.paths[p])) {
            stage_d3 = std::max(stage_d3, s.paths[p].d3);
            if (s.paths[p].mul3 % cw) cw = 16;
            // Copied rows cannot be zeroed: every K row of the tiles must exist.
            if (s.paths[p].mul1 * s.paths[p].mul2 % 16) dma = false;
          }
    dma = dma && stage_d3;
    Code kc;  // the kernel up to the unit bodies
    kc.line("extern \"C\" __global__ void __launch_bounds__(256) %sluna_uvw_bwd_xy_p%d(",
            four ? (s.bpf && !dma && stage_d3 ? "__attribute__((amdgpu_waves_per_eu(3))) "
                                              : "__attribute__((amdgpu_waves_per_eu(4))) ")
                 : "__attribute__((amdgpu_waves_per_eu(2))) ", phase);
    kc.line("    const real* __restrict__ x, const real* __restrict__ y, const real* __restrict__ wt,");
    kc.line("    const real* __restrict__ g, real* __restrict__ gx, real* __restrict__ part, int B, int tf) {");
    kc.line("  const int lane = threadIdx.x & 63, grp = lane >> 4, c16 = lane & 15;");
    emit_grid_order(kc);
    // The four waves of a workgroup take four K tiles of one input block for
    // the same 16 batch rows and share the staged seed rows.
    if (dma) {
      kc.line("  __shared__ __attribute__((aligned(16))) real gsd[2][%d];", 16 * cw * stage_d3);
      kc.line("  __shared__ __attribute__((aligned(16))) real wsd[2][4][%d];", 16 * cw);
    } else if (stage_d3) {
      kc.line("  __shared__ __attribute__((aligned(16))) real gs[2][16][%d];", cw * stage_d3 + s.gpad);
      kc.line("  __shared__ real wsh[4][16][%d];", cw + s.wpad);
      kc.line("  int chunk = 0;");
    }
    kc.line("  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);");
    kc.line("  const int b0 = rb * 16;");
    kc.line("  if (b0 >= B) return;");
    kc.line("  const bool rok = b0 + c16 < B;");
    kc.line("  const int brow = rok ? b0 + c16 : B - 1;");
    Code ub;  // the unit bodies
    {
    Code& c = ub;
    c.line("  int unit = ut;");
    for (const Unit& un : units) {
      if (un.phase != phase) continue;
      const UvwPath& head = s.paths[un.paths[0]];
      const int m2 = head.mul2, d1 = head.d1, Ktot = head.mul1 * head.mul2;
      const int kts = ktiles16(head);
      const int nq = 4 / m2;
      std::map<int, std::string> cols;
      for (int p : un.paths) {
        const UvwPath& q = s.paths[p];
        for (int v = 0; v < m2; ++v)
          for (int j : term_js(q)) cols[q.y_off + v * q.d2 + j] = "gc" + std::to_string(q.y_off + v * q.d2 + j);
      }
      c.line("  if (unit == 0)");
      c.line("  for (int kt0 = 0; kt0 < %d; kt0 += 4) {", kts);
      c.line("    const bool tok = kt0 + wave < %d;", kts);
      c.line("    const int kt = tok ? kt0 + wave : %d;", kts - 1);
      c.line("    const int ka = kt * 16 + c16;");  // A operand row (K index) of this lane
      c.line("    const bool kaok = ka < %d;", Ktot);
      c.line("    const int kb = kt * 16 + 4 * grp;");  // first of this lane's four D rows
      // Copied chunks: 16-byte piece pc of batch (or K) row r of a chunk lands
      // in LDS slot 16 pc + r (lane l of copy instruction j fills slot
      // 64 j + l), so the 16 rows of a tile read at one offset spread over 16
      // banks.  The seed pieces are shared by the workgroup
      // (instruction j issued by wave j % 4; waves past the last instruction
      // repeat it, the same bytes to the same place, rather than branch);
      // each wave copies its own 16 W rows.
      std::vector<std::pair<int, int>> items;  // (path, chunk) in order
      int item = 0;
      auto dma_copy = [&](int t) {
        const UvwPath& q = s.paths[items[t].first];
        const int cn = items[t].second, par = t & 1, nj = cw * q.d3 / 16;
        for (int i = 0; 4 * i < nj; ++i) {
          const std::string j = 4 * i + 4 <= nj ? "wave" : "min(wave, " + std::to_string(nj - 4 * i - 1) + ")";
          c.line("    lds_copy16(grow + %d + 16 * %s, (lvoid*)(G%d + %d + 256 * %s));", q.out_off + cn * cw * q.d3 + 64 * i,
                 j.c_str(), par, 1024 * i, j.c_str());
        }
        for (int j = 0; j < cw / 16; ++j)
          c.line("    lds_copy16(wt + (i64)ka * %d + %d + 4 * grp, (lvoid*)(W%d + %d));", q.mul3, q.w_off + cn * cw + 16 * j,
                 par, 256 * j);
      };
      if (dma) {
        for (int p : un.paths)
          if (staged_seeds(s, s.paths[p]))
            for (int cn = 0; cn < s.paths[p].mul3 / cw; ++cn) items.push_back({p, cn});
        if (!items.empty()) {
          c.line("    const real* grow = g + (i64)brow * %d + 4 * grp;", s.out);
          dma_copy(0);
        }
      }
      for (int qd = 0; qd < nq; ++qd)
        for (int i = 0; i < d1; ++i) c.line("    real gxa%d_%d = 0;", qd, i);
      for (const auto& kv : cols) c.line("    real %s = 0;", kv.second.c_str());
      // x of this lane's batch row at its four K indices.
      c.line("    const real* xr = x + (i64)brow * %d + %d;", s.in1, head.x_off);
      std::set<int> unit_is;
      for (int p : un.paths)
        for (int i : term_is(s.paths[p])) unit_is.insert(i);
      if (s.vec && m2 == 1 && Ktot % 16 == 0 && head.x_off % 4 == 0 && s.in1 % 4 == 0) {
        // The four K indices of the lane are four consecutive u: 4*d1 floats.
        c.line("    const float4* xv = (const float4*)(xr + (i64)kb * %d);", d1);
        for (int v4 = 0; v4 < d1; ++v4) c.line("    const float4 xq%d = xv[%d];", v4, v4);
        for (int r = 0; r < 4; ++r)
          for (int i : unit_is) {
            const int e = r * d1 + i;
            c.line("    const real x%d_%d = xq%d.%c;", r, i, e / 4, "xyzw"[e % 4]);
          }
      } else {
        for (int r = 0; r < 4; ++r) {
          c.line("    const int u%d = (kb + %d < %d ? kb + %d : %d) / %d;", r, r, Ktot, r, Ktot - 1, m2);
          for (int i : unit_is) c.line("    const real x%d_%d = xr[u%d * %d + %d];", r, i, r, d1, i);
        }
      }
      // Register staging of the gx/gy chunks: chunk `cc` of path q's seed rows
      // (float4 pieces idx = threadIdx.x + 256 it, consecutive lanes on
      // consecutive addresses) and of this wave's 16 W rows, through pg / pw,
      // then into the LDS buffers (rows padded by gpad floats).
      auto stage_per = [&](const UvwPath& q) { return (16 * cw * q.d3 / 4 + 255) / 256; };
      auto stage_load = [&](const UvwPath& q, const char* cc) {
        const int gw = cw * q.d3, total = 16 * gw / 4, per = stage_per(q);
        for (int it = 0; it < per; ++it) {
          c.line("        {");
          c.line("          const int idx = threadIdx.x + %d;", 256 * it);
          c.line("          const int r = idx / %d, e = idx - r * %d;", gw / 4, gw / 4);
          c.line("          const int rr = b0 + r < B ? b0 + r : B - 1;");
          c.line("          if (idx < %d) pg%d = *(const float4*)(g + %d + (%s) * %d + (i64)rr * %d + e * 4);", total, it,
                 q.out_off, cc, cw * q.d3, s.out);
          c.line("        }");
        }
        for (int t = 0; t < cw / 16; ++t) {
          c.line("        {");
          c.line("          const int pq = lane + %d, r = pq / %d, e = pq - r * %d, kr = kt * 16 + r;", 64 * t, cw / 4,
                 cw / 4);
          c.line("          pw%d = kr < %d ? *(const float4*)(wt + %d + (i64)kr * %d + (%s) * %d + e * 4)"
                 " : make_float4(0.0f, 0.0f, 0.0f, 0.0f);", t, Ktot, q.w_off, q.mul3, cc, cw);
          c.line("        }");
        }
      };
      auto stage_store = [&](const UvwPath& q) {
        const int gw = cw * q.d3, total = 16 * gw / 4, per = stage_per(q);
        c.line("        real (*gsb)[%d] = gs[chunk & 1];", cw * stage_d3 + s.gpad);
        for (int it = 0; it < per; ++it) {
          c.line("        {");
          c.line("          const int idx = threadIdx.x + %d;", 256 * it);
          c.line("          const int r = idx / %d, e = idx - r * %d;", gw / 4, gw / 4);
          c.line("          if (idx < %d) {", total);
          c.line("            real* dst = &gsb[r][e * 4];");
          if (s.gpad == 4)
            c.line("            *(float4*)dst = pg%d;", it);
          else if (s.gpad == 2)
            c.line("            ((float2*)dst)[0] = make_float2(pg%d.x, pg%d.y); ((float2*)dst)[1] = "
                   "make_float2(pg%d.z, pg%d.w);", it, it, it, it);
          else
            c.line("            dst[0] = pg%d.x; dst[1] = pg%d.y; dst[2] = pg%d.z; dst[3] = pg%d.w;", it, it, it, it);
          c.line("          }");
          c.line("        }");
        }
        for (int t = 0; t < cw / 16; ++t) {
          c.line("        {");
          c.line("          const int pq = lane + %d, r = pq / %d, e = pq - r * %d;", 64 * t, cw / 4, cw / 4);
          c.line("          real* dst = &wsh[wave][r][e * 4];");
          c.line("          dst[0] = pw%d.x; dst[1] = pw%d.y; dst[2] = pw%d.z; dst[3] = pw%d.w;", t, t, t, t);
          c.line("        }");
        }
      };
      for (int p : un.paths) {
        const UvwPath& q = s.paths[p];
        const int d3 = q.d3, mul3 = q.mul3;
        const int quarter = (mul3 + 3) / 4;
        const std::set<int> js = term_js(q);
        // Lane group grp contracts w in [grp*quarter, grp*quarter + quarter),
        // so each lane's W and g entries are consecutive (16-byte loads of four
        // steps when the layout allows it).
        const bool vec = staged_seeds(s, q);
        c.line("    {");
        c.line("      const real* wr = wt + %d + (i64)(kaok ? ka : %d) * %d + grp * %d;", q.w_off, Ktot - 1, mul3,
               quarter);
        c.line("      const real* gr = g + (i64)brow * %d + %d + grp * %d;", s.out, q.out_off, quarter * d3);
        c.line("      const real* yr = y + (i64)brow * %d + %d;", s.in2, q.y_off);
        for (int v = 0; v < m2; ++v)
          for (int j : js) c.line("      const real y%d_%d = yr[%d];", v, j, v * q.d2 + j);
        for (int v = 0; v < m2; ++v)
          for (int j : js) c.line("      real gp%d_%d = 0;", v, j);
        for (int k = 0; k < d3; ++k) c.line("      floatx4 dz%d = (floatx4)(0.0f);", k);
        if (vec && dma) {
          // Wait for this chunk's copies (all of this wave's copies in flight),
          // make the workgroup's visible, request the next chunk into the
          // other buffers, then the matrix work on this one.  Lane group grp
          // contracts w = 4 ss + grp: A at slot 16 ss + c16, offset grp; B
          // element f = (4 ss + grp) d3 + k of row c16 at slot 16 (f / 4) + c16,
          // offset f % 4, through per-lane bases bq[(k % 4)].  A half-wave
          // (32 banks) reads 16 rows at two offsets, so rows r and r + 8 share
          // a bank: two-way conflicts, which 16-byte pieces cannot pad away.
          c.line("      const int gq = grp * %d;", d3);
          for (int c0 = 0; c0 < std::min(4, d3); ++c0)
            c.line("      const int bq%d = 64 * ((gq + %d) >> 2) + c16 * 4 + ((gq + %d) & 3);", c0, c0, c0);
          for (int cn = 0; cn < mul3 / cw; ++cn, ++item) {
            const int par = item & 1;
            c.line("      {");
            c.line("        __builtin_amdgcn_s_waitcnt(%d);", vmcnt_imm(0));
            c.line("        asm volatile(\"\" ::: \"memory\");");
            c.line("        __builtin_amdgcn_sched_barrier(0);");
            c.line("        __syncthreads();");
            if (item + 1 < (int)items.size()) dma_copy(item + 1);
            c.line("        const lreal* al = W%d + c16 * 4 + grp;", par);
            for (int ss = 0; ss < cw / 4; ++ss) {
              c.line("        {");
              c.line("          const real a = al[%d];", 64 * ss);
              for (int k = 0; k < d3; ++k)
                c.line("          dz%d = mfma16(a, G%d[bq%d + %d], dz%d);", k, par, k & 3, 64 * (ss * d3 + (k >> 2)), k);
              c.line("        }");
            }
            c.line("      }");
          }
        } else if (vec) {
          // Chunks of cw w: the seed rows of the 16 batch rows and the W rows
          // of the 16 K indices go through LDS, read from HBM / L2 with
          // consecutive lanes on consecutive addresses; within a chunk lane
          // group grp takes w = 4 ss + grp.
          const int nch = mul3 / cw;
          for (int it = 0; it < stage_per(q); ++it)
            c.line("      float4 pg%d = make_float4(0.0f, 0.0f, 0.0f, 0.0f);", it);
          for (int t = 0; t < cw / 16; ++t) c.line("      float4 pw%d;", t);
          if (!s.bpf) {
            c.line("      #pragma unroll 1");
            c.line("      for (int cn = 0; cn < %d; ++cn) {", nch);
            stage_load(q, "cn");
            stage_store(q);
            c.line("        __syncthreads();");
          } else {
            // Chunk 0 requested before the loop; each iteration stores the
            // chunk in registers to LDS, then requests the next one before this
            // chunk's matrix work.  (Also requesting the next path's chunk 0
            // during the last chunk measured slower: 0.754 -> 0.801 ms.)
            stage_load(q, "0");
            c.line("      #pragma unroll 1");
            c.line("      for (int cn = 0; cn < %d; ++cn) {", nch);
            stage_store(q);
            c.line("        __syncthreads();");
            c.line("        if (cn + 1 < %d) {", nch);
            stage_load(q, "(cn + 1)");
            c.line("        }");
          }
          c.line("        const real* gl = &gs[chunk & 1][c16][0];");
          c.line("        const real* al = &wsh[wave][c16][0];");
          c.line("        ++chunk;");
          for (int ss = 0; ss < cw / 4; ++ss) {
            c.line("        {");
            c.line("          const int wl = %d + grp;", 4 * ss);
            c.line("          const real a = al[wl];");
            for (int k = 0; k < d3; ++k) c.line("          dz%d = mfma16(a, gl[wl * %d + %d], dz%d);", k, d3, k, k);
            c.line("        }");
          }
          c.line("      }");
        } else {
          c.line("      #pragma unroll 4");
          c.line("      for (int s = 0; s < %d; ++s) {", quarter);
          c.line("        const int w = grp * %d + s;", quarter);
          c.line("        const bool wok = w < %d;", mul3);
          c.line("        const int sc = wok ? s : %d - grp * %d;", mul3 - 1, quarter);
          c.line("        const real a = (kaok && wok) ? wr[sc] : 0.0f;");
          for (int k = 0; k < d3; ++k) c.line("        dz%d = mfma16(a, gr[sc * %d + %d], dz%d);", k, d3, k, k);
          c.line("      }");
        }
        // Per (i, k), over the lane's K rows: gx_i += c_ik dZ_k with c_ik = sum_j c_ijk y_j,
        // and gy_j += c_ijk s_ik with s_ik = sum x_i dZ_k (8 operations a pair and
        // 2 a term; term by term it was 13 a term, 83 terms on 79 pairs at lmax 2).
        // 200,000 rows, 64 channels, lmax 2: step 1,918 -> 1,904 us.
        for (const auto& ik : term_iks(q)) {
          const int i = ik.first, k = ik.second;
          for (int v = 0; v < m2; ++v) {
            std::string coupling;
            for (const auto& t : q.terms) {
              if (t.i != i || t.k != k) continue;
              const std::string yv = "y" + std::to_string(v) + "_" + std::to_string(t.j);
              coupling = coupling.empty() ? flit(t.c) + " * " + yv : "FMA(" + flit(t.c) + ", " + yv + ", " + coupling + ")";
            }
            c.line("      {");
            c.line("        const real cik = %s;", coupling.c_str());
            for (int r = v; r < 4; r += m2) c.line("        gxa%d_%d = FMA(cik, dz%d[%d], gxa%d_%d);", r / m2, i, k, r, r / m2, i);
            c.line("        real sik = x%d_%d * dz%d[%d];", v, i, k, v);
            for (int r = v + m2; r < 4; r += m2) c.line("        sik = FMA(x%d_%d, dz%d[%d], sik);", r, i, k, r);
            for (const auto& t : q.terms)
              if (t.i == i && t.k == k)
                c.line("        gp%d_%d = FMA(%s, sik, gp%d_%d);", v, t.j, flit(t.c).c_str(), v, t.j);
            c.line("      }");
          }
        }
        // Sum over the four lane groups that share a batch row.
        for (int v = 0; v < m2; ++v)
          for (int j : js) {
            c.line("      gp%d_%d += __shfl_xor(gp%d_%d, 16, 64);", v, j, v, j);
            c.line("      gp%d_%d += __shfl_xor(gp%d_%d, 32, 64);", v, j, v, j);
            c.line("      %s += gp%d_%d;", cols[q.y_off + v * q.d2 + j].c_str(), v, j);
          }
        c.line("    }");
      }
      c.line("    if (rok && tok) {");
      c.line("      real* gq = gx + (i64)brow * %d + %d;", s.in1, head.x_off);
      for (int qd = 0; qd < nq; ++qd) {
        const int r = qd * m2;
        c.line("      if (kb + %d < %d) {", r, Ktot);
        c.line("        const int ur = (kb + %d) / %d;", r, m2);
        for (int i = 0; i < d1; ++i)
          c.line("        gq[ur * %d + %d] %s gxa%d_%d;", d1, i, un.accumulate ? "+=" : "=", qd, i);
        c.line("      }");
      }
      c.line("      if (grp == 0 && tok) {");
      c.line("        real* pr = part + ((i64)(%d + kt) * B + brow) * %d;", un.slot_base, s.in2);
      for (const auto& kv : cols) c.line("        pr[%d] = %s;", kv.first, kv.second.c_str());
      c.line("      }");
      c.line("    }");
      // The next K tiles' first copy reuses buffer 0.
      if (dma && kts > 4 && !items.empty()) c.line("    __syncthreads();");
      c.line("  }");
      c.line("  unit -= 1;");
    }
    }
    if (dma) {
      c.line("__device__ __forceinline__ void bxy_units_%d(const real* __restrict__ x, const real* __restrict__ y,", phase);
      c.line("    const real* __restrict__ wt, const real* __restrict__ g, real* __restrict__ gx, real* __restrict__ part,");
      c.line("    int B, int lane, int grp, int c16, int wave, int b0, bool rok, int brow, int ut,");
      c.line("    lreal* __restrict__ G0, lreal* __restrict__ G1, lreal* __restrict__ W0, lreal* __restrict__ W1) {");
      c.s << ub.s.str();
      c.line("}");
      c.s << kc.s.str();
      c.line("  bxy_units_%d(x, y, wt, g, gx, part, B, lane, grp, c16, wave, b0, rok, brow, ut, (lreal*)&gsd[0][0],", phase);
      c.line("              (lreal*)&gsd[1][0], (lreal*)&wsd[0][wave][0], (lreal*)&wsd[1][wave][0]);");
    } else {
      c.s << kc.s.str() << ub.s.str();
    }
    c.line("}");
  }
  // gy[b, col] = sum of the partial slots that hold column col.
  std::vector<std::vector<int>> writers(s.in2);
  for (const Unit& un : units) {
    const UvwPath& head = s.paths[un.paths[0]];
    std::set<int> cols;
    for (int p : un.paths) {
      const UvwPath& q = s.paths[p];
      for (int v = 0; v < q.mul2; ++v)
        for (int j : term_js(q)) cols.insert(q.y_off + v * q.d2 + j);
    }
    for (int col : cols)
      for (int kt = 0; kt < ktiles16(head); ++kt) writers[col].push_back(un.slot_base + kt);
  }
  c.line("extern \"C\" __global__ void __launch_bounds__(256) luna_uvw_bwd_gy(");
  c.line("    const real* __restrict__ part, real* __restrict__ gy, int B) {");
  c.line("  const int b = blockIdx.x * 256 + threadIdx.x;");
  c.line("  if (b >= B) return;");
  for (int col = 0; col < s.in2; ++col) {
    std::string sum;
    for (int slot : writers[col]) {
      char term[96];
      std::snprintf(term, sizeof(term), "part[((i64)%d * B + b) * %d + %d]", slot, s.in2, col);
      sum += (sum.empty() ? "" : " + ") + std::string(term);
    }
    c.line("  gy[(i64)b * %d + %d] = %s;", s.in2, col, sum.empty() ? "0.0f" : sum.c_str());
  }
  c.line("}");
  return c.s.str();
}

// ---------------------------------------------------------------- backward: weights
// dW_p[K, w] = sum_{b,k} Z_p[b, k, K] g[b, oo + w*d3 + k]: A = Z_p (rows K,
// produced in-lane for K = 32 mt + l%32 from batch row 2s + l/32), B = the
// seed rows (columns w), contraction over (b, k) two batch rows per
// instruction and one instruction per k.  Each wave owns kChunkRows rows of
// one path and writes one partial of dW_p; a second kernel sums the partials.
// Weight-gradient paths whose x, seed and y rows are copied by global_load_lds
// into two LDS buffers per wave, UvwSpec::wrows rows at a time, the next rows in flight
// during the current rows' matrix work (UvwSpec::wdma).
// Rows stay row-major in LDS: a lane reads x[row][u d1 + i] and
// g[row][w d3 + k] for consecutive u or w, an odd stride, so no bank conflicts.
int bw_pieces(const UvwSpec& s, int floats_per_row) { return (s.wrows * floats_per_row / 4 + 63) / 64 * 64; }
// LDS of a workgroup (four waves, two buffers of x, seed and y rows) for one path.
int bw_lds_bytes(const UvwSpec& s, const UvwPath& q) {
  return 4 * 2 * (bw_pieces(s, q.mul1 * q.d1) * 4 + bw_pieces(s, q.mul3 * q.d3) * 4 + 64) * 4;
}
bool bw_dma_eligible(const UvwSpec& s, const UvwPath& q) {
  if (!s.wdma) return false;
  return q.mul2 == 1 && (q.mul1 * q.d1) % 4 == 0 && (q.mul3 * q.d3) % 4 == 0 && q.x_off % 4 == 0 &&
         q.out_off % 4 == 0 && s.in1 % 4 == 0 && s.out % 4 == 0 && q.d2 * s.wrows <= 64 &&
         bw_lds_bytes(s, q) <= 128 * 1024;
}
// The paths that use the LDS copies.  They share one buffer sized by the
// largest x block and the largest seed block over the set, which may come
// from different paths: the widest paths leave the set until that union fits
// the 128 KiB budget.
std::vector<bool> bw_dma_set(const UvwSpec& s) {
  std::vector<bool> in(s.paths.size());
  for (size_t p = 0; p < s.paths.size(); ++p) in[p] = bw_dma_eligible(s, s.paths[p]);
  for (;;) {
    int xmax = 0, gmax = 0, widest = -1, width = -1;
    for (size_t p = 0; p < s.paths.size(); ++p) {
      if (!in[p]) continue;
      const UvwPath& q = s.paths[p];
      const int x = bw_pieces(s, q.mul1 * q.d1) * 4, g = bw_pieces(s, q.mul3 * q.d3) * 4;
      xmax = std::max(xmax, x);
      gmax = std::max(gmax, g);
      if (x + g > width) width = x + g, widest = (int)p;
    }
    if (widest < 0 || 4 * 2 * (xmax + gmax + 64) * 4 <= 128 * 1024) return in;
    in[widest] = false;
  }
}
bool bw_dma_path(const UvwSpec& s, const UvwPath& q) {
  const size_t p = (size_t)(&q - s.paths.data());
  if (p >= s.paths.size()) return false;
  return bw_dma_set(s)[p];
}

// All such paths in one function (four __restrict__ buffers, so the
// compiler's waits before LDS reads cover only the copies into the buffer
// being read).  Returns false for other paths.
void emit_bw_dma(Code& c, const UvwSpec& s, int chunk_rows) {
  c.line("__device__ __forceinline__ bool bw_dma(int path, const real* __restrict__ x, const real* __restrict__ y,");
  c.line("    const real* __restrict__ g, real* __restrict__ part, int B, int chunk, int r0, int lane, int col,");
  c.line("    int hk, lreal* __restrict__ X0, lreal* __restrict__ X1, lreal* __restrict__ G0,");
  c.line("    lreal* __restrict__ G1, lreal* __restrict__ Y0, lreal* __restrict__ Y1) {");
  for (int p = 0; p < (int)s.paths.size(); ++p) {
    const UvwPath& q = s.paths[p];
    if (!bw_dma_path(s, q)) continue;
    const int K = q.mul1, mt = ktiles(q), nt = (q.mul3 + 31) / 32, d3 = q.d3, d1 = q.d1;
    const int px = q.mul1 * d1, pg = q.mul3 * d3;  // floats per row of the x block and of the seed block
    const int nx = bw_pieces(s, px) / 64, ng = bw_pieces(s, pg) / 64, ncopy = nx + ng + 1;
    const int d2 = q.d2;
    const int nch = chunk_rows / s.wrows;
    const std::set<int> is = term_is(q), js = term_js(q);
    const std::set<std::pair<int, int>> iks = term_iks(q);
    c.line("  if (path == %d) {", p);
    for (int m = 0; m < mt; ++m)
      for (int n = 0; n < nt; ++n) c.line("    floatx16 acc%d_%d = (floatx16)(0.0f);", m, n);
    for (int m = 0; m < mt; ++m) {
      c.line("    const bool kok%d = %d + col < %d;", m, m * 32, K);
      c.line("    const int xu%d = (kok%d ? %d + col : %d) * %d;", m, m, m * 32, K - 1, d1);
    }
    for (int n = 0; n < nt; ++n) {
      c.line("    const bool wok%d = %d + col < %d;", n, n * 32, q.mul3);
      c.line("    const int gw%d = (wok%d ? %d + col : %d) * %d;", n, n, n * 32, q.mul3 - 1, d3);
    }
    // Copy instruction i, lane l: 16-byte piece 64 i + l of the rows, row-major
    // (pieces past the rows re-read the last piece into the buffer's tail).
    for (int i = 0; i < nx; ++i) {
      c.line("    const int xpc%d = 64 * %d + lane < %d ? 64 * %d + lane : %d;", i, i, s.wrows * px / 4, i,
             s.wrows * px / 4 - 1);
      c.line("    const int xrow%d = xpc%d / %d, xoff%d = %d + (xpc%d - xrow%d * %d) * 4;", i, i, px / 4, i, q.x_off, i, i,
             px / 4);
    }
    for (int i = 0; i < ng; ++i) {
      c.line("    const int gpc%d = 64 * %d + lane < %d ? 64 * %d + lane : %d;", i, i, s.wrows * pg / 4, i,
             s.wrows * pg / 4 - 1);
      c.line("    const int grow%d = gpc%d / %d, goff%d = %d + (gpc%d - grow%d * %d) * 4;", i, i, pg / 4, i, q.out_off, i,
             i, pg / 4);
    }
    // y: one 4-byte copy per lane, lane l = (row l / d2, column l % d2).
    c.line("    const int yl = lane < %d ? lane : %d;", s.wrows * d2, s.wrows * d2 - 1);
    c.line("    const int yrow = yl / %d, ycol = %d + yl - yrow * %d;", d2, q.y_off, d2);
    auto copy = [&](const char* cb, const char* X, const char* G, const char* Y) {
      for (int i = 0; i < nx; ++i)
        c.line("      __builtin_amdgcn_global_load_lds((const void*)(x + (i64)min(%s + xrow%d, B - 1) * %d + xoff%d), "
               "(lvoid*)(%s + %d), 16, 0, 0);", cb, i, s.in1, i, X, 256 * i);
      for (int i = 0; i < ng; ++i)
        c.line("      __builtin_amdgcn_global_load_lds((const void*)(g + (i64)min(%s + grow%d, B - 1) * %d + goff%d), "
               "(lvoid*)(%s + %d), 16, 0, 0);", cb, i, s.out, i, G, 256 * i);
      c.line("      __builtin_amdgcn_global_load_lds((const void*)(y + (i64)min(%s + yrow, B - 1) * %d + ycol), "
             "(lvoid*)%s, 4, 0, 0);", cb, s.in2, Y);
    };
    // The empty asm with a memory clobber keeps the optimizer from moving LDS
    // reads above the wait (the wait intrinsic itself does not order memory
    // accesses); sched_barrier does the same for the machine scheduler.
    auto wait = [&](int left) {
      c.line("      __builtin_amdgcn_s_waitcnt(%d);", vmcnt_imm(left));
      c.line("      asm volatile(\"\" ::: \"memory\");");
      c.line("      __builtin_amdgcn_sched_barrier(0);");
    };
    auto compute = [&](const char* cb, const char* X, const char* G, const char* Y) {
      for (int sp = 0; sp < s.wrows / 2; ++sp) {
        c.line("      {");
        c.line("        const bool rok = %s + %d + hk < B;", cb, 2 * sp);
        for (int j : js) c.line("        const real y%d_%d = %s[(%d + hk) * %d + %d];", sp, j, Y, 2 * sp, d2, j);
        c.line("        const lreal* xl = %s + (%d + hk) * %d;", X, 2 * sp, px);
        c.line("        const lreal* gl = %s + (%d + hk) * %d;", G, 2 * sp, pg);
        emit_coupling(c, q, [&](int j) { return "y" + std::to_string(sp) + "_" + std::to_string(j); });
        // The shorter of the two forms: sum_k z_k g_k with z_k = sum_i x_i c_ik, or
        // sum_i x_i h_i with h_i = sum_k c_ik g_k (2 l1 + 1 < 2 l3 + 1 matrix steps).
        // Bound by the matrix instructions: at 64 channels, lmax 2, 108 of 140 remain
        // per pair of rows; 200,000 rows, beside the gx/gy kernel: step 1,998 -> 1,851 us.
        // A path of weight 0 has no terms and takes the first form, whose z are then 0.
        const bool seeds = d1 < d3 && !q.terms.empty();
        for (int m = 0; m < mt; ++m)
          for (int i : is)
            c.line("        const real x%d_%d = %sxl[xu%d + %d]%s;", m, i,
                   seeds ? ("(rok && kok" + std::to_string(m) + ") ? ").c_str() : "", m, i, seeds ? " : 0.0f" : "");
        for (int n = 0; n < nt; ++n)
          for (int k = 0; k < d3; ++k) c.line("        const real g%d_%d = wok%d ? gl[gw%d + %d] : 0.0f;", n, k, n, n, k);
        auto contract = [&](const char* to, const char* from, int tiles, int width, bool over_i) {
          for (int m = 0; m < tiles; ++m) {
            for (int v = 0; v < width; ++v) c.line("        real %s%d_%d = 0;", to, m, v);
            for (const auto& ik : iks)
              c.line("        %s%d_%d = FMA(%s%d_%d, c%d_%d, %s%d_%d);", to, m, over_i ? ik.second : ik.first, from, m,
                     over_i ? ik.first : ik.second, ik.first, ik.second, to, m, over_i ? ik.second : ik.first);
            for (int v = 0; v < width; ++v)
              c.line("        %s%d_%d = (rok%s) ? %s%d_%d : 0.0f;", to, m, v,
                     over_i ? (" && kok" + std::to_string(m)).c_str() : "", to, m, v);
          }
        };
        if (seeds)
          contract("h", "g", nt, d1, false);
        else
          contract("z", "x", mt, d3, true);
        for (int v = 0; v < (seeds ? d1 : d3); ++v)
          for (int m = 0; m < mt; ++m)
            for (int n = 0; n < nt; ++n)
              c.line("        acc%d_%d = mfma32(%s%d_%d, %s%d_%d, acc%d_%d);", m, n, seeds ? "x" : "z", m, v,
                     seeds ? "h" : "g", n, v, m, n);
        c.line("      }");
      }
    };
    c.line("    {");
    copy("r0", "X0", "G0", "Y0");
    c.line("    }");
    c.line("    #pragma unroll 1");
    c.line("    for (int cc = 0; cc < %d; cc += 2) {", nch);
    c.line("      const int ca = r0 + cc * %d, cb = ca + %d;", s.wrows, s.wrows);
    copy("cb", "X1", "G1", "Y1");
    wait(ncopy);
    compute("ca", "X0", "G0", "Y0");
    c.line("      if (cc + 2 < %d) {", nch);
    const std::string next = "cb + " + std::to_string(s.wrows);
    copy(next.c_str(), "X0", "G0", "Y0");
    wait(ncopy);
    c.line("      } else {");
    wait(0);
    c.line("      }");
    compute("cb", "X1", "G1", "Y1");
    c.line("    }");
    // Register r: K = 32 m + 8(r/4) + 4hk + r%4, w = 32 n + col.
    c.line("    real* pr = part + (i64)chunk * %d + %d;", s.wnum, q.w_off);
    for (int m = 0; m < mt; ++m)
      for (int n = 0; n < nt; ++n) {
        c.line("    if (wok%d) {", n);
        c.line("      #pragma unroll");
        c.line("      for (int r = 0; r < 16; ++r) {");
        c.line("        const int kr = %d + 8 * (r >> 2) + 4 * hk + (r & 3);", m * 32);
        c.line("        if (kr < %d) pr[(i64)kr * %d + %d + col] = acc%d_%d[r];", K, q.mul3, 32 * n, m, n);
        c.line("      }");
        c.line("    }");
      }
    c.line("    return true;");
    c.line("  }");
  }
  c.line("  return false;");
  c.line("}");
}

std::string emit_backward_w(const UvwSpec& s, int chunk_rows) {
  Code c;
  c.s << kPrelude;
  int xmax = 0, gmax = 0;
  for (const auto& q : s.paths)
    if (bw_dma_path(s, q)) {
      xmax = std::max(xmax, bw_pieces(s, q.mul1 * q.d1) * 4);
      gmax = std::max(gmax, bw_pieces(s, q.mul3 * q.d3) * 4);
    }
  if (xmax) emit_bw_dma(c, s, chunk_rows);
  c.line("extern \"C\" __global__ void __launch_bounds__(256) luna_uvw_bwd_w(");
  c.line("    const real* __restrict__ x, const real* __restrict__ y, const real* __restrict__ g,");
  c.line("    real* __restrict__ part, int B, int tf) {");
  if (xmax) c.line("  __shared__ __attribute__((aligned(16))) real buf[4][2][%d];", xmax + gmax + 64);
  emit_head(c);
  emit_grid_order(c);
  c.line("  const int chunk = rb * 4 + wave;");
  c.line("  const int r0 = chunk * %d;", chunk_rows);
  c.line("  if (r0 >= B) return;");
  c.line("  const int path = ut;");
  if (xmax) {
    c.line("  if (bw_dma(path, x, y, g, part, B, chunk, r0, lane, col, hk, (lreal*)&buf[wave][0][0],");
    c.line("             (lreal*)&buf[wave][1][0], (lreal*)&buf[wave][0][%d], (lreal*)&buf[wave][1][%d],", xmax, xmax);
    c.line("             (lreal*)&buf[wave][0][%d], (lreal*)&buf[wave][1][%d])) return;", xmax + gmax, xmax + gmax);
  }
  for (int p = 0; p < (int)s.paths.size(); ++p) {
    const UvwPath& q = s.paths[p];
    const int K = q.mul1 * q.mul2, mt = ktiles(q), nt = (q.mul3 + 31) / 32, d3 = q.d3;
    const std::set<int> is = term_is(q), js = term_js(q);
    c.line("  if (path == %d) {", p);
    for (int m = 0; m < mt; ++m)
      for (int n = 0; n < nt; ++n) c.line("    floatx16 acc%d_%d = (floatx16)(0.0f);", m, n);
    for (int m = 0; m < mt; ++m) {
      c.line("    const int k%d = %d + col;", m, m * 32);
      c.line("    const int u%d = (k%d < %d ? k%d : %d) / %d, v%d = (k%d < %d ? k%d : %d) %% %d;", m, m, K, m, K - 1,
             q.mul2, m, m, K, m, K - 1, q.mul2);
      c.line("    const bool kok%d = k%d < %d;", m, m, K);
    }
    for (int n = 0; n < nt; ++n) {
      c.line("    const int w%d = %d + col;", n, n * 32);
      c.line("    const bool wok%d = w%d < %d;", n, n, q.mul3);
    }
    c.line("    #pragma unroll 2");
    c.line("    for (int s = 0; s < %d; ++s) {", chunk_rows / 2);
    c.line("      const int row = r0 + 2 * s + hk;");
    c.line("      const bool rok = row < B;");
    c.line("      const int rc = rok ? row : B - 1;");
    c.line("      const real* xr = x + (i64)rc * %d + %d;", s.in1, q.x_off);
    c.line("      const real* yr = y + (i64)rc * %d + %d;", s.in2, q.y_off);
    c.line("      const real* gr = g + (i64)rc * %d + %d;", s.out, q.out_off);
    for (int m = 0; m < mt; ++m) {
      c.line("      const bool zok%d = rok && kok%d;", m, m);
      for (int i : is) c.line("      const real x%d_%d = xr[u%d * %d + %d];", m, i, m, q.d1, i);
      for (int j : js) c.line("      const real y%d_%d = yr[v%d * %d + %d];", m, j, m, q.d2, j);
      for (int k = 0; k < d3; ++k) c.line("      real z%d_%d = 0;", m, k);
      for (const auto& t : q.terms)
        c.line("      z%d_%d = FMA(%s, x%d_%d * y%d_%d, z%d_%d);", m, t.k, flit(t.c).c_str(), m, t.i, m, t.j, m, t.k);
      for (int k = 0; k < d3; ++k) c.line("      z%d_%d = zok%d ? z%d_%d : 0.0f;", m, k, m, m, k);
    }
    for (int n = 0; n < nt; ++n)
      for (int k = 0; k < d3; ++k)
        c.line("      const real g%d_%d = (rok && wok%d) ? gr[(wok%d ? w%d : 0) * %d + %d] : 0.0f;", n, k, n, n, n, d3,
               k);
    for (int k = 0; k < d3; ++k)
      for (int m = 0; m < mt; ++m)
        for (int n = 0; n < nt; ++n) c.line("      acc%d_%d = mfma32(z%d_%d, g%d_%d, acc%d_%d);", m, n, m, k, n, k, m, n);
    c.line("    }");
    // Register r: K = 32 m + 8(r/4) + 4hk + r%4, w = 32 n + col.
    c.line("    real* pr = part + (i64)chunk * %d + %d;", s.wnum, q.w_off);
    for (int m = 0; m < mt; ++m)
      for (int n = 0; n < nt; ++n) {
        c.line("    if (wok%d) {", n);
        c.line("      #pragma unroll");
        c.line("      for (int r = 0; r < 16; ++r) {");
        c.line("        const int kr = %d + 8 * (r >> 2) + 4 * hk + (r & 3);", m * 32);
        c.line("        if (kr < %d) pr[(i64)kr * %d + w%d] = acc%d_%d[r];", K, q.mul3, n, m, n);
        c.line("      }");
        c.line("    }");
      }
    c.line("    return;");
    c.line("  }");
  }
  c.line("}");
  // gw[i] = sum over chunks of part[chunk][i], in two passes: kReduceGroups
  // groups of chunks in parallel, then the group sums, for covered entries.
  c.line("extern \"C\" __global__ void __launch_bounds__(256) luna_uvw_bwd_w_reduce(");
  c.line("    const real* __restrict__ part, real* __restrict__ part2, int chunks) {");
  c.line("  const int i = blockIdx.x * 256 + threadIdx.x;");
  c.line("  if (i >= %d) return;", s.wnum);
  c.line("  const int per = (chunks + %d) / %d;", kReduceGroups - 1, kReduceGroups);
  c.line("  const int n0 = blockIdx.y * per, n1 = n0 + per < chunks ? n0 + per : chunks;");
  c.line("  real a0 = 0, a1 = 0, a2 = 0, a3 = 0;");
  c.line("  int n = n0;");
  c.line("  for (; n + 3 < n1; n += 4) {");
  c.line("    a0 += part[(i64)n * %d + i];", s.wnum);
  c.line("    a1 += part[(i64)(n + 1) * %d + i];", s.wnum);
  c.line("    a2 += part[(i64)(n + 2) * %d + i];", s.wnum);
  c.line("    a3 += part[(i64)(n + 3) * %d + i];", s.wnum);
  c.line("  }");
  c.line("  for (; n < n1; ++n) a0 += part[(i64)n * %d + i];", s.wnum);
  c.line("  part2[(i64)blockIdx.y * %d + i] = (a0 + a1) + (a2 + a3);", s.wnum);
  c.line("}");
  c.line("extern \"C\" __global__ void __launch_bounds__(256) luna_uvw_bwd_w_final(");
  c.line("    const real* __restrict__ part2, real* __restrict__ gw) {");
  c.line("  const int i = blockIdx.x * 256 + threadIdx.x;");
  c.line("  if (i >= %d) return;", s.wnum);
  std::string covered;
  for (const auto& q : s.paths) {
    char term[96];
    std::snprintf(term, sizeof(term), "(i >= %d && i < %d)", q.w_off, q.w_off + q.mul1 * q.mul2 * q.mul3);
    covered += (covered.empty() ? "" : " || ") + std::string(term);
  }
  c.line("  if (!(%s)) return;", covered.c_str());
  c.line("  real acc = 0;");
  c.line("  for (int n = 0; n < %d; ++n) acc += part2[(i64)n * %d + i];", kReduceGroups, s.wnum);
  c.line("  gw[i] = acc;");
  c.line("}");
  return c.s.str();
}

struct UvwPlan {
  UvwSpec spec;
  ModuleCache kernels;
  std::vector<Unit> fwd_units, bwd_units;
  int fwd_phases = 0, bwd_phases = 0;
  std::vector<int> fwd_phase_tiles, bwd_phase_tiles;  // grid.y per phase
  int gy_slots = 0;
  int chunk_rows = kChunkRows;
  bool out_needs_zero = false, gx_needs_zero = false, gy_needs_zero = false, gw_needs_zero = false;
};

std::string source_for(const UvwPlan& plan, const std::string& variant) {
  if (variant == "fwd") return emit_forward(plan.spec, plan.fwd_units, plan.fwd_phases);
  if (variant == "bxy") return emit_backward_xy(plan.spec, plan.bwd_units, plan.bwd_phases);
  return emit_backward_w(plan.spec, plan.chunk_rows);
}

bool covers(const std::vector<std::pair<long, long>>& ranges, long total) {
  std::vector<std::pair<long, long>> r = ranges;
  std::sort(r.begin(), r.end());
  long at = 0;
  for (const auto& x : r) {
    if (x.first > at) return false;
    at = std::max(at, x.second);
  }
  return at >= total;
}

}  // namespace
}  // namespace luna

using namespace luna;

struct LunaUvwPlan {
  UvwPlan plan;
};

namespace {

hipModule_t module_for(UvwPlan& plan, const std::string& variant) {
  return plan.kernels.module_for(variant, [&] { return source_for(plan, variant); });
}

int64_t chunks_for(const UvwPlan& p, int64_t rows) { return (rows + p.chunk_rows - 1) / p.chunk_rows; }

size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }
size_t gw_part_bytes(const UvwPlan& p, int64_t rows) {
  return align256((size_t)chunks_for(p, rows) * (size_t)p.spec.wnum * sizeof(float)) +
         align256((size_t)kReduceGroups * (size_t)p.spec.wnum * sizeof(float));
}
size_t gy_part_bytes(const UvwPlan& p, int64_t rows) {
  return align256((size_t)p.gy_slots * (size_t)rows * (size_t)p.spec.in2 * sizeof(float));
}
// LUNAEQ_AMD_UVW_CONC=0 runs the two backward kernels one after the other.
bool concurrent_backward() {
  const char* e = std::getenv("LUNAEQ_AMD_UVW_CONC");
  return !e || std::atoi(e) != 0;
}

// Grid of `blocks` row blocks by `tiles` tiles, the tile index fastest when the
// row blocks fit the grid's y extent (*tf = 1), else the row block fastest.
// The kernels read the order from tf.
dim3 grid2(unsigned blocks, unsigned tiles, int* tf) {
  const char* e = std::getenv("LUNAEQ_AMD_UVW_TF");
  *tf = (!e || std::atoi(e) != 0) && blocks <= 65535u;
  return *tf ? dim3(tiles, blocks) : dim3(blocks, tiles);
}

unsigned row_blocks(int64_t rows, int rows_per_wave) {  // 4 waves per workgroup
  return (unsigned)((rows + 4 * rows_per_wave - 1) / (4 * rows_per_wave));
}

}  // namespace

extern "C" {

int luna_uvw_plan_create(const char* spec, const char* cache_dir, LunaUvwPlan** out) {
  return guard_call([&] {
    if (!spec || !out) fail("luna_uvw_plan_create: null argument");
    auto holder = std::make_unique<LunaUvwPlan>();
    UvwPlan& p = holder->plan;
    p.spec = parse(spec);
    const char* vec = std::getenv("LUNAEQ_AMD_UVW_VEC");
    const char* wide = std::getenv("LUNAEQ_AMD_UVW_WIDE");
    const char* wdma = std::getenv("LUNAEQ_AMD_UVW_WDMA");
    p.spec.vec = !vec || std::atoi(vec) != 0;
    p.spec.wide = wide ? std::atoi(wide) : 2;
    p.spec.wdma = !wdma || std::atoi(wdma) != 0;
    if (const char* wr = std::getenv("LUNAEQ_AMD_UVW_WROWS")) p.spec.wrows = std::atoi(wr) == 4 ? 4 : 2;
    if (const char* gp = std::getenv("LUNAEQ_AMD_UVW_GPAD")) {
      const int v = std::atoi(gp);
      p.spec.gpad = v == 1 || v == 4 ? v : 2;
    }
    if (const char* wp = std::getenv("LUNAEQ_AMD_UVW_WPAD")) p.spec.wpad = std::atoi(wp) == 1 ? 1 : 2;
    if (const char* bcw = std::getenv("LUNAEQ_AMD_UVW_BCW")) p.spec.bcw = std::atoi(bcw) == 16 ? 16 : 32;
    if (const char* bd = std::getenv("LUNAEQ_AMD_UVW_BDMA")) p.spec.bdma = std::atoi(bd) != 0 ? 1 : 0;
    if (const char* bp = std::getenv("LUNAEQ_AMD_UVW_BPF")) p.spec.bpf = std::atoi(bp) != 0 ? 1 : 0;

    p.kernels.cache_dir = cache_dir ? cache_dir : "";
    p.kernels.tag = "uvw";
    std::vector<std::pair<long, long>> xs, ws;
    for (const auto& q : p.spec.paths) {
      xs.push_back({q.x_off, q.x_off + (long)q.mul1 * q.d1});
      ws.push_back({q.w_off, q.w_off + (long)q.mul1 * q.mul2 * q.mul3});
    }
    p.fwd_units = forward_units(p.spec);
    bool out_collision = false, gx_collision = false;
    p.fwd_phases = assign_phases(p.fwd_units, &out_collision);
    p.fwd_phase_tiles.assign(p.fwd_phases, 0);
    std::vector<std::pair<long, long>> outs;
    for (const Unit& u : p.fwd_units) {
      p.fwd_phase_tiles[u.phase] += fwd_tiles(p.spec, u);
      outs.push_back({u.lo, u.hi});
    }
    p.bwd_units = backward_units(p.spec);
    p.bwd_phases = assign_phases(p.bwd_units, &gx_collision);
    p.bwd_phase_tiles.assign(p.bwd_phases, 0);
    for (Unit& u : p.bwd_units) {
      u.slot_base = p.gy_slots;
      p.gy_slots += ktiles16(p.spec.paths[u.paths[0]]);
      p.bwd_phase_tiles[u.phase] += 1;
    }
    for (int t : p.fwd_phase_tiles)
      if (t > 65535) fail("uvw: too many output tiles for one launch");
    for (int t : p.bwd_phase_tiles)
      if (t > 65535) fail("uvw: too many input blocks for one launch");
    p.out_needs_zero = out_collision || !covers(outs, p.spec.out);
    p.gx_needs_zero = gx_collision || !covers(xs, p.spec.in1);
    p.gy_needs_zero = false;  // the gy reduction writes every column
    p.gw_needs_zero = !covers(ws, p.spec.wnum);
    *out = holder.release();
  });
}

int luna_uvw_plan_destroy(LunaUvwPlan* plan) {
  return guard_call([&] { delete plan; });
}

int luna_uvw_plan_needs_zero(const LunaUvwPlan* plan, int32_t* flags) {
  return guard_call([&] {
    if (!plan || !flags) fail("luna_uvw_plan_needs_zero: null argument");
    flags[0] = plan->plan.out_needs_zero;
    flags[1] = plan->plan.gx_needs_zero;
    flags[2] = plan->plan.gy_needs_zero;
    flags[3] = plan->plan.gw_needs_zero;
  });
}

int luna_uvw_plan_precompile(LunaUvwPlan* plan) {
  return guard_call([&] {
    if (!plan) fail("luna_uvw_plan_precompile: null plan");
    for (const char* v : {"fwd", "bxy", "bw"})
      plan->plan.kernels.code_for(v, [&] { return source_for(plan->plan, v); });
  });
}

int luna_uvw_fwd(const LunaUvwPlan* cplan, const void* x, const void* y, const void* weight, void* out,
                 int64_t rows, LunaStream stream) {
  return guard_call([&] {
    if (!cplan) fail("luna_uvw_fwd: null plan");
    if (rows < 0 || rows > 0x7fffffffLL) fail("luna_uvw_fwd: bad row count");
    if (rows == 0) return;
    if (!x || !y || !weight || !out) fail("luna_uvw_fwd: null tensor");
    UvwPlan& plan = const_cast<LunaUvwPlan*>(cplan)->plan;
    hipModule_t module = module_for(plan, "fwd");
    int B = (int)rows;
    int tf = 0;
    for (int phase = 0; phase < plan.fwd_phases; ++phase) {
      void* args[] = {&x, &y, &weight, &out, &B, &tf};
      launch("uvw_fwd", function_for(module, "luna_uvw_fwd_p" + std::to_string(phase)),
             grid2(row_blocks(rows, 32), (unsigned)plan.fwd_phase_tiles[phase], &tf), dim3(256), (hipStream_t)stream,
             args);
    }
  });
}

int luna_uvw_bwd_workspace(const LunaUvwPlan* plan, int64_t rows, size_t* bytes) {
  return guard_call([&] {
    if (!plan || !bytes) fail("luna_uvw_bwd_workspace: null argument");
    if (rows < 0) fail("negative row count");
    *bytes = gw_part_bytes(plan->plan, rows) + gy_part_bytes(plan->plan, rows);
  });
}

int luna_uvw_bwd(const LunaUvwPlan* cplan, const void* x, const void* y, const void* weight, const void* g,
                 void* gx, void* gy, void* gw, void* workspace, size_t workspace_bytes, int64_t rows,
                 LunaStream stream) {
  return guard_call([&] {
    if (!cplan) fail("luna_uvw_bwd: null plan");
    if (rows < 0 || rows > 0x7fffffffLL) fail("luna_uvw_bwd: bad row count");
    // An empty batch may come with null row tensors (gw is then zero).
    if (!weight || (rows > 0 && (!x || !y || !g))) fail("luna_uvw_bwd: null tensor");
    UvwPlan& plan = const_cast<LunaUvwPlan*>(cplan)->plan;
    hipStream_t s = (hipStream_t)stream;
    int B = (int)rows;
    const size_t need = gw_part_bytes(plan, rows) + gy_part_bytes(plan, rows);
    if ((((gx || gy) && rows > 0) || gw) && (!workspace || workspace_bytes < need))
      fail("luna_uvw_bwd: workspace too small");
    char* ws = (char*)workspace;
    void* gw_part = ws;
    void* gy_part = ws + gw_part_bytes(plan, rows);
    if ((gx || gy) && rows > 0 && (!gx || !gy)) fail("luna_uvw_bwd: gx and gy are produced together");
    // gx/gy and the weight gradient read the same inputs and write disjoint
    // outputs; each leaves the matrix cores partly idle, so with both wanted
    // the weight gradient runs on a second stream beside gx/gy.
    auto run_xy = [&](hipStream_t st) {
      hipModule_t module = module_for(plan, "bxy");
      int tf = 0;
      for (int phase = 0; phase < plan.bwd_phases; ++phase) {
        void* args[] = {&x, &y, &weight, &g, &gx, &gy_part, &B, &tf};
        launch("uvw_bwd_xy", function_for(module, "luna_uvw_bwd_xy_p" + std::to_string(phase)),
               grid2((unsigned)((rows + 15) / 16), (unsigned)plan.bwd_phase_tiles[phase], &tf), dim3(256), st, args);
      }
      void* args[] = {&gy_part, &gy, &B};
      launch("uvw_bwd_gy", function_for(module, "luna_uvw_bwd_gy"), dim3((unsigned)((rows + 255) / 256)), dim3(256),
             st, args);
    };
    auto run_w = [&](hipStream_t st) {
      hipModule_t module = module_for(plan, "bw");
      const int64_t chunks = chunks_for(plan, rows);
      if (rows > 0) {
        int tf = 0;
        void* args[] = {&x, &y, &g, &gw_part, &B, &tf};
        launch("uvw_bwd_w", function_for(module, "luna_uvw_bwd_w"),
               grid2((unsigned)((chunks + 3) / 4), (unsigned)plan.spec.paths.size(), &tf), dim3(256), st, args);
      }
      int n = (int)chunks;
      void* part2 = (char*)gw_part + align256((size_t)chunks * (size_t)plan.spec.wnum * sizeof(float));
      void* args[] = {&gw_part, &part2, &n};
      launch("uvw_bwd_w_reduce", function_for(module, "luna_uvw_bwd_w_reduce"),
             dim3((unsigned)((plan.spec.wnum + 255) / 256), kReduceGroups), dim3(256), st, args);
      void* args2[] = {&part2, &gw};
      launch("uvw_bwd_w_final", function_for(module, "luna_uvw_bwd_w_final"),
             dim3((unsigned)((plan.spec.wnum + 255) / 256)), dim3(256), st, args2);
    };
    const bool want_xy = (gx || gy) && rows > 0;
    if (want_xy && gw && concurrent_backward()) {
      // Load both modules first: nothing below may block between fork and join.
      module_for(plan, "bxy");
      module_for(plan, "bw");
      fork_join(s, run_w, [&] { run_xy(s); });
    } else {
      if (want_xy) run_xy(s);
      if (gw) run_w(s);
    }
  });
}

}  // extern "C"
