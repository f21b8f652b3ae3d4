"""Index arithmetic of the UVU kernels at the top of the int32 edge range, run on the host.

The emitted kernels of one-path layers are compiled as ordinary C++ and run lane by lane for nodes
that own the last k edges of a graph of 2^31 - 1 edges.  The edge arrays are sparse mappings between
unreadable pages, so an index that wraps ends the program; sums and per-edge results are whole
numbers and compared exactly.  The same runs with 64-bit offsets beyond 2^31 edges.
"""

import re
import shutil
import subprocess
from pathlib import Path

import pytest

from lunaequivariance_amd import _native

ROOT = Path(__file__).resolve().parents[1]
CLANG = shutil.which("clang++") or "/opt/rocm/llvm/bin/clang++"
HIP_INCLUDE = Path("/opt/rocm/include")

pytestmark = pytest.mark.skipif(not (Path(CLANG).exists() and HIP_INCLUDE.exists()), reason="needs clang++ and HIP headers")

EMIT = r"""
#include <fstream>
#include "%s/lunaequivariance_amd/csrc/uvu_plan.h"
int main(int argc, char** argv) {
  luna::Plan plan;
  plan.spec = luna::parse_spec(argv[1]);
  plan.edge_index_bits = std::stoi(argv[2]);
  luna::build_schedule(plan);
  const std::string to = argv[3];
  std::ofstream(to + "/fwd.h") << luna::emit_forward(plan, false, false, false);
  std::ofstream(to + "/fws.h") << luna::emit_forward(plan, false, false, true);
  std::ofstream(to + "/bwd.h") << luna::emit_backward(plan, false, false, true, true, true);
  std::ofstream(to + "/plan.h") << "constexpr int kTeams = " << luna::gather_teams(plan) << ", kColumns = "
                                << luna::gather_columns(plan) << ", kVector = " << luna::gather_vector_width(plan)
                                << ";\nconstexpr bool kComponentMajor = " << luna::message_component_major(plan) << ";\n";
}
"""

RUN = r"""
#include <sys/mman.h>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
struct Dim { unsigned x, y, z; } threadIdx, blockIdx, blockDim = {64, 1, 1}, gridDim = {1, 1, 1};
#define __device__
#define __global__
#define __forceinline__ inline
#define __launch_bounds__(n)
#define __shared__ static
#define __syncthreads()
#define __builtin_amdgcn_wave_barrier()
#define __builtin_amdgcn_readfirstlane(v) (v)
// Lanes of the one active channel keep their own share; the others hold zeros.
#define __builtin_amdgcn_mov_dpp(...) 0
#define __builtin_amdgcn_ds_swizzle(...) 0
#define __builtin_amdgcn_ds_bpermute(...) 0
inline int __float_as_int(float) { return 0; }
inline float __int_as_float(int) { return 0; }
inline int __double2hiint(double) { return 0; }
inline int __double2loint(double) { return 0; }
inline double __hiloint2double(int, int) { return 0; }
inline int min(int a, int b) { return a < b ? a : b; }
#include "plan.h"
namespace fwd {
#include "fwd.h"
}
namespace fws {
#include "fws.h"
}
namespace bwd {
#include "bwd.h"
}
typedef fwd::eix eix;
typedef float real;

// `n` zeros with 32 GB of unreadable addresses on both sides.
template <typename T>
T* sparse(long long n) {
  const size_t guard = 32ULL << 30, size = ((size_t)n * sizeof(T) + 4095) & ~(size_t)4095;
  char* p = (char*)mmap(nullptr, size + 2 * guard, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (p == MAP_FAILED || mprotect(p + guard, size, PROT_READ | PROT_WRITE)) { puts("no address space"); exit(77); }
  return (T*)(p + guard + size - (size_t)n * sizeof(T));
}
// Every lane of a workgroup in turn, twice: the second time the LDS holds the others' values.
template <typename F>
void workgroup(int threads, F kernel) {
  blockDim.x = threads;
  for (int pass = 0; pass < 2; ++pass)
    for (threadIdx.x = 0; threadIdx.x < (unsigned)threads; ++threadIdx.x) kernel();
}
#define EXPECT(c) if (!(c)) { printf("%s: %d edges\n", #c, k); return 1; }

int main() {
  const long long E = EDGES;
  const int C = CHANNELS;
  int* src = sparse<int>(E);
  eix* ebs = sparse<eix>(E);
  real *y = sparse<real>(E), *w = sparse<real>(E * C), *gw = sparse<real>(E * C), *msg = sparse<real>(E * C), *part = sparse<real>(2 * E);
  static real x[64], g[64], out[64], gx[64];
  static int order[1];
  for (int c = 0; c < C; ++c) x[c] = g[c] = 1;
  for (long long e = E - MOST; e < E; ++e) {
    y[e] = 1;
    ebs[e] = (eix)e;
    for (int c = 0; c < C; ++c) w[e * C + c] = 1;
  }
  for (int k = 0; k <= MOST; ++k) {
    const eix rowptr[2] = {(eix)(E - k), (eix)E};
    workgroup(64, [&] { fwd::luna_uvu_fwd_p0(x, y, w, nullptr, src, rowptr, order, out, nullptr); });
    for (int c = 0; c < C; ++c) EXPECT(out[c] == k);
    for (int split = 2; split <= 8; split *= 2) {
      workgroup(64 * split, [&] { fws::luna_uvu_fwd_p0(x, y, w, nullptr, src, rowptr, order, out, nullptr); });
      for (int c = 0; c < C; ++c) EXPECT(out[c] == k);
    }
    for (gridDim.z = 1; gridDim.z <= 8; gridDim.z *= 2) {
      for (long long e = E - MOST; e < E; ++e) part[2 * e] = 0;
      memset(gw + (E - MOST) * C, 0, sizeof(real) * MOST * C);
      memset(msg + (E - MOST) * C, 0, sizeof(real) * MOST * C);
      for (blockIdx.z = 0; blockIdx.z < gridDim.z; ++blockIdx.z)
        workgroup(64, [&] { bwd::luna_uvu_bwd_p0(x, y, w, nullptr, g, nullptr, src, rowptr, order, gw, msg, part, E); });
      blockIdx.z = 0;
      for (long long e = E - MOST; e < E; ++e) {
        const bool mine = e >= E - k;
        for (int c = 0; c < C; ++c) EXPECT(gw[e * C + c] == mine && msg[e * C + c] == mine);
        if (C == 1) EXPECT(part[2 * e] == mine);
      }
    }
    gridDim.z = 1;
    workgroup(kTeams * kColumns, [&] { bwd::luna_uvu_bwd_gather(msg, rowptr, ebs, gx); });
    for (int c = 0; c < C; ++c) EXPECT(gx[c] == k);
  }
  puts("ok");
}
"""


def host_source(text):
    """The kernels as host C++: no C linkage (three modules share names), no inline assembly."""
    text = text.replace('extern "C" ', "")
    text = text.replace("extern __shared__ __attribute__((aligned(16))) unsigned char obuf_lds[];",
                        "static __attribute__((aligned(16))) unsigned char obuf_lds[65536];")
    return re.sub(r"asm(?: volatile)?\([^;]*\);", ";", text)


@pytest.fixture(scope="module")
def emitter(tmp_path_factory):
    to = tmp_path_factory.mktemp("emit")
    (to / "emit.cpp").write_text(EMIT % ROOT)
    library = Path(_native.LIBRARY_PATH)
    subprocess.run([CLANG, "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", f"-I{HIP_INCLUDE}", str(to / "emit.cpp"),
                    str(library), f"-Wl,-rpath,{library.parent}", "-Wl,--allow-shlib-undefined", "-o", str(to / "emit")],
                   check=True)
    return to / "emit"


@pytest.mark.parametrize("channels", [1, 9, 17, 33])  # 8, 4, 2 edges at once and one
@pytest.mark.parametrize("bits,edges", [(32, 2 ** 31 - 1), (64, 2 ** 31 + 2 ** 12)])
def test_last_edges_of_a_graph(emitter, tmp_path, bits, edges, channels):
    spec = (f"LUNAUVU1 32 {channels} 1 {channels} {channels} 1 {channels}\n"
            f"0 0 0 0 1 {channels} 1 1 1 0 1 0 0 0 1.0\n")
    subprocess.run([str(emitter), spec, str(bits), str(tmp_path)], check=True)
    for name in ("fwd", "fws", "bwd"):
        path = tmp_path / f"{name}.h"
        path.write_text(host_source(path.read_text()))
    most = 2 * 8 * 8 * 2 + 3  # two rounds of the widest look-ahead and a remainder
    (tmp_path / "run.cpp").write_text(
        RUN.replace("EDGES", f"{edges}LL").replace("CHANNELS", str(channels)).replace("MOST", str(most)))
    # Signed sums wrap, as on the device.
    subprocess.run([CLANG, "-std=c++17", "-O1", "-w", "-fwrapv", str(tmp_path / "run.cpp"), "-o", str(tmp_path / "run")],
                   check=True)
    done = subprocess.run([str(tmp_path / "run")], capture_output=True, text=True)
    if done.returncode == 77:
        pytest.skip(done.stdout)
    assert done.returncode == 0 and done.stdout.strip() == "ok", (done.returncode, done.stdout)


# ---- the UUU convolution's loops

EMIT_UUU = r"""
#include <fstream>
#include "%s/lunaequivariance_amd/csrc/uuu.cpp"
int main(int argc, char** argv) {
  LunaUuuPlan* plan = nullptr;
  if (luna_uuu_plan_create_ex(argv[1], "", std::stoi(argv[2]), &plan)) return 1;
  const std::string to = argv[3];
  std::ofstream(to + "/fwd.h") << luna::emit_forward(plan->plan, false, true);
  std::ofstream(to + "/bwd.h") << luna::emit_backward(plan->plan, false, false, true, true, true, true);
}
"""

# Every edge's own results (scalar features; gy, gw and the env-gradient partials) are written by the
# lane that takes it; sums over lanes are not formed here.
RUN_UUU = RUN[:RUN.index('#include "plan.h"')] + r"""
#define __align__(n) __attribute__((aligned(n)))
namespace fwd {
#include "fwd.h"
}
namespace bwd {
#include "bwd.h"
}
typedef fwd::eix eix;
typedef float real;
""" + RUN[RUN.index("// `n` zeros"):RUN.index("int main()")] + r"""
int main() {
  const long long E = EDGES;
  const int C = CHANNELS;
  int* other = sparse<int>(E);
  eix* ids = sparse<eix>(E);
  real *y = sparse<real>(E * C), *w = sparse<real>(E * C), *l0 = sparse<real>(E * C), *gy = sparse<real>(E * C);
  real *gw = sparse<real>(E * C), *part = sparse<real>(E);
  static real x[64], g[64], out[64], gx[64];
  static int order[1];
  for (int c = 0; c < C; ++c) x[c] = g[c] = 1;
  for (long long e = E - MOST; e < E; ++e) {
    ids[e] = (eix)e;
    for (int c = 0; c < C; ++c) y[e * C + c] = w[e * C + c] = 1;
  }
  for (int k = 0; k <= MOST; k += k < 70 ? 1 : 61) {
    const eix rowptr[2] = {(eix)(E - k), (eix)E};
    for (int split = 1; split <= 8; split *= 2) {
      real* const results[] = {l0, gy, gw};
      for (real* p : results) memset(p + (E - MOST) * C, 0, sizeof(real) * MOST * C);
      memset(part + (E - MOST), 0, sizeof(real) * MOST);
      workgroup(64 * split, [&] { fwd::luna_uuu_fwd_g0(x, y, w, nullptr, other, rowptr, order, out, l0, split); });
      workgroup(64 * split, [&] {
        bwd::luna_uuu_bwd_g0(x, y, w, nullptr, g, nullptr, other, rowptr, ids, order, gx, gy, gw, part, split, E);
      });
      for (long long e = E - MOST; e < E; ++e) {
        const bool mine = e >= E - k;
        for (int c = 0; c < C; ++c) EXPECT(l0[e * C + c] == mine && gy[e * C + c] == mine && gw[e * C + c] == mine);
        EXPECT(part[e] == mine);
      }
    }
  }
  puts("ok");
}
"""


@pytest.fixture(scope="module")
def uuu_emitter(tmp_path_factory):
    to = tmp_path_factory.mktemp("emit_uuu")
    (to / "emit.cpp").write_text(EMIT_UUU % ROOT)
    library = Path(_native.LIBRARY_PATH)
    subprocess.run([CLANG, "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", f"-I{HIP_INCLUDE}", str(to / "emit.cpp"),
                    str(library), f"-Wl,-rpath,{library.parent}", "-Wl,--unresolved-symbols=ignore-all", "-o",
                    str(to / "emit")], check=True)
    return to / "emit"


@pytest.mark.parametrize("channels", [1, 3, 33])  # 64 and 16 edges at once, and one
@pytest.mark.parametrize("bits,edges", [(32, 2 ** 31 - 1), (64, 2 ** 31 + 2 ** 12)])
def test_last_edges_of_a_graph_uuu(uuu_emitter, tmp_path, bits, edges, channels):
    spec = (f"LUNAUUU1 32 {channels} {channels} {channels} {channels} 1 {channels}\n"
            f"0 0 0 0 {channels} 1 1 1 0 1 0 0 0 1.0\n")
    subprocess.run([str(uuu_emitter), spec, str(bits), str(tmp_path)], check=True)
    for name in ("fwd", "bwd"):
        path = tmp_path / f"{name}.h"
        text = host_source(path.read_text())
        path.write_text(re.sub(r"extern __shared__ __align__\(16\) unsigned char lds\[\];",
                               "static __align__(16) unsigned char lds[1 << 20];", text))
    most = 2 * 64 * 8 + 3  # two rounds of the widest step and a remainder
    (tmp_path / "run.cpp").write_text(
        RUN_UUU.replace("EDGES", f"{edges}LL").replace("CHANNELS", str(channels)).replace("MOST", str(most)))
    # Signed sums wrap, as on the device.
    subprocess.run([CLANG, "-std=c++17", "-O1", "-w", "-fwrapv", str(tmp_path / "run.cpp"), "-o", str(tmp_path / "run")],
                   check=True)
    done = subprocess.run([str(tmp_path / "run")], capture_output=True, text=True)
    if done.returncode == 77:
        pytest.skip(done.stdout)
    assert done.returncode == 0 and done.stdout.strip() == "ok", (done.returncode, done.stdout)


# ---- the graph tables' source segments

RUN_SEGMENTS = r"""
#include <cstdio>
struct Dim { unsigned x, y, z; } threadIdx, blockIdx;
typedef long long i64;
typedef unsigned u32;
#define __global__
#define __launch_bounds__(n)
#define __shfl_xor(v, m, w) (v)
#define __hip_atomic_load(p, order, scope) (*(p))
inline void atomicMax(long long* p, long long v) { if (v > *p) *p = v; }
inline int max(int a, int b) { return a > b ? a : b; }
inline int min(int a, int b) { return a < b ? a : b; }
KERNELS
int main() {
  const int E = 2147483646;  // the most edges of the builder
  for (int degree = 1; degree <= 100; ++degree) {
    const int rowptr[2] = {E - degree, E};
    int count, nodes[4], begin[4], end[4];
    u32 in_key, out_key, seg_key[4];
    i64 status[8] = {};
    luna_graph_segment_counts(rowptr, rowptr, 1, &count, status);
    if (count != (degree + 31) / 32 || status[5] != degree) { printf("count of %d\n", degree); return 1; }
    const int seg_rowptr[2] = {0, count};
    luna_graph_node_keys(rowptr, rowptr, seg_rowptr, 1, degree, &in_key, &out_key, nodes, begin, end, seg_key);
    for (int s = 0; s < count; ++s)
      if (begin[s] != E - degree + 32 * s || end[s] != (s + 1 < count ? begin[s] + 32 : E)) { printf("segment of %d\n", degree); return 1; }
  }
  // One node with every edge.
  const int hub[2] = {0, E};
  int count;
  i64 status[8] = {};
  luna_graph_segment_counts(hub, hub, 1, &count, status);
  if (count != E / 32 + 1) { puts("count of the hub"); return 1; }
  puts("ok");
}
"""


def test_segments_of_the_last_edges(tmp_path):
    source = (ROOT / "lunaequivariance_amd" / "csrc" / "graph.cpp").read_text()
    kernels = "\n".join(
        re.search(r'extern "C" __global__ void __launch_bounds__\(256\) ' + name + r"\(.*?\n}\n", source, re.S).group(0)
        for name in ("luna_graph_segment_counts", "luna_graph_node_keys"))
    (tmp_path / "run.cpp").write_text(RUN_SEGMENTS.replace("KERNELS", kernels))
    subprocess.run([CLANG, "-std=c++17", "-O1", "-w", "-fwrapv", str(tmp_path / "run.cpp"), "-o", str(tmp_path / "run")],
                   check=True)
    done = subprocess.run([str(tmp_path / "run")], capture_output=True, text=True)
    assert done.returncode == 0 and done.stdout.strip() == "ok", (done.returncode, done.stdout)
