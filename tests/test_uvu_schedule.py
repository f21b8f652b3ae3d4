"""Which lanes the UVU kernels give to channels and to edges, read from the built plans (no GPU)."""

import shutil
import subprocess
from pathlib import Path

import pytest

from lunaequivariance_amd import _native

ROOT = Path(__file__).resolve().parents[1]
CLANG = shutil.which("clang++") or "/opt/rocm/llvm/bin/clang++"
HIP_INCLUDE = Path("/opt/rocm/include")

pytestmark = pytest.mark.skipif(not (Path(CLANG).exists() and HIP_INCLUDE.exists()), reason="needs clang++ and HIP headers")


def run(tmp_path, body):
    (tmp_path / "plan.cpp").write_text(
        f'#include <cstdio>\n#include "{ROOT}/include/lunaeq_amd.h"\n'
        f'#include "{ROOT}/lunaequivariance_amd/csrc/uvu_plan.h"\n' + body)
    library = Path(_native.LIBRARY_PATH)
    subprocess.run([CLANG, "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", f"-I{HIP_INCLUDE}", str(tmp_path / "plan.cpp"),
                    str(library), f"-Wl,-rpath,{library.parent}", "-Wl,--unresolved-symbols=ignore-all", "-o",
                    str(tmp_path / "plan")], check=True)
    return subprocess.run([str(tmp_path / "plan")], capture_output=True, text=True, check=True).stdout.split()


PLAN = r"""
// One scalar path of `channels` channels.
LunaUvuPlan* plan_of(int channels) {
  char spec[128];
  snprintf(spec, sizeof(spec), "LUNAUVU1 32 %d 1 %d %d 1 %d\n0 0 0 0 1 %d 1 1 1 0 1 0 0 0 1.0\n", channels, channels,
           channels, channels, channels);
  LunaUvuPlan* plan = nullptr;
  if (luna_uvu_plan_create(spec, "", &plan)) puts("failed");
  return plan;
}
"""


def test_chunk_widths(tmp_path):
    """Up to 32 channels in chunks of a power of two from 8 on; more in whole waves only."""
    channels = [1, 8, 9, 16, 17, 32, 33, 64, 65, 80, 96, 129, 160]
    out = run(tmp_path, PLAN + r"""
int main() {
  for (int channels : {%s}) {
    LunaUvuPlan* plan = plan_of(channels);
    printf("%%d:%%d:%%d\n", plan->plan.fwd_groups[0].cw, plan->plan.fwd_groups[0].chunks, plan->plan.bwd_groups[0].cw);
  }
}""" % ",".join(map(str, channels)))
    width = [8, 8, 16, 16, 32, 32] + 7 * [64]
    assert out == [f"{w}:{-(-c // w)}:{w}" for c, w in zip(channels, width)]


def test_few_edges_per_node_are_taken_one_at_a_time(tmp_path):
    """Up to two per node, three where the plan takes two at once; the workspace is the same."""
    out = run(tmp_path, PLAN + r"""
int main() {
  for (int channels : {8, 12, 16, 17, 32, 33}) {
    LunaUvuPlan* plan = plan_of(channels);
    int most = 0;
    while (most < 8 && plan->few(1000, 1000 * (most + 1))) ++most;
    const bool exact = !plan->sparse || !plan->few(1000, 1000 * most + 1);
    const bool same = !plan->sparse || (luna::uvu_bwd_workspace_bytes(*plan->sparse, 999) == luna::uvu_bwd_workspace_bytes(plan->plan, 999) &&
                                        plan->sparse->fwd_groups[0].cw == 64 && plan->sparse->bwd_groups[0].cw == 64);
    printf("%d:%d:%d:%d\n", channels, most, exact, same);
  }
}""")
    assert out == ["8:2:1:1", "12:2:1:1", "16:2:1:1", "17:3:1:1", "32:3:1:1", "33:0:1:1"]


def test_all_kernels_of_a_plan_compile_without_gpu(tmp_path, monkeypatch):
    """Ahead of the first call: a narrow layer on any graph (no envelope or scalar features) and by rows."""
    from lunaequivariance_amd.build import standard_operators

    monkeypatch.setenv("LUNAEQ_AMD_CACHE", str(tmp_path))
    op = standard_operators()[2]
    assert op.max_channels == 32
    op.plan.precompile(everything=True)
    names = sorted(p.name.split("_")[1] for p in tmp_path.glob("uvu_*.co"))
    assert names == ["bwd00111", "bwd00111", "fwd00", "fwd00", "fws00", "rwb0111", "rwb1111", "rwf0", "rwf1"]
