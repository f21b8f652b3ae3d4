"""Workspace sizing of the graph tables, run on the host: the sizing pass takes what the launching one takes."""

import shutil
import subprocess
from pathlib import Path

import pytest

from lunaequivariance_amd import _native

ROOT = Path(__file__).resolve().parents[1]
CLANG = shutil.which("clang++") or "/opt/rocm/llvm/bin/clang++"
HIP_INCLUDE = Path("/opt/rocm/include")

pytestmark = pytest.mark.skipif(not (Path(CLANG).exists() and HIP_INCLUDE.exists()), reason="needs clang++ and HIP headers")

PROGRAM = r"""
#include <cstdio>
#include "%s/lunaequivariance_amd/csrc/graph.cpp"
// Peak scratch of one scan of n values, with and without memory behind it (nothing is launched).
size_t peak(char* base, size_t size, int64_t n) {
  luna::Arena arena{base, size};
  luna::Builder{nullptr, nullptr, arena}.scan(nullptr, n, nullptr, n);
  return arena.peak;
}
int main() {
  static char memory[1 << 20];
  // One tile, the most tiles whose sums every workgroup adds up, one more, and two levels of nested scans.
  for (int64_t n : {1LL, 2048LL, 64 * 2048LL, 64 * 2048LL + 1, 300 * 2048LL, 66000 * 2048LL})
    if (peak(nullptr, 0, n) != peak(memory, sizeof(memory), n)) { printf("%%lld values\n", (long long)n); return 1; }
  puts("ok");
}
"""


def test_nested_scans_are_counted(tmp_path):
    (tmp_path / "sizes.cpp").write_text(PROGRAM % ROOT)
    library = Path(_native.LIBRARY_PATH)
    subprocess.run([CLANG, "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", f"-I{HIP_INCLUDE}", str(tmp_path / "sizes.cpp"),
                    str(library), f"-Wl,-rpath,{library.parent}", "-Wl,--allow-shlib-undefined", "-o", str(tmp_path / "sizes")],
                   check=True)
    done = subprocess.run([str(tmp_path / "sizes")], capture_output=True, text=True)
    assert done.returncode == 0 and done.stdout.strip() == "ok", (done.returncode, done.stdout, done.stderr)
