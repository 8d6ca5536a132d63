"""The device lists of a batch's instances (each solver's list behind the list
of all): every list starts on an instance descriptor's alignment and ends
inside the allocation, whatever the numbers of instances. Compiled from the
header that the runtime and the kernels share; runs on the host."""
import os
import shutil
import subprocess

import pytest

from helpers import ROOT

PROGRAM = """
#include "step_kernels.hpp"
#include <cstdio>
using namespace athmi;
int main() {
  for (size_t n = 1; n <= 4099; n++) {
    const size_t all = inst_list_bytes(n);
    if (all < n * (sizeof(Inst) + NKINDS * sizeof(int))) return std::printf("small %zu\\n", n), 1;
    for (size_t roe : {size_t(0), size_t(1), n / 3, n / 2, n - 1, n}) {
      const size_t hlle = n - roe;
      // in the order they are packed: all, Roe's, HLLE's
      const size_t at_roe = all, at_hlle = all + inst_list_bytes(roe);
      if (at_roe % alignof(Inst) || at_hlle % alignof(Inst))
        return std::printf("misaligned: %zu instances, %zu Roe\\n", n, roe), 1;
      if (at_hlle + inst_list_bytes(hlle) > inst_lists_bytes(n))
        return std::printf("past the end: %zu instances, %zu Roe\\n", n, roe), 1;
    }
  }
  return 0;
}
"""


@pytest.mark.skipif(not shutil.which("g++") or not os.path.isdir("/opt/rocm/include"),
                    reason="needs g++ and the HIP headers")
def test_lists_are_aligned_and_fit(tmp_path):
    src, exe = tmp_path / "lists.cpp", tmp_path / "lists"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I",
                    os.path.join(ROOT, "athena-cuda_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
