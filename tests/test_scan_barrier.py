"""The order of a level's scan (scan_counts, csrc/pga_level.h), in the device
code's LLVM IR, on the CPU. The block totals cross a grid barrier without
fences, so each thread's store of its totals has to be complete before its
block arrives. That takes a wait that the compiler cannot move the store past:
an instruction that touches memory, not a hardware wait the optimiser takes
for unrelated to memory."""
import os
import re
import subprocess

from operatorgraph_amd import build as B

KERNEL = """
#include "pga_level.h"
extern "C" __global__ void scan_only(pga::KArgs a) {
    __shared__ pga::LevelLDS L;
    pga::scan_counts(a, L, 1u, 1u);
}
"""


def test_block_totals_are_waited_for(tmp_path):
    src, out = str(tmp_path / "scan.hip"), str(tmp_path / "scan.ll")
    with open(src, "w") as f:
        f.write(KERNEL)
    flags = [f for f in B.COMMON_FLAGS if f != "-fPIC"]
    subprocess.run([B.HIPCC, f"--offload-arch={B.ARCH}", *flags, "-I", B.CSRC, "-I", os.path.join(B.ROOT, "include"),
                    "--offload-device-only", "-emit-llvm", "-S", src, "-o", out], check=True, capture_output=True)
    text = open(out).read()
    body = re.search(r"define [^\n]*@scan_only\(.*?\n}\n", text, re.S).group(0).splitlines()
    assert any("store atomic i32" in l and 'syncscope("agent")' in l for l in body), "the totals' store was not found"
    # the function's first barrier is where the block's waves meet before its
    # arrival; blocks of code do not stand in order, so look at its own
    first = next(i for i, l in enumerate(body) if "@llvm.amdgcn.s.barrier()" in l)
    before = []
    while first > 0 and not re.match(r"\d+:|$", body[first - 1]):
        first -= 1
        before.append(body[first])
    assert any("asm sideeffect" in l and "vmcnt(0)" in l and "~{memory}" in l for l in before), \
        "no wait with a memory clobber before the block arrives"
