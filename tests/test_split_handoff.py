"""The split-k products' hand-off in the built library: the waves of a CTA add their partial sums with atomics that
nothing waits for, so each must wait for its own (vmcnt 0) before the barrier in front of the CTA's arrival on the
tile's counter. Read from the gfx950 code of this build: no run can be relied on to show a missing wait."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def split_kernels(tmp_path):
    """Each kernel with 64-bit atomic adds in memory: its instructions."""
    lib = shutil.copy(os.path.join(ROOT, "tritify_amd", "libkt_hip.so"), tmp_path)  # the bundles land beside it
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, stdout=subprocess.DEVNULL)
    kernels = {}
    for f in sorted(tmp_path.glob("*gfx950")):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(f)], check=True, capture_output=True, text=True).stdout
        name = None
        for line in text.splitlines():
            head = re.match(r"^[0-9a-f]+ <(.*)>:$", line)
            if head:
                name = head.group(1)
            elif name and line.strip():
                kernels.setdefault(name, []).append(line.split("//")[0].strip())
    return {n: c for n, c in kernels.items() if any(i.startswith("global_atomic_add_x2 ") for i in c)}


def test_partial_sums_are_waited_for_before_the_arrival(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    kernels = split_kernels(tmp_path)
    assert sum("plane_gemm_kernel" in n for n in kernels) >= 9 and sum("plane_dma_kernel" in n for n in kernels) == 3
    for name, code in kernels.items():
        # the arrival: the one 32-bit add whose old value is used
        arrive = [i for i, c in enumerate(code) if re.match(r"global_atomic_add v\d+, .*\bsc0\b", c)]
        assert len(arrive) == 1, name
        at = max(i for i in range(arrive[0]) if code[i].startswith("s_barrier"))
        before = []  # back from the barrier to the wait: no memory instruction in between
        while not re.match(r"s_waitcnt .*vmcnt\(0\)", code[at - 1 - len(before)]):
            before.append(code[at - 1 - len(before)])
            assert not re.match(r"(global|flat|buffer)_", before[-1]), f"{name}: {before[-1]} is not waited for"
            assert len(before) < 16, f"{name}: no wait before the arrival's barrier"
