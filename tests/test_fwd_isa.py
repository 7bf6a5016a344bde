"""The plain and fused forward kernels keep everything in registers.

A forward workgroup is 1024 threads, so a lane has 128 VGPRs, 64 of them the
codebook; a value that does not fit is stored to and reloaded from scratch
memory in every trellis step.  This compiles both translation units of the
kernels for gfx950 (hipcc, no GPU needed) and reads the compiler's resource
remarks: no instance of fwd_kernel, tailbite_fused_kernel or fwd_defer_kernel
spills a register.  (The column chain's kernel, which carries the feedback's
state around the steps, does and is not held to this.)
"""
import os
import re
import shutil
import subprocess

import pytest

from conftest import PKG

SRC = os.path.join(PKG, "csrc", "viterbi_kernels.hip")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
# K=3's batched forward has a translation unit of its own (see the Makefile)
UNITS = {"main": [], "k3": ["-DXTQ_FWD_K3_TU", "-mllvm", "-amdgpu-sched-strategy=max-ilp"]}
GROUPS = {2: (1,), 3: (1, 2), 4: (1, 2, 4), 5: (1, 2, 4, 8), 6: (1, 2, 4, 8), 7: (1, 2, 4, 8)}


@pytest.fixture(scope="module")
def resources(tmp_path_factory):
    """(kernel, template arguments) -> (VGPRs spilled, scratch bytes per lane)"""
    if not os.path.exists(HIPCC) and not shutil.which("hipcc"):
        pytest.skip("hipcc not available")
    tmp = tmp_path_factory.mktemp("fwd_isa")
    procs = [subprocess.Popen(
        [HIPCC if os.path.exists(HIPCC) else "hipcc", "--offload-arch=gfx950", "-O3",
         "-std=c++17", "-ffp-contract=off", "-fvisibility=hidden",
         "-fno-gpu-flush-denormals-to-zero",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", *flags,
         "-Rpass-analysis=kernel-resource-usage", "--cuda-device-only", "-S", SRC,
         "-o", str(tmp / (name + ".s"))], stderr=subprocess.PIPE, text=True)
        for name, flags in UNITS.items()]
    found = {}
    for p in procs:
        text = p.communicate()[1]
        assert p.returncode == 0, text[-2000:]
        for block in text.split("Function Name: ")[1:]:
            m = re.match(r"\S*?\d+((?:fwd|tailbite|fwd_defer)_(?:fused_)?kernel)I((?:Li\d+E)+)E",
                         block)
            if m:
                args = tuple(int(v) for v in re.findall(r"Li(\d+)E", m.group(2)))
                spill = int(re.search(r"VGPRs Spill: (\d+)", block).group(1))
                scratch = int(re.search(r"ScratchSize \[bytes/lane\]: (\d+)", block).group(1))
                found[m.group(1), args] = (spill, scratch)
    return found


@pytest.mark.parametrize("K", range(2, 8))
def test_forward_kernels_do_not_spill(resources, K):
    want = [("fwd_kernel", (K, T)) for T in GROUPS[K]] + [("tailbite_fused_kernel", (K,))]
    if K >= 4:
        want += [("fwd_defer_kernel", (K, T)) for T in GROUPS[K]]
    for kernel in want:
        assert resources[kernel] == (0, 0), (kernel, resources[kernel])
