"""No step kernel on CSR rows spills registers to scratch memory: it runs thousands of
times a call, and a spill comes back as traffic of every lane in every row (a batch step of
eight complex vectors took 3 to 4 times as long with 240 bytes a lane).  Read from the
code objects in the build's own object files."""
import os
import re
import subprocess

import pytest

from conftest import ROOT

LLVM = "/opt/rocm/llvm/bin"
OBJ = os.path.join(ROOT, "leo2d_amd", "_build")


@pytest.mark.parametrize("source", ["kpm.hip", "batch.hip", "cond.hip"])
def test_csr_step_kernels_use_no_scratch(tmp_path, source):
    obj = os.path.join(OBJ, source + ".o")
    tools = [os.path.join(LLVM, t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-readelf")]
    if not os.path.exists(obj) or not all(map(os.path.exists, tools)):
        pytest.skip("object files of a build and the LLVM tools are needed")
    bundle, code = str(tmp_path / "bundle"), str(tmp_path / "code")
    subprocess.run([tools[0], "--dump-section", ".hip_fatbin=" + bundle, obj, os.devnull], check=True)
    subprocess.run([tools[1], "--unbundle", "--type=o", "--input=" + bundle, "--output=" + code,
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
    notes = subprocess.run([tools[2], "--notes", code], check=True, capture_output=True, text=True).stdout
    kernels = re.findall(r"\.name: +(\S*kernel\S*)\n.*?\.private_segment_fixed_size: (\d+)\n.*?\.vgpr_spill_count: (\d+)",
                         notes, re.S)
    steps = {name: (int(scratch), int(spills)) for name, scratch, spills in kernels if "_step_" in name}
    assert steps
    assert all(v == (0, 0) for v in steps.values()), {k: v for k, v in steps.items() if v != (0, 0)}
