"""The built kernels start without 16-bit vector loads: their launch shape is read by
scalar loads (a blockDim that the compiler cannot fold is a select between two
16-bit values in memory, a wait of every work-group before its first own load)."""
import os
import re
import subprocess

import pytest

from cps_veloc_amd import dwf

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
TOOLS = [os.path.join(LLVM, t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-objdump")]


@pytest.mark.skipif(not os.path.exists(dwf.LIB_PATH), reason="library not built")
@pytest.mark.skipif(not all(os.path.exists(t) for t in TOOLS), reason="no LLVM tools")
def test_launch_shape_is_scalar(tmp_path):
    copy, bundler, dump = TOOLS
    fat, obj = str(tmp_path / "fat"), str(tmp_path / "dev.o")
    subprocess.run([copy, "--dump-section", f".hip_fatbin={fat}", dwf.LIB_PATH, os.devnull],
                   check=True)
    subprocess.run([bundler, "--type=o", "--unbundle", f"--input={fat}", f"--output={obj}",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
    text = subprocess.run([dump, "-d", "--no-show-raw-insn", obj], check=True,
                          capture_output=True, text=True).stdout
    kernels = re.split(r"^[0-9a-f]+ <(\S+)>:$", text, flags=re.M)
    seen, bad = 0, []
    for name, body in zip(kernels[1::2], kernels[2::2]):
        if not re.search(r"k_(mobius|dwf|x_flush|pnext|xpby|ms_|m5inv|cg_)", name):
            continue
        seen += 1
        if any("global_load_ushort" in line for line in body.splitlines()[:60]):
            bad.append(name)
    assert seen > 100 and not bad
