"""Build-time check of the single-token kernel of the recurrent layers: its threads keep a state's rows in registers, and no instance
in the built library has more than a few scalars in scratch (a row of four values is 16 bytes a lane)."""
import os
import re
import shutil
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin"


@pytest.mark.skipif(not os.path.exists(os.path.join(LLVM, "llvm-readelf")), reason="no LLVM tools")
def test_no_step_kernel_keeps_rows_of_a_state_in_scratch(tmp_path):
    from fandhe_ai_amd import capi
    lib = shutil.copy(capi.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", lib], check=True, capture_output=True, cwd=tmp_path)
    scratch = {}
    for f in tmp_path.iterdir():
        if "gfx950" not in f.name:
            continue
        notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", str(f)], check=True, capture_output=True, text=True).stdout
        for kernel in re.split(r"^ +- \.agpr_count", notes, flags=re.M)[1:]:
            name = re.search(r"^ +\.name: +(\S+)", kernel, flags=re.M).group(1)
            if "delta_step_kernel" in name:
                scratch[name] = int(re.search(r"\.private_segment_fixed_size: +(\d+)", kernel).group(1))
    assert len(scratch) >= 12
    assert max(scratch.values()) <= 64, sorted(scratch.items(), key=lambda x: -x[1])[:3]
