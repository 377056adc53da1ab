"""What the compiler makes of kernels whose speed hangs on it (gfx950 assembly; no GPU needed)."""
import os
import re
import subprocess

from forja_amd import build


def test_row_tile_kernels_read_memory_by_global_loads_only(tmp_path):
    """A load through a pointer that may point to LDS (flat_load) counts as an access to memory and to LDS: the waits
    of the loop's LDS reads then wait for it, and for every load requested before it."""
    source, assembly = os.path.join(build.CSRC, "qmm_rows.hip"), str(tmp_path / "qmm_rows.s")
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    subprocess.run([hipcc, "-x", "hip", "-S", "--cuda-device-only", source, "-o", assembly] + build.COMMON, check=True,
                   capture_output=True)
    text = open(assembly).read()
    kernels = re.findall(r"^(_Z\w*qmm_rows_kernel\w+):(.*?)^\.Lfunc_end", text, re.M | re.S)
    assert len(kernels) == 10
    for name, body in kernels:
        assert "global_load" in body and "flat_" not in body, name
