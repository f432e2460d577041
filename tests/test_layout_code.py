"""What the compiler makes of the weight layout conversion: its pieces stay in registers, its loads are in flight together."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs the ROCm toolchain")
def test_the_code_layout_kernel_waits_for_its_loads_together(tmp_path):
    out = tmp_path / "plk_mok.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-S",
                    f"-I{ROOT}/include", f"{ROOT}/pipelink_amd/csrc/plk_mok.cpp", "-o", str(out)], check=True, capture_output=True)
    body = re.search(r"^_Z\d+codes_to_k64_tiled_kernel\w*:.*?s_endpgm", out.read_text(), re.M | re.S).group(0)
    assert "ds_write" not in body and "ds_read" not in body
    loads = [m.start() for m in re.finditer(r"global_load_dwordx4", body)]
    assert len(loads) == 2 and "vmcnt" not in body[loads[0]:loads[1]]
