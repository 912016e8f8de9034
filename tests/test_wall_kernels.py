"""CPU check of what the compiler makes of the pure wall functions: no private array in
LDS and no read of the dispatch packet (the two go together: the place of such an array
depends on the size of the workgroup, which every wave then fetches from host memory)."""

import os
import re
import subprocess

from vivsim_amd import _build


def test_wall_kernels_hold_no_private_array(tmp_path):
    out = tmp_path / "ops.s"
    subprocess.run([_build.HIPCC, *_build.FLAGS, "--offload-device-only", "-S", os.path.join(_build.CSRC, "ops.hip"),
                    "-o", str(out)], check=True, capture_output=True)
    kernels = re.findall(r"\.amdhsa_kernel (\S+)\n(.*?)\.end_amdhsa_kernel", out.read_text(), re.S)
    wall = {k: v for k, v in kernels if re.search(r"\d(k_wall|k_wall_copy|k_cbc)I", k)}
    assert len(wall) == 6
    for name, v in wall.items():
        assert re.search(r"\.amdhsa_group_segment_fixed_size (\d+)", v).group(1) == "0", name
        assert re.search(r"\.amdhsa_user_sgpr_dispatch_ptr (\d+)", v).group(1) == "0", name
