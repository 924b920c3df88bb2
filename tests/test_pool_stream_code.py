"""The backward of 3x3 / 2 max pooling stores its gradient non-temporally where it is asked to: read from the code that it becomes (a
choice between the two stores at run time, though of a constant, was folded into the temporal one: 240 -> 263 us over 537 MB)."""
import os
import re
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "arraydiff_cuda_amd", "csrc")


def test_streaming_stores(tmp_path):
    out = tmp_path / "pool.s"
    subprocess.check_call(["hipcc", "-O3", "-std=c++17", "--offload-arch=gfx950", "--offload-device-only", "-S", "-Xclang", "-target-feature", "-Xclang",
                           "-packed-fp32-ops", "-I", CSRC, "-I", os.path.join(CSRC, "..", "..", "include"), "-o", str(out), os.path.join(CSRC, "pool.hip")])
    kernels = dict(re.findall(r"^_ZN3adh22pool_bwd_max3s2_kernel(\w+?)EEvNS_12PoolS2ParamsE:(.*?)s_endpgm", out.read_text(), re.S | re.M))
    found = 0
    for name, code in kernels.items():  # (type, [columns,] ragged rows, streaming)
        stores = re.findall(r"global_store_dwordx4 [^\n]*", code)
        if name.endswith("Lb0ELb1E") and stores:
            found += 1
            assert all(line.rstrip().endswith("nt") for line in stores), (name, stores)
        elif name.endswith("Lb0E"):
            assert not any(line.rstrip().endswith("nt") for line in stores), (name, stores)
    assert found == 2  # fp32 and bf16
