"""What load_vec and store_vec promise the compiler about an address: no more than an element's alignment, as flat copies, batch norm and
pooling run over rows that start anywhere.  Read from the code that they become (compiled here, nothing is run)."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "arraydiff_cuda_amd", "csrc")

SOURCE = """
#include "adh_common.h"
using namespace adh;
struct Wide { uint16_t v[8]; } __attribute__((aligned(16)));
template <typename V, typename T, bool STREAM> __device__ void copy(const T *from, T *to) { store_vec<STREAM>(to, load_vec<STREAM, V>(from)); }
__global__ void copy_f32(const float *from, float *to) { copy<float4, float, false>(from, to); }
__global__ void copy_f32_stream(const float *from, float *to) { copy<float4, float, true>(from, to); }
__global__ void copy_bf16(const uint16_t *from, uint16_t *to) { copy<Wide, uint16_t, false>(from, to); }
__global__ void copy_bf16_stream(const uint16_t *from, uint16_t *to) { copy<Wide, uint16_t, true>(from, to); }
"""


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    d = tmp_path_factory.mktemp("align")
    (d / "copies.hip").write_text(SOURCE)
    subprocess.check_call(["hipcc", "-O3", "-std=c++17", "--offload-arch=gfx950", "--offload-device-only", "-S", "-emit-llvm", "-Xclang", "-target-feature",
                           "-Xclang", "-packed-fp32-ops", "-I", CSRC, "-I", os.path.join(CSRC, "..", "..", "include"), "-o", str(d / "copies.ll"), str(d / "copies.hip")])
    return dict(re.findall(r"define [^@]*@_Z\d+(copy_\w+?)PK\w+\([^{]*\{(.*?)\n\}", (d / "copies.ll").read_text(), re.S))


@pytest.mark.parametrize("name,element", [("copy_f32", 4), ("copy_f32_stream", 4), ("copy_bf16", 2), ("copy_bf16_stream", 2)])
def test_vectors_at_element_alignment(kernels, name, element):
    accesses = [line for line in kernels[name].splitlines() if re.search(r"\b(load|store)\b.*ptr addrspace\(1\)", line)]
    assert len(accesses) == 2, accesses  # one of 16 bytes either way
    for line in accesses:
        assert re.search(r"<(4 x i32|8 x i16)>", line) and int(re.search(r"align (\d+)", line).group(1)) <= element, line
