"""Reads of a tile through a buffer resource (TileReader in partition_device.h) rely on the hardware's comparison of a
read's offset with the length of the resource.  The scalar offset operand of the instruction is left out of that
comparison (the contract of the raw buffer loads), so a read that carries a part of its place there can pass the check
and lie past the end of the caller's array.  Compiled here for gfx950 and looked at in the assembly; needs no GPU."""
import os
import re
import subprocess

import pytest

from mcsparse_amd import build

PROBE = """
#include "partition_device.h"
using mcsp::partition_detail::TileReader;
// the two ways in which the partition kernels name their places: slabs of 64 per item, and a workgroup's width per item
template <typename W, int STRIDE, int FIRST>
__global__ void probe(const W* in, uint32_t count, W* out) {
    const TileReader reader(in, count * sizeof(W));
    W got[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) got[i] = reader.template read<W>(threadIdx.x, i * STRIDE + FIRST);
    W sum = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) sum = sum * 3 + got[i];
    out[threadIdx.x] = sum;
}
template __global__ void probe<%s, %d, %d>(const %s*, uint32_t, %s*);
"""


@pytest.mark.parametrize("word", ["uint32_t", "uint64_t"])
@pytest.mark.parametrize("stride,first", [(64, 0), (512, 1)])
def test_a_read_carries_its_whole_place_where_the_hardware_checks_it(tmp_path, word, stride, first):
    src = tmp_path / "probe.hip"
    src.write_text(PROBE % (word, stride, first, word, word))
    flags = [f for f in build.COMPILE_FLAGS if f not in ("-fPIC", "-Wall")]
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    out = tmp_path / "probe.txt"
    subprocess.run([hipcc] + flags + ["-w", "--cuda-device-only", "-S", "-I", build.INCLUDE, "-I", build.CSRC, str(src), "-o",
                                      str(out)], check=True, stderr=subprocess.DEVNULL)
    # buffer_load_dword[x2] data, place, s[resource], scalar offset [modifiers]
    loads = re.findall(r"buffer_load_dword\S*\s+\S+ (\S+), s\[\d+:\d+\], (\S+) ([^\n]*)", out.read_text())
    assert len(loads) == 16, loads
    for place, scalar, modifiers in loads:
        assert place.startswith("v") and "offen" in modifiers, (place, modifiers)
        assert scalar == "0", (place, scalar, modifiers)
