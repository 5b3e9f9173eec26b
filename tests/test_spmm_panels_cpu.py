"""Which products without a schedule take rows of op(B) in panels of 512 bytes (csrc/internal.h): the matrices and widths that were
measured, on the side of the rule where they were faster.  Needs no GPU."""
import subprocess

import pytest

from mcsparse_amd import build

# row bytes, rows, nonzeros, longest row, neighbouring rows known to share columns, rows of op(B) of whole lines, panels; fp64 vectors
STENCIL, EVEN = (1000000, 26463592, 27), (100000, 1600000, 16)
CASES = [
    # 27-point stencil: whole panels, what is left of one where the columns are known to be shared
    (1024, *STENCIL, 0, 1, 1), (1024, *STENCIL, 0, 0, 0), (1024, *STENCIL, 1, 0, 1), (528, *STENCIL, 1, 0, 1), (768, *STENCIL, 1, 0, 1),
    (772, *STENCIL, 1, 0, 0), (528, *STENCIL, 0, 0, 0), (1560, *STENCIL, 1, 0, 1), (1560, *STENCIL, 0, 0, 0),
    # rows of 16 evenly spread columns: 129, 130, 160, 192 and 390 fp32 columns lost
    (516, *EVEN, 0, 0, 0), (520, *EVEN, 0, 0, 0), (640, *EVEN, 0, 1, 0), (768, *EVEN, 0, 1, 0), (1560, *EVEN, 0, 0, 0), (1024, *EVEN, 0, 1, 1),
    (1024, *EVEN, 0, 0, 0), (1536, *EVEN, 0, 1, 1), (1280, *EVEN, 0, 1, 1), (1280, *EVEN, 0, 0, 0), (1040, *EVEN, 0, 0, 1), (1792, *EVEN, 0, 1, 1),
    # short rows
    (520, 100000, 200000, 2, 0, 0, 1), (768, 100000, 400000, 4, 0, 1, 1), (776, 100000, 200000, 2, 0, 0, 1), (776, 100000, 400000, 4, 0, 0, 0), (768, 100000, 600000, 6, 0, 1, 0),
    (1024, 100000, 200000, 2, 0, 0, 1), (1024, 100000, 600000, 6, 0, 0, 0), (520, 5000, 10000, 2, 0, 0, 0),
    (640, 1000000, 8000000, 8, 0, 1, 1), (520, 1000000, 11000000, 11, 0, 0, 0), (1024, 1000000, 6000000, 6, 0, 0, 1),
    # rows of very different length
    (516, 100000, 824063, 1000, 0, 0, 0), (1024, 20000, 164801, 1000, 0, 1, 0), (1024, 100000, 824063, 1000, 0, 1, 0),
    (1024, 300000, 2472205, 1000, 0, 1, 0), (1024, 1000000, 8240658, 1000, 0, 1, 1), (1024, 100000, 472263, 128, 0, 1, 0),
    (1024, 300000, 1416799, 128, 0, 1, 1), (640, 100000, 384590, 64, 0, 1, 1), (640, 20000, 76915, 64, 0, 1, 0),
    # few rows
    (1024, 729, 15625, 27, 0, 1, 0), (528, 4913, 117649, 27, 1, 0, 0), (1024, 4913, 117649, 27, 0, 1, 1), (528, 20000, 500926, 27, 1, 0, 1),
    # more than half a panel left
    (800, 20000, 500926, 27, 1, 0, 0), (800, 128000, 3300000, 27, 1, 0, 1), (800, 198000, 5100000, 27, 0, 0, 0),
    # one panel; a length that is not known, no nonzeros
    (512, *STENCIL, 1, 1, 0), (1024, 1000000, 26463592, 0, 1, 1, 0), (1024, 1000, 0, 0, 1, 1, 0),
]


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    folder = tmp_path_factory.mktemp("panels")
    source, program = folder / "panels.cpp", folder / "panels"
    source.write_text('#include <cstdio>\n#include <cstdlib>\n#include "internal.h"\nint main(int, char** v) { return std::printf("%d\\n", '
                      "mcsp::spmm_takes_panels(atoll(v[1]), atoll(v[2]), atoll(v[3]), atoll(v[4]), atoi(v[5]), atoi(v[6]), atoi(v[7]))), 0; }\n")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I", build.INCLUDE, "-I", build.CSRC,
                    str(source), "-o", str(program)], check=True)
    return lambda *args: subprocess.run([str(program)] + [str(int(a)) for a in args], stdout=subprocess.PIPE, text=True).stdout == "1\n"


@pytest.mark.parametrize("case", CASES)
def test_rule(rule, case):
    assert rule(*case[:-1], 0) == bool(case[-1])


def test_rule_for_vectors_of_doubles(rule):
    # a million rows of a stencil, 100 columns: fp64, and fp32 or rows that begin at any element
    assert rule(800, *STENCIL, 1, 0, 1) and not rule(800, *STENCIL, 1, 0, 0) and not rule(800, *STENCIL, 0, 0, 1)
