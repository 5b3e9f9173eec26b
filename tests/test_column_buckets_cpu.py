"""The buckets of columns of the transposing SpMV without preprocess (csrc/internal.h): the bucket that a product's high word
names is column / width, at both ends of every bucket, for every width a bucket can have.  Needs no GPU."""
import subprocess

from mcsparse_amd import build

PROGRAM = r"""
#include <algorithm>
#include <cstdio>
#include "internal.h"
using namespace mcsp;
int main() {
    for (const uint32_t bits : {kBucketFewBits, kBucketManyBits}) {
        const uint32_t least = std::max<uint32_t>((kBucketMinColumns - 1 >> bits) + 1, 3);
        for (uint32_t width = least; width <= kBucketMaxColumns; ++width) {
            // the most and the fewest columns that have buckets of this width
            for (const uint32_t n : {width << bits, std::max<uint32_t>((width - 1 << bits) + 1, kBucketMinColumns)}) {
                const ColumnBuckets b = column_buckets(n, bits);
                if (b.width != width || b.bits != bits) return std::printf("%u columns: buckets of %u\n", n, b.width), 1;
                for (uint32_t k = 0; k < 1u << bits && k * width < n; ++k) {
                    const uint32_t first = k * width, last = std::min(first + width, n) - 1;
                    if (bucket_of(b, first) != k || bucket_of(b, last) != k)
                        return std::printf("%u columns of %u: bucket %u is %u to %u\n", n, width, k, bucket_of(b, first), bucket_of(b, last)), 1;
                }
            }
        }
    }
    return std::puts("ok"), 0;
}
"""


def test_bucket_of_a_column(tmp_path):
    source, program = tmp_path / "column_buckets.cpp", tmp_path / "column_buckets"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I", build.INCLUDE, "-I", build.CSRC,
                    str(source), "-o", str(program)], check=True)
    assert subprocess.run([str(program)], stdout=subprocess.PIPE, text=True).stdout == "ok\n"
