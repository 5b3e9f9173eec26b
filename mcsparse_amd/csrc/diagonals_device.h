// Rows that share diagonals, in slices of neighbouring rows: spmv_diagonals.hip (which finds them), spmm_diagonals.hip.
#ifndef MCSPARSE_AMD_DIAGONALS_DEVICE_H_
#define MCSPARSE_AMD_DIAGONALS_DEVICE_H_

#include "device_util.h"
#include "internal.h"

namespace mcsp {
namespace diagonals_detail {

template <typename T>
constexpr int lane_rows() { return 16 / static_cast<int>(sizeof(T)); }  // neighbouring rows of a lane
template <typename T>
constexpr uint32_t slice_rows() { return kWave * lane_rows<T>(); }
inline uint32_t slice_rows_of(size_t value_bytes) { return value_bytes == 4 ? slice_rows<float>() : slice_rows<double>(); }

// A diagonal of a slice: row r0 + R * lane + j holds column row + offset (mod 2^32) where bit `lane` of rows[j] is set.
template <int R>
struct SliceDiagonal {
    uint32_t offset, unused;
    unsigned long long rows[R];
};

// The slice of a workgroup, `of` of them to a grid padded to whole turns of the XCDs: neighbouring slices read the same
// operand, so an XCD takes a stretch of them.
__device__ __forceinline__ uint32_t block_in_stretch(uint32_t xcds) {
    return (blockIdx.x % xcds) * (gridDim.x / xcds) + blockIdx.x / xcds;
}

}  // namespace diagonals_detail
}  // namespace mcsp

#endif  // MCSPARSE_AMD_DIAGONALS_DEVICE_H_
