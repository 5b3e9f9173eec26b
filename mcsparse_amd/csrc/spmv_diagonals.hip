// SpMV from a copy along the diagonals for gfx950: y = alpha*A*x + beta*y.
//
// Neighbouring rows of a grid's matrix hold the same diagonals (column minus row).  Stored row by row every nonzero
// carries its column, a wavefront's lanes share a row (27 nonzeros on 32 lanes, rows that begin at any address) and add
// their products across lanes.  mcsparseSpMV_preprocess therefore tries a copy in slices of 64 lanes times 16 bytes of y:
// a diagonal that any row of the slice holds is its offset, a bit per row that holds it, and a value per row (zero where
// the row does not hold it: grid lines end, which costs a place in a hundred).  Values are then read 16 aligned bytes a
// lane, x 16 bytes a lane from wherever the diagonal lies, no sum crosses a lane, and a nonzero costs its value alone.
//
// Bounds: the values' stream, then the vector memory unit, which takes a load in the same time whatever its width (hence 16
// bytes a lane: with one row a lane 45 us in fp64).  27-point stencil 101 x 97 x 89 (23 M nonzeros), microseconds, row
// kernel and this: fp64 73.5 and 38.1 (203 MB, 5.3 TB/s), fp32 60.6 and 17.5; 150^3, fp64 (790 MB): 151.6 (5.2 TB/s); 128^3,
// fp32, copy in column order and this: 134 and 54; 5-point Laplacian 1900 x 1801, fp32: 49.6 and 18.
//
// Stands in, like spmv.hip, for the reference's row kernel (src/kernels/level2/spmv/csr_vector_device.hpp:22-79).
#include "diagonals_device.h"

namespace mcsp {

namespace {

using namespace diagonals_detail;

constexpr int kBlock = 256;
constexpr uint32_t kWaves = kBlock / kWave;
constexpr uint32_t kSampledSlices = 256;
// Values beyond half of the 256 MB behind the L2s are read past the caches: they are gone before the next product, and push
// x and y out.  Stencils, microseconds with plain and with streaming loads: fp64 101 x 97 x 89 (189 MB) 43.3 and 40.8, 33 x
// 149 x 150 (160 MB) 36.2 and 34.6, fp32 128^3 (226 MB) 56.1 and 54.0; fp32 101 x 97 x 89 (94 MB) 17.5 and 23.2.
constexpr uint64_t kKeptBytes = 128ull << 20;
// Diagonals of a slice up to which two wavefronts share it, with four loads of values in flight, and not four, with seven:
// 5-point Laplacian, 1900 x 1801, fp32: 18.0 and 40.7 us; the 27 diagonals of the fp64 stencil 41.9 and 38.1.
constexpr uint32_t kFewDiagonals = 12;
constexpr uint32_t kMostDiagonals = 512;  // of a slice; more: not a matrix for this copy

struct DiagonalTotals {
    unsigned long long diagonals, nonzeros;  // of the slices looked at
    uint32_t refused;                        // != 0: a row with unsorted or repeated columns, or too many diagonals
    uint32_t longest;                        // most nonzeros of a slice
};

// the smallest over the wavefront, in every lane
__device__ __forceinline__ int wave_min(int v) {
    constexpr int kRowShr = 0x110, kRowBcast15 = 0x142, kRowBcast31 = 0x143, kMost = 0x7fffffff;
    v = min(v, __builtin_amdgcn_update_dpp(kMost, v, kRowShr + 1, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(kMost, v, kRowShr + 2, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(kMost, v, kRowShr + 4, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(kMost, v, kRowShr + 8, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(kMost, v, kRowBcast15, 0xA, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(kMost, v, kRowBcast31, 0xC, 0xF, false));
    return __builtin_amdgcn_readlane(v, kWave - 1);
}

// A wavefront per slice merges its rows by offset.  The slice's columns (and values) are brought to LDS in one piece where
// they fit: walked where they lie, the rows of the slices in flight push each other's lines out of the caches (1000 us for
// both passes over 23 M nonzeros).  The diagonals are counted, into counts[slice] or, where that is null, added up (`stride`
// slices apart), or written, with or without their values.
enum SlicePass : int { kCount, kDescribe, kCopy };
template <typename T, int PASS>
__global__ __launch_bounds__(kWave) void slice_diagonals_kernel(idx_t m, idx_t base, uint32_t slices, uint32_t stride,
                                                                const idx_t* __restrict__ row_ptr,
                                                                const idx_t* __restrict__ col, const T* __restrict__ val,
                                                                uint32_t* counts, DiagonalTotals* totals,
                                                                SliceDiagonal<lane_rows<T>()>* __restrict__ diagonals,
                                                                T* __restrict__ vals_out) {
    constexpr int R = lane_rows<T>();
    constexpr uint32_t kRows = slice_rows<T>(), kStaged = kRows * 28;
    typedef T vec_t __attribute__((ext_vector_type(R)));
    __shared__ idx_t s_col[kStaged];
    __shared__ T s_val[PASS == kCopy ? kStaged : 1];
    const uint64_t slice = static_cast<uint64_t>(blockIdx.x) * stride;
    if (slice >= slices) return;  // whole workgroup
    const uint32_t lane = lane_id();
    const uint64_t row0 = slice * kRows;
    const uint32_t rows_here = m - row0 < kRows ? static_cast<uint32_t>(m - row0) : kRows;
    const idx_t first = row_ptr[row0] - base, nonzeros = row_ptr[row0 + rows_here] - base - first;
    const bool staged = nonzeros <= kStaged;  // the same for the wavefront
    if (staged) {
#pragma unroll 8
        for (uint32_t p = lane; p < nonzeros; p += kWave) {
            s_col[p] = col[first + p];
            if constexpr (PASS == kCopy) s_val[p] = val[first + p];
        }
        __syncthreads();
    }
    // half of the places filled, with some allowance for the slices where the diagonals change
    const uint32_t most = min(nonzeros / (kRows / 2) + 32, kMostDiagonals);
    constexpr int kNone = 0x7fffffff;
    idx_t at[R], end[R];  // inside the slice
    int offset[R];
    auto offset_at = [&](int j, idx_t p) {
        const uint32_t row = static_cast<uint32_t>(row0) + lane * R + j;
        return p < end[j] ? static_cast<int>((staged ? s_col[p] : col[first + p]) - base - row) : kNone;
    };
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const uint32_t r = lane * R + j;
        at[j] = r < rows_here ? row_ptr[row0 + r] - base - first : 0;
        end[j] = r < rows_here ? row_ptr[row0 + r + 1] - base - first : 0;
        offset[j] = offset_at(j, at[j]);
    }
    uint32_t found = 0;
    const uint64_t out = PASS != kCount ? counts[slice] : 0;
    bool refused = false;
    while (true) {
        int least = offset[0];
#pragma unroll
        for (int j = 1; j < R; ++j) least = min(least, offset[j]);
        least = wave_min(least);
        if (least == kNone) break;
        if (found == most) {
            refused = true;
            break;
        }
        vec_t v = vec_t(0);
        SliceDiagonal<R> d;
        d.offset = static_cast<uint32_t>(least);
        d.unused = 0;
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const bool mine = offset[j] == least;
            d.rows[j] = __ballot(mine);
            if (mine) {
                if constexpr (PASS == kCopy) v[j] = staged ? s_val[at[j]] : val[first + at[j]];
                offset[j] = offset_at(j, ++at[j]);
                refused |= offset[j] <= least;
            }
        }
        if constexpr (PASS == kCopy) reinterpret_cast<vec_t*>(vals_out)[(out + found) * kWave + lane] = v;
        if (PASS != kCount && lane == 0) diagonals[out + found] = d;
        ++found;
        if (__any(refused)) break;
    }
    if constexpr (PASS == kCount) {
        if (__any(refused)) {
            found = 0;
            if (lane == 0) totals->refused = 1;
        }
        if (lane == 0) {
            if (nonzeros > totals->longest) atomicMax(&totals->longest, nonzeros);  // (mostly not: no queue at the counter)
            if (counts != nullptr) {
                counts[slice] = found;
            } else {
                atomicAdd(&totals->diagonals, static_cast<unsigned long long>(found));
                atomicAdd(&totals->nonzeros, static_cast<unsigned long long>(nonzeros));
            }
        }
    }
}

__global__ void clear_totals_kernel(DiagonalTotals* totals, uint32_t* last_count) {
    *totals = DiagonalTotals{0, 0, 0, 0};
    *last_count = 0;  // the scan leaves the sum of all counts there
}

// WAVES wavefronts to a slice, each with a stretch of its diagonals, 4 / WAVES slices to a workgroup: a workgroup then reads
// one piece of the copy at a time, and small matrices have work for every compute unit.  What is read from the
// copy is clamped, so a copy the caller has overwritten gives wrong numbers but no access outside the arrays.
// Sums: fp32 products are added as doubles; fp64 ones into two sums a wavefront in turn, so that a row of 27 is chains of
// four and not one of 27.
template <typename T, bool BETA0, bool STREAM, int WAVES>
__global__ __launch_bounds__(kBlock) void spmv_diagonals_kernel(idx_t m, idx_t n, uint32_t slices, uint32_t total,
                                                                const uint32_t* __restrict__ diagonal_first,
                                                                const SliceDiagonal<lane_rows<T>()>* __restrict__ diagonals,
                                                                const T* __restrict__ vals, const T* __restrict__ x,
                                                                T* __restrict__ y, T alpha, T beta, uint32_t xcds) {
    constexpr int R = lane_rows<T>();
    constexpr int kAhead = WAVES == 2 ? 4 : 7;  // diagonals whose loads are in flight together
    constexpr int kSums = sizeof(T) == 8 ? 2 : 1;
    typedef T vec_t __attribute__((ext_vector_type(R)));
    typedef vec_t element_aligned __attribute__((aligned(sizeof(T))));  // a vector of x or y from any element on
    __shared__ double s_sum[kWaves][R][kWave];
    const uint32_t block = block_in_stretch(xcds);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t slice = block * (kWaves / WAVES) + wave / WAVES;
    const uint32_t lane = lane_id();
    const idx_t row0 = slice * slice_rows<T>(), row = row0 + lane * R;
    double sum[kSums][R] = {};
    if (slice < slices) {
        const uint32_t d1 = min(diagonal_first[slice + 1], total), d0 = min(diagonal_first[slice], d1);
        const uint32_t share = (d1 - d0 + WAVES - 1) / WAVES;
        const uint32_t from = min(d0 + wave % WAVES * share, d1), to = min(from + share, d1);
        for (uint32_t c = from; c < to; c += kWave) {
            SliceDiagonal<R> own = {};  // a lane keeps a diagonal (rows = 0: none)
            if (c + lane < to) own = diagonals[c + lane];
            const uint32_t here = min(to - c, static_cast<uint32_t>(kWave));
            // every vector of x lies inside it, also for rows that do not hold the diagonal?  (not so next to the ends of x)
            const int64_t x0 = static_cast<int64_t>(row0) + static_cast<int>(own.offset);
            const bool inside = __all(lane >= here || (x0 >= 0 && x0 + slice_rows<T>() <= n));
            auto run = [&](auto vectors_of_x) {
                for (uint32_t k0 = 0; k0 < here; k0 += kAhead) {
                    vec_t v[kAhead], xv[kAhead];
                    unsigned long long rows[kAhead][R];
#pragma unroll
                    for (int u = 0; u < kAhead; ++u) {
                        const uint32_t k = min(k0 + u, here - 1);
#pragma unroll
                        for (int j = 0; j < R; ++j) {
                            const uint32_t low = __builtin_amdgcn_readlane(static_cast<uint32_t>(own.rows[j]), k);
                            const uint32_t high = __builtin_amdgcn_readlane(static_cast<uint32_t>(own.rows[j] >> 32), k);
                            rows[u][j] = k0 + u < here ? static_cast<unsigned long long>(high) << 32 | low : 0;
                        }
                        const vec_t* from_copy = reinterpret_cast<const vec_t*>(vals) + static_cast<uint64_t>(c + k) * kWave + lane;
                        v[u] = STREAM ? load_stream(from_copy) : *from_copy;
                        const uint32_t column = row + static_cast<uint32_t>(__builtin_amdgcn_readlane(own.offset, k));
                        if constexpr (decltype(vectors_of_x)::value) {
                            xv[u] = *reinterpret_cast<const element_aligned*>(x + column);
                        } else {
#pragma unroll
                            for (int j = 0; j < R; ++j) xv[u][j] = x[min(column + j, n - 1)];
                        }
                    }
#pragma unroll
                    for (int u = 0; u < kAhead; ++u) {
#pragma unroll
                        for (int j = 0; j < R; ++j) {
                            // (a row without the diagonal must not touch its sum: 0 * x is NaN for an infinite x)
                            double& s = sum[u % kSums][j];
                            const double with = __builtin_fma(static_cast<double>(v[u][j]), static_cast<double>(xv[u][j]), s);
                            s = __builtin_amdgcn_inverse_ballot_w64(rows[u][j]) ? with : s;
                        }
                    }
                }
            };
            if (inside) run(std::true_type());
            else run(std::false_type());
        }
    }
    double all[R];
#pragma unroll
    for (int j = 0; j < R; ++j) all[j] = kSums == 2 ? sum[0][j] + sum[kSums - 1][j] : sum[0][j];
#pragma unroll
    for (int j = 0; j < R; ++j) s_sum[wave][j][lane] = all[j];
    __syncthreads();
    if (wave % WAVES != 0) return;  // whole wavefront
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
#pragma unroll
        for (int j = 0; j < R; ++j) all[j] += s_sum[wave + w][j][lane];
    }
    if (slice >= slices || row >= m) return;
    if (m - row >= R) {
        element_aligned* out = reinterpret_cast<element_aligned*>(y + row);
        vec_t s;
#pragma unroll
        for (int j = 0; j < R; ++j) s[j] = alpha * static_cast<T>(all[j]);
        if constexpr (!BETA0) {
            const vec_t old = *out;
#pragma unroll
            for (int j = 0; j < R; ++j) s[j] = beta * old[j] + alpha * static_cast<T>(all[j]);
        }
        *out = s;
    } else {
#pragma unroll
        for (int j = 0; j < R; ++j) {
            if (row + j < m) {
                const T s = static_cast<T>(all[j]);
                y[row + j] = BETA0 ? alpha * s : beta * y[row + j] + alpha * s;
            }
        }
    }
}

}  // namespace

SliceDiagonalsLayout slice_diagonals_layout(idx_t m, idx_t nnz, size_t value_bytes, bool with_values) {
    const uint32_t rows = slice_rows_of(value_bytes);
    const size_t diagonal = value_bytes == 4 ? sizeof(SliceDiagonal<4>) : sizeof(SliceDiagonal<2>);
    SliceDiagonalsLayout l;
    l.slices = static_cast<uint32_t>((static_cast<uint64_t>(m) + rows - 1) / rows);
    // two thirds of the places filled: with fewer, fp64 values alone are as long as values and columns in rows
    l.most = static_cast<uint32_t>(static_cast<uint64_t>(nnz) * 3 / (2 * rows));
    size_t off = 0;
    l.totals = off; off += align_up(sizeof(DiagonalTotals));
    l.diagonal_first = off; off += align_up((static_cast<size_t>(l.slices) + 1) * sizeof(uint32_t));
    l.diagonals = off; off += align_up(static_cast<size_t>(l.most) * diagonal);
    l.vals = off; off += with_values ? align_up(static_cast<size_t>(l.most) * rows * value_bytes) : 0;
    l.scan_ws = off; off += align_up(exclusive_scan_workspace_bytes(static_cast<uint64_t>(l.slices) + 1));
    l.total = off;
    return l;
}

bool slice_diagonals_shape(idx_t m, idx_t n, idx_t nnz) {
    return m != 0 && nnz >= kDiagonalsLeastNonzeros && m < (1u << 31) && n < (1u << 31);
}

namespace {

template <typename T>
bool build_typed(hipStream_t stream, idx_t m, idx_t nnz, idx_t base, const idx_t* row_ptr, const idx_t* col, const T* val,
                 void* region, uint32_t* total, uint32_t* longest) {
    const SliceDiagonalsLayout l = slice_diagonals_layout(m, nnz, sizeof(T), val != nullptr);
    char* w = static_cast<char*>(region);
    DiagonalTotals* totals = reinterpret_cast<DiagonalTotals*>(w + l.totals);
    uint32_t* counts = reinterpret_cast<uint32_t*>(w + l.diagonal_first);
    auto* diagonals = reinterpret_cast<SliceDiagonal<lane_rows<T>()>*>(w + l.diagonals);
    T* vals = reinterpret_cast<T*>(w + l.vals);
    auto read_back = [&](void* to, const void* from, size_t bytes) {
        return hipMemcpyAsync(to, from, bytes, hipMemcpyDeviceToHost, stream) == hipSuccess &&
               hipStreamSynchronize(stream) == hipSuccess;
    };
    auto run = [&](auto* kernel, uint32_t stride, uint32_t* per_slice) {
        hipLaunchKernelGGL(kernel, dim3((l.slices + stride - 1) / stride), dim3(kWave), 0, stream, m, base, l.slices, stride,
                           row_ptr, col, val, per_slice, totals, diagonals, vals);
    };
    hipLaunchKernelGGL(clear_totals_kernel, dim3(1), dim3(1), 0, stream, totals, counts + l.slices);
    // a sample first: most matrices are turned away here
    run(slice_diagonals_kernel<T, kCount>, l.slices / kSampledSlices + 1, nullptr);
    DiagonalTotals t;
    if (!read_back(&t, totals, sizeof(t))) return false;
    if (t.refused != 0 || t.diagonals * slice_rows<T>() * 2 > t.nonzeros * 3) return true;
    run(slice_diagonals_kernel<T, kCount>, 1, counts);
    launch_exclusive_scan_u32(stream, counts, static_cast<uint64_t>(l.slices) + 1, w + l.scan_ws);
    uint32_t found = 0;
    if (!read_back(&found, counts + l.slices, sizeof(found)) || !read_back(&t, totals, sizeof(t))) return false;
    if (t.refused != 0 || found > l.most) return true;
    if (val != nullptr) run(slice_diagonals_kernel<T, kCopy>, 1, counts);
    else run(slice_diagonals_kernel<T, kDescribe>, 1, counts);
    *total = found;
    if (longest != nullptr) *longest = t.longest;
    return true;
}

}  // namespace

bool build_slice_diagonals(hipStream_t stream, idx_t m, idx_t nnz, idx_t base, const idx_t* row_ptr, const idx_t* col,
                           const void* val, size_t value_bytes, void* region, uint32_t* total, uint32_t* longest) {
    *total = 0;
    return value_bytes == 4
               ? build_typed(stream, m, nnz, base, row_ptr, col, static_cast<const float*>(val), region, total, longest)
               : build_typed(stream, m, nnz, base, row_ptr, col, static_cast<const double*>(val), region, total, longest);
}

template <typename T>
bool launch_spmv_diagonals(hipStream_t stream, uint32_t total, const SpmvArgs& a, T alpha, T beta, void* region) {
    const SliceDiagonalsLayout l = slice_diagonals_layout(a.m, a.nnz, sizeof(T), true);
    char* w = static_cast<char*>(region);
    const uint32_t xcds = device_topology().xcds;
    auto launch = [&](auto waves, auto stream_values) {
        constexpr int kPerSlice = decltype(waves)::value;
        constexpr uint32_t kSlices = kWaves / kPerSlice;
        constexpr bool kStream = decltype(stream_values)::value;
        const uint32_t blocks = (l.slices + kSlices - 1) / kSlices;
        const dim3 grid((blocks + xcds - 1) / xcds * xcds);
        auto* kernel = beta == T(0) ? spmv_diagonals_kernel<T, true, kStream, kPerSlice>
                                    : spmv_diagonals_kernel<T, false, kStream, kPerSlice>;
        hipLaunchKernelGGL(kernel, grid, dim3(kBlock), 0, stream, a.m, a.n, l.slices, total,
                           reinterpret_cast<const uint32_t*>(w + l.diagonal_first),
                           reinterpret_cast<const SliceDiagonal<lane_rows<T>()>*>(w + l.diagonals),
                           reinterpret_cast<const T*>(w + l.vals), static_cast<const T*>(a.x), static_cast<T*>(a.y), alpha,
                           beta, xcds);
    };
    auto launch_waves = [&](auto stream_values) {
        if (total / l.slices <= kFewDiagonals) launch(std::integral_constant<int, 2>(), stream_values);
        else launch(std::integral_constant<int, 4>(), stream_values);
    };
    if (static_cast<uint64_t>(total) * slice_rows<T>() * sizeof(T) > kKeptBytes) launch_waves(std::true_type());
    else launch_waves(std::false_type());
    return launches_taken();
}

template bool launch_spmv_diagonals<float>(hipStream_t, uint32_t, const SpmvArgs&, float, float, void*);
template bool launch_spmv_diagonals<double>(hipStream_t, uint32_t, const SpmvArgs&, double, double, void*);

}  // namespace mcsp
