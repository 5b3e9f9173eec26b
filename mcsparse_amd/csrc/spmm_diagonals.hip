// CSR SpMM with op(B) and C in column-major order, for matrices whose neighbouring rows hold the same diagonals, on gfx950.
//
// Rows of op(B) are what the other SpMM kernels load, so a column-major op(B) is transposed for them first, and a
// column-major C is written in pieces (or transposed out).  A slice of rows that share diagonals reads a column of op(B) as a
// product with one vector does: 64 lanes times 16 bytes of neighbouring elements, from wherever the diagonal lies.  So nothing
// is transposed here: a workgroup takes a slice (spmv_diagonals.hip: mcsparseSpMM_preprocess finds the slices' diagonals), its
// values go to LDS, and every wavefront walks the diagonals for four columns of op(B), with the sums of its lanes' rows in
// registers, which are written as they lie.
//
// Bounds: the first cache of a compute unit, which serves 64 bytes of one line a cycle (a vector that begins at any element
// costs half as much again): three neighbouring diagonals therefore share one load (fp64 27-point stencil, 101 x 97 x 89, 16
// columns: 157 us with a load for each, 106 so; the transposes and the row kernel took 224).  A, op(B) and C
// are 408 MB, 85 us at the rate of a copy.  Other widths, microseconds with transposes and so: fp64 5, 8 and 37 columns 178,
// 186, 1004 and 67, 76, 293; fp32 9, 16, 64 and 128 columns 126, 158, 644, 1157 and 54, 65, 223, 477.  Columns a power of two apart fall on
// the same sets of the caches, which costs what the transposes do elsewhere: 128^3 (8 MB), fp32, 64 and 128 columns 676 with
// transposes and blocks and 684 so, 1353 and 1355; with 32 and 100 columns 374 and 347, 1480 and 1102; fp64, 64, 2495 and 1412.
//
// The reference copies the operands into the other order (src/kernels/level3/spmm/mcsp_spmm_gpu.cpp:119-133).
#include "diagonals_device.h"

namespace mcsp {

namespace {

using namespace diagonals_detail;

constexpr int kColumns = 4;      // of a wavefront, or half of them
constexpr uint32_t kPanelWaves = 4;  // as many columns as a slice is read for at a time, by the wavefronts of a workgroup
constexpr size_t kTwoLanes = 32;  // bytes of a row of op(B) up to which the kernels without a schedule are of another kind

// v of the next lane; the last lane gets `last`.
constexpr int kWaveShiftLeft = 0x130;
__device__ __forceinline__ float next_lane(float v, float last) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(last), __float_as_int(v), kWaveShiftLeft, 0xF, 0xF, false));
}
__device__ __forceinline__ double next_lane(double v, double last) {
    const long long bits = __double_as_longlong(v), of_last = __double_as_longlong(last);
    const int low = __builtin_amdgcn_update_dpp(static_cast<int>(of_last), static_cast<int>(bits), kWaveShiftLeft, 0xF, 0xF, false);
    const int high = __builtin_amdgcn_update_dpp(static_cast<int>(of_last >> 32), static_cast<int>(bits >> 32), kWaveShiftLeft, 0xF, 0xF, false);
    return __longlong_as_double(static_cast<long long>(high) << 32 | static_cast<unsigned int>(low));
}

template <typename T>
constexpr uint32_t staged_values() { return slice_rows<T>() * 28; }

// Sums are formed in the order of the diagonals, one multiply-add after the other, as the row kernels form them on the
// transposed operands: the same bits.
template <typename T, int COLUMNS, bool BETA0>
__global__ __launch_bounds__(kPanelWaves * kWave, 4) void spmm_diagonals_kernel(
    idx_t m, idx_t n, idx_t k, idx_t nnz, idx_t base, uint32_t slices, uint32_t total,
    const uint32_t* __restrict__ diagonal_first, const SliceDiagonal<lane_rows<T>()>* __restrict__ diagonals,
    const idx_t* __restrict__ row_ptr, const T* __restrict__ val, const T* __restrict__ B, int64_t ldb, T* __restrict__ C,
    int64_t ldc, T alpha, T beta, uint32_t xcds) {
    constexpr int R = lane_rows<T>();
    constexpr int kAhead = 2;  // runs of diagonals whose elements of op(B) are on their way
    constexpr int kRun = 3;
    static_assert(kRun - 1 <= R, "a run reaches into the next lane's elements and no further");
    constexpr uint32_t kRows = slice_rows<T>(), kStaged = staged_values<T>();
    typedef T vec_t __attribute__((ext_vector_type(R)));
    typedef vec_t element_aligned __attribute__((aligned(sizeof(T))));
    __shared__ __align__(16) T s_val[kStaged];
    const uint32_t slice = block_in_stretch(xcds);
    if (slice >= slices) return;  // whole workgroup
    const uint32_t lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const idx_t row0 = slice * kRows, row = row0 + lane * R;
    const uint32_t rows_here = min(m - row0, kRows);
    const idx_t first = row_ptr[row0] - base;
    const uint32_t count = min(min(row_ptr[row0 + rows_here] - base, nnz) - first, kStaged);
    uint32_t at[R];  // where the next unused value of each of the lane's rows lies
#pragma unroll
    for (int j = 0; j < R; ++j) at[j] = row_ptr[min(row + j, m)] - base - first;
    const uint32_t d1 = min(diagonal_first[slice + 1], total), d0 = min(diagonal_first[slice], d1);
    {
        constexpr int kBatch = 7;  // all of a slice in one trip, for four wavefronts
        const uint32_t vectors = count / R;
        for (uint32_t p0 = threadIdx.x; p0 < vectors; p0 += blockDim.x * kBatch) {
            vec_t got[kBatch];
#pragma unroll
            for (int i = 0; i < kBatch; ++i)
                got[i] = __builtin_nontemporal_load(reinterpret_cast<const element_aligned*>(val + first) + min(p0 + i * blockDim.x, vectors - 1));
#pragma unroll
            for (int i = 0; i < kBatch; ++i)
                if (p0 + i * blockDim.x < vectors) reinterpret_cast<vec_t*>(s_val)[p0 + i * blockDim.x] = got[i];
        }
        const uint32_t p = vectors * R + threadIdx.x;
        if (p < count) s_val[p] = val[first + p];
    }
    __syncthreads();
    const uint32_t column0 = (blockIdx.y * (blockDim.x / kWave) + wave) * COLUMNS;
    if (column0 >= n) return;  // whole wavefront
    const char* b[COLUMNS];
#pragma unroll
    for (int c = 0; c < COLUMNS; ++c)
        b[c] = reinterpret_cast<const char*>(B + static_cast<int64_t>(min(column0 + c, n - 1)) * ldb);
    T sum[COLUMNS][R] = {};
    for (uint32_t c0 = d0; c0 < d1; c0 += kWave) {
        SliceDiagonal<R> own = {};  // a lane keeps a diagonal (rows = 0: none)
        if (c0 + lane < d1) own = diagonals[c0 + lane];
        const uint32_t here = min(d1 - c0, static_cast<uint32_t>(kWave));
        // Up to kRun neighbouring diagonals are one run: a lane's elements of op(B) for the later ones are its own, moved on,
        // and the next lane's.
        const uint32_t before = __shfl_up(own.offset, 1, kWave);
        const unsigned long long breaks = __ballot(lane == 0 || own.offset != before + 1);
        const uint32_t in_row = __clzll(static_cast<long long>(breaks << (kWave - 1 - lane)));  // diagonals since the last break
        unsigned long long left = __ballot(lane < here && in_row % kRun == 0);
        struct Run {
            uint32_t first, width;
        };
        auto next_run = [&]() {  // width 0: none left
            Run r = {here - 1, 0};
            if (left != 0) {
                r.first = __builtin_ctzll(left);
                left &= left - 1;
                r.width = (left != 0 ? static_cast<uint32_t>(__builtin_ctzll(left)) : here) - r.first;
            }
            return r;
        };
        // every vector of op(B) lies inside it, also for rows that do not hold the diagonal?
        const int64_t x0 = static_cast<int64_t>(row0) + static_cast<int>(own.offset);
        const bool inside = __all(lane >= here || (x0 >= 0 && x0 + kRows + R <= k));
        auto walk = [&](auto vectors_of_b) {
            constexpr bool kVectors = decltype(vectors_of_b)::value;
            struct Elements {
                vec_t own[COLUMNS], more[COLUMNS];  // more: what follows the last lane's (kVectors), or this lane's
            };
            Elements x[kAhead];
            Run runs[kAhead];
            auto ask = [&](Elements& e, const Run& run) {
                const uint32_t offset = __builtin_amdgcn_readlane(own.offset, run.first);
#pragma unroll
                for (int c = 0; c < COLUMNS; ++c) {
                    if constexpr (kVectors) {
                        e.own[c] = *reinterpret_cast<const element_aligned*>(b[c] + (row + offset) * static_cast<uint32_t>(sizeof(T)));
                        e.more[c] = *reinterpret_cast<const element_aligned*>(b[c] + (row0 + kRows + offset) * static_cast<uint32_t>(sizeof(T)));
                    } else {
#pragma unroll
                        for (int j = 0; j < R; ++j) {
                            e.own[c][j] = *reinterpret_cast<const T*>(b[c] + min(row + offset + j, k - 1) * static_cast<uint32_t>(sizeof(T)));
                            e.more[c][j] = *reinterpret_cast<const T*>(b[c] + min(row + offset + R + j, k - 1) * static_cast<uint32_t>(sizeof(T)));
                        }
                    }
                }
            };
            auto add = [&](const Elements& e, const Run& run) {
                T after[COLUMNS][kRun - 1];
#pragma unroll
                for (int c = 0; c < COLUMNS; ++c) {
#pragma unroll
                    for (int i = 0; i < kRun - 1; ++i)
                        after[c][i] = kVectors ? next_lane(e.own[c][i], e.more[c][i]) : e.more[c][i];
                }
#pragma unroll
                for (int p = 0; p < kRun; ++p) {
                    if (p >= static_cast<int>(run.width)) break;  // whole wavefront
                    T v[R];
                    unsigned long long rows[R];
#pragma unroll
                    for (int j = 0; j < R; ++j) {
                        const uint32_t low = __builtin_amdgcn_readlane(static_cast<uint32_t>(own.rows[j]), run.first + p);
                        const uint32_t high = __builtin_amdgcn_readlane(static_cast<uint32_t>(own.rows[j] >> 32), run.first + p);
                        rows[j] = static_cast<unsigned long long>(high) << 32 | low;
                        v[j] = s_val[min(at[j], kStaged - 1)];
                        at[j] += __builtin_amdgcn_inverse_ballot_w64(rows[j]) ? 1u : 0u;
                    }
#pragma unroll
                    for (int j = 0; j < R; ++j) {
                        // (a row without the diagonal must not touch its sums: 0 * x is NaN for an infinite x)
                        if (__builtin_amdgcn_inverse_ballot_w64(rows[j])) {
#pragma unroll
                            for (int c = 0; c < COLUMNS; ++c)
                                sum[c][j] += v[j] * (j + p < R ? e.own[c][(j + p) % R] : after[c][(j + p) % R]);
                        }
                    }
                }
            };
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                runs[u] = next_run();
                ask(x[u], runs[u]);
            }
            while (runs[0].width != 0) {
#pragma unroll
                for (int u = 0; u < kAhead; ++u) {
                    add(x[u], runs[u]);
                    runs[u] = next_run();
                    ask(x[u], runs[u]);
                }
            }
        };
        if (inside) walk(std::true_type());
        else walk(std::false_type());
    }
    if (row >= m) return;
#pragma unroll
    for (int c = 0; c < COLUMNS; ++c) {
        if (column0 + c >= n) return;  // whole wavefront
        T* out = C + static_cast<int64_t>(column0 + c) * ldc + row;
        if (m - row >= R) {
            vec_t s;
#pragma unroll
            for (int j = 0; j < R; ++j) s[j] = alpha * sum[c][j];
            if constexpr (!BETA0) {
                const vec_t old = *reinterpret_cast<const element_aligned*>(out);
#pragma unroll
                for (int j = 0; j < R; ++j) s[j] = scaled_sum(alpha, sum[c][j], beta, old[j]);
            }
            __builtin_nontemporal_store(s, reinterpret_cast<element_aligned*>(out));
        } else {
#pragma unroll
            for (int j = 0; j < R; ++j) {
                if (row + j < m) out[j] = BETA0 ? alpha * sum[c][j] : scaled_sum(alpha, sum[c][j], beta, out[j]);
            }
        }
    }
}

}  // namespace

bool spmm_diagonals_usable(idx_t m, idx_t k, idx_t n, uint32_t longest, size_t value_bytes) {
    // Operands of one or two lanes a row run in kernels that add a row up as a tree: other bits.
    if (n * value_bytes <= kTwoLanes) return false;
    // A wavefront walks all diagonals of a slice in turn, which takes as long on the smallest matrix (fp32, 9 to 16 columns:
    // 14 to 18 us): with a workgroup or less to a compute unit the transposes are through before.  Fp32 27-point stencils on
    // cubes of 30, 35, 41 and 48 points, 9 columns, transposes and so: 12.0 and 15.0, 12.7 and 14.5, 15.1 and 15.4, 21.0
    // and 18.1; more columns need more transposing (30, 17 columns: 56 and 15), and slices of fp64 are half as long (30, 9
    // columns: 13.1 and 10.6).
    const uint32_t rows = slice_rows_of(value_bytes);
    if (value_bytes == 4 && n <= kColumns * kPanelWaves && (m - 1) / rows + 1 <= device_topology().cus) return false;
    // the values of a slice fit LDS; places in a column of op(B) fit 32 bits
    return longest <= (value_bytes == 4 ? staged_values<float>() : staged_values<double>()) &&
           static_cast<uint64_t>(k) * value_bytes < (1ull << 32);
}

template <typename T>
void launch_spmm_diagonals(hipStream_t stream, const SpmmArgs& a, uint32_t total, const void* region, T alpha, T beta) {
    const SliceDiagonalsLayout l = slice_diagonals_layout(a.m, a.nnz, sizeof(T), false);
    const char* w = static_cast<const char*>(region);
    const uint32_t xcds = device_topology().xcds;
    const uint32_t waves = (a.n + kColumns - 1) / kColumns;  // of all columns
    const uint32_t panels = (waves + kPanelWaves - 1) / kPanelWaves, panel_waves = (waves + panels - 1) / panels;
    const dim3 grid((l.slices + xcds - 1) / xcds * xcds, panels);
    auto launch = [&](auto columns) {
        constexpr int COLUMNS = decltype(columns)::value;
        auto* kernel = beta == T(0) ? spmm_diagonals_kernel<T, COLUMNS, true> : spmm_diagonals_kernel<T, COLUMNS, false>;
        hipLaunchKernelGGL(kernel, grid, dim3(panel_waves * (kColumns / COLUMNS) * kWave), 0, stream, a.m, a.n, a.k, a.nnz, a.base,
                           l.slices, total, reinterpret_cast<const uint32_t*>(w + l.diagonal_first),
                           reinterpret_cast<const SliceDiagonal<lane_rows<T>()>*>(w + l.diagonals), a.row_ptr,
                           static_cast<const T*>(a.val), static_cast<const T*>(a.B), a.ldb, static_cast<T*>(a.C), a.ldc, alpha,
                           beta, xcds);
    };
    // Up to half a panel: twice the wavefronts with half the columns each (fp64, 101 x 97 x 89, 5 and 8 columns 76.5 -> 67.4
    // and 81.0 -> 75.7 us, 41 x 37 x 29 11.8 -> 10.0 and 11.7 -> 10.2; 9 columns 85.6 with four each, 92.1 with two).
    if (a.n <= kColumns * kPanelWaves / 2) launch(std::integral_constant<int, kColumns / 2>());
    else launch(std::integral_constant<int, kColumns>());
}

template void launch_spmm_diagonals<float>(hipStream_t, const SpmmArgs&, uint32_t, const void*, float, float);
template void launch_spmm_diagonals<double>(hipStream_t, const SpmmArgs&, uint32_t, const void*, double, double);

}  // namespace mcsp
