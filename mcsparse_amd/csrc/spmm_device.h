// Device helpers shared by the SpMM kernels (spmm.hip, spmm_blocks.hip): 128-bit row accesses of op(B) and C,
// the XCD-aware workgroup order, and one row of A times op(B) for a lane group.
#ifndef MCSPARSE_AMD_SPMM_DEVICE_H_
#define MCSPARSE_AMD_SPMM_DEVICE_H_

#include "device_util.h"
#include "internal.h"

namespace mcsp {
namespace spmm_detail {

constexpr int kBlock = 256;

template <typename T, int V>
struct Vec {
    T v[V];
};

template <typename T, int V>
__device__ __forceinline__ Vec<T, V> load_vec(const T* p) {
    Vec<T, V> r;
    if constexpr (V == 1) {
        r.v[0] = p[0];
    } else if constexpr (sizeof(T) * V == 16) {
        typedef T Native __attribute__((ext_vector_type(V)));
        const Native n = *reinterpret_cast<const Native*>(p);
#pragma unroll
        for (int i = 0; i < V; ++i) r.v[i] = n[i];
    } else {
        static_assert(sizeof(T) * V == 8, "unsupported vector width");
        typedef T Native __attribute__((ext_vector_type(V)));
        const Native n = *reinterpret_cast<const Native*>(p);
#pragma unroll
        for (int i = 0; i < V; ++i) r.v[i] = n[i];
    }
    return r;
}

// A row of op(B) may begin at any element (widths and leading dimensions that are no multiple of the vector): the
// hardware takes 128-bit accesses at any multiple of four bytes, so ragged operands keep the wide loads.
template <typename T, int V>
__device__ __forceinline__ Vec<T, V> load_row(const T* p) {
    if constexpr (V == 1) {
        return load_vec<T, V>(p);
    } else {
        typedef T Native __attribute__((ext_vector_type(V), aligned(sizeof(T))));
        Vec<T, V> r;
        const Native n = *reinterpret_cast<const Native*>(p);
#pragma unroll
        for (int i = 0; i < V; ++i) r.v[i] = n[i];
        return r;
    }
}

// The columns of a lane of a row of n >= V columns: V from `own` on, moved back where fewer are left; the first `skip`
// of them then belong to the lane before.  Lanes past the last column (own >= n) get the row's first columns.
struct LaneColumns {
    uint64_t first;
    int skip;
    bool any;
};
template <int V, bool RAGGED = true>
__device__ __forceinline__ LaneColumns lane_columns(uint64_t own, uint64_t n) {
    LaneColumns c;
    c.any = own < n;
    if constexpr (RAGGED) {
        c.first = !c.any ? 0 : (own + V <= n ? own : n - V);
        c.skip = c.any ? static_cast<int>(own - c.first) : V;
    } else {  // n is a multiple of V
        c.first = c.any ? own : 0;
        c.skip = 0;
    }
    return c;
}

// Stores of C: written once and not read again by the call, so they are marked as streaming, which keeps the
// rows of op(B) in cache and lets the lines leave as they fill (N = 64: 552 -> 535 us, N = 256: 1.90 -> 1.82 ms).
template <typename T, int V>
__device__ __forceinline__ void store_vec(T* p, const Vec<T, V>& r) {
    if constexpr (V == 1) {
        __builtin_nontemporal_store(r.v[0], p);
    } else {
        typedef T Native __attribute__((ext_vector_type(V), aligned(sizeof(T))));
        Native n;
#pragma unroll
        for (int i = 0; i < V; ++i) n[i] = r.v[i];
        __builtin_nontemporal_store(n, reinterpret_cast<Native*>(p));
    }
}

// Byte offsets into op(B) are 32-bit when the whole operand lies within 4 GiB of its first
// element (WIDE = false): a row's offset then travels between lanes in one register and the
// load takes it next to the scalar base address, which leaves one vector instruction of address
// arithmetic per row of op(B).
template <bool WIDE>
struct ByteOffset { typedef uint32_t type; };
template <>
struct ByteOffset<true> { typedef uint64_t type; };

// Workgroups are handed to the XCDs of a device in turn (workgroup h runs on XCD h % xcds), each XCD with
// an L2 of its own.  Rows that are close in the matrix tend to read the same rows of op(B), so
// an XCD should work on a contiguous stretch of rows: this maps the hardware's workgroup number
// to a position such that every XCD takes `chunk` consecutive positions at a time.  chunk = 1 (or one XCD)
// is the identity; positions past `count` (the grid is padded to whole rounds) do no work.
__device__ __forceinline__ uint64_t xcd_position(uint32_t hw_block, uint32_t chunk, uint32_t xcds) {
    const uint32_t per_round = xcds * chunk;
    const uint32_t round = hw_block / per_round;
    const uint32_t rem = hw_block % per_round;
    return static_cast<uint64_t>(round) * per_round + (rem % xcds) * chunk + rem / xcds;
}
inline uint32_t xcd_padded_grid(uint64_t count, uint32_t chunk, uint32_t xcds) {
    const uint64_t per_round = static_cast<uint64_t>(xcds) * chunk;
    return static_cast<uint32_t>((count + per_round - 1) / per_round * per_round);
}

// Length of such a stretch for the kernels without a schedule, which know nothing of the structure: workgroups that
// hold kXcdStretchRows rows, but no more than leave every XCD kXcdStretchRounds turns, so that stretches of different
// weight even out.  Neighbouring rows of a stencil or a mesh read mostly the same rows of op(B); in plain turns all
// eight L2s fetch them.  27-point stencil 101 x 97 x 89, 16 fp64 columns, microseconds per product: 189 in plain turns,
// 179, 178, 180, 185, 186 with 1024, 2048, 4096, 8192, 16384 rows; a million power-law rows, 8 fp32 columns: 407 and
// 385, 392, 384, 390, 396.
constexpr uint64_t kXcdStretchRows = 2048;
constexpr uint64_t kXcdStretchRounds = 4;
inline uint32_t xcd_stretch(uint64_t blocks, uint64_t rows_per_block, uint32_t xcds) {
    uint32_t chunk = 1;
    if (xcds <= 1) return chunk;
    while (chunk * 2 * rows_per_block <= kXcdStretchRows && chunk * 2 * xcds * kXcdStretchRounds <= blocks) chunk *= 2;
    return chunk;
}

// acc += sum over the nonzeros [begin, end) of one row of A of value * (V columns of the row of
// op(B) the nonzero names), for a group of LR >= 4 lanes that all pass the same range.
// B_bytes is the operand's first element, lane_off the byte offset of this lane's columns.
//
// What bounds these kernels is the return path of the vector memory unit, and a load in which
// all lanes of a group ask for the same word still returns a word per lane.  So the lanes fetch
// LR nonzeros of the row at once, one each, turn them into row offsets, and pass offsets and
// values round in registers; the loop then loads rows of op(B) and nothing else.
//
// AHEAD: the group takes every step / LR-th stretch of LR nonzeros from begin on (several groups on one long row), and
// asks for the next one before the rows of op(B) of this one, so that a round costs one trip to memory instead of two
// (places past the end read the last nonzero again: no load sits under a test).  Not for the short rows of a stencil,
// which it makes slower (27 nonzeros, 16 fp64 columns: 178 -> 187 us): they have other rows to wait beside.
template <typename T, int LR, int V, bool WIDE, bool AHEAD = false>
__device__ __forceinline__ void row_times_b(idx_t begin, idx_t end, idx_t lane, idx_t base,
                                            const idx_t* __restrict__ col, const T* __restrict__ val,
                                            const char* __restrict__ B_bytes,
                                            typename ByteOffset<WIDE>::type lane_off,
                                            typename ByteOffset<WIDE>::type ldb_bytes, T (&acc)[V],
                                            idx_t step = LR) {
    typedef typename ByteOffset<WIDE>::type off_t;
    constexpr int kBatch = LR < 8 ? LR : 8;  // rows of op(B) in flight per lane
    if (begin >= end) return;  // whole lane groups
    idx_t c_next = 0;
    T a_next = T(0);
    if constexpr (AHEAD) {
        c_next = col[min(begin + lane, end - 1)];
        a_next = val[min(begin + lane, end - 1)];
    }
    for (idx_t j = begin; j < end; j += step) {
        const idx_t left = end - j;
        off_t roff;
        T aa;
        if constexpr (AHEAD) {
            roff = static_cast<off_t>(c_next - base) * ldb_bytes;
            aa = a_next;
            const idx_t next = left > step ? min(j + step + lane, end - 1) : end - 1;
            c_next = col[next];
            a_next = val[next];
        } else {
            const bool has = lane < left;
            roff = has ? static_cast<off_t>(col[j + lane] - base) * ldb_bytes : off_t(0);
            aa = has ? val[j + lane] : T(0);
        }
        auto chunk = [&](auto checked) {
            constexpr bool kChecked = decltype(checked)::value;
            static_for<LR / kBatch>([&](auto g) {
                constexpr int u0 = decltype(g)::value * kBatch;
                if (!kChecked || u0 < left) {
                    Vec<T, V> b[kBatch];
                    static_for<kBatch>([&](auto u) {
                        constexpr int k = u0 + decltype(u)::value;
                        if (!kChecked || k < left) {  // the same for all lanes of the group
                            const off_t off = group_bcast<LR, k>(roff) + lane_off;
                            b[decltype(u)::value] = load_row<T, V>(reinterpret_cast<const T*>(B_bytes + off));
                        }
                    });
                    static_for<kBatch>([&](auto u) {
                        constexpr int k = u0 + decltype(u)::value;
                        if (!kChecked || k < left) {
                            const T a = group_bcast<LR, k>(aa);
#pragma unroll
                            for (int i = 0; i < V; ++i) acc[i] += a * b[decltype(u)::value].v[i];
                        }
                    });
                }
            });
        };
        if (left >= LR) chunk(std::false_type{});
        else chunk(std::true_type{});
    }
}

// Writes V adjacent columns of one row of C but for the first `skip`: beta*C + alpha*acc, C untouched by reads if
// beta == 0.
template <typename T, int V>
__device__ __forceinline__ void store_c(T* __restrict__ C, int64_t ldc, bool c_row_major, uint64_t row, uint64_t c0,
                                        const T (&acc)[V], T alpha, T beta, int skip = 0) {
    const bool beta0 = beta == T(0);
    if (V > 1 && skip != 0) {
        T* Cp = c_row_major ? C + static_cast<int64_t>(row) * ldc + c0 : C + static_cast<int64_t>(c0) * ldc + row;
        const int64_t next = c_row_major ? 1 : ldc;
#pragma unroll
        for (int i = 1; i < V; ++i) {
            if (i >= skip) Cp[i * next] = beta0 ? alpha * acc[i] : scaled_sum(alpha, acc[i], beta, Cp[i * next]);
        }
    } else if (c_row_major) {
        T* Cp = C + static_cast<int64_t>(row) * ldc + c0;
        Vec<T, V> out;
        if (beta0) {
#pragma unroll
            for (int i = 0; i < V; ++i) out.v[i] = alpha * acc[i];
        } else {
            const Vec<T, V> old = load_row<T, V>(Cp);
#pragma unroll
            for (int i = 0; i < V; ++i) out.v[i] = scaled_sum(alpha, acc[i], beta, old.v[i]);
        }
        store_vec<T, V>(Cp, out);
    } else {
#pragma unroll
        for (int i = 0; i < V; ++i) {
            T* Cp = C + static_cast<int64_t>(c0 + i) * ldc + row;
            *Cp = beta0 ? alpha * acc[i] : scaled_sum(alpha, acc[i], beta, *Cp);
        }
    }
}

// Four consecutive rows of one column of a column-major C (16-byte aligned): beta*C + alpha*acc with
// 128-bit accesses, C untouched by reads if beta == 0.
template <typename T>
__device__ __forceinline__ void store_c_four_rows(T* __restrict__ Cp, T a0, T a1, T a2, T a3, T alpha, T beta) {
    constexpr int W = 16 / sizeof(T);  // elements per 128-bit access: 4 floats, 2 doubles
    const T acc[4] = {a0, a1, a2, a3};
    const bool beta0 = beta == T(0);
#pragma unroll
    for (int h = 0; h < 4 / W; ++h) {
        Vec<T, W> out;
        if (beta0) {
#pragma unroll
            for (int i = 0; i < W; ++i) out.v[i] = alpha * acc[h * W + i];
        } else {
            const Vec<T, W> old = load_vec<T, W>(Cp + h * W);
#pragma unroll
            for (int i = 0; i < W; ++i) out.v[i] = scaled_sum(alpha, acc[h * W + i], beta, old.v[i]);
        }
        store_vec<T, W>(Cp + h * W, out);
    }
}

// op(B) lies within 4 GiB of its first element: byte offsets into it fit 32 bits
inline bool narrow_offsets(const SpmmArgs& a, size_t value_bytes) {
    const uint64_t last = (a.k == 0 ? 0 : static_cast<uint64_t>(a.k) - 1) * static_cast<uint64_t>(a.ldb) + a.n;
    return last * value_bytes <= 0xffffffffull;
}

}  // namespace spmm_detail
}  // namespace mcsp

#endif  // MCSPARSE_AMD_SPMM_DEVICE_H_
