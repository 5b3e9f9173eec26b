// Long rows of a CSR SpMM.  The row kernels (spmm.hip) give a row of A to one lane group, which walks its
// nonzeros with a handful of loads in flight: a row of 50,000 nonzeros keeps that one group busy for
// milliseconds after every other row is done (1 M power-law rows, N = 16: 7.3 ms, of which the longest row is 7).
// The reference has the same shape (one wavefront per row and output column,
// src/kernels/level3/spmm/csr_spmm_device.hpp:121-137).  Here rows longer than the call's cut (256 to
// 1024 nonzeros, spmm_long_cut) are left out by the row kernels and taken in pieces of kSpmmLongChunk nonzeros, a workgroup each:
//   1. spmm_long_find_kernel lists the pieces (row, piece) and, for rows of several pieces, the rows, and notes whether any
//      row has more than kSpmmLongRow nonzeros: if none has, the row kernels take them all.  A call that does not know
//      that beforehand runs it in front of the row kernels, so what becomes of a row depends on the matrix alone;
//   2. spmm_long_chunk_kernel forms the sums of a piece, all 256 threads on its nonzeros, and writes the row of C
//      (one piece) or a row of partial sums (several);
//   3. spmm_long_reduce_kernel adds the partial sums of a row in the order of the pieces and writes the row of C.
// Where op(B) is far larger than the L2s, step 2 goes band by band of op(B): see the bands below.
// Every sum is formed in a fixed order, so results repeat bit for bit; where the pieces and partial sums of a row
// lie in the scratch area depends on the order in which the rows were found, which nothing else depends on.
#include "spmm_long_device.h"

namespace mcsp {

namespace {

using namespace spmm_detail;

__global__ void spmm_long_zero_kernel(LongCounters* c, bool known) {
    c->items = 0;
    c->several = 0;
    c->apart = known ? 1 : 0;
    c->unsorted = 0;
}

// item: {row, piece, pieces of the row, first row of partial sums of the row (unused for one piece)}
//
// The places in the three lists come off three counters, and atomic adds to one address take their turns (3.4 ns
// each: 12,000 long rows among 4 M, found by a thread each, 195 us).  So a workgroup looks at kFindRows rows,
// collects its long ones in LDS with places relative to the workgroup, and takes its share of the lists with one
// add per counter (the same matrix: 36 us).  4096 rows a workgroup instead of 8192 take 6 us off the call on 100,000
// rows (71 -> 65 us) and cost 14 on 4 M (1975 -> 1989).
constexpr uint32_t kFindRows = 4096;   // rows a workgroup looks at
constexpr uint32_t kFindList = 2048;   // long rows it can collect; further ones take their places one by one

__device__ __forceinline__ void write_long_row(uint32_t row, uint32_t pieces, uint32_t first, uint32_t slot, uint32_t at,
                                               uint4* __restrict__ items, uint4* __restrict__ rows, uint32_t cap_items,
                                               uint32_t cap_rows, uint32_t cap_slots) {
    // (the capacities hold for every structure whose offsets add up to nnz; for one that does not, nothing is
    // written out of bounds, and the rows that found no room are missing from the product)
    bool fits = first + pieces <= cap_items && first + pieces >= first;
    if (pieces > 1) {
        fits = fits && slot + pieces <= cap_slots && slot + pieces >= slot && at < cap_rows;
        if (at < cap_rows) rows[at] = fits ? make_uint4(row, slot, pieces, first) : make_uint4(row, 0u, 0u, 0u);
    }
    for (uint32_t j = 0; j < pieces && first + j < cap_items; ++j)
        items[first + j] = make_uint4(row, j, fits ? pieces : 0u, slot);
}

__global__ __launch_bounds__(kBlock) void spmm_long_find_kernel(idx_t m, idx_t long_row, const idx_t* __restrict__ row_ptr,
                                                                LongCounters* __restrict__ c, uint4* __restrict__ items,
                                                                uint4* __restrict__ rows, uint32_t cap_items,
                                                                uint32_t cap_rows, uint32_t cap_slots) {
    __shared__ uint4 s_list[kFindList];      // {row, pieces, first item, first slot}, relative to the workgroup
    __shared__ uint32_t s_list_row[kFindList];  // place in the list of rows of several pieces
    __shared__ uint32_t s_count, s_items, s_slots, s_rows, s_apart;
    __shared__ uint32_t s_base;
    __shared__ unsigned long long s_base_several;
    const uint32_t tid = threadIdx.x;
    if (tid == 0) {
        s_count = 0;
        s_items = 0;
        s_slots = 0;
        s_rows = 0;
        s_apart = 0;
    }
    __syncthreads();
    const uint64_t row0 = static_cast<uint64_t>(blockIdx.x) * kFindRows;
    constexpr uint32_t kAtOnce = 8;  // rows a thread asks for before it looks at any: one trip to memory for the lot
    static_assert(kFindRows % (kBlock * kAtOnce) == 0, "whole rounds");
    bool apart = false;
    for (uint32_t k0 = tid; k0 < kFindRows; k0 += kBlock * kAtOnce) {
        idx_t lens[kAtOnce];
#pragma unroll
        for (uint32_t u = 0; u < kAtOnce; ++u) {
            const uint64_t row = row0 + k0 + u * kBlock;
            const uint64_t r = row < m ? row : m - 1;  // m != 0 here
            lens[u] = row < m ? row_ptr[r + 1] - row_ptr[r] : 0;
        }
#pragma unroll
        for (uint32_t u = 0; u < kAtOnce; ++u) {
            const uint64_t row = row0 + k0 + u * kBlock;
            const idx_t len = lens[u];
            if (len <= long_row) continue;
            apart |= len > kSpmmLongRow;
            const uint32_t pieces = (len + kSpmmLongChunk - 1) / kSpmmLongChunk;
            const uint32_t at = atomicAdd(&s_count, 1u);
            if (at < kFindList) {
                const uint32_t first = atomicAdd(&s_items, pieces);
                const uint32_t slot = pieces > 1 ? atomicAdd(&s_slots, pieces) : 0u;
                s_list_row[at] = pieces > 1 ? atomicAdd(&s_rows, 1u) : 0u;
                s_list[at] = make_uint4(static_cast<uint32_t>(row), pieces, first, slot);
            } else {  // no room in the workgroup's list: places straight off the counters
                const uint32_t first = atomicAdd(&c->items, pieces);
                const unsigned long long there = pieces > 1 ? atomicAdd(&c->several, 1ull << 32 | pieces) : 0ull;
                write_long_row(static_cast<uint32_t>(row), pieces, first, static_cast<uint32_t>(there),
                               static_cast<uint32_t>(there >> 32), items, rows, cap_items, cap_rows, cap_slots);
            }
        }
    }
    if (apart) s_apart = 1;
    __syncthreads();
    const uint32_t listed = min(s_count, kFindList);
    if (listed == 0) return;  // whole workgroup
    if (tid == 0) {
        if (s_apart != 0) c->apart = 1;
        s_base = atomicAdd(&c->items, s_items);
        s_base_several = s_rows != 0 ? atomicAdd(&c->several, static_cast<unsigned long long>(s_rows) << 32 | s_slots) : 0ull;
    }
    __syncthreads();
    for (uint32_t k = tid; k < listed; k += kBlock) {
        const uint4 e = s_list[k];
        write_long_row(e.x, e.y, s_base + e.z, static_cast<uint32_t>(s_base_several) + e.w,
                       static_cast<uint32_t>(s_base_several >> 32) + s_list_row[k], items, rows, cap_items, cap_rows, cap_slots);
    }
}

__global__ __launch_bounds__(kBlock) void spmm_long_bounds_kernel(BoundsWork work, idx_t base, idx_t nnz,
                                                                  const idx_t* __restrict__ row_ptr,
                                                                  const idx_t* __restrict__ col) {
    cut_pieces(work, base, nnz, row_ptr, col);
}

// A wavefront's share of the bands: kBandTake pairs of band and item at a time, off one of its XCD's counters.  A round is up to 64 nonzeros of a pair, one
// asked for by every lane: nonzero t goes to lane group t % G, so that the groups load equally many rows of op(B).  The
// nonzeros of the next round, often the next pair's, are asked for before the rows of this one.
template <typename T, int LR, int V>
__device__ __forceinline__ void take_bands(const BandPlan& plan, const LaneColumns& own, idx_t base, const idx_t* __restrict__ col,
                                           const T* __restrict__ val, const T* __restrict__ B, int64_t ldb, int64_t ld_partials) {
    constexpr uint32_t G = kWave / LR;
    const uint32_t lane = threadIdx.x % kWave, group = lane / LR, place = lane % LR * G + group;
    const uint32_t stretch = blockIdx.x % kBandStretches;
    const uint32_t all = plan.bands / kBandStretches * plan.items;  // pairs of the stretch, band after band
    const uint32_t queue = (blockIdx.x / kBandStretches * (kBlock / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave)) % kBandQueues;
    uint32_t* taken = plan.taken + (stretch * kBandQueues + queue) * (kAlign / sizeof(uint32_t));
    T* sums = static_cast<T*>(plan.sums);
    const char* B_bytes = reinterpret_cast<const char*>(B);
    const uint32_t lane_off = static_cast<uint32_t>(own.first * sizeof(T)), ldb_bytes = static_cast<uint32_t>(ldb * sizeof(T));
    auto take = [&]() {
        uint32_t at = 0;
        if (lane == 0) at = atomicAdd(taken, 1u);
        return at;
    };
    uint32_t next = take();
    while (true) {
        const uint32_t from = (__builtin_amdgcn_readfirstlane(next) * kBandQueues + queue) * kBandTake;
        if (from >= all) break;  // whole wavefront
        next = take();  // on its way while this share is worked on
        const uint32_t pairs = min(kBandTake, all - from);
        // lane p keeps the bounds of pair p
        const uint32_t mine = from + min(lane, pairs - 1), turn = mine / plan.items, it = mine - turn * plan.items;
        const uint64_t at = static_cast<uint64_t>(it) * (plan.bands + 1) + turn * kBandStretches + stretch;
        const uint32_t my_begin = plan.bounds[at], my_end = plan.bounds[at + 1];
        const uint32_t my_sum = it * plan.bands + turn * kBandStretches + stretch;
        unsigned long long left = __ballot(lane < pairs && my_begin < my_end);
        if (left == 0) continue;  // whole wavefront
        uint32_t p = __builtin_ctzll(left);
        left &= left - 1;
        uint32_t j = __builtin_amdgcn_readlane(my_begin, p), end = __builtin_amdgcn_readlane(my_end, p);
        idx_t c_next = col[min(j + place, end - 1)];
        T a_next = val[min(j + place, end - 1)];
        T acc[V];
#pragma unroll
        for (int i = 0; i < V; ++i) acc[i] = T(0);
        while (true) {  // a round of pair p
            const uint32_t count = min(end - j, static_cast<uint32_t>(kWave));
            const uint32_t roff = (c_next - base) * ldb_bytes;
            const T aa = a_next;
            const bool last = j + kWave >= end;
            const uint32_t p_now = p;
            if (last) {
                if (left != 0) {
                    p = __builtin_ctzll(left);
                    left &= left - 1;
                    j = __builtin_amdgcn_readlane(my_begin, p);
                    end = __builtin_amdgcn_readlane(my_end, p);
                } else {
                    p = kWave;  // none
                }
            } else {
                j += kWave;
            }
            c_next = col[min(j + place, end - 1)];
            a_next = val[min(j + place, end - 1)];
            Vec<T, V> b[LR];
            static_for<LR>([&](auto k) {
                constexpr int kk = decltype(k)::value;
                if (kk * G < count)  // the same for the wavefront
                    b[kk] = load_row<T, V>(reinterpret_cast<const T*>(B_bytes + (group_bcast<LR, kk>(roff) + lane_off)));
            });
            T of_round[V];  // (a sum of its own, so that a pair of thousands is no chain of hundreds)
#pragma unroll
            for (int i = 0; i < V; ++i) of_round[i] = T(0);
            static_for<LR>([&](auto k) {
                constexpr int kk = decltype(k)::value;
                if (kk * G + group < count) {  // a lane without a nonzero stays out: 0 * inf would be NaN
                    const T a = group_bcast<LR, kk>(aa);
#pragma unroll
                    for (int i = 0; i < V; ++i) of_round[i] += a * b[kk].v[i];
                }
            });
#pragma unroll
            for (int i = 0; i < V; ++i) acc[i] += of_round[i];
            if (!last) continue;
#pragma unroll
            for (int i = 0; i < V; ++i) {
#pragma unroll
                for (int off = LR; off < kWave; off <<= 1) acc[i] += __shfl_xor(acc[i], off, kWave);
            }
            if (group == 0 && own.any) {
                T* out = sums + static_cast<int64_t>(__builtin_amdgcn_readlane(my_sum, p_now)) * ld_partials + own.first;
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    if (i >= own.skip) out[i] = acc[i];
                }
            }
            if (p == kWave) break;
#pragma unroll
            for (int i = 0; i < V; ++i) acc[i] = T(0);
        }
    }
}

// lanes: lane groups of `lanes` threads (a power of two up to 64) hold the columns of a panel of lanes * V columns
// (blockIdx.y walks the panels); the kBlock / lanes groups take the nonzeros of the piece in turn, kAhead rows of
// op(B) in flight each, and their sums meet in LDS, added in the order of the groups.
// op(B)(kk, j) lies at kk * b_rs + j * b_cs; V > 1 needs b_cs == 1 and n >= V (the launcher checks).
template <typename T, int V>
__global__ __launch_bounds__(kBlock) void spmm_long_chunk_kernel(idx_t n, idx_t base, uint32_t lanes,
                                                                 const idx_t* __restrict__ row_ptr,
                                                                 const idx_t* __restrict__ col, const T* __restrict__ val,
                                                                 const T* __restrict__ B, int64_t b_rs, int64_t b_cs,
                                                                 T* __restrict__ C, int64_t ldc, bool c_row_major,
                                                                 T alpha, T beta, const LongCounters* __restrict__ c,
                                                                 const uint4* __restrict__ items, uint32_t cap_items,
                                                                 T* __restrict__ partials, int64_t ld_partials, idx_t nnz) {
    constexpr int kAhead = 4;
    __shared__ T s_sum[kBlock * V];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid % lanes;
    const uint32_t group = tid / lanes;
    const uint32_t groups = kBlock / lanes;
    const LaneColumns own = lane_columns<V>((static_cast<uint64_t>(blockIdx.y) * lanes + lane) * V, n);
    const uint64_t c0 = own.first;
    const uint32_t count = c->apart != 0 ? min(c->items, cap_items) : 0u;
    const idx_t last_nonzero = nnz - 1;  // nnz != 0 where a row is long
    for (uint32_t it = blockIdx.x; it < count; it += gridDim.x) {
        const uint4 item = items[it];
        const uint32_t row = item.x, piece = item.y, pieces = item.z;
        if (pieces == 0) continue;  // whole workgroup: a row that found no room
        const idx_t row_start = row_ptr[row] - base;
        const idx_t row_end = min(row_ptr[row + 1] - base, nnz);
        const idx_t start = row_start + piece * kSpmmLongChunk;
        const idx_t end = min(start + static_cast<idx_t>(kSpmmLongChunk), row_end);
        T acc[V];
#pragma unroll
        for (int i = 0; i < V; ++i) acc[i] = T(0);
        for (idx_t e = start + group; e < end; e += groups * kAhead) {
            idx_t cc[kAhead];
            T aa[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const idx_t j = min(e + u * groups, last_nonzero);
                cc[u] = col[j] - base;
                aa[u] = val[j];
            }
            Vec<T, V> b[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u)
                b[u] = load_row<T, V>(B + static_cast<int64_t>(cc[u]) * b_rs + static_cast<int64_t>(c0) * b_cs);
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                if (e + u * groups < end) {  // a lane without a nonzero stays out: 0 * inf would be NaN
#pragma unroll
                    for (int i = 0; i < V; ++i) acc[i] += aa[u] * b[u].v[i];
                }
            }
        }
#pragma unroll
        for (int i = 0; i < V; ++i) s_sum[tid * V + i] = acc[i];
        __syncthreads();
        if (group == 0) {
            T sum[V];
#pragma unroll
            for (int i = 0; i < V; ++i) sum[i] = T(0);
            for (uint32_t g = 0; g < groups; ++g) {
#pragma unroll
                for (int i = 0; i < V; ++i) sum[i] += s_sum[(g * lanes + lane) * V + i];
            }
            if (own.any) {
                if (pieces == 1) {
                    store_c<T, V>(C, ldc, c_row_major, row, c0, sum, alpha, beta, own.skip);
                } else {
                    T* out = partials + static_cast<int64_t>(item.w + piece) * ld_partials + c0;
#pragma unroll
                    for (int i = 0; i < V; ++i) {
                        if (i >= own.skip) out[i] = sum[i];
                    }
                }
            }
        }
        __syncthreads();  // the sums are read before the next piece writes them
    }
}

// The same for operands of LR = 4 .. 64 lanes of whole vectors that lie within 4 GiB, where most of the work is: a
// wavefront's groups take neighbouring stretches of LR nonzeros, one per lane, read ahead, and pass them round in
// registers (row_times_b), so that a trip to memory brings eight rows of op(B) per lane; the kernel above makes two
// dependent trips for four, and every lane of its groups loads the same nonzero.  What bounds it is the gather of op(B):
// a million power-law rows, 32 fp32 columns, rows of more than 256 nonzeros: 325 us; before, with rows from 1024
// on: 270 us beside a row kernel of 369, which now takes 200.  The sums of a wavefront's groups meet
// in registers, those of the four wavefronts in LDS, in a fixed order.
template <typename T, int LR, int V>
__global__ __launch_bounds__(kBlock) void spmm_long_stretch_kernel(idx_t n, idx_t base, const idx_t* __restrict__ row_ptr,
                                                                   const idx_t* __restrict__ col,
                                                                   const T* __restrict__ val, const T* __restrict__ B,
                                                                   int64_t ldb, T* __restrict__ C, int64_t ldc,
                                                                   bool c_row_major, T alpha, T beta,
                                                                   const LongCounters* __restrict__ c,
                                                                   const uint4* __restrict__ items, uint32_t cap_items,
                                                                   T* __restrict__ partials, int64_t ld_partials, idx_t nnz,
                                                                   BandSpace space) {
    constexpr int kWaves = kBlock / kWave;
    __shared__ T s_sum[kWaves][LR * V];
    const uint32_t lane = threadIdx.x % LR;
    const uint32_t group = threadIdx.x / LR;
    const uint32_t wave = threadIdx.x / kWave;
    const LaneColumns own = lane_columns<V>((static_cast<uint64_t>(blockIdx.y) * LR + lane) * V, n);
    const BandPlan plan = band_plan(space, c, cap_items);
    if (plan.bands != 0) {  // the same for all workgroups
        if constexpr (LR <= kBandLanes) take_bands<T, LR, V>(plan, own, base, col, val, B, ldb, ld_partials);
        return;
    }
    const uint32_t count = c->apart != 0 ? min(c->items, cap_items) : 0u;
    for (uint32_t it = blockIdx.x; it < count; it += gridDim.x) {
        const uint4 item = items[it];
        const uint32_t row = item.x, piece = item.y, pieces = item.z;
        if (pieces == 0) continue;  // whole workgroup: a row that found no room
        const idx_t row_start = row_ptr[row] - base;
        const idx_t row_end = min(row_ptr[row + 1] - base, nnz);
        const idx_t start = row_start + piece * kSpmmLongChunk;
        const idx_t end = min(start + static_cast<idx_t>(kSpmmLongChunk), row_end);
        T acc[V];
#pragma unroll
        for (int i = 0; i < V; ++i) acc[i] = T(0);
        row_times_b<T, LR, V, false, true>(start + group * LR, end, lane, base, col, val, reinterpret_cast<const char*>(B),
                                           static_cast<uint32_t>(own.first * sizeof(T)),
                                           static_cast<uint32_t>(ldb * sizeof(T)), acc, kBlock);
#pragma unroll
        for (int i = 0; i < V; ++i) {
#pragma unroll
            for (int off = LR; off < kWave; off <<= 1) acc[i] += __shfl_xor(acc[i], off, kWave);
        }
        if (threadIdx.x % kWave < LR) {
#pragma unroll
            for (int i = 0; i < V; ++i) s_sum[wave][lane * V + i] = acc[i];
        }
        __syncthreads();
        if (group == 0 && own.any) {
#pragma unroll
            for (int w = 1; w < kWaves; ++w) {
#pragma unroll
                for (int i = 0; i < V; ++i) acc[i] += s_sum[w][lane * V + i];
            }
            if (pieces == 1) {
                store_c<T, V>(C, ldc, c_row_major, row, own.first, acc, alpha, beta, own.skip);
            } else {
                T* out = partials + static_cast<int64_t>(item.w + piece) * ld_partials + own.first;
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    if (i >= own.skip) out[i] = acc[i];
                }
            }
        }
        __syncthreads();  // the sums are read before the next piece writes them
    }
}

// One thread per (row of several pieces, V columns): the partial sums of the pieces in their order.
template <typename T, int V>
__global__ __launch_bounds__(kBlock) void spmm_long_reduce_kernel(idx_t n, T* __restrict__ C, int64_t ldc,
                                                                  bool c_row_major, T alpha, T beta,
                                                                  const LongCounters* __restrict__ c,
                                                                  const uint4* __restrict__ rows, uint32_t cap_rows,
                                                                  const T* __restrict__ partials, int64_t ld_partials,
                                                                  const uint4* __restrict__ items, uint32_t cap_items,
                                                                  BandSpace space) {
    const uint64_t per_row = (static_cast<uint64_t>(n) + V - 1) / V;
    const BandPlan plan = band_plan(space, c, cap_items);
    if (plan.bands != 0) {  // the same for all workgroups: the partial sums of all pieces of a row, band by band
        constexpr uint32_t kLanes = 8, kGroups = kWave / kLanes, kWaves = kBlock / kWave;
        static_assert(kBandStretches % kGroups == 0, "whole rounds");
        __shared__ T s_sum[kWaves][kLanes * V];
        const uint32_t wave_lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, lane = threadIdx.x % kLanes, group = wave_lane / kLanes;
        const uint64_t panels = (per_row + kLanes - 1) / kLanes;
        // sum += the sums of every `step`-th of `pieces` pieces of a row, the first of which is item `it`
        auto add_pieces = [&](uint32_t it, uint32_t pieces, uint32_t step, const LaneColumns& own, T (&sum)[V]) {
            // 64 bands of a piece at a time; the bounds of the next 64 are asked for before the sums of these
            const uint32_t rounds = (plan.bands + kWave - 1) / kWave;
            const uint64_t next_bounds = static_cast<uint64_t>(step) * (plan.bands + 1);
            const uint32_t* bounds = plan.bounds + static_cast<uint64_t>(it) * (plan.bands + 1);
            const T* in = static_cast<const T*>(plan.sums) + static_cast<int64_t>(it) * plan.bands * ld_partials + own.first;
            uint32_t b0 = 0, b = min(wave_lane, plan.bands - 1), begin = bounds[b], end = bounds[b + 1];
            for (uint32_t steps = (pieces + step - 1) / step * rounds; steps != 0; --steps) {
                const bool holds = b0 + wave_lane < plan.bands && begin != end;
                const uint32_t band_here = b;
                const T* in_here = in;
                b0 += kWave;
                if (b0 >= plan.bands) {
                    b0 = 0;
                    if (steps != 1) {
                        bounds += next_bounds;
                        in += static_cast<int64_t>(step) * plan.bands * ld_partials;
                    }
                }
                b = min(b0 + wave_lane, plan.bands - 1);
                begin = bounds[b];
                end = bounds[b + 1];
                // the bands that hold nonzeros of the piece (for the others nothing was written), the groups in turn
                const unsigned long long holding = __ballot(holds);
                const uint32_t rank = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(holding >> 32),
                                                                __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(holding), 0u));
                // lane r learns the r-th of them (lanes without one send to the last lane, where nobody looks unless all hold)
                const uint32_t bands_held = __popcll(holding);
                const uint32_t band = __builtin_amdgcn_ds_permute(static_cast<int>((holds ? rank : kWave - 1) * 4), static_cast<int>(band_here));
                constexpr uint32_t kAtOnce = 4;
                for (uint32_t r0 = 0; r0 < bands_held; r0 += kGroups * kAtOnce) {
                    Vec<T, V> part[kAtOnce];
#pragma unroll
                    for (uint32_t u = 0; u < kAtOnce; ++u) {
                        const uint32_t r = min(r0 + u * kGroups + group, bands_held - 1);
                        part[u] = load_row<T, V>(in_here + static_cast<int64_t>(__shfl(band, r, kWave)) * ld_partials);
                    }
#pragma unroll
                    for (uint32_t u = 0; u < kAtOnce; ++u) {
                        if (r0 + u * kGroups + group < bands_held) {
#pragma unroll
                            for (int i = 0; i < V; ++i) sum[i] += part[u].v[i];
                        }
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < V; ++i) {
#pragma unroll
                for (int off = kLanes; off < kWave; off <<= 1) sum[i] += __shfl_xor(sum[i], off, kWave);
            }
        };
        // A row of several pieces is a workgroup's, a wavefront every fourth piece (a wavefront for all 13 of the longest row
        // took as long as all other rows: 18.0 -> 15.0 us).
        const uint64_t several = static_cast<uint64_t>(min(c->rows(), cap_rows)) * panels;
        for (uint64_t w = blockIdx.x; w < several; w += gridDim.x) {
            const uint4 row = rows[w / panels];
            if (row.z == 0) continue;  // whole workgroup: a row that found no room
            const LaneColumns own = lane_columns<V>((w % panels * kLanes + lane) * V, n);
            T sum[V];
#pragma unroll
            for (int i = 0; i < V; ++i) sum[i] = T(0);
            if (wave < row.z) add_pieces(row.w + wave, row.z - wave, kWaves, own, sum);
            if (group == 0) {
#pragma unroll
                for (int i = 0; i < V; ++i) s_sum[wave][lane * V + i] = sum[i];
            }
            __syncthreads();
            if (wave == 0 && group == 0 && own.any) {
#pragma unroll
                for (uint32_t k = 1; k < kWaves; ++k) {
#pragma unroll
                    for (int i = 0; i < V; ++i) sum[i] += s_sum[k][lane * V + i];
                }
                store_c<T, V>(C, ldc, c_row_major, row.x, own.first, sum, alpha, beta, own.skip);
            }
            __syncthreads();  // the sums are read before the next row's are written
        }
        for (uint64_t w = static_cast<uint64_t>(blockIdx.x) * kWaves + wave; w < plan.items * panels;
             w += static_cast<uint64_t>(gridDim.x) * kWaves) {
            const uint32_t it = static_cast<uint32_t>(w / panels);
            const uint4 item = items[it];
            if (item.z != 1) continue;  // whole wavefront: of several pieces, or a row that found no room
            const LaneColumns own = lane_columns<V>((w % panels * kLanes + lane) * V, n);
            T sum[V];
#pragma unroll
            for (int i = 0; i < V; ++i) sum[i] = T(0);
            add_pieces(it, 1, 1, own, sum);
            if (group == 0 && own.any) store_c<T, V>(C, ldc, c_row_major, item.x, own.first, sum, alpha, beta, own.skip);
        }
        return;
    }
    const uint64_t work = c->apart != 0 ? static_cast<uint64_t>(min(c->rows(), cap_rows)) * per_row : 0;
    for (uint64_t w = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; w < work;
         w += static_cast<uint64_t>(gridDim.x) * kBlock) {
        const uint4 entry = rows[w / per_row];
        const LaneColumns own = lane_columns<V>((w % per_row) * V, n);
        const uint64_t c0 = own.first;
        if (entry.z == 0) continue;
        T sum[V];
#pragma unroll
        for (int i = 0; i < V; ++i) sum[i] = T(0);
        for (uint32_t j = 0; j < entry.z; ++j) {
            const T* in = partials + static_cast<int64_t>(entry.y + j) * ld_partials + c0;
#pragma unroll
            for (int i = 0; i < V; ++i) sum[i] += in[i];
        }
        store_c<T, V>(C, ldc, c_row_major, entry.x, c0, sum, alpha, beta, own.skip);
    }
}

struct LongLayout {
    size_t counters, items, rows, partials, total;
    uint32_t cap_items, cap_rows, cap_slots;
    int64_t ld_partials;
};

// A row of several pieces is longer than a piece, so there are at most nnz / piece such rows, with at most
// 2 * nnz / piece pieces (ceil(len / piece) <= 2 * len / piece); rows of one piece number at most
// nnz / kSpmmLongCutLeast.
LongLayout long_layout(idx_t nnz, int64_t n, size_t value_bytes) {
    LongLayout l;
    const uint64_t per_piece = static_cast<uint64_t>(nnz) / kSpmmLongChunk;
    l.cap_rows = static_cast<uint32_t>(per_piece + 1);
    l.cap_slots = static_cast<uint32_t>(2 * per_piece + 2);
    l.cap_items = static_cast<uint32_t>(static_cast<uint64_t>(nnz) / kSpmmLongCutLeast + 2 * per_piece + 2);
    l.ld_partials = (n + 3) / 4 * 4;
    size_t off = 0;
    // the first kAlign bytes are left to the row-length analysis of the call (34 counters)
    off += 2 * kAlign;
    l.counters = off; off += 2 * kAlign;
    l.items = off; off += align_up(static_cast<size_t>(l.cap_items) * sizeof(uint4));
    l.rows = off; off += align_up(static_cast<size_t>(l.cap_rows) * sizeof(uint4));
    l.partials = off; off += align_up(static_cast<size_t>(l.cap_slots) * l.ld_partials * value_bytes);
    l.total = off;
    return l;
}

}  // namespace

size_t spmm_long_rows_bytes(idx_t nnz, int64_t n, size_t value_bytes) { return long_layout(nnz, n, value_bytes).total; }

const uint32_t* launch_spmm_long_find(hipStream_t stream, const SpmmArgs& a, size_t value_bytes) {
    const LongLayout l = long_layout(a.nnz, a.long_n, value_bytes);
    char* w = static_cast<char*>(a.long_ws);
    LongCounters* c = reinterpret_cast<LongCounters*>(w + l.counters);
    hipLaunchKernelGGL(spmm_long_zero_kernel, dim3(1), dim3(1), 0, stream, c, a.long_known);
    hipLaunchKernelGGL(spmm_long_find_kernel, dim3((a.m + kFindRows - 1) / kFindRows), dim3(kBlock), 0, stream, a.m, a.long_row, a.row_ptr,
                       c, reinterpret_cast<uint4*>(w + l.items), reinterpret_cast<uint4*>(w + l.rows), l.cap_items,
                       l.cap_rows, l.cap_slots);
    return &c->apart;
}

// Workgroups of the row kernel that cut pieces, the first of its grid: few, and the last pieces are cut when the rows are through,
// many, and the first rows wait for them.  A million power-law rows, 32 fp32 columns, us a call: 128 495, 256 406, 512 394, 1024 396,
// 2048 404.
constexpr uint32_t kCutBlocks = 512;

spmm_detail::BoundsWork spmm_long_bounds(const SpmmArgs& a, size_t value_bytes) {
    BoundsWork w = {0, {nullptr, 0, 0, 0, 0}, nullptr, nullptr, 0};
    const int64_t per_vector = static_cast<int64_t>(16 / value_bytes), vectors = (a.n + per_vector - 1) / per_vector;
    // op(B) beyond the L2s, two to kBandLanes lanes a row of it, and nonzeros enough to be worth cutting
    if (!a.b_row_major || a.n < per_vector || vectors < 2 || vectors > kBandLanes || !narrow_offsets(a, value_bytes) ||
        a.band_ws == nullptr || a.nnz < kBandLeastNonzeros || static_cast<uint64_t>(a.k) * a.n * value_bytes < kBandLeastBytes)
        return w;
    const LongLayout l = long_layout(a.nnz, a.long_n, value_bytes);
    char* ws = static_cast<char*>(a.long_ws);
    w.blocks = kCutBlocks;
    w.space.ws = a.band_ws;
    w.space.bytes = static_cast<uint64_t>(a.nnz) * sizeof(idx_t);
    w.space.k = a.k;
    w.space.row_bytes = static_cast<uint32_t>(vectors * 16);
    w.space.sum_bytes = static_cast<uint32_t>(l.ld_partials * value_bytes);
    w.counters = reinterpret_cast<LongCounters*>(ws + l.counters);
    w.items = reinterpret_cast<const uint4*>(ws + l.items);
    w.cap_items = l.cap_items;
    return w;
}

template <typename T>
void launch_spmm_long_rows(hipStream_t stream, const SpmmArgs& a, T alpha, T beta) {
    const LongLayout l = long_layout(a.nnz, a.long_n, sizeof(T));
    char* w = static_cast<char*>(a.long_ws);
    const LongCounters* c = reinterpret_cast<const LongCounters*>(w + l.counters);
    const uint4* items = reinterpret_cast<const uint4*>(w + l.items);
    const uint4* rows = reinterpret_cast<const uint4*>(w + l.rows);
    T* partials = reinterpret_cast<T*>(w + l.partials);
    const T* val = static_cast<const T*>(a.val);
    const T* B = static_cast<const T*>(a.B);
    T* C = static_cast<T*>(a.C);
    const int64_t b_rs = a.b_row_major ? a.ldb : 1;
    const int64_t b_cs = a.b_row_major ? 1 : a.ldb;
    constexpr int kWide = 16 / sizeof(T);
    const bool wide = a.b_row_major && a.n >= kWide;
    const uint32_t v = wide ? kWide : 1;
    const uint64_t lanes_needed = (static_cast<uint64_t>(a.n) + v - 1) / v;
    uint32_t lanes = 1;
    while (lanes < kWave && lanes < lanes_needed) lanes *= 2;
    const uint32_t panels = static_cast<uint32_t>((lanes_needed + lanes - 1) / lanes);
    // pieces are few (a 2048th of the nonzeros at most): a grid that lets every compute unit hold several
    static_assert(2048 % kBandStretches == 0, "workgroups of a launch");
    const dim3 grid(2048, panels);
    const uint32_t reduce_blocks = 1024;
    const BoundsWork work = spmm_long_bounds(a, sizeof(T));
    const BandSpace space = work.space;
    // (Two lanes to a row: in groups of four, half of them idle, where that way leads band by band; its gathers count, not its
    // lanes.  Power-law rows, pieces whole and in bands: 1.1 M, 6 fp32 columns 425 -> 315 us a call, 3.3 M, 4 fp64 columns 1478 -> 1087.)
    if (work.blocks != 0 && lanes < 4) lanes = 4;
    const bool stretched = wide && lanes >= 4 && narrow_offsets(a, sizeof(T));
    if (work.blocks != 0 && !a.long_cut) {
        BoundsWork whole_launch = work;
        whole_launch.blocks = 8192;
        hipLaunchKernelGGL(spmm_long_bounds_kernel, dim3(whole_launch.blocks), dim3(kBlock), 0, stream, whole_launch, a.base, a.nnz,
                           a.row_ptr, a.col);
    }
    auto stretches = [&](auto lr) {
        constexpr int LR = decltype(lr)::value;
        hipLaunchKernelGGL((spmm_long_stretch_kernel<T, LR, kWide>), grid, dim3(kBlock), 0, stream, a.n, a.base, a.row_ptr, a.col, val, B, a.ldb, C, a.ldc, a.c_row_major, alpha, beta, c, items, l.cap_items,
                           partials, l.ld_partials, a.nnz, space);
    };
    if (stretched) {
        if (lanes == 4) stretches(std::integral_constant<int, 4>{});
        else if (lanes == 8) stretches(std::integral_constant<int, 8>{});
        else if (lanes == 16) stretches(std::integral_constant<int, 16>{});
        else if (lanes == 32) stretches(std::integral_constant<int, 32>{});
        else stretches(std::integral_constant<int, 64>{});
    } else if (wide) {
        hipLaunchKernelGGL((spmm_long_chunk_kernel<T, kWide>), grid, dim3(kBlock), 0, stream, a.n, a.base, lanes,
                           a.row_ptr, a.col, val, B, b_rs, b_cs, C, a.ldc, a.c_row_major, alpha, beta, c, items,
                           l.cap_items, partials, l.ld_partials, a.nnz);
    } else {
        hipLaunchKernelGGL((spmm_long_chunk_kernel<T, 1>), grid, dim3(kBlock), 0, stream, a.n, a.base, lanes, a.row_ptr,
                           a.col, val, B, b_rs, b_cs, C, a.ldc, a.c_row_major, alpha, beta, c, items, l.cap_items,
                           partials, l.ld_partials, a.nnz);
    }
    if (wide) {
        hipLaunchKernelGGL((spmm_long_reduce_kernel<T, kWide>), dim3(reduce_blocks), dim3(kBlock), 0, stream, a.n, C,
                           a.ldc, a.c_row_major, alpha, beta, c, rows, l.cap_rows, partials, l.ld_partials, items, l.cap_items,
                           space);
    } else {
        hipLaunchKernelGGL((spmm_long_reduce_kernel<T, 1>), dim3(reduce_blocks), dim3(kBlock), 0, stream, a.n, C, a.ldc,
                           a.c_row_major, alpha, beta, c, rows, l.cap_rows, partials, l.ld_partials, items, l.cap_items,
                           space);
    }
}

template void launch_spmm_long_rows<float>(hipStream_t, const SpmmArgs&, float, float);
template void launch_spmm_long_rows<double>(hipStream_t, const SpmmArgs&, double, double);

}  // namespace mcsp
