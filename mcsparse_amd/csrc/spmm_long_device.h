// Long rows taken apart (spmm_long.hip): what is known of them, and the cutting of their pieces where their columns pass from
// one band of op(B) to the next, which the row kernel of such matrices (spmm.hip) does beside its own rows.
#ifndef MCSPARSE_AMD_SPMM_LONG_DEVICE_H_
#define MCSPARSE_AMD_SPMM_LONG_DEVICE_H_

#include "spmm_device.h"

namespace mcsp {
namespace spmm_detail {

struct LongCounters {
    // the pieces listed; rows of several pieces << 32 | the pieces of those.  (Adds to one line take their turns, 5 ns each,
    // whichever counters they are for: three for each of 1024 workgroups were the time of the find kernel on 4 M rows, 17 us.)
    uint32_t items;
    unsigned long long several;
    __device__ uint32_t rows() const { return static_cast<uint32_t>(several >> 32); }
    // not zero: the listed rows are taken apart, since there is one of more than kSpmmLongRow nonzeros (on a line of its
    // own: a store among the adds to the counters makes the find kernel wait, 16.5 -> 27.5 us on a million rows)
    alignas(128) uint32_t apart;
    uint32_t unsorted;  // not zero: a piece whose columns do not ascend
};
static_assert(sizeof(LongCounters) <= 2 * kAlign, "what the layout has room for");

// ---- bands of op(B) --------------------------------------------------------------------------------------------
// The long rows of a matrix name every row of op(B) many times (a million power-law rows: 20 times), but a piece walks all of
// op(B), so each time it comes from behind the L2s.  Where op(B) is larger than they are, the pieces are taken band by band: a
// band is a stretch of rows of op(B) that fits an L2, an XCD works on every eighth band, and a wavefront takes the
// nonzeros that one piece has in one band, which lie side by side where columns ascend.  Their sum is a row of partial sums,
// added up per row in the order of pieces and bands.  Whether and how is decided on the device, from the number of pieces
// found, so that every way to a product comes to the same sums.
// A million power-law rows, 32 fp32 columns (20 M of 28 M nonzeros in rows of more than 256), microseconds: pieces whole 327,
// band by band 225 and 30 for the bounds (10 beside the row kernel), 560 -> 501 a call; 16 columns 520 -> 457; 3 M rows, 20 columns 1942 -> 1443; 400 K
// rows, 11 fp64 columns 258 -> 227.  Half of the rows of op(B) still come from behind the L2 (its wavefronts are not all in
// one band); bands of 2 MB bring that down to a quarter and the nonzeros of a pair to 32, half a round: 524.  Bands of 8 MB:
// 549.  Rows of op(B) wider than a panel of kBandLanes lanes keep their pieces whole: A's long rows would be read once per
// panel (100 fp32 columns: 1763 us whole, 2740 in panels).
constexpr uint64_t kBandBytes = size_t(4) << 20;  // of op(B)
constexpr uint32_t kBandStretches = 8;            // bands are dealt to so many XCDs
constexpr idx_t kBandLeastNonzeros = 1u << 20;
// (of 10 to 16 MB: 416 K rows and 5 fp64 columns 157 -> 140 us, 176 K and 17 fp32 columns 106 -> 100; of 6 to 10 MB 2 to 5 % slower
// as often as faster)
constexpr uint64_t kBandLeastBytes = size_t(10) << 20;
constexpr int kBandLanes = 8;
struct BandSpace {
    void* ws;            // null: no room, or no need
    uint64_t bytes;
    idx_t k;             // rows of op(B)
    uint32_t row_bytes, sum_bytes;  // of a row of op(B), and of a row of partial sums
};
// The pairs of a stretch are taken off kBandQueues counters, kBandTake at a time, every queue each kBandQueues-th take: adds to one
// address take their turns, some 14 ns each with all wavefronts of an XCD at it.  One counter, takes of 2, 4, 8 and 16 pairs: 622,
// 487, 457 and 475 us a call (a million rows, 32 fp32 columns, when the rest of it took 27 us more); 4 counters, takes of 2, 4, 8: 402,
// 401, 410 against 433; 8 counters 398, 398; 16 counters 397, 397.  3 M rows, 22 columns: 1464; 16 counters, takes of 2 and 4: 1458, 1417.
constexpr uint32_t kBandTake = 4;
constexpr uint32_t kBandQueues = 16;
struct BandPlan {
    uint32_t bands, items;  // 0 bands: pieces are taken whole
    uint32_t* taken;        // [stretch][queue], a line each: takes of kBandTake (band, item) pairs so far
    uint32_t* bounds;       // [item][band]: the item's first nonzero in that band or a later one; and behind the last band
    void* sums;             // [item][band]
    float of_column;        // band = column times this (whatever the rounding: it ascends with the column)
};
__device__ __forceinline__ BandPlan band_plan(const BandSpace& s, const LongCounters* __restrict__ c, uint32_t cap_items) {
    BandPlan p = {0, 0, nullptr, nullptr, nullptr, 0.0f};
    if (s.ws == nullptr || c->apart == 0 || c->unsorted != 0) return p;
    p.items = min(c->items, cap_items);
    if (p.items == 0) return p;
    const uint64_t wanted = (static_cast<uint64_t>(s.k) * s.row_bytes + kBandBytes - 1) / kBandBytes;
    uint64_t bands = (wanted + kBandStretches - 1) / kBandStretches * kBandStretches;
    auto bounds_bytes = [&](uint64_t n) { return (p.items * (n + 1) * sizeof(uint32_t) + kAlign - 1) / kAlign * kAlign; };
    constexpr uint64_t kTakenBytes = kBandStretches * kBandQueues * kAlign;
    while (bands != 0 && kTakenBytes + bounds_bytes(bands) + bands * p.items * s.sum_bytes > s.bytes) bands -= kBandStretches;
    if (2 * bands < wanted) return p;  // (bands of twice the size still keep half of their rows)
    p.bands = static_cast<uint32_t>(bands);
    p.taken = static_cast<uint32_t*>(s.ws);
    p.bounds = p.taken + kTakenBytes / sizeof(uint32_t);
    p.sums = reinterpret_cast<char*>(p.bounds) + bounds_bytes(bands);
    p.of_column = static_cast<float>(bands) / static_cast<float>(s.k);
    return p;
}

// The bounds of every item, by the first `blocks` workgroups of a launch, an item at a time.
struct BoundsWork {
    uint32_t blocks;  // 0: none
    BandSpace space;
    LongCounters* counters;
    const uint4* items;
    uint32_t cap_items;
};
__device__ __forceinline__ void cut_pieces(const BoundsWork& w, idx_t base, idx_t nnz, const idx_t* __restrict__ row_ptr,
                                           const idx_t* __restrict__ col) {
    const BandPlan plan = band_plan(w.space, w.counters, w.cap_items);  // (a workgroup that sees another's `unsorted` may stop early)
    if (plan.bands == 0) return;  // whole workgroup
    constexpr int kAtOnce = 2, kQuad = 4;
    typedef idx_t quad_t __attribute__((ext_vector_type(kQuad)));
    typedef quad_t element_aligned __attribute__((aligned(sizeof(idx_t))));
    static_assert(kBandStretches * kBandQueues <= kBlock, "a thread per counter");
    if (blockIdx.x == 0 && threadIdx.x < kBandStretches * kBandQueues) plan.taken[threadIdx.x * (kAlign / sizeof(uint32_t))] = 0;
    auto band_of = [&](idx_t column) {
        return min(static_cast<uint32_t>(static_cast<float>(column - base) * plan.of_column), plan.bands - 1);
    };
    for (uint32_t it = blockIdx.x; it < plan.items; it += w.blocks) {
        const uint4 item = w.items[it];
        uint32_t* bounds = plan.bounds + static_cast<uint64_t>(it) * (plan.bands + 1);
        const idx_t row_end = min(row_ptr[item.x + 1] - base, nnz);
        const idx_t start = min(row_ptr[item.x] - base + item.y * kSpmmLongChunk, row_end);
        const idx_t end = item.z != 0 ? min(start + static_cast<idx_t>(kSpmmLongChunk), row_end) : start;
        if (start == end) {  // whole workgroup: a row that found no room
            for (uint32_t b = threadIdx.x; b <= plan.bands; b += kBlock) bounds[b] = start;
            continue;
        }
        bool unsorted = false;
        // neighbouring nonzeros by fours to a thread: the one before its first is the thread's before
        for (idx_t j0 = start + threadIdx.x * kQuad; j0 < end; j0 += kBlock * kQuad * kAtOnce) {
            quad_t here[kAtOnce];
            idx_t before[kAtOnce];
#pragma unroll
            for (int u = 0; u < kAtOnce; ++u) {
                const idx_t j = j0 + u * kBlock * kQuad;
                if (j + kQuad <= end) {
                    here[u] = *reinterpret_cast<const element_aligned*>(col + j);
                } else {
#pragma unroll
                    for (int q = 0; q < kQuad; ++q) here[u][q] = col[min(j + q, end - 1)];
                }
                before[u] = col[min(j, end) - (j != start ? 1 : 0)];
            }
#pragma unroll
            for (int u = 0; u < kAtOnce; ++u) {
                idx_t last = before[u];
                uint32_t last_band = band_of(last);
#pragma unroll
                for (int q = 0; q < kQuad; ++q) {
                    const idx_t j = j0 + u * kBlock * kQuad + q;
                    if (j >= end) break;
                    unsorted |= here[u][q] < last;
                    const uint32_t band = band_of(here[u][q]);
                    for (uint32_t b = j == start ? 0 : last_band + 1; b <= band; ++b) bounds[b] = j;
                    if (j == end - 1) {
                        for (uint32_t b = band + 1; b <= plan.bands; ++b) bounds[b] = end;
                    }
                    last = here[u][q];
                    last_band = band;
                }
            }
        }
        if (unsorted) w.counters->unsorted = 1;
    }
}

}  // namespace spmm_detail
// What is to be cut for a call, once spmm_long_find_kernel has run; blocks = 0: its pieces are taken whole.
spmm_detail::BoundsWork spmm_long_bounds(const SpmmArgs& a, size_t value_bytes);
}  // namespace mcsp

#endif  // MCSPARSE_AMD_SPMM_LONG_DEVICE_H_
