// Building blocks of the kernels that partition entries by the bits of a key and read the parts back: partition.hip,
// spmv_transposed.hip.
#ifndef MCSPARSE_AMD_PARTITION_DEVICE_H_
#define MCSPARSE_AMD_PARTITION_DEVICE_H_

#include "device_util.h"
#include "internal.h"

namespace mcsp {
namespace partition_detail {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// ---- one wavefront ---------------------------------------------------------------------------------------------
// How many of the ascending values a[0 .. n) are <= g, with 64 probes per round.  Every lane of the wavefront must
// call this; all lanes return the same value.
__device__ __forceinline__ uint32_t wave_count_up_to(const uint32_t* __restrict__ a, uint32_t n, uint32_t base, uint32_t g) {
    uint64_t lo = 0, hi = n;
    const unsigned lane = lane_id();
    while (lo < hi) {
        const uint64_t step = (hi - lo + kWave - 1) / kWave;
        const uint64_t probe = lo + lane * step;
        const bool pred = probe < hi && a[probe] - base <= g;
        const unsigned count = __popcll(__ballot(pred));
        if (count == 0) {
            hi = lo;
        } else {
            const uint64_t new_hi = lo + static_cast<uint64_t>(count) * step;
            lo = lo + static_cast<uint64_t>(count - 1) * step + 1;
            hi = new_hi < hi ? new_hi : hi;
        }
    }
    return static_cast<uint32_t>(lo);
}

// lanes below this one among the bits of a 64-bit word
__device__ __forceinline__ uint32_t bits_below_lane(uint32_t lo, uint32_t hi) {
    return __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
}

// Clears, in the word (lo, hi) of candidate lanes, those whose digit differs from this lane's: per bit of the digit
// the lanes that voted as this lane did stay.  a & ~(b ^ c) is one v_bitop3 each for the low and the high half, so a
// bit costs four instructions.
template <int MAX_BITS>
__device__ __forceinline__ void keep_equal_digits(uint32_t d, uint32_t bits, uint32_t& lo, uint32_t& hi) {
#pragma unroll
    for (uint32_t b = 0; b < MAX_BITS; ++b) {
        if (b < bits) {
            const int own = __builtin_amdgcn_sbfe(static_cast<int>(d), b, 1);
            const uint64_t vote = __ballot(own < 0);
            lo = __builtin_amdgcn_bitop3_b32(lo, static_cast<uint32_t>(vote), static_cast<uint32_t>(own), 0x90);
            hi = __builtin_amdgcn_bitop3_b32(hi, static_cast<uint32_t>(vote >> 32), static_cast<uint32_t>(own), 0x90);
        }
    }
}

// Waits until this wavefront's stores have reached the L2.  A barrier does not (the L1 keeps a workgroup's accesses in
// order, so the compiler asks for no wait there): what all wavefronts have written can be released to other workgroups by
// one of them only if each has waited so before the barrier.
__device__ __forceinline__ void wait_for_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// ---- one workgroup ---------------------------------------------------------------------------------------------
// Exclusive sum over the threads of a workgroup; s_wave: THREADS / 64 words.  Holds one barrier; s_wave may be reused
// after the caller's next barrier.
template <int THREADS>
__device__ __forceinline__ uint32_t block_exclusive_sum(uint32_t v, uint32_t* s_wave, uint32_t* total = nullptr) {
    const uint32_t wave = threadIdx.x / kWave;
    const uint32_t upto = wave_inclusive_sum(v);
    if (threadIdx.x % kWave == kWave - 1) s_wave[wave] = upto;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (uint32_t w = 0; w < THREADS / kWave; ++w) {
        const uint32_t s = s_wave[w];
        if (w < wave) before += s;
        all += s;
    }
    if (total != nullptr) *total = all;
    return before + upto - v;
}

// Position inside the tile of a thread's i-th entry: wavefronts own consecutive slabs of `items` times 64 entries
// and the lanes are interleaved inside a slab, so (wavefront, i, lane) order is the order of the entries.
__device__ __forceinline__ uint32_t slab_place(uint32_t items, uint32_t i) {
    return (threadIdx.x / kWave * items + i) * kWave + threadIdx.x % kWave;
}
// slab_place(items, i) < count, as one comparison with a scalar.
__device__ __forceinline__ bool in_slab(uint32_t items, uint32_t i, uint32_t count) {
    return static_cast<int>(slab_place(items, 0)) < static_cast<int>(count) - static_cast<int>(i * kWave);
}

// array[index] for arrays of less than 4 GiB: a scalar base and a 32-bit offset.
template <typename W>
__device__ __forceinline__ W load_at(const void* array, uint32_t index) {
    return *reinterpret_cast<const W*>(static_cast<const char*>(array) + index * static_cast<uint32_t>(sizeof(W)));
}

// Reads of a tile of an array through a buffer resource that ends with the tile: places past the end read as zero
// without a test, and a thread's items differ by constants only.  A place, its constant part included, goes into the
// offset operand, which the hardware compares with the resource's length (constants below 4096 bytes travel in the
// instruction, larger ones cost an addition for every 4096 bytes); the scalar offset operand is no part of that
// comparison and stays zero.
struct TileReader {
    __amdgpu_buffer_rsrc_t tile;
    __device__ __forceinline__ TileReader(const void* first, uint32_t bytes) {
        constexpr int kRawDwords = 0x00027000;  // no stride, untyped
        tile = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(first), 0, static_cast<int>(bytes), kRawDwords);
    }
    template <typename W>
    __device__ __forceinline__ W read(uint32_t place, uint32_t constant_places) const {
        constexpr int kNonTemporal = 2;
        const int offset = static_cast<int>((place + constant_places) * sizeof(W));
        if constexpr (sizeof(W) == 4) {
            return __builtin_amdgcn_raw_buffer_load_b32(tile, offset, 0, kNonTemporal);
        } else {
            typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
            return __builtin_bit_cast(W, static_cast<u32x2>(__builtin_amdgcn_raw_buffer_load_b64(tile, offset, 0, kNonTemporal)));
        }
    }
};

// Stable rank of every entry among the entries of its wavefront with the same digit, two 16-bit ranks to a word;
// s_cnt[wave][digit] ends as the wavefront's count of the digit (zero on entry).  digit(i) is the digit of entry i;
// entries from `count` on are left out.
template <int ITEMS, int MAX_BITS, typename Digit>
__device__ __forceinline__ void rank_entries(uint32_t count, uint32_t bits, uint16_t* s_cnt,
                                             uint32_t (&rank)[(ITEMS + 1) / 2], Digit digit) {
    uint16_t* mine = s_cnt + (threadIdx.x / kWave << MAX_BITS);
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        uint32_t r = 0;
        const uint32_t d = digit(i);
        const bool live = in_slab(ITEMS, i, count);
        const uint64_t candidates = __ballot(live);
        uint32_t lo = static_cast<uint32_t>(candidates), hi = static_cast<uint32_t>(candidates >> 32);
        keep_equal_digits<MAX_BITS>(d, bits, lo, hi);
        const uint32_t below = bits_below_lane(lo, hi);
        if (live) {
            // Every peer reads the counter, then the lowest one adds the round's count.  The LDS operations of a
            // wavefront complete in program order; relaxed atomics keep the compiler from moving or merging them.
            const uint32_t before = __hip_atomic_load(mine + d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            r = before + below;
            if (below == 0) {
                __hip_atomic_store(mine + d, static_cast<uint16_t>(before + __popc(lo) + __popc(hi)), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WAVEFRONT);
            }
        }
        if (i % 2 == 0) rank[i / 2] = r;
        else rank[i / 2] |= r << 16;
        if (i % 2 != 0) forget(rank[i / 2]);  // (else the halves stay apart, in a register each, until they are used)
    }
}

// Ranks in no particular order, for callers that do not care how the entries of a digit follow each other: one LDS
// counter per digit (zero on entry) hands them out.  A quarter of the instructions of rank_entries.  Entries sorted by
// key (a long row) bring whole wavefronts of one digit, whose adds LDS would take one after the other: one lane adds
// for all of them.
template <int ITEMS, typename Digit>
__device__ __forceinline__ void rank_entries_unordered(uint32_t count, uint32_t* s_count, uint32_t (&rank)[(ITEMS + 1) / 2],
                                                       Digit digit) {
    const uint32_t lane = threadIdx.x % kWave;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t d = digit(i);
        const bool live = in_slab(ITEMS, i, count);
        const uint32_t lead = __builtin_amdgcn_readfirstlane(d);
        uint32_t r = 0;
        if (__all(live && d == lead)) {
            if (lane == 0) r = atomicAdd(&s_count[lead], static_cast<uint32_t>(kWave));
            r = __builtin_amdgcn_readfirstlane(r) + lane;
        } else if (live) {
            r = atomicAdd(&s_count[d], 1u);
        }
        if (i % 2 == 0) rank[i / 2] = r;
        else rank[i / 2] |= r << 16;
    }
}

// After rank_entries and a barrier: turns the counts of the wavefronts into the first place of each (wavefront, digit)
// in the ordered tile.  per_digit(digit, first place, count) is called once for every digit below 2^bits.  Ends with
// a barrier.
template <int THREADS, int MAX_BITS, typename PerDigit>
__device__ __forceinline__ void place_digits(uint32_t bits, uint16_t* s_cnt, uint32_t* s_wave, PerDigit per_digit) {
    constexpr int kWaves = THREADS / kWave;
    constexpr int kDigits = (1 << MAX_BITS) > THREADS ? (1 << MAX_BITS) / THREADS : 1;  // neighbouring digits per thread
    const uint32_t first = threadIdx.x * kDigits;
    uint32_t total[kDigits], sum = 0;
#pragma unroll
    for (int k = 0; k < kDigits; ++k) {
        total[k] = 0;
        if (first + k < (1u << MAX_BITS)) {
            uint32_t c[kWaves];
#pragma unroll
            for (int w = 0; w < kWaves; ++w) c[w] = s_cnt[(w << MAX_BITS) + first + k];
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                s_cnt[(w << MAX_BITS) + first + k] = static_cast<uint16_t>(total[k]);
                total[k] += c[w];
            }
        }
        sum += total[k];
    }
    uint32_t at = block_exclusive_sum<THREADS>(sum, s_wave);
#pragma unroll
    for (int k = 0; k < kDigits; ++k) {
        if (first + k < (1u << bits)) {
#pragma unroll
            for (int w = 0; w < kWaves; ++w) s_cnt[(w << MAX_BITS) + first + k] += static_cast<uint16_t>(at);
            per_digit(first + k, at, total[k]);
        }
        at += total[k];
    }
    __syncthreads();
}

// ---- runs of tiles ---------------------------------------------------------------------------------------------
// The entries of one bucket, in order, are the runs that its digit has in tiles 0, 1, ...: run t is `begins[t]` ..
// of them (ascending; the next run's begin, or `all`, ends it) and lies at place start(table[t]) of tile t.  A table
// word holds the run's place in the tile and its length.
__device__ __forceinline__ uint32_t table_word(uint32_t place, uint32_t length) { return place | length << 16; }
__device__ __forceinline__ uint32_t run_place(uint32_t word) { return word & 0xffffu; }
__device__ __forceinline__ uint32_t run_length(uint32_t word) { return word >> 16; }

// Where the entries q0 .. q0 + count - 1 of a bucket come from.  The runs they touch are listed in LDS, each as the
// difference between an entry's place in memory and its place in the chunk, and a bit marks where a run begins; the
// run of an entry is then a count of bits.
template <int CHUNK>
struct RunMap {
    unsigned long long begins[CHUNK / kWave];
    uint32_t before[CHUNK / kWave];  // runs that begin before each 64 entries, less one, the first entry's own included
    uint32_t wave[16];
};
// The last run of a bucket that begins at or before entry q0, found by search; for whole wavefronts.
__device__ __forceinline__ uint32_t find_first_run(const uint32_t* __restrict__ run_begins, uint32_t tiles, uint32_t q0) {
    const uint32_t upto = wave_count_up_to(run_begins, tiles, 0, q0);
    return upto != 0 ? upto - 1 : 0;
}

// first_run: the last run that begins at or before q0 (earlier ones will do).
template <int THREADS, int CHUNK>
__device__ __forceinline__ void map_runs(const uint32_t* __restrict__ run_begins, const uint32_t* __restrict__ table,
                                         uint32_t tiles, uint32_t all, uint32_t q0, uint32_t count, uint32_t first_run,
                                         uint32_t tile_stride, uint32_t source, RunMap<CHUNK>& s, uint32_t* s_delta) {
    constexpr uint32_t kWords = CHUNK / kWave;
    const uint32_t tid = threadIdx.x;
    for (uint32_t w = tid; w < kWords; w += THREADS) s.begins[w] = 0;
    __syncthreads();
    const uint32_t q1 = q0 + count;
    uint32_t listed = 0;
    for (uint32_t t0 = first_run; t0 < tiles; t0 += THREADS) {
        const uint32_t t = t0 + tid;
        uint32_t begin = all, end = all, word = 0;
        if (t < tiles) {
            begin = run_begins[t];
            end = t + 1 < tiles ? run_begins[t + 1] : all;
            word = table[t];
        }
        const uint32_t from = begin > q0 ? begin : q0;
        const uint32_t to = end < q1 ? end : q1;
        const bool used = from < to;
        uint32_t fresh = 0;
        const uint32_t at = listed + block_exclusive_sum<THREADS>(used ? 1u : 0u, s.wave, &fresh);
        if (used) {
            const uint32_t place = from - q0;
            if (at < static_cast<uint32_t>(CHUNK)) s_delta[at] = source + t * tile_stride + run_place(word) + (from - begin) - place;
            atomicOr(&s.begins[place / kWave], 1ull << (place % kWave));
        }
        listed += fresh;
        if (t0 + THREADS >= tiles) break;  // whole workgroup
        // past the chunk's end?  the last thread's run is the furthest
        if (!__syncthreads_or(tid == THREADS - 1 && end < q1)) break;  // whole workgroup
    }
    __syncthreads();
    if (tid < kWave) {
        uint32_t carried = 0;
        for (uint32_t w0 = 0; w0 < kWords; w0 += kWave) {
            const uint32_t w = w0 + tid;
            const unsigned long long word = w < kWords ? s.begins[w] : 0;
            const uint32_t c = __popcll(word);
            const uint32_t upto = wave_inclusive_sum(c);
            if (w < kWords) s.before[w] = carried + upto - c + static_cast<uint32_t>(word & 1u) - 1;
            carried += __shfl(upto, kWave - 1, kWave);
        }
    }
    __syncthreads();
}

// Place in memory of entry w * 64 + lane of a chunk of `count` entries (of the last one, for lanes past it).
template <int CHUNK>
__device__ __forceinline__ uint32_t mapped_place(const RunMap<CHUNK>& s, const uint32_t* s_delta, uint32_t w, uint32_t count) {
    const unsigned long long later = s.begins[w] >> 1;  // runs that begin at or before a lane, after the first lane
    const uint32_t run = s.before[w] + bits_below_lane(static_cast<uint32_t>(later), static_cast<uint32_t>(later >> 32));
    // (no run begins behind the last entry: lanes past it have found that entry's run)
    return s_delta[run] + min(w * kWave + threadIdx.x % kWave, count - 1);
}

// ---- stores of an ordered tile ---------------------------------------------------------------------------------
// Entries go to LDS in their new order and out as 16-byte pieces, `PLACES` of them (the tile and what its runs are
// padded with).  Every one of these begins and ends with the workgroup through with the buffer.
template <int ITEMS, int THREADS, uint32_t PLACES, typename Key>
__device__ __forceinline__ void store_keys(uint32_t* s_buf, uint32_t count, const uint32_t (&dest)[(ITEMS + 1) / 2], Key* out,
                                           const uint32_t (&key)[ITEMS], uint32_t mask) {
    Key* s = reinterpret_cast<Key*>(s_buf);
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if (in_slab(ITEMS, i, count)) s[(dest[i / 2] >> (i % 2 * 16)) & 0xffffu] = static_cast<Key>(key[i] & mask);
    }
    __syncthreads();
    static_assert(PLACES * sizeof(Key) % 16 == 0, "whole pieces");
    for (uint32_t v = threadIdx.x; v < PLACES * sizeof(Key) / 16; v += THREADS)
        __builtin_nontemporal_store(reinterpret_cast<const u32x4*>(s_buf)[v], reinterpret_cast<u32x4*>(out) + v);
    __syncthreads();
}

template <int ITEMS, int THREADS, uint32_t PLACES>
__device__ __forceinline__ void store_words(uint32_t* s_buf, uint32_t count, const uint32_t (&dest)[(ITEMS + 1) / 2],
                                            uint32_t* out, const uint32_t (&word)[ITEMS]) {
    constexpr uint32_t kPieces = PLACES / 4;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if (in_slab(ITEMS, i, count)) s_buf[(dest[i / 2] >> (i % 2 * 16)) & 0xffffu] = word[i];
    }
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < (kPieces + THREADS - 1) / THREADS; ++k) {
        const uint32_t v = k * THREADS + threadIdx.x;
        if (kPieces % THREADS == 0 || v < kPieces)
            __builtin_nontemporal_store(reinterpret_cast<const u32x4*>(s_buf)[v], reinterpret_cast<u32x4*>(out) + v);
    }
    __syncthreads();
}

// 64-bit words, word_of(half, i) being the lower and the upper half of entry i's, go through the buffer in two halves.  A
// thread has two words of a store to itself, so that a wavefront's store is one stretch (four, as two stores of 16 bytes a
// 32-byte stride apart: twice the requests to L2).
template <int ITEMS, int THREADS, uint32_t PLACES, typename WordOfHalf>
__device__ __forceinline__ void store_halves(uint32_t* s_buf, uint32_t count, const uint32_t (&dest)[(ITEMS + 1) / 2],
                                             uint64_t* out, WordOfHalf word_of) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    constexpr uint32_t kPieces = PLACES / 2;
    constexpr uint32_t kMine = (kPieces + THREADS - 1) / THREADS;
    u32x2 low[kMine];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            if (in_slab(ITEMS, i, count)) s_buf[(dest[i / 2] >> (i % 2 * 16)) & 0xffffu] = word_of(half, i);
        }
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < kMine; ++k) {
            const uint32_t v = k * THREADS + threadIdx.x;
            if (kPieces % THREADS != 0 && v >= kPieces) continue;
            const u32x2 got = reinterpret_cast<const u32x2*>(s_buf)[v];
            if (half == 0) {
                low[k] = got;
            } else {
                const u32x4 piece = {low[k].x, got.x, low[k].y, got.y};
                __builtin_nontemporal_store(piece, reinterpret_cast<u32x4*>(out) + v);
            }
        }
        __syncthreads();
    }
}
template <int ITEMS, int THREADS, uint32_t PLACES>
__device__ __forceinline__ void store_words(uint32_t* s_buf, uint32_t count, const uint32_t (&dest)[(ITEMS + 1) / 2],
                                            uint64_t* out, const uint64_t (&word)[ITEMS]) {
    store_halves<ITEMS, THREADS, PLACES>(s_buf, count, dest, out,
                                         [&](int half, int i) { return static_cast<uint32_t>(word[i] >> (32 * half)); });
}

// ---- packed entries --------------------------------------------------------------------------------------------
// Where what is left of an entry's key and its index share a word (Key = uint32_t), the entries are an array of such words
// and one of values, or, with 32-bit values, one of {word, value} pairs.
template <typename Key>
constexpr bool packed_entries() { return sizeof(Key) == 4; }
template <int VB>
__device__ __forceinline__ void load_packed(const void* words, const void* vals, uint32_t at, uint32_t& word,
                                            typename WordOf<VB>::type& val) {
    if constexpr (VB == 4) {
        const uint64_t pair = load_at<uint64_t>(words, at);
        word = static_cast<uint32_t>(pair);
        val = static_cast<uint32_t>(pair >> 32);
    } else {
        word = load_at<uint32_t>(words, at);
        if constexpr (VB != 0) val = load_at<uint64_t>(vals, at);
    }
}
template <int VB, int ITEMS, int THREADS, uint32_t PLACES, typename WordOfEntry, typename Values>
__device__ __forceinline__ void store_packed(uint32_t* s_buf, uint32_t count, const uint32_t (&dest)[(ITEMS + 1) / 2],
                                             void* words, void* vals, uint64_t out, WordOfEntry word_of, const Values& val) {
    if constexpr (VB == 4) {
        store_halves<ITEMS, THREADS, PLACES>(s_buf, count, dest, static_cast<uint64_t*>(words) + out,
                                             [&](int half, int i) { return half == 0 ? word_of(i) : val[i]; });
    } else {
        uint32_t word[ITEMS];
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) word[i] = word_of(i);
        store_words<ITEMS, THREADS, PLACES>(s_buf, count, dest, static_cast<uint32_t*>(words) + out, word);
        if constexpr (VB != 0) store_words<ITEMS, THREADS, PLACES>(s_buf, count, dest, static_cast<uint64_t*>(vals) + out, val);
    }
}

}  // namespace partition_detail
}  // namespace mcsp

#endif  // MCSPARSE_AMD_PARTITION_DEVICE_H_
