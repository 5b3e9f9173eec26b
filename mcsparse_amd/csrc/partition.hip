// Partition of entries by bits of a key, tile by tile, and the stable sort by key made of it, for gfx950.
//
// partition_kernel orders the entries of a tile by a digit of their keys, inside the tile only, and writes the tile back
// as one linear stream, with a table of where each digit's run begins.  Against a radix pass that writes every entry
// straight to its bucket (src/mcprim/device_radix_sort.hpp:90-309 of the reference) it needs no counting pass and makes
// no scattered store; the runs are put together by whoever reads them next.
//
// The sort orders (key, index, value) triples by a key of up to 24 bits: csr2csc
// (src/kernels/conversion/mcsp_csr2csc.cpp:97-98 of the reference) and the index sorts.  A stable sort has one result,
// so how it is reached is free.  What bounds it is the bytes its passes move; an LSD sort moves every triple whole, keys
// included, once per 8 bits and reads the keys once more per pass.  Here the most significant bits go first:
//   1. partition_kernel, by the top d1 bits;
//   2. where more than 2^11 buckets are wanted, repartition_kernel: the same on the tiles of each bucket, whose entries
//      it gathers from the runs of step 1, by the next d2 bits;
//   3. bucket_sort_kernel gathers a bucket, which fits LDS, orders it by the last d3 bits and writes it where it belongs,
//      a linear stream again.  Where the keys begin (col_ptr of a CSC) falls out of its digit counts.
// A key loses the bits that its place already tells: at most 16 of them travel to step 2, 8 or 16 to step 3.
// A sort by two keys (the index sorts) partitions by the major key alone: step 3 orders a bucket by the minor key first,
// then by what is left of the major one, in passes of up to eight bits that stay in LDS.  Where the two have room in one
// word (sort_packs) it is the words that are ordered.
// Buckets that do not fit LDS (popular keys) are sorted in chunks by oversize_kernel, which finds nothing to do elsewhere;
// inputs that would make such buckets only (few keys) are left to the LSD passes.
#include "partition_device.h"
#include "sort_shape.h"

#include <algorithm>

namespace mcsp {

namespace {

using namespace partition_detail;
using namespace sort_detail;

// ---- step 1 ----------------------------------------------------------------------------------------------------
// What the entries of a sort are.  CSR: `aux` holds the m + 1 row offsets (index base `base`) of a matrix whose
// nonzeros are the entries, and an entry's index is its row + base.
struct EntrySource {
    const uint32_t* keys;
    const uint32_t* aux;
    const void* vals;
    const void* x;         // products: the value that travels is value * x[row], and no index does
    uint32_t count;
    uint32_t key_bias;     // subtracted from a key before its bits are taken
    uint32_t m, base;
    const uint32_t* tile_rows;  // CSR: rows that begin at or before each tile's first nonzero
    // CSR, packed entries: the index is counted from the tile's first row; a tile with more rows than the word has room for
    // leaves its indices in an array of their own and sets *wide
    bool relative;
    uint32_t* wide;
    uint32_t minor_bits;  // plain, packed entries: bits of the index, which lies below the key's rest
    ColumnBuckets columns;  // products
};

// The order of tiles over the workgroups: an XCD takes a contiguous range, so the table words of neighbouring tiles,
// which share lines, meet in one L2.
__device__ __forceinline__ uint32_t tile_of_block(uint32_t tiles, uint32_t xcds) {
    const uint32_t per_xcd = (tiles + xcds - 1) / xcds;
    return (blockIdx.x % xcds) * per_xcd + blockIdx.x / xcds;
}

// The order of buckets over the workgroups: XCDs take kNeighbours in turn or, if `range` is not 0, that many each.  (A contiguous
// range of them each, as for tiles, leaves XCDs without work where the number of keys is no power of two and the last buckets are
// empty, or where the keys are not evenly spread: 22 M nonzeros in 1.2 M columns, a call of csr2csc 325 us, and 269 in turn; 11.5 M
// in 700 K 168 and 151; index sort of 10 M triples in 2^20 rows 280 and 216.  Neighbours meet on the lines at the ends of their
// runs, for which 2, 4, 8 and 16 of them do: 270, 269, 269, 269, and 60, 59, 59, 59 for 4 M nonzeros in 300 K columns, 68 before.)
constexpr uint32_t kNeighbours = 8;
// Few entries stay in the L2s from one step to the next.  A range of the buckets that have keys then finds in its own XCD's L2
// what the tiles of that part of a banded matrix left there: csr2csc of a million nonzeros in 65536 columns 29.4 us, in turn
// 31.9 (fp64 31.4 and 35.1), in 80 K columns 29.5 and 31.8 (fp64 33.3 and 35.6), of 1.4 M in 200 K 36.2 and 38.9.  Nonzeros from
// everywhere lose up to 3 % by it (33.5 and 32.4 us in 65536 columns).  2.4 M in 2^18 columns 46.9 and 47.6 (fp64 55.1 and 54.7;
// power-law columns 105 and 102), 3.5 M in 2^17 48.1 and 47.7.
constexpr uint32_t kEntriesThatStay = 1u << 21;
__device__ __forceinline__ uint32_t bucket_of_block(uint32_t range, uint32_t xcds) {
    const uint32_t turn = blockIdx.x / xcds, xcd = blockIdx.x - turn * xcds;
    if (range != 0) return turn < range ? xcd * range + turn : blockIdx.x;
    return turn / kNeighbours * kNeighbours * xcds + xcd * kNeighbours + turn % kNeighbours;
}

enum EntryKind : int { kPlain = 0, kCsr = 1, kProducts = 2 };
// Runs of products are padded with zeros to a multiple of kBucketRunPad entries, so that they can be read in pieces of
// that many.
constexpr uint32_t run_pad(int kind) { return kind == kProducts ? kBucketRunPad : 1; }
// Places a tile takes in memory once its 2^bits runs are padded.
constexpr uint32_t tile_places(uint32_t tile_size, int kind, uint32_t bits) { return tile_size + ((run_pad(kind) - 1) << bits); }

// The rows of a tile's nonzeros, without a load per nonzero: a bit marks every nonzero at which a row begins, and the
// row of a nonzero is the first row of the tile plus the bits at or before it.  Two rows that begin at one nonzero (an
// empty row) cannot be told from the bits: then the row starts, staged in LDS or in memory, are searched.
template <uint32_t TILE>
struct TileRows {
    unsigned long long begins[TILE / kWave];
    uint32_t before[TILE / kWave];
    uint32_t empty_rows;
};

// zero: before the barrier in front of mark_rows
template <int THREADS, uint32_t TILE>
__device__ __forceinline__ void clear_rows(TileRows<TILE>& s) {
    for (uint32_t i = threadIdx.x; i < TILE / kWave; i += THREADS) s.begins[i] = 0;
    if (threadIdx.x == 0) s.empty_rows = 0;
}
// at: the row starts of the tile, relative to it, as loaded by start_of_row (thread after thread, item after item)
template <int ITEMS, int THREADS>
__device__ __forceinline__ void mark_rows(TileRows<ITEMS * THREADS>& s, uint32_t* s_starts, uint32_t inside,
                                          uint32_t tile_first, const uint32_t (&start)[ITEMS]) {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t j = i * THREADS + threadIdx.x;
        if (j < inside) {
            const uint32_t at = start[i] - tile_first;
            s_starts[j] = at;
            if (at < static_cast<uint32_t>(ITEMS * THREADS)) {  // the tile's last row may end where the next tile begins
                const unsigned long long bit = 1ull << (at % kWave);
                if ((atomicOr(&s.begins[at / kWave], bit) & bit) != 0) s.empty_rows = 1;
            }
        }
    }
}
// the running count of the bits, by the first wavefront; a barrier on either side
template <uint32_t TILE>
__device__ __forceinline__ void count_rows(TileRows<TILE>& s) {
    if (threadIdx.x < kWave) {
        uint32_t carried = 0;
        for (uint32_t w0 = 0; w0 < TILE / kWave; w0 += kWave) {
            const uint32_t w = w0 + threadIdx.x;
            const uint32_t c = w < TILE / kWave ? __popcll(s.begins[w]) : 0;
            const uint32_t upto = wave_inclusive_sum(c);
            if (w < TILE / kWave) s.before[w] = carried + upto - c;
            carried += __shfl(upto, kWave - 1, kWave);
        }
    }
}

// A workgroup per tile.  Key: the type the rest of a key travels in.  Products: the digit is the bucket of ColumnBuckets.
//
// Bounds at 118 M entries (the products of a transposing SpMV, fp32): 0.98 GB read and 0.79 GB written in 340 us, nine
// tenths of the rate of a copy; tiles of 4096 or 16 wavefronts per workgroup are no faster (342 and 420 us).  The pass
// it replaces took 486 us, with a pass over the keys (111 us) in front of it to count them.  The first step of csr2csc
// (16 bytes per entry, the ranks by ballots): 1.9 GB in 350 us.
template <int VB, int KIND, int MAX_BITS, typename Key, int THREADS, int ITEMS>
__global__ __launch_bounds__(THREADS) void partition_kernel(EntrySource in, uint32_t shift, uint32_t bits, uint32_t tiles,
                                                               Key* __restrict__ keys_out, uint32_t* __restrict__ aux_out,
                                                               void* __restrict__ vals_out, uint32_t* __restrict__ table,
                                                               uint32_t xcds) {
    constexpr uint32_t kTile = THREADS * ITEMS;
    constexpr uint32_t kPad = run_pad(KIND);
    constexpr uint32_t kPlaces = tile_places(kTile, KIND, MAX_BITS);
    constexpr int kWaves = THREADS / kWave;
    constexpr bool kOrdered = KIND != kProducts;  // products: the entries of a digit may follow each other in any order
    typedef typename WordOf<VB>::type word_t;
    // plain: the counts' place is the words' afterwards (nothing is staged before)
    constexpr uint32_t kCounts = kOrdered ? kWaves << MAX_BITS : 2 << MAX_BITS;
    constexpr bool kOnePlace = KIND == kPlain;
    __shared__ __align__(16) uint32_t s_buf[kOnePlace && kCounts / 2 > kPlaces ? kCounts / 2 : kPlaces];
    __shared__ __align__(16) uint16_t s_apart[kOnePlace ? 8 : kCounts];
    uint16_t* const s_cnt = kOnePlace ? reinterpret_cast<uint16_t*>(s_buf) : s_apart;
    __shared__ uint32_t s_wave[kWaves];
    __shared__ TileRows<KIND != kPlain ? kTile : kWave> s_rows;

    const uint32_t tile = tile_of_block(tiles, xcds);
    if (tile >= tiles) return;  // whole workgroup
    const uint32_t tid = threadIdx.x;
    const uint64_t first = static_cast<uint64_t>(tile) * kTile;
    const uint32_t count = in.count - first < kTile ? static_cast<uint32_t>(in.count - first) : kTile;
    const uint32_t slab = slab_place(ITEMS, 0);

    uint32_t key[ITEMS], aux[ITEMS];
    word_t val[VB ? ITEMS : 1];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) key[i] = TileReader(in.keys + first, count * 4).read<uint32_t>(slab, i * kWave);
    uint32_t before = 0, inside = 0;
    bool staged = false;
    if constexpr (KIND != kPlain) {
        before = in.tile_rows[tile];
        inside = in.tile_rows[tile + 1] - before;
        staged = inside <= kTile;
        // (the row starts are in aux for the time being)
        const TileReader starts(in.aux + (before - 1), (min(inside, kTile) + 1) * 4);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) aux[i] = starts.read<uint32_t>(tid, i * THREADS + 1);
        clear_rows<THREADS>(s_rows);
    }
    // (64-bit values are asked for once the ranks are there: held through the ranking they cost the second workgroup
    // of a compute unit)
    constexpr bool kValuesEarly = VB == 4;
    auto load_values = [&]() {
        const word_t* vals_in = static_cast<const word_t*>(in.vals);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) val[i] = TileReader(vals_in + first, count * VB).template read<word_t>(slab, i * kWave);
    };
    if constexpr (kValuesEarly) load_values();
    for (uint32_t i = tid; i < kCounts / 8; i += THREADS) reinterpret_cast<u32x4*>(s_cnt)[i] = u32x4(0);
    __syncthreads();

    const uint32_t mask = (1u << bits) - 1u;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        key[i] -= in.key_bias;
        // the bucket above the column's low half, and no bucket but those that exist, whatever the column
        if constexpr (!kOrdered) key[i] = min(bucket_of(in.columns, key[i]), mask) << 16 | (key[i] & 0xffffu);
    }
    auto digit = [&](int i) { return kOrdered ? (key[i] >> shift) & mask : key[i] >> 16; };
    uint32_t dest[(ITEMS + 1) / 2];
    constexpr int kDigits = (1 << MAX_BITS) > THREADS ? (1 << MAX_BITS) / THREADS : 1;  // products: neighbouring digits of a thread
    uint32_t pad_from[kDigits], pad_to[kDigits];  // what they leave open behind their runs
    uint32_t* const s_count = reinterpret_cast<uint32_t*>(s_cnt);
    if constexpr (kOrdered) rank_entries<ITEMS, MAX_BITS>(count, bits, s_cnt, dest, digit);
    else rank_entries_unordered<ITEMS>(count, s_count, dest, digit);
    if constexpr (KIND != kPlain) {
        if (staged) mark_rows<ITEMS, THREADS>(s_rows, s_buf, inside, static_cast<uint32_t>(first) + in.base, aux);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) forget(key[i]);
    if constexpr (KIND != kPlain) count_rows(s_rows);
    if constexpr (kOrdered) {
        place_digits<THREADS, MAX_BITS>(bits, s_cnt, s_wave, [&](uint32_t d, uint32_t at, uint32_t n) {
            table[static_cast<uint64_t>(d) * tiles + tile] = table_word(at, n);
        });
    } else {
        uint32_t n[kDigits], padded[kDigits], sum = 0;
#pragma unroll
        for (int k = 0; k < kDigits; ++k) {
            const uint32_t d = tid * kDigits + k;
            n[k] = d < (1u << MAX_BITS) ? s_count[d] : 0;
            padded[k] = (n[k] + kPad - 1) / kPad * kPad;
            sum += padded[k];
        }
        uint32_t at = block_exclusive_sum<THREADS>(sum, s_wave);
#pragma unroll
        for (int k = 0; k < kDigits; ++k) {
            const uint32_t d = tid * kDigits + k;
            if (d < (1u << MAX_BITS)) {
                s_count[d] = at;
                if (d < (1u << bits)) table[static_cast<uint64_t>(d) * tiles + tile] = table_word(at, padded[k]);
            }
            pad_from[k] = at + n[k];
            at += padded[k];
            pad_to[k] = at;
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t at = kOrdered ? s_cnt[(tid / kWave << MAX_BITS) + digit(i)] : s_count[digit(i)];
        dest[i / 2] += at << (i % 2 * 16);
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) forget(key[i]);

    if constexpr (kOnePlace) __syncthreads();  // the counts have been read
    if constexpr (KIND == kPlain) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) aux[i] = TileReader(in.aux + first, count * 4).read<uint32_t>(slab, i * kWave);
    } else if (staged && s_rows.empty_rows == 0) {  // the same for the workgroup
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t w = tid / kWave * ITEMS + i;
            const unsigned long long word = s_rows.begins[w];
            const uint32_t upto = bits_below_lane(static_cast<uint32_t>(word), static_cast<uint32_t>(word >> 32)) +
                                  static_cast<uint32_t>((word >> (tid % kWave)) & 1u);
            aux[i] = before - 1 + s_rows.before[w] + upto;
        }
    } else {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t p = slab_place(ITEMS, i);
            uint32_t lo = 0, hi = inside;
            while (lo < hi) {
                const uint32_t mid = (lo + hi) >> 1;
                const uint32_t at = staged ? s_buf[mid] : in.aux[before + mid] - static_cast<uint32_t>(first) - in.base;
                if (at <= p) lo = mid + 1; else hi = mid;
            }
            aux[i] = before - 1 + lo;
        }
        __syncthreads();  // the staged starts have been read
    }
    if constexpr (VB != 0 && !kValuesEarly) load_values();
    const uint64_t out = static_cast<uint64_t>(tile) * kPlaces;
    if constexpr (packed_entries<Key>()) {
        static_assert(KIND != kProducts, "no index travels with a product");
        uint32_t origin = 0u - in.base;
        if (KIND == kCsr && in.relative) {  // (shift != 0: there is a second step)
            origin = before - 1;
            if (inside >> (32 - shift) != 0) {  // whole workgroup
#pragma unroll
                for (int i = 0; i < ITEMS; ++i) aux[i] += in.base;
                store_words<ITEMS, THREADS, kPlaces>(s_buf, count, dest, aux_out + out, aux);
                if (tid == 0) *in.wide = 1;
            }
        }
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t rest = key[i] & ((1u << shift) - 1u);
            // (a minor key that is out of range must not reach the bits above it)
            key[i] = KIND == kCsr ? rest | (aux[i] - origin) << shift
                                  : rest << in.minor_bits | (aux[i] & ((1u << in.minor_bits) - 1u));
            forget(key[i]);
        }
        store_packed<VB, ITEMS, THREADS, kPlaces>(s_buf, count, dest, keys_out, vals_out, out, [&](int i) { return key[i]; }, val);
        return;
    }
    store_keys<ITEMS, THREADS, kPlaces>(s_buf, count, dest, keys_out + out, key, kOrdered ? (1u << shift) - 1u : 0xffffu);
    if constexpr (KIND == kProducts) {
        typedef typename RealOf<VB>::type real_t;
        const real_t* x = static_cast<const real_t*>(in.x);
        constexpr int kAhead = ITEMS / 2;  // gathers in flight: all of them at once cost a wavefront per SIMD in registers
#pragma unroll
        for (int i0 = 0; i0 < ITEMS; i0 += kAhead) {
            real_t xr[kAhead];
#pragma unroll
            for (int i = 0; i < kAhead; ++i) xr[i] = x[in_slab(ITEMS, i0 + i, count) ? aux[i0 + i] : before - 1];
#pragma unroll
            for (int i = 0; i < kAhead; ++i)
                val[i0 + i] = __builtin_bit_cast(word_t, __builtin_bit_cast(real_t, val[i0 + i]) * xr[i]);
            __builtin_amdgcn_sched_barrier(0);
        }
        // (a product of 0 and whatever key lies beside it: both halves of a 64-bit zero are the same word)
#pragma unroll
        for (int k = 0; k < kDigits; ++k) {
            for (uint32_t p = pad_from[k]; p < pad_to[k]; ++p) s_buf[p] = 0;
        }
    } else {
        if constexpr (KIND == kCsr) {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) aux[i] += in.base;
        }
        store_words<ITEMS, THREADS, kPlaces>(s_buf, count, dest, aux_out + out, aux);
    }
    if constexpr (VB != 0) store_words<ITEMS, THREADS, kPlaces>(s_buf, count, dest, static_cast<word_t*>(vals_out) + out, val);
}

// tile_rows[t] = number of rows that begin at or before the first nonzero of tile t (t = tiles: all m + 1 offsets).
constexpr int kRowStartsBlock = 256;
__global__ __launch_bounds__(kRowStartsBlock) void partition_row_starts_kernel(const uint32_t* __restrict__ row_ptr,
                                                                               uint32_t m, uint32_t base, uint32_t nnz,
                                                                               uint32_t tile_size, uint32_t tiles,
                                                                               uint32_t* __restrict__ tile_rows,
                                                                               uint32_t* __restrict__ wide) {
    const uint32_t t = blockIdx.x * (kRowStartsBlock / kWave) + threadIdx.x / kWave;
    if (wide != nullptr && blockIdx.x == 0 && threadIdx.x == 0) *wide = 0;
    if (t > tiles) return;  // whole wavefront
    const uint64_t first = static_cast<uint64_t>(t) * tile_size;
    // (m + 1 < 2^32: the reference's limit on extents)
    const uint32_t starts = wave_count_up_to(row_ptr, m + 1, base, first < nnz ? static_cast<uint32_t>(first) : nnz);
    if (threadIdx.x % kWave == 0) tile_rows[t] = starts;
}

// run_begins[d * tiles + t] = entries of digit d in the tiles before t; totals[d] = all of them.  A workgroup per digit.
// first_runs (may be null), [d][first_stride]: for the entries q * kSecondTile of the digit the run they lie in.
// A wavefront has ITEMS * 64 tiles a round, neighbouring lanes neighbouring ones: bound by latency and by how many lines
// its reads and stores touch.  With a few neighbouring tiles a thread 256 digits of 14,400 tiles took 22.5 us and 2048 of 888
// 9.7; so 11.3 and 5.7.
template <int BLOCK, int ITEMS>
__global__ __launch_bounds__(BLOCK) void run_begins_kernel(uint32_t tiles, const uint32_t* __restrict__ table,
                                                           uint32_t* __restrict__ run_begins, uint32_t* __restrict__ totals,
                                                           uint32_t* __restrict__ first_runs, uint32_t first_stride) {
    __shared__ uint32_t s_wave[BLOCK / kWave];
    const uint32_t* in = table + static_cast<uint64_t>(blockIdx.x) * tiles;
    uint32_t* out = run_begins + static_cast<uint64_t>(blockIdx.x) * tiles;
    const uint32_t wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    uint32_t carried = 0;
    for (uint32_t t0 = 0; t0 < tiles; t0 += BLOCK * ITEMS) {
        const uint32_t first = t0 + wave * (ITEMS * kWave) + lane;
        uint32_t n[ITEMS], at[ITEMS], in_wave = 0;
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) n[k] = in[min(first + k * kWave, tiles - 1)];
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            n[k] = first + k * kWave < tiles ? run_length(n[k]) : 0;
            const uint32_t upto = wave_inclusive_sum(n[k]);
            at[k] = in_wave + upto - n[k];
            in_wave += __builtin_amdgcn_readlane(upto, kWave - 1);
        }
        if (lane == 0) s_wave[wave] = in_wave;
        __syncthreads();
        uint32_t before = carried;
#pragma unroll
        for (uint32_t w = 0; w < BLOCK / kWave; ++w) {
            const uint32_t sum = s_wave[w];
            if (w < wave) before += sum;
            carried += sum;
        }
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            const uint32_t t = first + k * kWave, begin = before + at[k];
            if (t < tiles) out[t] = begin;
            if (first_runs != nullptr && n[k] != 0) {  // (a run is no longer than a tile)
                for (uint32_t q = (begin + kSecondTile - 1) / kSecondTile; q * kSecondTile < begin + n[k]; ++q)
                    first_runs[static_cast<uint64_t>(blockIdx.x) * first_stride + q] = t;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = carried;
}

// ---- between workgroups of one launch --------------------------------------------------------------------------
// An XCD's L2 does not see what another XCD writes: what workgroups of a launch hand to each other goes past the caches on
// both sides.  (An L2 written back by each of its workgroups at the end of a phase: 70 us a phase.)
template <typename W>
__device__ __forceinline__ W load_shared(const W* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename W>
__device__ __forceinline__ void store_shared(W* p, W v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The same at array[index], for arrays of less than 4 GiB: a scalar base and a 32-bit offset.
template <typename W>
__device__ __forceinline__ W load_shared_at(const void* array, uint32_t index) {
    return load_shared(reinterpret_cast<const W*>(static_cast<const char*>(array) + index * static_cast<uint32_t>(sizeof(W))));
}
template <typename W>
__device__ __forceinline__ void store_at(void* array, uint32_t index, W v) {
    *reinterpret_cast<W*>(static_cast<char*>(array) + index * static_cast<uint32_t>(sizeof(W))) = v;
}
template <typename W>
__device__ __forceinline__ void store_shared_at(void* array, uint32_t index, W v) {
    store_shared(reinterpret_cast<W*>(static_cast<char*>(array) + index * static_cast<uint32_t>(sizeof(W))), v);
}
// One more of `all` has come: was it the last?  For the whole workgroup; whoever comes last may load_shared what the others
// have written with store_shared.
__device__ __forceinline__ bool last_to_arrive(uint32_t* counter, uint32_t all, uint32_t* s_last) {
    wait_for_stores();
    __syncthreads();
    if (threadIdx.x == 0)
        *s_last = (__hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1) % all == 0;
    __syncthreads();
    return *s_last != 0;
}

// ---- step 2 ----------------------------------------------------------------------------------------------------
// What the kernels after step 1 read of it and of each other.  One level: the buckets of step 1 are sorted as they are.
// Two levels: tile t of bucket b (its entries [t * kSecondTile, ...)) is tile number tile_first[b] + t.
struct SortTables {
    // step 1: [digit][tile]
    const uint32_t* table1;
    const uint32_t* begins1;
    const uint32_t* totals1;
    uint32_t tiles1, places1;
    // step 2: [bucket][digit][tile of the bucket]
    uint32_t* table2;
    uint32_t* begins2;
    uint32_t* bucket_first;  // entries before each bucket of step 1, 2^d1 + 1 of them
    uint32_t* tile_first;    // tiles before each bucket of step 1, 2^d1 + 1 of them
    const uint32_t* first_runs;  // [bucket][first_stride]: the run of step 1 in which each of its tiles begins
    uint32_t first_stride;       // tiles of step 2 that one bucket can have
    // step 1, packed entries: rows that begin at or before each tile's first entry, less one and the index base; whether
    // there are tiles whose indices lie in an array of their own
    const uint32_t* tile_rows;
    const uint32_t* wide;
    uint32_t tile1_shift, base;  // log2 of the places of a tile of step 1
    uint2* tile_map;         // the order in which the tiles are taken: {bucket << 24 | tile of the bucket, its first run}
    // both: entries before each bucket of step 3, 2^(d1 + d2) + 1 of them
    uint32_t* sub_first;
    uint32_t* sub_arrived;  // workgroups that are through with a bucket of step 1
    // buckets of step 3 that do not fit LDS, in the order in which they were listed
    struct OversizeState* oversize;
    uint32_t* oversize_bucket;
    uint32_t* oversize_first;     // chunks of the buckets before
    uint32_t* oversize_counted;   // groups of chunks that have been counted, over all passes
    uint32_t* oversize_arrived;   // [group]: chunks of it that have been counted, over all passes
    uint32_t* oversize_counts;    // [chunk][digit]
    uint32_t* oversize_begins;    // [group][digit]
    uint32_t* oversize_aux[2];    // where the passes over such a bucket leave its entries in between
    void* oversize_vals[2];
    uint16_t* oversize_keys[2];
    uint32_t oversize_passes, oversize_width;  // passes of so many bits over the minor and the major key together
    uint32_t d1, d2, d3, count;
    // step 3: `minor_passes` passes of minor_width bits (the last one: what is left) over the minor_bits of aux, then
    // passes of key_width bits over the d3 bits of the keys
    uint32_t minor_bits, minor_passes, minor_width, key_width, passes;
};
struct SortPass {
    bool on_aux;
    uint32_t shift, bits;
};
__device__ __forceinline__ SortPass sort_pass(const SortTables& t, uint32_t p) {
    SortPass s;
    s.on_aux = p < t.minor_passes;
    s.shift = s.on_aux ? p * t.minor_width : (p - t.minor_passes) * t.key_width;
    s.bits = s.on_aux ? min(t.minor_width, t.minor_bits - s.shift) : min(t.key_width, t.d3 - s.shift);
    return s;
}

// The same over the words of packed pairs.
__device__ __forceinline__ SortPass word_pass(const SortTables& t, uint32_t p) {
    const uint32_t shift = p * t.oversize_width;
    return {false, shift, min(t.oversize_width, t.minor_bits + t.d3 - shift)};
}

// A bucket that does not fit LDS is sorted in chunks, by passes of up to kPassBits over the bits that are left of its
// keys.  A pass has two phases: the digits of the chunks are counted, then the chunks are written where they belong.
constexpr uint32_t kOversizeChunk = kBucketRoom;
constexpr uint32_t kOversizeGroup = 16;  // chunks whose counts are added up together
constexpr uint32_t kMaxOversizePhases = 10;  // of 24 bits of the minor key and 16 of the major one
struct OversizeState {
    unsigned long long listed;  // buckets | chunks << 32
    // chunks of a phase that somebody works on or has done, and that are done; on lines of their own, since idle
    // workgroups keep reading `done`
    alignas(128) uint32_t taken[kMaxOversizePhases];
    alignas(128) uint32_t done[kMaxOversizePhases];
};
// The groups of a listed bucket are numbered from here on (a bucket has at most chunks / kOversizeGroup + 1 of them).
__device__ __forceinline__ uint32_t oversize_slot(uint32_t first, uint32_t listed_at) { return first / kOversizeGroup + listed_at; }
__device__ __forceinline__ void note_oversize(const SortTables& t, uint32_t bucket, uint32_t entries) {
    if (entries <= kBucketRoom) return;
    const uint32_t chunks = (entries + kOversizeChunk - 1) / kOversizeChunk;
    const unsigned long long at = atomicAdd(&t.oversize->listed, static_cast<unsigned long long>(chunks) << 32 | 1u);
    const uint32_t k = static_cast<uint32_t>(at), first = static_cast<uint32_t>(at >> 32);
    t.oversize_bucket[k] = bucket;
    t.oversize_first[k] = first;
    t.oversize_counted[k] = 0;
    const uint32_t groups = (chunks + kOversizeGroup - 1) / kOversizeGroup;
    for (uint32_t g = 0; g < groups; ++g) t.oversize_arrived[oversize_slot(first, k) + g] = 0;
}

// Exclusive sums over the buckets of step 1 (at most 2^11), in one workgroup: of entries, and (two levels) of tiles.
// One level: the buckets of step 1 are those of step 3.
constexpr int kPlanBlock = 1024;
__global__ __launch_bounds__(kPlanBlock) void sort_plan_kernel(SortTables t) {
    __shared__ uint32_t s_wave[kPlanBlock / kWave];
    if (threadIdx.x == 0) {
        t.oversize->listed = 0;
        for (uint32_t p = 0; p < kMaxOversizePhases; ++p) t.oversize->taken[p] = t.oversize->done[p] = 0;
        __threadfence();  // before the adds of this workgroup's other threads
    }
    const uint32_t buckets = 1u << t.d1;
    uint32_t* first = t.d2 != 0 ? t.bucket_first : t.sub_first;
    uint32_t entries_before = 0, tiles_before = 0;
    __syncthreads();
    for (uint32_t b0 = 0; b0 < buckets; b0 += kPlanBlock) {
        const uint32_t b = b0 + threadIdx.x;
        const uint32_t n = b < buckets ? t.totals1[b] : 0;
        uint32_t all = 0;
        const uint32_t at = block_exclusive_sum<kPlanBlock>(n, s_wave, &all);
        if (b < buckets) first[b] = entries_before + at;
        entries_before += all;
        __syncthreads();
        if (t.d2 != 0) {
            const uint32_t tiles = (n + kSecondTile - 1) / kSecondTile;
            const uint32_t tile_at = block_exclusive_sum<kPlanBlock>(tiles, s_wave, &all);
            if (b < buckets) {
                t.tile_first[b] = tiles_before + tile_at;
                t.sub_arrived[b] = 0;
            }
            tiles_before += all;
            __syncthreads();
        } else if (b < buckets) {
            note_oversize(t, b, n);
        }
    }
    if (threadIdx.x == 0) {
        first[buckets] = entries_before;
        if (t.d2 != 0) t.tile_first[buckets] = tiles_before;
    }
}

// The order in which repartition_kernel takes its tiles: an eighth of the buckets at a time (what an XCD works on),
// inside it the first tiles of all buckets, then the second ones, ...  Tiles of the same number of neighbouring buckets
// read neighbouring runs of the same tiles of step 1 and meet on the lines at the ends of the runs.
constexpr int kMapBlock = 256;
__global__ __launch_bounds__(kMapBlock) void tile_map_kernel(SortTables t) {
    __shared__ uint32_t s_first[257];
    const uint32_t buckets = 1u << t.d1;  // at most 256
    for (uint32_t b = threadIdx.x; b <= buckets; b += kMapBlock) s_first[b] = t.tile_first[b];
    __syncthreads();
    const uint32_t q = blockIdx.x * kMapBlock + threadIdx.x;
    if (q >= s_first[buckets]) return;
    uint32_t lo = 0, hi = buckets;  // the bucket whose tile q is: the last one that begins at or before it
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (s_first[mid] <= q) lo = mid; else hi = mid;
    }
    const uint32_t tile = q - s_first[lo];
    const uint32_t group = buckets >= 8 ? buckets / 8 : 1;
    const uint32_t g0 = lo / group * group;
    uint32_t at = s_first[g0];
    for (uint32_t b = g0; b < g0 + group; ++b) {
        const uint32_t tiles = s_first[b + 1] - s_first[b];
        at += tiles < tile ? tiles : tile;
        if (b < lo && tiles > tile) ++at;
    }
    t.tile_map[at] = make_uint2(lo << 24 | tile, t.first_runs[static_cast<uint64_t>(lo) * t.first_stride + tile]);
}

// 118 M entries (16 bytes each): 0.99 GB read, 1.10 GB written in 415 us.
// Key: the type the rest of a key travels in from here on, or the packed entries' word (on both sides; PAIRS, a sort by two
// keys: only from here on).
template <int VB, typename Key, bool PAIRS>
__global__ __launch_bounds__(kSecondThreads) void repartition_kernel(SortTables t, const void* __restrict__ keys_in,
                                                                     const uint32_t* __restrict__ aux_in,
                                                                     const void* __restrict__ vals_in,
                                                                     Key* __restrict__ keys_out,
                                                                     uint32_t* __restrict__ aux_out,
                                                                     void* __restrict__ vals_out, uint32_t xcds) {
    constexpr int kWaves = kSecondThreads / kWave;
    constexpr int kMaxBits = 8;
    typedef typename WordOf<VB>::type word_t;
    __shared__ __align__(16) uint32_t s_buf[kSecondTile];
    __shared__ __align__(16) uint16_t s_cnt[kWaves << kMaxBits];
    __shared__ uint32_t s_wave[kWaves];
    __shared__ RunMap<kSecondTile> s_map;
    const uint32_t all_tiles = t.tile_first[1u << t.d1];  // at most as many as the grid has workgroups
    const uint32_t at = tile_of_block(all_tiles, xcds);
    if (at >= all_tiles || blockIdx.x / xcds >= (all_tiles + xcds - 1) / xcds) return;  // whole workgroup
    const uint2 mine = t.tile_map[at];
    const uint32_t bucket = mine.x >> 24, tile = mine.x & 0xffffffu;
    const uint32_t tid = threadIdx.x, wave = tid / kWave;
    const uint32_t all = t.totals1[bucket];
    const uint32_t q0 = tile * kSecondTile;
    const uint32_t count = min(all - q0, kSecondTile);
    for (uint32_t i = tid; i < sizeof(s_cnt) / 16; i += kSecondThreads) reinterpret_cast<u32x4*>(s_cnt)[i] = u32x4(0);
    const uint64_t row = static_cast<uint64_t>(bucket) * t.tiles1;
    map_runs<kSecondThreads, kSecondTile>(t.begins1 + row, t.table1 + row, t.tiles1, all, q0, count, mine.y, t.places1, 0, s_map,
                                          s_buf);
    constexpr bool kPacked = packed_entries<Key>() && !PAIRS;
    uint32_t key[kPacked ? 1 : kSecondItems], aux[kSecondItems];  // packed: aux is the word that goes on from here,
    uint32_t digits[kPacked ? (kSecondItems + 3) / 4 : 1];        // digits the bits of it this step sorts by
    word_t val[VB ? kSecondItems : 1];
    const uint32_t last_word = (count - 1) / kWave;
    // (past the last entry: some entry of the last runs, which is not used)
    uint32_t own_wave = wave;
    auto place_of = [&](int i) { return mapped_place(s_map, s_buf, min(own_wave * kSecondItems + i, last_word), count); };
    const uint32_t mask = (1u << t.d2) - 1u;
    if constexpr (kPacked) {
        const uint32_t rest_bits = t.d2 + t.d3, low_mask = (1u << t.d3) - 1u;
        uint32_t first_row[kSecondItems];
#pragma unroll
        for (int i = 0; i < kSecondItems; ++i) {
            const uint32_t from = place_of(i);
            load_packed<VB>(keys_in, vals_in, from, aux[i], val[VB ? i : 0]);
            first_row[i] = load_at<uint32_t>(t.tile_rows, from >> t.tile1_shift);  // the row the word counts from, plus one
            if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // (places of so many at a time are held in registers)
        }
        if (*t.wide != 0) {  // the same for all workgroups
            forget(own_wave);  // (places found again and not held in registers)
#pragma unroll
            for (int i = 0; i < kSecondItems; ++i) {
                const uint32_t from = place_of(i), tile1 = from >> t.tile1_shift;
                if ((t.tile_rows[tile1 + 1] - t.tile_rows[tile1]) >> (32 - rest_bits) != 0) {
                    first_row[i] = aux_in[from] - t.base + 1;
                    aux[i] &= (1u << rest_bits) - 1u;
                }
            }
        }
#pragma unroll
        for (int i = 0; i < kSecondItems; ++i) {
            const uint32_t word = aux[i], d = ((word >> t.d3) & mask) << (i % 4 * 8);
            if (i % 4 == 0) digits[i / 4] = d;
            else digits[i / 4] |= d;
            aux[i] = ((word >> rest_bits) + first_row[i] - 1 + t.base) << t.d3 | (word & low_mask);
            forget(aux[i]);
            if (i % 4 == 3) forget(digits[i / 4]);
        }
    } else {
#pragma unroll
        for (int i = 0; i < kSecondItems; ++i) {
            const uint32_t from = place_of(i);
            key[i] = load_at<uint16_t>(keys_in, from);
            aux[i] = load_at<uint32_t>(aux_in, from);
            if constexpr (VB != 0) val[i] = load_at<word_t>(vals_in, from);
        }
    }
    auto digit = [&](int i) {
        if constexpr (kPacked) return (digits[i / 4] >> (i % 4 * 8)) & 0xffu;
        else return (key[kPacked ? 0 : i] >> t.d3) & mask;
    };
    uint32_t dest[kSecondItems / 2];
    rank_entries<kSecondItems, kMaxBits>(count, t.d2, s_cnt, dest, digit);
    __syncthreads();
    const uint32_t first_tile = t.tile_first[bucket], tiles = t.tile_first[bucket + 1] - first_tile;
    uint32_t* table = t.table2 + (static_cast<uint64_t>(first_tile) << t.d2) + tile;
    place_digits<kSecondThreads, kMaxBits>(t.d2, s_cnt, s_wave, [&](uint32_t d, uint32_t place, uint32_t n) {
        table[static_cast<uint64_t>(d) * tiles] = table_word(place, n);
    });
#pragma unroll
    for (int i = 0; i < kSecondItems; ++i)
        dest[i / 2] += static_cast<uint32_t>(s_cnt[(wave << kMaxBits) + digit(i)]) << (i % 2 * 16);
    const uint64_t out = static_cast<uint64_t>(first_tile + tile) * kSecondTile;
    if constexpr (packed_entries<Key>()) {
        auto word_of = [&](int i) {
            if (kPacked) return aux[i];
            return (key[kPacked ? 0 : i] & ((1u << t.d3) - 1u)) << t.minor_bits | (aux[i] & ((1u << t.minor_bits) - 1u));
        };
        store_packed<VB, kSecondItems, kSecondThreads, kSecondTile>(s_buf, count, dest, keys_out, vals_out, out, word_of, val);
    } else {
        store_keys<kSecondItems, kSecondThreads, kSecondTile>(s_buf, count, dest, keys_out + out, key, (1u << t.d3) - 1u);
        store_words<kSecondItems, kSecondThreads, kSecondTile>(s_buf, count, dest, aux_out + out, aux);
        if constexpr (VB != 0)
            store_words<kSecondItems, kSecondThreads, kSecondTile>(s_buf, count, dest, static_cast<word_t*>(vals_out) + out, val);
    }
}

// begins2 and sub_first from table2; kSubParts workgroups per bucket of step 1, a wavefront per digit at a time, and
// whoever comes last says where the bucket's digits begin.  One workgroup per bucket and one round of 64 tiles in flight
// took 514 us where a bucket holds two thirds of 67 M entries (some 7000 tiles), now 96.
constexpr int kSubBlock = 256;
constexpr uint32_t kSubParts = 8;
__global__ __launch_bounds__(kSubBlock) void sub_begins_kernel(SortTables t) {
    __shared__ uint32_t s_wave[kSubBlock / kWave];
    __shared__ uint32_t s_last;
    constexpr uint32_t kAhead = 8;
    const uint32_t bucket = blockIdx.x / kSubParts, part = blockIdx.x % kSubParts, tid = threadIdx.x, lane = tid % kWave;
    const uint32_t digits = 1u << t.d2;  // at most 256
    const uint32_t first_tile = t.tile_first[bucket], tiles = t.tile_first[bucket + 1] - first_tile;
    const uint64_t row0 = static_cast<uint64_t>(first_tile) << t.d2;
    uint32_t* first = t.sub_first + (bucket << t.d2);
    for (uint32_t d = part * (kSubBlock / kWave) + tid / kWave; d < digits; d += kSubParts * (kSubBlock / kWave)) {
        const uint64_t row = row0 + static_cast<uint64_t>(d) * tiles;
        uint32_t carried = 0;
        for (uint32_t t0 = 0; t0 < tiles; t0 += kWave * kAhead) {
            uint32_t n[kAhead];
#pragma unroll
            for (uint32_t k = 0; k < kAhead; ++k) n[k] = t.table2[row + min(t0 + k * kWave + lane, tiles - 1)];
#pragma unroll
            for (uint32_t k = 0; k < kAhead; ++k) {
                const uint32_t at = t0 + k * kWave + lane;
                n[k] = at < tiles ? run_length(n[k]) : 0;
                const uint32_t upto = wave_inclusive_sum(n[k]);
                if (at < tiles) t.begins2[row + at] = carried + upto - n[k];
                carried += __builtin_amdgcn_readlane(upto, kWave - 1);
            }
        }
        if (lane == 0) store_shared(first + d, carried);
    }
    if (!last_to_arrive(t.sub_arrived + bucket, kSubParts, &s_last)) return;  // whole workgroup
    static_assert(kSubBlock == 256, "a thread per digit");
    const uint32_t n = tid < digits ? load_shared(first + tid) : 0;
    const uint32_t at = t.bucket_first[bucket] + block_exclusive_sum<kSubBlock>(n, s_wave);
    if (tid < digits) {
        first[tid] = at;
        note_oversize(t, (bucket << t.d2) + tid, n);
    }
    if (bucket == (1u << t.d1) - 1 && tid == 0) t.sub_first[1u << (t.d1 + t.d2)] = t.count;
}

// ---- step 3 ----------------------------------------------------------------------------------------------------
struct SortOutput {
    uint32_t* keys;    // may be null
    uint32_t* aux;
    void* vals;
    uint32_t* key_ptr; // may be null: where each of the `key_count` keys begins, + base, and the end
    uint32_t key_count, base, key_bias;
};

// Runs of a bucket of step 3.
struct BucketRuns {
    const uint32_t* begins;
    const uint32_t* table;
    uint32_t tiles, places, source;
};
__device__ __forceinline__ BucketRuns runs_of_bucket(const SortTables& t, uint32_t sub) {
    BucketRuns r;
    if (t.d2 == 0) {
        const uint64_t row = static_cast<uint64_t>(sub) * t.tiles1;
        r.begins = t.begins1 + row;
        r.table = t.table1 + row;
        r.tiles = t.tiles1;
        r.places = t.places1;
        r.source = 0;
    } else {
        const uint32_t bucket = sub >> t.d2, digit = sub & ((1u << t.d2) - 1u);
        const uint32_t first_tile = t.tile_first[bucket];
        r.tiles = t.tile_first[bucket + 1] - first_tile;
        const uint64_t row = (static_cast<uint64_t>(first_tile) << t.d2) + static_cast<uint64_t>(digit) * r.tiles;
        r.begins = t.begins2 + row;
        r.table = t.table2 + row;
        r.places = kSecondTile;
        r.source = first_tile * kSecondTile;
    }
    return r;
}

__device__ __forceinline__ void write_key_ptr(const SortOutput& out, uint32_t sub, uint32_t d3, uint32_t digit, uint32_t at,
                                              uint32_t count) {
    if (out.key_ptr == nullptr) return;
    const uint64_t key = (static_cast<uint64_t>(sub) << d3) + digit;
    if (key < out.key_count) out.key_ptr[key] = at + out.base;
    if (key + 1 == out.key_count) out.key_ptr[out.key_count] = count + out.base;
}

struct BucketLds {
    __align__(16) uint32_t buf[kBucketRoom];
    __align__(16) uint16_t cnt[kBucketThreads / kWave << kPassBits];
    uint32_t wave[kBucketThreads / kWave];
    uint16_t key_begin[(1 << kPassBits) + 1];  // first place of each key, for short runs of keys
    uint16_t long_run;                         // != 0: one of the runs is not short
    RunMap<kBucketRoom> map;
    __device__ __forceinline__ void clear_counts() {
        for (uint32_t i = threadIdx.x; i < sizeof(cnt) / 16; i += kBucketThreads) reinterpret_cast<u32x4*>(cnt)[i] = u32x4(0);
    }
};

// Entries with one major key (a row of a mesh's matrix: 16 triples) up to which the sort by the minor key is a count:
// ordered by the major key first, an entry looks at the minor keys of its run, which lie together in LDS and are read by
// neighbouring lanes together.  A pass of the radix sort costs an entry some 60 instructions, three of them as many as 40
// comparisons.  A bucket with a run of more than kShortRun goes on with the passes by minor and major key, which give the
// same order from any order that is stable in the major key; buckets whose mean run is above kUsualRun don't try.
// Assembly, all calls, with the radix passes alone and with this: 7.2 M triples of a mesh 219 -> 200 us; random triples,
// 2 a row (8 M) 452 -> 423, 16 a row (8 M) 423 -> 393; tried with 30 a row (12 M) 555 -> 562, with 60 a row 549 -> 580.
// Packed words: the first pass takes the eight upper bits of the word, also where more or fewer of them are the major key's,
// and entries are compared as words, four at a time from where the run's stretch of 16 bytes begins: the words of the runs
// around it compare as they should.  One bound serves four of them: words in front of an entry's own four go before it also
// if they are equal, those of its four are its neighbours' and are looked at there.  (With a bound for every word, 21
// instructions for four words and not 13, the assembly of the 7.2 M triples took 174 us, where it takes 168.)  (Tried
// wherever the minor key's upper bits may cut the runs short: bands of 216 and 400 triples a row 212 -> 252 and 306 -> 357
// us, for there they seldom do.)
constexpr uint32_t kShortRun = 64, kUsualRun = 20;

// place + how many of the four words are below the bound.  (The compiler waits for every comparison by itself and sends half
// of them through a register.)  An SGPR that a vector instruction has written may be read by another one, as its carry, two
// instructions later at the earliest: nobody else looks after that inside the block, so three stand between a comparison and its
// add, and no fewer than two may.
__device__ __forceinline__ uint32_t add_smaller(uint32_t place, u32x4 words, uint32_t bound) {
    uint64_t a, b, c, d;
    asm("v_cmp_lt_u32_e64 %1, %5, %9\n\t"
        "v_cmp_lt_u32_e64 %2, %6, %9\n\t"
        "v_cmp_lt_u32_e64 %3, %7, %9\n\t"
        "v_cmp_lt_u32_e64 %4, %8, %9\n\t"
        "v_addc_co_u32_e64 %0, %1, 0, %0, %1\n\t"
        "v_addc_co_u32_e64 %0, %2, 0, %0, %2\n\t"
        "v_addc_co_u32_e64 %0, %3, 0, %0, %3\n\t"
        "v_addc_co_u32_e64 %0, %4, 0, %0, %4"
        : "+v"(place), "=&s"(a), "=&s"(b), "=&s"(c), "=&s"(d)
        : "v"(words.x), "v"(words.y), "v"(words.z), "v"(words.w), "v"(bound));
    return place;
}

// How many of the lanes below this one in its four hold the same word.
__device__ __forceinline__ uint32_t equal_below_in_quad(uint32_t word) {
    const uint32_t lane = threadIdx.x % 4;
    const int w = static_cast<int>(word);
    const bool first = __builtin_amdgcn_update_dpp(0, w, 0x00, 0xF, 0xF, false) == w;
    const bool second = __builtin_amdgcn_update_dpp(0, w, 0x55, 0xF, 0xF, false) == w;
    const bool third = __builtin_amdgcn_update_dpp(0, w, 0xAA, 0xF, 0xF, false) == w;
    return (first && lane > 0 ? 1u : 0u) + (second && lane > 1 ? 1u : 0u) + (third && lane > 2 ? 1u : 0u);
}

// Sorts a bucket of at most ITEMS * kBucketThreads entries, the runs of which are mapped in LDS.  MANY: in several passes.
template <int VB, typename Key, bool MANY, int ITEMS>
__device__ __forceinline__ void sort_bucket(const SortTables& t, uint32_t sub, uint32_t first, uint32_t count,
                                            const Key* keys_in, const uint32_t* aux_in, const void* vals_in,
                                            const SortOutput& out, BucketLds& s) {
    typedef typename WordOf<VB>::type word_t;
    static_assert(!MANY || VB != 8, "64-bit values are sorted in one pass");
    const uint32_t tid = threadIdx.x, wave = tid / kWave;
    // (aux is then the whole word: the key's rest below the index, or, MANY, above it, so that words sort as pairs do)
    constexpr bool kPacked = packed_entries<Key>();
    uint32_t key[kPacked ? 1 : ITEMS], aux[ITEMS];
    word_t val[VB ? ITEMS : 1];
    const uint32_t last_word = (count - 1) / kWave;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t from = mapped_place(s.map, s.buf, min(wave * ITEMS + i, last_word), count);
        if constexpr (kPacked) {
            load_packed<VB>(keys_in, vals_in, from, aux[i], val[VB ? i : 0]);
        } else {
            key[i] = load_at<Key>(keys_in, from);
            aux[i] = load_at<uint32_t>(aux_in, from);
            if constexpr (VB != 0) val[i] = load_at<word_t>(vals_in, from);
        }
    }
    uint32_t dest[(ITEMS + 1) / 2];
    // into LDS in the new order
    auto ordered = [&](auto word_of) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            if (in_slab(ITEMS, i, count)) s.buf[(dest[i / 2] >> (i % 2 * 16)) & 0xffffu] = word_of(i);
        }
        __syncthreads();
    };
    // MANY: one pass by the key first (-1), packed: by the upper bits of the word, where its runs are likely to be short; see
    // kShortRun.
    const uint32_t upper = kPacked ? min(t.minor_bits + t.d3, kPassBits) : t.d3;
    const uint32_t below = kPacked ? t.minor_bits + t.d3 - upper : 0;
    const bool key_first = MANY && upper <= kPassBits && (kPacked ? t.oversize_passes > 2 : t.minor_passes > 1) &&
                           count <= kUsualRun << min(t.d3, kPassBits);
    for (int p = key_first ? -1 : 0;; ++p) {
        SortPass pass = {false, MANY ? below : 0u, MANY ? upper : t.d3};
        if (MANY && p >= 0) pass = kPacked ? word_pass(t, static_cast<uint32_t>(p)) : sort_pass(t, static_cast<uint32_t>(p));
        if (MANY && p < 0 && tid == 0) {
            s.long_run = 0;
            s.key_begin[1u << upper] = static_cast<uint16_t>(count);
        }
        const uint32_t mask = (1u << pass.bits) - 1u;
        auto digit = [&](int i) {
            const uint32_t of_aux = aux[i];  // (the values, so that neither array needs an address)
            if constexpr (kPacked) return (of_aux >> pass.shift) & mask;
            const uint32_t of_key = key[kPacked ? 0 : i];
            return MANY ? ((pass.on_aux ? of_aux : of_key) >> pass.shift) & mask : of_key;
        };
        rank_entries<ITEMS, kPassBits>(count, pass.bits, s.cnt, dest, digit);
        __syncthreads();
        if constexpr (MANY && kPacked) {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) forget(aux[i]);
        }
        place_digits<kBucketThreads, kPassBits>(pass.bits, s.cnt, s.wave, [&](uint32_t d, uint32_t at, uint32_t entries) {
            if (!MANY) {
                write_key_ptr(out, sub, t.d3, d, first + at, t.count);
            } else if (p < 0) {
                s.key_begin[d] = static_cast<uint16_t>(at);
                if (entries > kShortRun) s.long_run = 1;
            }
        });
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
            dest[i / 2] += static_cast<uint32_t>(s.cnt[(wave << kPassBits) + digit(i)]) << (i % 2 * 16);
        if constexpr (MANY && kPacked) {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) forget(aux[i]);
        }
        if (!MANY || p + 1 == static_cast<int>(kPacked ? t.oversize_passes : t.passes)) break;
        auto back = [&](uint32_t (&word)[ITEMS]) {
            ordered([&](int i) { return word[i]; });
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) word[i] = s.buf[slab_place(ITEMS, i)];
            __syncthreads();
        };
        if constexpr (MANY) {
            if constexpr (!kPacked) back(key);
            if constexpr (VB == 4) back(val);
            back(aux);
            if (kPacked && p < 0) {
                // (the words behind the last one are looked at too, and must not go in front of any)
                if (tid < 4 - count % 4 && count % 4 != 0) s.buf[count + tid] = ~0u;
                __syncthreads();
            }
            if (p < 0 && s.long_run == 0) {  // the same for the workgroup
                // buf still holds the minor keys in this order: an entry's place is that of its run, plus the entries
                // of the run that go before it
#pragma unroll
                for (int i = 0; i < ITEMS; ++i) {
                    const bool live = in_slab(ITEMS, i, count);
                    const uint32_t here = slab_place(ITEMS, i), mine = aux[i];
                    const uint32_t run = !live ? 0u : kPacked ? mine >> below : key[kPacked ? 0 : i] & mask;
                    uint32_t q = s.key_begin[run];
                    const uint32_t end = live ? s.key_begin[run + 1] : q;
                    uint32_t place = q;
                    if constexpr (kPacked) {
                        // (no word is all ones: see sort_packs)
                        // (of equal words those in front count: in front of this four by the bound, in it by the lanes below)
                        q &= ~3u;
                        uint32_t own = mine;
                        forget(own);  // (not all items' at the start, a register each)
                        place = q + equal_below_in_quad(own);
                        const uint32_t four = here & ~3u;
                        const u32x4* others = reinterpret_cast<const u32x4*>(&s.buf[q]);
                        for (; q < end; q += 4, ++others) place = add_smaller(place, *others, mine + (q < four ? 1u : 0u));
                    } else {
#pragma unroll 4
                        for (; q < end; ++q) {
                            const uint32_t other = s.buf[q];
                            place += other < mine || (other == mine && q < here);
                        }
                    }
                    if (i % 2 == 0) dest[i / 2] = place;
                    else dest[i / 2] |= place << 16;
                }
                __syncthreads();
                break;
            }
            s.clear_counts();
            __syncthreads();
        }
    }
    // every array out as a linear stream
    auto stream_out = [&](auto store) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t p = i * kBucketThreads + tid;
            if (p < count) store(i, p, s.buf[p]);
        }
        __syncthreads();
    };
    const uint32_t minor_mask = (1u << t.minor_bits) - 1u;
    ordered([&](int i) { return !kPacked ? aux[i] : MANY ? aux[i] & minor_mask : aux[i] >> t.d3; });
    stream_out([&](int, uint32_t p, uint32_t w) { out.aux[first + p] = w; });
    if constexpr (VB == 4) {
        ordered([&](int i) { return val[i]; });
        stream_out([&](int, uint32_t p, uint32_t w) { static_cast<uint32_t*>(out.vals)[first + p] = w; });
    } else if constexpr (VB == 8) {  // in two halves
        uint32_t low[ITEMS];
        ordered([&](int i) { return static_cast<uint32_t>(val[i]); });
        stream_out([&](int i, uint32_t, uint32_t w) { low[i] = w; });
        ordered([&](int i) { return static_cast<uint32_t>(val[i] >> 32); });
        stream_out([&](int i, uint32_t p, uint32_t w) {
            static_cast<uint64_t*>(out.vals)[first + p] = static_cast<uint64_t>(w) << 32 | low[i];
        });
    }
    if constexpr (MANY) {
        const uint32_t high = (sub << t.d3) + out.key_bias;
        ordered([&](int i) { return kPacked ? aux[i] >> t.minor_bits : key[kPacked ? 0 : i]; });
        stream_out([&](int, uint32_t p, uint32_t w) { out.keys[first + p] = high + w; });
    }
}

// A workgroup per bucket.  118 M entries (16 bytes each) in buckets of 3600: 390 us, bound by vector instructions as much
// as by memory; so most buckets, below two thirds of the room, run a version without the last third of the items (458 -> 445
// us when an entry was 17 bytes in three arrays).  Packed pairs: another one without the last quarter, for the buckets of a
// mean size (1.5 M rows, 6 M triples, all of the assembly: 274 -> 263 us), and 64 registers, so that a compute unit has four
// workgroups and not three (7.2 M triples of a mesh 181 -> 177, 2 M random ones 97 -> 93, 7.9 M 331 -> 322; with
// __syncthreads_or for long_run, which holds the thread's three numbers all along, six registers went to scratch memory: 180, 94,
// 326, and 0.6 M triples 52.8 -> 53.8, where it is 53.0 so).
template <int VB, typename Key, bool MANY>
__global__ __launch_bounds__(kBucketThreads, VB == 8 || (MANY && !packed_entries<Key>()) ? 6 : 8) void bucket_sort_kernel(SortTables t, const Key* __restrict__ keys_in,
                                                                                      const uint32_t* __restrict__ aux_in,
                                                                                      const void* __restrict__ vals_in,
                                                                                      SortOutput out, uint32_t buckets,
                                                                                      uint32_t range, uint32_t xcds) {
    constexpr int kUsualItems = kBucketItems * 2 / 3, kFewItems = kBucketItems / 3;
    constexpr int kMoreItems = MANY && packed_entries<Key>() ? kBucketItems * 3 / 4 : kUsualItems;
    __shared__ BucketLds s;
    const uint32_t sub = bucket_of_block(range, xcds);
    if (sub >= buckets) return;  // whole workgroup
    const uint32_t tid = threadIdx.x;
    const uint32_t first = t.sub_first[sub], count = t.sub_first[sub + 1] - first;
    if (count > kBucketRoom) return;  // whole workgroup: oversize_kernel's work
    if (count == 0) {
        for (uint32_t d = tid; d < (1u << t.d3) && !MANY; d += kBucketThreads) write_key_ptr(out, sub, t.d3, d, first, t.count);
        return;
    }
    s.clear_counts();
    const BucketRuns runs = runs_of_bucket(t, sub);
    map_runs<kBucketThreads, kBucketRoom>(runs.begins, runs.table, runs.tiles, count, 0, count, 0, runs.places, runs.source,
                                          s.map, s.buf);
    if (count <= static_cast<uint32_t>(kFewItems * kBucketThreads))
        sort_bucket<VB, Key, MANY, kFewItems>(t, sub, first, count, keys_in, aux_in, vals_in, out, s);
    else if (count <= static_cast<uint32_t>(kUsualItems * kBucketThreads))
        sort_bucket<VB, Key, MANY, kUsualItems>(t, sub, first, count, keys_in, aux_in, vals_in, out, s);
    else if (kMoreItems != kUsualItems && count <= static_cast<uint32_t>(kMoreItems * kBucketThreads))
        sort_bucket<VB, Key, MANY, kMoreItems>(t, sub, first, count, keys_in, aux_in, vals_in, out, s);
    else
        sort_bucket<VB, Key, MANY, kBucketItems>(t, sub, first, count, keys_in, aux_in, vals_in, out, s);
}

// ---- buckets that do not fit LDS -------------------------------------------------------------------------------
// One launch works on all of them, phase by phase: a workgroup takes the next chunk of the phase off a counter until none
// is left, adds what it has done to the phase's other counter, and waits there for the rest.  It only ever waits for chunks
// that running workgroups have taken, so every wait ends whether or not the other workgroups of the grid are resident.
// Entries and counts that are read in a later phase go past the caches.  The counts of a chunk become places in two steps:
// whoever counts the last chunk of a group adds the group up, whoever adds up the last group of a bucket says where every
// group's entries begin, and the second phase adds the chunks of the group in front of its own.
//
// Before, a workgroup looked for work among all buckets with two device-wide fences a chunk, one workgroup placed all
// chunks of a bucket, the counting phase read whole entries, and entries were written from where they lay in registers:
// csr2csc of 67 M nonzeros with columns by Zipf's law (53 M of them in such buckets) 3690 us, now 1458 (LSD passes: 1484);
// an index sort of 10 M triples with rows by that law 1870 us, then 953.  Since then: a workgroup looks a chunk's bucket up only
// where it is another one than before, waits for the end of a phase with fewer looks at the counter (848 -> 833 us; 512 of them
// looking hold the workgroups up that add to it), and pairs of keys that share a word stay one to the last pass (833 -> 748).
// Index sorts by a skewed major key stay slower than the LSD passes: 503 us for those, 936 against 1609 for 21.8 M triples
// in a million power-law rows of up to 50,000 (38 % of them in such buckets), 156 against 188 in a hundred thousand rows.
// A pass over such a bucket costs two phases of 45 us at least, and there are four or five of them.  How the keys are
// spread is not known on the host, where the choice is made, and evenly spread ones gain as much (10 M: 481 and 330 us);
// so does csr2csc under any spread.
constexpr uint32_t kOversizeGrid = 512;
// Up to that many workgroups may look more often than 512: waits are what a phase of few chunks takes.  By Zipf's law, with the long
// waits and with the short ones: csr2csc of 20 K nonzeros 48.4 and 46.1 us, 160 K 55.8 and 53.6, 1.05 M 68.5 and 67.2; index sorts of
// 10 K triples 96.6 and 89, 300 K 132 and 124, a million 149 and 145.  Of more chunks: csr2csc of 3.5 M 101 and 103, index sort of
// 4.8 M 434 and 450.  (With 128 for 256 csr2csc of 1.05 M 69, of 1.4 M 77.6 for 74.5; with 384 as with 256.)
constexpr uint32_t kFewOversizeChunks = 256;

struct OversizeChunk {
    uint32_t listed_at, bucket, first, entries;  // first: place of the bucket's first entry in the output
    uint32_t chunk, chunks, slot;                // slot: the bucket's first group
    uint32_t before;                             // chunks of the buckets listed before
};
// For whole wavefronts; every lane returns the same.
__device__ __forceinline__ OversizeChunk oversize_chunk(const SortTables& t, uint32_t listed, uint32_t number) {
    OversizeChunk c;
    c.listed_at = wave_count_up_to(t.oversize_first, listed, 0, number) - 1;
    c.before = t.oversize_first[c.listed_at];
    c.bucket = t.oversize_bucket[c.listed_at];
    c.first = t.sub_first[c.bucket];
    c.entries = t.sub_first[c.bucket + 1] - c.first;
    c.chunk = number - c.before;
    c.chunks = (c.entries + kOversizeChunk - 1) / kOversizeChunk;
    c.slot = oversize_slot(c.before, c.listed_at);
    return c;
}

// The next chunk of a phase that nobody has taken.
__device__ __forceinline__ uint32_t take_chunk(const SortTables& t, uint32_t phase) {
    return __hip_atomic_fetch_add(&t.oversize->taken[phase], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The counts of a bucket's groups, digit by digit, become places in the output.
__device__ __forceinline__ void place_groups(const SortTables& t, const OversizeChunk& c, const SortOutput& out, bool write_ptr,
                                             uint32_t bits, uint32_t (&s_sum)[kBucketThreads], uint32_t* s_wave) {
    constexpr uint32_t kDigits = 1 << kPassBits, kShares = kBucketThreads / kDigits;  // threads per digit
    const uint32_t d = threadIdx.x % kDigits, share = threadIdx.x / kDigits;
    const uint32_t groups = (c.chunks + kOversizeGroup - 1) / kOversizeGroup;
    const uint32_t mine = (groups + kShares - 1) / kShares;
    const uint32_t from = min(share * mine, groups), to = min(from + mine, groups);
    uint32_t* column = t.oversize_begins + (static_cast<uint64_t>(c.slot) << kPassBits) + d;
    constexpr uint32_t kBatch = 16;  // loads on their way at a time
    auto counts_of = [&](uint32_t g0, uint32_t (&n)[kBatch]) {
#pragma unroll
        for (uint32_t i = 0; i < kBatch; ++i) n[i] = load_shared(column + (static_cast<uint64_t>(min(g0 + i, to - 1)) << kPassBits));
    };
    uint32_t sum = 0, n[kBatch];
    for (uint32_t g = from; g < to; g += kBatch) {
        counts_of(g, n);
#pragma unroll
        for (uint32_t i = 0; i < kBatch; ++i) sum += g + i < to ? n[i] : 0u;
    }
    s_sum[threadIdx.x] = sum;
    __syncthreads();
    uint32_t total = 0, before = 0;
#pragma unroll
    for (uint32_t k = 0; k < kShares; ++k) {
        if (k == share) before = total;
        total += s_sum[k * kDigits + d];
    }
    const uint32_t first = c.first + block_exclusive_sum<kBucketThreads>(share == 0 ? total : 0u, s_wave);
    if (share == 0) {
        s_sum[d] = first;  // (every thread has read the sums: the barrier in the scan)
        if (write_ptr && d < (1u << bits)) write_key_ptr(out, c.bucket, t.d3, d, first, t.count);
    }
    __syncthreads();
    uint32_t at = s_sum[d] + before;
    for (uint32_t g = from; g < to; g += kBatch) {
        counts_of(g, n);
#pragma unroll
        for (uint32_t i = 0; i < kBatch; ++i) {
            if (g + i < to) store_shared(column + (static_cast<uint64_t>(g + i) << kPassBits), at);
            at += n[i];
        }
    }
}

template <int VB, typename Key, bool MANY>
__global__ __launch_bounds__(kBucketThreads, VB == 8 ? 2 : 4) void oversize_kernel(SortTables t, const Key* __restrict__ keys_in,
                                                                  const uint32_t* __restrict__ aux_in,
                                                                  const void* __restrict__ vals_in, SortOutput out) {
    typedef typename WordOf<VB>::type word_t;
    constexpr uint32_t kDigits = 1 << kPassBits;
    static_assert(kDigits <= kBucketThreads, "a thread per digit");
    constexpr bool kWords = MANY && packed_entries<Key>();  // both keys in a word, as which they travel to the last pass
    const unsigned long long counted = t.oversize->listed;
    const uint32_t listed = static_cast<uint32_t>(counted), all_chunks = static_cast<uint32_t>(counted >> 32);
    if (blockIdx.x >= all_chunks) return;  // whole workgroup: more workgroups than chunks
    __shared__ BucketLds s;
    __shared__ uint32_t s_count[kDigits];
    __shared__ uint32_t s_sum[kBucketThreads];
    __shared__ uint32_t s_ticket, s_last;
    const uint32_t tid = threadIdx.x, wave = tid / kWave;
    const uint32_t phases = 2 * t.oversize_passes;
    OversizeChunk c = {};
    for (uint32_t phase = 0; phase < phases; ++phase) {
        const uint32_t p = phase / 2;
        const uint32_t shift = p * t.oversize_width, bits = min(t.oversize_width, t.minor_bits + t.d3 - shift);
        const uint32_t mask = (1u << bits) - 1u;
        // which of the two keys the pass looks at
        const bool by_aux = MANY && shift < t.minor_bits, by_key = !MANY || shift + bits > t.minor_bits;
        auto digit_of = [&](uint32_t of_key, uint32_t of_aux) {
            if (!MANY || kWords) return of_key >> shift & mask;
            return static_cast<uint32_t>((static_cast<uint64_t>(of_key) << t.minor_bits | of_aux) >> shift) & mask;
        };
        // the first pass reads the runs, the others what the one before has left in the bucket's stretch
        const uint16_t* between_keys = t.oversize_keys[(p + 1) % 2];
        const uint32_t* between_aux = t.oversize_aux[(p + 1) % 2];
        const word_t* between_vals = static_cast<const word_t*>(t.oversize_vals[(p + 1) % 2]);
        if (tid == 0) {
            for (uint32_t idle = 0; phase != 0 && load_shared(&t.oversize->done[phase - 1]) < all_chunks; ++idle) {
                if (all_chunks <= kFewOversizeChunks)
                    for (uint32_t n = 0; n < (1u << min(idle, 2u)); ++n) __builtin_amdgcn_s_sleep(32);  // some 1, 2, 4 us
                else
                    for (uint32_t n = 0; n < (1u << min(idle, 1u)); ++n) __builtin_amdgcn_s_sleep(100);  // some 3, 6 us
            }
            s_ticket = take_chunk(t, phase);
        }
        __syncthreads();
        uint32_t finished = 0, number = s_ticket;
        while (number < all_chunks) {
            ++finished;
            // The next ticket: on its way while this chunk is worked on, unless that would take the last chunks away from
            // workgroups that have none yet.
            const bool ahead = all_chunks - number > gridDim.x;
            uint32_t next = 0;
            if (tid == 0 && ahead) next = take_chunk(t, phase);
            // (a chunk of the same bucket as the one before, as a rule where there are many: no search, five trips to memory)
            if (number - c.before < c.chunks) c.chunk = number - c.before;
            else c = oversize_chunk(t, listed, number);
            const uint32_t q0 = c.chunk * kOversizeChunk, count = min(c.entries - q0, kOversizeChunk);
            const uint32_t group = c.chunk / kOversizeGroup, in_group = c.chunk % kOversizeGroup;
            uint32_t* counts = t.oversize_counts + (static_cast<uint64_t>(number) << kPassBits);
            uint32_t* begins = t.oversize_begins + (static_cast<uint64_t>(c.slot + group) << kPassBits);
            if (p == 0) {
                const BucketRuns runs = runs_of_bucket(t, c.bucket);
                map_runs<kBucketThreads, kBucketRoom>(runs.begins, runs.table, runs.tiles, c.entries, q0, count,
                                                      find_first_run(runs.begins, runs.tiles, q0), runs.places, runs.source,
                                                      s.map, s.buf);
            }
            const uint32_t last_word = (count - 1) / kWave;
            // (worked out for every chunk again: as what it is, the same for all chunks, each item's share of it is held in
            // a register from the start on, and the kernel needs scratch memory)
            uint32_t own_wave = wave, own_slab = slab_place(kBucketItems, 0), own_thread = tid;
            forget(own_wave);
            forget(own_slab);
            forget(own_thread);
            auto place_of = [&](int i) {
                return p == 0 ? mapped_place(s.map, s.buf, min(own_wave * kBucketItems + i, last_word), count)
                              : c.first + q0 + min(own_slab + i * kWave, count - 1);
            };
            if (phase % 2 == 0) {
                if (tid < kDigits) s_count[tid] = 0;
                uint32_t key[kBucketItems], aux[MANY && !kWords ? kBucketItems : 1];
#pragma unroll
                for (int i = 0; i < kBucketItems; ++i) {
                    const uint32_t from = place_of(i);
                    key[i] = 0;
                    if constexpr (packed_entries<Key>()) {
                        key[i] = !MANY || p == 0 ? load_at<uint32_t>(keys_in, VB == 4 ? 2 * from : from)
                                                 : load_shared_at<uint32_t>(between_aux, from);
                    } else {
                        if (by_key) key[i] = p == 0 ? load_at<Key>(keys_in, from) : load_shared_at<uint16_t>(between_keys, from);
                        if constexpr (MANY) {
                            aux[i] = 0;
                            if (by_aux) aux[i] = p == 0 ? load_at<uint32_t>(aux_in, from) : load_shared_at<uint32_t>(between_aux, from);
                        }
                    }
                }
                __syncthreads();
#pragma unroll
                for (int i = 0; i < kBucketItems; ++i) {
                    if (in_slab(kBucketItems, i, count)) atomicAdd(&s_count[digit_of(key[i], MANY && !kWords ? aux[MANY && !kWords ? i : 0] : 0u)], 1u);
                }
                __syncthreads();
                if (tid < kDigits) store_shared(counts + tid, s_count[tid]);
                const uint32_t chunks_here = min(c.chunks - group * kOversizeGroup, kOversizeGroup);
                if (last_to_arrive(t.oversize_arrived + c.slot + group, chunks_here, &s_last)) {  // whole workgroup
                    if (tid < kDigits) {
                        const uint32_t* column = counts - (static_cast<uint64_t>(in_group) << kPassBits) + tid;
                        uint32_t n[kOversizeGroup], sum = 0;
#pragma unroll
                        for (uint32_t k = 0; k < kOversizeGroup; ++k) n[k] = load_shared(column + (min(k, chunks_here - 1) << kPassBits));
#pragma unroll
                        for (uint32_t k = 0; k < kOversizeGroup; ++k) sum += k < chunks_here ? n[k] : 0u;
                        store_shared(begins + tid, sum);
                    }
                    const uint32_t groups = (c.chunks + kOversizeGroup - 1) / kOversizeGroup;
                    if (last_to_arrive(t.oversize_counted + c.listed_at, groups, &s_last))
                        place_groups(t, c, out, !MANY, bits, s_sum, s.wave);
                }
            } else {
                s.clear_counts();
                if (tid < kDigits) {  // where the chunk's entries of each digit begin
                    const uint32_t* column = counts - (static_cast<uint64_t>(in_group) << kPassBits) + tid;
                    uint32_t n[kOversizeGroup], sum = load_shared(begins + tid);
#pragma unroll
                    for (uint32_t k = 0; k < kOversizeGroup; ++k) n[k] = load_shared(column + (min(k, in_group) << kPassBits));
#pragma unroll
                    for (uint32_t k = 0; k < kOversizeGroup; ++k) sum += k < in_group ? n[k] : 0u;
                    s_sum[tid] = sum;
                }
                uint32_t key[kBucketItems], aux[kWords ? 1 : kBucketItems];  // words: in key
                word_t val[VB ? kBucketItems : 1];
#pragma unroll
                for (int i = 0; i < kBucketItems; ++i) {
                    const uint32_t from = place_of(i);
                    if constexpr (kWords) {
                        if (p == 0) {
                            load_packed<VB>(keys_in, vals_in, from, key[i], val[VB ? i : 0]);
                        } else {
                            key[i] = load_shared_at<uint32_t>(between_aux, from);
                            if constexpr (VB != 0) val[i] = load_shared_at<word_t>(between_vals, from);
                        }
                    } else if (packed_entries<Key>()) {
                        load_packed<VB>(keys_in, vals_in, from, key[i], val[VB ? i : 0]);
                        aux[kWords ? 0 : i] = key[i] >> t.d3;
                    } else if (!MANY || p == 0) {
                        key[i] = load_at<Key>(keys_in, from);
                        aux[kWords ? 0 : i] = load_at<uint32_t>(aux_in, from);
                        if constexpr (VB != 0) val[i] = load_at<word_t>(vals_in, from);
                    } else {
                        key[i] = load_shared_at<uint16_t>(between_keys, from);
                        aux[kWords ? 0 : i] = load_shared_at<uint32_t>(between_aux, from);
                        if constexpr (VB != 0) val[i] = load_shared_at<word_t>(between_vals, from);
                    }
                }
                __syncthreads();
                auto digit = [&](int i) { return digit_of(key[i], aux[kWords ? 0 : i]); };
                uint32_t dest[kBucketItems / 2];
                rank_entries<kBucketItems, kPassBits>(count, bits, s.cnt, dest, digit);
                __syncthreads();
                // (s_count: where the digit's first entry of the chunk goes, less its place in the chunk)
                place_digits<kBucketThreads, kPassBits>(bits, s.cnt, s.wave,
                                                        [&](uint32_t d, uint32_t at, uint32_t) { s_count[d] = s_sum[d] - at; });
#pragma unroll
                for (int i = 0; i < kBucketItems; ++i)
                    dest[i / 2] += static_cast<uint32_t>(s.cnt[(wave << kPassBits) + digit(i)]) << (i % 2 * 16);
                // into LDS in the new order, and out of it with neighbouring lanes on neighbouring entries
                auto in_order = [&](auto word_of, auto use) {
#pragma unroll
                    for (int i = 0; i < kBucketItems; ++i) {
                        if (in_slab(kBucketItems, i, count)) s.buf[(dest[i / 2] >> (i % 2 * 16)) & 0xffffu] = word_of(i);
                    }
                    __syncthreads();
#pragma unroll
                    for (int i = 0; i < kBucketItems; ++i) {
                        const uint32_t at = i * kBucketThreads + own_thread;
                        if (at < count) use(i, at, s.buf[at]);
                    }
                    __syncthreads();
                };
                uint32_t put[kBucketItems];
                in_order([&](int i) { return s_count[digit(i)]; }, [&](int i, uint32_t at, uint32_t w) { put[i] = w + at; });
                // (what the last pass writes nobody reads in this launch)
                const bool to_output = !MANY || p + 1 == t.oversize_passes;
                auto move = [&](auto word_of, auto* between, auto* output, auto finish) {
                    if (to_output)
                        in_order(word_of, [&](int i, uint32_t, uint32_t w) { store_at(output, put[i], finish(i, w)); });
                    else
                        in_order(word_of, [&](int i, uint32_t, uint32_t w) { store_shared_at(between, put[i], finish(i, w)); });
                };
                auto as_it_is = [](int, uint32_t w) { return w; };
                if constexpr (kWords) {
                    const uint32_t minor_mask = to_output ? (1u << t.minor_bits) - 1u : ~0u;
                    move([&](int i) { return key[i]; }, t.oversize_aux[p % 2], out.aux, [&](int, uint32_t w) { return w & minor_mask; });
                } else {
                    move([&](int i) { return aux[i]; }, t.oversize_aux[p % 2], out.aux, as_it_is);
                }
                if constexpr (VB == 4) {
                    move([&](int i) { return val[i]; }, static_cast<uint32_t*>(t.oversize_vals[p % 2]),
                         static_cast<uint32_t*>(out.vals), as_it_is);
                } else if constexpr (VB == 8) {  // in two halves
                    uint32_t low[kBucketItems];
                    in_order([&](int i) { return static_cast<uint32_t>(val[i]); }, [&](int i, uint32_t, uint32_t w) { low[i] = w; });
                    move([&](int i) { return static_cast<uint32_t>(val[i] >> 32); }, static_cast<uint64_t*>(t.oversize_vals[p % 2]),
                         static_cast<uint64_t*>(out.vals), [&](int i, uint32_t w) { return static_cast<uint64_t>(w) << 32 | low[i]; });
                }
                if constexpr (kWords) {
                    if (to_output) {
                        const uint32_t high = (c.bucket << t.d3) + out.key_bias;
                        in_order([&](int i) { return key[i] >> t.minor_bits; },
                                 [&](int i, uint32_t, uint32_t w) { store_at(out.keys, put[i], high + w); });
                    }
                } else if constexpr (MANY) {
                    if (!to_output) {
                        uint16_t* keys_to = t.oversize_keys[p % 2];
                        in_order([&](int i) { return key[i]; },
                                 [&](int i, uint32_t, uint32_t w) { store_shared_at(keys_to, put[i], static_cast<uint16_t>(w)); });
                    } else {
                        const uint32_t high = (c.bucket << t.d3) + out.key_bias;
                        in_order([&](int i) { return key[i]; }, [&](int i, uint32_t, uint32_t w) { store_at(out.keys, put[i], high + w); });
                    }
                }
            }
            // (both barriers here: with the second one at the head of the loop the compiler, ROCm 7.2, leaves out the wait
            // for the store of the ticket in front of it, and some wavefronts go on with the old one)
            __syncthreads();
            if (tid == 0) s_ticket = ahead ? next : take_chunk(t, phase);
            __syncthreads();
            number = s_ticket;
        }
        wait_for_stores();
        __syncthreads();
        if (tid == 0 && finished != 0)
            __hip_atomic_fetch_add(&t.oversize->done[phase], finished, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

static_assert(kTileSmall == kBucketTileMin, "what the sums over buckets make room for");

template <int VB, int KIND, int MAX_BITS, typename Key>
void launch_partition(hipStream_t stream, const EntrySource& in, uint32_t shift, uint32_t bits, uint32_t tile_size,
                      void* keys_out, uint32_t* aux_out, void* vals_out, uint32_t* table) {
    const uint32_t tiles = tiles_of(in.count, tile_size);
    const uint32_t xcds = device_topology().xcds;
    const dim3 grid((tiles + xcds - 1) / xcds * xcds);
    // 16 wavefronts with half the items each need half the registers and fill a compute unit: packed entries of csr2csc (118 M,
    // 1163 -> 1139 us; with the counters of 11 bits they would fill it with one workgroup, 2 M: 85.6 -> 89.6), and index sorts,
    // whose counts and words share their place (7.2 M triples, partition 42.9 -> 39.5 us; all of the assembly 185 -> 181).
    constexpr int kThreads = KIND == kPlain || (packed_entries<Key>() && MAX_BITS <= 8) ? 1024 : 512;
    if (tile_size == kTileLarge) {
        hipLaunchKernelGGL((partition_kernel<VB, KIND, MAX_BITS, Key, kThreads, kTileLarge / kThreads>), grid, dim3(kThreads), 0,
                           stream, in, shift, bits, tiles, static_cast<Key*>(keys_out), aux_out, vals_out, table, xcds);
    } else {
        hipLaunchKernelGGL((partition_kernel<VB, KIND, MAX_BITS, Key, 512, 8>), grid, dim3(512), 0, stream, in, shift, bits,
                           tiles, static_cast<Key*>(keys_out), aux_out, vals_out, table, xcds);
    }
}

void launch_row_starts(hipStream_t stream, const EntrySource& in, uint32_t tile_size, uint32_t* tile_rows, uint32_t* wide) {
    const uint32_t tiles = tiles_of(in.count, tile_size);
    constexpr uint32_t kPerBlock = kRowStartsBlock / kWave;
    hipLaunchKernelGGL(partition_row_starts_kernel, dim3(tiles / kPerBlock + 1), dim3(kRowStartsBlock), 0, stream, in.aux,
                       in.m, in.base, in.count, tile_size, tiles, tile_rows, wide);
}

struct BucketedLayout {
    size_t keys, products, table, totals, tile_rows, spare;
};
BucketedLayout bucketed_layout(idx_t nnz, uint32_t bits, size_t value_bytes) {
    const uint32_t tile_size = tile_size_for(nnz);
    const size_t tiles = tiles_of(nnz, tile_size);
    BucketedLayout l;
    size_t off = 0;
    const size_t places = tile_places(tile_size, kProducts, bits);
    l.keys = off; off += align_up(tiles * places * sizeof(uint16_t));
    l.products = off; off += align_up(tiles * places * value_bytes);
    l.table = off; off += align_up((tiles << bits) * sizeof(uint32_t));
    l.totals = off; off += align_up(sizeof(uint32_t) << bits);
    l.tile_rows = off; off += align_up((tiles + 1) * sizeof(uint32_t));
    l.spare = off;
    return l;
}

// ---- the sort --------------------------------------------------------------------------------------------------
void sort_passes(const SortShape& s, SortTables* t) {
    const uint32_t minor = s.minor_bits == kNoMinorKey ? 0 : s.minor_bits;
    auto passes_for = [](uint32_t bits) { return (bits + kPassBits - 1) / kPassBits; };
    auto width_for = [&](uint32_t bits) { return bits == 0 ? 0 : (bits + passes_for(bits) - 1) / passes_for(bits); };
    t->minor_bits = minor;
    t->minor_passes = passes_for(minor);
    t->minor_width = width_for(minor);
    t->key_width = width_for(s.d3);
    t->passes = t->minor_passes + passes_for(s.d3);
    if (t->passes == 0) t->passes = 1;  // everything in order already: one pass over no bits
    t->oversize_passes = std::max(passes_for(minor + s.d3), 1u);
    t->oversize_width = (minor + s.d3 + t->oversize_passes - 1) / t->oversize_passes;
}

// Tiles of step 2 that one bucket of step 1 can have: all entries may lie in one (tiles of step 1 hold more entries, so
// their number is no bound).
uint32_t second_tiles_most(uint32_t count) { return (count - 1) / kSecondTile + 1; }

struct SortLayout {
    size_t keys1, aux1, vals1, keys2, aux2, vals2, wide, table1, begins1, totals1, tile_rows, table2, begins2, bucket_first,
        tile_first, first_runs, tile_map, sub_first, sub_arrived, oversize, oversize_bucket, oversize_first, oversize_counted, oversize_arrived,
        oversize_counts, oversize_begins, oversize_keys[2], oversize_aux[2], oversize_vals[2], total;
};
SortLayout sort_layout(uint32_t count, const SortShape& s, size_t value_bytes) {
    const size_t places1 = static_cast<size_t>(s.tiles1) * s.tile_size;
    const size_t places2 = static_cast<size_t>(s.max_tiles2) * kSecondTile;
    const size_t runs1 = static_cast<size_t>(s.tiles1) << s.d1, runs2 = static_cast<size_t>(s.max_tiles2) << s.d2;
    const size_t subs = size_t(1) << (s.d1 + s.d2);
    const size_t oversize = static_cast<size_t>(count) / kBucketRoom + 1;
    const size_t chunks = 2 * (static_cast<size_t>(count) / kOversizeChunk) + 1;  // every oversize bucket has two at least
    const size_t groups = chunks / kOversizeGroup + oversize + 1;
    SortLayout l;
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t at = off;
        off += align_up(bytes);
        return at;
    };
    // packed: words, or {word, value} pairs
    const bool pairs = value_bytes == sizeof(uint32_t);
    const size_t entry = pairs ? sizeof(uint64_t) : sizeof(uint32_t), apart = pairs ? 0 : value_bytes;
    const bool rows_apart = s.minor_bits == kNoMinorKey && s.d2 != 0;  // of tiles that span many
    l.keys1 = take(places1 * (packs_first(s) ? entry : bytes_of(first_key_word(s))));
    l.aux1 = take(!packs_first(s) || rows_apart ? places1 * sizeof(uint32_t) : 0);
    l.vals1 = take(places1 * (packs_first(s) ? apart : value_bytes));
    l.keys2 = take(places2 * (s.packed ? entry : bytes_of(second_key_word(s))));
    l.aux2 = take(s.packed ? 0 : places2 * sizeof(uint32_t));
    l.vals2 = take(places2 * (s.packed ? apart : value_bytes));
    l.wide = take(sizeof(uint32_t));
    l.table1 = take(runs1 * sizeof(uint32_t));
    l.begins1 = take(runs1 * sizeof(uint32_t));
    l.totals1 = take(sizeof(uint32_t) << s.d1);
    l.tile_rows = take((static_cast<size_t>(s.tiles1) + 1) * sizeof(uint32_t));
    l.table2 = take(runs2 * sizeof(uint32_t));
    l.begins2 = take(runs2 * sizeof(uint32_t));
    l.bucket_first = take((sizeof(uint32_t) << s.d1) + sizeof(uint32_t));
    l.tile_first = take((sizeof(uint32_t) << s.d1) + sizeof(uint32_t));
    l.first_runs = take(s.d2 != 0 ? (static_cast<size_t>(second_tiles_most(count)) << s.d1) * sizeof(uint32_t) : 0);
    l.tile_map = take(static_cast<size_t>(s.max_tiles2) * sizeof(uint2));
    l.sub_first = take((subs + 1) * sizeof(uint32_t));
    l.sub_arrived = take(sizeof(uint32_t) << s.d1);
    l.oversize = take(sizeof(OversizeState));
    l.oversize_bucket = take(oversize * sizeof(uint32_t));
    l.oversize_first = take(oversize * sizeof(uint32_t));
    l.oversize_counted = take(oversize * sizeof(uint32_t));
    l.oversize_arrived = take(groups * sizeof(uint32_t));
    l.oversize_counts = take((chunks << kPassBits) * sizeof(uint32_t));
    l.oversize_begins = take((groups << kPassBits) * sizeof(uint32_t));
    SortTables passes;
    sort_passes(s, &passes);
    for (uint32_t k = 0; k < 2; ++k) {
        const size_t between = count > kBucketRoom && passes.oversize_passes > k + 1 ? count : 0;
        l.oversize_keys[k] = take(between * sizeof(uint16_t));
        l.oversize_aux[k] = take(between * sizeof(uint32_t));
        l.oversize_vals[k] = take(between * value_bytes);
    }
    l.total = off;
    return l;
}

template <int VB, int KIND>
void launch_sort(hipStream_t stream, EntrySource in, const SortShape& s, const SortOutput& out, char* w) {
    const SortLayout l = sort_layout(in.count, s, VB);
    auto words = [&](size_t at) { return reinterpret_cast<uint32_t*>(w + at); };
    const uint32_t xcds = device_topology().xcds;
    if constexpr (KIND == kCsr) {
        in.wide = words(l.wide);
        in.relative = s.packed && s.d2 != 0;
        launch_row_starts(stream, in, s.tile_size, words(l.tile_rows), in.wide);
        in.tile_rows = words(l.tile_rows);
    }
    SortTables t;
    t.tile_rows = words(l.tile_rows);
    t.wide = words(l.wide);
    t.tile1_shift = bit_length(s.tile_size) - 1;
    t.base = in.base;
    t.table1 = words(l.table1);
    t.begins1 = words(l.begins1);
    t.totals1 = words(l.totals1);
    t.tiles1 = s.tiles1;
    t.places1 = s.tile_size;
    t.table2 = words(l.table2);
    t.begins2 = words(l.begins2);
    t.bucket_first = words(l.bucket_first);
    t.tile_first = words(l.tile_first);
    t.first_runs = words(l.first_runs);
    t.first_stride = second_tiles_most(in.count);
    t.tile_map = reinterpret_cast<uint2*>(w + l.tile_map);
    t.sub_first = words(l.sub_first);
    t.sub_arrived = words(l.sub_arrived);
    t.oversize = reinterpret_cast<OversizeState*>(w + l.oversize);
    t.oversize_bucket = words(l.oversize_bucket);
    t.oversize_first = words(l.oversize_first);
    t.oversize_counted = words(l.oversize_counted);
    t.oversize_arrived = words(l.oversize_arrived);
    t.oversize_counts = words(l.oversize_counts);
    t.oversize_begins = words(l.oversize_begins);
    for (uint32_t k = 0; k < 2; ++k) {
        t.oversize_keys[k] = reinterpret_cast<uint16_t*>(w + l.oversize_keys[k]);
        t.oversize_aux[k] = words(l.oversize_aux[k]);
        t.oversize_vals[k] = w + l.oversize_vals[k];
    }
    sort_passes(s, &t);
    t.d1 = s.d1;
    t.d2 = s.d2;
    t.d3 = s.d3;
    t.count = in.count;
    const uint32_t shift = s.d2 + s.d3;
    constexpr bool kMany = KIND == kPlain;  // the sorts by two keys
    in.minor_bits = t.minor_bits;
    auto with_digits = [&](auto key) {
        typedef decltype(key) Key;
        return s.d1 <= 8 ? launch_partition<VB, KIND, 8, Key> : launch_partition<VB, KIND, kMaxOneLevelBits, Key>;
    };
    // (a sort by one key: 8 or 32 bits, or 16 to step 2; by two keys: 16 or 32)
    auto with_word = [&](KeyWord word, auto launch) {
        if (word == KeyWord::k32) return launch(uint32_t());
        if constexpr (kMany) launch(uint16_t());
        else launch(uint8_t());
    };
    const KeyWord first_word = first_key_word(s);
    if (!kMany && first_word == KeyWord::k16) {
        with_digits(uint16_t())(stream, in, shift, s.d1, s.tile_size, w + l.keys1, words(l.aux1), w + l.vals1, words(l.table1));
    } else {
        with_word(first_word, [&](auto key) {
            with_digits(key)(stream, in, shift, s.d1, s.tile_size, w + l.keys1, words(l.aux1), w + l.vals1, words(l.table1));
        });
    }
    // (few tiles: a round of small workgroups, several digits to a compute unit; many: few rounds)
    auto* run_begins = s.tiles1 > 1024 ? run_begins_kernel<1024, 8> : run_begins_kernel<256, 4>;
    hipLaunchKernelGGL(run_begins, dim3(1u << s.d1), dim3(s.tiles1 > 1024 ? 1024 : 256), 0, stream, s.tiles1, t.table1,
                       words(l.begins1), words(l.totals1), s.d2 != 0 ? words(l.first_runs) : nullptr, t.first_stride);
    hipLaunchKernelGGL(sort_plan_kernel, dim3(1), dim3(kPlanBlock), 0, stream, t);
    const void* keys = w + l.keys1;
    const uint32_t* aux = words(l.aux1);
    const void* vals = w + l.vals1;
    if (s.d2 != 0) {
        hipLaunchKernelGGL(tile_map_kernel, dim3((s.max_tiles2 + kMapBlock - 1) / kMapBlock), dim3(kMapBlock), 0, stream, t);
        const dim3 grid((s.max_tiles2 + xcds - 1) / xcds * xcds);
        auto repartition = [&](auto key) {
            typedef decltype(key) Key;
            hipLaunchKernelGGL((repartition_kernel<VB, Key, kMany>), grid, dim3(kSecondThreads), 0, stream, t, keys, aux, vals,
                               reinterpret_cast<Key*>(w + l.keys2), words(l.aux2), w + l.vals2, xcds);
        };
        with_word(second_key_word(s), repartition);
        hipLaunchKernelGGL(sub_begins_kernel, dim3(kSubParts << s.d1), dim3(kSubBlock), 0, stream, t);
        keys = w + l.keys2;
        aux = words(l.aux2);
        vals = w + l.vals2;
    }
    const uint32_t buckets = 1u << (s.d1 + s.d2);
    // (what a contiguous range is of: the buckets that have keys, which the sorts by two keys don't tell)
    const uint32_t used = ((out.key_count - 1) >> s.d3) + 1, range = !kMany && in.count <= kEntriesThatStay ? (used + xcds - 1) / xcds : 0;
    const uint32_t per_round = xcds * (range != 0 ? range : kNeighbours);
    const dim3 grid((buckets + per_round - 1) / per_round * per_round);
    auto sort = [&](auto key) {
        typedef decltype(key) Key;
        hipLaunchKernelGGL((bucket_sort_kernel<VB, Key, kMany>), grid, dim3(kBucketThreads), 0, stream, t,
                           static_cast<const Key*>(keys), aux, vals, out, buckets, range, xcds);
        if (in.count > kBucketRoom)  // else no bucket is larger than that
            hipLaunchKernelGGL((oversize_kernel<VB, Key, kMany>), dim3(kOversizeGrid), dim3(kBucketThreads), 0, stream, t,
                               static_cast<const Key*>(keys), aux, vals, out);
    };
    with_word(s.d2 != 0 ? second_key_word(s) : first_word, sort);
}

}  // namespace

bool partition_sort_usable(idx_t count, idx_t key_count) {
    SortShape s;
    return sort_shape(count, key_count, kNoMinorKey, &s);
}
size_t partition_sort_workspace_bytes(idx_t count, idx_t key_count, size_t value_bytes) {
    SortShape s;
    if (!sort_shape(count, key_count, kNoMinorKey, &s)) return 0;
    const size_t apart = sort_layout(count, s, value_bytes).total;  // (the rows are not known here)
    s.packed = true;
    return std::max(apart, sort_layout(count, s, value_bytes).total);
}
bool partition_sort_pairs_usable(idx_t count, idx_t major_count, idx_t minor_count) {
    SortShape s;
    return sort_shape(count, major_count, bit_length(minor_count - 1), &s);
}
size_t partition_sort_pairs_workspace_bytes(idx_t count, idx_t major_count, idx_t minor_count) {
    SortShape s;
    if (!sort_shape(count, major_count, bit_length(minor_count - 1), &s)) return 0;
    s.packed = sort_packs(s, minor_count);
    return sort_layout(count, s, sizeof(idx_t)).total;
}

void launch_partition_sort(hipStream_t stream, idx_t count, const PartitionSortArgs& a, size_t value_bytes, void* workspace) {
    SortShape s;
    if (!sort_shape(count, a.key_count, kNoMinorKey, &s)) return;
    s.packed = sort_packs(s, a.csr_rows);
    EntrySource in;
    in.keys = a.keys_in;
    in.aux = a.row_ptr;
    in.vals = a.vals_in;
    in.x = nullptr;
    in.count = count;
    in.key_bias = a.key_bias;
    in.m = a.csr_rows;
    in.base = a.base;
    in.tile_rows = nullptr;
    SortOutput out;
    out.keys = nullptr;
    out.aux = a.aux_out;
    out.vals = a.vals_out;
    out.key_ptr = a.key_ptr;
    out.key_count = a.key_count;
    out.base = a.base;
    out.key_bias = a.key_bias;
    auto* launch = value_bytes == 0 ? launch_sort<0, kCsr> : value_bytes == 4 ? launch_sort<4, kCsr> : launch_sort<8, kCsr>;
    launch(stream, in, s, out, static_cast<char*>(workspace));
}

void launch_partition_sort_pairs(hipStream_t stream, idx_t count, idx_t major_count, idx_t minor_count, idx_t* major,
                                 idx_t* minor, idx_t* perm, void* workspace) {
    SortShape s;
    if (!sort_shape(count, major_count, bit_length(minor_count - 1), &s)) return;
    s.packed = sort_packs(s, minor_count);
    EntrySource in = {};
    in.keys = major;
    in.aux = minor;
    in.vals = perm;
    in.count = count;
    SortOutput out = {};
    out.keys = major;
    out.aux = minor;
    out.vals = perm;
    auto* launch = perm == nullptr ? launch_sort<0, kPlain> : launch_sort<4, kPlain>;
    launch(stream, in, s, out, static_cast<char*>(workspace));
}

bool bucketed_products_shape(idx_t n, ColumnBuckets* columns) {
    // fewer columns than that: the full sort is two short passes; more: a bucket's sums no longer fit in LDS
    if (n < kBucketMinColumns) return false;
    for (const uint32_t bits : {kBucketFewBits, kBucketManyBits}) {
        *columns = column_buckets(n, bits);
        if (columns->width <= kBucketMaxColumns) return true;
    }
    return false;
}

size_t bucketed_products_workspace_bytes(idx_t nnz, uint32_t bits, size_t value_bytes) {
    return bucketed_layout(nnz, bits, value_bytes).spare;
}

// One partition by the buckets of the columns (index base taken off), the values multiplied by x[row] on the
// way.  What lies behind workspace_bytes is not touched.
void launch_bucketed_products(hipStream_t stream, idx_t m, idx_t n, idx_t nnz, const void* csr_val, const idx_t* row_ptr,
                              const idx_t* col, const void* x, size_t value_bytes, idx_t base, void* workspace,
                              size_t workspace_bytes, BucketedProducts* out) {
    if (m == 0 || nnz == 0 || !bucketed_products_shape(n, &out->columns)) return;
    const uint32_t bits = out->columns.bits;
    const BucketedLayout l = bucketed_layout(nnz, bits, value_bytes);
    char* w = static_cast<char*>(workspace);
    EntrySource in;
    in.keys = col;
    in.aux = row_ptr;
    in.vals = csr_val;
    in.x = x;
    in.count = nnz;
    in.key_bias = base;
    in.m = m;
    in.base = base;
    in.tile_rows = reinterpret_cast<uint32_t*>(w + l.tile_rows);
    const uint32_t tile_size = tile_size_for(nnz);
    uint32_t* table = reinterpret_cast<uint32_t*>(w + l.table);
    launch_row_starts(stream, in, tile_size, reinterpret_cast<uint32_t*>(w + l.tile_rows), nullptr);
    auto of_bits = [&](auto vb) {
        constexpr int VB = decltype(vb)::value;
        return bits == kBucketFewBits ? launch_partition<VB, kProducts, kBucketFewBits, uint16_t>
                                      : launch_partition<VB, kProducts, kBucketManyBits, uint16_t>;
    };
    auto* launch = value_bytes == 4 ? of_bits(std::integral_constant<int, 4>{}) : of_bits(std::integral_constant<int, 8>{});
    in.columns = out->columns;
    launch(stream, in, 0, bits, tile_size, w + l.keys, nullptr, w + l.products, table);
    out->keys = reinterpret_cast<const uint16_t*>(w + l.keys);
    out->products = w + l.products;
    out->table = table;
    out->totals = reinterpret_cast<uint32_t*>(w + l.totals);
    out->tiles = tiles_of(nnz, tile_size);
    out->tile_places = tile_places(tile_size, kProducts, bits);
    out->spare = w + l.spare;
    out->spare_bytes = workspace_bytes > l.spare ? workspace_bytes - l.spare : 0;
}

}  // namespace mcsp
