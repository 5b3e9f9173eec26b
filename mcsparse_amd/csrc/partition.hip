// Partition of entries by the top bits of a key, tile by tile, for gfx950.
//
// partition_kernel orders the entries of a tile by a digit of their keys, inside the tile only, and writes the tile back
// as one linear stream, with a table of where each digit's run begins.  Against a radix pass that writes every entry
// straight to its bucket (src/mcprim/device_radix_sort.hpp:90-309 of the reference) it needs no counting pass and makes
// no scattered store; the runs are put together by whoever reads them next.
#include "partition_device.h"

namespace mcsp {

namespace {

using namespace partition_detail;

template <int VB>
struct WordOf { typedef uint32_t type; };
template <>
struct WordOf<8> { typedef uint64_t type; };
template <int VB>
struct RealOf { typedef float type; };
template <>
struct RealOf<8> { typedef double type; };

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
};

// The order of tiles over the workgroups: an XCD takes a contiguous range, so the table words of neighbouring tiles,
// which share lines, meet in one L2.
__device__ __forceinline__ uint32_t tile_of_block(uint32_t tiles, uint32_t xcds) {
    const uint32_t per_xcd = (tiles + xcds - 1) / xcds;
    return (blockIdx.x % xcds) * per_xcd + blockIdx.x / xcds;
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

// A workgroup per tile.  Key: the type the rest of a key travels in.
//
// Bounds at 118 M entries (the products of a transposing SpMV, fp32): 0.98 GB read and 0.79 GB written in 340 us, nine
// tenths of the rate of a copy; tiles of 4096 or 16 wavefronts per workgroup are no faster (342 and 420 us).  The pass
// it replaces took 486 us, with a pass over the keys (111 us) in front of it to count them.
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
    __shared__ __align__(16) uint32_t s_buf[kPlaces];
    __shared__ __align__(16) uint16_t s_cnt[kOrdered ? kWaves << MAX_BITS : 2 << MAX_BITS];
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
    for (uint32_t i = tid; i < sizeof(s_cnt) / 16; i += THREADS) reinterpret_cast<u32x4*>(s_cnt)[i] = u32x4(0);
    __syncthreads();

    const uint32_t mask = (1u << bits) - 1u;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) key[i] -= in.key_bias;
    auto digit = [&](int i) { return (key[i] >> shift) & mask; };
    uint32_t dest[(ITEMS + 1) / 2];
    uint32_t pad_from = 0, pad_to = 0;  // what this thread's digit leaves open behind its run
    uint32_t* const s_count = reinterpret_cast<uint32_t*>(s_cnt);
    if constexpr (kOrdered) rank_entries<ITEMS, MAX_BITS, kWaves>(count, ITEMS, bits, s_cnt, dest, digit);
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
        static_assert(1 << MAX_BITS <= THREADS, "a thread per digit");
        const uint32_t n = tid < (1u << MAX_BITS) ? s_count[tid] : 0;
        const uint32_t padded = (n + kPad - 1) / kPad * kPad;
        const uint32_t at = block_exclusive_sum<THREADS>(padded, s_wave);
        if (tid < (1u << MAX_BITS)) {
            s_count[tid] = at;
            if (tid < (1u << bits)) table[static_cast<uint64_t>(tid) * tiles + tile] = table_word(at, padded);
        }
        pad_from = at + n;
        pad_to = at + padded;
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t at = kOrdered ? s_cnt[(tid / kWave << MAX_BITS) + digit(i)] : s_count[digit(i)];
        dest[i / 2] += at << (i % 2 * 16);
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) forget(key[i]);

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
    store_keys<ITEMS, THREADS, kPlaces>(s_buf, count, dest, keys_out + out, key, (1u << shift) - 1u);
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
        for (uint32_t p = pad_from; p < pad_to; ++p) s_buf[p] = 0;
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
                                                                               uint32_t* __restrict__ tile_rows) {
    const uint32_t t = blockIdx.x * (kRowStartsBlock / kWave) + threadIdx.x / kWave;
    if (t > tiles) return;  // whole wavefront
    const uint64_t first = static_cast<uint64_t>(t) * tile_size;
    // (m + 1 < 2^32: the reference's limit on extents)
    const uint32_t starts = wave_count_up_to(row_ptr, m + 1, base, first < nnz ? static_cast<uint32_t>(first) : nnz);
    if (threadIdx.x % kWave == 0) tile_rows[t] = starts;
}

// Small inputs get small tiles, so that there are a few workgroups per compute unit.
constexpr uint32_t kTileLarge = 8192, kTileSmall = 2048;
constexpr uint32_t kSmallTileEntries = 512 * kTileLarge;
static_assert(kTileSmall == kBucketTileMin, "what the sums over buckets make room for");
uint32_t tile_size_for(uint32_t count) { return count <= kSmallTileEntries ? kTileSmall : kTileLarge; }
uint32_t tiles_of(uint32_t count, uint32_t tile_size) {
    return static_cast<uint32_t>((static_cast<uint64_t>(count) + tile_size - 1) / tile_size);
}

template <int VB, int KIND, int MAX_BITS, typename Key>
void launch_partition(hipStream_t stream, const EntrySource& in, uint32_t shift, uint32_t bits, uint32_t tile_size,
                      void* keys_out, uint32_t* aux_out, void* vals_out, uint32_t* table) {
    const uint32_t tiles = tiles_of(in.count, tile_size);
    const uint32_t xcds = device_topology().xcds;
    const dim3 grid((tiles + xcds - 1) / xcds * xcds);
    if (tile_size == kTileLarge) {
        hipLaunchKernelGGL((partition_kernel<VB, KIND, MAX_BITS, Key, 512, 16>), grid, dim3(512), 0, stream, in, shift, bits,
                           tiles, static_cast<Key*>(keys_out), aux_out, vals_out, table, xcds);
    } else {
        hipLaunchKernelGGL((partition_kernel<VB, KIND, MAX_BITS, Key, 256, 8>), grid, dim3(256), 0, stream, in, shift, bits,
                           tiles, static_cast<Key*>(keys_out), aux_out, vals_out, table, xcds);
    }
}

void launch_row_starts(hipStream_t stream, const EntrySource& in, uint32_t tile_size, uint32_t* tile_rows) {
    const uint32_t tiles = tiles_of(in.count, tile_size);
    constexpr uint32_t kPerBlock = kRowStartsBlock / kWave;
    hipLaunchKernelGGL(partition_row_starts_kernel, dim3(tiles / kPerBlock + 1), dim3(kRowStartsBlock), 0, stream, in.aux,
                       in.m, in.base, in.count, tile_size, tiles, tile_rows);
}

struct BucketedLayout {
    size_t keys, products, table, totals, tile_rows, spare;
};
BucketedLayout bucketed_layout(idx_t nnz, size_t value_bytes) {
    const uint32_t tile_size = tile_size_for(nnz);
    const size_t tiles = tiles_of(nnz, tile_size);
    BucketedLayout l;
    size_t off = 0;
    const size_t places = tile_places(tile_size, kProducts, 8);
    l.keys = off; off += align_up(tiles * places * sizeof(uint16_t));
    l.products = off; off += align_up(tiles * places * value_bytes);
    l.table = off; off += align_up(256 * tiles * sizeof(uint32_t));
    l.totals = off; off += align_up(256 * sizeof(uint32_t));
    l.tile_rows = off; off += align_up((tiles + 1) * sizeof(uint32_t));
    l.spare = off;
    return l;
}

}  // namespace

bool bucketed_products_shape(idx_t n, uint32_t* shift) {
    const uint32_t bits = bit_length(n - 1);  // of the columns without their index base
    // fewer keys than that: the full sort is two short passes; more: a bucket's sums no longer fit in LDS
    if (bits < kBucketMinKeyBits || bits > 8 + kBucketMaxShift) return false;
    *shift = bits - 8;
    return true;
}

size_t bucketed_products_workspace_bytes(idx_t nnz, size_t value_bytes) { return bucketed_layout(nnz, value_bytes).spare; }

// One partition by the top eight bits of the columns (index base taken off), the values multiplied by x[row] on the
// way.  What lies behind workspace_bytes is not touched.
void launch_bucketed_products(hipStream_t stream, idx_t m, idx_t n, idx_t nnz, const void* csr_val, const idx_t* row_ptr,
                              const idx_t* col, const void* x, size_t value_bytes, idx_t base, void* workspace,
                              size_t workspace_bytes, BucketedProducts* out) {
    uint32_t shift = 0;
    if (m == 0 || nnz == 0 || !bucketed_products_shape(n, &shift)) return;
    const BucketedLayout l = bucketed_layout(nnz, value_bytes);
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
    launch_row_starts(stream, in, tile_size, reinterpret_cast<uint32_t*>(w + l.tile_rows));
    auto* launch = value_bytes == 4 ? launch_partition<4, kProducts, 8, uint16_t> : launch_partition<8, kProducts, 8, uint16_t>;
    launch(stream, in, shift, 8, tile_size, w + l.keys, nullptr, w + l.products, table);
    out->keys = reinterpret_cast<const uint16_t*>(w + l.keys);
    out->products = w + l.products;
    out->table = table;
    out->totals = reinterpret_cast<uint32_t*>(w + l.totals);
    out->tiles = tiles_of(nnz, tile_size);
    out->tile_places = tile_places(tile_size, kProducts, 8);
    out->shift = shift;
    out->buckets = static_cast<uint32_t>((n - 1) >> shift) + 1;
    out->spare = w + l.spare;
    out->spare_bytes = workspace_bytes > l.spare ? workspace_bytes - l.spare : 0;
}

}  // namespace mcsp
