// A^T x without a preprocess call, for matrices of more than 2^14 and at most 18.8 million columns: the products
// value * x[row] are ordered by column bucket inside tiles of the matrix (launch_bucketed_products in partition.hip)
// and a bucket's sums are formed in LDS from its runs in all the tiles.
//
// The reference builds the transpose in the scratch buffer on every call and runs its row kernel on it
// (src/kernels/level2/spmv/mcsp_spmv_gpu.cpp:797-845).
#include "bucket_deal.h"
#include "partition_device.h"

namespace mcsp {

namespace {

using namespace partition_detail;

constexpr int kBlock = 256;
// One workgroup per bucket of neighbouring columns: the sums of the bucket's columns live in LDS as
// doubles (fp32 products are widened: ds_add_f64 runs at four times the rate of ds_add_f32 on this chip), and every
// column of the bucket is written at the end, with or without products.
// BUCKETS: rows of the table of runs.  With 1024 of them (more than 4.7 M columns) a run is 8 entries instead of 32 and
// 3072 of a tile's 11264 places may be padding (tiles of 4096 entries: 3072 of 7168), but a sort by the columns takes three times as long.
constexpr int kBucketBlock = 1024;

// Which part of which bucket a workgroup takes.  A bucket whose pairs number more than twice `share` (the mean of
// a bucket, rounded up) is dealt to several workgroups, ceil(count / share) of them, so that columns that crowd
// into a few buckets (a matrix sorted by degree) do not leave the work to a few CUs: workgroup b < BUCKETS takes the
// first part of bucket b, the workgroups from BUCKETS on the further parts, bucket by bucket.  The parts of a split
// bucket leave their sums as planes in `planes`, numbered in the same order, for bucket_merge_kernel.
struct BucketPart {
    uint32_t bucket;  // BUCKETS: none
    uint32_t part, parts;
    uint32_t plane;   // of part 0 of this bucket, when parts > 1
};
// every thread of the workgroup must call this (it holds barriers); s_parts: BUCKETS words of LDS
template <uint32_t BUCKETS>
__device__ __forceinline__ BucketPart bucket_part(uint32_t group, bool merge, const uint32_t* __restrict__ totals,
                                                  uint32_t share, uint32_t* s_parts, uint32_t* s_out) {
    for (uint32_t b = threadIdx.x; b < BUCKETS; b += blockDim.x) {
        const uint32_t count = totals[b];
        s_parts[b] = count / 2 > share ? (count + share - 1) / share : 1u;  // more than twice the share: split
    }
    __syncthreads();
    if (threadIdx.x < kWave) {  // the first wavefront: a few buckets per lane, prefix sums over the lanes
        constexpr uint32_t kMine = BUCKETS / kWave;
        const uint32_t lane = threadIdx.x;
        uint32_t parts[kMine], extra = 0, planes = 0;
#pragma unroll
        for (uint32_t k = 0; k < kMine; ++k) {
            parts[k] = s_parts[kMine * lane + k];
            extra += parts[k] - 1;
            planes += parts[k] > 1 ? parts[k] : 0;
        }
        uint32_t extra_upto = extra, planes_upto = planes;  // inclusive over lanes
#pragma unroll
        for (int d = 1; d < kWave; d *= 2) {
            const uint32_t e = __shfl_up(extra_upto, d, kWave), q = __shfl_up(planes_upto, d, kWave);
            if (lane >= static_cast<uint32_t>(d)) {
                extra_upto += e;
                planes_upto += q;
            }
        }
        uint32_t bucket = BUCKETS, part = 0;
        if (merge || group < BUCKETS) {
            bucket = group;
        } else {
            // the further part number `further` lies with the lane whose buckets hold it
            const uint32_t further = group - BUCKETS;
            const bool here = further >= extra_upto - extra && further < extra_upto;
            const uint64_t owner = __ballot(here);
            if (owner != 0) {
                const int src = __ffsll(static_cast<long long>(owner)) - 1;
                uint32_t left = further - __shfl(extra_upto - extra, src, kWave);
                uint32_t found = BUCKETS, found_part = 0;
#pragma unroll
                for (uint32_t k = 0; k < kMine; ++k) {
                    const uint32_t e = __shfl(parts[k], src, kWave) - 1;
                    if (found == BUCKETS) {
                        if (left < e) {
                            found = kMine * src + k;
                            found_part = left + 1;
                        } else {
                            left -= e;
                        }
                    }
                }
                bucket = found;
                part = found_part;
            }
        }
        // planes of the split buckets before `bucket`
        uint32_t plane = 0;
        if (bucket < BUCKETS) {
            const int src = bucket / kMine;
            plane = __shfl(planes_upto - planes, src, kWave);
#pragma unroll
            for (uint32_t k = 0; k < kMine; ++k) {
                const uint32_t q = __shfl(parts[k], src, kWave);
                if (k < bucket % kMine) plane += q > 1 ? q : 0;
            }
        }
        if (lane == 0) {
            s_out[0] = bucket;
            s_out[1] = part;
            s_out[2] = plane;
        }
    }
    __syncthreads();
    BucketPart p;
    p.bucket = s_out[0];
    p.part = s_out[1];
    p.plane = s_out[2];
    p.parts = p.bucket < BUCKETS ? s_parts[p.bucket] : 0;
    return p;
}


// A wavefront takes the runs of kGroupTiles neighbouring tiles at a time, a lane per run, and their entries in pieces of
// kPiece: with runs of 32 entries (8192 per tile, 256 buckets) that is just under one batch of eight pieces per lane.
constexpr int kPiece = kBucketRunPad;
static_assert(kPiece == 4, "a piece is a 16-byte load of fp32 products and an 8-byte load of keys");
constexpr uint32_t kGroupTiles = 57;
constexpr uint32_t kWindow = 1024;   // pieces of a group that are mapped to their runs together
constexpr uint32_t kWords = kWindow / kWave;
constexpr int kBatch = 8;            // pieces per lane in flight
constexpr uint32_t kHeavyGroup = 4 * kWindow;  // groups with more pieces are shared by the workgroup's wavefronts
constexpr uint32_t kMaxGroups = ((1ull << 32) / kBucketTileMin + kGroupTiles - 1) / kGroupTiles;

struct WaveRuns {
    unsigned long long begins[kWords];
    uint32_t delta[kWave];
};

template <typename T>
struct Piece { typedef T type __attribute__((ext_vector_type(kPiece))); };

// Adds the products of the windows first, first + step, ... of group g to the sums.  Returns the number of windows of
// the group.
template <typename T>
__device__ __forceinline__ uint32_t add_group(uint32_t word, uint32_t g, uint32_t tile_places, uint32_t first, uint32_t step,
                                          WaveRuns& s, const uint16_t* __restrict__ keys, const T* __restrict__ products,
                                          uint32_t first_column, uint32_t last, double* s_acc) {
    typedef typename Piece<T>::type piece_t;
    typedef uint32_t key_piece_t __attribute__((ext_vector_type(2)));
    const key_piece_t* key_pieces = reinterpret_cast<const key_piece_t*>(keys);
    const piece_t* product_pieces = reinterpret_cast<const piece_t*>(products);
    const uint32_t lane = threadIdx.x % kWave;
    // a column's place in the bucket from its low half (what pads a run has any, and a product of 0)
    auto add = [&](uint32_t low_half, T product) {
        unsafeAtomicAdd(&s_acc[min(low_half - first_column & 0xffffu, last)], static_cast<double>(product));
    };
    const uint32_t length = run_length(word) / kPiece;
    const uint32_t end = wave_inclusive_sum(length);
    const uint32_t begin = end - length;
    const uint32_t total = __builtin_amdgcn_readlane(end, kWave - 1);
    const uint64_t runs = __ballot(length != 0);
    const uint32_t number = bits_below_lane(static_cast<uint32_t>(runs), static_cast<uint32_t>(runs >> 32));
    // place of a piece = its place among the group's pieces plus its run's delta (mod 2^32)
    if (length != 0) s.delta[number] = (g * kGroupTiles + lane) * (tile_places / kPiece) + run_place(word) / kPiece - begin;
    for (uint32_t w0 = first * kWindow; w0 < total; w0 += step * kWindow) {
        const uint32_t count = min(total - w0, kWindow);
        // A bit in front of every piece at which a run begins, the window's first piece left out: the bits below a
        // piece's own, plus the run the window begins in, number its run.  (LDS operations of a wavefront complete in
        // order: no barrier between these lines.)
        __builtin_amdgcn_wave_barrier();
        if (lane < kWords) __hip_atomic_store(&s.begins[lane], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        const uint32_t at = begin - 1 - w0;  // wraps for runs that begin at or before w0
        if (length != 0 && begin > w0 && at < kWindow)
            __hip_atomic_fetch_or(&s.begins[at / kWave], 1ull << (at % kWave), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        const unsigned long long mine =
            lane < kWords ? __hip_atomic_load(&s.begins[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT) : 0ull;
        __builtin_amdgcn_wave_barrier();
        const uint32_t first_run = __popcll(__ballot(length != 0 && begin <= w0)) - 1;
        const uint32_t run_of_word = first_run + wave_inclusive_sum(__popcll(mine)) - __popcll(mine);
        const uint32_t rounds = (count + kWave - 1) / kWave;
        for (uint32_t r0 = 0; r0 < rounds; r0 += kBatch) {
            key_piece_t key[kBatch];
            piece_t p[kBatch];
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                const uint32_t r = r0 + i < rounds ? r0 + i : rounds - 1;
                const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(mine), r);
                const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(mine >> 32), r);
                const uint32_t run = __builtin_amdgcn_readlane(run_of_word, r) + bits_below_lane(lo, hi);
                // (no run begins behind the window's last piece: lanes past it find that piece's run)
                const uint32_t place = s.delta[run] + w0 + min(r * kWave + lane, count - 1);
                // (plain loads: the lines at the ends of a run are shared with the neighbouring buckets' workgroups on
                // this XCD, and a streaming load drops them from L2 before they come for them: 178 -> 153 us)
                key[i] = key_pieces[place];
                p[i] = product_pieces[place];
            }
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                if ((r0 + i) * kWave + lane < count) {
                    add(key[i].x, p[i].x);
                    add(key[i].x >> 16, p[i].y);
                    add(key[i].y, p[i].z);
                    add(key[i].y >> 16, p[i].w);
                }
            }
        }
    }
    return (total + kWindow - 1) / kWindow;
}

template <typename T, uint32_t BUCKETS>
__global__ __launch_bounds__(kBucketBlock) void bucket_sums_kernel(idx_t n, ColumnBuckets columns, uint32_t tiles,
                                                                  uint32_t tile_places, uint32_t share,
                                                                  const uint32_t* __restrict__ totals,
                                                                  const uint32_t* __restrict__ table,
                                                                  const uint16_t* __restrict__ keys,
                                                                  const T* __restrict__ products, T* __restrict__ y,
                                                                  double* __restrict__ planes, T alpha, T beta,
                                                                  uint32_t xcds) {
    constexpr uint32_t kWaves = kBucketBlock / kWave;
    extern __shared__ __align__(16) unsigned char s_raw[];
    __shared__ WaveRuns s_runs[kWaves];
    __shared__ uint32_t s_heavy[(kMaxGroups + 31) / 32];
    __shared__ uint32_t s_parts[BUCKETS];
    __shared__ uint32_t s_mine[3];
    double* s_acc = reinterpret_cast<double*>(s_raw);
    const uint32_t tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
    // Neighbouring buckets go to one XCD: their runs are neighbours in every tile and share lines at the ends.
    uint32_t block = blockIdx.x;
    if (block < BUCKETS && BUCKETS % xcds == 0 && gridDim.x >= BUCKETS) block = block % xcds * (BUCKETS / xcds) + block / xcds;
    // a workgroup whose own bucket is in one piece (the common case) need not look at the others
    BucketPart mine = {block, 0, 1, 0};
    if (block >= BUCKETS || totals[block] / 2 > share)  // the same for the whole workgroup
        mine = bucket_part<BUCKETS>(block, false, totals, share, s_parts, s_mine);
    const uint32_t bucket = mine.bucket;
    if (bucket >= BUCKETS) return;  // whole workgroup: no further part left for it
    const uint32_t first = bucket * columns.width;
    if (first >= n) return;  // whole workgroup: no such bucket
    const uint32_t width = min(columns.width, n - first);
    for (uint32_t r = tid; r < width; r += kBucketBlock) s_acc[r] = 0.0;
    const uint32_t groups = (tiles + kGroupTiles - 1) / kGroupTiles;
    for (uint32_t r = tid; r < (groups + 31) / 32; r += kBucketBlock) s_heavy[r] = 0;
    __syncthreads();
    const uint32_t* row = table + static_cast<uint64_t>(bucket) * tiles;
    auto words_of = [&](uint32_t g) {
        const uint32_t t = g * kGroupTiles + lane;
        return lane < kGroupTiles && t < tiles ? row[t] : 0u;
    };
    // light groups are dealt to the parts (bucket_deal.h), heavy ones are shared by all wavefronts of all parts
    uint32_t word = wave < groups ? words_of(wave) : 0u;
    for (uint32_t g = wave; g < groups; g += kWaves) {
        const uint32_t next = g + kWaves < groups ? words_of(g + kWaves) : 0u;  // on its way while this group is added
        const uint32_t total = __builtin_amdgcn_readlane(wave_inclusive_sum(run_length(word) / kPiece), kWave - 1);
        if (total > kHeavyGroup) {
            if (lane == 0) atomicOr(&s_heavy[g / 32], 1u << (g % 32));
        } else if (total != 0 && part_of_group(g, kWaves, mine.parts) == mine.part) {
            add_group(word, g, tile_places, 0, 1, s_runs[wave], keys, products, first, width - 1, s_acc);
        }
        word = next;
    }
    __syncthreads();
    const uint32_t takers = mine.parts * kWaves;
    uint32_t turn = mine.part * kWaves + wave;  // which of the next group's windows is this wavefront's first
    for (uint32_t w = 0; w < (groups + 31) / 32; ++w) {
        uint32_t left = s_heavy[w];
        while (left != 0) {
            const uint32_t b = __ffs(left) - 1;
            left &= left - 1;
            const uint32_t windows = add_group(words_of(w * 32 + b), w * 32 + b, tile_places, turn, takers, s_runs[wave], keys,
                                               products, first, width - 1, s_acc);
            turn = (turn + takers - windows % takers) % takers;
        }
    }
    __syncthreads();
    if (mine.parts > 1) {  // whole workgroup
        double* out = planes + (static_cast<uint64_t>(mine.plane) + mine.part) * columns.width;
        for (uint32_t r = tid; r < width; r += kBucketBlock) out[r] = s_acc[r];
        return;
    }
    for (uint32_t r = tid; r < width; r += kBucketBlock) {
        const uint64_t c = first + r;
        const T s = alpha * static_cast<T>(s_acc[r]);
        y[c] = beta == T(0) ? s : s + beta * y[c];
    }
}

// totals[d] = entries of digit d in all tiles.  A workgroup per digit.
__global__ __launch_bounds__(kBlock) void bucket_totals_kernel(uint32_t tiles, const uint32_t* __restrict__ table,
                                                               uint32_t* __restrict__ totals) {
    __shared__ uint32_t s_wave[kBlock / kWave];
    const uint32_t* row = table + static_cast<uint64_t>(blockIdx.x) * tiles;
    constexpr int kAhead = 8;
    uint32_t sum = 0;
    for (uint32_t t0 = 0; t0 < tiles; t0 += kAhead * kBlock) {
        uint32_t got[kAhead];
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
            const uint32_t t = t0 + k * kBlock + threadIdx.x;
            got[k] = row[t < tiles ? t : tiles - 1];
        }
#pragma unroll
        for (int k = 0; k < kAhead; ++k) sum += t0 + k * kBlock + threadIdx.x < tiles ? run_length(got[k]) : 0u;
    }
    uint32_t all = 0;
    block_exclusive_sum<kBlock>(sum, s_wave, &all);
    if (threadIdx.x == 0) totals[blockIdx.x] = all;
}

// The columns of the buckets that were dealt to several workgroups: their planes added up.  kBucketMergeParts
// workgroups per bucket, each with its share of the bucket's columns; those of a bucket in one piece have nothing
// to do.
constexpr uint32_t kBucketMergeParts = 16;
template <typename T, uint32_t BUCKETS>
__global__ __launch_bounds__(kBlock) void bucket_merge_kernel(idx_t n, ColumnBuckets columns, uint32_t share,
                                                              const uint32_t* __restrict__ totals,
                                                              const double* __restrict__ planes, T* __restrict__ y,
                                                              T alpha, T beta) {
    __shared__ uint32_t s_parts[BUCKETS];
    __shared__ uint32_t s_mine[3];
    if (totals[blockIdx.x / kBucketMergeParts] / 2 <= share) return;  // whole workgroup
    const BucketPart mine = bucket_part<BUCKETS>(blockIdx.x / kBucketMergeParts, true, totals, share, s_parts, s_mine);
    const uint32_t first = mine.bucket * columns.width;
    if (first >= n || mine.parts < 2) return;  // whole workgroup
    const uint32_t width = min(columns.width, n - first);
    const uint32_t slice = (width + kBucketMergeParts - 1) / kBucketMergeParts;
    const uint32_t r0 = (blockIdx.x % kBucketMergeParts) * slice;
    const uint32_t r1 = r0 + slice < width ? r0 + slice : width;
    const double* in = planes + static_cast<uint64_t>(mine.plane) * columns.width;
    for (uint32_t r = r0 + threadIdx.x; r < r1; r += kBlock) {
        const uint64_t c = first + r;
        double sum = 0.0;
        for (uint32_t part = 0; part < mine.parts; ++part) sum += in[static_cast<uint64_t>(part) * columns.width + r];
        const T s = alpha * static_cast<T>(sum);
        y[c] = beta == T(0) ? s : s + beta * y[c];
    }
}

template <typename T, uint32_t BUCKETS>
bool launch_sums(hipStream_t stream, idx_t n, const BucketedProducts& b, T* y, T alpha, T beta) {
    const size_t lds = sizeof(double) * b.columns.width;
    hipLaunchKernelGGL(bucket_totals_kernel, dim3(BUCKETS), dim3(kBlock), 0, stream, b.tiles, b.table, b.totals);
    // A bucket with more than twice `share` entries is dealt to several workgroups, ceil(count / share) of them.  share
    // is the mean of a bucket, so that at most BUCKETS further workgroups are needed, or more where the spare scratch is
    // short: the split buckets leave fewer than 2 * entries / share planes (one per `share` entries, and one more for
    // each of the fewer than entries / share buckets that are split at all).  Entries: with the padding of the runs.
    const uint64_t max_planes = b.spare_bytes / lds;
    const bool split = max_planes >= 4;
    const uint64_t entries = static_cast<uint64_t>(b.tiles) * b.tile_places;
    uint64_t share = 0xffffffffull;  // no bucket holds more
    if (split) {
        share = (entries + BUCKETS - 1) / BUCKETS;
        const uint64_t fits = (2 * entries + max_planes - 1) / max_planes + 1;
        share = share > fits ? share : fits;
        share = share < 0xffffffffull ? share : 0xffffffffull;
    }
    double* planes = static_cast<double*>(b.spare);
    if (!allow_dynamic_lds(reinterpret_cast<const void*>(bucket_sums_kernel<T, BUCKETS>), lds)) return false;
    hipLaunchKernelGGL((bucket_sums_kernel<T, BUCKETS>), dim3(split ? 2 * BUCKETS : BUCKETS), dim3(kBucketBlock), lds,
                       stream, n, b.columns, b.tiles, b.tile_places, static_cast<uint32_t>(share),
                       static_cast<const uint32_t*>(b.totals), b.table, b.keys, static_cast<const T*>(b.products), y,
                       planes, alpha, beta, device_topology().xcds);
    if (split) {
        hipLaunchKernelGGL((bucket_merge_kernel<T, BUCKETS>), dim3(BUCKETS * kBucketMergeParts), dim3(kBlock), 0, stream, n,
                           b.columns, static_cast<uint32_t>(share), static_cast<const uint32_t*>(b.totals),
                           static_cast<const double*>(planes), y, alpha, beta);
    }
    return launches_taken();
}

}  // namespace

template <typename T>
bool launch_bucket_sums(hipStream_t stream, idx_t n, const BucketedProducts& b, T* y, T alpha, T beta) {
    if (b.columns.width == 0 || b.columns.width > kBucketMaxColumns) return false;
    if (b.columns.bits == kBucketFewBits) return launch_sums<T, 1u << kBucketFewBits>(stream, n, b, y, alpha, beta);
    if (b.columns.bits == kBucketManyBits) return launch_sums<T, 1u << kBucketManyBits>(stream, n, b, y, alpha, beta);
    return false;
}

template bool launch_bucket_sums<float>(hipStream_t, idx_t, const BucketedProducts&, float*, float, float);
template bool launch_bucket_sums<double>(hipStream_t, idx_t, const BucketedProducts&, double*, double, double);

}  // namespace mcsp
