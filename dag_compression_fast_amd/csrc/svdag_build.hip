// svdag_build.hip -- gfx950 kernels of the bottom-up DAG build.
//
// Reference path (src/DAGCompression.cu):
//   SelectUnique + leaf ReduceByKey  :1035-1068  -> k_cell_reduce /
//       k_cell_compact (keys grouped by 64^3 cell, code >> 18, with known cell
//       starts) or k_leaf_reduce / k_leaf_compact (keys grouped by code >> 15):
//       one pass over the keys; duplicates OR into the same 4^3 mask, so no
//       separate unique step is needed
//   SortLevel(Leaves)               :1070-1071  -> k_table_clear / k_leaf_insert
//       (hash table keyed by the mask) + a sample sort of its occupied slots
//       (k_leaf_sample, k_order_*)
//   ExtractLevel + ComputeHashes    :916-974, :827-833 -> k_level_count /
//       k_level_build (parent masks, child ranks, Murmur hash, insert into the
//       level's dedup table)
//   SortLevel(level)                :864-914    -> k_extract_count /
//       k_level_extract (ordered linear-probing table: home slot = top bits of
//       the hash, so sorting each probe cluster orders the whole table; rank =
//       occupied slots before it)
//   CreateFinalDAG / WriteTo        :834-861, :1550-1610 -> k_final_count /
//       k_final_positions / k_final_write
// Every compaction is reduce-then-scan: a count kernel writes one count per
// part (the consecutive tiles of one workgroup of the main kernel), and each
// workgroup of the main kernel sums the counts before its own; k_leaf_compact
// takes its offsets from a one-workgroup scan (k_scan_counts).  No workgroup
// waits on another; element counts come from device memory, so the build runs without
// host round trips.
#include "svdag_device.hpp"
#include "svdag_internal.hpp"

#include <algorithm>
#include <type_traits>

namespace svdag {

namespace {

constexpr int kThreads = 256;
constexpr int kScanThreads = 1024;
constexpr int kScanItems = 4;

__host__ int grid_for(uint64_t tiles, int per_cu)
{
    const uint64_t cap = uint64_t(device_cu_count()) * per_cu;
    return int(std::max<uint64_t>(1, std::min<uint64_t>(tiles, cap)));
}

__global__ void k_fill_u64(uint64_t* __restrict__ p, uint64_t count, uint64_t value, uint64_t set_at,
                           uint64_t set_value)
{
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += stride)
        p[i] = i == set_at ? set_value : value;
}

// Exclusive scan of counts[0, ntiles) into offsets, ntiles = ceil(*items / per_tile);
// the grand total goes to *total_out when given.  One workgroup.
__global__ __launch_bounds__(kScanThreads) void k_scan_counts(const uint32_t* __restrict__ counts,
                                                              uint64_t* __restrict__ offsets,
                                                              const uint64_t* __restrict__ items, uint64_t per_tile,
                                                              uint64_t* __restrict__ total_out, uint64_t items_host)
{
    __shared__ uint64_t s_scan[kScanThreads / kWave];
    const uint64_t ntiles = ((items ? *items : items_host) + per_tile - 1) / per_tile;
    uint64_t running = 0;
    // kScanItems consecutive counts per thread per block scan.
    for (uint64_t chunk = 0; chunk < ntiles; chunk += uint64_t(kScanThreads) * kScanItems) {
        const uint64_t i0 = chunk + uint64_t(threadIdx.x) * kScanItems;
        uint32_t v[kScanItems];
        uint64_t sum = 0;
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            v[k] = i0 + k < ntiles ? counts[i0 + k] : 0u;
            sum += v[k];
        }
        uint64_t total;
        uint64_t run = running + block_exclusive_scan64<kScanThreads>(sum, s_scan, total);
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            if (i0 + k < ntiles) offsets[i0 + k] = run;
            run += v[k];
        }
        running += total;
    }
    if (total_out && threadIdx.x == 0) *total_out = running;
}

// Parts of a stage: workgroup b of P takes the consecutive tiles [t0, t1) of
// ntiles.  A tile t lies in part part_of_tile.
__device__ __forceinline__ void part_tiles(uint64_t ntiles, uint32_t b, uint32_t P, uint64_t& t0, uint64_t& t1)
{
    t0 = ntiles * b / P;
    t1 = ntiles * (uint64_t(b) + 1) / P;
}
__device__ __forceinline__ uint32_t part_of_tile(uint64_t ntiles, uint64_t t, uint32_t P)
{
    return uint32_t(((t + 1) * P - 1) / ntiles);
}

// Sum of the parts before this workgroup's (two barriers; every thread must
// call it).  At most kMaxParts words from L2: a scan kernel between the count
// and the main kernel took 4.6 us at the smallest, 27 us over 65536 tiles.
__device__ __forceinline__ uint64_t parts_before(const uint32_t* __restrict__ parts, uint64_t* scratch)
{
    uint64_t sum = 0;
    for (uint32_t i = threadIdx.x; i < blockIdx.x; i += kThreads) sum += parts[i];
    return block_reduce_sum<kThreads>(sum, scratch);
}

// ---------------------------------------------------------------------------
// Leaf reduce: keys sorted by code >> (6 + r), with r = min(9, 3 * depth - 6)
// -> (code >> 6, OR of 1 << (code & 63)) per 4^3 block, in code order.
// A run of keys with equal code >> (6 + r) (a "block group", at most 2^r
// leaves) is reduced in a wave-private LDS table of 2^r words indexed by the
// leaf's low r bits; the keys of a group may come in any order, so the sort
// skips the low r bits of the leaf code as well as the 6 voxel bits.
// Wave work unit: a chunk of kPackTileItems consecutive keys.  A wave owns the
// groups whose first key lies in its chunk (reading on past the chunk to
// finish its last one) and writes their leaves into its own region of
// kPackTileItems + 512 entries: groups inside the chunk have at most one leaf
// per key, the last group at most 2^r leaves.  k_leaf_compact then moves the
// regions together.
// ---------------------------------------------------------------------------
constexpr uint32_t kReduceChunk = uint32_t(kPackTileItems);
constexpr uint32_t kReduceTable = 1u << kLeafGroupBits;
constexpr uint32_t kReduceRegion = uint32_t(kLeafRegionItems);
static_assert(kReduceRegion == kReduceChunk + kReduceTable, "region bound");
// Groups of 64 keys loaded together: 2 KiB of keys per wave in flight.
template <typename K>
constexpr int kReduceGroups = int(2048 / (kWave * sizeof(K)));
constexpr int kReduceWaves = kThreads / kWave;
static_assert(kReduceTable == 8 * kWave, "one lane holds the 8 leaves of one parent");

// Value of lane l (a wave-uniform l), as a scalar.
__device__ __forceinline__ uint64_t readlane64(uint64_t v, uint32_t l)
{
    const uint32_t lo = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(v)), int(l)));
    const uint32_t hi = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(v >> 32)), int(l)));
    return uint64_t(hi) << 32 | lo;
}

// G groups of 64 raw keys from `base`; indices past the end read
// the last key (n >= 1), and the caller ignores those lanes.  No use of the
// values here, so the loads stay in flight until the keys are needed.
template <typename K, int G, typename KC>
__device__ __forceinline__ void load_groups(const K* __restrict__ sorted, uint64_t base, uint64_t n,
                                            KC (&k)[G])
{
    const uint32_t lane = lane_id();
#pragma unroll
    for (int g = 0; g < G; ++g)  // read once: non-temporal
        k[g] = KC(__builtin_nontemporal_load(sorted + min(base + g * kWave + lane, n - 1)));
}

// Lane l's value of v (wave-uniform result), for 32- and 64-bit values.
__device__ __forceinline__ uint32_t readlane_of(uint32_t v, uint32_t l)
{
    return uint32_t(__builtin_amdgcn_readlane(int(v), int(l)));
}
__device__ __forceinline__ uint64_t readlane_of(uint64_t v, uint32_t l) { return readlane64(v, l); }
__device__ __forceinline__ uint32_t shfl_up_of(uint32_t v) { return uint32_t(__shfl_up(int(v), 1, kWave)); }
__device__ __forceinline__ uint64_t shfl_up_of(uint64_t v) { return __shfl_up(v, 1, kWave); }

// Bucket of position p among Morton-ordered buckets with starts start(0..num)
// (start(num) > p): the last b >= lo with start(b) <= p (empty buckets share
// their start with the next one).
template <typename Start>
__device__ __forceinline__ uint64_t bucket_of(const Start& start, uint64_t lo, uint64_t num, uint64_t p)
{
    uint64_t hi = num;
    while (hi - lo > 1) {
        const uint64_t mid = (lo + hi) / 2;
        if (start(mid) <= p) lo = mid;
        else hi = mid;
    }
    return lo;
}

constexpr uint32_t kLdsBuckets = 512;  // bucket tables up to this size are staged in LDS

// Where the leaf reduce finds bucket starts: no buckets (keys are codes), a
// copy in LDS (small tables), or the table in global memory.
enum BucketMode { kBucketsNone = 0, kBucketsLds = 1, kBucketsGlobal = 2 };

// BM != kBucketsNone: 32-bit bucket-local keys (see launch_leaf_reduce); each
// wave keeps the bucket of its current position and its end, so a batch inside
// one bucket takes the prefix from a register; batches that cross a bucket end
// (a few per bucket) search per lane.
template <typename K, int BM>
__global__ __launch_bounds__(kThreads) void k_leaf_reduce(const K* __restrict__ sorted,
                                                          const uint64_t* __restrict__ n_ptr, uint64_t code_mask,
                                                          uint32_t r, uint64_t* __restrict__ reg_code,
                                                          uint64_t* __restrict__ reg_mask,
                                                          uint32_t* __restrict__ counts,
                                                          unsigned long long* __restrict__ err, ChunkPrefix bk)
{
    __shared__ uint64_t s_tab[kReduceWaves][kReduceTable];
    constexpr int G = kReduceGroups<K>;
    constexpr bool BUCKETED = BM != kBucketsNone;
    // Keys and group indices in registers: 32-bit for 32-bit keys (a group
    // index then has at most 32 - 15 local bits and the bucket's 12 above
    // them), 64-bit otherwise.
    using KC = std::conditional_t<sizeof(K) == 4, uint32_t, uint64_t>;
    // Bucket starts (positions < 2^30) staged in LDS when the table is small.
    __shared__ uint32_t s_bstart[BM == kBucketsLds ? kLdsBuckets + 1 : 1];
    if constexpr (BM == kBucketsLds) {
        for (uint32_t i = threadIdx.x; i <= bk.num_chunks; i += kThreads) s_bstart[i] = uint32_t(bk.offsets[i]);
        __syncthreads();
    }
    auto start_of = [&](uint64_t b) -> uint64_t {
        if constexpr (BM == kBucketsLds) return s_bstart[b];
        else return bk.offsets[b];
    };
    const uint32_t lane = lane_id();
    // The wave index as a scalar, so that the chunk loop and the group
    // bookkeeping below compile to scalar control flow.
    const uint32_t w = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x / kWave)));
    uint64_t* const tab = s_tab[w];
#pragma unroll
    for (int e = 0; e < 8; ++e) tab[e * kWave + lane] = 0ull;
    __builtin_amdgcn_wave_barrier();
    const uint64_t n = *n_ptr;
    const uint64_t nchunks = (n + kReduceChunk - 1) / kReduceChunk;
    const uint32_t sh = 6 + r;
    const uint32_t low_mask = (1u << r) - 1u;
    bool overflow = false;

    for (uint64_t chunk = uint64_t(blockIdx.x) * kReduceWaves + w; chunk < nchunks;
         chunk += uint64_t(gridDim.x) * kReduceWaves) {
        const uint64_t c0 = chunk * kReduceChunk;
        const uint64_t c1 = min(c0 + kReduceChunk, n);
        uint64_t* const oc = reg_code + chunk * kReduceRegion;
        uint64_t* const om = reg_mask + chunk * kReduceRegion;
        uint32_t written = 0;
        // Bucket of the chunk's current batch and that bucket's end.
        uint64_t cur = 0, cur_end = ~0ull;
        if constexpr (BUCKETED) {
            cur = bucket_of(start_of, 0, bk.num_chunks, c0 > 0 ? c0 - 1 : 0);
            cur_end = start_of(cur + 1);
        }
        // Group indices (code >> sh) of the batch of keys v at bb: the key's own
        // bits above sh, with its bucket above those (bucketed keys).
        const uint32_t gsh = BUCKETED ? bk.chunk_bits - sh : 0u;  // chunk_bits > sh
        auto group_of = [&](uint64_t bb, const KC (&v)[G], KC (&out)[G]) {
            if constexpr (BUCKETED) {
                const uint64_t last = min(bb + uint64_t(G) * kWave - 1, n - 1);
                if (last < cur_end) {
                    const KC pre = KC(cur) << gsh;
#pragma unroll
                    for (int g = 0; g < G; ++g) out[g] = pre | (v[g] >> sh);
                } else {
#pragma unroll
                    for (int g = 0; g < G; ++g) {
                        const uint64_t p = min(bb + uint64_t(g) * kWave + lane, n - 1);
                        out[g] = (KC(bucket_of(start_of, cur, bk.num_chunks, p)) << gsh) | (v[g] >> sh);
                    }
                    cur = bucket_of(start_of, cur, bk.num_chunks, last);
                    cur_end = start_of(cur + 1);
                }
            } else {
#pragma unroll
                for (int g = 0; g < G; ++g) out[g] = v[g] >> sh;
            }
        };
        // Group of the key before the chunk (~0 never equals a group index).
        KC prev_b = KC(~0ull);
        if (c0 > 0) {
            const KC pk = KC(sorted[c0 - 1]) & KC(code_mask);
            if constexpr (BUCKETED) prev_b = (KC(cur) << gsh) | (pk >> sh);  // cur: the bucket of c0 - 1
            else prev_b = pk >> sh;
        }
        bool open = false;  // a group owned by this wave is being accumulated
        KC cur_b = 0;
        bool done = false;

        // Writes the open group's leaves in order and clears the table.  Row e
        // of the table is read by lanes 0..63 (leaves 64e + lane), so a leaf's
        // output position is the count of nonzero rows' ballots before it.
        auto flush = [&]() {
            __builtin_amdgcn_wave_barrier();
            // A full table fits the region for valid bounds: the groups before
            // the last hold at most one leaf per chunk key, so written <= 4095.
            // Past that, an internal bound failed: reported, nothing written.
            const bool room = written + kReduceTable <= kReduceRegion;
            if (!room) overflow = true;
            // Row by row, with the per-row bookkeeping in vector registers:
            // this runs once per group and its scalar work had been about half
            // of the kernel's scalar instructions (the scalar unit is its
            // limit).
            uint32_t pos = written;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint64_t m = tab[e * kWave + lane];
                tab[e * kWave + lane] = 0ull;
                const uint64_t B = __ballot(m != 0ull);
                if (m && room) {
                    const uint32_t p = pos + uint32_t(__popcll(B & lanemask_lt()));
                    oc[p] = (uint64_t(cur_b) << r) | uint64_t(e * kWave + lane);
                    om[p] = m;
                }
                pos += uint32_t(__popcll(B));
            }
            if (room) written = pos;
            __builtin_amdgcn_wave_barrier();
            open = false;
        };

        KC k[G], nxt[G], gb[G];
        load_groups(sorted, c0, n, k);
        // No load may be pending at the loop head (see the wait at its end).
        __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
#pragma unroll
        for (int g = 0; g < G; ++g) k[g] &= KC(code_mask);
        group_of(c0, k, gb);
        for (uint64_t base = c0; !done; base += uint64_t(G) * kWave) {
            // The next batch of the chunk is in flight while this one is reduced.
            const uint64_t next = base + uint64_t(G) * kWave;
            const bool prefetch = next < c1;
            if (prefetch) load_groups(sorted, next, n, nxt);
            // Group starts of the whole batch first: a lane starts a group when
            // its group index differs from the previous lane's (lane 0: from
            // the previous batch group's last lane).  A shuffle and a ballot
            // for every batch group: the shortcut of comparing the first and
            // last lanes (no start inside when they agree) cost more scalar
            // work and a branch than it saved.  Lanes past the end repeat the
            // last key: they never start a group, and OR-ing their bit again is
            // harmless.
            uint64_t H[G];
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const KC b = gb[g];
                KC pb = shfl_up_of(b);
                if (lane == 0) pb = prev_b;
                H[g] = __ballot(b != pb);
                prev_b = readlane_of(b, kWave - 1);
            }
            // A batch that ends before both the chunk's and the keys' end (all
            // but the last of a chunk) cannot end the wave's work: FAST drops
            // the per-group end checks (scalar work; the scalar unit is this
            // kernel's limit).
            auto reduce_batch = [&](auto fast_tag) {
                constexpr bool FAST = decltype(fast_tag)::value;
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    if (!FAST && done) break;
                    const uint64_t gi = base + uint64_t(g) * kWave;  // index of lane 0's key
                    const KC key = k[g];
                    uint64_t* const word = &tab[uint32_t(key >> 6) & low_mask];
                    const uint64_t bit = 1ull << (uint32_t(key) & 63u);
                    uint64_t heads = H[g];
                    const bool keys_end = !FAST && gi + kWave >= n;  // the last key is in this batch group
                    // Segments [lo, next start), then [lo, 64): lanes before the first
                    // start continue the open group, or one owned by an earlier wave
                    // when none is open.  One flush site (the open group ends at a
                    // start, or at the keys' end): every call site is a copy of it.
                    uint32_t lo = 0;
                    while (true) {
                        const uint32_t hi = heads ? uint32_t(__ffsll((long long)heads) - 1) : uint32_t(kWave);
                        if (open && lane >= lo && lane < hi) atomicOr((unsigned long long*)word, bit);
                        const bool last = hi == uint32_t(kWave);
                        if (open && (!last || keys_end)) flush();
                        if (last) {
                            // The keys end here, or no group starts in the chunk.
                            if (!FAST && (keys_end || (!open && gi + kWave >= c1))) done = true;
                            break;
                        }
                        if (!FAST && gi + hi >= c1) {
                            done = true;
                            break;
                        }
                        open = true;
                        cur_b = readlane_of(gb[g], hi);
                        heads &= heads - 1ull;
                        lo = hi;
                    }
                }
            };
            if (next < c1 && next < n) reduce_batch(std::true_type{});
            else reduce_batch(std::false_type{});
            if (done) break;
            if (!prefetch) load_groups(sorted, next, n, nxt);
            // Settle every load here (vmcnt 0, other counters left alone): the
            // next batch's keys are then complete at the loop head, so the
            // batch's first uses do not wait behind the prefetch issued there.
            __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
#pragma unroll
            for (int g = 0; g < G; ++g) k[g] = nxt[g] & KC(code_mask);
            group_of(next, k, gb);
        }
        if (lane == 0) counts[chunk] = written;
    }
    if (overflow && lane == 0) atomicOr(err, (unsigned long long)kErrInternal);
}

// Region of chunk c (counts[c] leaves) -> lp_code / lp_mask at offsets[c].
// One wave per chunk.  A total beyond the capacity (distinct leaves never
// exceed it) is reported, not written.
__global__ __launch_bounds__(kThreads) void k_leaf_compact(const uint64_t* __restrict__ reg_code,
                                                           const uint64_t* __restrict__ reg_mask,
                                                           const uint32_t* __restrict__ counts,
                                                           const uint64_t* __restrict__ offsets,
                                                           const uint64_t* __restrict__ n_ptr,
                                                           uint64_t* __restrict__ lp_code,
                                                           uint64_t* __restrict__ lp_mask, uint64_t capacity,
                                                           unsigned long long* __restrict__ err)
{
    const uint32_t lane = lane_id();
    const uint64_t nchunks = (*n_ptr + kReduceChunk - 1) / kReduceChunk;
    for (uint64_t chunk = uint64_t(blockIdx.x) * kReduceWaves + threadIdx.x / kWave; chunk < nchunks;
         chunk += uint64_t(gridDim.x) * kReduceWaves) {
        const uint32_t cnt = counts[chunk];
        const uint64_t dst = offsets[chunk];
        const uint64_t src = chunk * kReduceRegion;
        if (dst + cnt > capacity) {
            if (lane == 0) atomicOr(err, (unsigned long long)kErrInternal);
            continue;
        }
        for (uint32_t j = lane; j < cnt; j += kWave) {
            lp_code[dst + j] = reg_code[src + j];
            lp_mask[dst + j] = reg_mask[src + j];
        }
    }
}

// ---------------------------------------------------------------------------
// Leaf reduce of keys grouped by 64^3 cell (code >> kCellShift) with known cell
// starts: one workgroup ORs a cell's keys into a table of its 4096 leaves in
// LDS (32 KB; four workgroups of 8 waves per CU) and writes the leaves present
// in order.  Against the 32^3 groups of k_leaf_reduce the sort orders 3 bits
// less (one pass instead of two up to depth 9 in a chunk), no wave looks for
// group starts, and the table words are 32 bits wide (64-bit LDS atomics take
// twice the bank cycles).  Bound by the keys' read and the LDS atomics where
// cells are full (512^3 noise, 67M keys: 304 -> 56 us, with 268 us of sort
// saved; 2048^3 triangles 153 -> 125), by the two barriers and the table pass a
// cell where they are not (512 chunks, 645 keys a cell: 364 -> 390 us, with 640
// us of sort saved; 690 before the next cell's keys were loaded ahead).  Full
// rounds of keys go without their guards (138 -> 125 us of the triangles);
// registers are held to 64 for the fourth workgroup per CU, which gains 26 us of
// the chunks and loses 18 of 1024^3 noise (540).
// A cell of k keys emits at most min(k, 4096) leaves, so a run of cells writes
// into its own keys' positions of the regions; codes there are 32-bit, local to
// the run.
// ---------------------------------------------------------------------------
constexpr int kCellThreads = 512;
constexpr int kCellWaves = kCellThreads / kWave;
constexpr int kCellKeys = 8;  // keys per thread in flight
constexpr int kCellRows = int(kCellLeaves) / kCellThreads;
static_assert(kCellRows * kCellThreads == int(kCellLeaves) && kMaxRunCells < kWave, "rows and starts per lane");

__global__ __launch_bounds__(kCellThreads, 8) void k_cell_reduce(CellArgs a, const uint64_t* __restrict__ n_ptr)
{
    __shared__ uint64_t s_tab[kCellLeaves];
    __shared__ uint32_t s_cnt[kCellWaves];
    uint32_t* const tab = reinterpret_cast<uint32_t*>(s_tab);
    const uint32_t lane = lane_id();
    const uint32_t w = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x / kWave)));
    for (uint32_t i = threadIdx.x; i < kCellLeaves; i += kCellThreads) s_tab[i] = 0ull;
    __syncthreads();
    const uint32_t n = uint32_t(*n_ptr);
    const uint64_t runs = cell_runs(a.cells, a.run_cells);
    // Bounds of a run's cells: lane l holds cell l's start (l == cells: the last
    // one's end).  No keys (or offsets a check rejected): every cell is empty.
    auto bounds_of = [&](uint64_t run) -> uint32_t {
        const uint64_t c = run * a.run_cells + min(lane, a.run_cells);
        return n != 0 && run < runs && c < a.cells ? a.starts[c] : n;
    };
    // Walk over the workgroup's cells that hold keys; the next run's bounds are
    // in flight while a run is walked.
    uint64_t run = blockIdx.x;
    uint32_t bound = bounds_of(run), ahead = bounds_of(run + gridDim.x);
    uint64_t todo = 0;  // cells of the run left to do
    bool fresh = true;  // no cell of the run has been taken yet
    uint32_t cell = 0, s = 0, e = 0;
    auto cells_with_keys = [&]() -> uint64_t {
        const uint32_t end = uint32_t(__shfl_down(int(bound), 1, kWave));
        return __ballot(lane < a.run_cells && bound < end);
    };
    auto next_cell = [&]() -> bool {
        while (todo == 0) {
            if (run >= runs) return false;
            if (fresh && threadIdx.x == 0) a.run_counts[run] = 0;  // no keys at all
            run += gridDim.x;
            bound = ahead;
            ahead = bounds_of(run + gridDim.x);
            todo = run < runs ? cells_with_keys() : 0ull;
            fresh = true;
        }
        fresh = false;
        cell = uint32_t(__builtin_amdgcn_readfirstlane(int(__ffsll((long long)todo) - 1)));
        todo &= todo - 1ull;
        s = uint32_t(__builtin_amdgcn_readlane(int(bound), int(cell)));
        e = uint32_t(__builtin_amdgcn_readlane(int(bound), int(cell + 1)));
        return true;
    };
    // The keys of one round, from p on; rows past the cell's end stay unread.
    uint32_t k[kCellKeys];
    auto load = [&](uint32_t p, uint32_t left) {
        if (left >= uint32_t(kCellThreads * kCellKeys)) {
#pragma unroll
            for (int i = 0; i < kCellKeys; ++i)
                k[i] = __builtin_nontemporal_load(a.keys + p + uint32_t(i) * kCellThreads + threadIdx.x);
            return;
        }
#pragma unroll
        for (int i = 0; i < kCellKeys; ++i)
            if (uint32_t(i) * kCellThreads < left)
                k[i] = __builtin_nontemporal_load(a.keys + p + min(uint32_t(i) * kCellThreads + threadIdx.x, left - 1));
    };
    todo = run < runs ? cells_with_keys() : 0ull;
    bool have = next_cell();
    if (have) load(s, e - s);
    uint32_t written = 0;
    while (have) {
        const uint64_t cur_run = run;
        const uint32_t cur_cell = cell;
        const uint32_t base = uint32_t(__builtin_amdgcn_readlane(int(bound), 0));
        for (uint32_t p = s;;) {
            const uint32_t left = e - p;
            auto add = [&](uint32_t key) { atomicOr(&tab[(key >> 5) & (2 * kCellLeaves - 1)], 1u << (key & 31u)); };
            if (left >= uint32_t(kCellThreads * kCellKeys)) {
#pragma unroll
                for (int i = 0; i < kCellKeys; ++i) add(k[i]);
            } else {
#pragma unroll
                for (int i = 0; i < kCellKeys; ++i)
                    if (uint32_t(i) * kCellThreads < left && uint32_t(i) * kCellThreads + threadIdx.x < left) add(k[i]);
            }
            if (left <= uint32_t(kCellThreads * kCellKeys)) break;
            p += kCellThreads * kCellKeys;
            load(p, e - p);
        }
        // The next cell's first keys are in flight while this one is written.
        have = next_cell();
        if (have) load(s, e - s);
        __syncthreads();
        // Wave w holds the leaves [w * 512, ...) in rows of 64.
        uint64_t m[kCellRows];
        uint32_t cnt = 0;
#pragma unroll
        for (int r = 0; r < kCellRows; ++r) {
            const uint32_t leaf = (w * kCellRows + uint32_t(r)) * kWave + lane;
            m[r] = s_tab[leaf];
            s_tab[leaf] = 0ull;
        }
#pragma unroll
        for (int r = 0; r < kCellRows; ++r) cnt += uint32_t(__popcll(__ballot(m[r] != 0ull)));
        if (lane == 0) s_cnt[w] = cnt;
        __syncthreads();
        uint32_t pos = base + written;
#pragma unroll
        for (int i = 0; i < kCellWaves; ++i) {
            const uint32_t x = s_cnt[i];
            pos += uint32_t(i) < w ? x : 0u;
            written += x;
        }
#pragma unroll
        for (int r = 0; r < kCellRows; ++r) {
            const uint64_t B = __ballot(m[r] != 0ull);
            if (m[r]) {
                const uint32_t q = pos + uint32_t(__popcll(B & lanemask_lt()));
                a.reg_code[q] = cur_cell * kCellLeaves + (w * kCellRows + uint32_t(r)) * kWave + lane;
                a.reg_mask[q] = m[r];
            }
            pos += uint32_t(__popcll(B));
        }
        if (!have || run != cur_run) {
            if (threadIdx.x == 0) a.run_counts[cur_run] = written;
            written = 0;
        }
    }
}

// The runs' leaves, concatenated.  A workgroup takes consecutive runs, a wave a
// run at a time, and finds its place by summing the counts before them (at most
// a few tens of KB from L2; a scan kernel and its launch cost more).
constexpr int kCompactAhead = 8;

__global__ __launch_bounds__(kThreads) void k_cell_compact(CellArgs a, const uint64_t* __restrict__ n_ptr,
                                                           uint64_t* __restrict__ total_out,
                                                           unsigned long long* __restrict__ err)
{
    __shared__ uint64_t s_red[kThreads / kWave];
    const uint64_t runs = cell_runs(a.cells, a.run_cells);
    const uint64_t first = runs * blockIdx.x / gridDim.x, last = runs * (blockIdx.x + 1) / gridDim.x;
    const uint32_t lane = lane_id(), w = threadIdx.x / kWave;
    uint64_t sum = 0;
    for (uint64_t i = threadIdx.x; i < first; i += kThreads) sum += a.run_counts[i];
    uint64_t before = block_reduce_sum<kThreads>(sum, s_red);
    const bool any = *n_ptr != 0;
    for (uint64_t batch = first; batch < last; batch += kWave) {
        // Lane l holds run batch + l's count, place and first key.
        const bool mine = any && batch + lane < last;
        const uint32_t count = mine ? a.run_counts[batch + lane] : 0u;
        const uint32_t start = mine ? a.starts[(batch + lane) * a.run_cells] : 0u;
        const uint32_t upto = wave_inclusive_scan(count);
        const uint32_t here = uint32_t(min(uint64_t(kWave), last - batch));
        for (uint32_t r = w; r < here; r += kThreads / kWave) {
            const uint32_t cnt = uint32_t(__shfl(int(count), int(r), kWave));
            const uint64_t src = uint32_t(__shfl(int(start), int(r), kWave));
            const uint64_t dst = before + uint32_t(__shfl(int(upto), int(r), kWave)) - cnt;
            uint64_t cell = (batch + r) * a.run_cells;
            if (a.chunk_ids)
                cell = uint64_t(a.chunk_ids[cell / a.chunk_cells]) * a.chunk_cells + cell % a.chunk_cells;
            const uint64_t high = cell * kCellLeaves;
            if (dst + cnt > a.lp_capacity) {
                if (lane == 0) atomicOr(err, (unsigned long long)kErrInternal);
                continue;
            }
            for (uint32_t j0 = 0; j0 < cnt; j0 += kWave * kCompactAhead) {
                uint32_t code[kCompactAhead];
                uint64_t mask[kCompactAhead];
#pragma unroll
                for (int q = 0; q < kCompactAhead; ++q) {
                    const uint32_t j = min(j0 + uint32_t(q) * kWave + lane, cnt - 1);
                    code[q] = a.reg_code[src + j];
                    mask[q] = a.reg_mask[src + j];
                }
#pragma unroll
                for (int q = 0; q < kCompactAhead; ++q) {
                    const uint32_t j = j0 + uint32_t(q) * kWave + lane;
                    if (j < cnt) {
                        a.lp_code[dst + j] = high + code[q];
                        a.lp_mask[dst + j] = mask[q];
                    }
                }
            }
        }
        before += uint32_t(__shfl(int(upto), kWave - 1, kWave));
    }
    if (blockIdx.x + 1 == gridDim.x && threadIdx.x == 0) *total_out = before;
}

// Clears slots [0, 2^lg + overflow) of each table, lg = max(8,
// ceil(log2(count << load_shift))), and records lg.
__device__ __forceinline__ void clear_tables(const TableClears& a)
{
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
    for (int t = 0; t < a.num; ++t) {
        const uint64_t cnt = *a.table[t].count;
        const uint32_t need = ceil_log2_u64((cnt ? cnt : 1ull) << a.load_shift);
        const uint32_t lg = need > 8u ? need : 8u;
        const uint64_t total = (1ull << lg) + a.table[t].overflow;
        uint64_t* __restrict__ keys = a.table[t].keys;
        if (blockIdx.x == 0 && threadIdx.x == 0) *a.table[t].log2_out = lg;
        for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total; i += stride) keys[i] = 0;
    }
}

__global__ void k_table_clear(TableClears a) { clear_tables(a); }

// Inserts key h (never 0) into a wrap-around table of 2^lg slots; `won` tells
// whether this call placed the key.  A probe never exceeds the table size; a
// full table reports kErrTableOverflow.
__device__ __forceinline__ uint32_t hashed_insert(uint64_t* __restrict__ tk, uint32_t lg, uint64_t h, bool& won,
                                                  unsigned long long* err)
{
    won = false;
    const uint64_t wrap = (1ull << lg) - 1;
    uint64_t slot = fmix64(h) >> (64 - lg);
    for (uint64_t probe = 0; probe <= wrap; ++probe, slot = (slot + 1) & wrap) {
        const uint64_t cur = probe_load(&tk[slot]);
        if (cur == h) return uint32_t(slot);
        if (cur == 0) {
            const uint64_t prev = atomicCAS((unsigned long long*)&tk[slot], 0ull, (unsigned long long)h);
            if (prev == 0) {
                won = true;
                return uint32_t(slot);
            }
            if (prev == h) return uint32_t(slot);
        }
    }
    atomicOr(err, (unsigned long long)kErrTableOverflow);
    return 0;
}

// Per-wave election among lanes holding equal 64-bit keys: every valid lane
// writes its lane index into the wave's LDS bucket (kElectBuckets words) for
// its key, one write wins; a lane whose bucket winner holds the same key is a
// follower of that winner and returns it, other lanes return themselves.
// Every lane of the wave must call it.
constexpr uint32_t kElectBuckets = 128;

__device__ __forceinline__ uint32_t elect_leader(uint64_t key, bool valid, uint32_t* buckets, bool& follower)
{
    const uint32_t lane = lane_id();
    const uint32_t bucket = uint32_t(fmix64(key)) & (kElectBuckets - 1);
    if (valid) buckets[bucket] = lane;
    __builtin_amdgcn_wave_barrier();
    const uint32_t winner = valid ? buckets[bucket] : lane;
    __builtin_amdgcn_wave_barrier();
    const uint64_t winner_key = __shfl(key, int(winner), kWave);
    follower = valid && winner != lane && winner_key == key;
    return follower ? winner : lane;
}

// Every leaf position's mask (never 0) enters the table and records its slot.
// A mask shared by many leaves (all-ones inside a solid, the same few patterns
// along a flat surface) would otherwise turn into a stream of probes and
// atomics on one table slot: a CU whose L1 still holds the slot's old 0
// settles each such probe with a CAS on the same L2 line.  So each wave first
// elects one lane per distinct mask: every lane writes its lane index into a
// per-wave LDS bucket chosen by its mask (one write wins), and a lane whose
// bucket winner holds the same mask takes the winner's slot instead of probing.
// Lanes that lose their bucket to another mask probe themselves.
constexpr int kInsertIpt = 8;

__global__ __launch_bounds__(kThreads) void k_leaf_insert(const uint64_t* __restrict__ lp_mask,
                                                          const uint64_t* __restrict__ count_ptr,
                                                          uint64_t* __restrict__ tk,
                                                          const uint32_t* __restrict__ log2_ptr,
                                                          uint32_t* __restrict__ lp_slot,
                                                          unsigned long long* __restrict__ err)
{
    __shared__ uint32_t s_elect[kThreads / kWave][kElectBuckets];
    const uint64_t n = *count_ptr;
    const uint32_t lg = *log2_ptr;
    const uint32_t lane = lane_id();
    uint32_t* const elect = s_elect[threadIdx.x / kWave];
    constexpr uint64_t per_round = uint64_t(kThreads) * kInsertIpt;
    // The loop bound is wave-uniform, so every lane of a wave takes part in the
    // shuffles below.
    for (uint64_t r0 = uint64_t(blockIdx.x) * per_round + (threadIdx.x & ~uint32_t(kWave - 1)); r0 < n;
         r0 += uint64_t(gridDim.x) * per_round) {
        // The round's masks are all in flight before the first insert (indices
        // past the end read the last mask and are not inserted).
        uint64_t masks[kInsertIpt];
#pragma unroll
        for (int j = 0; j < kInsertIpt; ++j) masks[j] = lp_mask[min(r0 + uint64_t(j) * kThreads + lane, n - 1)];
#pragma unroll
        for (int j = 0; j < kInsertIpt; ++j) {
            const uint64_t q = r0 + uint64_t(j) * kThreads + lane;
            const bool valid = q < n;
            const uint64_t mask = valid ? masks[j] : 0ull;
            bool follower;
            const uint32_t leader = elect_leader(mask, valid, elect, follower);
            uint32_t slot = 0;
            if (valid && !follower) {
                bool won;
                slot = hashed_insert(tk, lg, mask, won, err);
            }
            slot = uint32_t(__shfl(int(slot), int(leader), kWave));
            if (valid) lp_slot[q] = slot;
        }
    }
}

// ---------------------------------------------------------------------------
// Distinct-count estimate of the leaf masks (HyperLogLog: Flajolet, Fusy,
// Gandouet, Meunier 2007), so the leaf table is sized by unique leaves rather
// than by leaf positions and its slot arrays stay cache-sized.  Only the table
// size depends on it; the result does not.
// ---------------------------------------------------------------------------
constexpr int kSketchIpt = 8;

__global__ __launch_bounds__(kThreads) void k_sketch(const uint64_t* __restrict__ values,
                                                     const uint64_t* __restrict__ count_ptr,
                                                     uint32_t* __restrict__ regs)
{
    __shared__ uint32_t s_reg[kSketchRegs];
    for (uint32_t i = threadIdx.x; i < uint32_t(kSketchRegs); i += kThreads) s_reg[i] = 0;
    __syncthreads();
    const uint64_t n = *count_ptr;
    // kSketchIpt values per thread and round, all loaded before any is used
    // (one workgroup per CU holds too few waves to hide one load at a time).
    // Positions past the end read the last value again: a register maximum
    // does not change when a value is counted twice.
    constexpr uint64_t kRound = uint64_t(kThreads) * kSketchIpt;
    for (uint64_t b = uint64_t(blockIdx.x) * kRound; b < n; b += uint64_t(gridDim.x) * kRound) {
        uint64_t v[kSketchIpt];
#pragma unroll
        for (int i = 0; i < kSketchIpt; ++i)
            v[i] = __builtin_nontemporal_load(values + min(b + uint64_t(i) * kThreads + threadIdx.x, n - 1));
#pragma unroll
        for (int i = 0; i < kSketchIpt; ++i) {
            // A mixer unrelated to the table's home-slot hash.
            const uint64_t h = fmix64(v[i] * 0x9E3779B97F4A7C15ull + 0x632BE59BD9B4E019ull);
            const uint32_t idx = uint32_t(h >> (64 - kSketchBits));
            const uint64_t rest = h << kSketchBits;
            const uint32_t rho = rest ? uint32_t(__clzll((long long)rest)) + 1u : uint32_t(64 - kSketchBits + 1);
            atomicMax(&s_reg[idx], rho);
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < uint32_t(kSketchRegs); i += kThreads)
        if (s_reg[i]) atomicMax(&regs[i], s_reg[i]);
}

constexpr int kEstimateThreads = 1024;

__global__ __launch_bounds__(kEstimateThreads) void k_sketch_estimate(const uint32_t* __restrict__ regs,
                                                                      const uint64_t* __restrict__ bound_ptr,
                                                                      uint64_t* __restrict__ estimate)
{
    __shared__ double s_sum[kEstimateThreads / kWave];
    __shared__ uint32_t s_zero[kEstimateThreads / kWave];
    double sum = 0.0;
    uint32_t zeros = 0;
    for (uint32_t i = threadIdx.x; i < uint32_t(kSketchRegs); i += kEstimateThreads) {
        sum += ldexp(1.0, -int(regs[i]));
        zeros += regs[i] == 0 ? 1u : 0u;
    }
#pragma unroll
    for (int d = kWave / 2; d >= 1; d >>= 1) {
        sum += __shfl_xor(sum, d, kWave);
        zeros += __shfl_xor(zeros, d, kWave);
    }
    const uint32_t w = threadIdx.x / kWave;
    if (lane_id() == 0) {
        s_sum[w] = sum;
        s_zero[w] = zeros;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double total = 0.0;
        uint32_t z = 0;
        for (int i = 0; i < kEstimateThreads / kWave; ++i) {
            total += s_sum[i];
            z += s_zero[i];
        }
        const double m = double(kSketchRegs);
        double e = 0.7213 / (1.0 + 1.079 / m) * m * m / total;
        if (e <= 2.5 * m && z) e = m * log(m / double(z));  // small-range (linear counting) correction
        const uint64_t want = uint64_t(e * 1.25) + 16;
        const uint64_t bound = *bound_ptr;
        *estimate = want < bound ? want : bound;
    }
}

// ---------------------------------------------------------------------------
// Leaf order: the occupied slots of a hashed table -> the masks in ascending
// order, and each slot's rank.  A sample sort in four launches:
//   k_leaf_sample   one workgroup: a sample of the masks, sorted, gives the
//                   splitters of 2^b buckets of about 1024 masks.  The table is
//                   hashed, so its first slots are a uniform sample; their
//                   density also gives the mask count that b is chosen from.
//   k_order_count   keys per bucket (each tile of slots classifies its masks by
//                   binary search in the splitters, in LDS)
//   k_order_scatter masks and slots into their buckets' ranges, in any order
//   k_order_sort    one workgroup per bucket: LDS sort, masks and ranks out.
//                   The masks are distinct, so the result does not depend on
//                   the order of the scatter.
// Bound by launches and by the dependent LDS steps of the two sorts, not by
// bytes.  An LSD radix sort of the same pairs took eight passes of three
// launches: 25 launches and 130 us (100k masks) to 330 us (360k masks) of
// kernel time, 130 us of a 350 us build of 1000 keys.
// A bucket too large for LDS (the sample missed, or over 4M masks) is sorted in
// pieces that its workgroup merges in global memory.
// ---------------------------------------------------------------------------
constexpr int kSampleThreads = 1024;
constexpr uint32_t kSampleMax = 4096;        // masks sampled at most
constexpr uint32_t kSamplePerBucket = 8;     // aimed at; fewer past 2^9 buckets
constexpr uint32_t kSampleScanMax = 1u << 18;  // slots looked at for a small sample
constexpr uint32_t kOrderMean = 1024;        // masks per bucket aimed at
constexpr int kOrderSortThreads = 512;
constexpr int kOrderIpt = 16;
constexpr uint32_t kOrderTile = kThreads * kOrderIpt;
static_assert(kOrderTile <= 65536 && kOrderMaxBuckets <= 65536, "bucket and rank packed in 16 bits each");

// Ascending sort of the n <= THREADS * E keys of s_key (LDS; the rest of its
// THREADS * E entries is overwritten with ~0), E consecutive ones per thread: a
// sort in registers, then log2(n / E) rounds in which each thread finds its
// place in a pair of runs (merge path) and merges its E keys.  Bound by the
// chain of dependent LDS reads, about 16 per round; a bitonic network's n log^2 n
// exchanges kept the CU's LDS busy for 40 us at 4096 keys.  Ends with a barrier;
// every thread of the block must call it.
template <int THREADS, int E>
__device__ __forceinline__ void block_merge_sort(uint64_t* s_key, uint32_t n)
{
    const uint32_t first = threadIdx.x * E;
    uint64_t v[E];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = first + e < n ? s_key[first + e] : ~0ull;
#pragma unroll
    for (int r = 0; r < E; ++r) {
#pragma unroll
        for (int e = r & 1; e + 1 < E; e += 2) {
            const uint64_t a = v[e], b = v[e + 1];
            v[e] = a < b ? a : b;
            v[e + 1] = a < b ? b : a;
        }
    }
#pragma unroll
    for (int e = 0; e < E; ++e) s_key[first + e] = v[e];
    __syncthreads();
    for (uint32_t run = E; run < n; run *= 2) {
        const uint32_t base = first & ~(2 * run - 1), diag = first - base;
        const bool live = base < n;  // threads past the keys hold padding only
        if (live) {
            const uint64_t *A = s_key + base, *B = A + run;
            uint32_t lo = diag > run ? diag - run : 0u, hi = min(diag, run);
            while (lo < hi) {
                const uint32_t mid = (lo + hi) / 2;
                if (A[mid] <= B[diag - 1 - mid]) lo = mid + 1;
                else hi = mid;
            }
            uint32_t ia = lo, ib = diag - lo;
            // Reads past a run's end stay inside s_key and are not taken.
            uint64_t ka = A[min(ia, run - 1)], kb = B[min(ib, run - 1)];
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const bool take = ib >= run || (ia < run && ka <= kb);
                v[e] = take ? ka : kb;
                ia += take ? 1u : 0u;
                ib += take ? 0u : 1u;
                const uint64_t next = take ? A[min(ia, run - 1)] : B[min(ib, run - 1)];
                ka = take ? next : ka;
                kb = take ? kb : next;
            }
        }
        __syncthreads();
        if (live) {
#pragma unroll
            for (int e = 0; e < E; ++e) s_key[first + e] = v[e];
        }
        __syncthreads();
    }
}

// split[1 .. 2^b): the splitters; split[0] = b.
__global__ __launch_bounds__(kSampleThreads) void k_leaf_sample(const uint64_t* __restrict__ tk,
                                                                const uint32_t* __restrict__ log2_ptr,
                                                                uint64_t* __restrict__ split)
{
    constexpr int IPT = 4;
    constexpr uint32_t kRound = kSampleThreads * IPT;
    __shared__ uint64_t s_key[kSampleMax];
    __shared__ uint32_t s_scan[kSampleThreads / kWave];
    const uint64_t total = 1ull << *log2_ptr;
    uint64_t scanned = 0, found = 0;
    uint32_t m = 0, b = 0;
    while (true) {
        uint64_t v[IPT];
#pragma unroll
        for (int i = 0; i < IPT; ++i) v[i] = tk[min(scanned + uint64_t(i) * kSampleThreads + threadIdx.x, total - 1)];
        uint32_t mine = 0;
#pragma unroll
        for (int i = 0; i < IPT; ++i) {
            if (scanned + uint64_t(i) * kSampleThreads + threadIdx.x >= total) v[i] = 0;
            mine += v[i] != 0 ? 1u : 0u;
        }
        uint32_t round;
        uint32_t o = m + block_exclusive_scan<kSampleThreads>(mine, s_scan, round);
#pragma unroll
        for (int i = 0; i < IPT; ++i) {
            if (v[i] != 0) {
                if (o < kSampleMax) s_key[o] = v[i];
                ++o;
            }
        }
        found += round;
        m = uint32_t(min(uint64_t(kSampleMax), m + uint64_t(round)));
        scanned = min(scanned + kRound, total);
        // Expected masks in the whole table, and the buckets for them.
        const float expect = float(found) * (float(total) / float(scanned));
        b = 0;
        while (b < kOrderMaxLog2 && float(kOrderMean << b) < expect) ++b;
        const uint32_t want = min(max(kSamplePerBucket << b, 64u), kSampleMax);
        if (scanned == total || m >= want || scanned >= kSampleScanMax) break;
    }
    while (b > 0 && (2u << b) > m) --b;  // at least two samples per bucket
    if (b > 0) {
        block_merge_sort<kSampleThreads, int(kSampleMax) / kSampleThreads>(s_key, m);
        const uint32_t buckets = 1u << b;
        for (uint32_t j = 1 + threadIdx.x; j < buckets; j += kSampleThreads)
            split[j] = s_key[uint32_t(uint64_t(j) * m >> b)];
    }
    if (threadIdx.x == 0) split[0] = b;
}

// Buckets of N keys: the number of splitters at or below each.  The N searches
// run in step, so that their LDS reads are in flight together.
template <int N>
__device__ __forceinline__ void buckets_by_split(const uint64_t* s_split, uint32_t b, const uint64_t (&key)[N],
                                                 uint32_t (&idx)[N])
{
#pragma unroll
    for (int j = 0; j < N; ++j) idx[j] = 0;
    for (uint32_t step = (1u << b) >> 1; step > 0; step >>= 1) {
#pragma unroll
        for (int j = 0; j < N; ++j) idx[j] += s_split[idx[j] + step] <= key[j] ? step : 0u;
    }
}

__global__ __launch_bounds__(kThreads) void k_order_count(const uint64_t* __restrict__ tk,
                                                          const uint32_t* __restrict__ log2_ptr,
                                                          const uint64_t* __restrict__ split,
                                                          uint32_t* __restrict__ totals)
{
    __shared__ uint64_t s_split[kOrderMaxBuckets];
    __shared__ uint32_t s_cnt[kOrderMaxBuckets];
    const uint64_t total = 1ull << *log2_ptr;
    const uint64_t ntiles = (total + kOrderTile - 1) / kOrderTile;
    if (blockIdx.x >= ntiles) return;
    const uint32_t b = uint32_t(split[0]), buckets = 1u << b;
    for (uint32_t i = threadIdx.x; i < buckets; i += kThreads) {
        s_split[i] = split[i];
        s_cnt[i] = 0;
    }
    __syncthreads();
    for (uint64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        uint64_t v[kOrderIpt];
#pragma unroll
        for (int j = 0; j < kOrderIpt; ++j)
            v[j] = tk[min(tile * kOrderTile + uint64_t(j) * kThreads + threadIdx.x, total - 1)];
        uint32_t k[kOrderIpt];
        buckets_by_split(s_split, b, v, k);
#pragma unroll
        for (int j = 0; j < kOrderIpt; ++j) {
            const bool here = tile * kOrderTile + uint64_t(j) * kThreads + threadIdx.x < total && v[j] != 0;
            if (b == 0) {
                // One bucket: one add per wave instead of one word for all.
                const uint32_t c = uint32_t(__popcll(__ballot(here)));
                if (lane_id() == 0 && c) atomicAdd(&s_cnt[0], c);
            } else if (here) {
                atomicAdd(&s_cnt[k[j]], 1u);
            }
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < buckets; i += kThreads)
        if (s_cnt[i]) atomicAdd(&totals[i], s_cnt[i]);
}

__global__ __launch_bounds__(kThreads) void k_order_scatter(const uint64_t* __restrict__ tk,
                                                            const uint32_t* __restrict__ log2_ptr,
                                                            const uint64_t* __restrict__ split,
                                                            const uint32_t* __restrict__ totals,
                                                            uint32_t* __restrict__ cursors,
                                                            uint64_t* __restrict__ list_keys,
                                                            uint32_t* __restrict__ list_slots)
{
    constexpr int BPT = int(kOrderMaxBuckets) / kThreads;  // buckets per thread in the scan
    __shared__ uint64_t s_split[kOrderMaxBuckets];
    __shared__ uint32_t s_start[kOrderMaxBuckets];
    __shared__ uint32_t s_cnt[kOrderMaxBuckets];
    __shared__ uint32_t s_scan[kThreads / kWave];
    const uint64_t total = 1ull << *log2_ptr;
    const uint64_t ntiles = (total + kOrderTile - 1) / kOrderTile;
    if (blockIdx.x >= ntiles) return;
    const uint32_t b = uint32_t(split[0]), buckets = 1u << b;
    for (uint32_t i = threadIdx.x; i < buckets; i += kThreads) s_split[i] = split[i];
    // Bucket starts: exclusive scan of the totals, BPT consecutive per thread.
    uint32_t t[BPT], sum = 0;
#pragma unroll
    for (int k = 0; k < BPT; ++k) {
        const uint32_t i = threadIdx.x * BPT + k;
        t[k] = i < buckets ? totals[i] : 0u;
        sum += t[k];
    }
    uint32_t unused;
    uint32_t run = block_exclusive_scan<kThreads>(sum, s_scan, unused);
#pragma unroll
    for (int k = 0; k < BPT; ++k) {
        const uint32_t i = threadIdx.x * BPT + k;
        if (i < buckets) s_start[i] = run;
        run += t[k];
    }
    for (uint64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        __syncthreads();  // the previous tile's counts have been read
        for (uint32_t i = threadIdx.x; i < buckets; i += kThreads) s_cnt[i] = 0;
        uint64_t v[kOrderIpt];
        uint32_t br[kOrderIpt];  // bucket << 16 | rank within the tile's bucket
#pragma unroll
        for (int j = 0; j < kOrderIpt; ++j)
            v[j] = tk[min(tile * kOrderTile + uint64_t(j) * kThreads + threadIdx.x, total - 1)];
        __syncthreads();
        buckets_by_split(s_split, b, v, br);
#pragma unroll
        for (int j = 0; j < kOrderIpt; ++j) {
            if (tile * kOrderTile + uint64_t(j) * kThreads + threadIdx.x >= total) v[j] = 0;
            if (v[j] != 0) br[j] = br[j] << 16 | atomicAdd(&s_cnt[br[j]], 1u);
        }
        __syncthreads();
        // The tile's place in each bucket's range.
        for (uint32_t i = threadIdx.x; i < buckets; i += kThreads) {
            const uint32_t c = s_cnt[i];
            if (c) s_cnt[i] = s_start[i] + atomicAdd(&cursors[i], c);
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kOrderIpt; ++j) {
            if (v[j] != 0) {
                const uint32_t o = s_cnt[br[j] >> 16] + (br[j] & 0xFFFFu);
                list_keys[o] = v[j];
                list_slots[o] = uint32_t(tile * kOrderTile + uint64_t(j) * kThreads + threadIdx.x);
            }
        }
    }
}

// The place of `key` among the n ascending keys of s_key that hold it.
__device__ __forceinline__ uint32_t place_in(const uint64_t* s_key, uint32_t n, uint64_t key)
{
    uint32_t lo = 0;
    for (uint32_t len = n; len > 1;) {
        const uint32_t half = len / 2;
        lo += s_key[lo + half] <= key ? half : 0u;
        len -= half;
    }
    return lo;
}

// Only the masks are sorted; a slot's rank is its mask's place among them.
__global__ __launch_bounds__(kOrderSortThreads) void k_order_sort(const uint64_t* __restrict__ split,
                                                                  const uint32_t* __restrict__ totals,
                                                                  uint64_t* keys_a, uint32_t* slots_a,
                                                                  uint64_t* keys_b, uint32_t* slots_b,
                                                                  uint64_t* __restrict__ out,
                                                                  uint32_t* __restrict__ rank_of_slot,
                                                                  uint64_t* __restrict__ count)
{
    constexpr uint32_t T = kOrderSortThreads;
    constexpr int E = int(kOrderCap / T);
    __shared__ uint64_t s_key[kOrderCap];
    __shared__ uint64_t s_red[T / kWave];
    const uint32_t buckets = 1u << uint32_t(split[0]);
    for (uint32_t bucket = blockIdx.x; bucket < buckets; bucket += gridDim.x) {
        uint64_t below = 0;
        for (uint32_t i = threadIdx.x; i < bucket; i += T) below += totals[i];
        const uint64_t start = block_reduce_sum<T>(below, s_red);
        const uint32_t cnt = totals[bucket];
        if (bucket + 1 == buckets && threadIdx.x == 0) *count = start + cnt;
        const bool whole = cnt <= kOrderCap;
        for (uint32_t c0 = 0; c0 < cnt; c0 += kOrderCap) {
            const uint32_t n = min(kOrderCap, cnt - c0);
            const uint64_t at = start + c0;
            // The thread's masks and slots, kept for their ranks.
            uint64_t key[E];
            uint32_t slot[E];
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const uint32_t i = min(threadIdx.x + uint32_t(e) * T, n - 1);
                key[e] = keys_a[at + i];
                slot[e] = slots_a[at + i];
            }
#pragma unroll
            for (int e = 0; e < E; ++e)
                if (threadIdx.x + uint32_t(e) * T < n) s_key[threadIdx.x + uint32_t(e) * T] = key[e];
            block_merge_sort<int(T), E>(s_key, n);
            uint64_t* const dst = whole ? out + start : keys_b + at;
            for (uint32_t i = threadIdx.x; i < n; i += T) dst[i] = s_key[i];
#pragma unroll
            for (int e = 0; e < E; ++e) {
                if (threadIdx.x + uint32_t(e) * T < n) {
                    const uint32_t p = place_in(s_key, n, key[e]);
                    if (whole) rank_of_slot[slot[e]] = uint32_t(start) + p;
                    else slots_b[at + p] = slot[e];
                }
            }
            __syncthreads();
        }
        if (whole) continue;
        // Pairs of sorted pieces, merged by each key's place in the other one.
        uint64_t *ka = keys_b + start, *kb = keys_a + start;
        uint32_t *sa = slots_b + start, *sb = slots_a + start;
        for (uint64_t piece = kOrderCap; piece < cnt; piece *= 2) {
            for (uint64_t i = threadIdx.x; i < cnt; i += T) {
                const uint64_t first = i / (2 * piece) * (2 * piece);
                const uint64_t mid = min(first + piece, uint64_t(cnt)), last = min(first + 2 * piece, uint64_t(cnt));
                const uint64_t key = ka[i];
                uint64_t lo = i < mid ? mid : first, hi = i < mid ? last : mid;
                const uint64_t own = i < mid ? i : i - mid + first, base = lo;
                while (lo < hi) {
                    const uint64_t at = (lo + hi) / 2;
                    if (ka[at] < key) lo = at + 1;
                    else hi = at;
                }
                kb[own + (lo - base)] = key;
                sb[own + (lo - base)] = sa[i];
            }
            __syncthreads();
            uint64_t* const kt = ka;
            ka = kb;
            kb = kt;
            uint32_t* const st = sa;
            sa = sb;
            sb = st;
        }
        for (uint64_t i = threadIdx.x; i < cnt; i += T) {
            out[start + i] = ka[i];
            rank_of_slot[sa[i]] = uint32_t(start + i);
        }
        __syncthreads();
    }
}

// The whole order of at most kOrderCap masks in one workgroup: occupied slots
// gathered into LDS in any order, sorted, and each slot's rank found by a search.
// Four launches less three: 1000 keys, whose build is bound by launches (6 us
// each), 199 -> 163 us with the sketch's two and the layout's count left out too.
__global__ __launch_bounds__(kSampleThreads) void k_order_small(const uint64_t* __restrict__ table_keys,
                                                                const uint32_t* __restrict__ table_log2,
                                                                uint64_t* __restrict__ out,
                                                                uint32_t* __restrict__ rank_of_slot,
                                                                uint64_t* __restrict__ count)
{
    __shared__ uint64_t s_key[kOrderCap];
    __shared__ uint32_t s_n;
    const uint32_t slots = 1u << *table_log2;
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < slots; i += kSampleThreads) {
        const uint64_t k = table_keys[i];
        if (k) {
            const uint32_t at = atomicAdd(&s_n, 1u);
            if (at < kOrderCap) s_key[at] = k;  // always: the caller's bound
        }
    }
    __syncthreads();
    const uint32_t n = min(s_n, kOrderCap);
    block_merge_sort<kSampleThreads, int(kOrderCap) / kSampleThreads>(s_key, n);
    for (uint32_t i = threadIdx.x; i < n; i += kSampleThreads) out[i] = s_key[i];
    for (uint32_t i = threadIdx.x; i < slots; i += kSampleThreads) {
        const uint64_t k = table_keys[i];
        if (k) {
            uint32_t lo = 0, hi = n;
            while (lo < hi) {
                const uint32_t mid = (lo + hi) / 2;
                if (s_key[mid] < k) lo = mid + 1;
                else hi = mid;
            }
            rank_of_slot[i] = lo;
        }
    }
    if (threadIdx.x == 0) *count = n;
}

// Ordered-table probe: home = top lg bits of the hash, linear probing forward
// into an overflow tail (no wrap), so every key sits at or after its home slot.
// `won` tells whether this call placed the key.
__device__ __forceinline__ uint32_t ordered_probe(uint64_t* __restrict__ tk, uint32_t lg, uint64_t limit, uint64_t h,
                                                  bool& won, unsigned long long* err)
{
    won = false;
    uint64_t slot = h >> (64 - lg);
    for (; slot < limit; ++slot) {
        const uint64_t cur = probe_load(&tk[slot]);
        if (cur == h) return uint32_t(slot);
        if (cur == 0) {
            const uint64_t prev = atomicCAS((unsigned long long*)&tk[slot], 0ull, (unsigned long long)h);
            if (prev == 0) {
                won = true;
                return uint32_t(slot);
            }
            if (prev == h) return uint32_t(slot);
        }
    }
    atomicOr(err, (unsigned long long)kErrTableOverflow);
    return uint32_t(limit - 1);
}

// Ordered-table insert; the placing call records p as the key's representative.
__device__ __forceinline__ uint32_t ordered_insert(uint64_t* __restrict__ tk, uint32_t* __restrict__ rep, uint32_t lg,
                                                   uint64_t limit, uint64_t h, uint32_t p, BuildCounters* c)
{
    bool won;
    const uint32_t slot = ordered_probe(tk, lg, limit, h, won, (unsigned long long*)&c->error);
    if (won) rep[slot] = p;
    return slot;
}

// ---------------------------------------------------------------------------
// Level build: children (Morton-sorted codes of the level below, their table
// slots) -> parents.  A parent belongs to the tile holding its first child and
// has at most 8 children, so a run extends at most 7 children past the tile.
// ---------------------------------------------------------------------------
constexpr int kBuildIpt = 2;
constexpr int kBuildTile = kThreads * kBuildIpt;

// The parents that each part of the children starts (the workgroups of
// k_level_build take the same parts).  With pre set, also the node counts of
// all levels from `level` down to `lowest`, from the children's codes alone:
// child i starts a node of level `level - j` when its code differs from its
// predecessor's above bit 3 (j + 1).
__global__ __launch_bounds__(kThreads) void k_level_count(const uint64_t* __restrict__ codes,
                                                          const uint64_t* __restrict__ n_ptr,
                                                          uint32_t* __restrict__ parts, uint64_t* __restrict__ pre,
                                                          int level, int lowest)
{
    constexpr int kTriples = 22;  // of a 64-bit code
    __shared__ uint32_t s_diff[kTriples];
    __shared__ uint64_t s_red[kThreads / kWave];
    const uint64_t n = *n_ptr;
    const uint64_t ntiles = (n + kBuildTile - 1) / kBuildTile;
    if (threadIdx.x < uint32_t(kTriples)) s_diff[threadIdx.x] = 0;
    __syncthreads();
    uint64_t t0, t1;
    part_tiles(ntiles, blockIdx.x, gridDim.x, t0, t1);
    // Starts of parents, grandparents; the levels above them from a histogram
    // of the highest triple that differs (one child in 64 or fewer).
    uint32_t starts = 0, gstarts = 0;
    for (uint64_t tile = t0; tile < t1; ++tile) {
        // Coalesced: lane i of a round reads code i and its predecessor (all
        // loads issued first, indices clamped into [0, n)).
        const uint64_t base = tile * kBuildTile + threadIdx.x;
        uint64_t cv[kBuildIpt], pv[kBuildIpt];
#pragma unroll
        for (int j = 0; j < kBuildIpt; ++j) {
            const uint64_t i = base + uint64_t(j) * kThreads;
            cv[j] = codes[min(i, n - 1)];
            pv[j] = codes[i > 0 ? min(i - 1, n - 1) : 0];
        }
#pragma unroll
        for (int j = 0; j < kBuildIpt; ++j) {
            const uint64_t i = base + uint64_t(j) * kThreads;
            const uint64_t x = i == 0 ? ~0ull : i < n ? cv[j] ^ pv[j] : 0ull;
            starts += (x >> 3) != 0 ? 1u : 0u;
            gstarts += (x >> 6) != 0 ? 1u : 0u;
            if (pre && (x >> 9) != 0) atomicAdd(&s_diff[(63 - __clzll((long long)x)) / 3], 1u);
        }
    }
    const uint64_t heads = block_reduce_sum<kThreads>(starts, s_red);
    const uint64_t ghead = block_reduce_sum<kThreads>(gstarts, s_red);
    if (threadIdx.x == 0) parts[blockIdx.x] = uint32_t(heads);
    if (!pre) return;
    for (int j = int(threadIdx.x); level - j >= lowest; j += kThreads) {
        uint64_t sum = j == 0 ? heads : j == 1 ? ghead : 0;
        for (int t = j + 1; j >= 2 && t < kTriples; ++t) sum += s_diff[t];
        if (sum) atomicAdd((unsigned long long*)&pre[level - j], (unsigned long long)sum);
    }
}

// A tile's children are read coalesced and staged in LDS with the starts of
// their parents; then one thread per parent takes its children from LDS (they
// are sorted, so slot s's child is the popcount of the mask below s), writes the
// record and inserts the hash into the level's table.  The next tile's children
// are loaded before the inserts.  Bound by the chain of each tile's dependent
// steps (loads, two barriers, probe, CAS) and the waves in flight to hide it.
// All builds of 2048^3 triangles 359 -> 285 us, of 64 chunks (12.8M keys) 137 ->
// 96, against a thread per run of children whose last parent walked on through
// global memory child by child.  Two children per thread: with four the
// registers (130) leave 12 waves per CU (331 us), with one a tile has too little
// between its barriers (356); not loading ahead takes 305.
constexpr int kBuildHalo = 8;
constexpr int kBuildWaves = kThreads / kWave;

__global__ __launch_bounds__(kThreads) void k_level_build(LevelBuildArgs g)
{
    __shared__ uint64_t s_hash[kBuildTile + kBuildHalo];
    __shared__ uint32_t s_slot[kBuildTile + kBuildHalo];
    __shared__ uint8_t s_sub[kBuildTile + kBuildHalo];
    __shared__ uint16_t s_start[kBuildTile + 1];
    __shared__ uint32_t s_cnt[kBuildIpt * kBuildWaves];
    __shared__ uint32_t s_heads[kBuildWaves];
    __shared__ uint32_t s_end;
    __shared__ uint64_t s_red[kBuildWaves];
    __shared__ uint32_t s_elect[kBuildWaves][kElectBuckets];
    const uint64_t n = *g.child_count;
    const uint64_t ntiles = (n + kBuildTile - 1) / kBuildTile;
    const uint64_t next_tiles = g.next_parts ? (*g.parent_count + kBuildTile - 1) / kBuildTile : 0;
    uint64_t t0, t1;
    part_tiles(ntiles, blockIdx.x, gridDim.x, t0, t1);
    if (t0 >= t1) return;  // the whole workgroup
    const uint32_t tid = threadIdx.x, lane = lane_id();
    const uint32_t w = uint32_t(__builtin_amdgcn_readfirstlane(int(tid / kWave)));
    const uint32_t lg = *g.table_log2;
    const uint64_t limit = (1ull << lg) + kTableOverflow;

    // A tile's children in registers: row j holds child j * kThreads + tid, the
    // halo (threads 0 .. 7) those past the tile; before[j]: the code before the
    // wave's row.  Indices are clamped into [0, n): what lies past the end is
    // not used.
    uint64_t code[kBuildIpt], hash[kBuildIpt], before[kBuildIpt], halo_code = 0, halo_hash = 0;
    uint32_t slot[kBuildIpt], halo_slot = 0;
    auto child = [&](uint64_t i, uint64_t& h, uint32_t& sl) {
        if (g.child_hash_seq) {
            sl = g.child_slots[i];
            h = g.child_hash_seq[i];
        } else {
            sl = g.child_rank_of_slot[g.child_slots[i]];
            h = g.child_hashes[sl];
        }
    };
    auto load = [&](uint64_t tile) {
        const uint64_t base = tile * kBuildTile;
#pragma unroll
        for (int j = 0; j < kBuildIpt; ++j) {
            const uint64_t row = base + uint64_t(j) * kThreads + w * kWave;
            code[j] = g.child_codes[min(row + lane, n - 1)];
            before[j] = g.child_codes[row > 0 ? min(row - 1, n - 1) : 0];
        }
#pragma unroll
        for (int j = 0; j < kBuildIpt; ++j) child(min(base + uint64_t(j) * kThreads + tid, n - 1), hash[j], slot[j]);
        if (tid < uint32_t(kBuildHalo)) {
            const uint64_t i = min(base + kBuildTile + tid, n - 1);
            halo_code = g.child_codes[i];
            child(i, halo_hash, halo_slot);
        }
    };
    load(t0);
    uint64_t p0 = parts_before(g.parts, s_red);
    for (uint64_t tile = t0; tile < t1; ++tile) {
        const uint64_t base = tile * kBuildTile;
        const uint32_t here = uint32_t(min(uint64_t(kBuildTile), n - base));
        // Row by row: which children start a parent (a grandparent), as ballots.
        uint64_t starts[kBuildIpt], gstarts[kBuildIpt];
#pragma unroll
        for (int j = 0; j < kBuildIpt; ++j) {
            const uint32_t i = uint32_t(j) * kThreads + tid;
            uint64_t prev = __shfl_up(code[j], 1, kWave);
            if (lane == 0) prev = before[j];
            const uint64_t x = base + i == 0 ? ~0ull : code[j] ^ prev;
            starts[j] = __ballot(i < here && (x >> 3) != 0);
            gstarts[j] = __ballot(i < here && (x >> 6) != 0);
            if (lane == 0) s_cnt[j * kBuildWaves + w] = uint32_t(__popcll(starts[j]));
            s_hash[i] = hash[j];
            s_slot[i] = slot[j];
            s_sub[i] = uint8_t(code[j] & 7u);
        }
        if (tid < uint32_t(kBuildHalo)) {
            s_hash[kBuildTile + tid] = halo_hash;
            s_slot[kBuildTile + tid] = halo_slot;
            s_sub[kBuildTile + tid] = uint8_t(halo_code & 7u);
        }
        // End of the tile's last run: the halo's children of the last child's
        // parent (a prefix of it, the codes being sorted).  The last wave holds
        // that child, the first the halo: through LDS.
        if (tid == uint32_t(kThreads - 1)) s_red[0] = code[kBuildIpt - 1] >> 3;
        __syncthreads();
        if (w == 0) {
            const uint64_t B = __ballot(lane < uint32_t(kBuildHalo) && base + kBuildTile + lane < n &&
                                        (halo_code >> 3) == s_red[0]);
            if (lane == 0) s_end = here + uint32_t(__popcll(B));
        }
        uint32_t local[kBuildIpt], tile_parents = 0;
#pragma unroll
        for (int i = 0; i < kBuildIpt * kBuildWaves; ++i) {
            if (uint32_t(i % kBuildWaves) == w) local[i / kBuildWaves] = tile_parents;
            tile_parents += s_cnt[i];
        }
        // The tile's nodes [p0, p0 + tile_parents) lie in at most two tiles of
        // the next build: its parents in the first (low half) and the second.
        const uint32_t cut = uint32_t(kBuildTile - p0 % kBuildTile);
        uint32_t heads = 0;
#pragma unroll
        for (int j = 0; j < kBuildIpt; ++j) {
            const uint32_t q = local[j] + uint32_t(__popcll(starts[j] & lanemask_lt()));
            if ((starts[j] >> lane) & 1ull) {
                s_start[q] = uint16_t(uint32_t(j) * kThreads + tid);
                g.parent_codes[p0 + q] = code[j] >> 3;
            }
            heads += ((gstarts[j] >> lane) & 1ull) ? (q < cut ? 1u : 1u << 16) : 0u;
        }
        if (g.next_parts) {
            heads = wave_reduce_sum32(heads);
            if (lane == 0) s_heads[w] = heads;
        }
        if (tile + 1 < t1) load(tile + 1);
        __syncthreads();
        if (g.next_parts && tid < 2) {
            uint32_t sum = 0;
#pragma unroll
            for (int i = 0; i < kBuildWaves; ++i) sum += (s_heads[i] >> (16 * tid)) & 0xFFFFu;
            const uint64_t t = p0 / kBuildTile + tid;
            if (sum) atomicAdd(&g.next_parts[part_of_tile(next_tiles, t, g.next_num)], sum);
        }
        for (uint32_t k0 = 0; k0 < tile_parents; k0 += kThreads) {
            const uint32_t k = k0 + tid;
            const bool valid = k < tile_parents;
            uint64_t h = 0;
            if (valid) {
                const uint32_t st = s_start[k], en = k + 1 < tile_parents ? s_start[k + 1] : s_end;
                uint32_t mask = 0;
#pragma unroll
                for (uint32_t c = 0; c < 8; ++c) mask |= st + c < en ? 1u << s_sub[min(st + c, en - 1)] : 0u;
                uint32_t ch[8];
                uint64_t hs[8];
#pragma unroll
                for (uint32_t c = 0; c < 8; ++c) {
                    const bool there = (mask >> c) & 1u;
                    const uint32_t i = st + uint32_t(__popc(mask & ((1u << c) - 1u)));
                    const uint32_t at = min(i, en - 1);
                    ch[c] = there ? s_slot[at] : kEmptyChild;
                    hs[c] = there ? s_hash[at] : 0ull;
                }
                const uint64_t p = p0 + k;
                g.parent_masks[p] = uint8_t(mask);
                uint4* dst = reinterpret_cast<uint4*>(g.parent_children + 8 * p);
                dst[0] = make_uint4(ch[0], ch[1], ch[2], ch[3]);
                dst[1] = make_uint4(ch[4], ch[5], ch[6], ch[7]);
                h = hash_children(hs);
                if (g.parent_hashes) g.parent_hashes[p] = h;
            }
            // Equal parents (identical subtrees) often sit side by side: one lane
            // per distinct hash in a wave probes the table, the others take its
            // slot.
            bool follower;
            const uint32_t leader = elect_leader(h, valid, s_elect[w], follower);
            uint32_t at = 0;
            if (valid && !follower)
                at = ordered_insert(g.table_keys, g.table_rep, lg, limit, h, uint32_t(p0 + k), g.counters);
            at = uint32_t(__shfl(int(at), int(leader), kWave));
            if (valid) g.parent_slots[p0 + k] = at;
        }
        p0 += tile_parents;
        __syncthreads();  // the staged children are rewritten by the next tile
    }
}

// ---------------------------------------------------------------------------
// Small top levels in one workgroup, all in LDS.  Level l <= 3 has at most 8^l
// <= 512 nodes, so its children lie in a dense array indexed by code (empty:
// rank kEmptyChild, hash 0): parent p's are entries 8p .. 8p + 7, and a parent's
// rank and hash are an entry of the next level's array.  Per level: one thread
// per parent forms its mask and hash; the (hash, parent) pairs are sorted (each
// wave 64 of them in registers, then merges by binary search); equal hashes get
// one rank, and the level is written in ascending hash order.  Bound by latency
// (one workgroup): four levels take 20 to 24 us; with the children scattered
// through global memory and a bitonic sort of 45 barriers they took 45 to 58.
// ---------------------------------------------------------------------------
constexpr int kTailThreads = 1024;
constexpr int kTailChildren = int(kTailMaxChildren) / kTailThreads;

// True when (ka, ia) sorts before (kb, ib).
__device__ __forceinline__ bool pair_less(uint64_t ka, uint32_t ia, uint64_t kb, uint32_t ib)
{
    return ka < kb || (ka == kb && ia < ib);
}

__global__ __launch_bounds__(kTailThreads) void k_level_tail(TailArgs a)
{
    // Children of level l (dense), then of level l - 1 behind them: 8^(l + 1)
    // entries each, in two arrays used in turn.
    __shared__ uint64_t s_hash[kTailMaxChildren + kTailMaxParents];
    __shared__ uint32_t s_rank[kTailMaxChildren + kTailMaxParents];
    __shared__ uint64_t s_key[kTailMaxParents];
    __shared__ uint16_t s_idx[kTailMaxParents];
    __shared__ uint32_t s_scan[kTailThreads / kWave];
    __shared__ uint64_t s_red[kTailThreads / kWave];
    const uint32_t tid = threadIdx.x, lane = lane_id();
    BuildCounters* c = a.counters;
    {
        // The children of level `top`; all loads of a step are issued together.
        const uint32_t C = uint32_t(min(*a.child_count, uint64_t(kTailMaxChildren)));
        uint32_t code[kTailChildren], r[kTailChildren];
        uint64_t h[kTailChildren];
#pragma unroll
        for (int k = 0; k < kTailChildren; ++k) {
            const uint32_t i = min(uint32_t(k) * kTailThreads + tid, C ? C - 1 : 0u);
            code[k] = C ? uint32_t(a.child_codes[i]) & (kTailMaxChildren - 1) : 0u;
            r[k] = C ? a.child_slots[i] : 0u;
        }
#pragma unroll
        for (int k = 0; k < kTailChildren; ++k) r[k] = C ? a.child_rank_of_slot[r[k]] : 0u;
#pragma unroll
        for (int k = 0; k < kTailChildren; ++k) h[k] = C ? a.child_hashes[r[k]] : 0ull;
        for (uint32_t i = tid; i < kTailMaxChildren; i += kTailThreads) {
            s_rank[i] = kEmptyChild;
            s_hash[i] = 0;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kTailChildren; ++k) {
            if (uint32_t(k) * kTailThreads + tid < C) {
                s_rank[code[k]] = r[k];
                s_hash[code[k]] = h[k];
            }
        }
        __syncthreads();
    }
    uint32_t in = 0, out = kTailMaxChildren;  // where the children and the parents' entries are
    for (int l = a.top; l >= 0; --l) {
        const uint32_t P = 1u << (3 * l);  // parents there may be
        // 1. Parents: mask and hash (absent ones sort last).
        const uint32_t p = tid;
        uint32_t mask = 0;
        uint64_t key = ~0ull;
        uint32_t idx = 0xFFFFu;
        if (p < P) {
            uint64_t hs[8];
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) {
                mask |= s_rank[in + 8 * p + k] != kEmptyChild ? 1u << k : 0u;
                hs[k] = s_hash[in + 8 * p + k];
            }
            if (mask) {
                key = hash_children(hs);
                idx = p;
            } else {
                idx = 0x8000u | p;
            }
            s_rank[out + p] = kEmptyChild;
            s_hash[out + p] = mask ? key : 0ull;
        }
        // 2. Ascending sort of (key, idx): each wave's 64 by a bitonic network
        //    in registers, then runs of 64, 128, ... merged in pairs: an
        //    element's place is its own plus the elements of the other run
        //    before it.  Waves without parents only keep the barriers.
        const bool mine = (tid & ~uint32_t(kWave - 1)) < P;
        const uint32_t net = min(P, uint32_t(kWave));  // lanes of one network
        if (mine) {
            for (uint32_t size = 2; size <= net; size <<= 1) {
                for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
                    const uint64_t ok = __shfl_xor(key, int(stride), kWave);
                    const uint32_t oi = uint32_t(__shfl_xor(int(idx), int(stride), kWave));
                    const bool up = (lane & size) == 0 || size == net;
                    const bool keep_low = ((lane & stride) == 0) == up;
                    const bool less = pair_less(key, idx, ok, oi);
                    // Equal pairs (padding) may stay.
                    if (less != keep_low && pair_less(ok, oi, key, idx) == keep_low) {
                        key = ok;
                        idx = oi;
                    }
                }
            }
        }
        uint32_t pos = tid;
        if (mine) {
            s_key[pos] = key;
            s_idx[pos] = uint16_t(idx);
        }
        __syncthreads();
        for (uint32_t run = kWave; run < P; run *= 2) {
            if (mine) {
                const uint32_t other = (pos & ~(run - 1)) ^ run;
                uint32_t lo = 0, hi = run;
                while (lo < hi) {
                    const uint32_t mid = (lo + hi) / 2;
                    if (pair_less(s_key[other + mid], s_idx[other + mid], key, idx)) lo = mid + 1;
                    else hi = mid;
                }
                pos = (pos & ~(2 * run - 1)) + (pos & (run - 1)) + lo;
            }
            __syncthreads();
            if (mine) {
                s_key[pos] = key;
                s_idx[pos] = uint16_t(idx);
            }
            __syncthreads();
        }
        // 3. Unique ranks; the first of each equal-hash run represents it.  One
        //    scan carries the ranks and, above them, the totals: duplicates
        //    (at most 511: 9 bits from bit 10) and the representatives'
        //    children (at most 4096: 13 bits from bit 19).
        const uint32_t q = tid;
        uint64_t bad = 0;
        const uint32_t qp = q < P ? s_idx[q] : 0xFFFFu;
        const bool there = qp < kTailMaxParents;
        const uint64_t qk = there ? s_key[q] : 0ull;
        const bool lead = there && (q == 0 || qk != s_key[q - 1]);
        uint32_t ch[8], m = 0;
        if (there) {
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) {
                ch[k] = s_rank[in + 8 * qp + k];
                m |= ch[k] != kEmptyChild ? 1u << k : 0u;
            }
        }
        uint32_t total;
        const uint32_t ex = block_exclusive_scan<kTailThreads>(
            lead ? 1u | uint32_t(__popc(m)) << 19 : there ? 1u << 10 : 0u, s_scan, total) & 1023u;
        const uint32_t Q = total & 1023u;
        if (there) {
            const uint32_t r = ex + (lead ? 1u : 0u) - 1u;
            s_rank[out + qp] = r;
            if (lead) {
                a.out_hashes[l][r] = qk;
                a.out_masks[l][r] = uint8_t(m);
                uint4* dst = reinterpret_cast<uint4*>(a.out_children[l] + 8 * uint64_t(r));
                dst[0] = make_uint4(ch[0], ch[1], ch[2], ch[3]);
                dst[1] = make_uint4(ch[4], ch[5], ch[6], ch[7]);
            } else if (a.check_collisions) {
                // Compare with the run's representative (content must be equal).
                uint32_t f = q;
                while (f > 0 && s_key[f - 1] == qk) --f;
                const uint32_t rp = s_idx[f];
                bool diff = false;
                for (uint32_t k = 0; k < 8; ++k) diff |= ch[k] != s_rank[in + 8 * rp + k];
                bad = diff ? 1 : 0;
            }
        }
        if (a.check_collisions) bad = block_reduce_sum<kTailThreads>(bad, s_red);
        if (tid == 0) {
            c->pre[l] = Q + (total >> 10 & 511u);
            c->uniq[l] = Q;
            c->words[l] = Q + (total >> 19);
            if (bad) c->collisions += bad;
        }
        __syncthreads();  // ranks written, keys read
        const uint32_t t = in;
        in = out;
        out = t;
    }
}

// Exact-content check of every parent against its table representative.
__global__ void k_level_check(const uint32_t* __restrict__ parent_slots, const uint32_t* __restrict__ table_rep,
                              const uint8_t* __restrict__ masks, const uint32_t* __restrict__ children,
                              const uint64_t* __restrict__ count_ptr, uint64_t* __restrict__ collisions)
{
    const uint64_t n = *count_ptr;
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
    uint32_t bad = 0;
    for (uint64_t p = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; p < n; p += stride) {
        const uint32_t r = table_rep[parent_slots[p]];
        bool diff = masks[p] != masks[r];
        for (int s = 0; s < 8; ++s) diff |= children[8 * p + s] != children[8 * uint64_t(r) + s];
        bad += diff ? 1u : 0u;
    }
    if (bad) atomicAdd((unsigned long long*)collisions, (unsigned long long)bad);
}

// ---------------------------------------------------------------------------
// Level extract: ordered table -> the level's arrays in ascending hash order.
// For occupied slot k in probe cluster [js, je]:
//   rank(k) = (#occupied slots before k) - (k - js) + #{keys in cluster < key(k)}
// Slots are read through an LDS window with a halo; clusters reaching past it
// fall back to global loads.
// ---------------------------------------------------------------------------
constexpr int kExtractIpt = 1;
constexpr int kExtractTile = kThreads * kExtractIpt;
constexpr int kHalo = 128;

// Occupied slots of every part of the tables given (one workgroup per part;
// the workgroups of k_level_extract take the same parts).  With clear.num, the
// workgroups also clear those tables.
__global__ __launch_bounds__(kThreads) void k_extract_count(ExtractCounts a, TableClears clear)
{
    __shared__ uint64_t s_red[kThreads / kWave];
    uint32_t b = blockIdx.x;
    int t = 0;
    while (b >= a.table[t].num_parts) b -= a.table[t++].num_parts;
    const uint64_t* __restrict__ keys = a.table[t].keys;
    const uint64_t total = (1ull << *a.table[t].log2) + kTableOverflow;
    const uint64_t ntiles = (total + kExtractTile - 1) / kExtractTile;
    uint64_t t0, t1;
    part_tiles(ntiles, b, a.table[t].num_parts, t0, t1);
    const uint64_t end = min(t1 * kExtractTile, total);
    uint32_t occ = 0;
    constexpr int kAhead = 8;
    for (uint64_t i = t0 * kExtractTile + threadIdx.x; i < end; i += kAhead * kThreads) {
        // All in flight at once; slots past the part read its last and are not
        // counted.
        uint64_t v[kAhead];
#pragma unroll
        for (int k = 0; k < kAhead; ++k) v[k] = keys[min(i + uint64_t(k) * kThreads, end - 1)];
#pragma unroll
        for (int k = 0; k < kAhead; ++k) occ += (i + uint64_t(k) * kThreads < end && v[k] != 0) ? 1u : 0u;
    }
    const uint64_t cnt = block_reduce_sum<kThreads>(occ, s_red);
    if (threadIdx.x == 0) a.table[t].parts[b] = uint32_t(cnt);
    clear_tables(clear);
}

__global__ __launch_bounds__(kThreads) void k_level_extract(LevelExtractArgs g)
{
    __shared__ uint64_t s_win[kExtractTile + 2 * kHalo];
    __shared__ uint32_t s_scan[kThreads / kWave];
    __shared__ uint64_t s_red[kThreads / kWave];
    const uint32_t lg = *g.table_log2;
    const uint64_t total = (1ull << lg) + kTableOverflow;
    const uint64_t ntiles = (total + kExtractTile - 1) / kExtractTile;
    uint64_t wsum = 0;
    uint64_t t0, t1;
    part_tiles(ntiles, blockIdx.x, gridDim.x, t0, t1);
    uint64_t tile_before = parts_before(g.parts, s_red);  // occupied slots before the tile
    for (uint64_t tile = t0; tile < t1; ++tile) {
        const int64_t tile_base = int64_t(tile) * kExtractTile;
        const int64_t win_lo = tile_base - kHalo;
        const int64_t win_hi = tile_base + kExtractTile + kHalo;
        // Unconditional loads of the window (clamped into the table; slots
        // outside it read as empty), all in flight at once.
        constexpr int kWinPerThread = (kExtractTile + 2 * kHalo + kThreads - 1) / kThreads;
        uint64_t wv[kWinPerThread];
#pragma unroll
        for (int q = 0; q < kWinPerThread; ++q) {
            const int64_t s = win_lo + q * kThreads + int64_t(threadIdx.x);
            wv[q] = g.table_keys[min(max(s, int64_t(0)), int64_t(total) - 1)];
        }
#pragma unroll
        for (int q = 0; q < kWinPerThread; ++q) {
            const int i = q * kThreads + int(threadIdx.x);
            const int64_t s = win_lo + i;
            if (i < kExtractTile + 2 * kHalo) s_win[i] = (s >= 0 && s < int64_t(total)) ? wv[q] : 0;
        }
        __syncthreads();
        auto key_at = [&](int64_t s) -> uint64_t {
            if (s < 0 || s >= int64_t(total)) return 0;
            if (s >= win_lo && s < win_hi) return s_win[s - win_lo];
            return g.table_keys[s];
        };
        const int64_t first = tile_base + int64_t(threadIdx.x) * kExtractIpt;
        uint32_t occ = 0;
#pragma unroll
        for (int j = 0; j < kExtractIpt; ++j) occ |= (s_win[first + j - win_lo] != 0 ? 1u : 0u) << j;
        uint32_t tile_slots;
        const uint32_t local = block_exclusive_scan<kThreads>(__popc(occ), s_scan, tile_slots);
        uint64_t before = tile_before + local;  // occupied slots before the current one
        tile_before += tile_slots;
        // Representatives' records, gathered up front (unoccupied slots read
        // parent 0, which is then ignored).
        uint32_t mask[kExtractIpt];
        uint4 ch0[kExtractIpt], ch1[kExtractIpt];
#pragma unroll
        for (int j = 0; j < kExtractIpt; ++j) {
            const uint32_t r = g.table_rep[min(uint64_t(first + j), total - 1)];
            const uint64_t rep = ((occ >> j) & 1u) ? r : 0u;
            mask[j] = g.parent_masks[rep];
            const uint4* src = reinterpret_cast<const uint4*>(g.parent_children + 8 * rep);
            ch0[j] = src[0];
            ch1[j] = src[1];
        }
        if (g.child_rank_of_slot) {
            // Child slots of the level below -> its ranks.  Only occupied
            // slots' real children are translated (the others hold parent 0's
            // record, which may be unset); every gather is issued, reading
            // rank 0 for the rest, so that all are in flight at once.
            const uint32_t* __restrict__ rk = g.child_rank_of_slot;
            uint32_t r[kExtractIpt][8];
#pragma unroll
            for (int j = 0; j < kExtractIpt; ++j) {
                const bool live = (occ >> j) & 1u;
                const uint32_t c[8] = {ch0[j].x, ch0[j].y, ch0[j].z, ch0[j].w, ch1[j].x, ch1[j].y, ch1[j].z, ch1[j].w};
#pragma unroll
                for (int e = 0; e < 8; ++e) r[j][e] = rk[live && c[e] != kEmptyChild ? c[e] : 0u];
            }
            auto tr = [](uint32_t v, uint32_t rank) { return v == kEmptyChild ? v : rank; };
#pragma unroll
            for (int j = 0; j < kExtractIpt; ++j) {
                ch0[j] = make_uint4(tr(ch0[j].x, r[j][0]), tr(ch0[j].y, r[j][1]), tr(ch0[j].z, r[j][2]),
                                    tr(ch0[j].w, r[j][3]));
                ch1[j] = make_uint4(tr(ch1[j].x, r[j][4]), tr(ch1[j].y, r[j][5]), tr(ch1[j].z, r[j][6]),
                                    tr(ch1[j].w, r[j][7]));
            }
        }
#pragma unroll
        for (int j = 0; j < kExtractIpt; ++j) {
            if ((occ >> j) & 1u) {
                const int64_t k = first + j;
                const uint64_t key = s_win[k - win_lo];
                int64_t js = k;
                while (key_at(js - 1) != 0) --js;
                int64_t je = k;
                while (key_at(je + 1) != 0) ++je;
                uint64_t lt = 0;
                for (int64_t x = js; x <= je; ++x) lt += key_at(x) < key ? 1 : 0;
                const uint64_t rank = before - uint64_t(k - js) + lt;
                g.rank_of_slot[k] = uint32_t(rank);
                g.out_hashes[rank] = key;
                g.out_masks[rank] = uint8_t(mask[j]);
                uint4* dst = reinterpret_cast<uint4*>(g.out_children + 8 * rank);
                dst[0] = ch0[j];
                dst[1] = ch1[j];
                wsum += 1 + __popc(mask[j]);
                ++before;
            }
        }
        __syncthreads();  // the window is rewritten by the next tile
    }
    const uint64_t wtot = block_reduce_sum<kThreads>(wsum, s_red);
    if (threadIdx.x == 0 && wtot) atomicAdd((unsigned long long*)g.w_count, (unsigned long long)wtot);
    if (threadIdx.x == 0 && blockIdx.x + 1 == gridDim.x) *g.q_count = tile_before;
}

// ---------------------------------------------------------------------------
// Final layout.  Node g of the level concatenation (levels 0.., in order) starts
// at word positions[g] = exclusive prefix of (1 + popc(mask)); leaves follow.
// ---------------------------------------------------------------------------
constexpr int kFinalIpt = 16;
constexpr int kFinalTile = kThreads * kFinalIpt;
static_assert(kBuildTile == kBuildTileItems && kExtractTile == kExtractTileItems &&
                  kFinalTile == kFinalTileItems,
              "tile sizes shared with the scratch planner");

// Per-level starts and arrays of the layout, staged in LDS once per block:
// a lane's level lookup then reads LDS rather than indexing the kernel
// argument block by a per-lane level (a dependent memory load per step).
struct FinalLds {
    uint64_t first[SVDAG_MAX_LEVELS + 1];  // first node of each level; [num_levels] = total_nodes
    const uint8_t* masks[SVDAG_MAX_LEVELS];
    const uint32_t* children[SVDAG_MAX_LEVELS];
};

// Every thread of the block must call it (one barrier).
__device__ __forceinline__ void stage_levels(const FinalArgs& a, FinalLds& s)
{
    const int t = int(threadIdx.x);
    if (t < a.num_levels) {
        s.first[t] = a.levels[t].first_node;
        s.masks[t] = a.levels[t].masks;
        s.children[t] = a.levels[t].children;
    }
    if (t == a.num_levels) s.first[t] = a.total_nodes;
    __syncthreads();
}

// Level of node g (< total_nodes): the last level starting at or before g;
// empty levels start where the next one does and are passed over.
__device__ __forceinline__ int level_of(const FinalLds& s, int num_levels, uint64_t g)
{
    int l = 0;
    while (l + 1 < num_levels && g >= s.first[l + 1]) ++l;
    return l;
}

// Word counts (1 + popc(mask)) of the thread's nodes.  The levels of the
// nodes are found first (they depend only on the index), so that all mask
// loads are in flight at once; nodes past the end read the last node's mask
// and count 0.
__device__ __forceinline__ uint32_t node_words(const FinalArgs& a, const FinalLds& s, uint64_t first,
                                               uint32_t (&sizes)[kFinalIpt])
{
    const uint64_t last = a.total_nodes - 1;  // total_nodes >= 1 (the root)
    int l = level_of(s, a.num_levels, min(first, last));
    const uint8_t* src[kFinalIpt];
#pragma unroll
    for (int j = 0; j < kFinalIpt; ++j) {
        const uint64_t gi = min(first + j, last);
        while (gi >= s.first[l + 1]) ++l;
        src[j] = s.masks[l] + (gi - s.first[l]);
    }
    uint8_t m[kFinalIpt];
#pragma unroll
    for (int j = 0; j < kFinalIpt; ++j) m[j] = *src[j];
    uint32_t sum = 0;
#pragma unroll
    for (int j = 0; j < kFinalIpt; ++j) {
        sizes[j] = first + j < a.total_nodes ? 1 + __popc(uint32_t(m[j])) : 0u;
        sum += sizes[j];
    }
    return sum;
}

__global__ __launch_bounds__(kThreads) void k_final_count(FinalArgs a)
{
    __shared__ uint64_t s_red[kThreads / kWave];
    __shared__ FinalLds s_lv;
    stage_levels(a, s_lv);
    const uint64_t ntiles = (a.total_nodes + kFinalTile - 1) / kFinalTile;
    uint64_t t0, t1;
    part_tiles(ntiles, blockIdx.x, gridDim.x, t0, t1);
    uint64_t sum = 0;
    for (uint64_t tile = t0; tile < t1; ++tile) {
        uint32_t sizes[kFinalIpt];
        sum += node_words(a, s_lv, tile * kFinalTile + uint64_t(threadIdx.x) * kFinalIpt, sizes);
    }
    const uint64_t tot = block_reduce_sum<kThreads>(sum, s_red);
    if (threadIdx.x == 0) a.parts[blockIdx.x] = uint32_t(tot);
}

__global__ __launch_bounds__(kThreads) void k_final_positions(FinalArgs a)
{
    __shared__ uint32_t s_scan[kThreads / kWave];
    __shared__ uint64_t s_red[kThreads / kWave];
    __shared__ FinalLds s_lv;
    stage_levels(a, s_lv);
    const uint64_t ntiles = (a.total_nodes + kFinalTile - 1) / kFinalTile;
    uint64_t t0, t1;
    part_tiles(ntiles, blockIdx.x, gridDim.x, t0, t1);
    uint64_t before = parts_before(a.parts, s_red);
    for (uint64_t tile = t0; tile < t1; ++tile) {
        const uint64_t first = tile * kFinalTile + uint64_t(threadIdx.x) * kFinalIpt;
        uint32_t sizes[kFinalIpt];
        const uint32_t sum = node_words(a, s_lv, first, sizes);
        uint32_t tile_words;
        const uint32_t local = block_exclusive_scan<kThreads>(sum, s_scan, tile_words);
        uint64_t pos = before + local;
        before += tile_words;
#pragma unroll
        for (int j = 0; j < kFinalIpt; ++j) {
            if (first + j < a.total_nodes) a.positions[first + j] = uint32_t(pos);
            pos += sizes[j];
        }
    }
}

__global__ __launch_bounds__(kThreads) void k_final_write(FinalArgs a)
{
    __shared__ FinalLds s_lv;
    stage_levels(a, s_lv);
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
    for (uint64_t gi = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; gi < a.total_nodes; gi += stride) {
        const int l = level_of(s_lv, a.num_levels, gi);
        const uint64_t i = gi - s_lv.first[l];
        const uint32_t mask = s_lv.masks[l][i];
        const uint32_t pos = a.positions[gi];
        a.words[pos] = mask;
        const bool last = l + 1 == a.num_levels;
        const uint4* src = reinterpret_cast<const uint4*>(s_lv.children[l] + 8 * i);
        const uint4 c0 = src[0], c1 = src[1];
        const uint32_t ch[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
        // Every child's target first (absent children read node 0's position
        // and are dropped), so that all gathers are in flight at once.
        uint32_t target[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const uint32_t c = (mask >> s) & 1u ? ch[s] : 0u;
            target[s] = last ? uint32_t(a.leaves_start + 2ull * c) : a.positions[s_lv.first[l + 1] + c];
        }
        uint32_t off = 1;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            if ((mask >> s) & 1u) {
                a.words[pos + off] = target[s];
                ++off;
            }
        }
    }
    for (uint64_t r = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; r < a.num_leaves; r += stride) {
        const uint64_t leaf = a.leaves[r];
        a.words[a.leaves_start + 2 * r] = uint32_t(leaf);
        a.words[a.leaves_start + 2 * r + 1] = uint32_t(leaf >> 32);
    }
}

// ---------------------------------------------------------------------------
// A DAG's arrays to pinned host memory in one launch.  A workgroup takes pieces
// of 16 KB: 4 loads of 16 bytes per thread in flight, then 4 stores over the
// link.  A DAG has three arrays a level: as copies of their own, most of them a
// few KB, they took 7 to 10 us each (0.56 MB in 19 arrays: 125 us, now 26; 10.5
// MB in 28: 389 and 207; 73 MB: 1479 and 1358, the link's 54 GB/s).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads) void k_copy_out(CopyOut a)
{
    constexpr uint32_t kWords = uint32_t(kCopyPiece / 16), kAhead = kWords / kThreads;
    for (uint32_t piece = blockIdx.x; piece < a.pieces; piece += gridDim.x) {
        uint32_t at = piece;
        int g = 0;
        for (;; ++g) {
            const uint32_t here = uint32_t((a.seg[g].bytes + kCopyPiece - 1) / kCopyPiece);
            if (at < here) break;
            at -= here;
        }
        const uint64_t bytes = a.seg[g].bytes;
        const uint64_t words = bytes / 16, first = uint64_t(at) * kWords + threadIdx.x;
        const uint4* __restrict__ src = static_cast<const uint4*>(a.seg[g].src);
        uint4* __restrict__ dst = static_cast<uint4*>(a.seg[g].dst);
        if (words) {
            uint4 v[kAhead];
#pragma unroll
            for (uint32_t k = 0; k < kAhead; ++k) v[k] = src[min(first + uint64_t(k) * kThreads, words - 1)];
#pragma unroll
            for (uint32_t k = 0; k < kAhead; ++k)
                if (first + uint64_t(k) * kThreads < words) dst[first + uint64_t(k) * kThreads] = v[k];
        }
        // The last bytes of a segment, with its first piece.
        const uint64_t tail = 16 * words + threadIdx.x;
        if (at == 0 && tail < bytes)
            static_cast<uint8_t*>(a.seg[g].dst)[tail] = static_cast<const uint8_t*>(a.seg[g].src)[tail];
    }
}

// ---------------------------------------------------------------------------
// Merge insert (MergeDAGs, src/DAGCompression.cu:1109-1320): the nodes of one
// level of many sub-DAGs, concatenated, enter one shared dedup table.  A node's
// hash depends only on its content, so it is reused; its children are remapped
// from sub-DAG-local indices to the merged level below through that level's
// slot and rank arrays.  Leaves (ordered == 0) go into the hashed leaf table.
// ---------------------------------------------------------------------------
__global__ void k_merge_insert(const MergeSource* __restrict__ src, uint32_t nsrc, uint64_t total,
                               const uint32_t* __restrict__ child_slot_of,
                               const uint32_t* __restrict__ child_rank_of_slot, uint8_t* __restrict__ masks_out,
                               uint32_t* __restrict__ children_out, uint64_t* __restrict__ tk,
                               uint32_t* __restrict__ trep, const uint32_t* __restrict__ log2_ptr,
                               uint32_t* __restrict__ slot_of, BuildCounters* __restrict__ c, int ordered)
{
    const uint32_t lg = *log2_ptr;
    const uint64_t limit = (1ull << lg) + kTableOverflow;
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
    for (uint64_t gi = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; gi < total; gi += stride) {
        uint32_t lo = 0, hi = nsrc;  // src[lo].first <= gi < src[hi].first
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) / 2;
            if (src[mid].first <= gi) lo = mid;
            else hi = mid;
        }
        const MergeSource& s = src[lo];
        const uint64_t i = gi - s.first;
        if (!ordered) {
            bool won;
            slot_of[gi] = hashed_insert(tk, lg, s.hashes[i], won, (unsigned long long*)&c->error);
            continue;
        }
        const uint64_t key = s.hashes[i];
        const uint4* cs = reinterpret_cast<const uint4*>(s.children + 8 * i);
        const uint4 a = cs[0], b = cs[1];
        uint32_t ch[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (ch[k] != kEmptyChild) ch[k] = child_rank_of_slot[child_slot_of[s.child_first + ch[k]]];
        masks_out[gi] = s.masks[i];
        uint4* dst = reinterpret_cast<uint4*>(children_out + 8 * gi);
        dst[0] = make_uint4(ch[0], ch[1], ch[2], ch[3]);
        dst[1] = make_uint4(ch[4], ch[5], ch[6], ch[7]);
        slot_of[gi] = ordered_insert(tk, trep, lg, limit, key, uint32_t(gi), c);
    }
}

// ---------------------------------------------------------------------------
// Resident DAG (served mode): one dedup table per level that persists across
// insertions.  A resident node is identified by its table slot; its record
// (mask, children as slots of the level below) is stored at that slot by the
// call that placed its key, and rep[slot] = slot, so the level extract reads
// a resident table like a build's.  Wave-aggregated counts of placed keys
// track each table's occupancy.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void count_placed(bool won, unsigned long long* occupied)
{
    const uint64_t wins = __ballot(won);
    if (wins && lane_id() == uint32_t(__ffsll((long long)wins) - 1))
        atomicAdd(occupied, (unsigned long long)__popcll(wins));
}

// Leaves of a round (unique masks) into the resident leaf table.
__global__ void k_resident_leaves(const uint64_t* __restrict__ leaves, uint64_t count, uint64_t* __restrict__ tk,
                                  uint32_t lg, uint32_t* __restrict__ slot_of, unsigned long long* __restrict__ occupied,
                                  unsigned long long* __restrict__ err)
{
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
    // Wave-uniform trip count (count_placed is a wave ballot).
    for (uint64_t base = uint64_t(blockIdx.x) * blockDim.x; base < count; base += stride) {
        const uint64_t i = base + threadIdx.x;
        bool won = false;
        if (i < count) slot_of[i] = hashed_insert(tk, lg, leaves[i], won, err);
        count_placed(won, occupied);
    }
}

// Nodes of one round level into the resident table of that level; children
// (round ranks of the level below) become resident slots through child_slot_of.
__global__ void k_resident_level(ResidentLevelArgs a)
{
    const uint64_t limit = (1ull << a.lg) + kTableOverflow;
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
    for (uint64_t base = uint64_t(blockIdx.x) * blockDim.x; base < a.count; base += stride) {
        const uint64_t i = base + threadIdx.x;
        bool won = false;
        if (i < a.count) {
            const uint32_t slot = ordered_probe(a.table_keys, a.lg, limit, a.hashes[i], won, a.err);
            if (won) {
                const uint4* cs = reinterpret_cast<const uint4*>(a.children + 8 * i);
                const uint4 c0 = cs[0], c1 = cs[1];
                uint32_t ch[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    if (ch[k] != kEmptyChild) ch[k] = a.child_slot_of[ch[k]];
                uint4* dst = reinterpret_cast<uint4*>(a.rec_children + 8 * uint64_t(slot));
                dst[0] = make_uint4(ch[0], ch[1], ch[2], ch[3]);
                dst[1] = make_uint4(ch[4], ch[5], ch[6], ch[7]);
                a.rec_masks[slot] = a.masks[i];
                a.table_rep[slot] = slot;
            }
            a.slot_of[i] = slot;
        }
        count_placed(won, a.occupied);
    }
}

// One thread per chunk slot s: walks the round's top levels along s's child
// indices; a chunk present in the round gets its root's resident slot and hash.
// A chunk at a slot that already holds one sets kErrSlotFilled.
constexpr int kRootThreads = 256;

__global__ __launch_bounds__(kRootThreads) void k_resident_roots(ResidentRootArgs a)
{
    const uint32_t slots = 1u << (3 * a.top_levels);
    for (uint32_t s = threadIdx.x; s < slots; s += kRootThreads) {
        uint64_t node = 0;
        bool present = a.has_root;
        for (int l = 0; l < a.top_levels && present; ++l) {
            const uint32_t b = (s >> (3 * (a.top_levels - 1 - l))) & 7u;
            if (!((a.masks[l][node] >> b) & 1u)) present = false;
            else node = a.children[l][8 * node + b];
        }
        uint64_t hash = 0;
        if (present) {
            const uint32_t slot = a.root_slot_of[node];
            if (a.root_slot[s] != kEmptyChild) {
                atomicOr(a.err, (unsigned long long)kErrSlotFilled);
            } else {
                a.root_slot[s] = slot;
                hash = a.root_table_keys[slot];
            }
        }
        a.root_hash[s] = hash;
    }
}

// One workgroup checks the device chunk offsets of a batched build and sets
// its key count (0 when they are invalid, so that no kernel reads past them).
constexpr int kCountThreads = 1024;

__global__ __launch_bounds__(kCountThreads) void k_batch_count(const uint64_t* __restrict__ offsets,
                                                               uint64_t num_chunks, uint64_t n_bound,
                                                               uint64_t* __restrict__ n_out,
                                                               unsigned long long* __restrict__ err)
{
    __shared__ uint32_t s_bad;
    if (threadIdx.x == 0) s_bad = offsets[0] != 0 || offsets[num_chunks] > n_bound;
    __syncthreads();
    for (uint64_t c = threadIdx.x; c < num_chunks; c += kCountThreads)
        if (offsets[c + 1] < offsets[c]) s_bad = 1;
    __syncthreads();
    if (threadIdx.x == 0) {
        *n_out = s_bad ? 0 : offsets[num_chunks];
        if (s_bad) atomicOr(err, (unsigned long long)kErrOffsets);
    }
}

// Keys of several device arrays, back to back.  A workgroup copies a tile of
// kGatherTile destination keys: one binary search finds the tile's first
// source, then the sources overlapping the tile are copied in turn, each as a
// contiguous, coalesced range.
constexpr uint32_t kGatherTile = 4096;

__global__ __launch_bounds__(kThreads) void k_gather_keys(const GatherSource* __restrict__ src, uint32_t nsrc,
                                                          uint64_t total, uint64_t* __restrict__ dst)
{
    __shared__ uint32_t s_first;
    const uint64_t ntiles = (total + kGatherTile - 1) / kGatherTile;
    for (uint64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const uint64_t t0 = tile * kGatherTile;
        const uint64_t t1 = min(t0 + kGatherTile, total);
        if (threadIdx.x == 0) {
            uint32_t lo = 0, hi = nsrc;  // src[lo].start <= t0 < src[hi].start
            while (hi - lo > 1) {
                const uint32_t mid = (lo + hi) / 2;
                if (src[mid].start <= t0) lo = mid;
                else hi = mid;
            }
            s_first = lo;
        }
        __syncthreads();
        uint32_t sidx = s_first;
        for (uint64_t pos = t0; pos < t1; ++sidx) {
            const GatherSource g = src[sidx];
            const uint64_t end = min(t1, sidx + 1 < nsrc ? src[sidx + 1].start : total);
            for (uint64_t i = pos + threadIdx.x; i < end; i += kThreads)
                dst[i] = __builtin_nontemporal_load(g.keys + (i - g.start));
            pos = end;
        }
        __syncthreads();  // s_first is rewritten by the next tile
    }
}

// The filled chunk slots in slot (Morton) order: codes, root slots, count.
__global__ __launch_bounds__(kRootThreads) void k_resident_root_list(const uint32_t* __restrict__ root_slot,
                                                                     uint32_t slots, uint64_t* __restrict__ codes,
                                                                     uint32_t* __restrict__ list_slots,
                                                                     uint64_t* __restrict__ count)
{
    __shared__ uint32_t s_scan[kRootThreads / kWave];
    uint32_t placed = 0;
    for (uint32_t base = 0; base < slots; base += kRootThreads) {
        const uint32_t s = base + threadIdx.x;
        const bool filled = s < slots && root_slot[s] != kEmptyChild;
        uint32_t total;
        const uint32_t ex = block_exclusive_scan<kRootThreads>(filled ? 1u : 0u, s_scan, total);
        if (filled) {
            codes[placed + ex] = s;
            list_slots[placed + ex] = root_slot[s];
        }
        placed += total;
    }
    if (threadIdx.x == 0) *count = placed;
}

}  // namespace

// ---------------------------------------------------------------------------
// Host launchers.
// ---------------------------------------------------------------------------
void launch_fill_u64(hipStream_t s, uint64_t* p, uint64_t count, uint64_t value, uint64_t set_at, uint64_t set_value)
{
    if (count == 0) return;
    TimedLaunch t(kKFill, s);
    hipLaunchKernelGGL(k_fill_u64, dim3(grid_for((count + kThreads - 1) / kThreads, 8)), dim3(kThreads), 0, s, p, count,
                       value, set_at, set_value);
}

void launch_scan_counts(hipStream_t s, const uint32_t* counts, uint64_t* offsets, const uint64_t* items_dev,
                        uint64_t per_tile, uint64_t* total_out, uint64_t items_host)
{
    TimedLaunch t(kKScanCounts, s);
    hipLaunchKernelGGL(k_scan_counts, dim3(1), dim3(kScanThreads), 0, s, counts, offsets, items_dev, per_tile, total_out,
                       items_host);
}

void launch_cell_reduce(hipStream_t s, const CellArgs& a, BuildCounters* c)
{
    const uint64_t runs = cell_runs(a.cells, a.run_cells);
    {
        TimedLaunch t(kKLeafReduce, s);
        hipLaunchKernelGGL(k_cell_reduce, dim3(resident_grid(k_cell_reduce, kCellThreads, runs)), dim3(kCellThreads), 0,
                           s, a, &c->n);
    }
    TimedLaunch t(kKLeafCompact, s);
    hipLaunchKernelGGL(k_cell_compact, dim3(resident_grid(k_cell_compact, kThreads, runs)), dim3(kThreads), 0, s, a,
                       &c->n, &c->leaf_positions, reinterpret_cast<unsigned long long*>(&c->error));
}

template <typename K>
void launch_leaf_reduce(hipStream_t s, const K* sorted, BuildCounters* c, uint32_t group_bits, uint64_t* reg_code,
                        uint64_t* reg_mask, uint64_t* lp_code, uint64_t* lp_mask, uint64_t lp_capacity,
                        uint32_t* tile_counts, uint64_t* tile_offsets, uint64_t n_bound,
                        uint64_t code_mask, const ChunkPrefix& buckets)
{
    const uint64_t chunks = (n_bound + kReduceChunk - 1) / kReduceChunk;
    const uint64_t units = (chunks + kReduceWaves - 1) / kReduceWaves;
    {
        TimedLaunch t(kKLeafReduce, s);
        bool bucketed = false;
        if constexpr (sizeof(K) == 4) {
            if (buckets.offsets) {
                bucketed = true;
                if (buckets.num_chunks <= kLdsBuckets)
                    hipLaunchKernelGGL((k_leaf_reduce<K, kBucketsLds>),
                                       dim3(resident_grid(k_leaf_reduce<K, kBucketsLds>, kThreads, units)),
                                       dim3(kThreads), 0, s, sorted, &c->n, code_mask, group_bits, reg_code, reg_mask,
                                       tile_counts,
                                       reinterpret_cast<unsigned long long*>(&c->error), buckets);
                else
                    hipLaunchKernelGGL((k_leaf_reduce<K, kBucketsGlobal>),
                                       dim3(resident_grid(k_leaf_reduce<K, kBucketsGlobal>, kThreads, units)),
                                       dim3(kThreads), 0, s, sorted, &c->n, code_mask, group_bits, reg_code, reg_mask,
                                       tile_counts,
                                       reinterpret_cast<unsigned long long*>(&c->error), buckets);
            }
        }
        if (!bucketed)
            hipLaunchKernelGGL((k_leaf_reduce<K, kBucketsNone>),
                               dim3(resident_grid(k_leaf_reduce<K, kBucketsNone>, kThreads, units)), dim3(kThreads), 0,
                               s, sorted, &c->n, code_mask, group_bits, reg_code, reg_mask, tile_counts, reinterpret_cast<unsigned long long*>(&c->error), ChunkPrefix{});
    }
    launch_scan_counts(s, tile_counts, tile_offsets, &c->n, kReduceChunk, &c->leaf_positions);
    {
        TimedLaunch t(kKLeafCompact, s);
        hipLaunchKernelGGL(k_leaf_compact, dim3(grid_for(units, 8)), dim3(kThreads), 0, s, reg_code, reg_mask, tile_counts,
                           tile_offsets, &c->n, lp_code, lp_mask, lp_capacity,
                           reinterpret_cast<unsigned long long*>(&c->error));
    }
}
template void launch_leaf_reduce<uint64_t>(hipStream_t, const uint64_t*, BuildCounters*, uint32_t, uint64_t*,
                                           uint64_t*, uint64_t*, uint64_t*, uint64_t, uint32_t*, uint64_t*, uint64_t, uint64_t, const ChunkPrefix&);
template void launch_leaf_reduce<uint32_t>(hipStream_t, const uint32_t*, BuildCounters*, uint32_t, uint64_t*,
                                           uint64_t*, uint64_t*, uint64_t*, uint64_t, uint32_t*, uint64_t*, uint64_t, uint64_t, const ChunkPrefix&);

void launch_table_clear(hipStream_t s, const TableClears& a)
{
    TimedLaunch t(kKTableClear, s);
    uint64_t most = 1;
    for (int i = 0; i < a.num; ++i) most = std::max(most, a.table[i].slot_bound);
    hipLaunchKernelGGL(k_table_clear, dim3(grid_for((most + kThreads - 1) / kThreads, 8)), dim3(kThreads), 0, s, a);
}

void launch_leaf_insert(hipStream_t s, const uint64_t* lp_mask, const uint64_t* count_ptr, uint64_t* table_keys,
                        const uint32_t* log2_ptr, uint32_t* lp_slot, uint64_t n_bound, unsigned long long* err)
{
    TimedLaunch t(kKLeafInsert, s);
    hipLaunchKernelGGL(k_leaf_insert, dim3(grid_for((n_bound + kThreads * kInsertIpt - 1) / (kThreads * kInsertIpt), 8)),
                       dim3(kThreads), 0, s, lp_mask, count_ptr, table_keys, log2_ptr, lp_slot, err);
}

void launch_leaf_order(hipStream_t s, const LeafOrderArgs& a, uint64_t slot_bound, uint64_t leaf_bound)
{
    TimedLaunch t(kKLeafOrder, s);
    if (order_is_small(slot_bound, leaf_bound)) {
        hipLaunchKernelGGL(k_order_small, dim3(1), dim3(kSampleThreads), 0, s, a.table_keys, a.table_log2, a.out,
                           a.rank_of_slot, a.count);
        return;
    }
    const int grid = grid_for((slot_bound + kOrderTile - 1) / kOrderTile, 4);
    hipLaunchKernelGGL(k_leaf_sample, dim3(1), dim3(kSampleThreads), 0, s, a.table_keys, a.table_log2, a.split);
    hipLaunchKernelGGL(k_order_count, dim3(grid), dim3(kThreads), 0, s, a.table_keys, a.table_log2, a.split, a.totals);
    hipLaunchKernelGGL(k_order_scatter, dim3(grid), dim3(kThreads), 0, s, a.table_keys, a.table_log2, a.split, a.totals,
                       a.totals + kOrderMaxBuckets, a.list_keys[0], a.list_slots[0]);
    // At most one bucket per kOrderMean / 2 leaves (the sample's error aside;
    // the workgroups stride over the buckets there are).
    const uint64_t buckets = std::min<uint64_t>(kOrderMaxBuckets, std::max<uint64_t>(1, leaf_bound / (kOrderMean / 2)));
    hipLaunchKernelGGL(k_order_sort, dim3(uint32_t(buckets)), dim3(kOrderSortThreads), 0, s, a.split, a.totals, a.list_keys[0],
                       a.list_slots[0], a.list_keys[1], a.list_slots[1], a.out, a.rank_of_slot, a.count);
}

void launch_sketch(hipStream_t s, const uint64_t* values, const uint64_t* count_ptr, uint32_t* regs, uint64_t n_bound)
{
    TimedLaunch t(kKSketch, s);
    // Few workgroups: each merges its registers into the global ones once.
    const uint64_t rounds = (n_bound + uint64_t(kThreads) * kSketchIpt - 1) / (uint64_t(kThreads) * kSketchIpt);
    hipLaunchKernelGGL(k_sketch, dim3(grid_for(rounds, 1)), dim3(kThreads), 0, s, values, count_ptr, regs);
}

void launch_sketch_estimate(hipStream_t s, const uint32_t* regs, const uint64_t* bound_ptr, uint64_t* estimate)
{
    TimedLaunch t(kKSketch, s);
    hipLaunchKernelGGL(k_sketch_estimate, dim3(1), dim3(kEstimateThreads), 0, s, regs, bound_ptr, estimate);
}

uint32_t level_build_parts(uint64_t child_bound)
{
    return uint32_t(std::min<uint64_t>(kMaxParts, resident_grid(k_level_build, kThreads, tiles(child_bound, kBuildTile))));
}

uint32_t level_extract_parts(uint64_t slot_bound)
{
    return uint32_t(std::min<uint64_t>(kMaxParts, resident_grid(k_level_extract, kThreads, tiles(slot_bound, kExtractTile))));
}

void launch_level_count(hipStream_t s, const uint64_t* codes, const uint64_t* count, uint64_t bound, uint32_t* parts,
                        uint64_t* pre, int level, int lowest)
{
    TimedLaunch t(kKLevelCount, s);
    hipLaunchKernelGGL(k_level_count, dim3(level_build_parts(bound)), dim3(kThreads), 0, s, codes, count, parts, pre,
                       level, lowest);
}

void launch_level_build(hipStream_t s, const LevelBuildArgs& a, uint64_t child_bound)
{
    TimedLaunch t(kKLevelBuild, s);
    hipLaunchKernelGGL(k_level_build, dim3(level_build_parts(child_bound)), dim3(kThreads), 0, s, a);
}

void launch_level_tail(hipStream_t s, const TailArgs& a)
{
    TimedLaunch t(kKLevelTail, s);
    hipLaunchKernelGGL(k_level_tail, dim3(1), dim3(kTailThreads), 0, s, a);
}

void launch_extract_count(hipStream_t s, const ExtractCounts& a, const TableClears* clear)
{
    uint32_t grid = 0;
    for (int i = 0; i < a.num; ++i) grid += a.table[i].num_parts;
    if (grid == 0) return;
    TimedLaunch t(kKExtractCount, s);
    const TableClears tc = clear ? *clear : TableClears{};
    hipLaunchKernelGGL(k_extract_count, dim3(grid), dim3(kThreads), 0, s, a, tc);
}

void launch_level_extract(hipStream_t s, const LevelExtractArgs& a, uint64_t slot_bound)
{
    TimedLaunch t(kKLevelExtract, s);
    hipLaunchKernelGGL(k_level_extract, dim3(level_extract_parts(slot_bound)), dim3(kThreads), 0, s, a);
}

void launch_level_check(hipStream_t s, const uint32_t* parent_slots, const uint32_t* table_rep,
                        const uint8_t* parent_masks, const uint32_t* parent_children, const uint64_t* count_ptr,
                        uint64_t* collisions, uint64_t n_bound)
{
    TimedLaunch t(kKLevelCheck, s);
    hipLaunchKernelGGL(k_level_check, dim3(grid_for((n_bound + kThreads - 1) / kThreads, 8)), dim3(kThreads), 0, s,
                       parent_slots, table_rep, parent_masks, parent_children, count_ptr, collisions);
}

// ---------------------------------------------------------------------------
// Point query against the flat layout, walking it as the reference's tracer
// does (src/DAGTracer.cu:85-176): a node is its child mask word followed by
// one absolute word index per set slot; after depth - 2 nodes the index
// names a leaf, two words of 4x4x4 occupancy (low word first).  The slot of
// level l is bits [3(depth-1-l), 3(depth-l)) of the code.
// out[i]: 1 set, 0 not set (or the code is outside 2^(3*depth)), 2 the walk
// left the words (not a valid layout).
// ---------------------------------------------------------------------------
__global__ void k_query_voxels(const uint32_t* __restrict__ words, uint64_t n_words, int depth,
                               const uint64_t* __restrict__ codes, uint64_t n, uint8_t* __restrict__ out)
{
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
        const uint64_t c = codes[i];
        uint8_t r = 3;  // walk in progress
        if (n_words == 0 || (c >> (3 * depth)) != 0) r = 0;
        uint64_t idx = 0;
        for (int l = 0; r == 3 && l < depth - 2; ++l) {
            if (idx >= n_words) {
                r = 2;
                break;
            }
            const uint32_t mask = words[idx];
            const uint32_t slot = uint32_t(c >> (3 * (depth - 1 - l))) & 7u;
            if (mask > 0xFFu) {
                r = 2;
            } else if (!((mask >> slot) & 1u)) {
                r = 0;
            } else {
                const uint64_t at = idx + 1 + uint32_t(__popc(mask & ((1u << slot) - 1u)));
                if (at >= n_words) r = 2;
                else idx = words[at];
            }
        }
        if (r == 3) {
            if (idx + 1 >= n_words) {
                r = 2;
            } else {
                const uint32_t bit = uint32_t(c & 63u);
                r = uint8_t((words[idx + (bit >> 5)] >> (bit & 31u)) & 1u);
            }
        }
        out[i] = r;
    }
}

void launch_query_voxels(hipStream_t s, const uint32_t* words, uint64_t n_words, int depth, const uint64_t* codes,
                         uint64_t n, uint8_t* out)
{
    if (n == 0) return;
    TimedLaunch t(kKQueryVoxels, s);
    hipLaunchKernelGGL(k_query_voxels, dim3(grid_for((n + kThreads - 1) / kThreads, 8)), dim3(kThreads), 0, s, words,
                       n_words, depth, codes, n, out);
}

void launch_final(hipStream_t s, const FinalArgs& a)
{
    if (a.total_nodes == 0 && a.num_leaves == 0) return;
    if (a.total_nodes) {
        const uint64_t tiles = (a.total_nodes + kFinalTile - 1) / kFinalTile;
        const uint32_t parts = uint32_t(std::min<uint64_t>(kMaxParts, resident_grid(k_final_positions, kThreads, tiles)));
        if (parts > 1) {  // one part starts at 0
            TimedLaunch t(kKFinalCount, s);
            hipLaunchKernelGGL(k_final_count, dim3(parts), dim3(kThreads), 0, s, a);
        }
        {
            TimedLaunch t(kKFinalPositions, s);
            hipLaunchKernelGGL(k_final_positions, dim3(parts), dim3(kThreads), 0, s, a);
        }
    }
    const uint64_t work = std::max(a.total_nodes, a.num_leaves);
    {
        TimedLaunch t(kKFinalWrite, s);
        hipLaunchKernelGGL(k_final_write, dim3(grid_for((work + kThreads - 1) / kThreads, 8)), dim3(kThreads), 0, s, a);
    }
}

void launch_copy_out(hipStream_t s, const CopyOut& a)
{
    if (a.pieces == 0) return;
    TimedLaunch t(kKCopyOut, s);
    hipLaunchKernelGGL(k_copy_out, dim3(grid_for(a.pieces, 2)), dim3(kThreads), 0, s, a);
}

void launch_resident_leaves(hipStream_t s, const uint64_t* leaves, uint64_t count, uint64_t* table_keys, uint32_t lg,
                            uint32_t* slot_of, unsigned long long* occupied, unsigned long long* err)
{
    if (count == 0) return;
    TimedLaunch t(kKResidentInsert, s);
    hipLaunchKernelGGL(k_resident_leaves, dim3(grid_for((count + kThreads - 1) / kThreads, 8)), dim3(kThreads), 0, s,
                       leaves, count, table_keys, lg, slot_of, occupied, err);
}

void launch_resident_level(hipStream_t s, const ResidentLevelArgs& a)
{
    if (a.count == 0) return;
    TimedLaunch t(kKResidentInsert, s);
    hipLaunchKernelGGL(k_resident_level, dim3(grid_for((a.count + kThreads - 1) / kThreads, 8)), dim3(kThreads), 0, s,
                       a);
}

void launch_batch_count(hipStream_t s, const uint64_t* offsets, uint64_t num_chunks, uint64_t n_bound, uint64_t* n_out,
                        unsigned long long* err)
{
    TimedLaunch t(kKFill, s);
    hipLaunchKernelGGL(k_batch_count, dim3(1), dim3(kCountThreads), 0, s, offsets, num_chunks, n_bound, n_out, err);
}

void launch_gather_keys(hipStream_t s, const GatherSource* src, uint32_t nsrc, uint64_t total, uint64_t* dst)
{
    if (total == 0 || nsrc == 0) return;
    TimedLaunch t(kKFill, s);
    hipLaunchKernelGGL(k_gather_keys, dim3(grid_for((total + kGatherTile - 1) / kGatherTile, 8)), dim3(kThreads), 0, s,
                       src, nsrc, total, dst);
}

void launch_resident_roots(hipStream_t s, const ResidentRootArgs& a)
{
    TimedLaunch t(kKResidentInsert, s);
    hipLaunchKernelGGL(k_resident_roots, dim3(1), dim3(kRootThreads), 0, s, a);
}

void launch_resident_root_list(hipStream_t s, const uint32_t* root_slot, uint32_t slots, uint64_t* codes,
                               uint32_t* list_slots, uint64_t* count)
{
    TimedLaunch t(kKResidentInsert, s);
    hipLaunchKernelGGL(k_resident_root_list, dim3(1), dim3(kRootThreads), 0, s, root_slot, slots, codes, list_slots,
                       count);
}

void launch_merge_insert(hipStream_t s, const MergeSource* d_sources, uint32_t num_sources, uint64_t total,
                         const uint32_t* child_slot_of, const uint32_t* child_rank_of_slot, uint8_t* masks_out,
                         uint32_t* children_out, uint64_t* table_keys, uint32_t* table_rep, const uint32_t* table_log2,
                         uint32_t* slot_of, BuildCounters* counters, int ordered)
{
    if (total == 0) return;
    TimedLaunch t(kKMergeInsert, s);
    hipLaunchKernelGGL(k_merge_insert, dim3(grid_for((total + kThreads - 1) / kThreads, 8)), dim3(kThreads), 0, s,
                       d_sources, num_sources, total, child_slot_of, child_rank_of_slot, masks_out, children_out,
                       table_keys, table_rep, table_log2, slot_of, counters, ordered);
}

}  // namespace svdag
