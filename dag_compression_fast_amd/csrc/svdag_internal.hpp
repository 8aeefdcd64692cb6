// svdag_internal.hpp -- host-side launchers and device-memory layouts shared by
// the kernels (svdag_sort.hip, svdag_build.hip) and the C-ABI driver
// (svdag_api.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "svdag.h"

namespace svdag {

// ---- per-kernel timing ----------------------------------------------------
// Counterpart of the reference's per-operation event timer
// (src/CudaPerfRecorder.h:5-60, used at src/DAGCompression.cu:352, 384, 413...),
// which synchronises after every operation.  Here a launch is bracketed by two
// events on its stream when a recorder is active on the calling thread; the
// pairs are resolved after the call's single synchronisation.
enum KernelId : int {
    kKHistogram = 0,
    kKSortCount,
    kKSortScan,
    kKSortScatterKeys,
    kKFill,
    kKScanCounts,
    kKLeafReduce,
    kKLeafCompact,
    kKTableClear,
    kKLeafInsert,
    kKLeafOrder,  // ascending order of the unique leaves
    kKLevelCount,
    kKLevelBuild,
    kKLevelCheck,
    kKExtractCount,
    kKLevelExtract,
    kKFinalCount,
    kKFinalPositions,
    kKFinalWrite,
    kKMergeInsert,
    kKSketch,
    kKLevelTail,
    kKQueryVoxels,
    kKVoxSetup,
    kKVoxCount,
    kKVoxWrite,
    kKTracePaths,
    kKResidentInsert,
    kKSortScatterTop,  // top-digit pass of a top-digit-first key sort (64-bit in, 32-bit out)
    kKSegCount,        // segmented sort: per-tile counts
    kKSegScatter,      // segmented sort: scatter passes
    kKCopyOut,         // results to the host
    kNumKernelIds
};

struct KernelRecorder {
    virtual void begin(hipStream_t s, int id) = 0;
    virtual void end(hipStream_t s, int id) = 0;
    virtual ~KernelRecorder() = default;
};

// The recorder of the calling thread (null: no timing).
KernelRecorder*& active_recorder();

struct TimedLaunch {
    int id;
    hipStream_t s;
    TimedLaunch(int kernel, hipStream_t stream) : id(kernel), s(stream)
    {
        if (KernelRecorder* r = active_recorder()) r->begin(s, id);
    }
    ~TimedLaunch()
    {
        if (KernelRecorder* r = active_recorder()) r->end(s, id);
    }
};

// ---- radix sort -----------------------------------------------------------
// Digits are at most kMaxRadixBits wide; kRadix digit slots are reserved in
// every LDS and count array.
constexpr int kMaxRadixBits = 9;
constexpr int kRadix = 1 << kMaxRadixBits;
constexpr int kMaxPasses = 8;
// A tile is 256 threads x ipt keys: 16 (4096 keys) or 32 (8192 keys).
constexpr int kSortThreads = 256;
constexpr int kSortIptSmall = 16;
constexpr int kSortIptLarge = 32;

struct SortPlan {
    int passes;
    uint32_t shift[kMaxPasses];
    uint32_t bits[kMaxPasses];
    int ipt;  // keys per thread and tile
    // Key-only sorts rank their first pass unstably unless this is set; keys
    // equal on the sorted bits then keep their input order (a stable sort).
    bool stable;
};

// Digits of width <= max_bits covering bits [lo, hi), spread evenly.
SortPlan make_sort_plan(int lo, int hi, int max_bits = kMaxRadixBits, int ipt = kSortIptSmall);

inline uint64_t sort_tiles(uint64_t n, int ipt)
{
    const uint64_t tile = uint64_t(kSortThreads) * ipt;
    return (n + tile - 1) / tile;
}

// Device scratch of one sort: the all-pass digit histogram (passes * kRadix
// u32, zero before launch_sort) and the per-tile digit counts
// (sort_count_words u32 for any tile size, any contents).
inline uint64_t sort_zero_words(const SortPlan& p) { return uint64_t(p.passes) * kRadix; }
inline uint64_t sort_count_words(uint64_t n_bound) { return uint64_t(kRadix) * sort_tiles(n_bound, kSortIptSmall); }

// LSD radix sort of keys on the plan's bits.  With plan.stable, keys equal on
// those bits keep their input order; otherwise their order is unspecified (the first pass ranks unstably).
// n is read from device memory (*n_ptr, < 2^30); n_bound is a host upper bound
// sizing the grid and the count buffer.  Passes ping-pong between (keys_a,
// keys_b); the first pass reads keys_in.  Returns which buffer holds the result
// (0 = a, 1 = b, 2 = final); if final_keys is non-null the last
// pass writes there instead.  key_or (optional) receives the OR of all keys.
// Chunk-local input of a batched build: key i, with offsets[c] <= i <
// offsets[c + 1], becomes (c << chunk_bits) | key when the sort first reads it
// (chunk order = Morton order of the sub-volumes, src/Utils/Aabb.h:83-105).
struct ChunkPrefix {
    const uint64_t* offsets = nullptr;  // device, num_chunks + 1 entries; null: keys are global
    uint64_t num_chunks = 0;
    uint32_t chunk_bits = 0;
    unsigned long long* err = nullptr;  // receives kErrKeyRange for a key >= 2^chunk_bits
};

// Segmented key sort of a batched build (chunks back to back, in chunk order):
// tiles of at most kSegTileItems keys, none crossing a chunk, planned on the
// device from the chunk offsets (chunk_start: num_chunks + 1 device entries;
// *n_ptr keys in all, at most n_bound; *n_ptr == 0 plans nothing).  Sorts the
// chunk-local bits [lo, chunk_bits) (at most kSegMaxBits of them, in one or
// two passes of at most kMaxSegDigitBits) and writes the keys as 32-bit
// chunk-local keys (chunk_bits <= 32); a reader restores key i's chunk index
// from chunk_start (ChunkPrefix).  Returns 0 (result in keys_a), 1 (keys_b),
// or -1 when the bit span does not fit.  first_bits: the first pass's digit width (0: half the
// bits), clamped so both passes have at most kMaxSegDigitBits.
struct SegTile {
    uint64_t start;
    uint32_t count;
    uint32_t chunk;
};
constexpr uint32_t kSegTileItems = 4096;
constexpr uint32_t kSegMaxBits = 12;
constexpr uint32_t kMaxSegDigitBits = 9;
inline uint64_t seg_tile_bound(uint64_t n_bound, uint64_t num_chunks) { return n_bound / kSegTileItems + num_chunks; }
// When plain builds of 64-bit keys sort top digit first (option
// SVDAG_OPT_TOP_DIGIT_FIRST): never, from kTopFirstMinKeys keys on, always
// (where the bits fit).
constexpr int kTopFirstNever = 0, kTopFirstAuto = 1, kTopFirstAlways = 2;
constexpr uint64_t kTopFirstMinKeys = 1ull << 20;
// Scratch of the segmented sort: tiles (seg_tile_bound entries), chunk_tiles
// (num_chunks + 1), counts (tile bound << kMaxSegDigitBits), totals and starts
// (num_chunks << kMaxSegDigitBits each), the tile count.
struct SegScratch {
    SegTile* tiles;
    uint32_t* chunk_tiles;
    uint32_t* counts;
    uint32_t* totals;
    uint32_t* starts;
    uint64_t* ntiles;
    uint32_t* slices;      // sums over several tiles, slice_words words (any number)
    uint64_t slice_words;
};
template <typename KI>
int launch_segmented_sort(hipStream_t stream, const KI* keys_in, uint32_t* keys_a, uint32_t* keys_b,
                          const uint64_t* chunk_start, uint64_t num_chunks, const uint64_t* n_ptr, uint64_t n_bound,
                          const SegScratch& sc, uint32_t lo, uint32_t chunk_bits, unsigned long long* err,
                          uint32_t first_bits = 0);

// Key sort of a plain build of 64-bit keys on bits [lo, top_shift + top_bits),
// top digit first: a pass on the top digit writes each key's bits below
// top_shift (< 2^32) into `local`, grouped by top digit, with the groups'
// starts in bucket_start (2^top_bits + 1 entries); the segmented sort then
// sorts [lo, top_shift) inside each group, still as 32-bit bucket-local keys.  zero:
// kRadix u32, zero at launch; counts: sort_count_words(n_bound) u32.  Returns
// as launch_segmented_sort (0: keys_a, 1: keys_b), -1 when the bits do not fit
// (top_shift > 32, or more than kSegMaxBits below it).
int launch_top_digit_sort(hipStream_t stream, const uint64_t* keys_in, uint32_t* local, uint32_t* keys_a,
                          uint32_t* keys_b, int ipt, uint32_t top_shift, uint32_t top_bits, uint32_t lo,
                          const uint64_t* n_ptr, uint64_t n_bound, uint32_t* zero, uint32_t* counts,
                          unsigned long long* key_or, uint64_t* bucket_start, const SegScratch& sc,
                          unsigned long long* err);

// One pass grouping the keys by their top digit [shift, shift + bits) (shift +
// bits <= 32), written as 32-bit keys (the bits below shift at least); starts[d]
// = first key of digit d, 2^bits entries.  zero, counts, key_or as above.
// Returns 0, or -1 when the digit does not fit.
template <typename K>
int launch_cell_sort(hipStream_t stream, const K* keys_in, uint32_t* keys_out, int ipt, uint32_t shift, uint32_t bits,
                     const uint64_t* n_ptr, uint64_t n_bound, uint32_t* zero, uint32_t* counts,
                     unsigned long long* key_or, uint32_t* starts);

// Stable sort of 64-bit keys on bits [0, top_shift + top_bits) (top_shift <=
// 32), top digit first.  launch_top_histogram: the digit totals (zero), the
// top digit's tile counts and group starts, and the OR of the keys, also into
// *or_out (pinned).  launch_top_plan: the tables that the passes need.
// launch_top_passes: below = digits covering [0, top_shift); KL = uint32_t when
// no key has a bit above the sorted ones, else uint64_t; first and second: n
// keys each, used in turn (for uint64_t, second may be keys_out if below.passes
// is odd, and first if it is even; neither may overlap keys_in then).  The
// segmented sort's scratch has 2^top_bits chunks and digits of below's widths.
void launch_top_histogram(hipStream_t stream, const uint64_t* keys_in, uint32_t top_shift, uint32_t top_bits,
                          const uint64_t* n_ptr, uint64_t n, uint32_t* zero, uint32_t* counts,
                          unsigned long long* key_or, uint64_t* bucket_start, unsigned long long* or_out);
void launch_top_plan(hipStream_t stream, uint32_t top_bits, const uint64_t* n_ptr, uint64_t n, const uint32_t* zero,
                     uint32_t* counts, const uint64_t* bucket_start, const SegScratch& sc);
template <typename KL>
void launch_top_passes(hipStream_t stream, const uint64_t* keys_in, KL* first, KL* second, uint64_t* keys_out,
                       uint32_t top_shift, uint32_t top_bits, const SortPlan& below, const uint64_t* n_ptr, uint64_t n,
                       uint32_t* counts, const uint64_t* bucket_start, const SegScratch& sc);
// From how many keys svdag_sort_keys takes it.
constexpr uint64_t kTopSortMinKeys = 1ull << 22;

template <typename K>
int launch_sort(hipStream_t stream, const SortPlan& plan, const K* keys_in, K* keys_a, K* keys_b, K* final_keys,
                const uint64_t* n_ptr, uint64_t n_bound, uint32_t* zero, uint32_t* counts,
                unsigned long long* key_or, const ChunkPrefix& prefix = ChunkPrefix{});

// ---- build ----------------------------------------------------------------
constexpr uint32_t kTableOverflow = 4096;  // slots past 2^log2 for ordered tables

// Device counters of one build; zeroed at the start.
struct BuildCounters {
    uint64_t n;
    unsigned long long key_or;
    uint64_t leaf_positions;                  // L0
    uint64_t unique_leaves;                   // L
    uint64_t pre[SVDAG_MAX_LEVELS];           // M_l
    uint64_t uniq[SVDAG_MAX_LEVELS];          // Q_l
    uint64_t words[SVDAG_MAX_LEVELS];         // W_l
    uint64_t collisions;
    uint64_t error;                           // kErr* bits
    uint32_t table_log2[SVDAG_MAX_LEVELS + 1];  // [l] level tables, [MAX] leaf table
    uint64_t leaf_estimate;                   // table sizing count of the leaf dedup table
};

constexpr uint64_t kErrTableOverflow = 1;
constexpr uint64_t kErrKeyRange = 2;
constexpr uint64_t kErrInternal = 4;  // a bound the kernels rely on did not hold
constexpr uint64_t kErrSlotFilled = 8;  // a resident chunk slot received a second chunk
constexpr uint64_t kErrOffsets = 16;    // device chunk offsets invalid or past the key capacity

// Tile sizes of the compaction stages; a stage over at most n items needs
// tiles(n, kXxxTile) u32 counts and u64 offsets of scratch.
constexpr uint64_t kPackTileItems = 4096;     // grouped keys per leaf-reduce chunk
constexpr uint32_t kLeafGroupBits = 9;        // low leaf-code bits the key sort leaves unsorted
constexpr uint64_t kLeafRegionItems = kPackTileItems + (1u << kLeafGroupBits);  // leaves one chunk may emit
constexpr uint64_t kBuildTileItems = 512;     // child codes per level-build tile
constexpr uint64_t kExtractTileItems = 256;   // table slots per extract tile
constexpr uint64_t kFinalTileItems = 4096;    // nodes per final-layout tile
inline uint64_t tiles(uint64_t n, uint64_t per) { return (n + per - 1) / per; }

int device_cu_count();

// Workgroups of `threads` threads of `kernel` that the device holds at once
// (its occupancy times the CU count; cached per kernel).  A kernel whose
// workgroups each walk several tiles launches at most this many: a larger grid
// leaves a partial second round of workgroups, each with a full share of tiles.
int kernel_slots(const void* kernel, int threads);
template <typename F>
inline int kernel_slots(F kernel, int threads)
{
    return kernel_slots(reinterpret_cast<const void*>(kernel), threads);
}
// Grid for `tiles` units of work: one workgroup per unit, at most kernel_slots.
template <typename F>
inline int resident_grid(F kernel, int threads, uint64_t tiles)
{
    return int(std::max<uint64_t>(1, std::min<uint64_t>(tiles, uint64_t(kernel_slots(kernel, threads)))));
}

// p[0, count) = value, except p[set_at] = set_value when set_at < count.
void launch_fill_u64(hipStream_t s, uint64_t* p, uint64_t count, uint64_t value, uint64_t set_at = ~0ull,
                     uint64_t set_value = 0);

// *n_out = offsets[num_chunks] when the device offsets start at 0, never
// decrease and end at most at n_bound; else *n_out = 0 and kErrOffsets in *err.
void launch_batch_count(hipStream_t s, const uint64_t* offsets, uint64_t num_chunks, uint64_t n_bound, uint64_t* n_out,
                        unsigned long long* err);

// One-workgroup exclusive scan of tile counts into offsets; the number of tiles
// is ceil(items / per_tile), items = *items_dev, or items_host when items_dev is
// null; the total goes to *total_out when non-null.
void launch_scan_counts(hipStream_t s, const uint32_t* counts, uint64_t* offsets, const uint64_t* items_dev,
                        uint64_t per_tile, uint64_t* total_out, uint64_t items_host = 0);


// Leaf ReduceByKey over keys grouped by code >> (6 + group_bits): per-chunk
// leaves into the regions reg_code / reg_mask (kLeafRegionItems per chunk of
// kPackTileItems keys), then compacted into lp_code / lp_mask (lp_capacity
// entries); sets
// c->leaf_positions.
// buckets.offsets non-null (32-bit keys only): the keys are local to the
// buckets of a segmented sort, key i's code is (b << buckets.chunk_bits) | key
// for the bucket b holding position i.
template <typename K>
void launch_leaf_reduce(hipStream_t s, const K* sorted, BuildCounters* c, uint32_t group_bits, uint64_t* reg_code,
                        uint64_t* reg_mask, uint64_t* lp_code, uint64_t* lp_mask, uint64_t lp_capacity,
                        uint32_t* tile_counts, uint64_t* tile_offsets, uint64_t n_bound,
                        uint64_t code_mask, const ChunkPrefix& buckets = ChunkPrefix{});

// Leaf ReduceByKey over keys grouped by cell (code >> kCellShift: 64^3 voxels,
// 4096 leaves), cell c at keys[starts[c], starts[c + 1]) (the last up to
// c->n): one workgroup per cell.  Runs of run_cells cells write their leaves
// into reg_code / reg_mask from their first key's position on (n_bound
// entries), counted in run_counts (cell_runs entries), then compacted as
// above.  Which builds take it: cells_pay.
constexpr uint32_t kCellShift = 18;
constexpr uint32_t kCellLeaves = 1u << (kCellShift - 6);
constexpr uint32_t kMaxRunCells = 32;
// Cells per run: a power of two, at most `most`; the shortest with at most
// max_runs (and 16384) runs, if `most` allows it.
inline uint32_t cell_run_length(uint64_t cells, uint64_t max_runs, uint64_t most)
{
    const uint64_t runs = std::min<uint64_t>(16384, max_runs), top = std::min<uint64_t>(kMaxRunCells, most);
    uint32_t len = 1;
    while (len < top && cells > len * runs) len *= 2;
    return len;
}
__host__ __device__ inline uint64_t cell_runs(uint64_t cells, uint32_t run_cells) { return (cells + run_cells - 1) / run_cells; }
// A cell costs its workgroup a pass over 4096 table words however few keys it
// holds: below 16 keys a cell the wave-sized groups of launch_leaf_reduce read
// less, unless there are so few cells that launches cost more than the tables.
inline bool cells_pay(uint64_t cells, uint64_t n) { return cells <= 8192 || cells <= n / 16; }
struct CellArgs {
    const uint32_t* keys;
    const uint32_t* starts;
    uint64_t cells;
    uint32_t run_cells;
    uint32_t* reg_code;
    uint64_t* reg_mask;
    uint32_t* run_counts;
    uint64_t* lp_code;
    uint64_t* lp_mask;
    uint64_t lp_capacity;
    // Non-null: the cells are those of some chunks only, chunk_cells each (a
    // power of two that run_cells divides), chunk j's at chunk_ids[j] in the
    // order of all chunks.
    const uint32_t* chunk_ids;
    uint32_t chunk_cells;
};
void launch_cell_reduce(hipStream_t s, const CellArgs& a, BuildCounters* c);

// Clears ordered (overflow > 0) and hashed tables, each sized from its count
// (device memory), and records their log2 sizes.
struct TableClears {
    int num;
    uint32_t load_shift;
    struct {
        uint64_t* keys;
        const uint64_t* count;
        uint32_t* log2_out;
        uint32_t overflow;
        uint64_t slot_bound;
    } table[SVDAG_MAX_LEVELS + 1];
    void add(uint64_t* keys, const uint64_t* count, uint32_t* log2_out, uint32_t overflow, uint64_t slot_bound)
    {
        table[num++] = {keys, count, log2_out, overflow, slot_bound};
    }
};
void launch_table_clear(hipStream_t s, const TableClears& a);

// Inserts every leaf mask into the hashed table and records its slot.
void launch_leaf_insert(hipStream_t s, const uint64_t* lp_mask, const uint64_t* count_ptr, uint64_t* table_keys,
                        const uint32_t* log2_ptr, uint32_t* lp_slot, uint64_t n_bound, unsigned long long* err);

// The occupied slots of a hashed table (2^*table_log2 slots, at most
// slot_bound; at most leaf_bound occupied): their keys in ascending order to
// out, each slot's rank to rank_of_slot, their number to *count.
constexpr uint32_t kOrderMaxLog2 = 11;
constexpr uint32_t kOrderMaxBuckets = 1u << kOrderMaxLog2;
constexpr uint64_t kOrderZeroWords = 2 * kOrderMaxBuckets;  // u32 words that must be zero at launch
// Orders that one workgroup takes whole: they need no split, totals or lists.
constexpr uint32_t kOrderCap = 4096;  // masks one LDS sort takes
constexpr uint32_t kOrderSmallSlots = 8 * kOrderCap;
inline bool order_is_small(uint64_t slot_bound, uint64_t leaf_bound)
{
    return leaf_bound <= kOrderCap && slot_bound <= kOrderSmallSlots;
}
struct LeafOrderArgs {
    const uint64_t* table_keys;
    const uint32_t* table_log2;
    uint64_t* split;          // kOrderMaxBuckets entries
    uint32_t* totals;         // kOrderZeroWords, zero: bucket totals, then cursors
    uint64_t* list_keys[2];   // leaf_bound entries each
    uint32_t* list_slots[2];
    uint64_t* out;
    uint32_t* rank_of_slot;
    uint64_t* count;
};
void launch_leaf_order(hipStream_t s, const LeafOrderArgs& a, uint64_t slot_bound, uint64_t leaf_bound);

// Distinct-count sketch (HyperLogLog, kSketchRegs registers, zero before the
// first launch) of values[0, *count_ptr), and the count a hashed table is sized
// from: 1.25 x the estimate, at most *bound_ptr.
constexpr int kSketchBits = 12;
constexpr int kSketchRegs = 1 << kSketchBits;
void launch_sketch(hipStream_t s, const uint64_t* values, const uint64_t* count_ptr, uint32_t* regs, uint64_t n_bound);
void launch_sketch_estimate(hipStream_t s, const uint32_t* regs, const uint64_t* bound_ptr, uint64_t* estimate);

// Children come in one of two forms.  With child_hash_seq, child i's hash is
// child_hash_seq[i] and its table slot is recorded as the pointer (the level's
// extract turns slots into ranks); otherwise its rank is
// child_rank_of_slot[child_slots[i]] and its hash child_hashes[rank].
struct LevelBuildArgs {
    const uint64_t* child_codes;
    const uint32_t* child_slots;
    const uint64_t* child_hash_seq;
    const uint32_t* child_rank_of_slot;
    const uint64_t* child_hashes;
    const uint64_t* child_count;
    uint64_t* parent_hashes;  // hash of parent p at p, or null
    uint64_t* parent_codes;
    uint32_t* parent_slots;
    uint8_t* parent_masks;
    uint32_t* parent_children;
    uint64_t* table_keys;
    uint32_t* table_rep;
    const uint32_t* table_log2;
    const uint32_t* parts;    // parents started in each part of the children
    // Non-null: the same counts for the level above (zero before; next_num
    // parts of *parent_count, this level's node count).
    uint32_t* next_parts;
    uint32_t next_num;
    const uint64_t* parent_count;
    BuildCounters* counters;
};
// Workgroups of a level's build and extract (their parts; at most kMaxParts and
// at most one per tile).
constexpr uint32_t kMaxParts = 2048;
uint32_t level_build_parts(uint64_t child_bound);
uint32_t level_extract_parts(uint64_t slot_bound);
// Parents started in each part of the sorted child codes (level_build_parts of
// them); with pre also the node counts of levels lowest .. level, added to
// pre[...], which the codes below determine.
void launch_level_count(hipStream_t s, const uint64_t* codes, const uint64_t* count, uint64_t bound, uint32_t* parts,
                        uint64_t* pre, int level, int lowest);
void launch_level_build(hipStream_t s, const LevelBuildArgs& a, uint64_t child_bound);

// ---- small top levels -------------------------------------------------------
// Levels 0..top with top <= kTailTopLevel hold at most 8^top <= 512 nodes; one
// workgroup builds, dedups (LDS sort by hash) and writes all of them.
constexpr int kTailTopLevel = 3;
constexpr uint32_t kTailMaxParents = 1u << (3 * kTailTopLevel);
constexpr uint32_t kTailMaxChildren = 1u << (3 * (kTailTopLevel + 1));

struct TailArgs {
    int top;                              // highest level built here
    // Children of level `top`: codes (sorted), table slots and the child level's
    // slot -> rank map, hashes by rank, and their count.
    const uint64_t* child_codes;
    const uint32_t* child_slots;
    const uint32_t* child_rank_of_slot;
    const uint64_t* child_hashes;
    const uint64_t* child_count;
    // Output levels 0..top.
    uint64_t* out_hashes[kTailTopLevel + 1];
    uint8_t* out_masks[kTailTopLevel + 1];
    uint32_t* out_children[kTailTopLevel + 1];
    BuildCounters* counters;
    int check_collisions;
};
void launch_level_tail(hipStream_t s, const TailArgs& a);

struct LevelExtractArgs {
    const uint64_t* table_keys;
    const uint32_t* table_rep;
    const uint32_t* table_log2;
    uint32_t* rank_of_slot;
    const uint8_t* parent_masks;
    const uint32_t* parent_children;
    const uint32_t* child_rank_of_slot;  // non-null: parent_children hold child slots, written as ranks
    uint64_t* out_hashes;
    uint8_t* out_masks;
    uint32_t* out_children;
    const uint32_t* parts;    // occupied slots of each part (launch_extract_count)
    uint64_t* q_count;        // receives the level's unique node count
    uint64_t* w_count;        // receives the level's word count (atomic adds)
};
void launch_level_extract(hipStream_t s, const LevelExtractArgs& a, uint64_t slot_bound);
// Occupied slots per part (level_extract_parts of its slot bound) of each of
// several ordered tables; also clears the tables of `clear`.
struct ExtractCounts {
    int num;
    struct {
        const uint64_t* keys;
        const uint32_t* log2;
        uint32_t* parts;
        uint32_t num_parts;
    } table[SVDAG_MAX_LEVELS];
    void add(const uint64_t* keys, const uint32_t* log2, uint32_t* parts, uint32_t num_parts)
    {
        table[num++] = {keys, log2, parts, num_parts};
    }
};
void launch_extract_count(hipStream_t s, const ExtractCounts& a, const TableClears* clear = nullptr);

void launch_level_check(hipStream_t s, const uint32_t* parent_slots, const uint32_t* table_rep,
                        const uint8_t* parent_masks, const uint32_t* parent_children, const uint64_t* count_ptr,
                        uint64_t* collisions, uint64_t n_bound);

// ---- final layout ---------------------------------------------------------
struct FinalLevel {
    const uint8_t* masks;
    const uint32_t* children;
    uint64_t first_node;   // index of the level's first node in the concatenation
    uint64_t num_nodes;
};
struct FinalArgs {
    FinalLevel levels[SVDAG_MAX_LEVELS];
    int num_levels;
    uint64_t total_nodes;
    const uint64_t* leaves;
    uint64_t num_leaves;
    uint64_t leaves_start;   // word index of the first leaf
    uint32_t* positions;     // [total_nodes] absolute word offset of each node
    uint32_t* words;
    uint32_t* parts;         // words of each part of the nodes (one per tile at most)
};
void launch_final(hipStream_t s, const FinalArgs& a);

// ---- device voxeliser ------------------------------------------------------
// Per-triangle constants of the thin surface rule: normal n, n . v0, the
// projected edge functions (nx, ny, d) per axis plane and edge, the dominant
// axis a with the column axes u, w, the planes that are not edge-on, and the
// column rectangle (u0, w0, nw columns along w).
struct TriSetup {
    double n[3];
    double nd;
    double ex[3][3], ey[3][3], ed[3][3];
    int64_t u0, w0;
    uint32_t nw;
    int32_t a, u, w, planes;
};
constexpr uint64_t kVoxTileItems = 2048;  // rows per tile of the row stages
constexpr uint64_t kVoxUnitTile = 256;    // units (at most 8 columns of one row) per voxeliser tile

// Per-row table of the triangles' column rectangles (a row runs along w).
struct VoxRows {
    uint32_t* tri;       // triangle of the row
    uint32_t* u;         // its u coordinate
    uint32_t* w0;        // first column kept
    uint32_t* cols;      // columns kept (a conservative superset of those the rule can emit)
    uint64_t* unit_off;  // exclusive scan of the rows' units
};

// rows[t] = rows of triangle t's rectangle (tris: 9 doubles per triangle);
// *rect_columns += the rectangles' columns (a bound on the kept columns); a
// non-finite coordinate sets kErrKeyRange in *err.
void launch_tri_setup(hipStream_t s, const double* tris, uint64_t n_tris, int depth, TriSetup* setup, uint32_t* rows,
                      uint64_t* rect_columns, unsigned long long* err);
// rows.tri / u / w0 / cols / unit_off for the *n_rows_dev rows (n_rows on the
// host), the unit total into *total_units_dev; row_off = exclusive scan of
// the per-triangle row counts; tile_units / tile_off: one entry per
// kVoxTileItems rows; a tile of rows with 2^32 or more columns sets
// kErrInternal in *err.
void launch_row_setup(hipStream_t s, const TriSetup* setup, const uint64_t* row_off, const uint64_t* n_tris_dev,
                      const uint64_t* n_rows_dev, uint64_t n_rows, const VoxRows& rows, uint32_t* tile_units,
                      uint64_t* tile_off, uint64_t* total_units_dev, unsigned long long* err);
// Voxels per tile of kVoxUnitTile units (total_units in all, also in
// *total_units_dev) into tile_counts, and per unit the voxels that are in
// (bits, may be null).  tile_row (tiles + 1 entries) receives each tile's first
// row; the write pass reads both (with null bits it makes the tests again).
void launch_vox_count(hipStream_t s, const TriSetup* setup, const VoxRows& rows, const uint64_t* n_rows_dev,
                      const uint64_t* total_units_dev, uint64_t total_units, int depth, uint64_t* tile_row,
                      uint16_t* bits, uint32_t* tile_counts);
// The keys, each tile's at tile_offsets[tile] (exclusive scan of the counts).
void launch_vox_write(hipStream_t s, const TriSetup* setup, const VoxRows& rows, const uint64_t* tile_row,
                      const uint64_t* total_units_dev, uint64_t total_units, int depth, const uint16_t* bits,
                      const uint64_t* tile_offsets, uint64_t* keys);

// Per pixel: the first voxel hit and its colour (the reference's trace_paths).
void launch_trace_paths(hipStream_t s, const uint32_t* words, uint64_t n_words, int depth,
                        const svdag_trace_params& p, uint32_t* paths, uint32_t* colors);

// out[i] = occupancy of voxel codes[i] in the flat layout (1 set, 0 not set,
// 2 the walk left the words).
void launch_query_voxels(hipStream_t s, const uint32_t* words, uint64_t n_words, int depth, const uint64_t* codes,
                         uint64_t n, uint8_t* out);

// ---- copies to the host ----------------------------------------------------
// Arrays in device memory to pinned host memory; both ends 16-byte aligned, any
// length.
constexpr int kMaxCopySegments = 3 * SVDAG_MAX_LEVELS + 1;
constexpr uint64_t kCopyPiece = 16384;  // bytes per workgroup step
// DAGs from this size on leave by the copy engine, array by array: it reaches 57
// GB/s against the kernel's 53.5 but takes about 7 us more an array (28 arrays,
// kernel and copies: 126 MB 2337 and 2398 us, 228 MB 4223 and 4190, 314 MB 5860
// and 5710, 1.76 GB 32.9 and 31.0 ms).  Copies of the large arrays beside a
// kernel for the others took 2 to 3% less than either, but a few processes in
// thirty then kept to 31 GB/s.
constexpr uint64_t kCopyOutMaxBytes = 160ull << 20;
struct CopyOut {
    int num;
    uint32_t pieces;  // of all segments
    struct {
        const void* src;
        void* dst;
        uint64_t bytes;
    } seg[kMaxCopySegments];
};
void launch_copy_out(hipStream_t s, const CopyOut& a);

// ---- merge ----------------------------------------------------------------
// Remaps and inserts the nodes of many sub-DAG levels into one shared table.
struct MergeSource {
    const uint8_t* masks;
    const uint32_t* children;
    const uint64_t* hashes;
    uint64_t first;          // index of the source's first node in the concatenation
    uint64_t num;
    uint64_t child_first;    // index of the source's first child in the child concatenation
};
void launch_merge_insert(hipStream_t s, const MergeSource* d_sources, uint32_t num_sources, uint64_t total,
                         const uint32_t* child_slot_of, const uint32_t* child_rank_of_slot, uint8_t* masks_out,
                         uint32_t* children_out, uint64_t* table_keys, uint32_t* table_rep, const uint32_t* table_log2,
                         uint32_t* slot_of, BuildCounters* counters, int ordered);

// ---- gathered chunks ------------------------------------------------------
// Source i's keys go to dst[start, start of source i + 1) (the last source up
// to `total`); starts strictly increase.
struct GatherSource {
    const uint64_t* keys;
    uint64_t start;
};
void launch_gather_keys(hipStream_t s, const GatherSource* src, uint32_t nsrc, uint64_t total, uint64_t* dst);

// ---- resident DAG (served mode) ------------------------------------------
// Nodes of one round level into the persistent table of that level.
struct ResidentLevelArgs {
    const uint64_t* hashes;       // the round level (ascending hash order)
    const uint8_t* masks;
    const uint32_t* children;     // round ranks of the level below
    uint64_t count;
    const uint32_t* child_slot_of;  // round rank of the level below -> resident slot
    uint64_t* table_keys;         // resident ordered table (2^lg + kTableOverflow slots)
    uint32_t* table_rep;
    uint32_t lg;
    uint8_t* rec_masks;           // slot-indexed records
    uint32_t* rec_children;
    uint32_t* slot_of;            // out: resident slot of each round node
    unsigned long long* occupied; // += keys placed
    unsigned long long* err;
};
void launch_resident_level(hipStream_t s, const ResidentLevelArgs& a);
void launch_resident_leaves(hipStream_t s, const uint64_t* leaves, uint64_t count, uint64_t* table_keys, uint32_t lg,
                            uint32_t* slot_of, unsigned long long* occupied, unsigned long long* err);

// Chunk roots of a round: its levels 0 .. top_levels - 1 lead to the chunk
// slots (8^top_levels of them, Morton order).
constexpr int kMaxResidentTop = kTailTopLevel + 1;
struct ResidentRootArgs {
    int top_levels;
    bool has_root;                               // the round has a root node
    const uint8_t* masks[kMaxResidentTop];       // round levels 0 .. top_levels - 1
    const uint32_t* children[kMaxResidentTop];
    const uint32_t* root_slot_of;                // round rank at level top_levels -> resident slot
    const uint64_t* root_table_keys;             // resident table of level top_levels
    uint32_t* root_slot;                         // per chunk slot: resident root slot (kEmptyChild: none)
    uint64_t* root_hash;                         // out: per chunk slot, its root's hash if added now, else 0
    unsigned long long* err;
};
void launch_resident_roots(hipStream_t s, const ResidentRootArgs& a);
// Filled chunk slots in slot order: codes[i] = slot index, list_slots[i] = root slot, *count.
void launch_resident_root_list(hipStream_t s, const uint32_t* root_slot, uint32_t slots, uint64_t* codes,
                               uint32_t* list_slots, uint64_t* count);

}  // namespace svdag
