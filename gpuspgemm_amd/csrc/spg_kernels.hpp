// Compiled kernel variants and host-side launchers.
//
// A variant fixes how a workgroup works on rows: R rows per workgroup (so
// L = WG / R lanes per row), A entries per chunk, products per lane per
// round, and the LDS table size.  The runtime bin tables (BinTable) map
// rows to variants; they replace the reference's hand-set per-arch tables
// (src/libproposal/include/proposal/parameters.cuh:22-413) and can be
// rewritten at run time by the tuner.
#pragma once

#include "spg_common.hpp"
#include "spg_wave.hpp"

namespace spg {

struct SymVariant {
    int wg, r, t, ec, pmax;  // workgroup, rows per workgroup, table slots, A entries per chunk, products per lane
};
struct NumVariant {
    int wg, r, p, ec, pmax;  // ... p = sorted-list capacity (the hash table has 2p slots)
    int t;                   // table slots of the one-wave rows
};
// Rows of one wave each (wg / r == 64): see symnum_wave_row; rows that a
// workgroup's waves share, with values in the table: symnum_group_row.
constexpr bool num_is_wave(const NumVariant& v) { return v.wg / v.r == kWave; }
constexpr bool num_is_group(const NumVariant& v) { return v.wg / v.r > kWave && v.t > 0 && v.t <= 4096; }
// The longest rows that fit LDS: only the columns do, see symnum_long_row.
constexpr bool num_is_long(const NumVariant& v) { return v.t > 4096; }


// Symbolic (count) variants.  0..8 run inside one launch of 256-thread
// workgroups: 0..4 several rows to a wave, 5 and 6 a row to a wave, 7 and 8 a
// row to a workgroup; 9 is the largest LDS table (sym1.cuh:169-245).  A bin
// may take rows of NIP below its table size; variant 8 takes rows of any NIP
// and hands those with more than kSymOverThreshold distinct columns to
// variant 9, which hands those above kSymMaxThreshold to the global tables.
// A row's NIP says little about its distinct columns: a structural matrix of
// 81 entries a row has 6,561 products and 375 columns, and a 1024-thread
// workgroup with a 128 KB table per such row took 1.54 ms for 59,049 rows.
constexpr SymVariant kSymVariants[] = {
    {256, 256, 16, 4, 8},  {256, 128, 32, 4, 8},  {256, 64, 64, 8, 8},    {256, 32, 128, 16, 8},
    {256, 16, 256, 32, 8}, {256, 4, 512, 64, 4},  {256, 4, 1024, 64, 4},  {256, 1, 4096, 64, 4},
    {256, 1, 4096, 64, 4}, {1024, 1, 32768, 64, 4},
};
constexpr int kSymMultiVariants = 9;
constexpr int kSymOverVariant = 8;
constexpr int kSymMaxVariant = 9;
// Distinct columns at which a wave of these variants stops inserting; every
// wave may have a round of 64 * 4 more in flight.  Linear probing gets slow
// as a table fills: with 70 % here a row that overflowed (95 % with the
// rounds in flight) took 200 us, with 50 % under 20.
constexpr int kSymOverThreshold = 2048;  // 50 % of 4096
constexpr int kSymMaxThreshold = 26214;  // 80 % of 32768
static_assert(kSymOverThreshold + 4 * 256 < 4096 && kSymMaxThreshold + 16 * 256 < 32768,
              "a counting table keeps room for the rounds in flight");
// Rows that variant 8 hands on and that have at most kSymSmallNip products are
// counted by the largest-table launch four at a time, in tables of twice
// their products.
constexpr int kSymSmallNip = 4096;
constexpr SymVariant kSymSmall = {256, 1, 2 * kSymSmallNip, 64, 4};
constexpr int kSymMultiMinWaves = 7;  // waves per SIMD that the multi-bin launch keeps: at most 72 VGPRs
constexpr int kSymMultiLds = 160 * 1024 / kSymMultiMinWaves;  // bytes a workgroup of it may use: as many on a CU
constexpr bool sym_is_wave(const SymVariant& v) { return v.wg / v.r == kWave; }
constexpr bool sym_is_group(const SymVariant& v) { return v.wg / v.r > kWave; }

// Fused sorted-columns + numeric variants, one kernel each: all use 256
// threads except 9 and 20 (a 1024-thread workgroup per row); rows above every
// capacity use global-memory tables (variant 19).  4, 5 and 13: a row to a
// wave; 6 and 7: a row to a workgroup's waves, values in the table; 20: the
// longest rows, columns in LDS; 8 and 9: a row to a workgroup in step, with
// searches in the sorted list; the others several rows to a wave.  10 to 13
// (and 5) sort rows with a product per lane (two) in registers.  The tuner
// picks among those that fit a bin.
constexpr NumVariant kNumVariants[] = {
    {256, 256, 8, 4, 16},   {256, 128, 16, 4, 16}, {256, 64, 32, 8, 16},  {256, 32, 64, 16, 16},
    {256, 4, 256, 64, 4, 512}, {256, 4, 128, 64, 4, 256}, {256, 1, 512, 64, 4, 1024}, {256, 1, 1024, 64, 4, 2048},
    {256, 1, 2048, 256, 8}, {1024, 1, 8192, 1024, 4}, {256, 32, 8, 8, 2}, {256, 16, 16, 16, 2},
    {256, 8, 32, 32, 4},    {256, 4, 64, 64, 4, 128}, {256, 64, 8, 8, 4},    {256, 128, 8, 4, 8},
    {256, 32, 16, 8, 4},    {256, 64, 16, 8, 8},   {256, 32, 32, 16, 8},  {1024, 1, 1, 1, 1},
    {1024, 1, 26214, 64, 4, 32768},
};
constexpr int kNumVariantCount = 21;
constexpr int kNumGlobalVariant = 19;  // (its entry above only holds the place)
// Waves per SIMD that each fused variant's kernel must keep (its register
// budget is 512 / waves VGPRs).  The floors of the narrow variants keep the
// residency that they had when a lane's products were fetched one by one
// (power-law: 198k-row bin 70 -> 53 us with the batch inside it); the wave
// rows' eight waves (64 VGPRs) beat six by 7 % (96^3 stencil).
constexpr int kNumMinWaves[kNumVariantCount] = {3, 3, 3, 3, 5, 8, 8, 5, 3, 4, 8, 8, 7, 8, 7, 5, 7, 5, 5, 1, 4};

// Fused variants whose bins share one launch.  Set 0, small rows (256
// threads, up to a wave per row, about 78 VGPRs; floors of seven and eight
// waves measured +4 and +1 % on the power-law, -2 and -3 % on a batch):
// their bins hold most rows of skewed matrices, and one launch keeps the GPU filled across them
// where separate launches would queue behind each other on the lane's few
// hardware queues.  Set 1, the 256-thread variants of longer rows: merged
// only while their bins are small (a few thousand units, as the heavy tail
// of a skewed matrix), so that those long-latency units all start at once
// beside set 0 instead of queueing one launch after another; a large bin
// of set 1 (the 96^3 stencil's) keeps its own launch and its own register
// budget.  kNumMultiMinWaves is each merged kernel's residency floor.
constexpr int kNumMultiSet0[] = {10, 11, 12, 13, 14, 16};
constexpr int kNumMultiSet1[] = {4, 5, 6, 7, 8};
constexpr int kNumMultiMinWaves[2] = {6, 3};
constexpr int kNumMultiMaxUnits1 = 4096;  // set 1 merges while its bins hold at most this many units
constexpr int num_multi_set(int v) {
    for (int m : kNumMultiSet0)
        if (m == v) return 0;
    for (int m : kNumMultiSet1)
        if (m == v) return 1;
    return -1;
}

// Bins of one merged launch: bin b's rows are items [off[b], off[b] +
// count[b]) in units of its variant's rows.  Every XCD takes one contiguous
// slice of every bin: the workgroups with local index (blockIdx.x / 8) in
// [slice0[b], slice0[b + 1]) work on bin b, slice0[b + 1] - slice0[b] =
// ceil(units of bin b / 8) of them per XCD.
struct NumMultiBins {
    int32_t n;
    int32_t variant[kMaxBins];
    int32_t off[kMaxBins];
    int32_t count[kMaxBins];
    int32_t slice0[kMaxBins + 1];
};

constexpr int kGlobalSortChunk = 4096;  // LDS chunk of the global-bin column sort

// Ints of one row slot in LDS: `bytes` rounded up to 8-byte words and
// padded so that the number of words is odd.  Slots of one wave then start
// in different LDS banks; with a power-of-two stride the same offset of
// every row of the wave falls in one bank, and the small-row variants (up
// to 64 rows per wave) serialise on bank conflicts.
constexpr int padded_row_ints(int bytes) {
    const int words = (bytes + 7) / 8;
    return 2 * (words % 2 ? words : words + 1);
}
// Fused variant: table 2p ints (reused for p sums in double), sorted
// list p ints, chunk metadata when the row has more than one lane.
constexpr int num_row_ints(const NumVariant& v) {
    return num_is_long(v) ? long_row_bytes(v.t, v.wg / kWave) / 4
         : num_is_group(v) ? group_row_bytes(v.p, v.t, v.wg / kWave) / 4
         : num_is_wave(v) ? wave_row_bytes(v.p, v.t) / 4
                           : padded_row_ints(12 * v.p + (v.wg / v.r > 1 ? 16 * v.ec : 0));
}
// Symbolic variant: table t ints, walk metadata without values.
constexpr int sym_row_ints(const SymVariant& v) {
    if (sym_is_group(v)) return v.t + v.wg / kWave * static_cast<int>(sizeof(WaveChunk<false>)) / 4 + 4;
    if (sym_is_wave(v)) return v.t + static_cast<int>(sizeof(WaveChunk<false>)) / 4;
    return padded_row_ints(4 * v.t + (v.wg / v.r > 1 ? 8 * v.ec + 8 : 0));
}
constexpr int kSymMaxLds = 4 * (sym_row_ints(kSymVariants[kSymMaxVariant]) > 4 * sym_row_ints(kSymSmall)
                                    ? sym_row_ints(kSymVariants[kSymMaxVariant])
                                    : 4 * sym_row_ints(kSymSmall));
constexpr int max_sym_multi_lds() {
    int m = 0;
    for (int i = 0; i < kSymMultiVariants; ++i) {
        const int b = 4 * kSymVariants[i].r * sym_row_ints(kSymVariants[i]);
        m = m > b ? m : b;
    }
    return m;
}
constexpr int max_num_lds() {
    int m = 0;
    for (int i = 0; i < kNumVariantCount; ++i) {
        const int b = 4 * kNumVariants[i].r * num_row_ints(kNumVariants[i]);
        m = m > b ? m : b;
    }
    return m;
}
constexpr int max_num_multi_lds(int set) {
    int m = 0;
    for (int v = 0; v < kNumVariantCount; ++v) {
        const int b = 4 * kNumVariants[v].r * num_row_ints(kNumVariants[v]);
        if (num_multi_set(v) == set) m = m > b ? m : b;
    }
    return m;
}
constexpr int kNumBigLds = max_num_lds();
static_assert(max_sym_multi_lds() <= kSymMultiLds, "symbolic multi-bin LDS budget");

// Slots of a global-memory hash table for a row with `keys` distinct keys.
__host__ __device__ __forceinline__ long long global_table_slots(long long keys) {
    long long t = kGlobalSortChunk;
    while (t < 2 * keys) t <<= 1;
    return t;
}

// ---- launchers (defined next to their kernels) ----
void launch_clear(DevMeta* meta, int from_word, hipStream_t s);
void launch_signal(int* host_flag, hipStream_t s);
void launch_readback(const int* src, int* host_dst, int words, const long long* src2, long long* host_dst2, int n2,
                     DevMeta* clear, int* host_flag, hipStream_t s);
void launch_total_nip(const int32_t* a_rpt, const int32_t* a_col, const int32_t* b_rpt, int m,
                      unsigned long long* out, hipStream_t s);

// NIP per row and the scatter into the symbolic bin lists (bin b's list
// starts at items + b * bin_cap); entries: of A, over all products
template <typename V>
void launch_nip(const ProbSet<V>& ps, const BinTable& sym, DevMeta* meta, int2* items, int bin_cap, long long entries,
                hipStream_t s);
template <typename V>
void launch_scan_count(const ProbSet<V>& ps, const BinTable& num, DevMeta* meta, long long* tile_sums,
                       int after_fail, hipStream_t s);
// with tile_prefix_min or more tiles, k_tile_prefix turns tile_sums into
// their exclusive prefix first (in place)
template <typename V>
void launch_scan_apply(const ProbSet<V>& ps, const BinTable& num, DevMeta* meta, long long* tile_sums,
                       RowItem* items, long long* gpool_off, long long* inst_nnz, int after_fail,
                       int tile_prefix_min, hipStream_t s);

// symbolic count: one launch over bins [0, n_multi) of `sym` (rows that
// overflow variant 8 join the list of the last bin), then the last bin
template <typename V>
void launch_sym_multi(const ProbSet<V>& ps, int2* items, int bin_cap, const BinTable& sym, int n_multi, DevMeta* meta,
                      int grid, hipStream_t s);
template <typename V>
void launch_sym_max(const ProbSet<V>& ps, const int2* items, int bin_cap, int bin, DevMeta* meta, int2* fail_items,
                    long long* fail_off, int grid, hipStream_t s);
template <typename V>
void launch_sym_global(const ProbSet<V>& ps, const int2* fail_items, const long long* fail_off, int* pool,
                       int count, hipStream_t s);

// fused pass: one launch per variant (all but the global one) over one bin's items
template <typename V>
hipError_t launch_symnum_bin(int variant, const ProbSet<V>& ps, const RowItem* items, int item_off, int count,
                             DevMeta* meta, int grid, hipStream_t s);
// fused pass: one launch over the units of several bins whose variants are
// in merged set `set` (a workgroup per unit)
template <typename V>
hipError_t launch_symnum_multi(int set, const ProbSet<V>& ps, const RowItem* items, const NumMultiBins& mb,
                               DevMeta* meta, hipStream_t s);
template <typename V>
void launch_symnum_global(const ProbSet<V>& ps, const RowItem* items, const long long* gpool_off, int item_off,
                          int count, int* pool, DevMeta* meta, hipStream_t s);

// has the runtime load the fused kernels (a query of each), for which the first
// multiply would otherwise wait (5.1 instead of 2.1 ms)
template <typename V>
void load_symnum();

// occupancy (workgroups per CU) of the persistent launches
template <typename V>
int occupancy_sym_multi();
template <typename V>
int occupancy_sym_max();

}  // namespace spg
