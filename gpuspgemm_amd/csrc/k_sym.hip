// Symbolic count: exact nnz of every row of C from an open-addressing hash
// table of the row's B columns (sym1.cuh:28-306), written into c_rpt.
//
// A workgroup unit holds R rows; a row owns L = WG/R consecutive lanes of a
// wave (spg_rows.hpp), a wave or the workgroup (spg_wave.hpp), which walk its
// products and insert their columns into the row's LDS table.  Rows that
// overflow a table move on to the next larger one, in the end to global
// memory.
#include "spg_kernels.hpp"
#include "spg_rows.hpp"

namespace spg {

template <typename V, int WG, int R, int T, int EC, int PMAX>
__device__ __forceinline__ void sym_rows(const ProbSet<V>& ps, const int2* __restrict__ items, int first,
                                         int end, int* smem, int* s_tmp) {
    constexpr int L = WG / R;
    static_assert(WG % R == 0, "bad variant shape");
    static_assert(L < kWave, "longer rows: sym_wave_rows, sym_group_row");
    using Meta = ChunkMeta<V, EC, false>;
    constexpr int ROW_INTS = sym_row_ints(SymVariant{WG, R, T, EC, PMAX});
    const int slot = threadIdx.x / L;
    const int lr = threadIdx.x % L;
    int* tab = smem + slot * ROW_INTS;
    Meta* cm = reinterpret_cast<Meta*>(tab + T);
    lds_fill<T, L>(tab, kEmpty, lr);
    gsync<L>();

    const int idx = first + slot;
    const bool active = idx < end;
    const int2 it = active ? items[idx] : make_int2(0, 0);
    const GProb<V> P = ps.get(it.x);
    int a0 = 0, a1 = 0;
    if (active) {
        a0 = P.a_rpt[it.y];
        a1 = P.a_rpt[it.y + 1];
    }
    int mine = 0;
    for_each_round<V, L, EC, PMAX, false>(
        P, a0, a1, lr, cm, s_tmp,
        [&](const int(&key)[PMAX], const V(&)[PMAX], const bool(&ok)[PMAX]) { mine += table_insert_all<T>(tab, key, ok); });
    const int nnz = group_sum<L>(mine);
    if (active && lr == 0) P.c_rpt[it.y] = nnz;
    gsync<L>();  // the table is reused by the next unit
}

// Rows of one wave each (tables of T slots): rows idx, idx + step, ... below
// end of the bin's list.  A wave walks a row's products (wave_products) and
// counts its inserts in a scalar register.  A row starts with a chain of
// dependent loads (its item, its bounds in A, its entries, B's columns), so
// the next row's item and bounds are fetched while this one is counted.
template <typename V, int T, int N>
__device__ __forceinline__ void sym_wave_rows(const ProbSet<V>& ps, const int2* __restrict__ items, int idx, int step,
                                              int end, int* smem) {
    typedef int Words __attribute__((vector_size(16)));
    static_assert(T % (4 * kWave) == 0, "every lane clears a whole share");
    const int lane = lane_id();
    int* tab = smem;
    auto* walk = reinterpret_cast<WaveChunk<false>*>(smem + T);
    if (idx >= end) return;
    int2 it = items[idx];
    int inst = uniform(it.x), row = uniform(it.y);
    GProb<V> P = ps.get(inst);
    int a0 = uniform(P.a_rpt[row]), a1 = uniform(P.a_rpt[row + 1]);
    while (true) {
        const bool more = idx + step < end;
        const int2 it_next = items[more ? idx + step : idx];
#pragma unroll
        for (int i = 0; i < T / (4 * kWave); ++i)
            reinterpret_cast<Words*>(tab)[i * kWave + lane] = Words{kEmpty, kEmpty, kEmpty, kEmpty};
        const WaveOperands<V> W{nullptr, uniform_ptr(P.bref), uniform_ptr(P.b_col), nullptr, uniform(P.wide)};
        wave_sync();
        const int inst_next = uniform(it_next.x), row_next = uniform(it_next.y);
        const GProb<V> P_next = ps.get(inst_next);
        const int b0 = P_next.a_rpt[row_next], b1 = P_next.a_rpt[row_next + 1];
        int n = 0;
        wave_products<V, N, false>(
            W, a0, a1, walk,
            [&](const int(&key)[N], const LdsSum(&)[N], const unsigned long long(&ok)[N], auto far) {
                uint32_t h[N];
                table_slots<T, far, N, true>(tab, key, ok, h, n);
            });
        if (lane == 0) P.c_rpt[row] = n;
        if (!more) break;
        wave_sync();  // the table is reused by the next row
        idx += step;
        inst = inst_next;
        row = row_next;
        P = P_next;
        a0 = uniform(b0);
        a1 = uniform(b1);
    }
}

// A row of WG threads (tid: the thread's place among them), a whole workgroup
// or an equal share of one whose shares all call this together: every wave
// walks a share of the products on its own (no barrier inside the walk), all
// insert into one table.  SHARE: a share, whose row may be -1, none.  LIMIT > 0: a wave stops inserting
// once the row has more than LIMIT distinct columns; with GUESS also once
// 15/16 of the first four rounds' products or more were new columns and so
// many products promise more than LIMIT.  Returns the count (above LIMIT: too
// many, or so it seems), the same on every lane.
template <typename V, int WG, int T, int N, int LIMIT, bool GUESS = false, bool SHARE = false>
__device__ __forceinline__ int sym_group_row(const GProb<V>& P, int row, int* smem, int tid) {
    typedef int Words __attribute__((vector_size(16)));
    constexpr int kWaves = WG / kWave;
    static_assert(T % (4 * WG) == 0, "every thread clears a whole share");
    const int wave = uniform(tid / kWave);
    int* tab = smem;
    auto* walk = reinterpret_cast<WaveChunk<false>*>(smem + T);
    int* total = reinterpret_cast<int*>(walk + kWaves);
#pragma unroll
    for (int i = 0; i < T / (4 * WG); ++i)
        reinterpret_cast<Words*>(tab)[i * WG + tid] = Words{kEmpty, kEmpty, kEmpty, kEmpty};
    if (tid == 0) *total = 0;
    const WaveOperands<V> W{nullptr, uniform_ptr(P.bref), uniform_ptr(P.b_col), nullptr, uniform(P.wide)};
    int a0 = 0, a1 = 0, nip = 0;
    if (!SHARE || row >= 0) {
        a0 = uniform(P.a_rpt[row]);
        a1 = uniform(P.a_rpt[row + 1]);
        nip = uniform(P.nip[row]);
    }
    // GUESS: `total` holds the products so far (modulo 2^18) above the count
    constexpr int kCountBits = GUESS ? 14 : 31;
    constexpr unsigned kCount = (1u << kCountBits) - 1;
    static_assert(!GUESS || LIMIT + N * WG <= static_cast<int>(kCount), "the count's bits");
    const unsigned sample = nip > LIMIT + LIMIT / 16 ? N * WG : UINT_MAX;
    __syncthreads();
    int added = 0;
    auto report = [&]() {
        if (lane_id() == 0 && added) atomicAdd(total, added);
        added = 0;
    };
    wave_products<V, N, false>(
        W, a0, a1, walk + wave,
        [&](const int(&key)[N], const LdsSum(&)[N], const unsigned long long(&ok)[N], auto far) -> bool {
            if constexpr (LIMIT > 0) {
                const int have = uniform(lds_load(total));
                if constexpr (GUESS) {
                    const unsigned seen = static_cast<unsigned>(have) >> kCountBits, count = have & kCount;
                    if (count > LIMIT || (seen >= sample && 16 * count >= 15 * seen)) return false;
                } else {
                    if (have > LIMIT) return false;
                }
                // Near the limit a slot at a time, which leaves the table with LIMIT + 64 columns a wave instead
                // of LIMIT + 256: with 16 waves 83 % full instead of 92 (500 rows of 40,000 columns stop after
                // 610 us with whole rounds, after 230 so).
                if (kWaves > 4 && have > LIMIT - N * WG) {
#pragma unroll
                    for (int j = 0; j < N; ++j) {
                        if (uniform(lds_load(total)) > LIMIT) return false;
                        const int one[1] = {key[j]};
                        const unsigned long long one_ok[1] = {ok[j]};
                        uint32_t at[1];
                        table_slots<T, far, 1, true>(tab, one, one_ok, at, added);
                        report();
                    }
                    return true;
                }
            }
            uint32_t h[N];
            table_slots<T, far, N, true>(tab, key, ok, h, added);
            if constexpr (GUESS) {
#pragma unroll
                for (int j = 0; j < N; ++j) added += __popcll(ok[j]) << kCountBits;
            }
            if constexpr (LIMIT > 0) report();
            return true;
        },
        wave, kWaves, wave_by_chunk<kWaves>(a1 - a0, nip));
    report();
    __syncthreads();
    int n = *total;
    if constexpr (GUESS) {
        const unsigned missing = (static_cast<unsigned>(n) ^ static_cast<unsigned>(nip) << kCountBits) >> kCountBits;
        n = missing ? LIMIT + 1 : n & kCount;  // (stopped: not all products)
    }
    __syncthreads();  // the table and the total are reused by the next row
    return n;
}

// Where the rows go that variant 8 hands on to the largest-table launch.
struct OverLists {
    int2* items;  // behind the last bin's list: rows of more than kSymSmallNip products
    int2* last;   // from here down: the others
};

// One wave hands on rows k, k + step, ... (n <= 64 of them) below end: an
// atomic for each of the two lists, however many rows it takes (about 10 ns
// each from all workgroups: 200 us for 20,000 rows one by one).
template <typename V>
__device__ __forceinline__ void hand_on(const ProbSet<V>& ps, const int2* __restrict__ bin_items, int k, int step,
                                        int n, int end, const OverLists& over, DevMeta* meta) {
    const int lane = lane_id();
    const bool ok = lane < n && k + lane * static_cast<long long>(step) < end;
    int2 it = make_int2(0, 0);
    int nip = 0;
    if (ok) {
        it = bin_items[k + lane * step];
        nip = ps.get(it.x).nip[it.y];
    }
    const unsigned long long small = __ballot(ok && nip <= kSymSmallNip), large = __ballot(ok && nip > kSymSmallNip);
    int at_small = 0, at_large = 0;
    if (lane == 0) {
        if (small) at_small = atomicAdd(&meta->fail_count.over_small, __popcll(small));
        if (large) at_large = atomicAdd(&meta->fail_count.over, __popcll(large));
    }
    at_small = uniform(at_small);
    at_large = uniform(at_large);
    if (in_mask(small)) over.last[-(at_small + rank_in(small))] = it;
    if (in_mask(large)) over.items[at_large + rank_in(large)] = it;
}

// The units k0, k0 + step, ... below k_end (kV.r rows each) of a bin of
// variant VV.  After a row that overflows variant 8's table the workgroup
// hands its next ones on untried, a few and then more each time (rows of one
// matrix are alike), until it tries one that fits.
template <typename V, int VV>
__device__ __forceinline__ void sym_units(const ProbSet<V>& ps, const int2* __restrict__ bin_items, int k0, int step,
                                          int k_end, int count, int* smem, int* s_tmp, const OverLists& over,
                                          DevMeta* meta) {
    constexpr SymVariant kV = kSymVariants[VV];
    const int end = min(count, k_end * kV.r);
    if constexpr (sym_is_wave(kV)) {
        const int wave = uniform(static_cast<int>(threadIdx.x) / kWave);
        sym_wave_rows<V, kV.t, kV.pmax>(ps, bin_items, k0 * kV.r + wave, step * kV.r, end,
                                        smem + wave * sym_row_ints(kV));
    } else if constexpr (sym_is_group(kV)) {
        constexpr int kLimit = VV == kSymOverVariant ? kSymOverThreshold : 0;
        // A dozen scalar instructions a round: 59,049 rows of 6,561 products on 375 columns took 458 us instead of
        // 393 while every row was guessed at.  The first one is, and those after one that overflowed.
        bool guess = true;
        int untried = 0;
        for (int k = k0; k < end; k += step) {
            const int2 it = bin_items[k];
            const GProb<V> P = ps.get(uniform(it.x));
            const int row = uniform(it.y);
            const int n = kLimit > 0 && guess
                              ? sym_group_row<V, kV.wg, kV.t, kV.pmax, kLimit, true>(P, row, smem, threadIdx.x)
                              : sym_group_row<V, kV.wg, kV.t, kV.pmax, kLimit>(P, row, smem, threadIdx.x);
            guess = kLimit > 0 && n > kLimit;
            if (guess) {
                untried = min(2 * untried + 3, kWave - 1);
                if (uniform(static_cast<int>(threadIdx.x) / kWave) == 0)
                    hand_on<V>(ps, bin_items, k, step, untried + 1, end, over, meta);
                if (end - k <= untried * static_cast<long long>(step)) break;
                k += untried * step;
            } else {
                untried = 0;
                if (threadIdx.x == 0) P.c_rpt[row] = n;
            }
        }
    } else {
        for (int first = k0 * kV.r; first < end; first += step * kV.r)
            sym_rows<V, kV.wg, kV.r, kV.t, kV.ec, kV.pmax>(ps, bin_items, first, end, smem, s_tmp);
    }
}

// One launch serves the bins [0, n_multi) of the symbolic table.  Bin sizes
// are read on the device, so the launch needs no host round trip; the grid
// is persistent.  Every XCD takes a contiguous slice of every bin, the bins
// of long rows first, and its workgroups deal the slices' units among
// themselves.  One kernel for all variants (72 VGPRs with 52 bytes spilled a
// lane, 21.6 KB of LDS, seven waves per SIMD) keeps the whole symbolic phase on one stream: in three
// launches on three streams, the fork cost 7 to 14 us and the join 10 to 58.
template <typename V>
__global__ __launch_bounds__(kMultiThreads) SPG_WAVES_PER_EU(kSymMultiMinWaves) void k_sym_multi(
    ProbSet<V> ps, int2* __restrict__ items, int bin_cap, BinTable sym, int n_multi, DevMeta* __restrict__ meta) {
    __shared__ __align__(16) int smem[max_sym_multi_lds() / 4];
    __shared__ int s_tmp[kMultiThreads / kWave];
    __shared__ int s_cnt[kMaxBins];
    if (static_cast<int>(threadIdx.x) < n_multi) s_cnt[threadIdx.x] = meta->sym_count[threadIdx.x].v;
    __syncthreads();
    const int xcd = blockIdx.x % kXcds;
    const int step = gridDim.x / kXcds;
    int2* last_bin = items + static_cast<long long>(sym.n - 1) * bin_cap;
    const OverLists over{last_bin + meta->sym_count[sym.n - 1].v, last_bin + bin_cap - 1};
    int k0 = blockIdx.x / kXcds;  // this workgroup's first unit in the XCD's slice of the bin
    for (int b = n_multi - 1; b >= 0; --b) {
        const int count = s_cnt[b];
        const int per = ((count + sym.rows[b] - 1) / sym.rows[b] + kXcds - 1) / kXcds;  // units of the slice
        if (k0 >= per) {
            k0 -= per;
            continue;
        }
        const int2* bin_items = items + static_cast<long long>(b) * bin_cap;  // bin b's list
        const int first = xcd * per;
#define SPG_SYM_CASE(v)                                                                                            \
    case v:                                                                                                        \
        sym_units<V, v>(ps, bin_items, first + k0, step, first + per, count, smem, s_tmp, over, meta);             \
        break;
        switch (sym.variant[b]) {
            SPG_SYM_CASE(0)
            SPG_SYM_CASE(1)
            SPG_SYM_CASE(2)
            SPG_SYM_CASE(3)
            SPG_SYM_CASE(4)
            SPG_SYM_CASE(5)
            SPG_SYM_CASE(6)
            SPG_SYM_CASE(7)
            SPG_SYM_CASE(8)
            default:
                break;
        }
#undef SPG_SYM_CASE
        k0 += (per - k0 + step - 1) / step * step - per;
        // The next bin may lay out LDS differently, and rows of L <= 64 lanes
        // only synchronise inside their wave: no wave may start on it while
        // another wave still uses this one.  Units of one bin give every
        // wave the same LDS slots, so between them the waves run on.
        __syncthreads();
    }
}

// Largest LDS table (32768 slots, 128 KiB) with overflow detection
// (sym1.cuh:169-245): a row whose distinct count passes 80 % of the table
// stops early and is queued, with its global-table slot range, for
// k_sym_global.  Then, where they are many, the rows handed on that cannot
// fill a table of 8192, four at a time with a quarter of the workgroup each: one
// by one they took 304 us for 20,000 rows of 2,304 products, so 175 us.
template <typename V>
__global__ __launch_bounds__(1024) void k_sym_max(ProbSet<V> ps, const int2* __restrict__ items, int bin_cap,
                                                  int bin, DevMeta* __restrict__ meta,
                                                  int2* __restrict__ fail_items, long long* __restrict__ fail_off) {
    constexpr SymVariant kV = kSymVariants[kSymMaxVariant];
    __shared__ __align__(16) int smem[kSymMaxLds / 4];
    const int2* bin_items = items + static_cast<long long>(bin) * bin_cap;
    const int large = meta->sym_count[bin].v + meta->fail_count.over;
    const int small = meta->fail_count.over_small;
    const bool shares = small > static_cast<int>(gridDim.x);  // (fewer have a workgroup each)
    const int count = large + (shares ? 0 : small);
    for (int u = blockIdx.x; u < count; u += gridDim.x) {
        const int2 it = bin_items[u < large ? u : bin_cap - 1 - (u - large)];
        const GProb<V> P = ps.get(uniform(it.x));
        const int row = uniform(it.y);
        const int n = sym_group_row<V, kV.wg, kV.t, kV.pmax, kSymMaxThreshold>(P, row, smem, threadIdx.x);
        if (threadIdx.x == 0) {
            if (n <= kSymMaxThreshold) {
                P.c_rpt[row] = n;
            } else {
                const int f = atomicAdd(&meta->fail_count.v, 1);
                fail_items[f] = it;
                fail_off[f] = static_cast<long long>(
                    atomicAdd(&meta->fail_pool.v, static_cast<unsigned long long>(global_table_slots(P.nip[row]))));
            }
        }
    }
    constexpr int kShares = kV.wg / kSymSmall.wg;
    static_assert(kShares * sym_row_ints(kSymSmall) * 4 <= kSymMaxLds && sym_row_ints(kSymSmall) % 4 == 0,
                  "a share's LDS");
    if (!shares) return;
    const int share = uniform(static_cast<int>(threadIdx.x) / kSymSmall.wg);
    for (int u = blockIdx.x * kShares; u < small; u += gridDim.x * kShares) {
        const bool mine = u + share < small;
        const int2 it = bin_items[bin_cap - 1 - (mine ? u + share : u)];
        const GProb<V> P = ps.get(uniform(it.x));
        const int row = mine ? uniform(it.y) : -1;
        const int n = sym_group_row<V, kSymSmall.wg, kSymSmall.t, kSymSmall.pmax, 0, false, true>(
            P, row, smem + share * sym_row_ints(kSymSmall), threadIdx.x % kSymSmall.wg);
        if (mine && threadIdx.x % kSymSmall.wg == 0) P.c_rpt[row] = n;
    }
}

// Global-memory table per overflowed row (sym1.cuh:247-306), sized from the
// row's NIP (an upper bound of its distinct count) rather than from the
// largest NIP of the matrix.
template <typename V>
__global__ __launch_bounds__(1024) void k_sym_global(ProbSet<V> ps, const int2* __restrict__ fail_items,
                                                     const long long* __restrict__ fail_off, int* pool) {
    constexpr int WG = 1024;
    constexpr int EC = 1024;
    constexpr int PMAX = 4;
    using Meta = ChunkMeta<V, EC, false>;
    __shared__ Meta cm;
    __shared__ int s_tmp[WG / kWave];
    const int2 it = fail_items[blockIdx.x];
    const GProb<V> P = ps.get(it.x);
    const long long slots = global_table_slots(P.nip[it.y]);
    const int bits = __builtin_ctzll(static_cast<unsigned long long>(slots));
    int* tab = pool + fail_off[blockIdx.x];
    for (long long j = threadIdx.x; j < slots; j += WG) tab[j] = kEmpty;
    __threadfence();
    __syncthreads();
    const uint32_t mask = static_cast<uint32_t>(slots - 1);
    int mine = 0;
    for_each_product<V, WG, EC, PMAX, false>(P, P.a_rpt[it.y], P.a_rpt[it.y + 1], threadIdx.x, &cm, s_tmp,
                                             [&](int key, V) {
                                                 uint32_t h = hash_slot_rt(key, bits);
                                                 while (true) {
                                                     const int cur = __hip_atomic_load(
                                                         tab + h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                                                     if (cur == key) break;
                                                     if (cur == kEmpty) {
                                                         const int old = atomicCAS(tab + h, kEmpty, key);
                                                         if (old == kEmpty) {
                                                             ++mine;
                                                             break;
                                                         }
                                                         if (old == key) break;
                                                     }
                                                     h = (h + 1) & mask;
                                                 }
                                             });
    int total;
    (void)group_excl_scan<WG>(mine, threadIdx.x, s_tmp, total);
    if (threadIdx.x == 0) P.c_rpt[it.y] = total;
}

// ----------------------------------------------------------------- launchers

template <typename V>
void launch_sym_multi(const ProbSet<V>& ps, int2* items, int bin_cap, const BinTable& sym, int n_multi, DevMeta* meta,
                      int grid, hipStream_t s) {
    hipLaunchKernelGGL(k_sym_multi<V>, dim3(grid), dim3(kMultiThreads), 0, s, ps, items, bin_cap, sym, n_multi, meta);
}

template <typename V>
void launch_sym_max(const ProbSet<V>& ps, const int2* items, int bin_cap, int bin, DevMeta* meta, int2* fail_items,
                    long long* fail_off, int grid, hipStream_t s) {
    hipLaunchKernelGGL(k_sym_max<V>, dim3(grid), dim3(1024), 0, s, ps, items, bin_cap, bin, meta, fail_items,
                       fail_off);
}

template <typename V>
void launch_sym_global(const ProbSet<V>& ps, const int2* fail_items, const long long* fail_off, int* pool,
                       int count, hipStream_t s) {
    hipLaunchKernelGGL(k_sym_global<V>, dim3(count), dim3(1024), 0, s, ps, fail_items, fail_off, pool);
}

template <typename V>
int occupancy_sym_multi() {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_sym_multi<V>, kMultiThreads, 0) != hipSuccess) n = 1;
    return n > 0 ? n : 1;
}

template <typename V>
int occupancy_sym_max() {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_sym_max<V>, 1024, 0) != hipSuccess) n = 1;
    return n > 0 ? n : 1;
}

#define SPG_INSTANTIATE_SYM(V)                                                                               \
    template void launch_sym_multi<V>(const ProbSet<V>&, int2*, int, const BinTable&, int, DevMeta*, int,     \
                                      hipStream_t);                                                          \
    template void launch_sym_max<V>(const ProbSet<V>&, const int2*, int, int, DevMeta*, int2*, long long*, int, \
                                    hipStream_t);                                                            \
    template void launch_sym_global<V>(const ProbSet<V>&, const int2*, const long long*, int*, int,           \
                                       hipStream_t);                                                         \
    template int occupancy_sym_multi<V>();                                                                   \
    template int occupancy_sym_max<V>();

SPG_INSTANTIATE_SYM(float)
SPG_INSTANTIATE_SYM(double)

}  // namespace spg
