// Fused second symbolic pass and numeric pass.  For every row:
//   1. insert the row's B columns into an LDS hash table of 2P slots
//      (sym2.cuh:27-121 without the count);
//   2. compact the occupied slots and sort them ascending with a bitonic
//      network in LDS (the reference sorts the whole table with CUB merge
//      sort, sym2.cuh:104-113); write them to C.col (sym2.cuh:116-120);
//   3. reuse the table's LDS as the row's value accumulator, zeroed
//      (num.cuh:97-100), and for every product a_ik * b_kj find the slot of
//      column j by binary search in the sorted LDS column list (find_key,
//      num.cuh:28-41) and add the product there (num.cuh:104-116);
//   4. write the values to C.val.
// Fusing the two passes keeps the sorted column list in LDS between them,
// so C.col is written once and never read back.  Rows of 64 lanes add their
// values in the hash table itself (symnum_wave_row).  A row whose products fit
// in one chunk and in the lanes' PMAX register slots keeps (column, a*b)
// in registers from step 1 to step 3 and reads A and B only once.
#include "spg_kernels.hpp"
#include "spg_rows.hpp"

namespace spg {

// Compact the occupied slots of a row's table into cols[0..min(n, P))
// (unsorted); returns the number n of occupied slots.  Every lane reads its
// T/L slots first, then one group scan of the per-lane counts places them.
template <int L, int T, int P>
__device__ __forceinline__ int compact_table(const int* tab, int* cols, int lr, int* s_tmp) {
    static_assert(T % L == 0, "table must be a multiple of the group");
    constexpr int S = T / L;
    constexpr int B = L > kWave && S > 8 ? 8 : S;  // slots read per batch (workgroup-wide rows: bounded registers)
    int n = 0;
    for (int b0 = 0; b0 < S; b0 += B) {
        int key[B];
        int mine = 0;
#pragma unroll
        for (int s = 0; s < B; ++s) {
            key[s] = tab[lr + (b0 + s) * L];
            mine += key[s] != kEmpty;
        }
        int tot;
        int pos = n + group_excl_scan<L>(mine, lr, s_tmp, tot);
#pragma unroll
        for (int s = 0; s < B; ++s) {
            if (key[s] == kEmpty) continue;
            if (pos < P) cols[pos] = key[s];
            ++pos;
        }
        n += tot;
    }
    return n;
}

// Sorted column list of a row: the occupied slots of its table in
// ascending order in cols[0..n), padded with INT_MAX up to P; returns n.
// Groups inside one wave sort in registers (bitonic_sort_regs) and also
// leave lane lr's share cols[lr*E .. lr*E + E) in x; workgroup-wide rows
// sort wave blocks in registers and merge them in LDS (bitonic_sort_block).
template <int L, int T, int P>
__device__ __forceinline__ int sort_row(const int* tab, int* cols, int lr, int* s_tmp, int (&x)[L <= kWave ? P / L : 1]) {
    const int found = compact_table<L, T, P>(tab, cols, lr, s_tmp);
    const int n = min(found, P);
    if constexpr (L <= kWave) {
        constexpr int E = P / L;
        gsync<L>();
#pragma unroll
        for (int s = 0; s < E; ++s) x[s] = lr * E + s < n ? cols[lr * E + s] : INT_MAX;
        bitonic_sort_regs<P, L>(x, lr);
        gsync<L>();
#pragma unroll
        for (int s = 0; s < E; ++s) cols[lr * E + s] = x[s];
    } else {
        for (int j = n + lr; j < P; j += L) cols[j] = INT_MAX;
        gsync<L>();
        bitonic_sort_block<P, L>(cols, lr);
    }
    return found;
}

// Rows of at most L * K products, a group of L lanes to a row (K = 1, or L =
// 64), when the whole wave's rows are such: sorted in registers instead of
// hashed.  A row's products take one slot each, product j * 64 + lane of the
// wave; the slots' entries come from a bitmap of entry starts as in
// wave_products.  Every slot packs its column above its slot number into one
// word, the groups sort the words, a slot whose column differs from the one
// below starts an entry of C, and its place in the row is the number of such
// slots before it.  No table, no probing, and LDS sums only for waves that
// have a repeated column.  About 100 vector instructions for the 8 rows of a
// wave at L = 8, where the hashed path spends 25 a row: on the power-law matrix
// 47 of the launch's 113 us, which is bound by the lines of B that it fetches
// past L2.  A row to a wave (L = 64) is bound by the instructions of its sort,
// so rows of few columns are hashed (the bin tables).
template <int K>
struct alignas(16) SortSlots {
    unsigned long long starts[K];
    union {
        WaveEntry<true> ent[kWave];
        LdsSum prod[kWave * K];
    };
    LdsSum sum[kWave * K];
};
template <int K>
constexpr int kSortColBits = K == 1 ? 26 : 25;  // column bits beside the slot number (all ones: no product)

template <typename V, int L, int K>
__device__ __forceinline__ void symnum_sorted(const GProb<V>& Pr, const RowItem& it, bool active, SortSlots<K>& sl,
                                              DevMeta* meta) {
    static_assert(K == 1 || (K == 2 && L == kWave), "slot order");
    constexpr int kSlotBits = K == 1 ? 6 : 7;
    const int lane = lane_id();
    const int lr = lane % L;
    const WaveOperands<V> W{uniform_ptr(Pr.a_val), uniform_ptr(Pr.bref), uniform_ptr(Pr.b_col),
                            uniform_ptr(Pr.b_val), 0};
    const auto c_col = uniform_ptr(Pr.c_col);
    const auto c_val = uniform_ptr(Pr.c_val);
    if (lane < K) sl.starts[lane] = 0;
    const int nip = active ? it.nip : 0;
    // an entry of A to a lane
    long long ref = 0;
    V av = V(0);
    if (active && it.a0 + lr < it.a1) {
        ref = W.bref[it.a0 + lr];
        av = W.a_val[it.a0 + lr];
    }
    const int len = bref_len(ref);
    const int start = group_excl_sum<L>(len);
    wave_sync();
    if (len > 0) {
        const int at = lane - lr + start;  // the slot of the entry's first product
        atomicOr(&sl.starts[K == 1 ? 0 : at >> 6], 1ull << (at & 63));
    }
    const unsigned long long filled = __ballot(len > 0);
    if (len > 0) {
        WaveEntry<true> w;
        w.av = av;
        w.d = (bref_start(ref) - start) * 4;  // bytes of b_col, modulo 2^32
        sl.ent[rank_in(filled)] = w;
    }
    wave_sync();
    uint32_t word[K];
    LdsSum prod[K];
    int before = -1;
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const unsigned long long m = sl.starts[j];
        const unsigned lo = static_cast<unsigned>(uniform(static_cast<int>(m)));
        const unsigned hi = static_cast<unsigned>(uniform(static_cast<int>(m >> 32)));
        const unsigned long long mu = static_cast<unsigned long long>(hi) << 32 | lo;
        const int e = before + rank_in(mu) + (in_mask(mu) ? 1 : 0);
        before += __popcll(mu);
        const bool ok = j * kWave + lr < nip;
        const WaveEntry<true> w = sl.ent[ok ? e : 0];
        const uint32_t pos = static_cast<uint32_t>(w.d) + static_cast<uint32_t>((j * kWave + lr) * 4);
        const uint32_t o = ok ? pos : 0u;
        const int key = *(const int32_t SPG_GLOBAL*)((const char SPG_GLOBAL*)W.b_col + o);
        const V bv = *(const V SPG_GLOBAL*)((const char SPG_GLOBAL*)W.b_val + o * static_cast<uint32_t>(sizeof(V) / 4));
        prod[j] = w.av * static_cast<LdsSum>(bv);
        word[j] = ok ? static_cast<uint32_t>(key) << kSlotBits | static_cast<uint32_t>(j * kWave + lane) : ~0u;
    }
    wave_sync();  // every lane has read its entries
#pragma unroll
    for (int j = 0; j < K; ++j) {
        sl.prod[j * kWave + lane] = prod[j];
        sl.sum[j * kWave + lane] = 0;
    }
    wave_sort<K, L>(word);
    wave_sync();
    // sorted slot lane * K + s of the wave; heads: first of its column in its row
    uint32_t below = lane_below(word[K - 1]);
    bool head[K], real[K];
    unsigned long long heads[K], repeats = 0;
    const unsigned long long group = L == kWave ? ~0ull : ((1ull << (L % kWave)) - 1) << (lane - lr);
#pragma unroll
    for (int s = 0; s < K; ++s) {
        real[s] = word[s] != ~0u;
        head[s] = real[s] && ((s == 0 && lr == 0) || (word[s] >> kSlotBits) != (below >> kSlotBits));
        heads[s] = __ballot(head[s]);
        repeats |= __ballot(real[s] && !head[s]);
        below = word[s];
    }
    int rank[K];
    int found = 0;
#pragma unroll
    for (int s = 0; s < K; ++s) found += __popcll(heads[s] & group);
#pragma unroll
    for (int s = 0; s < K; ++s) {
        rank[s] = 0;
#pragma unroll
        for (int t = 0; t < K; ++t) rank[s] += rank_in(heads[t] & group) + (t < s && head[t] ? 1 : 0);
    }
    if (active && lr == 0 && found != it.cn) atomicOr(&meta->flags.v, kFlagMismatch);
    LdsSum val[K];
#pragma unroll
    for (int s = 0; s < K; ++s) val[s] = sl.prod[word[s] & (kWave * K - 1)];
    if (repeats) {
        const int g0 = (lane - lr) * K;  // the row's first place among the sums
#pragma unroll
        for (int s = 0; s < K; ++s)
            if (real[s]) lds_add(&sl.sum[g0 + rank[s] - (head[s] ? 0 : 1)], val[s]);
        wave_sync();
#pragma unroll
        for (int s = 0; s < K; ++s)
            if (head[s]) val[s] = sl.sum[g0 + rank[s]];
    }
#pragma unroll
    for (int s = 0; s < K; ++s)
        if (head[s] && rank[s] < it.cn) {
            c_col[it.c0 + rank[s]] = static_cast<int32_t>(word[s] >> kSlotBits);
            c_val[it.c0 + rank[s]] = static_cast<V>(val[s]);
        }
    wave_sync();  // LDS is reused by the next rows
}

// Whether symnum_sorted takes a wave's rows (every lane: its row's item).
template <typename V, int L, int K>
__device__ __forceinline__ bool sorted_fits(const GProb<V>& Pr, const RowItem& it, bool active) {
    const bool fits = it.nip <= L * K && it.a1 - it.a0 <= L && it.inst == uniform(it.inst) &&
                      !(Pr.wide & kWideOffsets) && Pr.n < 1 << kSortColBits<K>;
    return __ballot(active && !fits) == 0;
}

template <typename V, int WG, int R, int P, int EC, int PMAX>
__device__ __forceinline__ void symnum_rows(const ProbSet<V>& ps, const RowItem* __restrict__ items, int first,
                                            int end, int* smem, int* s_tmp, DevMeta* meta) {
    constexpr int L = WG / R;
    constexpr int T = 2 * P;
    constexpr int ROW_INTS = num_row_ints(NumVariant{WG, R, P, EC, PMAX});
    static_assert(WG % R == 0, "bad variant shape");
    static_assert(L <= kWave || R == 1, "a row spans several waves only when it owns the workgroup");
    static_assert(T * sizeof(int) >= P * sizeof(LdsSum), "values must fit in the table's LDS");
    static_assert(ROW_INTS % 2 == 0, "row slots must stay 8-byte aligned");
    using Meta = ChunkMeta<V, EC, true>;
    using KeyMeta = ChunkMeta<V, EC, false>;
    const int slot = threadIdx.x / L;
    const int lr = threadIdx.x % L;
    int* tab = smem + slot * ROW_INTS;
    int* cols = tab + T;
    Meta* cm = reinterpret_cast<Meta*>(cols + P);
    LdsSum* vals = reinterpret_cast<LdsSum*>(tab);

    const int idx = first + slot;
    const bool active = idx < end;
    const RowItem it = active ? load_item(items, idx) : RowItem{0, 0, 0, 0, 0, 0, 0, 0};
    if constexpr (L >= 8 && L < kWave && P == L) {
        if (__ballot(active) == 0) return;  // no row, and so no product whose B could be read
        const GProb<V> Pu = ps.get(uniform(it.inst));
        if (sorted_fits<V, L, 1>(Pu, it, active)) {
            static_assert(kWave / L * ROW_INTS * 4 >= static_cast<int>(sizeof(SortSlots<1>)) &&
                              kWave / L * ROW_INTS % 4 == 0, "a wave's slots lie in its rows' LDS");
            symnum_sorted<V, L, 1>(Pu, it, active, *reinterpret_cast<SortSlots<1>*>(tab - slot % (kWave / L) * ROW_INTS),
                                   meta);
            return;
        }
    }
    lds_fill<T, L>(tab, kEmpty, lr);
    gsync<L>();
    const GProb<V> Pr = ps.get(it.inst);
    const int a0 = it.a0, a1 = it.a1, nip = it.nip, c0 = it.c0, cn = it.cn;
    // products staged in registers when the whole row fits in one round
    const bool fits = a1 - a0 <= EC && nip <= L * PMAX;
    int key[PMAX];
    V prod[PMAX];
    bool ok[PMAX];
    if (fits) {
        int total;
        if constexpr (L == 1) {
            Meta rm;
            total = load_chunk_lane<V, EC, true>(Pr, a0, a1, rm);
            fetch_products_lane<V, EC, PMAX, true>(Pr, rm, total, 0, key, prod, ok);
        } else {
            total = load_chunk<V, L, EC, true>(Pr, a0, a1, lr, cm, s_tmp);
            fetch_products<V, L, EC, PMAX, true>(Pr, cm, total, 0, lr, key, prod, ok);
        }
        table_insert_all<T>(tab, key, ok);
    } else {
        for_each_round<V, L, EC, PMAX, false>(
            Pr, a0, a1, lr, reinterpret_cast<KeyMeta*>(cm), s_tmp,
            [&](const int(&k)[PMAX], const V(&)[PMAX], const bool(&o)[PMAX]) { table_insert_all<T>(tab, k, o); });
    }
    gsync<L>();

    constexpr int E = L <= kWave ? P / L : 1;
    int x[E];
    const int found = sort_row<L, T, P>(tab, cols, lr, s_tmp, x);
    const int n = min(found, P);

    int w = 0;
    if (active) {
        if (lr == 0 && cn != found) atomicOr(&meta->flags.v, kFlagMismatch);
        w = min(n, cn);
    }
    if constexpr (L <= kWave) {
#pragma unroll
        for (int s = 0; s < E; ++s)
            if (lr * E + s < w) Pr.c_col[c0 + lr * E + s] = x[s];
    } else {
        for (int j = lr; j < w; j += L) Pr.c_col[c0 + j] = cols[j];
    }
    for (int j = lr; j < P; j += L) vals[j] = 0;
    gsync<L>();

    // binary search of every product's column in the sorted list
    // (find_key, num.cuh:28-41), all of a lane's products in lockstep, then
    // LDS atomic adds that nothing waits for
    // (in groups of up to 8 keys, which bounds the registers in flight)
    auto accumulate = [&](const int(&k)[PMAX], const V(&v)[PMAX], const bool(&o)[PMAX]) {
        constexpr int G = PMAX % 8 == 0 ? 8 : (PMAX % 6 == 0 ? 6 : (PMAX % 4 == 0 ? 4 : PMAX));
        static_for<0, PMAX / G>([&](auto gi) {
            constexpr int J0 = decltype(gi)::value * G;
            int pos[G];
            lower_bound_all<P, G, J0>(cols, k, pos);
#pragma unroll
            for (int j = 0; j < G; ++j)
                if (o[J0 + j]) lds_add(vals + pos[j], static_cast<LdsSum>(v[J0 + j]));
        });
    };
    if (fits)
        accumulate(key, prod, ok);
    else
        for_each_round<V, L, EC, PMAX, true>(Pr, a0, a1, lr, cm, s_tmp, accumulate);
    gsync<L>();
    for (int j = lr; j < w; j += L) Pr.c_val[c0 + j] = static_cast<V>(vals[j]);
    gsync<L>();  // LDS is reused by the next unit
}

// A row of one wave (64 lanes).  The hash table carries a value beside every
// key: a product is looked up (or its column inserted) once and its value
// added to its slot right away, so the row's products are walked once, however
// many there are, and nothing of them outlives the walk.  (The narrower
// variants keep or re-read the products and binary-search the sorted list for
// each: seven dependent LDS reads a product at P = 128.)  The occupied slots
// are then compacted, sorted in registers, and every sorted column picks its
// value up from the table, one probe per entry of C instead of one search per
// product.  Bound by VALU issue and LDS latency: four slots a round and 64
// VGPRs (eight waves per SIMD) beat six or eight slots at six or five waves
// by 7 and 18 %, and a table of 4P slots (fewer probes, five waves) by 6 %.
// 96^3 stencil (729 products and 125 entries a row, FP64): 2.70 ms for the
// launch with staged products and binary searches, 1.23 ms so.
template <typename V, int P, int T, int N>
__device__ __forceinline__ void symnum_wave_row(const ProbSet<V>& ps, const RowItem* __restrict__ items, int idx,
                                                WaveRow<P, T>& row, DevMeta* meta) {
    constexpr int E = P / kWave;
    constexpr int S = T / kWave;
    static_assert(T % (2 * kWave) == 0 && P % kWave == 0, "every lane clears and compacts whole shares");
    const int lane = lane_id();
    const RowItem it = load_item(items, idx);
    const GProb<V> Pr = ps.get(uniform(it.inst));
    if constexpr (P <= 2 * kWave) {
        if (sorted_fits<V, kWave, P / kWave>(Pr, it, true)) {
            symnum_sorted<V, kWave, P / kWave>(Pr, it, true, *reinterpret_cast<SortSlots<P / kWave>*>(&row), meta);
            return;
        }
    }
    {
        typedef int Words __attribute__((vector_size(16)));
        Words* k = reinterpret_cast<Words*>(row.keys);
        Words* v = reinterpret_cast<Words*>(row.vals);
#pragma unroll
        for (int i = lane; i < T / 4; i += kWave) k[i] = Words{kEmpty, kEmpty, kEmpty, kEmpty};
#pragma unroll
        for (int i = 0; i < T * static_cast<int>(sizeof(LdsSum)) / (16 * kWave); ++i)
            v[i * kWave + lane] = Words{0, 0, 0, 0};
    }
    const WaveOperands<V> W{uniform_ptr(Pr.a_val), uniform_ptr(Pr.bref), uniform_ptr(Pr.b_col),
                            uniform_ptr(Pr.b_val), uniform(Pr.wide)};
    wave_sync();
    wave_products<V, N, true>(
        W, uniform(it.a0), uniform(it.a1), &row.walk,
        [&](const int(&key)[N], const LdsSum(&prod)[N], const unsigned long long(&ok)[N], auto far) {
            uint32_t h[N];
            int fresh = 0;
            table_slots<T, far>(row.keys, key, ok, h, fresh);
#pragma unroll
            for (int j = 0; j < N; ++j)
                if (in_mask(ok[j])) lds_add(row.vals + h[j], prod[j]);
        });
    wave_sync();

    // the occupied slots, S consecutive ones to a lane, in front of each other
    const SlotWord<T> sw(uniform(Pr.n));
    int key[S];
    int mine = 0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        key[s] = row.keys[lane * S + s];
        mine += key[s] != kEmpty ? 1 : 0;
    }
    const int incl = wave_incl_scan(mine);
    const int found = wave_last(incl);
    int pos = incl - mine;
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (key[s] != kEmpty) {
            if (pos < P) row.words[pos] = sw.pack(key[s], lane * S + s);
            ++pos;
        }
    wave_sync();
    const int cn = uniform(it.cn);
    if (lane == 0 && cn != found) atomicOr(&meta->flags.v, kFlagMismatch);
    const int w = min(min(found, P), cn);
    uint32_t x[E];
#pragma unroll
    for (int s = 0; s < E; ++s) {
        x[s] = row.words[lane * E + s];
        if (lane * E + s >= found) x[s] = ~0u;
    }
    wave_sort<E>(x);
    const auto ccol = uniform_ptr(Pr.c_col) + uniform(it.c0);
    const auto cval = uniform_ptr(Pr.c_val) + uniform(it.c0);
#pragma unroll
    for (int s = 0; s < E; ++s)
        if (lane * E + s < w) {
            ccol[lane * E + s] = sw.column(x[s]);
            cval[lane * E + s] = static_cast<V>(row.vals[sw.slot(row.keys, x[s])]);
        }
    wave_sync();  // LDS is reused by the next row
}

// The same for a row of a whole workgroup.  Every wave walks a share of the
// products on its own and all add into one table.  Each wave then sorts a
// block of the compacted columns in registers; a column's place in C is its
// place in its block plus the number of smaller columns in every other block
// (binary searches in LDS), where it leaves its table slot for the coalesced
// write of C.  27^3 nodes of 3 unknowns (6,561 products, 375 columns a row,
// FP64): 1.74 ms for the launch with two walks and a search per product,
// 0.46 ms so.  Rows up to 512 columns have a variant of their own, whose
// 18 KB of LDS let eight workgroups share a CU (31 KB for 1024: five).
template <typename V, int WG, int P, int T, int N>
__device__ __forceinline__ void symnum_group_row(const ProbSet<V>& ps, const RowItem* __restrict__ items, int idx,
                                                 GroupRow<P, T, WG / kWave>& row, DevMeta* meta) {
    constexpr int kWaves = WG / kWave;
    constexpr int B = P / kWaves;  // columns of a wave's block
    constexpr int E = B / kWave;
    constexpr int S = T / WG;
    static_assert(T % (4 * WG) == 0 && P % WG == 0, "every thread clears and compacts whole shares");
    const int lane = lane_id();
    const int wave = uniform(static_cast<int>(threadIdx.x) / kWave);
    {
        typedef int Words __attribute__((vector_size(16)));
        Words* k = reinterpret_cast<Words*>(row.keys);
        Words* v = reinterpret_cast<Words*>(row.vals);
#pragma unroll
        for (int i = 0; i < T / (4 * WG); ++i) k[i * WG + threadIdx.x] = Words{kEmpty, kEmpty, kEmpty, kEmpty};
#pragma unroll
        for (int i = 0; i < T / (2 * WG); ++i) v[i * WG + threadIdx.x] = Words{0, 0, 0, 0};
    }
    const RowItem it = load_item(items, idx);
    const GProb<V> Pr = ps.get(uniform(it.inst));
    const WaveOperands<V> W{uniform_ptr(Pr.a_val), uniform_ptr(Pr.bref), uniform_ptr(Pr.b_col),
                            uniform_ptr(Pr.b_val), uniform(Pr.wide)};
    const int a0 = uniform(it.a0), a1 = uniform(it.a1);
    __syncthreads();
    wave_products<V, N, true>(
        W, a0, a1, &row.walk[wave],
        [&](const int(&key)[N], const LdsSum(&prod)[N], const unsigned long long(&ok)[N], auto far) {
            uint32_t h[N];
            int fresh = 0;
            table_slots<T, far>(row.keys, key, ok, h, fresh);
#pragma unroll
            for (int j = 0; j < N; ++j)
                if (in_mask(ok[j])) lds_add(row.vals + h[j], prod[j]);
        },
        wave, kWaves, wave_by_chunk<kWaves>(a1 - a0, uniform(it.nip)));
    __syncthreads();

    // the occupied slots, S consecutive ones to a thread, in front of each other
    const SlotWord<T> sw(uniform(Pr.n));
    int key[S];
    int mine = 0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        key[s] = row.keys[threadIdx.x * S + s];
        mine += key[s] != kEmpty ? 1 : 0;
    }
    const int incl = wave_incl_scan(mine);
    if (lane == kWave - 1) row.wave_sum[wave] = incl;
    __syncthreads();
    int found = 0, pos = incl - mine;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        const int n = row.wave_sum[w];
        pos += w < wave ? n : 0;
        found += n;
    }
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (key[s] != kEmpty) {
            if (pos < P) row.words[pos] = sw.pack(key[s], static_cast<int>(threadIdx.x) * S + s);
            ++pos;
        }
    __syncthreads();
    const int cn = uniform(it.cn);
    if (threadIdx.x == 0 && cn != found) atomicOr(&meta->flags.v, kFlagMismatch);
    const int n = min(found, P);
    const int w = min(n, cn);
    const int mine0 = wave * B + lane * E;
    uint32_t x[E];
#pragma unroll
    for (int s = 0; s < E; ++s) x[s] = mine0 + s < n ? row.words[mine0 + s] : ~0u;
    if (wave * B < n) {
        wave_sort<E>(x);
#pragma unroll
        for (int s = 0; s < E; ++s) row.words[mine0 + s] = x[s];
    }
    __syncthreads();
    if (wave * B < n) {
        int rank[E];
#pragma unroll
        for (int s = 0; s < E; ++s) rank[s] = lane * E + s;
#pragma unroll
        for (int o = 1; o < kWaves; ++o) {
            const int other = (wave + o) % kWaves;
            if (other * B >= n) continue;
            int at[E];
            lower_bound_all<B, E>(row.words + other * B, x, at);
#pragma unroll
            for (int s = 0; s < E; ++s) {
                // (a block of B columns may hold none as large: B steps of the search end one short)
                at[s] += row.words[other * B + at[s]] < x[s] ? 1 : 0;
                rank[s] += at[s];
            }
        }
#pragma unroll
        for (int s = 0; s < E; ++s)
            if (mine0 + s < n) row.slots[rank[s]] = static_cast<unsigned short>(sw.slot(row.keys, x[s]));
    }
    __syncthreads();
    const auto ccol = uniform_ptr(Pr.c_col) + uniform(it.c0);
    const auto cval = uniform_ptr(Pr.c_val) + uniform(it.c0);
    for (int j = threadIdx.x; j < w; j += WG) {
        const int h = row.slots[j];
        ccol[j] = row.keys[h];
        cval[j] = static_cast<V>(row.vals[h]);
    }
    __syncthreads();  // LDS is reused by the next row
}

// Rows of up to P columns whose table takes most of LDS (a workgroup of 16
// waves on a CU of its own): the columns are found in LDS and compacted
// through C.col, their sorted list takes the table's place, and a second walk
// finds every product in it (15 LDS steps, four products of a lane in
// lockstep) and adds it to C.val in memory.  The searches are what the
// global-memory path below is slow at: a row of 16,767 products and 14,389
// columns took 460 us there, most of it dependent reads of the sorted list.
template <typename V, int WG, int P, int T, int N>
__device__ __forceinline__ void symnum_long_row(const ProbSet<V>& ps, const RowItem* __restrict__ items, int idx,
                                                LongRow<T, WG / kWave>& row, int* s_tmp, DevMeta* meta) {
    constexpr int kWaves = WG / kWave;
    static_assert(P < T && T % (4 * WG) == 0, "the table keeps free slots");
    const int wave = uniform(static_cast<int>(threadIdx.x) / kWave);
    typedef int Words __attribute__((vector_size(16)));
    for (int i = threadIdx.x; i < T / 4; i += WG)
        reinterpret_cast<Words*>(row.keys)[i] = Words{kEmpty, kEmpty, kEmpty, kEmpty};
    const RowItem it = load_item(items, idx);
    const GProb<V> Pr = ps.get(uniform(it.inst));
    const WaveOperands<V> W{uniform_ptr(Pr.a_val), uniform_ptr(Pr.bref), uniform_ptr(Pr.b_col),
                            uniform_ptr(Pr.b_val), uniform(Pr.wide)};
    const int a0 = uniform(it.a0), a1 = uniform(it.a1), cn = uniform(it.cn);
    const bool by_chunk = wave_by_chunk<kWaves>(a1 - a0, uniform(it.nip));
    const auto ccol = uniform_ptr(Pr.c_col) + uniform(it.c0);
    const auto cval = uniform_ptr(Pr.c_val) + uniform(it.c0);
    for (int j = threadIdx.x; j < cn; j += WG) cval[j] = V(0);
    __syncthreads();
    // (the walk without values uses the front of the same metadata)
    wave_products<V, N, false>(
        W, a0, a1, reinterpret_cast<WaveChunk<false>*>(&row.walk[wave]),
        [&](const int(&key)[N], const LdsSum(&)[N], const unsigned long long(&ok)[N], auto far) {
            uint32_t h[N];
            int fresh = 0;
            table_slots<T, far>(row.keys, key, ok, h, fresh);
        },
        wave, kWaves, by_chunk);
    __syncthreads();
    // the occupied slots into C.col, unsorted, WG * 4 slots at a time
    int found = 0;
    for (int base = 0; base < T; base += 4 * WG) {
        const Words k = reinterpret_cast<const Words*>(row.keys)[base / 4 + threadIdx.x];
        int mine = 0;
#pragma unroll
        for (int s = 0; s < 4; ++s) mine += k[s] != kEmpty ? 1 : 0;
        int total;
        int pos = found + group_excl_scan<WG>(mine, threadIdx.x, s_tmp, total);
#pragma unroll
        for (int s = 0; s < 4; ++s)
            if (k[s] != kEmpty) {
                if (pos < cn) ccol[pos] = k[s];
                ++pos;
            }
        found += total;
    }
    if (threadIdx.x == 0 && found != cn) atomicOr(&meta->flags.v, kFlagMismatch);
    const int n = min(found, cn);
    __threadfence();  // C.val is zero, C.col written, before other waves read or add
    __syncthreads();
    // the smallest power of two of columns that holds them all
    auto sort_as = [&](auto size) {
        constexpr int kP = decltype(size)::value;
        for (int j = threadIdx.x; j < kP; j += WG)
            row.keys[j] = j < n ? __hip_atomic_load(ccol + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : INT_MAX;
        __syncthreads();
        bitonic_sort_block<kP, WG>(row.keys, threadIdx.x);
    };
    if (n <= T / 2)
        sort_as(std::integral_constant<int, T / 2>{});
    else
        sort_as(std::integral_constant<int, T>{});
    for (int j = threadIdx.x; j < n; j += WG) ccol[j] = row.keys[j];
    const int half = n <= T / 2 ? T / 4 : T / 2;
    wave_products<V, N, true>(
        W, a0, a1, &row.walk[wave],
        [&](const int(&key)[N], const LdsSum(&prod)[N], const unsigned long long(&ok)[N], auto far) {
            int pos[N];
#pragma unroll
            for (int j = 0; j < N; ++j) pos[j] = 0;
            for (int step = half; step > 0; step >>= 1) {
                int probe[N];
#pragma unroll
                for (int j = 0; j < N; ++j) probe[j] = row.keys[pos[j] + step - 1];
#pragma unroll
                for (int j = 0; j < N; ++j) pos[j] += probe[j] < key[j] ? step : 0;
            }
#pragma unroll
            for (int j = 0; j < N; ++j)
                if (in_mask(ok[j]) && pos[j] < n)
                    __hip_atomic_fetch_add(cval + pos[j], static_cast<V>(prod[j]), __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
        },
        wave, kWaves, by_chunk);
    __syncthreads();  // LDS is reused by the next row
}

// The rows [first, end) of one unit of variant VV.
template <typename V, int VV>
__device__ __forceinline__ void symnum_unit(const ProbSet<V>& ps, const RowItem* __restrict__ items, int first,
                                            int end, int* smem, int* s_tmp, DevMeta* meta) {
    constexpr NumVariant kV = kNumVariants[VV];
    if constexpr (num_is_wave(kV)) {
        const int wave = uniform(static_cast<int>(threadIdx.x) / kWave);
        if (first + wave < end)
            symnum_wave_row<V, kV.p, kV.t, kV.pmax>(ps, items, first + wave,
                                                    reinterpret_cast<WaveRow<kV.p, kV.t>*>(smem)[wave], meta);
    } else if constexpr (num_is_long(kV)) {
        symnum_long_row<V, kV.wg, kV.p, kV.t, kV.pmax>(ps, items, first,
                                                       *reinterpret_cast<LongRow<kV.t, kV.wg / kWave>*>(smem), s_tmp, meta);
    } else if constexpr (num_is_group(kV)) {
        symnum_group_row<V, kV.wg, kV.p, kV.t, kV.pmax>(
            ps, items, first, *reinterpret_cast<GroupRow<kV.p, kV.t, kV.wg / kWave>*>(smem), meta);
    } else {
        symnum_rows<V, kV.wg, kV.r, kV.p, kV.ec, kV.pmax>(ps, items, first, end, smem, s_tmp, meta);
    }
}

// One launch per fused variant over the units (R rows each) of one bin; the
// host launches a workgroup per unit (residency is the hardware's), and the
// unit of a workgroup is chosen so that consecutive units stay on one XCD.
// A smaller grid walks the units persistently.
template <typename V, int VV>
__global__ __launch_bounds__(kNumVariants[VV].wg) SPG_WAVES_PER_EU(kNumMinWaves[VV]) void k_symnum_bin(ProbSet<V> ps, const RowItem* __restrict__ items,
                                                                    int item_off, int count, DevMeta* meta) {
    constexpr NumVariant kV = kNumVariants[VV];
    __shared__ __align__(16) int smem[kV.r * num_row_ints(kV)];
    __shared__ int s_tmp[kV.wg / kWave];
    const int units = (count + kV.r - 1) / kV.r;
    const UnitRange ur = xcd_units(units);
    for (int u = ur.first; u < ur.end; u += ur.stride)
        symnum_unit<V, VV>(ps, items, item_off + u * kV.r, item_off + count, smem, s_tmp, meta);
}

#define SPG_NUM_VARIANTS(X) \
    X(0) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15) X(16) X(17) X(18) X(20)

// Several bins of the fused pass in one launch, a workgroup per unit.
// Each XCD gets a contiguous slice of every bin (balanced work across the
// XCDs, and neighbouring rows, which read the same rows of B, meet in one
// L2).  Registers are the largest member's (kept within the set's
// residency floor), LDS the largest member's; a workgroup runs one unit, so
// no LDS layout is reused by another variant.
template <typename V, int SET>
__global__ __launch_bounds__(256) SPG_WAVES_PER_EU(kNumMultiMinWaves[SET]) void k_symnum_multi(
    ProbSet<V> ps, const RowItem* __restrict__ items, NumMultiBins mb, DevMeta* meta) {
    __shared__ __align__(16) int smem[max_num_multi_lds(SET) / 4];
    __shared__ int s_tmp[256 / kWave];
    const int xcd = blockIdx.x % kXcds;
    const int local = blockIdx.x / kXcds;
    int b = 0;
    while (b + 1 < mb.n && local >= mb.slice0[b + 1]) ++b;
    const int per = mb.slice0[b + 1] - mb.slice0[b];
    const int k = xcd * per + (local - mb.slice0[b]);  // unit of bin b
    const int end = mb.off[b] + mb.count[b];
#define SPG_MULTI_CASE(v)                                                                                   \
    case v:                                                                                                 \
        if constexpr (num_multi_set(v) == SET) {                                                            \
            static_assert(kNumVariants[v].wg == 256, "merged launches run 256-thread variants");           \
            if (mb.off[b] + k * kNumVariants[v].r < end)                                                    \
                symnum_unit<V, v>(ps, items, mb.off[b] + k * kNumVariants[v].r, end, smem, s_tmp, meta);    \
        }                                                                                                   \
        break;
    switch (mb.variant[b]) {
        SPG_NUM_VARIANTS(SPG_MULTI_CASE)
        default:
            break;
    }
#undef SPG_MULTI_CASE
}

// Lower bound in a sorted global list (values read coherently).
template <typename Ptr>
__device__ __forceinline__ int lower_bound_global(Ptr cols, int n, int key) {
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (__hip_atomic_load(cols + mid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < key)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

// Rows above every LDS capacity: hash table in global memory, compaction
// into C.col, a sort of C.col in LDS-sized chunks followed by a merge by
// rank (each key's position = its rank in its chunk + the number of smaller
// keys in every other chunk), then binary search + global atomic adds into
// C.val (num.cuh:251-298).  The reference's O(nnz^2) rank sort
// (sym2.cuh:279-287) becomes O(nnz * chunks * log chunk).
template <typename V>
__global__ __launch_bounds__(1024) void k_symnum_global(ProbSet<V> ps, const RowItem* __restrict__ items,
                                                        const long long* __restrict__ gpool_off, int item_off,
                                                        int* pool, DevMeta* meta) {
    constexpr int WG = 1024;
    constexpr int EC = 1024;
    constexpr int PMAX = 4;
    constexpr int CH = kGlobalSortChunk;
    using Meta = ChunkMeta<V, EC, true>;
    __shared__ __align__(16) int chunk[CH];
    __shared__ Meta cm;
    __shared__ int s_tmp[WG / kWave];
    __shared__ int s_n;
    const RowItem it = load_item(items, item_off + blockIdx.x);
    const GProb<V> P = ps.get(it.inst);
    const int c0 = it.c0;
    const int nnz = it.cn;
    const long long slots = global_table_slots(nnz);
    const int bits = __builtin_ctzll(static_cast<unsigned long long>(slots));
    const uint32_t mask = static_cast<uint32_t>(slots - 1);
    int* tab = pool + gpool_off[item_off + blockIdx.x];
    auto ccol = P.c_col + c0;
    auto cval = P.c_val + c0;
    for (long long j = threadIdx.x; j < slots; j += WG) tab[j] = kEmpty;
    for (int j = threadIdx.x; j < nnz; j += WG) cval[j] = V(0);
    if (threadIdx.x == 0) s_n = 0;
    __threadfence();
    __syncthreads();

    const int a0 = it.a0;
    const int a1 = it.a1;
    for_each_product<V, WG, EC, PMAX, false>(
        P, a0, a1, threadIdx.x, reinterpret_cast<ChunkMeta<V, EC, false>*>(&cm), s_tmp, [&](int key, V) {
            uint32_t h = hash_slot_rt(key, bits);
            while (true) {
                const int cur = __hip_atomic_load(tab + h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (cur == key) break;
                if (cur == kEmpty) {
                    const int old = atomicCAS(tab + h, kEmpty, key);
                    if (old == kEmpty || old == key) break;
                }
                h = (h + 1) & mask;
            }
        });
    __threadfence();
    __syncthreads();

    // compact the occupied slots into C.col (unsorted)
    for (long long j = threadIdx.x; j < slots; j += WG) {
        const int key = __hip_atomic_load(tab + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (key != kEmpty) {
            const int pos = atomicAdd(&s_n, 1);
            if (pos < nnz) ccol[pos] = key;
        }
    }
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0 && s_n != nnz) atomicOr(&meta->flags.v, kFlagMismatch);
    const int n = min(s_n, nnz);

    // sort chunks in LDS, staging them in the (now free) table
    const int nch = (n + CH - 1) / CH;
    for (int c = 0; c < nch; ++c) {
        for (int j = threadIdx.x; j < CH; j += WG) {
            const int e = c * CH + j;
            chunk[j] = e < n ? __hip_atomic_load(ccol + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : INT_MAX;
        }
        __syncthreads();
        bitonic_sort_block<CH, WG>(chunk, threadIdx.x);
        for (int j = threadIdx.x; j < CH; j += WG) tab[static_cast<long long>(c) * CH + j] = chunk[j];
        __syncthreads();
    }
    __threadfence();
    __syncthreads();
    // merge by rank
    for (int e = threadIdx.x; e < n; e += WG) {
        const int c = e / CH;
        const int x = __hip_atomic_load(tab + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        int rank = e - c * CH;
        for (int o = 0; o < nch; ++o) {
            if (o == c) continue;
            const int len = min(CH, n - o * CH);
            rank += lower_bound_global(tab + static_cast<long long>(o) * CH, len, x);
        }
        ccol[rank] = x;
    }
    __threadfence();
    __syncthreads();

    for_each_product<V, WG, EC, PMAX, true>(P, a0, a1, threadIdx.x, &cm, s_tmp, [&](int key, V v) {
        const int pos = lower_bound_global(ccol, n, key);
        if (pos < n) __hip_atomic_fetch_add(cval + pos, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    });
}

// ----------------------------------------------------------------- launchers

template <typename V, int VV>
static hipError_t launch_variant(const ProbSet<V>& ps, const RowItem* items, int item_off, int count, DevMeta* meta,
                                 int grid, hipStream_t s) {
    constexpr auto kernel = k_symnum_bin<V, VV>;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kNumVariants[VV].wg), 0, s, ps, items, item_off, count, meta);
    return hipGetLastError();
}

template <typename V>
hipError_t launch_symnum_bin(int variant, const ProbSet<V>& ps, const RowItem* items, int item_off, int count,
                             DevMeta* meta, int grid, hipStream_t s) {
#define SPG_LAUNCH_CASE(v) \
    case v:                \
        return launch_variant<V, v>(ps, items, item_off, count, meta, grid, s);
    switch (variant) {
        SPG_NUM_VARIANTS(SPG_LAUNCH_CASE)
        default:
            return hipErrorInvalidValue;
    }
#undef SPG_LAUNCH_CASE
}

template <typename V>
hipError_t launch_symnum_multi(int set, const ProbSet<V>& ps, const RowItem* items, const NumMultiBins& mb,
                               DevMeta* meta, hipStream_t s) {
    const int grid = kXcds * mb.slice0[mb.n];  // one unit per workgroup
    if (set == 0)
        hipLaunchKernelGGL((k_symnum_multi<V, 0>), dim3(grid), dim3(256), 0, s, ps, items, mb, meta);
    else if (set == 1)
        hipLaunchKernelGGL((k_symnum_multi<V, 1>), dim3(grid), dim3(256), 0, s, ps, items, mb, meta);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

template <typename V>
void launch_symnum_global(const ProbSet<V>& ps, const RowItem* items, const long long* gpool_off, int item_off,
                          int count, int* pool, DevMeta* meta, hipStream_t s) {
    hipLaunchKernelGGL(k_symnum_global<V>, dim3(count), dim3(1024), 0, s, ps, items, gpool_off, item_off, pool,
                       meta);
}

template <typename V>
void load_symnum() {
    int n = 0;
#define SPG_LOAD_CASE(v)                                                                                             \
    {                                                                                                                \
        constexpr auto kernel = k_symnum_bin<V, v>;                                                                  \
        (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, kNumVariants[v].wg, 0);                       \
    }
    SPG_NUM_VARIANTS(SPG_LOAD_CASE)
#undef SPG_LOAD_CASE
}

#define SPG_INSTANTIATE_NUM(V)                                                                               \
    template hipError_t launch_symnum_bin<V>(int, const ProbSet<V>&, const RowItem*, int, int, DevMeta*, int,    \
                                             hipStream_t);                                                    \
    template hipError_t launch_symnum_multi<V>(int, const ProbSet<V>&, const RowItem*, const NumMultiBins&,       \
                                               DevMeta*, hipStream_t);                                        \
    template void launch_symnum_global<V>(const ProbSet<V>&, const RowItem*, const long long*, int, int, int*, \
                                          DevMeta*, hipStream_t);                                             \
    template void load_symnum<V>();

SPG_INSTANTIATE_NUM(float)
SPG_INSTANTIATE_NUM(double)

}  // namespace spg
