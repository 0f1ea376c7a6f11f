// Building blocks of the rows that whole waves work on (long rows): a wave
// walks a row's products 64 to a slot, kSlots slots to a round, and keeps
// everything that is the same for its 64 lanes (the row, the operands'
// pointers, product counts) in scalar registers.
//
// These passes are bound by the vector instructions they issue per product
// (a SIMD issues one per 4 cycles), so the helpers below are written by
// instruction count: prefix sums on DPP operands instead of cross-lane
// reads through LDS, a 24-bit multiply for the hash (a 32-bit one takes
// four times as long), 32-bit byte offsets from a scalar base for B's
// columns and values, and compare-exchanges whose direction is a constant
// lane mask.
#pragma once

#include "spg_common.hpp"

namespace spg {

__device__ __forceinline__ int uniform(int v) {
    return static_cast<int>(__builtin_amdgcn_readfirstlane(static_cast<unsigned>(v)));
}
template <typename T>
__device__ __forceinline__ T SPG_GLOBAL* uniform_ptr(T SPG_GLOBAL* p) {
    const unsigned long long v = (unsigned long long)p;
    const unsigned long long lo = static_cast<unsigned>(uniform(static_cast<int>(v)));
    const unsigned long long hi = static_cast<unsigned>(uniform(static_cast<int>(v >> 32)));
    return (T SPG_GLOBAL*)(lo | hi << 32);
}

// The lanes of a constant mask, as a per-lane predicate (no instruction on
// the vector side).
__device__ __forceinline__ bool in_mask(unsigned long long mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }

// Set bits of a wave mask below this lane.
__device__ __forceinline__ int rank_in(unsigned long long mask) {
    return static_cast<int>(__builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(mask >> 32),
                                                      __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(mask), 0u)));
}

// Inclusive prefix sum over the wave: four DPP row shifts, then the two row
// broadcasts.
__device__ __forceinline__ int wave_incl_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true);   // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, true);   // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, true);   // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, true);   // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2 and 3
    return v;
}
// The value of lane 63.
__device__ __forceinline__ int wave_last(int v) { return __builtin_amdgcn_readlane(v, kWave - 1); }

// Slot of a column below 2^24 in a table of T <= 2^16 slots: the fraction of
// column * golden ratio, from the low 24 bits of both factors.  Matrices of
// more columns (FAR) take hash_slot: here columns that differ by a multiple of
// 2^24 would share a slot, and 20,000 rows of 27 x 27 products on columns 2^24
// apart took 5.9 ms instead of 0.12 (2^20 apart: 1.4 instead of 0.32).
template <int T>
__device__ __forceinline__ uint32_t slot24(int key) {
    constexpr int kBits = __builtin_ctz(T);
    static_assert((T & (T - 1)) == 0 && kBits >= 1 && kBits <= 16, "bad table size");
    constexpr uint32_t kGolden = 0x9E3779u;
    uint32_t x;
#if defined(__HIP_DEVICE_COMPILE__)
    // (from plain code the compiler picks the slower 32-bit multiply)
    asm("v_mul_u32_u24 %0, %1, %2" : "=v"(x) : "v"(key), "s"(kGolden));
#else
    x = (static_cast<uint32_t>(key) & 0xFFFFFFu) * kGolden;
#endif
    return (x >> (24 - kBits)) & (T - 1);
}

template <int T, bool FAR>
__device__ __forceinline__ uint32_t walk_slot(int key) {
    if constexpr (FAR)
        return hash_slot<T>(key);
    else
        return slot24<T>(key);
}

// Slots of N keys in an LDS table of T slots (open addressing, linear
// probing), inserting those that are new; ok[j]: the lanes that have a key j.
// The probes of all keys advance together, each a compare-and-swap.  Lane
// sets are scalar masks throughout (a ballot of one comparison is that
// comparison's result register, so combining them costs no vector
// instruction), and a key whose lanes are all done costs nothing more.
// The table never fills (its row has fewer distinct columns than T).  With
// COUNT, `fresh` grows by the number of keys the wave inserted.
template <int T, bool FAR, int N, bool COUNT = false>
__device__ __forceinline__ void table_slots(int* tab, const int (&key)[N], const unsigned long long (&ok)[N],
                                            uint32_t (&h)[N], int& fresh) {
    int old[N];
    unsigned long long pend[N], any = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        h[j] = walk_slot<T, FAR>(key[j]);
        if (in_mask(ok[j])) old[j] = atomicCAS(tab + h[j], kEmpty, key[j]);
    }
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const unsigned long long taken = __ballot(old[j] != kEmpty);
        if constexpr (COUNT) fresh += __popcll(ok[j] & ~taken);
        pend[j] = ok[j] & taken & __ballot(old[j] != key[j]);
        h[j] = (h[j] + (in_mask(pend[j]) ? 1u : 0u)) & (T - 1);
        any |= pend[j];
    }
    while (any) {
#pragma unroll
        for (int j = 0; j < N; ++j)
            if (pend[j] && in_mask(pend[j])) old[j] = atomicCAS(tab + h[j], kEmpty, key[j]);
        any = 0;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            if (pend[j]) {
                const unsigned long long taken = __ballot(old[j] != kEmpty);
                if constexpr (COUNT) fresh += __popcll(pend[j] & ~taken);
                pend[j] &= taken & __ballot(old[j] != key[j]);
                h[j] = (h[j] + (in_mask(pend[j]) ? 1u : 0u)) & (T - 1);
                any |= pend[j];
            }
        }
    }
}

// A column as the sort carries it: above its table slot where both fit one
// word (B has fewer columns than leave room for the slot; all ones marks no
// column), alone otherwise, and then its slot is looked up again after the
// sort (four LDS probes a column in the worst lane of a wave).
template <int T>
struct SlotWord {
    static constexpr int kBits = __builtin_ctz(T);
    int shift;       // scalar: kBits or 0
    uint32_t slots;  // scalar: T - 1 or 0
    bool far;        // scalar: more than 2^24 columns
    __device__ __forceinline__ explicit SlotWord(int columns)
        : shift(columns < (1 << (32 - kBits)) ? kBits : 0), slots(shift ? T - 1 : 0), far(columns > 1 << 24) {}
    __device__ __forceinline__ uint32_t pack(int key, int slot) const {
        return static_cast<uint32_t>(key) << shift | (static_cast<uint32_t>(slot) & slots);
    }
    __device__ __forceinline__ int column(uint32_t w) const { return static_cast<int>(w >> shift); }
    __device__ __forceinline__ uint32_t slot(const int* tab, uint32_t w) const;
};

// Slot of a key that is in the table.
template <int T>
__device__ __forceinline__ uint32_t table_find(const int* tab, int key, bool far) {
    uint32_t h = far ? walk_slot<T, true>(key) : walk_slot<T, false>(key);
    while (lds_load(tab + h) != key) h = (h + 1) & (T - 1);
    return h;
}
template <int T>
__device__ __forceinline__ uint32_t SlotWord<T>::slot(const int* tab, uint32_t w) const {
    return shift ? w & (T - 1) : table_find<T>(tab, static_cast<int>(w), far);
}

// Sort of 64 * E keys, lane l holding keys l*E .. l*E + E-1 of the result
// (ascending): the bitonic network of bitonic_sort_regs for one whole wave,
// a compare and a select per key and stage.
template <int LJ>
__device__ __forceinline__ int wave_xor(int v) {
    if constexpr (LJ == 1)
        return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, false);  // quad_perm [1,0,3,2]
    else if constexpr (LJ == 2)
        return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, false);  // quad_perm [2,3,0,1]
    else if constexpr (LJ == 8)
        return __builtin_amdgcn_mov_dpp(v, 0x128, 0xF, 0xF, false);  // row_ror:8
    else if constexpr (LJ < 32)
        return __builtin_amdgcn_ds_swizzle(v, (LJ << 10) | 0x1F);
    else
        return __shfl_xor(v, LJ);
}

// Lanes that keep the larger key of their pair at stage (K, J) for key s.
template <int E, int K, int J>
constexpr unsigned long long larger_lanes(int s) {
    unsigned long long m = 0;
    for (int l = 0; l < kWave; ++l) {
        const bool asc = ((l * E + s) & K) == 0;
        const bool lower = (l & (J / E)) == 0;
        if (lower != asc) m |= 1ull << l;
    }
    return m;
}
// Lanes whose in-lane pair falls at level K.
template <int E, int K>
constexpr unsigned long long falling_lanes(int s) {
    unsigned long long m = 0;
    for (int l = 0; l < kWave; ++l)
        if (((l * E + s) & K) != 0) m |= 1ull << l;
    return m;
}

template <int E, int K, int J, typename X>
__device__ __forceinline__ void wave_sort_stage(X (&x)[E]) {
    if constexpr (J >= E) {
        X other[E];
#pragma unroll
        for (int s = 0; s < E; ++s) other[s] = static_cast<X>(wave_xor<J / E>(static_cast<int>(x[s])));
        static_for<0, E>([&](auto si) {
            constexpr int s = decltype(si)::value;
            constexpr unsigned long long kLarger = larger_lanes<E, K, J>(s);
            x[s] = (x[s] < other[s]) != in_mask(kLarger) ? x[s] : other[s];
        });
    } else {
        static_for<0, E>([&](auto si) {
            constexpr int s = decltype(si)::value;
            if constexpr ((s & J) == 0) {
                const X a = x[s], b = x[s + J];
                bool keep = a < b;
                if constexpr (K < E)  // the direction is the same for every lane
                    keep = keep != ((s & K) != 0);
                else
                    keep = keep != in_mask(falling_lanes<E, K>(s));
                x[s] = keep ? a : b;
                x[s + J] = keep ? b : a;
            }
        });
    }
}
template <int E, int K, int J, typename X>
__device__ __forceinline__ void wave_sort_level(X (&x)[E]) {
    if constexpr (J >= 1) {
        wave_sort_stage<E, K, J>(x);
        wave_sort_level<E, K, J / 2>(x);
    }
}
// The last level of a sort: ascending in every group (the level's direction
// bit lies above every index).
template <int E, int J, typename X>
__device__ __forceinline__ void wave_sort_last(X (&x)[E]) {
    wave_sort_level<E, 2 * kWave * E, J>(x);
}
// Every aligned group of L lanes sorts its L * E keys.
template <int E, int L = kWave, int K = 2, typename X = int>
__device__ __forceinline__ void wave_sort(X (&x)[E]) {
    if constexpr (K < L * E) {
        wave_sort_level<E, K, K / 2>(x);
        wave_sort<E, L, 2 * K>(x);
    } else if constexpr (K == L * E) {
        wave_sort_last<E, K / 2>(x);
    }
}

// The value of the lane below (lane 0: its own).
__device__ __forceinline__ unsigned lane_below(unsigned v) {
    return static_cast<unsigned>(__builtin_amdgcn_update_dpp(static_cast<int>(v), static_cast<int>(v), 0x138, 0xF, 0xF,
                                                             false));  // wave_shr:1
}

// Exclusive prefix sum over aligned groups of L lanes (8 <= L <= 64).
template <int L>
__device__ __forceinline__ int group_excl_sum(int v) {
    static_assert(L == 8 || L == 16 || L == 32 || L == 64, "bad group");
    int x = v;
    if constexpr (L == 8) {
        // row_shr:1 and :2 without the lanes that would read the group below
        const int a = __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, true);
        x += in_mask(0xFEFEFEFEFEFEFEFEull) ? a : 0;
        const int b = __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, true);
        x += in_mask(0xFCFCFCFCFCFCFCFCull) ? b : 0;
        x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xA, false);  // row_shr:4 into banks 1 and 3
    } else {
        x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, true);
        x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, true);
        x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, true);
        x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, true);
        if constexpr (L >= 32) x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);
        if constexpr (L >= 64) x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);
    }
    return x - v;
}

// An entry of A as the wave's lanes read it: a_ik and where its row of B
// lies (position of the row's first product, minus the entry's product
// offset in the chunk).
template <bool VALS>
struct WaveEntry;
template <>
struct alignas(16) WaveEntry<true> {
    double av;
    int d, pad;
};
template <>
struct WaveEntry<false> {
    int d;
};

constexpr int kWaveWords = 32;  // 64-bit words of the entry-start bitmap (a window of 2048 products)
constexpr int kWavePad = 8;     // zero words after it (a round may end past the window)

// Per-wave LDS of the product walk.
template <bool VALS>
struct alignas(16) WaveChunk {
    unsigned long long starts[kWaveWords + kWavePad];
    int before[kWaveWords + kWavePad];  // entries that start before each word (and before the window)
    WaveEntry<VALS> ent[kWave];
};

// LDS of a fused row of one wave: the hash table of T slots with a value
// beside every key, and the product walk's metadata, whose place the
// compacted columns take once the walk is over.  Values are summed in double
// whatever the operands' type (LdsSum).
template <int P, int T>
struct alignas(16) WaveRow {
    LdsSum vals[T];
    int keys[T];
    union {
        WaveChunk<true> walk;
        uint32_t words[P];
    };
};
constexpr int wave_row_bytes(int p, int t) {
    const int walk = static_cast<int>(sizeof(WaveChunk<true>));
    const int cols = 4 * p;
    return t * static_cast<int>(sizeof(LdsSum) + sizeof(int)) + (walk > cols ? walk : cols);
}
static_assert(sizeof(WaveRow<128, 256>) == wave_row_bytes(128, 256) &&
                  sizeof(WaveRow<512, 1024>) == wave_row_bytes(512, 1024),
              "LDS size of a wave's row");

// The same for a row that WAVES waves share: the compacted columns, then the
// table slots of the row's columns in ascending order.
template <int P, int T, int WAVES>
struct alignas(16) GroupRow {
    LdsSum vals[T];
    int keys[T];
    union {
        WaveChunk<true> walk[WAVES];
        struct {
            uint32_t words[P];
            unsigned short slots[P];
        };
    };
    int wave_sum[WAVES];
};
constexpr int group_row_bytes(int p, int t, int waves) {
    const int walk = waves * static_cast<int>(sizeof(WaveChunk<true>));
    const int sorted = 6 * p;
    const int all = t * static_cast<int>(sizeof(LdsSum) + sizeof(int)) + (walk > sorted ? walk : sorted) + 4 * waves;
    return (all + 15) / 16 * 16;
}
static_assert(sizeof(GroupRow<512, 1024, 4>) == group_row_bytes(512, 1024, 4) &&
                  sizeof(GroupRow<1024, 2048, 4>) == group_row_bytes(1024, 2048, 4),
              "LDS size of a workgroup's row");

// A row whose columns fill most of LDS: the table, then the sorted columns in
// its place.
template <int T, int WAVES>
struct alignas(16) LongRow {
    int keys[T];
    WaveChunk<true> walk[WAVES];
    int wave_sum[WAVES];
};
constexpr int long_row_bytes(int t, int waves) {
    const int all = 4 * t + waves * (static_cast<int>(sizeof(WaveChunk<true>)) + 4);
    return (all + 15) / 16 * 16;
}
static_assert(sizeof(LongRow<32768, 16>) == long_row_bytes(32768, 16), "LDS size of a long row");

// Where a wave's walk reads (all scalar).
template <typename V>
struct WaveOperands {
    const V SPG_GLOBAL* a_val;
    const long long SPG_GLOBAL* bref;
    const int32_t SPG_GLOBAL* b_col;
    const V SPG_GLOBAL* b_val;
    int wide;  // WideFlags
};

// The products of A's entries [a0, a1), in rounds of N * 64:
// f(key[N], prod[N], ok[N], far), ok[j] the lanes with a product j, far the
// constant WIDE (B has one of the WideFlags: 64-bit offsets and a 32-bit
// hash).  The wave takes 64 entries at a time, one to a
// lane; entries with an empty row of B drop out.  A product's entry is the
// number of entries that start at or before it (less one): the chunk's
// starts are marked in a bitmap, 64 products to a word and one position
// early, so that a lane counts the marks below its own bit (two mbcnt on
// top of the count before the word).  `first` and `step` let
// several waves share a row: this wave takes the rounds first, first + step,
// ... of the row, counted on over its windows and chunks, or, with `by_chunk`,
// every round of the chunks first, first + step, ... instead.  An f that
// returns false (the same on every lane) ends the walk.
template <typename V, int N, bool VALS, bool SHARED, bool WIDE, typename F>
__device__ __forceinline__ void wave_products_at(const WaveOperands<V>& W, int a0, int a1, WaveChunk<VALS>* wc, F&& f,
                                                 int first, int step, bool by_chunk) {
    static_assert(N <= kWavePad, "a round may pass the window by N - 1 words");
    const int lane = lane_id();
    const int round_step = by_chunk ? 1 : step;
    int r = by_chunk ? 0 : first;  // this wave's next round, from the window's first on
    for (int ebase = a0 + (by_chunk ? first * kWave : 0); ebase < a1; ebase += by_chunk ? step * kWave : kWave) {
        const int e = ebase + lane;
        long long ref = 0;
        V av = V(0);
        if (e < a1) {
            ref = W.bref[e];
            if constexpr (VALS) av = W.a_val[e];
        }
        const int len = bref_len(ref);
        const int incl = wave_incl_scan(len);
        const int total = wave_last(incl);
        const int start = incl - len;
        const unsigned long long filled = __ballot(len > 0);
        wave_sync();  // the previous chunk's reads are done
        if (len > 0) {
            WaveEntry<VALS> w;
            if constexpr (VALS) w.av = av;
            w.d = (bref_start(ref) - start) * (WIDE ? 1 : 4);  // narrow: in bytes of b_col, modulo 2^32
            wc->ent[rank_in(filled)] = w;
        }
        for (int win = 0; win < total; win += kWave * kWaveWords) {
            const int in_win = min(total - win, kWave * kWaveWords);
            const int n_rounds = (in_win + N * kWave - 1) / (N * kWave);
            if constexpr (SHARED) {
                if (r >= n_rounds) {  // the other waves' rounds
                    r -= n_rounds;
                    continue;
                }
            } else {
                r = 0;
            }
            wave_sync();  // the previous window's reads are done
            if (lane < kWaveWords + kWavePad) wc->starts[lane] = 0;
            wave_sync();
            const int mark = start - 1 - win;
            const bool marks = len > 0 && start > 0;
            if (marks && mark >= 0 && mark < kWave * kWaveWords)
                atomicOr(&wc->starts[mark >> 6], 1ull << (mark & 63));
            const int earlier = __popcll(__ballot(marks && mark < 0));
            wave_sync();
            if (lane < kWave) {
                const int c = lane < kWaveWords ? __popcll(wc->starts[lane]) : 0;
                const int up = wave_incl_scan(c);
                if (lane < kWaveWords + kWavePad) wc->before[lane] = earlier + up - c;
            }
            wave_sync();
            for (; r < n_rounds; r += round_step) {
                const int base = r * N * kWave;  // in the window
                int en[N];
#pragma unroll
                for (int j = 0; j < N; ++j) {
                    const unsigned long long w = wc->starts[r * N + j];
                    en[j] = static_cast<int>(__builtin_amdgcn_mbcnt_hi(
                        static_cast<unsigned>(w >> 32),
                        __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(w),
                                                  static_cast<unsigned>(wc->before[r * N + j]))));
                }
                unsigned long long ok[N];
                int key[N];
                V bv[N];
#pragma unroll
                for (int j = 0; j < N; ++j) {
                    // a lane past the last product reads B's first entry
                    const int p0 = base + j * kWave;
                    ok[j] = __ballot(lane < in_win - p0);
                    if constexpr (WIDE) {
                        const int pos = wc->ent[en[j]].d + lane + (win + p0);
                        const int at = in_mask(ok[j]) ? pos : 0;
                        key[j] = W.b_col[at];
                        if constexpr (VALS) bv[j] = W.b_val[at];
                    } else {
                        const uint32_t pos = static_cast<uint32_t>(wc->ent[en[j]].d) + static_cast<uint32_t>(lane * 4) +
                                             static_cast<uint32_t>((win + p0) * 4);
                        const uint32_t o = in_mask(ok[j]) ? pos : 0u;
                        key[j] = *(const int32_t SPG_GLOBAL*)((const char SPG_GLOBAL*)W.b_col + o);
                        if constexpr (VALS)
                            bv[j] = *(const V SPG_GLOBAL*)((const char SPG_GLOBAL*)W.b_val +
                                                           o * static_cast<uint32_t>(sizeof(V) / 4));
                    }
                }
                LdsSum prod[N];
                if constexpr (VALS) {
                    LdsSum a[N];
#pragma unroll
                    for (int j = 0; j < N; ++j) a[j] = wc->ent[en[j]].av;
#pragma unroll
                    for (int j = 0; j < N; ++j) prod[j] = a[j] * static_cast<LdsSum>(bv[j]);
                }
                constexpr std::bool_constant<WIDE> far{};
                if constexpr (std::is_same_v<decltype(f(key, prod, ok, far)), bool>) {
                    if (!f(key, prod, ok, far)) return;
                } else {
                    f(key, prod, ok, far);
                }
            }
            r -= n_rounds;
        }
    }
}

template <typename V, int N, bool VALS, bool SHARED, typename F>
__device__ __forceinline__ void wave_products_shared(const WaveOperands<V>& W, int a0, int a1, WaveChunk<VALS>* wc, F&& f,
                                                     int first, int step, bool by_chunk) {
    // Two copies of the walk: choosing the hash round by round cost the 96^3 stencil 5 %, a third copy for wide
    // columns at narrow offsets 1.6 %.
    if (W.wide)
        wave_products_at<V, N, VALS, SHARED, true>(W, a0, a1, wc, f, first, step, by_chunk);
    else
        wave_products_at<V, N, VALS, SHARED, false>(W, a0, a1, wc, f, first, step, by_chunk);
}
// A row of this wave alone.
template <typename V, int N, bool VALS, typename F>
__device__ __forceinline__ void wave_products(const WaveOperands<V>& W, int a0, int a1, WaveChunk<VALS>* wc, F&& f) {
    wave_products_shared<V, N, VALS, false>(W, a0, a1, wc, f, 0, 1, true);
}
// This wave's share of a row.
template <typename V, int N, bool VALS, typename F>
__device__ __forceinline__ void wave_products(const WaveOperands<V>& W, int a0, int a1, WaveChunk<VALS>* wc, F&& f,
                                              int first, int step, bool by_chunk) {
    wave_products_shared<V, N, VALS, true>(W, a0, a1, wc, f, first, step, by_chunk);
}

// How the waves of a workgroup share a row: by chunks of 64 entries, or by
// rounds, for which every wave reads every chunk.  Reading a chunk takes a
// wave about as long as two rounds of 256 products, so chunks are dealt where
// the busiest wave's share of them, with their rounds, is the shorter.
template <int WAVES>
__device__ __forceinline__ bool wave_by_chunk(int entries, int nip) {
    constexpr unsigned kRead = 2;  // rounds that take as long as reading a chunk
    // Four waves, of which a launch has many rows, do with less (the sum below took the count of 81-entry rows 1.5 %
    // longer): the two meet at four rounds a chunk with two chunks and about sixteen with four to seven, and the way
    // picked so is at most 1.43 times as long as the other (three chunks of five rounds).
    if constexpr (WAVES <= 4)
        return entries >= 2 * WAVES * kWave || (entries > kWave && nip >> (entries > 3 * kWave ? 6 : 4) <= entries);
    if (entries <= kWave) return false;
    if (entries >= 8 * WAVES * kWave) return true;
    const unsigned chunks = static_cast<unsigned>(entries + kWave - 1) / kWave;
    const unsigned share = (chunks + WAVES - 1) / WAVES;
    const unsigned rounds = static_cast<unsigned>(nip) / (4 * kWave) + chunks;
    // share * (kRead + rounds / chunks) < kRead * chunks + rounds / WAVES
    return rounds * (share * WAVES - chunks) < kRead * WAVES * chunks * (chunks - share);
}

}  // namespace spg
