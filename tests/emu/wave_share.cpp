// How the waves of a workgroup share a row's products (spg_wave.hpp), on the
// CPU: for the two ways of sharing and the one that wave_by_chunk picks, one
// line "way: rounds of each wave : fewest and most waves that took a product".
//
//     wave_share <4 or 16 waves> <entries of the row> <products per entry>
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <vector>

#include "spg_wave.hpp"

namespace spg {

constexpr int kN = 4;  // slots of a round, as in the kernels

template <int WAVES>
void k_share(const long long* bref, const int32_t* b_col, int entries, bool by_chunk, int* rounds, int* hits) {
    __shared__ WaveChunk<false> walk[WAVES];
    const int wave = uniform(static_cast<int>(threadIdx.x) / kWave);
    const WaveOperands<double> W{nullptr, bref, b_col, nullptr, 0};
    wave_products<double, kN, false>(
        W, 0, entries, &walk[wave],
        [&](const int(&key)[kN], const LdsSum(&)[kN], const unsigned long long(&ok)[kN], auto) {
            if (lane_id() == 0) ++rounds[wave];
            for (int j = 0; j < kN; ++j)
                if (in_mask(ok[j])) atomicAdd(&hits[key[j]], 1);
        },
        wave, WAVES, by_chunk);
}

template <int WAVES>
void share(const char* how, int entries, int b_row, bool by_chunk) {
    std::vector<long long> bref(entries);
    std::vector<int32_t> b_col(entries * b_row);
    for (int e = 0; e < entries; ++e) bref[e] = pack_bref(e * b_row, b_row);
    for (size_t i = 0; i < b_col.size(); ++i) b_col[i] = static_cast<int32_t>(i);
    std::vector<int> rounds(WAVES, 0), hits(b_col.size(), 0);
    const long long* refs = bref.data();
    const int32_t* cols = b_col.data();
    int *r_out = rounds.data(), *h_out = hits.data();
    hipLaunchKernelGGL(k_share<WAVES>, 1, WAVES * kWave, 0, hipStreamPerThread, refs, cols, entries, by_chunk, r_out,
                       h_out);
    (void)hipDeviceSynchronize();
    std::printf("%s:", how);
    for (int n : rounds) std::printf(" %d", n);
    std::printf(" : %d %d\n", *std::min_element(hits.begin(), hits.end()), *std::max_element(hits.begin(), hits.end()));
}

template <int WAVES>
void all(int entries, int b_row) {
    share<WAVES>("rounds", entries, b_row, false);
    share<WAVES>("chunks", entries, b_row, true);
    share<WAVES>("rule", entries, b_row, wave_by_chunk<WAVES>(entries, entries * b_row));
}

}  // namespace spg

int main(int argc, char** argv) {
    if (argc != 4) return 2;
    const int entries = std::atoi(argv[2]), b_row = std::atoi(argv[3]);
    if (std::atoi(argv[1]) == 4)
        spg::all<4>(entries, b_row);
    else
        spg::all<16>(entries, b_row);
    return 0;
}
