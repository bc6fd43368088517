// How one launch of several GEMVs deals its blocks out to the calls, and what each wavefront takes.  Plain C++ (the kernel
// calls first_batch, which constexpr makes device code as well).
#pragma once
#include <cstdint>

namespace mi {

// Call i works on the blocks first[i] .. first[i + 1] - 1 (per row of x), waves[i] wavefronts in all, which take its
// nbatch[i] row batches in turn: wavefront w the batches w, w + waves[i], w + 2 waves[i], ...  Every wavefront gets about the
// same bytes, and all of them, of all M rows of x, are resident at once: the bytes per wavefront grow until the blocks fit
// (with that many blocks per row of x instead, 15 rows of a 576-wide Q4 layer took 19.7 us where they now take 17.0 and
// launches of a run each 18.7; 8 fp16 rows 14.1 against 8 and 17).  For several rows of x the launch has a multiple of 8
// blocks per row: the blocks that read the same weights for different rows then share an XCD's L2.  Returns the blocks
// per row of x, the blocks added for that multiple among them, which belong to no call.
inline long deal_blocks(int n, const int* nbatch, const int* batch_bytes, int M, long resident_waves, int waves_per_block,
                        uint16_t* first, int* waves) {
    double bytes = 0.0;
    for (int i = 0; i < n; ++i) bytes += static_cast<double>(nbatch[i]) * batch_bytes[i];
    const long cap = resident_waves / waves_per_block / M;
    for (double share = bytes * M / resident_waves;; share *= 1.05) {
        long blocks = 0;
        for (int i = 0; i < n; ++i) {
            const long per_wave = share > batch_bytes[i] ? static_cast<long>(share / batch_bytes[i]) : 1;
            const long b = ((nbatch[i] + per_wave - 1) / per_wave + waves_per_block - 1) / waves_per_block;
            first[i] = static_cast<uint16_t>(blocks);
            waves[i] = static_cast<int>(b * waves_per_block);
            blocks += b;
        }
        const long padded = M > 1 ? (blocks + 7) / 8 * 8 : blocks;
        if (padded <= cap || blocks <= n) return padded;
    }
}

// The first row batch of wavefront `wave` of block `block`, where the last call that starts at or before that block starts
// at `first` and has `waves` wavefronts.  -1: none, the block belongs to no call.
constexpr int first_batch(int block, int wave, int first, int waves, int waves_per_block) {
    const int w = (block - first) * waves_per_block + wave;
    return w < waves ? w : -1;
}

}  // namespace mi
