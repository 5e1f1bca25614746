// tt_quant_grid.h -- launch sizes of the quantisers and dequantisers, host
// arithmetic only. A dispatch counts its work-items in 32 bits, so every
// launch's grid times 256 threads stays within kMaxThreads.
#pragma once

#include <algorithm>

namespace tt {

constexpr long long kMaxThreads = 0xFFFFFF00LL;  // whole workgroups of 256

// Blocks per quantize_k launch, a thread per (block, channel) of `row` channels.
inline int quant_k_slice(const int num_blocks, const long long row) {
    return static_cast<int>(std::min<long long>(num_blocks, kMaxThreads / row));
}

// The wide K dequantiser holds four channels per thread.
inline bool deq_k_wide_fits(const long long quads) { return quads <= kMaxThreads; }

// The wide V dequantiser holds kDeqVPer channel quads per thread, 256 apart:
// 64 kDeqVPer words of 16 channels per workgroup, four threads to a word of
// each step, so twice as many threads as words.
constexpr int kDeqVPer = 2;
constexpr long long kDeqVWords = 64 * kDeqVPer;
inline long long deq_v_wide_groups(const long long words) { return (words + kDeqVWords - 1) / kDeqVWords; }
inline bool deq_v_wide_fits(const long long words) { return 256 * deq_v_wide_groups(words) <= kMaxThreads; }

}  // namespace tt
