// tt_quant_grid.h -- launch sizes and choice of stores of the quantisers and
// dequantisers, host arithmetic only. A dispatch counts its work-items in 32
// bits, so every launch's grid times 256 threads stays within kMaxThreads.
#pragma once

#include <algorithm>

namespace tt {

constexpr long long kMaxThreads = 0xFFFFFF00LL;  // whole workgroups of 256

// Blocks per quantize_k launch, a thread per (block, channel) of `row` channels.
inline int quant_k_slice(const int num_blocks, const long long row) {
    return static_cast<int>(std::min<long long>(num_blocks, kMaxThreads / row));
}

// Launches of at most a wave per SIMD (256 CUs of four; K in blocks of 32, whose
// lanes hold twice the values: two) are over with their slowest wave: there the
// quantisers divide every value (K in blocks of 16, 2 MB, 3.4 us against 3.6 with
// the reciprocal codes, 5 MB 4.0 against 3.7; in blocks of 32, 2 MB 4.6 against
// 5.8, 10 MB 5.8 against 6.3, 20 MB 7.1 against 6.8; V, 2 MB 3.6 against 3.7, 5 MB
// 4.0 against 3.8).
inline bool quant_one_wave(const long long threads) { return threads <= 4 * 256 * 64; }

// The wide K dequantiser holds four channels per thread.
inline bool deq_k_wide_fits(const long long quads) { return quads <= kMaxThreads; }

// The wide V dequantiser holds kDeqVPer channel quads per thread, 256 apart:
// 64 kDeqVPer words of 16 channels per workgroup, four threads to a word of
// each step, so twice as many threads as words.
constexpr int kDeqVPer = 2;
constexpr long long kDeqVWords = 64 * kDeqVPer;
inline long long deq_v_wide_groups(const long long words) { return (words + kDeqVWords - 1) / kDeqVWords; }
inline bool deq_v_wide_fits(const long long words) { return 256 * deq_v_wide_groups(words) <= kMaxThreads; }

// Outputs go out as non-temporal stores where they and the tiers together
// exceed the last-level cache (256 MiB), and stay cached for their reader
// below. Over six shapes at outputs of 208 to 320 MB the two cross there for V
// (per launch, plain against non-temporal, tiers and output in MiB: 242 36.9
// against 39.8 us, 259 46.3 against 42.2, 276 64.3 against 45.6) and for K with
// f32 metadata (252 39.4 against 43.2, 261 47.8 against 43.9, 288 56.0 against
// 48.1), and at 261 to 300 for K with f16 metadata (262 43.3 against 45.8, 280 48.3
// against 48.2, 298 56.2 against 51.7; head_dim 128 in blocks of 16: 288 53.0
// against 54.5, 306 58.1 against 57.5).
inline long long deq_bytes(const long long values, const int per_meta, const int meta_fp16) {
    return 4 * values + values / 4 + 2 * (meta_fp16 ? 2 : 4) * (values / per_meta);
}
inline bool deq_k_streams(const long long values, const int kgs, const int meta_fp16) {
    return deq_bytes(values, kgs, meta_fp16) > ((meta_fp16 ? 280LL : 256LL) << 20);
}
inline bool deq_v_streams(const long long values, const int D, const int meta_fp16) {
    return deq_bytes(values, D, meta_fp16) > (256LL << 20);
}

}  // namespace tt
