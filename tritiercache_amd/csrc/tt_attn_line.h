// tt_attn_line.h -- which contexts of head_dim 128 and 64 the VALU attention
// kernel takes from the matrix cores; host arithmetic only.
#pragma once

namespace tt {

// Query heads per workgroup of a group of G: the next power of two, at most 8.
inline int gp_for(const int G) { return G > 4 ? 8 : (G > 2 ? 4 : G); }

// Workgroups per slot: head chunks of all KV heads.
inline long long head_chunks(const int Hq, const int Hkv) {
    const int G = Hq / Hkv;
    return static_cast<long long>(Hkv) * ((G + gp_for(G) - 1) / gp_for(G));
}

// Whether the matrix-core kernel serves a shape at all (head_dim 64: two KV heads as one of 128 channels).
inline bool use_matrix_cores(const int D, const int Hkv) { return D == 128 || (D == 64 && Hkv % 2 == 0); }

// Units (16-token tiles of either kind) per KV head up to which the VALU kernel
// serves the head dims of the matrix-core kernel too. At short contexts a
// launch is one chain of latencies, and the VALU kernel's is shorter: no
// lay-out in LDS, no coefficients, a unit per wave. Its arithmetic grows with
// units x query heads x channels, so the line is a number of units x heads per
// CU for each group size and head dim, below the point where the matrix cores
// win with blocks of 32 tokens. It was measured with the waves per SIMD that
// the resource test of this kernel asks for (another register count moves the
// times, not the line). Partials per launch, VALU against matrix cores, at
// units x heads per CU:
//   one head per group of 128 (line at 35): 32/32 heads at 2k (16) 6.7 against
//     8.9 us, at 4k (32) 9.9 against 11.9, at 5k (39) 10.2 against 10.8, at
//     6k (47) 12.5 against 12.0;
//   two (16): 16/8 heads at 4k (8) 5.7 against 7.9, at 8k (16) 7.6 against 7.9;
//   four (4.5): 32/8 heads at 580 (1.2) 5.5 against 5.9, at 2k (3.9) 5.9 against
//     7.0, at 2.3k (4.5) 7.0 against 7.0, at 3k (5.9) 7.3 against 7.2;
//   more (0): 28/4 heads at 1k (1) 7.3 against 6.0;
//   head_dim 64: one (28): 64/64 heads at 1.5k (24) 6.9 against 8.2, at 2k (32)
//     7.9 against 8.6, at 2.6k (41) 9.8 against 9.6;
//   two (20): 32/16 heads at 5k (20) 7.2 against 8.5, at 6k (24) 7.8 against 8.4;
//   four (16): 32/8 heads at 6k (12) 6.9 against 7.5, at 8k (16) 8.0 against 8.0;
//   more (1.5): 14/2 heads at 3k (1.5) 6.2 against 6.4, at 4k (2) 6.2 against 7.5.
// (The lines of 64 channels with one, two and eight heads leave room above:
// contexts up to a third longer would still gain.)
inline long long short_units(const int Hq, const int Hkv, const int D, const int cus) {
    const int gp = gp_for(Hq / Hkv);
    const int halves = D == 64 ? (gp == 1 ? 56 : gp == 2 ? 40 : gp == 4 ? 32 : 3)
                               : (gp == 1 ? 70 : gp == 2 ? 32 : gp == 4 ? 9 : 0);
    return static_cast<long long>(cus) * halves / (2 * head_chunks(Hq, Hkv));
}

// Whether the VALU kernel runs a context.
inline bool use_valu(const int dense, const int blocks, const int Hq, const int Hkv, const int D, const int kgs,
                     const int cus) {
    const long long units = (static_cast<long long>(dense) + 15) / 16 + static_cast<long long>(blocks) * (kgs / 16);
    return !use_matrix_cores(D, Hkv) || units <= short_units(Hq, Hkv, D, cus);
}

}  // namespace tt
