// tt_quant.hip -- 2-bit asymmetric quantisers and dequantisers (gfx950).
//
// Bit-exact restatements of the reference AVX2 kernels:
//   K: csrc/cpu/quantize_k_avx2.cpp:26-110   (per channel over the block's tokens)
//   V: csrc/cpu/quantize_v_avx2.cpp:44-108   (per token over the head's channels)
//   dequant: csrc/cpu/dequantize_avx2.cpp:24-110 and :138-204
// The semantics are exact: explicit operand order for min/max, codes as IEEE
// division and round-to-nearest-even give them, software F16C-equivalent
// rounding. They run once per 16 evictions, or in bulk at prefill.
#include "tt_quant_dev.h"
#include "tt_quant_grid.h"

namespace tt {

namespace {

constexpr int kMaxGridY = 65535;  // largest grid y extent

__device__ __forceinline__ float4 load_meta4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 load_meta4(const uint16_t* p) {
    const ushort4 v = *reinterpret_cast<const ushort4*>(p);
    return make_float4(f16_to_f32(v.x), f16_to_f32(v.y), f16_to_f32(v.z), f16_to_f32(v.w));
}
template <bool NT>
__device__ __forceinline__ void store4(float* p, const float4 v) {
    typedef float f4v __attribute__((ext_vector_type(4)));
    if constexpr (NT)
        __builtin_nontemporal_store(f4v{v.x, v.y, v.z, v.w}, reinterpret_cast<f4v*>(p));
    else
        *reinterpret_cast<float4*>(p) = v;
}
inline bool aligned(const void* p, const size_t n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; }

// One thread per (block, head, channel), flat over all blocks, so that short
// rows leave no lane idle. Channels below 8*floor(D/8) follow the 8-wide
// vector body of the reference (MINPS/MAXPS operand order), the rest follow
// its scalar tail (std::min/std::max). `K` and the outputs start at the
// launch's first block; the output block is b + *base_dev when base_dev is
// given (engine prefill).
//
// One f32 read per value is what bounds it: 134 MB in 23.4 us (5.7 TB/s; 25.8
// us with a grid row per block and a division per value). Two and four
// channels per thread (8- and 16-byte loads) took 24.2 and 26.3 us. Launches of
// at most a wave per SIMD divide every value (see quant_codes).
template <typename MetaT, bool FAST>
__global__ void __launch_bounds__(256) quantize_k_kernel(const float* __restrict__ K, uint32_t* __restrict__ packed,
                                                         MetaT* __restrict__ scale, MetaT* __restrict__ zero,
                                                         unsigned items, unsigned row, unsigned D, int kgs,
                                                         const int* __restrict__ base_dev) {
    const unsigned item = blockIdx.x * 256u + threadIdx.x;
    if (item >= items) return;
    const unsigned b = item / row, hc = item - b * row, c = hc % D;
    const size_t ob = static_cast<size_t>(b) + (base_dev ? *base_dev : 0);
    const size_t mi = ob * row + hc;
    quant_k_channel<MetaT, FAST>(K + static_cast<size_t>(b) * kgs * row + hc, row, kgs, c < (D / 8) * 8, scale + mi,
                           zero + mi, packed + ob * (kgs / 16) * row + hc, row);
}

// One lane per packed word of a (token, head) row: the row's D / 16 words
// on an aligned group of `group` lanes (a power of two, at most 64, so the
// group lies in one wave; lanes past D / 16 only pad the min/max tree), the
// loads of a row coalesced. D % 16 == 0 (checked by the host).
template <typename MetaT, bool FAST>
__global__ void __launch_bounds__(256) quantize_v_kernel(const float* __restrict__ V, int32_t* __restrict__ packed,
                                                         MetaT* __restrict__ scale, MetaT* __restrict__ zero,
                                                         int tokens, int H, int D, int group,
                                                         const int* __restrict__ base_dev, int tokens_per_block) {
    const int wpr = D / 16;
    const long long th = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    // whole groups leave together: the total is a multiple of the group size
    if (th >= static_cast<long long>(tokens) * H * group) return;
    const int r = static_cast<int>(th / group), w = static_cast<int>(th % group);
    const int t = r / H, h = r % H;
    const int ot = t + (base_dev ? (*base_dev) * tokens_per_block : 0);
    const size_t mi = static_cast<size_t>(ot) * H + h;
    quant_v_row_lanes<MetaT, FAST>(V + static_cast<size_t>(t) * H * D + static_cast<size_t>(h) * D, w, wpr, group,
                             scale + mi, zero + mi, packed + mi * wpr);
}

// Rows of more than 64 words (D > 1024): one thread per (token, head) row.
template <typename MetaT>
__global__ void __launch_bounds__(256) quantize_v_serial_kernel(const float* __restrict__ V,
                                                                int32_t* __restrict__ packed,
                                                                MetaT* __restrict__ scale, MetaT* __restrict__ zero,
                                                                int tokens, int H, int D) {
    const int wpr = D / 16;
    const long long r = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (r >= static_cast<long long>(tokens) * H) return;
    const size_t mi = static_cast<size_t>(r);
    quant_v_row_serial<MetaT>(V + mi * D, wpr, scale + mi, zero + mi, packed + mi * wpr);
}

// Dequantisers, x = fmaf((float)q, scale, zero). Both only write: 16 bytes of
// f32 for each packed byte, so what bounds them is the rate of the stores.
//
// K with four channels per thread: a wave stores 1 KB runs of a token's row
// (16 bytes per lane). Threads are laid flat over (block, channel quad), so
// short rows leave no lane idle. 268 MB: 47.9 us (5.6 TB/s) against 66 with
// one channel per thread, 20 MB in blocks of 32 5.2 against 6.2. Up to a wave
// per SIMD with one channel per thread that is the shorter chain (2 MB in
// blocks of 32 3.0 us against 3.1, 0.5 MB 2.7 against 2.9).
template <typename MetaT, bool NT>
__global__ void __launch_bounds__(256) dequantize_k4_kernel(const int32_t* __restrict__ packed,
                                                            const MetaT* __restrict__ scale,
                                                            const MetaT* __restrict__ zero, float* __restrict__ out,
                                                            unsigned row, unsigned items, int kgs) {
    const unsigned item = blockIdx.x * 256u + threadIdx.x;
    if (item >= items) return;
    const unsigned quads = row / 4;
    const unsigned b = item / quads, c = 4 * (item - b * quads);
    const size_t mi = static_cast<size_t>(b) * row + c;
    const float4 s = load_meta4(scale + mi), z = load_meta4(zero + mi);
    const int words = kgs / 16;
    auto put = [&](const int w, const int4 p) {
        float* o = out + (static_cast<size_t>(b) * words + w) * 16 * row + c;
#pragma unroll
        for (int st = 0; st < 16; ++st) {
            auto x = [&](const int v, const float sc, const float ze) {
                return __builtin_fmaf(static_cast<float>((static_cast<uint32_t>(v) >> (2 * st)) & 3u), sc, ze);
            };
            store4<NT>(o + static_cast<size_t>(st) * row,
                   make_float4(x(p.x, s.x, z.x), x(p.y, s.y, z.y), x(p.z, s.z, z.z), x(p.w, s.w, z.w)));
        }
    };
    const int32_t* src = packed + static_cast<size_t>(b) * words * row + c;
    if constexpr (NT) {
        for (int w = 0; w < words; ++w) put(w, *reinterpret_cast<const int4*>(src + static_cast<size_t>(w) * row));
    } else {
        // both words of a block of 32 before the first store (268 MB with it and non-temporal stores 2.5 us more)
        int4 p[2];
#pragma unroll
        for (int w = 0; w < 2; ++w)
            if (w < words) p[w] = *reinterpret_cast<const int4*>(src + static_cast<size_t>(w) * row);
#pragma unroll
        for (int w = 0; w < 2; ++w)
            if (w < words) put(w, p[w]);
    }
}

// V with four channels (one byte of a word) per thread and kDeqVPer such
// quads, 256 apart: a wave's store covers 1 KB of consecutive channels. 268 MB:
// 45.1 us (5.9 TB/s) against 85.7 with a word's 16 channels per thread, whose
// stores leave 64 bytes between lanes; four quads per thread 47.8. (row, rem)
// of a quad's word are stepped rather than divided anew.
template <typename MetaT, bool NT>
__global__ void __launch_bounds__(256) dequantize_v4_kernel(const int32_t* __restrict__ packed,
                                                            const MetaT* __restrict__ scale,
                                                            const MetaT* __restrict__ zero, float* __restrict__ out,
                                                            unsigned words, unsigned wpr) {
    // 64 words (256 quads) per workgroup and step
    const size_t w0 = static_cast<size_t>(blockIdx.x) * kDeqVWords + (threadIdx.x >> 2);
    const int sh = 8 * (threadIdx.x & 3);
    unsigned row = static_cast<unsigned>(w0) / wpr, rem = static_cast<unsigned>(w0) - row * wpr;
    const unsigned drow = 64 / wpr, drem = 64 - drow * wpr;
    uint32_t p[kDeqVPer];
    float s[kDeqVPer], z[kDeqVPer];
#pragma unroll
    for (int u = 0; u < kDeqVPer; ++u) {
        const size_t w = w0 + 64 * u;
        if (w < words) {
            p[u] = static_cast<uint32_t>(packed[w]) >> sh;
            s[u] = Meta<MetaT>::load(scale, row);
            z[u] = Meta<MetaT>::load(zero, row);
        }
        row += drow;
        rem += drem;
        if (rem >= wpr) {
            rem -= wpr;
            ++row;
        }
    }
#pragma unroll
    for (int u = 0; u < kDeqVPer; ++u) {
        const size_t w = w0 + 64 * u;
        if (w < words) {
            auto x = [&](const int i) {
                return __builtin_fmaf(static_cast<float>((p[u] >> (2 * i)) & 3u), s[u], z[u]);
            };
            store4<NT>(out + 16 * w + 4 * (threadIdx.x & 3), make_float4(x(0), x(1), x(2), x(3)));
        }
    }
}

// Outputs or tiers that are not aligned for the wide accesses (a caller's
// view at an odd offset, K rows that are no multiple of four channels), and
// small K launches: one thread per (block, head, channel) ...
template <typename MetaT>
__global__ void __launch_bounds__(256) dequantize_k_kernel(const int32_t* __restrict__ packed,
                                                           const MetaT* __restrict__ scale,
                                                           const MetaT* __restrict__ zero, float* __restrict__ out,
                                                           int H, int D, int kgs, int b_off) {
    const int row = H * D;
    const int hc = blockIdx.x * blockDim.x + threadIdx.x;
    if (hc >= row) return;
    const int b = b_off + static_cast<int>(blockIdx.y);
    const float s = Meta<MetaT>::load(scale, static_cast<size_t>(b) * row + hc);
    const float z = Meta<MetaT>::load(zero, static_cast<size_t>(b) * row + hc);
    const int words = kgs / 16;
    for (int w = 0; w < words; ++w) {
        const uint32_t p = static_cast<uint32_t>(packed[(static_cast<size_t>(b) * words + w) * row + hc]);
        for (int st = 0; st < 16; ++st) {
            const size_t tok = static_cast<size_t>(b) * kgs + w * 16 + st;
            out[tok * row + hc] = __builtin_fmaf(static_cast<float>((p >> (2 * st)) & 3u), s, z);
        }
    }
}

// ... and one per (token, head, 16-channel group).
template <typename MetaT>
__global__ void __launch_bounds__(256) dequantize_v_kernel(const int32_t* __restrict__ packed,
                                                           const MetaT* __restrict__ scale,
                                                           const MetaT* __restrict__ zero, float* __restrict__ out,
                                                           int tokens, int H, int D) {
    const int qhd = D / 16;
    const long long idx = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= static_cast<long long>(tokens) * H * qhd) return;
    const int g = static_cast<int>(idx % qhd);
    const long long th = idx / qhd;  // token * H + head
    const float s = Meta<MetaT>::load(scale, static_cast<size_t>(th));
    const float z = Meta<MetaT>::load(zero, static_cast<size_t>(th));
    const uint32_t p = static_cast<uint32_t>(packed[idx]);
    float* o = out + static_cast<size_t>(th) * D + g * 16;
#pragma unroll
    for (int i = 0; i < 16; ++i) o[i] = __builtin_fmaf(static_cast<float>((p >> (2 * i)) & 3u), s, z);
}

}  // namespace

int launch_quantize_k(const float* K, uint32_t* packed, void* scale, void* zero, int num_blocks, int H, int D,
                      int kgs, int meta_fp16, const int* base_dev, hipStream_t stream) {
    if (num_blocks <= 0 || H * D <= 0) return TT_OK;
    // slices of whole blocks that a 1-D launch can hold
    const unsigned row = static_cast<unsigned>(H * D);
    const int per = quant_k_slice(num_blocks, row);
    const int words = kgs / 16;
    for (int b0 = 0; b0 < num_blocks; b0 += per) {
        const int nb = std::min(per, num_blocks - b0);
        const unsigned items = static_cast<unsigned>(nb) * row;
        const dim3 grid((items + 255u) / 256u);
        const float* k = K + static_cast<size_t>(b0) * kgs * row;
        uint32_t* p = packed + static_cast<size_t>(b0) * words * row;
        const size_t m = static_cast<size_t>(b0) * row;
        const auto launch = [&](auto kernel, auto meta) {
            using MetaT = decltype(meta);
            hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, k, p, static_cast<MetaT*>(scale) + m,
                               static_cast<MetaT*>(zero) + m, items, row, static_cast<unsigned>(D), kgs, base_dev);
        };
        const bool fast = !quant_one_wave(items / words);
        if (meta_fp16)
            fast ? launch(quantize_k_kernel<uint16_t, true>, uint16_t{}) : launch(quantize_k_kernel<uint16_t, false>, uint16_t{});
        else
            fast ? launch(quantize_k_kernel<float, true>, float{}) : launch(quantize_k_kernel<float, false>, float{});
        TT_LAUNCH_CHECK();
    }
    return TT_OK;
}

int launch_quantize_v(const float* V, int32_t* packed, void* scale, void* zero, int tokens, int H, int D,
                      int meta_fp16, const int* base_dev, int tokens_per_block, hipStream_t stream) {
    if (tokens <= 0 || H <= 0) return TT_OK;
    const int group = quant_v_group(D / 16);
    if (group == 0) {
        if (base_dev) TT_FAIL(TT_ERR_INVALID_ARGUMENT, "quantize_v: head_dim above 1024 in the engine");
        const long long rows = static_cast<long long>(tokens) * H;
        if (rows > kMaxThreads) TT_FAIL(TT_ERR_INVALID_ARGUMENT, "quantize_v: tokens x heads too large for one call");
        const dim3 grid(static_cast<unsigned>((rows + 255) / 256));
        if (meta_fp16)
            hipLaunchKernelGGL(quantize_v_serial_kernel<uint16_t>, grid, dim3(256), 0, stream, V, packed,
                               static_cast<uint16_t*>(scale), static_cast<uint16_t*>(zero), tokens, H, D);
        else
            hipLaunchKernelGGL(quantize_v_serial_kernel<float>, grid, dim3(256), 0, stream, V, packed,
                               static_cast<float*>(scale), static_cast<float*>(zero), tokens, H, D);
        TT_LAUNCH_CHECK();
        return TT_OK;
    }
    const long long n = static_cast<long long>(tokens) * H * group;
    if (n > kMaxThreads) TT_FAIL(TT_ERR_INVALID_ARGUMENT, "quantize_v: tokens x heads too large for one call");
    const dim3 grid(static_cast<unsigned>((n + 255) / 256));
    const auto launch = [&](auto kernel, auto meta) {
        using MetaT = decltype(meta);
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, V, packed, static_cast<MetaT*>(scale),
                           static_cast<MetaT*>(zero), tokens, H, D, group, base_dev, tokens_per_block);
    };
    const bool fast = !quant_one_wave(n);
    if (meta_fp16)
        fast ? launch(quantize_v_kernel<uint16_t, true>, uint16_t{}) : launch(quantize_v_kernel<uint16_t, false>, uint16_t{});
    else
        fast ? launch(quantize_v_kernel<float, true>, float{}) : launch(quantize_v_kernel<float, false>, float{});
    TT_LAUNCH_CHECK();
    return TT_OK;
}

int launch_dequantize_k(const int32_t* packed, const void* scale, const void* zero, float* out, int num_blocks,
                        int H, int D, int kgs, int meta_fp16, hipStream_t stream) {
    if (num_blocks <= 0 || H * D <= 0) return TT_OK;
    const size_t meta4 = meta_fp16 ? 8 : 16;
    const long long items = static_cast<long long>(num_blocks) * (H * D / 4);
    if (H * D % 4 == 0 && !quant_one_wave(4 * items) && deq_k_wide_fits(items) && aligned(packed, 16) && aligned(out, 16) &&
        aligned(scale, meta4) && aligned(zero, meta4)) {
        const dim3 grid(static_cast<unsigned>((items + 255) / 256));
        const unsigned row = static_cast<unsigned>(H * D), n = static_cast<unsigned>(items);
        const auto launch = [&](auto kernel, auto meta) {
            using MetaT = decltype(meta);
            hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, packed, static_cast<const MetaT*>(scale),
                               static_cast<const MetaT*>(zero), out, row, n, kgs);
        };
        const bool nt = deq_k_streams(static_cast<long long>(num_blocks) * kgs * row, kgs, meta_fp16);
        if (meta_fp16)
            nt ? launch(dequantize_k4_kernel<uint16_t, true>, uint16_t{})
               : launch(dequantize_k4_kernel<uint16_t, false>, uint16_t{});
        else
            nt ? launch(dequantize_k4_kernel<float, true>, float{}) : launch(dequantize_k4_kernel<float, false>, float{});
        TT_LAUNCH_CHECK();
        return TT_OK;
    }
    for (int b0 = 0; b0 < num_blocks; b0 += kMaxGridY) {
        const dim3 grid((H * D + 255) / 256, std::min(kMaxGridY, num_blocks - b0));
        if (meta_fp16)
            hipLaunchKernelGGL(dequantize_k_kernel<uint16_t>, grid, dim3(256), 0, stream, packed,
                               static_cast<const uint16_t*>(scale), static_cast<const uint16_t*>(zero), out, H, D,
                               kgs, b0);
        else
            hipLaunchKernelGGL(dequantize_k_kernel<float>, grid, dim3(256), 0, stream, packed,
                               static_cast<const float*>(scale), static_cast<const float*>(zero), out, H, D, kgs, b0);
        TT_LAUNCH_CHECK();
    }
    return TT_OK;
}

int launch_dequantize_v(const int32_t* packed, const void* scale, const void* zero, float* out, int tokens, int H,
                        int D, int meta_fp16, hipStream_t stream) {
    const long long n = static_cast<long long>(tokens) * H * (D / 16);
    if (n <= 0) return TT_OK;
    if (n > kMaxThreads) TT_FAIL(TT_ERR_INVALID_ARGUMENT, "dequantize_v: tokens x heads too large for one call");
    // (from 2^31 words on, 137 GB of output, the wide kernel's threads are too many for a dispatch)
    if (aligned(out, 16) && deq_v_wide_fits(n)) {
        const dim3 grid(static_cast<unsigned>(deq_v_wide_groups(n)));
        const unsigned words = static_cast<unsigned>(n), wpr = static_cast<unsigned>(D / 16);
        const auto launch = [&](auto kernel, auto meta) {
            using MetaT = decltype(meta);
            hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, packed, static_cast<const MetaT*>(scale),
                               static_cast<const MetaT*>(zero), out, words, wpr);
        };
        const bool nt = deq_v_streams(16 * n, D, meta_fp16);
        if (meta_fp16)
            nt ? launch(dequantize_v4_kernel<uint16_t, true>, uint16_t{})
               : launch(dequantize_v4_kernel<uint16_t, false>, uint16_t{});
        else
            nt ? launch(dequantize_v4_kernel<float, true>, float{}) : launch(dequantize_v4_kernel<float, false>, float{});
        TT_LAUNCH_CHECK();
        return TT_OK;
    }
    const dim3 grid(static_cast<unsigned>((n + 255) / 256));
    if (meta_fp16)
        hipLaunchKernelGGL(dequantize_v_kernel<uint16_t>, grid, dim3(256), 0, stream, packed,
                           static_cast<const uint16_t*>(scale), static_cast<const uint16_t*>(zero), out, tokens, H, D);
    else
        hipLaunchKernelGGL(dequantize_v_kernel<float>, grid, dim3(256), 0, stream, packed,
                           static_cast<const float*>(scale), static_cast<const float*>(zero), out, tokens, H, D);
    TT_LAUNCH_CHECK();
    return TT_OK;
}

}  // namespace tt
