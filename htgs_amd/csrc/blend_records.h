// What the training forward pass does with a finished pixel: the unclamped colour and the per-pixel records for the backward
// pass.  Shared by the kernels with one wave per tile, with several, and for very long lists.
#pragma once

#include "blend_long.h"

namespace htgs {

__device__ __forceinline__ float one_minus_alpha_rcp(float one_minus_alpha)
{
    return 1.0f / (one_minus_alpha > kOneMinusAlphaEps ? one_minus_alpha : kOneMinusAlphaEps);
}

// What the training pass does with a pixel's finished core and tail (HYBRID_BLEND): the unclamped colour and the records
// of R/include/hybrid_blend/kernels/forward.cuh:170-233.  Called once per pixel inside the image, by the kernel with one wave
// per tile and by the one for tiles with very long lists.  records: entries per record plane (64 per tile of the frame).
struct HybridRecords {
    float *image;
    uint32_t *core_idx;
    float4 *core_info;
    float *tail_info;
    uint32_t width, height;
    size_t records;
    template <int K>
    __device__ __forceinline__ void operator()(const float4 *__restrict__ prim, uint32_t tile, const TilePixel &px, float (&cd)[K], float (&c3)[K], float (&ci)[K],
                                               HybridTail &tail) const
    {
        constexpr int MODE = HTGS_MODE_HYBRID_BLEND;
        const uint32_t x = px.x, y = px.y;
        float tail0 = tail.c0, tail1 = tail.c1, tail2 = tail.c2;
        const float tail3 = tail.alpha, T_tail = tail.T;
        const size_t pix = (size_t)width * y + x, np = (size_t)width * height;
        const size_t rp = record_pixel(tile, x, y), rnp = records;
        float c0[K], c1[K], c2[K];
#pragma unroll
        for (int i = 0; i < K; ++i) {
            float4 c = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (c3[i] > 0.0f) c = prim[(size_t)float_to_bits(ci[i]) * (HTGS_PRIM_FLOATS_TRAIN / 4) + 4];
            c0[i] = c.x; c1[i] = c.y; c2[i] = c.z;
        }
#pragma unroll
        for (int i = 0; i < K; ++i) {
            tail0 = __builtin_fmaf(-c3[i], c0[i], tail0);
            tail1 = __builtin_fmaf(-c3[i], c1[i], tail1);
            tail2 = __builtin_fmaf(-c3[i], c2[i], tail2);
        }
        tail0 = clamp_pos(tail0); tail1 = clamp_pos(tail1); tail2 = clamp_pos(tail2);   // colours are >= 0, so is the exact difference
        float r = 0.0f, g = 0.0f, b = 0.0f, T_core = 1.0f;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            if (T_core >= kTransmittanceThreshold) {
                const float bw = T_core * c3[i];
                r = __builtin_fmaf(bw, c0[i], r);
                g = __builtin_fmaf(bw, c1[i], g);
                b = __builtin_fmaf(bw, c2[i], b);
                T_core *= 1.0f - c3[i];
                if (T_core < kTransmittanceThreshold) T_core = 0.0f;
            }
        }
        float w0 = 0.0f, w1 = 0.0f, w2 = 0.0f;
        float t0 = 0.0f, t1 = 0.0f, t2 = 0.0f, t3 = 0.0f, t4 = 0.0f, t5 = 0.0f;
        if (tail3 >= ModeCfg<MODE>::min_alpha) {
            const float asr = 1.0f / tail3;
            const float s = (T_core * (1.0f - T_tail)) * asr;
            w0 = s * tail0; w1 = s * tail1; w2 = s * tail2;
            t0 = tail0; t1 = tail1; t2 = tail2; t3 = asr; t4 = T_tail; t5 = T_core;
        }
        tail_info[rp] = t0; tail_info[rnp + rp] = t1; tail_info[2 * rnp + rp] = t2;
        tail_info[3 * rnp + rp] = t3; tail_info[4 * rnp + rp] = t4; tail_info[5 * rnp + rp] = t5;

        float n0 = 0.0f, n1 = 0.0f, n2 = 0.0f;
        T_core = 1.0f;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            const bool skip = !(c3[i] > 0.0f) || T_core < kTransmittanceThreshold;      // an empty slot has alpha 0
            __builtin_nontemporal_store(skip ? 0xffffffffu : float_to_bits(ci[i]), core_idx + ((size_t)i * rnp + rp));
            float4 info = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (!skip) {
                const float bw = T_core * c3[i];
                n0 = __builtin_fmaf(bw, c0[i], n0);
                n1 = __builtin_fmaf(bw, c1[i], n1);
                n2 = __builtin_fmaf(bw, c2[i], n2);
                const float oma = 1.0f - c3[i];
                const float omar = one_minus_alpha_rcp(oma);
                info.x = __builtin_fmaf(c0[i], T_core, -(((r - n0) + w0) * omar));
                info.y = __builtin_fmaf(c1[i], T_core, -(((g - n1) + w1) * omar));
                info.z = __builtin_fmaf(c2[i], T_core, -(((b - n2) + w2) * omar));
                info.w = bw;
                T_core *= oma;
            }
            // (0.7 GB of records per frame at 1080p, read back once by the backward pass: streaming stores)
            typedef float streamed_float4 __attribute__((ext_vector_type(4)));
            streamed_float4 packed; packed.x = info.x; packed.y = info.y; packed.z = info.z; packed.w = info.w;
            __builtin_nontemporal_store(packed, reinterpret_cast<streamed_float4 *>(core_info + ((size_t)i * rnp + rp)));
        }
        image[pix] = r + w0; image[np + pix] = g + w1; image[2 * np + pix] = b + w2;
    }
};

// ALPHA_BLEND_FIRST_K: R/include/alpha_blend_first_k/kernels/forward.cuh:160-213
struct FirstKRecords {
    float *image;
    uint32_t *core_idx;
    float4 *core_info;
    uint32_t width, height;
    size_t records;
    template <int K>
    __device__ __forceinline__ void operator()(const float4 *__restrict__ prim, uint32_t tile, const TilePixel &px, const float (&cd)[K], const float (&ca)[K],
                                               const uint32_t (&ci)[K]) const
    {
        const uint32_t x = px.x, y = px.y;
        const size_t pix = (size_t)width * y + x, np = (size_t)width * height;
        const size_t rp = record_pixel(tile, x, y), rnp = records;
        float r = 0.0f, g = 0.0f, b = 0.0f, T = 1.0f;
        float k0[K], k1[K], k2[K];
        bool open = true;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            open = open && T >= kTransmittanceThreshold && ci[i] != 0xffffffffu;
            k0[i] = k1[i] = k2[i] = 0.0f;
            if (open) {
                const float bw = T * ca[i];
                const float4 col = prim[(size_t)ci[i] * (HTGS_PRIM_FLOATS_TRAIN / 4) + 4];
                k0[i] = col.x; k1[i] = col.y; k2[i] = col.z;
                r = __builtin_fmaf(bw, col.x, r);
                g = __builtin_fmaf(bw, col.y, g);
                b = __builtin_fmaf(bw, col.z, b);
                T *= 1.0f - ca[i];
            }
        }
        float n0 = 0.0f, n1 = 0.0f, n2 = 0.0f;
        T = 1.0f;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            const bool skip = ci[i] == 0xffffffffu || T < kTransmittanceThreshold;
            __builtin_nontemporal_store(skip ? 0xffffffffu : ci[i], core_idx + ((size_t)i * rnp + rp));     // (streaming, as in HybridRecords)
            float4 info = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (!skip) {
                const float bw = T * ca[i];
                n0 = __builtin_fmaf(bw, k0[i], n0);
                n1 = __builtin_fmaf(bw, k1[i], n1);
                n2 = __builtin_fmaf(bw, k2[i], n2);
                const float oma = 1.0f - ca[i];
                const float omar = one_minus_alpha_rcp(oma);
                info.x = __builtin_fmaf(k0[i], T, -((r - n0) * omar));
                info.y = __builtin_fmaf(k1[i], T, -((g - n1) * omar));
                info.z = __builtin_fmaf(k2[i], T, -((b - n2) * omar));
                info.w = bw;
                T *= oma;
            }
            typedef float streamed_float4 __attribute__((ext_vector_type(4)));
            streamed_float4 packed; packed.x = info.x; packed.y = info.y; packed.z = info.z; packed.w = info.w;
            __builtin_nontemporal_store(packed, reinterpret_cast<streamed_float4 *>(core_info + ((size_t)i * rnp + rp)));
        }
        image[pix] = r; image[np + pix] = g; image[2 * np + pix] = b;
    }
};

// OIT_BLEND: R/include/oit_blend/kernels/forward.cuh:140-163
struct OitRecords {
    float *image, *tail_info;
    uint32_t width, height;
    size_t records;
    __device__ __forceinline__ void operator()(uint32_t tile, const TilePixel &px, const OitSums &sum) const
    {
        constexpr int MODE = HTGS_MODE_OIT_BLEND;
        const uint32_t x = px.x, y = px.y;
        const size_t pix = (size_t)width * y + x, np = (size_t)width * height;
        const size_t rp = record_pixel(tile, x, y), rnp = records;
        float r = 0.0f, g = 0.0f, b = 0.0f, t0 = 0.0f, t1 = 0.0f, t2 = 0.0f, t3 = 0.0f, t4 = 0.0f, t5 = 0.0f;
        if (sum.alpha >= ModeCfg<MODE>::min_alpha) {
            const float asr = 1.0f / sum.alpha;
            const float s = (1.0f - sum.T) * asr;
            r = s * sum.a0; g = s * sum.a1; b = s * sum.a2;
            t0 = sum.a0; t1 = sum.a1; t2 = sum.a2; t3 = asr; t4 = sum.T; t5 = 1.0f;   // row 5 plays the hybrid mode's T_core
        }
        tail_info[rp] = t0; tail_info[rnp + rp] = t1; tail_info[2 * rnp + rp] = t2;
        tail_info[3 * rnp + rp] = t3; tail_info[4 * rnp + rp] = t4; tail_info[5 * rnp + rp] = t5;
        image[pix] = r; image[np + pix] = g; image[2 * np + pix] = b;
    }
};

}  // namespace htgs
