// ntc_bc_source.h - how the block-compression kernels read their source image.
#ifndef NTC_BC_SOURCE_H
#define NTC_BC_SOURCE_H
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "ntc_decode_kernel.h"

namespace ntc_hip_dev {

typedef uint32_t __attribute__((aligned(1))) u32_unaligned;
typedef uint32_t u32x2_unaligned __attribute__((ext_vector_type(2), aligned(1)));

// fminf / fmaxf as single instructions.  The compiler brackets the library functions with two
// canonicalising instructions (it cannot know that its operands are already quiet); v_min_f32 /
// v_max_f32 themselves return the other operand when one is a NaN, which is all fminf / fmaxf promise.
__device__ __forceinline__ float min_f32(float a, float b) { float r; asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b)); return r; }
__device__ __forceinline__ float max_f32(float a, float b) { float r; asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b)); return r; }

__device__ __forceinline__ float min3_f32(float a, float b, float c) { float r; asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c)); return r; }
__device__ __forceinline__ float max3_f32(float a, float b, float c) { float r; asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c)); return r; }

// k / d for an integer k in [0, d], d = 255 or 65535, r = 1 / d rounded: one Newton step on k * r gives the
// correctly rounded quotient for every such k (all 256 + 65536 cases are checked in the tests with exact
// rational arithmetic) at a third of the instructions of a division.
__device__ __forceinline__ float unorm_quotient(float k, float d, float r)
{
    float const q = k * r;
    return __builtin_fmaf(__builtin_fmaf(-q, d, k), r, q);
}

// Channel c of the pixel at (x, y) of the source image, as a texture load gives it: outside the image
// everything reads as 0; channels the image does not have read as 0, alpha as 1.  A stored -0 becomes
// +0 (the "+ 0.f"): minima and maxima of +0 and -0 depend on the operand order otherwise.
__device__ __forceinline__ float source_channel(BlockCompressArgs const& a, int x, int y, int c)
{
    if (x < 0 || y < 0 || x >= a.srcWidth || y >= a.srcHeight) return 0.f;
    if (c >= a.numChannels) return c == 3 ? 1.f : 0.f;
    uint8_t const* px = a.src + size_t(y) * a.rowPitch + size_t(x) * a.pixelStride;
    switch (a.format) {
    case NTC_HIP_DEV_FORMAT_UNORM8:  return unorm_quotient(float(px[c]), 255.f, 1.f / 255.f);
    case NTC_HIP_DEV_FORMAT_UNORM16: return unorm_quotient(float(reinterpret_cast<uint16_t const*>(px)[c]), 65535.f, 1.f / 65535.f);
    case NTC_HIP_DEV_FORMAT_FLOAT16: return float(reinterpret_cast<_Float16 const*>(px)[c]) + 0.f;
    case NTC_HIP_DEV_FORMAT_FLOAT32: return reinterpret_cast<float const*>(px)[c] + 0.f;
    default:                         return float(reinterpret_cast<uint32_t const*>(px)[c]);
    }
}

// All four channels of a pixel.  The common source, four UNORM8 channels with every pixel on a 4-byte
// boundary (args.packedRgba8, set by the host), takes one 32-bit load per pixel.
__device__ __forceinline__ void source_packed_pixel(BlockCompressArgs const& a, int x, int y, float (&rgba)[4])
{
    uint32_t v = 0;
    if (x >= 0 && y >= 0 && x < a.srcWidth && y < a.srcHeight)
        v = *reinterpret_cast<uint32_t const*>(a.src + size_t(y) * a.rowPitch + size_t(x) * a.pixelStride);
#pragma unroll
    for (int c = 0; c < 4; ++c) rgba[c] = unorm_quotient(float((v >> (8 * c)) & 0xffu), 255.f, 1.f / 255.f);
}
__device__ __forceinline__ void source_pixel(BlockCompressArgs const& a, int x, int y, float (&rgba)[4])
{
    if (a.packedRgba8) {
        source_packed_pixel(a, x, y, rgba);
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) rgba[c] = source_channel(a, x, y, c);
    }
}

// Channels first ... first + CHANNELS - 1 of four pixels from (x, y) on and of those below them, ROWS rows, as source_channel()
// gives them: x, y >= 0.  All loads are under way before the first value is made, 16 bytes each where pixels are dwords side
// by side; pixels outside the image are read inside it.  (A branch by format or alignment around each load is a wait for each:
// sixteen trips to memory one after the other, 16 thousand cycles of the 45 thousand that a wave spent on 64 given BC7 blocks.)
typedef uint32_t u32x4_dwords __attribute__((ext_vector_type(4), aligned(4)));
template <int CHANNELS, int ROWS>
__device__ __forceinline__ void source_rows(BlockCompressArgs const& a, int x, int y, int first, float (&values)[ROWS][4][CHANNELS])
{
    auto const row = [&](int r) { return a.src + size_t(min(y + r, a.srcHeight - 1)) * a.rowPitch; };
    if (a.packedRgba8 && a.pixelStride == 4u && a.srcWidth >= 4) {   // uniform
        u32x4_dwords words[ROWS];
        int const start = min(x, a.srcWidth - 4);
#pragma unroll
        for (int r = 0; r < ROWS; ++r) words[r] = *reinterpret_cast<u32x4_dwords const*>(row(r) + size_t(start) * 4u);
        if (x != start) {                                    // the right edge
#pragma unroll
            for (int r = 0; r < ROWS; ++r)
#pragma unroll
                for (int i = 0; i < 4; ++i) words[r][i] = *reinterpret_cast<uint32_t const*>(row(r) + size_t(min(x + i, a.srcWidth - 1)) * 4u);
#pragma unroll
            for (int r = 0; r < ROWS; ++r) asm volatile("" : "+v"(words[r]));            // (waited for here)
        }
#pragma unroll
        for (int r = 0; r < ROWS; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int c = 0; c < CHANNELS; ++c) values[r][i][c] = unorm_quotient(float((words[r][i] >> (8 * (first + c))) & 0xffu), 255.f, 1.f / 255.f);
    } else {
        auto const load = [&](auto zero, auto convert) {
            using T = decltype(zero);
            T stored[ROWS][4][CHANNELS];
#pragma unroll
            for (int r = 0; r < ROWS; ++r)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int c = 0; c < CHANNELS; ++c)
                        stored[r][i][c] = reinterpret_cast<T const*>(row(r) + size_t(min(x + i, a.srcWidth - 1)) * a.pixelStride)[min(first + c, a.numChannels - 1)];
#pragma unroll
            for (int r = 0; r < ROWS; ++r)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int c = 0; c < CHANNELS; ++c) values[r][i][c] = convert(stored[r][i][c]);
        };
        switch (a.format) {                                  // uniform
        case NTC_HIP_DEV_FORMAT_UNORM8:  load(uint8_t{}, [](uint8_t v) { return unorm_quotient(float(v), 255.f, 1.f / 255.f); }); break;
        case NTC_HIP_DEV_FORMAT_UNORM16: load(uint16_t{}, [](uint16_t v) { return unorm_quotient(float(v), 65535.f, 1.f / 65535.f); }); break;
        case NTC_HIP_DEV_FORMAT_FLOAT16: load(_Float16{}, [](_Float16 v) { return float(v) + 0.f; }); break;
        case NTC_HIP_DEV_FORMAT_FLOAT32: load(float{}, [](float v) { return v + 0.f; }); break;
        default:                         load(uint32_t{}, [](uint32_t v) { return float(v); }); break;
        }
        if (first + CHANNELS > a.numChannels) {              // uniform
#pragma unroll
            for (int r = 0; r < ROWS; ++r)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int c = 0; c < CHANNELS; ++c) if (first + c >= a.numChannels) values[r][i][c] = first + c == 3 ? 1.f : 0.f;
        }
    }
    if (x + 4 > a.srcWidth || y + ROWS > a.srcHeight) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int c = 0; c < CHANNELS; ++c) if (x + i >= a.srcWidth || y + r >= a.srcHeight) values[r][i][c] = 0.f;
    }
}

} // namespace ntc_hip_dev
#endif
