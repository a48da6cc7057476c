// ntc_copy_kernel.hip - internal fp16 texture layout <-> user pitch-linear image, image loss (gfx950).
//
// The 1:1 branch of the reference's CopyImageKernel as ITextureSet::ReadChannels / WriteChannels
// use it (src/ImageProcessing.cu:86-164,220-265, src/TextureSet.cpp:835-985): no resize; colour
// space decode/encode and dithering as the reference defines them.  Pixels of at most eight bytes go four to a lane
// (read_groups_kernel, write_groups_kernel), larger ones one to a lane; the planar layout is read and written as half2
// pairs, coalesced across x.  2 bytes read and 1-4 bytes written per channel: bound by memory where colours are linear,
// by the draws and the rounding where 8-bit codes are dithered.  Then the copies between images of different sizes, the
// image loss and the image difference.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <atomic>
#include <type_traits>
#include "ntc_decode_kernel.h"
#include "ntc_launch.h"

namespace ntc_hip_dev {

typedef float    v2f __attribute__((ext_vector_type(2)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

// u(clamp(roundf(p), 0, top)) of WriteImageChannel (src/ImageProcessing.cu:141-152) for the UNORM formats.
// roundf rounds halves away from zero; for |p| < 2^23 it equals trunc(p + copysign(c, p)) with c the
// largest float below 1/2 (the sum rounds up to the next integer exactly when the fraction is at
// least 1/2), and negative p end at 0 either way, so: max with 0, add c, cap, truncating conversion.
__device__ __forceinline__ uint32_t unorm_code(float p, float top)
{
    return uint32_t(fminf(fmaxf(p, 0.f) + 0.49999997f, top));
}

// unorm_code(p, 255) as byte `at` of a word: the conversion that packs it saturates at both ends, in three instructions for
// five (equal for every float: tests).
__device__ __forceinline__ uint32_t put_unorm8(float p, uint32_t at, uint32_t word)
{
    return __builtin_amdgcn_cvt_pk_u8_f32(__builtin_floorf(p + 0.49999997f), at, word);
}

// Transfer functions, src/CudaUtils.h:61-114 (sRGB, Hybrid Log-Gamma) and src/ImageProcessing.cu:86-111.
// The transcendental parts are the device math library's, so results agree with a CPU
// evaluation to a few units in the last place, not bit for bit.
__device__ __forceinline__ float decode_color_space(int colorSpace, float v)
{
    if (colorSpace == 1) return (v <= 0.04045f) ? v / 12.92f : powf((v + 0.055f) / 1.055f, 2.4f);
    if (colorSpace == 2) {
        float const sign = (v < 0.f) ? -1.f : 1.f;
        float const h = fabsf(v);
        return (h < 0.5f) ? 4.f * h * h * sign : (expf((h - 0.55991073f) / 0.17883277f) + 0.28466892f) * sign;
    }
    return v;
}
__device__ __forceinline__ float encode_color_space(int colorSpace, float v)
{
    if (colorSpace == 1) return (v <= 0.0031308f) ? v * 12.92f : 1.055f * powf(v, 1.0f / 2.4f) - 0.055f;
    if (colorSpace == 2) {
        float const sign = (v < 0.f) ? -1.f : 1.f;
        float const e = fabsf(v);
        return (e < 1.f) ? 0.5f * sqrtf(e) * sign : (0.17883277f * logf(e - 0.28466892f) + 0.55991073f) * sign;
    }
    return v;
}

// ---- the transfer functions of stored values, by table -----------------------------------------------
//
// What the copies convert is a half (the internal layout, FLOAT16 images) or a UNORM code: a function of 16 bits, so
// encode(dst, decode(src, value)) is tabulated for the eight pairs of colour spaces that change a value, by the
// device functions above (same bits), once per device when its first context is created.  A powf costs some seventy
// vector instructions, sRGB to sRGB takes two of them and two divisions per channel: 2048 x 2048 sRGB pixels of 8
// bits, dithered, took 103 us to read that way and 91 us to write.
//
// With the tables (and the groups of four pixels below) they take 19 and 11 us.
//
// The floats of the halves in [1/64, 1], which is nearly everything a texture holds, are copied into LDS by launches
// large enough to pay for it; other halves are read from the table in memory (256 KB a pair, cached).
constexpr int kTransferPairs = 8;                            // src * 3 + dst - 1; linear to linear has no table
constexpr uint32_t kStageFirst = 0x2400u, kStageCount = 0x1801u;     // halves 1/64 .. 1
constexpr uint32_t kStageStride = kStageCount + 3u;          // of the copies in LDS, whole vectors
constexpr uint32_t kStagingThreads = 1024;
static __device__ float transferOfHalf[kTransferPairs][65536];
static __device__ uint16_t storedOfUnorm16[kTransferPairs][65536];   // UNORM16 code -> half of the internal layout
static __device__ uint16_t storedOfUnorm8[kTransferPairs + 1][256];  // UNORM8 code -> half; [8]: linear

__device__ __forceinline__ uint16_t stored_half(float v)     // WriteImageChannel FLOAT16, src/ImageProcessing.cu:154-156
{
    v = fmaxf(-65504.f, fminf(65504.f, v));
    asm volatile("" : "+v"(v));
    return __builtin_bit_cast(uint16_t, (_Float16)v);
}

__device__ __forceinline__ uint16_t unit_half(float v)       // of a v in [0, 1]
{
    asm volatile("" : "+v"(v));                              // (a multiply-add that rounds to a half rounds once)
    return __builtin_bit_cast(uint16_t, (_Float16)v);
}

// stored_half(encode_color_space(space, v)) for a value computed in fp32, most of the time without the math library: the
// hardware's log2, exp2 and square root are good to 2^-21 of what encode_color_space makes of v (over every v of the
// ranges below), so where y - e and y + e, e = 2^-20, round to the same half, that is the answer.  The few lanes in
// doubt (one in five hundred), and values outside the ranges, take the exact function.  `space` is uniform.
__device__ __forceinline__ uint32_t encoded_half(int space, float v)
{
    if (space == 0) return stored_half(v);
    constexpr float kError = 0x1p-20f;
    float y, e;
    bool certain;
    if (space == 1) {
        y = 1.055f * __builtin_amdgcn_exp2f(__builtin_amdgcn_logf(v) * (1.0f / 2.4f)) - 0.055f;
        e = __builtin_fmaf(y, kError, 0.055f * kError);
        certain = v > 0.0031308f && v <= 1.f;
    } else {
        y = 0.5f * __builtin_amdgcn_sqrtf(v);
        e = y * kError;
        certain = v >= 0x1p-100f && v < 1.f;
    }
    v2h const around = __builtin_convertvector(v2f{ y - e, y + e }, v2h);
    uint32_t const bits = __builtin_bit_cast(uint32_t, around), half = bits & 0xffffu;
    if (!certain || half != bits >> 16) return stored_half(encode_color_space(space, v));
    return half;
}

__global__ void __launch_bounds__(256)
transfer_tables_kernel()
{
    int const pair = blockIdx.y, src = pair == kTransferPairs ? 0 : (pair + 1) / 3, dst = pair == kTransferPairs ? 0 : (pair + 1) % 3;
    uint32_t const i = blockIdx.x * 256u + threadIdx.x;      // 65536 values
    auto transfer = [&](float v) { return encode_color_space(dst, decode_color_space(src, v)); };
    if (pair < kTransferPairs) {
        transferOfHalf[pair][i] = transfer(float(__builtin_bit_cast(_Float16, uint16_t(i))));
        storedOfUnorm16[pair][i] = stored_half(transfer(float(i) / 65535.f));
    }
    if (i < 256u) storedOfUnorm8[pair][i] = stored_half(transfer(float(i) / 255.f));
}

hipError_t launch_transfer_tables(hipStream_t stream)
{
    hipLaunchKernelGGL(transfer_tables_kernel, dim3(256, kTransferPairs + 1), dim3(256), 0, stream);
    return hipGetLastError();
}

__host__ __device__ __forceinline__ int transfer_pair(int src, int dst) { return src * 3 + dst - 1; }     // -1: linear to linear

// encode(dst, decode(src, half)) for a channel of the pair of colour spaces `pair` (uniform).
__device__ __forceinline__ float transfer_half(int pair, uint32_t bits)
{
    return pair < 0 ? float(__builtin_bit_cast(_Float16, uint16_t(bits))) : transferOfHalf[pair][bits];
}
// The same for four pixels' halves of one channel through the copies in LDS: slot 1 or 2 (uniform) names the copy that
// holds the pair, 0 none.  (The look-up in LDS happens for every half, out-of-range ones clamped: a choice between the
// two tables per half would become a choice of address and a flat load.  Look-ups in memory are waited for where they
// are made, or every path would wait there for all loads in flight, the next pixels' among them.)
__device__ __forceinline__ void transfer_halves(float const* staged, int slot, int pair, uint32_t const (&bits)[4], float (&value)[4])
{
    if (pair < 0) {                                          // uniform
#pragma unroll
        for (int k = 0; k < 4; ++k) value[k] = float(__builtin_bit_cast(_Float16, uint16_t(bits[k])));
    } else if (slot == 0) {
#pragma unroll
        for (int k = 0; k < 4; ++k) value[k] = transferOfHalf[pair][bits[k]];
#pragma unroll
        for (int k = 0; k < 4; ++k) asm volatile("" : "+v"(value[k]));
    } else {
        float const* const copy = staged + (slot - 1) * int(kStageStride);
        uint32_t at[4];
        bool beyond = false;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            at[k] = bits[k] - kStageFirst;
            value[k] = copy[min(at[k], kStageCount - 1u)];
            beyond |= at[k] >= kStageCount;
        }
        if (beyond) {
#pragma unroll
            for (int k = 0; k < 4; ++k) if (at[k] >= kStageCount) value[k] = transferOfHalf[pair][bits[k]];
#pragma unroll
            for (int k = 0; k < 4; ++k) asm volatile("" : "+v"(value[k]));
        }
    }
}
// a / b for b = 255 or 65535 and every a that occurs here (codes, dither draws): the product with the reciprocal as the sum
// of two floats, rounded once, is the correctly rounded quotient for all of them (checked exhaustively).
__device__ __forceinline__ float divide_by_top(float a, float top, float reciprocal)
{
    return __builtin_fmaf(a, reciprocal, a * float(1.0 / double(top) - double(reciprocal)));
}

// HashBasedRNG, src/CudaUtils.h:117-184: Jenkins hash of the pixel index seeds a Murmur3 round per draw.  The round turns
// the exclusive or of the seed and the draw's word by 13 bits; here each is turned by itself, the seed once for all draws.
// And an instruction of three operands takes the place of one with a shifted one, which shares no issue slot (2048 x 2048
// RGBA of 8 bits, dithered, 18.7 -> 18.3 us).
__device__ __forceinline__ constexpr uint32_t turned_left(uint32_t v, int bits) { return v << bits | v >> (32 - bits); }
struct DitherRng {
    uint32_t seed, index;                                    // the seed turned by 13 bits
    __device__ DitherRng() {}
    __device__ explicit DitherRng(uint32_t linearIndex) : index(0)
    {
        uint32_t a = linearIndex;
        a = (a + 0x7ed55d16u) + (a << 12);
        a = (a ^ 0xc761c23cu) ^ (a >> 19);
        a = (a + 0x165667b1u) + (a << 5);
        a = (a + 0xd3a2646cu) ^ (a << 9);
        a = (a + 0xfd7046c5u) + (a << 3);
        a = (a ^ 0xb55a4f09u) ^ (a >> 16);
        seed = turned_left(a, 13);
    }
    __device__ float next_offset()                           // a draw of [0, 1) less one half (both differences are exact)
    {
        return offset(index++);
    }
    __device__ float offset(uint32_t draw) const             // that of one draw, counted from 0
    {
        uint32_t const k = turned_left(turned_left((draw + 1u) * 0xcc9e2d51u, 15) * 0x1b873593u, 13);
        uint32_t h = (seed ^ k) * 5u + 0xe6546b64u;
        h = __builtin_amdgcn_bitop3_b32(h, h >> 16, 4u, 0x96);               // h ^= 4, h ^= h >> 16
        h *= 0x85ebca6bu;
        h ^= h >> 13; h *= 0xc2b2ae35u;
        h ^= h >> 16;
        return __builtin_bit_cast(float, (h & 0x7fffffu) | 0x3f800000u) - 1.5f;
    }
};

constexpr int bytes_per_channel(int format)
{
    return format == NTC_HIP_DEV_FORMAT_UNORM8 ? 1 : (format == NTC_HIP_DEV_FORMAT_UNORM16 || format == NTC_HIP_DEV_FORMAT_FLOAT16) ? 2 : 4;
}

// Lane -> pixel of the copy kernels: a workgroup covers 256 pixels of one row, or 64 pixels of four
// rows for images narrower than 256 (xShift = 8 or 6, chosen on the host).
struct CopyGrid {
    int x, y;
    __device__ explicit CopyGrid(int xShift)
        : x((int(blockIdx.x) << xShift) + (int(threadIdx.x) & ((1 << xShift) - 1))),
          y(int(blockIdx.y) * (256 >> xShift) + (int(threadIdx.x) >> xShift)) {}
};
inline dim3 copy_grid(int width, int height, int& xShift, bool wide = true)
{
    xShift = (wide && width >= 256) ? 8 : 6;
    int const rows = 256 >> xShift;
    return dim3((width + (1 << xShift) - 1) >> xShift, (height + rows - 1) / rows);
}

// WriteImageChannel (src/ImageProcessing.cu:141-164): the bits, in the destination format, of a channel whose
// value is in the destination's colour space already.
template <int FORMAT>
__device__ __forceinline__ uint32_t encode_value(float value, bool dithering, float dither)
{
    if constexpr (FORMAT == NTC_HIP_DEV_FORMAT_UNORM8) {
        if (dithering) value += divide_by_top(dither, 255.f, 1.f / 255.f);
        return unorm_code(value * 255.f, 255.f);
    } else if constexpr (FORMAT == NTC_HIP_DEV_FORMAT_UNORM16) {
        if (dithering) value += divide_by_top(dither, 65535.f, 1.f / 65535.f);
        return unorm_code(value * 65535.f, 65535.f);
    } else if constexpr (FORMAT == NTC_HIP_DEV_FORMAT_FLOAT16) {
        return stored_half(value);
    } else if constexpr (FORMAT == NTC_HIP_DEV_FORMAT_FLOAT32) {
        return __builtin_bit_cast(uint32_t, value);
    } else {
        return uint32_t(fmaxf(value, 0.f));
    }
}
template <int FORMAT>
__device__ __forceinline__ uint32_t encode_channel(int colorSpace, float value, bool dithering, float dither)
{
    return encode_value<FORMAT>(encode_color_space(colorSpace, value), dithering, dither);
}

// One lane per pixel.  All the half2 pairs the pixel needs are loaded before any arithmetic (the
// loads of a lane overlap; issued one by one behind their uses the kernel ran at half the rate),
// coalesced across the lanes of a row.  The pixel is produced 16 bytes at a time (16 / 8 / 4
// channels for 1 / 2 / 4-byte formats) and stored with the widest access the image's alignment allows
// (a.vectorBytes, decided on the host from base, pitch and stride).  PLAIN = every colour space
// linear and no dithering: the transfer functions and the generator are compiled out.
template <int FORMAT, bool PLAIN>
__global__ void __launch_bounds__(256)
read_channels_kernel(ReadChannelsArgs a)
{
    constexpr int BPC = bytes_per_channel(FORMAT), PER = 16 / BPC;
    CopyGrid const at(a.xShift);
    int const x = at.x, y = at.y;
    if (x >= a.width || y >= a.height) return;
    // GetPixelBaseAddress / GetChannelAddress, src/RegressionKernels.h:36-45
    uint16_t const* src = a.planarPairs + size_t(y) * size_t(a.width) * size_t(a.setChannels) + size_t(x) * 2;
    uint8_t* px = a.dst + size_t(y) * a.rowPitch + size_t(x) * a.pixelStride;
    int const firstPair = a.firstChannel >> 1;
    bool const odd = (a.firstChannel & 1) != 0;
    int const pairs = ((a.firstChannel + a.numChannels + 1) >> 1) - firstPair;     // at most 8
    uint32_t pr[NTC_HIP_DEV_MAX_CHANNELS / 2];
#pragma unroll
    for (int p = 0; p < NTC_HIP_DEV_MAX_CHANNELS / 2; ++p) {
        pr[p] = 0u;
        if (p < pairs) pr[p] = *reinterpret_cast<uint32_t const*>(src + size_t(2 * (firstPair + p)) * size_t(a.width));     // uniform
    }
    auto half_of = [&](int k) -> uint32_t {                  // half k of the loaded pairs, k a compile-time constant after unrolling
        return k < NTC_HIP_DEV_MAX_CHANNELS ? ((k & 1) ? pr[(k >> 1) & 7] >> 16 : pr[(k >> 1) & 7] & 0xffffu) : 0u;
    };
    [[maybe_unused]] DitherRng rng(uint32_t(x) + uint32_t(y) * uint32_t(a.width));
#pragma unroll
    for (int piece = 0; piece < NTC_HIP_DEV_MAX_CHANNELS / PER; ++piece) {
        int const base = piece * PER;
        if (base >= a.dstChannels) break;                    // uniform
        uint32_t words[4] = { 0u, 0u, 0u, 0u };
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            int const ch = base + k;
            if (ch >= a.dstChannels) continue;               // uniform
            float value;
            if (ch < a.numChannels) {
                uint32_t const bits = odd ? half_of(ch + 1) : half_of(ch);
                value = transfer_half(PLAIN ? -1 : transfer_pair(a.srcColorSpaces[ch], a.dstColorSpaces[ch]), bits);
            } else {
                value = (ch == 3) ? 1.f : 0.f;               // GetDefaultChannelValue, src/ImageProcessing.cu:166-170
                if constexpr (!PLAIN) value = encode_color_space(a.dstColorSpaces[ch], value);
            }
            uint32_t bits;
            if constexpr (PLAIN) {
                bits = encode_value<FORMAT>(value, false, 0.f);
            } else {
                float const dither = a.useDithering ? rng.next_offset() : 0.f;  // one draw per destination channel
                bits = encode_value<FORMAT>(value, a.useDithering != 0, dither);
            }
            words[(k * BPC) >> 2] |= bits << (8 * ((k * BPC) & 3));
        }
        int const bytes = min(PER, a.dstChannels - base) * BPC;
        uint8_t* const out = px + base * BPC;
        if (bytes == 16 && a.vectorBytes >= 16) {
            *reinterpret_cast<uint4*>(out) = make_uint4(words[0], words[1], words[2], words[3]);
        } else if ((bytes & 7) == 0 && a.vectorBytes >= 8) {
            for (int q = 0; q < bytes / 8; ++q) reinterpret_cast<uint2*>(out)[q] = make_uint2(words[2 * q], words[2 * q + 1]);
        } else if ((bytes & 3) == 0 && a.vectorBytes >= 4) {
            for (int q = 0; q < bytes / 4; ++q) reinterpret_cast<uint32_t*>(out)[q] = words[q];
        } else if constexpr (BPC == 1) {
            for (int q = 0; q < bytes; ++q) out[q] = uint8_t(words[q >> 2] >> (8 * (q & 3)));
        } else if constexpr (BPC == 2) {
            for (int q = 0; q < bytes / 2; ++q) reinterpret_cast<uint16_t*>(out)[q] = uint16_t(words[q >> 1] >> (16 * (q & 1)));
        } else {
            for (int q = 0; q < bytes / 4; ++q) reinterpret_cast<uint32_t*>(out)[q] = words[q];
        }
    }
    // Destination channels beyond the sixteen a set can hold (a pixel stride of more than 16 components): the
    // default value 0 in every format and colour space, dithered or not (|noise| < 1/2 step rounds to 0).
    int const tailBegin = NTC_HIP_DEV_MAX_CHANNELS * BPC, tailEnd = a.dstChannels * BPC;      // bytes; uniform
    if (tailEnd > tailBegin) {
        if (((tailEnd - tailBegin) & 3) == 0 && a.vectorBytes >= 4) {
            for (int b = tailBegin; b < tailEnd; b += 4) *reinterpret_cast<uint32_t*>(px + b) = 0u;
        } else if constexpr (BPC == 2) {
            for (int b = tailBegin; b < tailEnd; b += 2) *reinterpret_cast<uint16_t*>(px + b) = uint16_t(0);
        } else {
            for (int b = tailBegin; b < tailEnd; ++b) px[b] = uint8_t(0);
        }
    }
}

// ---- small pixels: four at a time ---------------------------------------------------------------------
//
// Images of at most eight bytes a pixel: a lane takes four adjacent pixels, so that it reads 16 bytes of each channel
// pair and writes its pixels as whole dwords.  (One pixel a lane, the kernel above, moved 5 bytes per lane for a
// single-channel 8-bit image and took 16.5 us for 2048 x 2048 of it, five times what its bytes take.)  The lanes of a
// wave cover 64, 32, 16 or 8 such groups of a row, whatever is the least that covers the row.  Accesses are whole
// vectors at whatever alignment the image has; the last group of a row that is no multiple of four goes pixel by pixel.
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(1)));
typedef uint32_t u32x2_any __attribute__((ext_vector_type(2), aligned(1)));
typedef uint32_t u32_any   __attribute__((aligned(1)));
typedef uint32_t u32x2_a4  __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t u32x4_a4  __attribute__((ext_vector_type(4), aligned(4)));

// Which pixels a lane works on: tiles of lanesX groups by threads / lanesX rows, a workgroup takes tiles
// blockIdx.x, blockIdx.x + step, ...
// (perRow: 2^40 / tilesX rounded up, 0 where a product with a tile's number could be inexact or too large.)
struct GroupGrid {
    int32_t tilesX, tiles, step;
    uint16_t log2LanesX, log2Rows;
    uint64_t perRow;
    __device__ __forceinline__ int row_of(int tile) const { return perRow ? int((uint32_t(tile) * perRow) >> 40) : tile / tilesX; }
};

int compute_units_of_current_device()
{
    static std::atomic<int> units[64];
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return 256;
    int n = units[device & 63].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || n < 1) n = 256;
        units[device & 63].store(n, std::memory_order_relaxed);
    }
    return n;
}

static GroupGrid group_grid(int width, int height, int threads)
{
    GroupGrid g;
    int const groups = (width + 3) / 4;
    g.log2LanesX = uint16_t(groups > 32 ? 6 : groups > 16 ? 5 : groups > 8 ? 4 : 3);
    int const rows = threads >> g.log2LanesX;
    g.log2Rows = uint16_t(__builtin_ctz(unsigned(rows)));
    g.tilesX = (groups + (1 << g.log2LanesX) - 1) >> g.log2LanesX;
    g.tiles = g.tilesX * ((height + rows - 1) / rows);
    g.step = g.tiles;
    g.perRow = g.tiles < 1 << 23 && g.tilesX < 1 << 16 ? ((uint64_t(1) << 40) + unsigned(g.tilesX) - 1u) / unsigned(g.tilesX) : 0u;
    return g;
}

// The pairs of colour spaces of a launch's channels, and the tables that it copies into LDS: the first two that they use.
// (In words: bytes of a kernel's arguments can be vector loads, and those indexed by a loop's variable always are.)
struct Transfers {
    uint32_t pairs = 0;                                      // four bits a channel: its pair + 1 (0: linear)
    uint32_t rest = 0;                                       // two bits a channel: the copy that holds it (0 none); from bit 16 on the number of copies and their pairs
    void set(int channel, int pair, int copy) { pairs |= uint32_t(pair + 1) << (4 * channel); rest |= uint32_t(copy) << (2 * channel); }
    int copy_of(int pair) const
    {
        for (int k = 0; k < count(); ++k) if (staged(k) == pair) return k + 1;
        return 0;
    }
    int stage(int pair)                                      // the copy that holds it, a new one while there are less than two
    {
        int const n = count();
        if (int const k = copy_of(pair)) return k;
        if (n == 2) return 0;
        rest += 1u << 16;
        rest |= uint32_t(pair) << (20 + 4 * n);
        return n + 1;
    }
    __host__ __device__ __forceinline__ int pair(int channel) const { return int((pairs >> (4 * channel)) & 15u) - 1; }
    __host__ __device__ __forceinline__ int slot(int channel) const { return int((rest >> (2 * channel)) & 3u); }
    __host__ __device__ __forceinline__ int count() const { return int((rest >> 16) & 3u); }
    __host__ __device__ __forceinline__ int staged(int k) const { return int((rest >> (20 + 4 * k)) & 15u); }
};

// Launch shape of the group kernels.  Images of two million pixels and more stage: workgroups of 1024 threads, two to
// a compute unit, that share a copy among two tiles or more each (2048 x 2048 read as dithered sRGB: 22.9 us, 24.4 with
// 512 threads, 28 with 256, 24.8 straight from the table in memory; HLG to linear halves: 19.6, 23.4, 22.6, 24.5; before
// the copies' loads were made at once and the next tile's pixels loaded ahead: 18.6 and 14.3 now).
// Smaller images, and those of linear channels, take small workgroups.  Either way no more than are resident: a workgroup
// loads its next tile's pixels before it works on one's, and its first tile's before it fills its tables.
struct GroupLaunch {
    GroupGrid grid;
    Transfers transfers;
    unsigned threads, ldsBytes;
};

static GroupLaunch plan_groups(int width, int height, uint8_t const* src, uint8_t const* dst, int channels, bool readsHalves)
{
    constexpr int kSmallThreads = 256, kTilesPerStaging = 2;
    GroupLaunch l{};
    Transfers& s = l.transfers;
    int const units = compute_units_of_current_device();
    l.grid = group_grid(width, height, int(kStagingThreads));
    bool const stage = readsHalves && l.grid.tiles >= kTilesPerStaging * units;
    for (int c = 0; c < channels; ++c) {
        int const pair = transfer_pair(src[c], dst[c]);
        s.set(c, pair, pair >= 0 && stage ? s.stage(pair) : 0);
    }
    if (s.count()) {
        int const share = (l.grid.tiles + kTilesPerStaging - 1) / kTilesPerStaging;
        l.threads = kStagingThreads;
        l.grid.step = 2 * units < share ? 2 * units : share;
        l.ldsBytes = unsigned(s.count() * kStageStride * sizeof(float));
    } else {
        l.grid = group_grid(width, height, kSmallThreads);
        l.threads = kSmallThreads;
        int const resident = 8 * units;                      // then a workgroup's next pixels are under way while it works
        if (l.grid.step > resident) l.grid.step = resident;
    }
    return l;
}

// Copies them: workgroups of kStagingThreads, 16 bytes a load and all loads in flight before the first is stored.  (A loop of
// dword loads, each waited for before the next, was a chain of six or twelve trips to the L2 in front of every launch's
// pixels: 2048 x 2048, sRGB dithered 19.6 us, HLG halves written 15.5, the 2 : 1 reduction 34.)
__device__ __forceinline__ void copy_staged(Transfers const& s, float* lds)
{
    if (s.count() == 0) return;
    constexpr uint32_t VECTORS = kStageCount / 4, STEPS = (VECTORS + kStagingThreads - 1) / kStagingThreads;
    static_assert(kStageCount == 4 * VECTORS + 1, "the table's end is 1");
    float4 v[2][STEPS];
    float last[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {                            // (one table twice if there is one)
        float const* const from = &transferOfHalf[k < s.count() ? s.staged(k) : s.staged(0)][kStageFirst];
#pragma unroll
        for (uint32_t i = 0; i < STEPS; ++i) v[k][i] = reinterpret_cast<float4 const*>(from)[min(threadIdx.x + i * kStagingThreads, VECTORS - 1u)];
        last[k] = from[kStageCount - 1u];
    }
    // (here, or each is loaded where it is stored)
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        asm volatile("" : "+v"(last[k]));
#pragma unroll
        for (uint32_t i = 0; i < STEPS; ++i) asm volatile("" : "+v"(v[k][i].x), "+v"(v[k][i].y), "+v"(v[k][i].z), "+v"(v[k][i].w));
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        if (k >= s.count()) continue;
        float* const to = lds + k * int(kStageStride);
#pragma unroll
        for (uint32_t i = 0; i < STEPS; ++i)
            if (uint32_t const at = threadIdx.x + i * kStagingThreads; at < VECTORS) reinterpret_cast<float4*>(to)[at] = v[k][i];
        if (threadIdx.x == 0) to[kStageCount - 1u] = last[k];
    }
    __syncthreads();
}

// What the kernels need of a ReadChannelsArgs or WriteChannelsArgs, in as few bytes as launches are quick with.
struct GroupsArgs {
    uint16_t* planar;
    uint8_t* image;
    uint64_t rowPitch;
    int32_t width, height;
    GroupGrid grid;
    Transfers transfers;
    uint8_t setChannels, firstChannel, channels;             // channels: copied ones
    uint8_t fillSpace;                                       // read: the destination's colour space of a fourth channel the set does not have
    uint32_t verticalFlip;                                   // write
};
static_assert(sizeof(GroupsArgs) <= 128, "");

// Where a lane works in a tile: the first of its four pixels.
struct GroupPlace {
    GroupGrid const& grid;
    int lx, ly;
    __device__ __forceinline__ explicit GroupPlace(GroupsArgs const& a)
        : grid(a.grid), lx(int(threadIdx.x) & ((1 << a.grid.log2LanesX) - 1)), ly(int(threadIdx.x) >> a.grid.log2LanesX) {}
    __device__ __forceinline__ void of_tile(int tile, int& x, int& y) const
    {
        int const tileY = grid.row_of(tile), tileX = tile - tileY * grid.tilesX;
        x = ((tileX << grid.log2LanesX) + lx) * 4; y = (tileY << grid.log2Rows) + ly;
    }
};

// CHANNELS = channels of a destination pixel.
template <int FORMAT, int CHANNELS, bool DITHER>
__global__ void __launch_bounds__(1024, 8)
read_groups_kernel(GroupsArgs a)
{
    constexpr int BPC = bytes_per_channel(FORMAT), PIXEL = CHANNELS * BPC, PAIRS = CHANNELS / 2 + 1;
    static_assert(PIXEL <= 8, "the words of four pixels stay in registers");
    extern __shared__ float staged[];
    GroupPlace const place(a);
    int const firstPair = a.firstChannel >> 1;
    bool const odd = (a.firstChannel & 1) != 0;
    int const copied = min(int(a.channels), CHANNELS);
    int const pairs = ((a.firstChannel + copied + 1) >> 1) - firstPair;      // at most PAIRS
    auto const pair_at = [&](int x, int y, int p) {
        return reinterpret_cast<uint32_t const*>(a.planar + size_t(y) * size_t(a.width) * size_t(a.setChannels) + size_t(2 * (firstPair + min(p, pairs - 1))) * size_t(a.width) + size_t(x) * 2);
    };
    // (four pixels of the row wherever the lane's group lies; a group that the row cuts off is read again)
    u32x4_a4 ahead[PAIRS];
    auto const load = [&](int tile) {
        int x, y;
        place.of_tile(tile, x, y);
        if (a.width < 4) return;                             // uniform
#pragma unroll
        for (int p = 0; p < PAIRS; ++p) ahead[p] = *reinterpret_cast<u32x4_a4 const*>(pair_at(min(x, a.width - 4), min(y, a.height - 1), p));
    };
    load(blockIdx.x);
    copy_staged(a.transfers, staged);
    for (int tile = blockIdx.x; tile < a.grid.tiles; tile += a.grid.step) {
        uint32_t pr[PAIRS][4];
#pragma unroll
        for (int p = 0; p < PAIRS; ++p)
#pragma unroll
            for (int k = 0; k < 4; ++k) pr[p][k] = ahead[p][k];
        if (tile + a.grid.step < a.grid.tiles) load(tile + a.grid.step);     // uniform
        int x, y;
        place.of_tile(tile, x, y);
        if (x >= a.width || y >= a.height) continue;
        // (what the channels' bits say is found out here again: kept from before the loop it is thirty spilled registers)
        Transfers transfers = a.transfers;
        asm volatile("" : "+s"(transfers.pairs), "+s"(transfers.rest));
        bool const whole = x + 4 <= a.width;
        if (!whole) {
#pragma unroll
            for (int p = 0; p < PAIRS; ++p)
#pragma unroll
                for (int k = 0; k < 4; ++k) pr[p][k] = pair_at(x, y, p)[min(k, a.width - 1 - x)];
#pragma unroll
            for (int p = 0; p < PAIRS; ++p)
#pragma unroll
                for (int k = 0; k < 4; ++k) asm volatile("" : "+v"(pr[p][k]));           // (waited for here)
        }
        uint32_t words[PIXEL];                               // four pixels
#pragma unroll
        for (int w = 0; w < PIXEL; ++w) words[w] = 0u;
        uint32_t const index = uint32_t(x) + uint32_t(y) * uint32_t(a.width);
        [[maybe_unused]] DitherRng rng[4];                   // one draw per pixel and destination channel, in channel order
        if constexpr (DITHER) {
#pragma unroll
            for (int k = 0; k < 4; ++k) rng[k] = DitherRng(index + uint32_t(k));
        }
        // (all look-ups before the first use of one: small images wait for their latency)
        float values[CHANNELS][4];
#pragma unroll
        for (int ch = 0; ch < CHANNELS; ++ch) {
            float (&value)[4] = values[ch];
            if (ch < copied) {                               // uniform
                uint32_t bits[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    uint32_t const even = (ch & 1) ? pr[ch >> 1][k] >> 16 : pr[ch >> 1][k] & 0xffffu;
                    uint32_t const next = (ch & 1) ? pr[(ch >> 1) + 1][k] & 0xffffu : pr[ch >> 1][k] >> 16;
                    bits[k] = odd ? next : even;
                }
                transfer_halves(staged, transfers.slot(ch), transfers.pair(ch), bits, value);
            } else {                                         // GetDefaultChannelValue; 0 is 0 in every colour space
                float const fill = (ch == 3) ? transfer_half(transfer_pair(0, a.fillSpace), 0x3C00u) : 0.f;
#pragma unroll
                for (int k = 0; k < 4; ++k) value[k] = fill;
            }
        }
#pragma unroll
        for (int ch = 0; ch < CHANNELS; ++ch) {
            // A filled channel whose code is the same for the least and the greatest draw has it for all between them, and
            // its draws, of which each is a seventh of a pixel's work, need not be made.
            if (DITHER && ch >= copied) {
                uint32_t const least = encode_value<FORMAT>(values[ch][0], true, -0.5f), greatest = encode_value<FORMAT>(values[ch][0], true, 0.5f - 0x1p-23f);
                if (__builtin_amdgcn_readfirstlane(least ^ greatest) == 0u) {    // uniform
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        int const at = k * PIXEL + ch * BPC; // byte of the group
                        words[at >> 2] |= least << (8 * (at & 3));
                    }
                    continue;
                }
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                int const at = k * PIXEL + ch * BPC;
                float value = values[ch][k];
                if constexpr (FORMAT == NTC_HIP_DEV_FORMAT_UNORM8) {
                    if constexpr (DITHER) value += divide_by_top(rng[k].offset(ch), 255.f, 1.f / 255.f);
                    words[at >> 2] = put_unorm8(value * 255.f, at & 3, words[at >> 2]);
                } else {
                    uint32_t const bits = encode_value<FORMAT>(value, DITHER, DITHER ? rng[k].offset(ch) : 0.f);
                    words[at >> 2] |= BPC == 4 ? bits : bits << (8 * (at & 3));
                }
            }
        }
        uint8_t* const out = a.image + size_t(y) * a.rowPitch + size_t(x) * PIXEL;
        if (whole) {
            constexpr int FOURS = PIXEL & ~3, TWOS = FOURS + (PIXEL & 2);
#pragma unroll
            for (int w = 0; w < FOURS; w += 4)
                *reinterpret_cast<u32x4_any*>(out + 4 * w) = u32x4_any{ words[w], words[w + 1], words[w + 2], words[w + 3] };
            if constexpr ((PIXEL & 2) != 0) *reinterpret_cast<u32x2_any*>(out + 4 * FOURS) = u32x2_any{ words[FOURS], words[FOURS + 1] };
            if constexpr ((PIXEL & 1) != 0) *reinterpret_cast<u32_any*>(out + 4 * TWOS) = words[TWOS];
        } else {
#pragma unroll
            for (int b = 0; b < 4 * PIXEL; b += BPC) {
                if (x + b / PIXEL >= a.width) continue;
                uint32_t const bits = words[b >> 2] >> (8 * (b & 3));
                if constexpr (BPC == 1)      out[b] = uint8_t(bits);
                else if constexpr (BPC == 2) *reinterpret_cast<uint16_t*>(out + b) = uint16_t(bits);
                else                         *reinterpret_cast<uint32_t*>(out + b) = bits;
            }
        }
    }
}

// ReadImageChannel, src/ImageProcessing.cu:113-139: channel k of a 16-byte piece of the pixel.
template <int FORMAT>
__device__ __forceinline__ float decode_channel(uint32_t const (&words)[4], int k, float const* unorm8Table)
{
    constexpr int BPC = bytes_per_channel(FORMAT);
    uint32_t const w = words[(k * BPC) >> 2] >> (8 * ((k * BPC) & 3));
    if constexpr (FORMAT == NTC_HIP_DEV_FORMAT_UNORM8)       return unorm8Table[w & 0xffu];          // = float(code) / 255.f
    else if constexpr (FORMAT == NTC_HIP_DEV_FORMAT_UNORM16) return float(w & 0xffffu) / 65535.f;
    else if constexpr (FORMAT == NTC_HIP_DEV_FORMAT_FLOAT16) return float(__builtin_bit_cast(_Float16, uint16_t(w)));
    else if constexpr (FORMAT == NTC_HIP_DEV_FORMAT_FLOAT32) return __builtin_bit_cast(float, w);
    else                                                     return float(w);
}

// The half of the internal layout that a channel of the user image becomes: its bits (upper bits are ignored by the
// narrow formats) through the pair of colour spaces (uniform).
template <int FORMAT>
__device__ __forceinline__ uint32_t stored_half_of(uint32_t bits, int pair)
{
    if constexpr (FORMAT == NTC_HIP_DEV_FORMAT_UNORM8) {
        return storedOfUnorm8[pair < 0 ? kTransferPairs : pair][bits & 0xffu];
    } else if constexpr (FORMAT == NTC_HIP_DEV_FORMAT_UNORM16) {
        return pair < 0 ? unit_half(divide_by_top(float(bits & 0xffffu), 65535.f, 1.f / 65535.f)) : storedOfUnorm16[pair][bits & 0xffffu];
    } else if constexpr (FORMAT == NTC_HIP_DEV_FORMAT_FLOAT16) {
        return stored_half(transfer_half(pair, bits & 0xffffu));
    } else {
        float const v = FORMAT == NTC_HIP_DEV_FORMAT_FLOAT32 ? __builtin_bit_cast(float, bits) : float(bits);
        return stored_half(pair < 0 ? v : encode_color_space((pair + 1) % 3, decode_color_space((pair + 1) / 3, v)));
    }
}

// Four pixels of at most eight bytes a lane, like read_groups_kernel the other way round: whole dwords of the pixels
// in, 16 bytes of each complete channel pair out; where the image has only one channel of a pair, its halves go out
// one by one between those of the other.  CHANNELS = channels of a source pixel, of which a.numChannels are stored.
// 8-bit codes of linear channels become halves by a product, others through a table in LDS, a row of 256 per channel.
// Bound by memory, and by the start and end of a launch where there is little of it: 2048 x 2048 of 8 bits, RGBA with sRGB
// 11.0 us (its bytes take 7), two channels in halves of two pairs 10.5 (4), one 7.8 (2), HLG halves 14.9 (10); one pixel a
// lane took 91, 15 (one channel) and 29, tables filled before the first pixels were asked for 11.9, 11.5, 7.9 and 15.5.
template <int FORMAT, int CHANNELS>
__global__ void __launch_bounds__(1024, 8)
write_groups_kernel(GroupsArgs a)
{
    constexpr int BPC = bytes_per_channel(FORMAT), PIXEL = CHANNELS * BPC, PAIRS = CHANNELS / 2 + 1;
    constexpr bool CODES = FORMAT == NTC_HIP_DEV_FORMAT_UNORM8, HALVES = FORMAT == NTC_HIP_DEV_FORMAT_FLOAT16;
    static_assert(PIXEL <= 8, "the words of four pixels stay in registers");
    __shared__ uint16_t codes[CODES ? CHANNELS : 1][256];
    extern __shared__ float staged[];
    GroupPlace const place(a);
    int const lx = place.lx, odd = a.firstChannel & 1;
    auto const pixel_at = [&](int x, int y) { return a.image + size_t(a.verticalFlip ? a.height - 1 - y : y) * a.rowPitch + size_t(x) * PIXEL; };
    constexpr int FOURS = PIXEL & ~3, TWOS = FOURS + (PIXEL & 2);
    // (four pixels of the row wherever the lane's group lies; a group that the row cuts off is read again)
    uint32_t ahead[PIXEL];
    auto const load = [&](int tile) {
        int x, y;
        place.of_tile(tile, x, y);
        if (a.width < 4) return;                             // uniform
        uint8_t const* const in = pixel_at(min(x, a.width - 4), min(y, a.height - 1));
#pragma unroll
        for (int w = 0; w < FOURS; w += 4) {
            u32x4_any const v = *reinterpret_cast<u32x4_any const*>(in + 4 * w);
            ahead[w] = v[0]; ahead[w + 1] = v[1]; ahead[w + 2] = v[2]; ahead[w + 3] = v[3];
        }
        if constexpr ((PIXEL & 2) != 0) {
            u32x2_any const v = *reinterpret_cast<u32x2_any const*>(in + 4 * FOURS);
            ahead[FOURS] = v[0]; ahead[FOURS + 1] = v[1];
        }
        if constexpr ((PIXEL & 1) != 0) ahead[TWOS] = *reinterpret_cast<u32_any const*>(in + 4 * TWOS);
    };
    load(blockIdx.x);
    if constexpr (CODES) {
        // (256 threads; the tables' loads are all in flight before the first is stored)
        if (a.transfers.pairs != 0u) {                       // uniform
            uint32_t code[CHANNELS];
#pragma unroll
            for (int ch = 0; ch < CHANNELS; ++ch) code[ch] = storedOfUnorm8[max(a.transfers.pair(ch), 0)][threadIdx.x & 255u];
#pragma unroll
            for (int ch = 0; ch < CHANNELS; ++ch) codes[ch][threadIdx.x & 255u] = uint16_t(code[ch]);
            __syncthreads();
        }
    }
    if constexpr (HALVES) copy_staged(a.transfers, staged);
    for (int tile = blockIdx.x; tile < a.grid.tiles; tile += a.grid.step) {
        uint32_t words[PIXEL];
#pragma unroll
        for (int w = 0; w < PIXEL; ++w) words[w] = ahead[w];
        if (tile + a.grid.step < a.grid.tiles) load(tile + a.grid.step);     // uniform
        int x, y;
        place.of_tile(tile, x, y);
        if (y >= a.height) continue;                         // (uniform across a wave that covers one row)
        int const tileX = (x >> 2) >> a.grid.log2LanesX;
        bool const whole = x + 4 <= a.width;
        if (!whole) {
            uint8_t const* const in = pixel_at(x, y);
#pragma unroll
            for (int w = 0; w < PIXEL; ++w) words[w] = 0u;
#pragma unroll
            for (int b = 0; b < 4 * PIXEL; b += BPC) {
                if (x + b / PIXEL >= a.width) continue;
                if constexpr (BPC == 1)      words[b >> 2] |= uint32_t(in[b]) << (8 * (b & 3));
                else if constexpr (BPC == 2) words[b >> 2] |= uint32_t(*reinterpret_cast<uint16_t const*>(in + b)) << (8 * (b & 3));
                else                         words[b >> 2] = *reinterpret_cast<uint32_t const*>(in + b);
            }
#pragma unroll
            for (int w = 0; w < PIXEL; ++w) asm volatile("" : "+v"(words[w]));           // (waited for here)
        }
        uint32_t half[CHANNELS][4];
#pragma unroll
        for (int ch = 0; ch < CHANNELS; ++ch) {
            uint32_t bits[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                int const at = k * PIXEL + ch * BPC;         // byte of the group
                bits[k] = words[at >> 2] >> (8 * (at & 3));
                if constexpr (BPC == 1) bits[k] &= 0xffu;
                if constexpr (BPC == 2) bits[k] &= 0xffffu;
            }
            if constexpr (CODES) {
                if (a.transfers.pair(ch) < 0) {              // uniform
#pragma unroll
                    for (int k = 0; k < 4; ++k) half[ch][k] = unit_half(divide_by_top(float(bits[k]), 255.f, 1.f / 255.f));
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k) half[ch][k] = codes[ch][bits[k]];
                }
            } else if constexpr (HALVES) {
                float value[4];
                transfer_halves(staged, a.transfers.slot(ch), a.transfers.pair(ch), bits, value);
#pragma unroll
                for (int k = 0; k < 4; ++k) half[ch][k] = stored_half(value[k]);
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k) half[ch][k] = stored_half_of<FORMAT>(bits[k], a.transfers.pair(ch));
            }
        }
        uint16_t* const dst = a.planar + size_t(y) * size_t(a.width) * size_t(a.setChannels) + size_t(x) * 2;
#pragma unroll
        for (int p = 0; p < PAIRS; ++p) {
            int const lower = 2 * p - odd;                   // the image's channel in the pair's first half, lower + 1 in its second
            if (lower >= int(a.channels)) continue;          // uniform, and so is everything about p
            uint16_t* const to = dst + size_t((a.firstChannel & ~1) + 2 * p) * size_t(a.width);
            bool const hasLower = lower >= 0, hasUpper = lower + 1 < int(a.channels);
            uint32_t pair[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                uint32_t const even = 2 * p < CHANNELS ? half[2 * p < CHANNELS ? 2 * p : 0][k] : 0u, before = p > 0 ? half[p > 0 ? 2 * p - 1 : 0][k] : 0u;
                uint32_t const after = 2 * p + 1 < CHANNELS ? half[2 * p + 1 < CHANNELS ? 2 * p + 1 : 0][k] : 0u;
                pair[k] = odd ? before | (even << 16) : even | (after << 16);
            }
            if (hasLower && hasUpper) {
                if (whole) {
                    *reinterpret_cast<u32x4_a4*>(to) = u32x4_a4{ pair[0], pair[1], pair[2], pair[3] };
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k) if (x + k < a.width) *reinterpret_cast<uint32_t*>(to + 2 * k) = pair[k];
                }
            } else if (a.grid.log2LanesX == 6) {
                // One half of a pair, a wave per row: the wave's 256 halves are dealt out anew, 64 neighbours to a
                // store, so that a store touches 256 bytes and not 1 KB (one channel 12 -> 10 us, two
                // 19 -> 13 us).  Lane i's pixel of store s is element i % 4
                // of lane 16 s + i / 4.
                uint32_t const low = hasLower ? __builtin_amdgcn_perm(pair[1], pair[0], 0x05040100u) : __builtin_amdgcn_perm(pair[1], pair[0], 0x07060302u);
                uint32_t const high = hasLower ? __builtin_amdgcn_perm(pair[3], pair[2], 0x05040100u) : __builtin_amdgcn_perm(pair[3], pair[2], 0x07060302u);
                uint16_t* const from = to - 2 * 4 * lx + 2 * lx + (hasLower ? 0 : 1);      // the wave's first pixel, then the lane's
                int const left = a.width - tileX * 256 - lx;                                 // pixels of the row from the lane's first on
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    int const source = (16 * s + (lx >> 2)) * 4;
                    uint32_t const l = uint32_t(__builtin_amdgcn_ds_bpermute(source, int(low))), h = uint32_t(__builtin_amdgcn_ds_bpermute(source, int(high)));
                    uint32_t const two = (lx & 2) ? h : l;
                    if (64 * s < left) from[2 * 64 * s] = uint16_t((lx & 1) ? two >> 16 : two);
                }
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (x + k < a.width) to[2 * k + (hasLower ? 0 : 1)] = uint16_t(hasLower ? pair[k] : pair[k] >> 16);
            }
        }
    }
}

// User image -> internal fp16 planar pairs: ITextureSet::WriteChannels through CopyImageKernel's 1:1
// branch (src/TextureSet.cpp:835-913, src/ImageProcessing.cu:220-265), optional vertical flip.
// The pixel is read 16 bytes at a time with the widest loads its alignment allows; channel pairs
// that fall on a half2 of the internal layout are written as one dword.  PLAIN as above.
template <int FORMAT, bool PLAIN>
__global__ void __launch_bounds__(256)
write_channels_kernel(WriteChannelsArgs a)
{
    constexpr int BPC = bytes_per_channel(FORMAT), PER = 16 / BPC;
    __shared__ float unorm8Table[FORMAT == NTC_HIP_DEV_FORMAT_UNORM8 ? 256 : 1];
    if constexpr (FORMAT == NTC_HIP_DEV_FORMAT_UNORM8 && PLAIN) {     // one correctly rounded division per code instead of per channel
        unorm8Table[threadIdx.x & 255] = float(threadIdx.x & 255) / 255.f;
        __syncthreads();
    }
    CopyGrid const at(a.xShift);
    int const x = at.x, y = at.y;
    if (x >= a.width || y >= a.height) return;
    int const srcY = a.verticalFlip ? a.height - 1 - y : y;          // SetupBilinearFilter flips the read position
    uint8_t const* px = a.src + size_t(srcY) * a.rowPitch + size_t(x) * a.pixelStride;
    uint16_t* dst = a.planarPairs + size_t(y) * size_t(a.width) * size_t(a.setChannels) + size_t(x) * 2;
    uint32_t pending = 0;                                            // low half of a pair waiting for its partner
#pragma unroll
    for (int piece = 0; piece < NTC_HIP_DEV_MAX_CHANNELS / PER; ++piece) {
        int const base = piece * PER;
        if (base >= a.numChannels) break;                            // uniform
        int const bytes = min(PER, a.numChannels - base) * BPC;
        uint8_t const* const in = px + base * BPC;
        uint32_t words[4] = { 0u, 0u, 0u, 0u };
        if (bytes == 16 && a.vectorBytes >= 16) {
            uint4 const v = *reinterpret_cast<uint4 const*>(in);
            words[0] = v.x; words[1] = v.y; words[2] = v.z; words[3] = v.w;
        } else if ((bytes & 3) == 0 && a.vectorBytes >= 4) {
            for (int q = 0; q < bytes / 4; ++q) words[q] = reinterpret_cast<uint32_t const*>(in)[q];
        } else if constexpr (BPC == 1) {
            for (int q = 0; q < bytes; ++q) words[q >> 2] |= uint32_t(in[q]) << (8 * (q & 3));
        } else if constexpr (BPC == 2) {
            for (int q = 0; q < bytes / 2; ++q) words[q >> 1] |= uint32_t(reinterpret_cast<uint16_t const*>(in)[q]) << (16 * (q & 1));
        } else {
            for (int q = 0; q < bytes / 4; ++q) words[q] = reinterpret_cast<uint32_t const*>(in)[q];
        }
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            int const ch = base + k;
            if (ch >= a.numChannels) continue;                       // uniform
            uint32_t half;
            if constexpr (PLAIN) half = stored_half(decode_channel<FORMAT>(words, k, unorm8Table));
            else                 half = stored_half_of<FORMAT>(words[(k * BPC) >> 2] >> (8 * ((k * BPC) & 3)), transfer_pair(a.srcColorSpaces[ch], a.dstColorSpaces[ch]));
            int const c = a.firstChannel + ch;
            uint16_t* const to = dst + size_t(c & ~1) * size_t(a.width);
            if ((c & 1) == 0) {
                if (ch + 1 < a.numChannels) pending = half;          // partner follows: store both together
                else to[0] = uint16_t(half);
            } else {
                if (ch > 0) *reinterpret_cast<uint32_t*>(to) = pending | (half << 16);
                else to[1] = uint16_t(half);
            }
        }
    }
}

// ---- resampling copies (src/ImageProcessing.cu:24-72: SetupBilinearFilter) -------------------------
//
// The position of destination pixel (x, y) in the source is ((x + 1/2) / dstW) * srcW - 1/2, clamped
// to the source image; the four taps around it are weighted bilinearly, and a tap whose weight is
// zero is not used (at the right and bottom edges it would lie outside the image; here its index is
// clamped and its value dropped).  The blend is a * w0 + b * w1 + c * w2 + d * w3 evaluated as one
// multiply and three fused multiply-adds, which is what the reference's compiler makes of that
// expression.  These kernels are general rather than fast: one lane per destination pixel, one
// channel at a time.
struct BilinearTaps { int x0, y0, x1, y1; float w[4]; };

__device__ __forceinline__ BilinearTaps setup_bilinear(int srcW, int srcH, int dstW, int dstH, int x, int y)
{
    if (srcW == dstW && srcH == dstH) return BilinearTaps{ x, y, x, y, { 1.f, 0.f, 0.f, 0.f } };   // the reference's 1:1 shortcut
    float const u = (float(x) + 0.5f) / float(dstW), v = (float(y) + 0.5f) / float(dstH);
    float const px = fmaxf(0.f, fminf(float(srcW) - 1.f, u * float(srcW) - 0.5f));
    float const py = fmaxf(0.f, fminf(float(srcH) - 1.f, v * float(srcH) - 0.5f));
    float const fx = px - floorf(px), fy = py - floorf(py);
    BilinearTaps t;
    t.x0 = int(floorf(px)); t.y0 = int(floorf(py));
    t.x1 = min(t.x0 + 1, srcW - 1); t.y1 = min(t.y0 + 1, srcH - 1);
    t.w[0] = (1.f - fx) * (1.f - fy); t.w[1] = fx * (1.f - fy); t.w[2] = (1.f - fx) * fy; t.w[3] = fx * fy;
    return t;
}

// ALL_WEIGHTED: the caller knows that no weight is zero.
template <bool ALL_WEIGHTED = false>
__device__ __forceinline__ float blend_taps(BilinearTaps const& t, float a, float b, float c, float d)
{
    if constexpr (!ALL_WEIGHTED) {
        a = t.w[0] > 0.f ? a : 0.f; b = t.w[1] > 0.f ? b : 0.f; c = t.w[2] > 0.f ? c : 0.f; d = t.w[3] > 0.f ? d : 0.f;
    }
    return __builtin_fmaf(d, t.w[3], __builtin_fmaf(c, t.w[2], __builtin_fmaf(b, t.w[1], a * t.w[0])));
}

__device__ __forceinline__ float planar_half(uint16_t const* image, int width, int setChannels, int x, int y, int c)
{
    uint16_t const bits = image[size_t(y) * size_t(width) * size_t(setChannels) + size_t(c & ~1) * size_t(width) + size_t(x) * 2 + size_t(c & 1)];
    return float(__builtin_bit_cast(_Float16, bits));
}

// Channel `k` of a pixel of the user image, any format and alignment the format allows.
__device__ __forceinline__ float user_channel(uint8_t const* px, int format, int k)
{
    switch (format) {
    case NTC_HIP_DEV_FORMAT_UNORM8:  return float(px[k]) / 255.f;
    case NTC_HIP_DEV_FORMAT_UNORM16: return float(reinterpret_cast<uint16_t const*>(px)[k]) / 65535.f;
    case NTC_HIP_DEV_FORMAT_FLOAT16: return float(reinterpret_cast<_Float16 const*>(px)[k]);
    case NTC_HIP_DEV_FORMAT_FLOAT32: return reinterpret_cast<float const*>(px)[k];
    default:                         return float(reinterpret_cast<uint32_t const*>(px)[k]);
    }
}

template <int FORMAT>
__global__ void __launch_bounds__(256)
read_channels_resize_kernel(ReadChannelsArgs a)
{
    constexpr int BPC = bytes_per_channel(FORMAT);
    int const x = blockIdx.x * 64 + (threadIdx.x & 63), y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= a.dstWidth || y >= a.dstHeight) return;
    BilinearTaps const t = setup_bilinear(a.width, a.height, a.dstWidth, a.dstHeight, x, y);
    uint8_t* const px = a.dst + size_t(y) * a.rowPitch + size_t(x) * a.pixelStride;
    DitherRng rng(uint32_t(x) + uint32_t(y) * uint32_t(a.dstWidth));
    for (int ch = 0; ch < a.dstChannels; ++ch) {
        float value;
        if (ch < a.numChannels) {
            int const c = a.firstChannel + ch, space = a.srcColorSpaces[ch];
            value = blend_taps(t, decode_color_space(space, planar_half(a.planarPairs, a.width, a.setChannels, t.x0, t.y0, c)),
                                  decode_color_space(space, planar_half(a.planarPairs, a.width, a.setChannels, t.x1, t.y0, c)),
                                  decode_color_space(space, planar_half(a.planarPairs, a.width, a.setChannels, t.x0, t.y1, c)),
                                  decode_color_space(space, planar_half(a.planarPairs, a.width, a.setChannels, t.x1, t.y1, c)));
        } else {
            value = (ch == 3) ? 1.f : 0.f;
        }
        float const dither = a.useDithering ? rng.next_offset() : 0.f;
        uint32_t const bits = encode_channel<FORMAT>(ch < 16 ? a.dstColorSpaces[ch] : 0, value, a.useDithering != 0, dither);
        if constexpr (BPC == 1) px[ch] = uint8_t(bits);
        else if constexpr (BPC == 2) reinterpret_cast<uint16_t*>(px)[ch] = uint16_t(bits);
        else reinterpret_cast<uint32_t*>(px)[ch] = bits;
    }
}

__global__ void __launch_bounds__(256)
write_channels_resize_kernel(WriteChannelsArgs a)
{
    int const x = blockIdx.x * 64 + (threadIdx.x & 63), y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= a.width || y >= a.height) return;
    BilinearTaps const t = setup_bilinear(a.srcWidth, a.srcHeight, a.width, a.height, x, a.verticalFlip ? a.height - 1 - y : y);
    uint8_t const* const p00 = a.src + size_t(t.y0) * a.rowPitch + size_t(t.x0) * a.pixelStride;
    uint8_t const* const p10 = a.src + size_t(t.y0) * a.rowPitch + size_t(t.x1) * a.pixelStride;
    uint8_t const* const p01 = a.src + size_t(t.y1) * a.rowPitch + size_t(t.x0) * a.pixelStride;
    uint8_t const* const p11 = a.src + size_t(t.y1) * a.rowPitch + size_t(t.x1) * a.pixelStride;
    uint16_t* const dst = a.planarPairs + size_t(y) * size_t(a.width) * size_t(a.setChannels) + size_t(x) * 2;
    for (int ch = 0; ch < a.numChannels; ++ch) {
        int const space = a.srcColorSpaces[ch];
        float const value = blend_taps(t, decode_color_space(space, user_channel(p00, a.format, ch)), decode_color_space(space, user_channel(p10, a.format, ch)),
                                          decode_color_space(space, user_channel(p01, a.format, ch)), decode_color_space(space, user_channel(p11, a.format, ch)));
        int const c = a.firstChannel + ch;
        dst[size_t(c & ~1) * size_t(a.width) + size_t(c & 1)] = stored_half(encode_color_space(a.dstColorSpaces[ch], value));
    }
}

// ResizeMultichannelImageKernel (src/ImageProcessing.cu:178-207): every channel of one image of the
// internal layout resampled into another; a channel pair is read as dwords and written as one.
//
// A lane makes one pixel of a range of channel pairs.  The two taps of a source row are neighbours: one 8-byte load
// (shifted left by a pixel at the right edge), and the next pair's are under way while a pair is filtered.  Stored
// values are decoded by table (from LDS in launches large enough, as in the copies above; a powf per tap and channel
// kept the kernel at 0.9 TB/s), the filtered value is encoded by the device function.  Images too small to fill the
// GPU are split by channel pairs: one mip of 64 x 64 and six pairs is 64 waves, not 4, in a chain a sixth as long.
// This kernel is for sizes that are no exact halves (a mip of an odd one); the others are halve_planar_kernel's.
struct ResizePlanarArgs {
    uint16_t const* src; uint16_t* dst;
    int32_t srcWidth, srcHeight, dstWidth, dstHeight, setChannels;
    int32_t tilesX, tiles, pairsPerLane;                     // tiles of 64 pixels x a row per wave
    int32_t step, threads;                                   // workgroups in x, threads of each
    Transfers transfers;                                     // of the decoding pairs; those of the colour spaces in the place of channels
    uint32_t spaces;                                         // two bits a channel
    __host__ __device__ __forceinline__ int space(int channel) const { return int(spaces >> (2 * channel)) & 3; }
};

template <bool LINEAR>
__global__ void __launch_bounds__(1024, 8)
resize_planar_kernel(ResizePlanarArgs a)
{
    extern __shared__ float staged[];
    if constexpr (!LINEAR) copy_staged(a.transfers, staged);
    int const pairBegin = int(blockIdx.y) * a.pairsPerLane, pairEnd = min(a.setChannels >> 1, pairBegin + a.pairsPerLane);
    size_t const srcRow = size_t(a.srcWidth) * size_t(a.setChannels), pairStride = size_t(a.srcWidth) * 2;
    for (int tile = blockIdx.x; tile < a.tiles; tile += a.step) {
        int const tileY = tile / a.tilesX, tileX = tile - tileY * a.tilesX;
        int const x = tileX * 64 + int(threadIdx.x & 63), y = tileY * (a.threads >> 6) + int(threadIdx.x >> 6);
        if (x >= a.dstWidth || y >= a.dstHeight) continue;
        BilinearTaps const t = setup_bilinear(a.srcWidth, a.srcHeight, a.dstWidth, a.dstHeight, x, y);
        int const left = max(0, min(t.x0, a.srcWidth - 2));  // columns left and left + 1 hold both taps
        bool const shift0 = t.x0 != left, shift1 = t.x1 != left;
        uint16_t const* const r0 = a.src + size_t(t.y0) * srcRow + size_t(left) * 2;
        uint16_t const* const r1 = a.src + size_t(t.y1) * srcRow + size_t(left) * 2;
        uint32_t* const out = reinterpret_cast<uint32_t*>(a.dst + size_t(y) * size_t(a.dstWidth) * size_t(a.setChannels) + size_t(x) * 2);
        auto load = [&](uint16_t const* row, int p, uint32_t (&taps)[2]) {
            if (a.srcWidth < 2) {                            // uniform
                taps[0] = taps[1] = *reinterpret_cast<uint32_t const*>(row + size_t(p) * pairStride);
            } else {
                u32x2_a4 const v = *reinterpret_cast<u32x2_a4 const*>(row + size_t(p) * pairStride);
                taps[0] = v[0]; taps[1] = v[1];
            }
        };
        // (taps of zero weight have to be dropped: the product with an infinity would not be zero.  Away from the
        // edges of a 2 : 1 reduction no lane has one.)
        auto pairs = [&](auto allWeighted) __attribute__((always_inline)) {
            constexpr bool ALL = decltype(allWeighted)::value;
            uint32_t top[2], bottom[2];
            load(r0, pairBegin, top);
            load(r1, pairBegin, bottom);
            for (int p = pairBegin; p < pairEnd; ++p) {
                uint32_t const v00 = shift0 ? top[1] : top[0], v10 = shift1 ? top[1] : top[0];
                uint32_t const v01 = shift0 ? bottom[1] : bottom[0], v11 = shift1 ? bottom[1] : bottom[0];
                int const next = min(p + 1, pairEnd - 1);
                load(r0, next, top);
                load(r1, next, bottom);
                uint32_t packed = 0;
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    int const space = LINEAR ? 0 : a.space(2 * p + k);
                    uint32_t const bits[4] = { (v00 >> (16 * k)) & 0xffffu, (v10 >> (16 * k)) & 0xffffu, (v01 >> (16 * k)) & 0xffffu, (v11 >> (16 * k)) & 0xffffu };
                    float v[4];
                    if constexpr (LINEAR) transfer_halves(staged, 0, -1, bits, v);
                    else                  transfer_halves(staged, a.transfers.slot(space), a.transfers.pair(space), bits, v);
                    packed |= encoded_half(space, blend_taps<ALL>(t, v[0], v[1], v[2], v[3])) << (16 * k);
                }
                out[size_t(p) * size_t(a.dstWidth)] = packed;
            }
        };
        if (__all(t.w[0] > 0.f && t.w[1] > 0.f && t.w[2] > 0.f && t.w[3] > 0.f)) pairs(std::true_type{});
        else                                                                     pairs(std::false_type{});
    }
}

// The same for an image of exactly half the width and height, what each mip is of an even one above it: the taps of pixel x
// are pixels 2 x and 2 x + 1 whatever the roundings of its position (which is off by less than 0.01 up to 65536 pixels),
// none of them without weight.  A lane makes two pixels from 16 bytes of each row, and a pair's are under way while the one
// before is filtered.  Bound by memory where the image is large, by the tables' gathers in the middle, by the launch below
// 128 x 128.  4096 x 4096, 2048 x 2048 and 1024 x 1024 of 12 channels, three sRGB and three HLG: 162, 35 and 12.2 us with 8
// bytes a load, colour spaces read from memory at each pair (a wait for everything in flight, the next pair's taps too) and
// tables copied dword by dword; 106, 24 and 10.5 now, 5.0 of 5.7 TB/s that linear channels reach.  Tables in LDS for the
// 1024 x 1024 image as well take longer to copy than they save (13.4).
template <bool LINEAR>
__global__ void __launch_bounds__(1024, 8)
halve_planar_kernel(ResizePlanarArgs a)
{
    extern __shared__ float staged[];
    int const pairBegin = int(blockIdx.y) * a.pairsPerLane, pairEnd = min(a.setChannels >> 1, pairBegin + a.pairsPerLane);
    size_t const srcRow = size_t(a.srcWidth) * size_t(a.setChannels), pairStride = size_t(a.srcWidth) * 2;
    int const lane = int(threadIdx.x & 63), row = int(threadIdx.x >> 6);
    // (the last lane of an odd row makes the pixel before the last one too, like the lane that it is another's)
    auto const row_of = [&](int tile, int& x, int& y) -> uint16_t const* {
        int const tileY = tile / a.tilesX, tileX = tile - tileY * a.tilesX;
        x = min((tileX * 64 + lane) * 2, a.dstWidth - 2); y = min(tileY * (a.threads >> 6) + row, a.dstHeight - 1);
        return a.src + size_t(2 * y) * srcRow + size_t(x) * 4;
    };
    u32x4_a4 top, bottom;
    auto const load = [&](uint16_t const* from) {
        top = *reinterpret_cast<u32x4_a4 const*>(from);
        bottom = *reinterpret_cast<u32x4_a4 const*>(from + srcRow);
    };
    int x, y;
    uint16_t const* from = row_of(blockIdx.x, x, y);
    load(from + size_t(pairBegin) * pairStride);
    if constexpr (!LINEAR) copy_staged(a.transfers, staged);
    for (int tile = blockIdx.x; tile < a.tiles; tile += a.step) {
        int const tileY = tile / a.tilesX, tileX = tile - tileY * a.tilesX;
        bool const inside = (tileX * 64 + lane) * 2 < a.dstWidth && tileY * (a.threads >> 6) + row < a.dstHeight;
        BilinearTaps const t0 = setup_bilinear(a.srcWidth, a.srcHeight, a.dstWidth, a.dstHeight, x, y);
        BilinearTaps const t1 = setup_bilinear(a.srcWidth, a.srcHeight, a.dstWidth, a.dstHeight, x + 1, y);
        uint16_t* const to = a.dst + size_t(y) * size_t(a.dstWidth) * size_t(a.setChannels) + size_t(x) * 2;
        for (int p = pairBegin; p < pairEnd; ++p) {
            u32x4_a4 const upper = top, lower = bottom;
            if (p + 1 < pairEnd) {
                load(from + size_t(p + 1) * pairStride);
            } else if (tile + a.step < a.tiles) {            // (uniform, both)
                int nextX, nextY;
                load(row_of(tile + a.step, nextX, nextY) + size_t(pairBegin) * pairStride);
            }
            uint32_t packed[2] = { 0u, 0u };
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                int const space = LINEAR ? 0 : a.space(2 * p + k);
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    uint32_t const bits[4] = { (upper[2 * i] >> (16 * k)) & 0xffffu, (upper[2 * i + 1] >> (16 * k)) & 0xffffu,
                                               (lower[2 * i] >> (16 * k)) & 0xffffu, (lower[2 * i + 1] >> (16 * k)) & 0xffffu };
                    float v[4];
                    if constexpr (LINEAR) transfer_halves(staged, 0, -1, bits, v);
                    else                  transfer_halves(staged, a.transfers.slot(space), a.transfers.pair(space), bits, v);
                    packed[i] |= encoded_half(space, blend_taps<true>(i ? t1 : t0, v[0], v[1], v[2], v[3])) << (16 * k);
                }
            }
            if (inside) *reinterpret_cast<u32x2_a4*>(to + size_t(p) * size_t(a.dstWidth) * 2) = u32x2_a4{ packed[0], packed[1] };
        }
        if (tile + a.step < a.tiles) from = row_of(tile + a.step, x, y);
    }
}

hipError_t launch_resize_planar(uint16_t const* src, int srcWidth, int srcHeight, uint16_t* dst, int dstWidth, int dstHeight,
                                int setChannels, uint8_t const* colorSpaces, hipStream_t stream)
{
    ResizePlanarArgs a{};
    a.src = src; a.dst = dst; a.srcWidth = srcWidth; a.srcHeight = srcHeight; a.dstWidth = dstWidth; a.dstHeight = dstHeight; a.setChannels = setChannels;
    bool linear = true;
    for (int i = 0; i < 16; ++i) {
        uint32_t const space = colorSpaces && i < setChannels ? colorSpaces[i] : 0u;
        a.spaces |= space << (2 * i);
        linear = linear && space == 0u;
    }
    int const units = compute_units_of_current_device(), pairs = setChannels / 2;
    bool const half = dstWidth >= 2 && srcWidth == 2 * dstWidth && srcHeight == 2 * dstHeight && srcWidth <= 65536 && srcHeight <= 65536;
    int const tileWidth = half ? 128 : 64;
    auto tile = [&](int threads) {
        a.tilesX = (dstWidth + tileWidth - 1) / tileWidth;
        a.tiles = a.tilesX * ((dstHeight + threads / 64 - 1) / (threads / 64));
    };
    int threads = int(kStagingThreads);
    tile(threads);
    bool const stage = !linear && a.tiles * tileWidth >= 128 * units;            // as in plan_groups: each copy serves two pixels a thread or more
    for (int space = 1; space <= 2; ++space) {
        bool used = false;
        for (int i = 0; i < setChannels; ++i) used = used || a.space(i) == space;
        int const pair = transfer_pair(space, 0);
        a.transfers.set(space, pair, stage && used ? a.transfers.stage(pair) : 0);
    }
    dim3 grid(1);
    a.pairsPerLane = pairs;
    if (stage) {
        grid.x = unsigned(2 * units < a.tiles ? 2 * units : a.tiles);
    } else {
        threads = 256;
        tile(threads);
        // as many ranges of pairs as it takes to have eight waves for every SIMD
        int const waves = a.tiles * (threads / 64), wanted = (32 * units + waves - 1) / waves;
        int const ranges = wanted < 1 ? 1 : wanted > pairs ? pairs : wanted;
        a.pairsPerLane = (pairs + ranges - 1) / ranges;
        grid = dim3(unsigned(a.tiles), unsigned((pairs + a.pairsPerLane - 1) / a.pairsPerLane));
    }
    size_t const lds = size_t(a.transfers.count()) * kStageStride * sizeof(float);
    a.step = int(grid.x);
    a.threads = threads;
    if (half) return linear ? launch_kernel<halve_planar_kernel<true>>(grid, dim3(threads), lds, stream, a)
                            : launch_kernel<halve_planar_kernel<false>>(grid, dim3(threads), lds, stream, a);
    return linear ? launch_kernel<resize_planar_kernel<true>>(grid, dim3(threads), lds, stream, a)
                  : launch_kernel<resize_planar_kernel<false>>(grid, dim3(threads), lds, stream, a);
}

static bool plain_copy(uint8_t const* srcSpaces, uint8_t const* dstSpaces, int useDithering)
{
    bool plain = useDithering == 0;
    for (int i = 0; i < 16; ++i) plain = plain && srcSpaces[i] == 0 && dstSpaces[i] == 0;
    return plain;
}

template <int FORMAT>
static hipError_t launch_write_groups_of(GroupsArgs const& args, int srcChannels, GroupLaunch const& plan, hipStream_t stream)
{
    auto launch = [&](auto channels) -> hipError_t {
        constexpr int CHANNELS = decltype(channels)::value;
        if constexpr (CHANNELS * bytes_per_channel(FORMAT) <= 8)
            return launch_kernel<write_groups_kernel<FORMAT, CHANNELS>>(dim3(plan.grid.step), dim3(plan.threads), plan.ldsBytes, stream, args);
        else
            return hipErrorInvalidValue;
    };
    switch (srcChannels) {
    case 1: return launch(std::integral_constant<int, 1>{});
    case 2: return launch(std::integral_constant<int, 2>{});
    case 3: return launch(std::integral_constant<int, 3>{});
    case 4: return launch(std::integral_constant<int, 4>{});
    case 5: return launch(std::integral_constant<int, 5>{});
    case 6: return launch(std::integral_constant<int, 6>{});
    case 7: return launch(std::integral_constant<int, 7>{});
    case 8: return launch(std::integral_constant<int, 8>{});
    default: return hipErrorInvalidValue;
    }
}

static hipError_t launch_write_groups(WriteChannelsArgs const& a, hipStream_t stream)
{
    GroupLaunch const plan = plan_groups(a.width, a.height, a.srcColorSpaces, a.dstColorSpaces, a.numChannels, a.format == NTC_HIP_DEV_FORMAT_FLOAT16);
    GroupsArgs const args{ a.planarPairs, const_cast<uint8_t*>(a.src), a.rowPitch, a.width, a.height, plan.grid, plan.transfers,
                           uint8_t(a.setChannels), uint8_t(a.firstChannel), uint8_t(a.numChannels), 0, a.verticalFlip != 0 };
    int const channels = int(a.pixelStride) / bytes_per_channel(a.format);
    switch (a.format) {
    case NTC_HIP_DEV_FORMAT_UNORM8:  return launch_write_groups_of<NTC_HIP_DEV_FORMAT_UNORM8>(args, channels, plan, stream);
    case NTC_HIP_DEV_FORMAT_UNORM16: return launch_write_groups_of<NTC_HIP_DEV_FORMAT_UNORM16>(args, channels, plan, stream);
    case NTC_HIP_DEV_FORMAT_FLOAT16: return launch_write_groups_of<NTC_HIP_DEV_FORMAT_FLOAT16>(args, channels, plan, stream);
    case NTC_HIP_DEV_FORMAT_FLOAT32: return launch_write_groups_of<NTC_HIP_DEV_FORMAT_FLOAT32>(args, channels, plan, stream);
    case NTC_HIP_DEV_FORMAT_UINT32:  return launch_write_groups_of<NTC_HIP_DEV_FORMAT_UINT32>(args, channels, plan, stream);
    default: return hipErrorInvalidValue;
    }
}

template <int FORMAT>
static hipError_t launch_write_format(WriteChannelsArgs const& a, dim3 grid, bool plain, hipStream_t stream)
{
    return plain ? launch_kernel<write_channels_kernel<FORMAT, true>>(grid, dim3(256), 0, stream, a)
                 : launch_kernel<write_channels_kernel<FORMAT, false>>(grid, dim3(256), 0, stream, a);
}

hipError_t launch_write_channels(WriteChannelsArgs const& args, hipStream_t stream)
{
    WriteChannelsArgs a = args;
    if (a.srcWidth > 0) {                                    // resampling copy
        return launch_kernel<write_channels_resize_kernel>(dim3((a.width + 63) / 64, (a.height + 3) / 4), dim3(256), 0, stream, a);
    }
    if (a.pixelStride <= 8 && a.wholePixels) return launch_write_groups(a, stream);
    dim3 const grid = copy_grid(a.width, a.height, a.xShift, false);
    bool const plain = plain_copy(a.srcColorSpaces, a.dstColorSpaces, 0);
    switch (a.format) {
    case NTC_HIP_DEV_FORMAT_UNORM8:  return launch_write_format<NTC_HIP_DEV_FORMAT_UNORM8>(a, grid, plain, stream);
    case NTC_HIP_DEV_FORMAT_UNORM16: return launch_write_format<NTC_HIP_DEV_FORMAT_UNORM16>(a, grid, plain, stream);
    case NTC_HIP_DEV_FORMAT_FLOAT16: return launch_write_format<NTC_HIP_DEV_FORMAT_FLOAT16>(a, grid, plain, stream);
    case NTC_HIP_DEV_FORMAT_FLOAT32: return launch_write_format<NTC_HIP_DEV_FORMAT_FLOAT32>(a, grid, plain, stream);
    case NTC_HIP_DEV_FORMAT_UINT32:  return launch_write_format<NTC_HIP_DEV_FORMAT_UINT32>(a, grid, plain, stream);
    default: return hipErrorInvalidValue;
    }
}

// Per-channel sum of squared differences between a decoded mip and its reference image, both in the
// internal layout: the loss branch of InferenceKernel (src/Inference.cu:77-118) as a pass of its own.
// With a mask channel (maskChannel >= 0) the decoded mask channel is first clamped to [0, 1] and stored back
// clamped (Inference.cu:96-97,112; a negative zero becomes +0 as the device max() of the reference
// returns), and with discardMaskedOut a texel whose REFERENCE mask value is zero counts on the mask
// channel only (Inference.cu:80-84,107-108).
// Squares are fp32 as in the reference; the sum of two texels' (where the width is odd, each texel's) goes into a double
// accumulator, and the workgroup writes 16 double partial sums; ReduceLoss likewise finishes in double
// (src/Optimizer.cu:382-387).
//
// The same launch finishes the sum and hands it to the host (a second kernel, a copy and a stream synchronisation made
// most of the 28 us a call on 64 x 64 texels took).  Workgroups form at most kLossRows groups; the last one of a group
// to arrive adds the group's partial sums, in a fixed order, so results are reproducible, and stores them into pinned
// host memory, where the caller is looking and adds the rows, of which an image of up to 128 x 128 texels has one per
// workgroup.  What such a call waits for is a chain of trips to memory: a second level of groups on the device, and a
// serial number stored once the totals were acknowledged, made it 2 us longer.
// The partial sums pass between workgroups of different dies, whose caches do not see each other: they are stored and
// loaded as device-scope atomics, which go past those caches, and a store is acknowledged before its workgroup counts
// itself as arrived.  (Fences instead write back and invalidate a die's whole L2, a thousand times in a launch over
// 2048 x 2048 texels: 154 us against 50.)
__device__ __forceinline__ void publish(double* to, double v) { __hip_atomic_store(to, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ double published(double const* from) { return __hip_atomic_load(from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// Sums over the workgroup of the 16 channels' terms entries[i * 16 + channel], i < count, in a fixed order.
__device__ __forceinline__ double sum_entries(double const* entries, int count, double (&scratch)[16][NTC_HIP_DEV_MAX_CHANNELS])
{
    int const c = threadIdx.x & 15, part = threadIdx.x >> 4;                     // 16 threads per channel
    double v = 0.0;
    for (int i = part; i < count; i += 32) {                 // (two loads in flight: groups have at most 32 members up to 4096 x 4096)
        double const one = published(entries + size_t(i) * NTC_HIP_DEV_MAX_CHANNELS + c);
        double const two = published(entries + size_t(min(i + 16, count - 1)) * NTC_HIP_DEV_MAX_CHANNELS + c);
        v += one;
        if (i + 16 < count) v += two;
    }
    scratch[part][c] = v;
    __syncthreads();
    double total = 0.0;
    if (threadIdx.x < NTC_HIP_DEV_MAX_CHANNELS)
#pragma unroll
        for (int k = 0; k < 16; ++k) total += scratch[k][c];
    return total;                                            // in threads 0 ... 15
}

// Whether this workgroup is the last of `count` to come here (uniform).  Each wave has its own stores in place first.
__device__ __forceinline__ bool arrived_last(uint32_t* counter, uint32_t count, int& scratch)
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0);
    asm volatile("" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        bool const last = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == count - 1u;
        if (last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);      // as the next launch expects it
        scratch = last;
    }
    __syncthreads();
    return scratch != 0;
}

// v plus the v of another lane of the row of 16: CONTROL is a DPP control.
template <int CONTROL>
__device__ __forceinline__ double add_from_row(double v)
{
    uint64_t const bits = __builtin_bit_cast(uint64_t, v);
    uint32_t const low = uint32_t(__builtin_amdgcn_mov_dpp(int(uint32_t(bits)), CONTROL, 0xF, 0xF, true));
    uint32_t const high = uint32_t(__builtin_amdgcn_mov_dpp(int(uint32_t(bits >> 32)), CONTROL, 0xF, 0xF, true));
    return v + __builtin_bit_cast(double, uint64_t(high) << 32 | low);
}

// The sums of 256 lanes' 16 accumulators and their way to the host.  Across the workgroup: 16 threads per channel add 16 of
// its 256 values each, then each other's.  (With exchanges between lanes, 17 of a double and 1500 instructions when every
// lane hands over half of what it holds at a step, this took 1 us longer.)
__device__ __forceinline__ void hand_over_sums(double const (&acc)[NTC_HIP_DEV_MAX_CHANNELS], int setChannels, uint32_t validChannelMask,
                                               uint32_t block, uint32_t blocks, uint32_t groupSize, LossWorkspace const& work)
{
    constexpr int STRIDE = 256 + 16;                         // (channels half the banks apart)
    __shared__ double lanes[NTC_HIP_DEV_MAX_CHANNELS * STRIDE];
    __shared__ double sums[NTC_HIP_DEV_MAX_CHANNELS];
    int const lane = threadIdx.x & 63;
#pragma unroll
    for (int c = 0; c < NTC_HIP_DEV_MAX_CHANNELS; ++c) lanes[c * STRIDE + int(threadIdx.x)] = acc[c];
    __syncthreads();
    int const channel = int(threadIdx.x) >> 4, part = int(threadIdx.x) & 15;
    double mine = 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) mine += lanes[channel * STRIDE + part + 16 * k];
    mine = add_from_row<0xB1>(mine);                         // quad_perm: the neighbour,
    mine = add_from_row<0x4E>(mine);                         // the other pair,
    mine = add_from_row<0x141>(mine);                        // row_half_mirror: the other quad,
    mine = add_from_row<0x140>(mine);                        // row_mirror: the other eight
    if (channel >= setChannels || !((validChannelMask >> channel) & 1u)) mine = 0.0;
    uint32_t const group = block / groupSize, first = group * groupSize, members = min(groupSize, blocks - first);
    double total;                                            // threads 0 ... 15: a channel's each
    if (members > 1) {
        __shared__ double scratch[16][NTC_HIP_DEV_MAX_CHANNELS];
        __shared__ int last;
        if (part == 0) publish(work.partials + size_t(block) * NTC_HIP_DEV_MAX_CHANNELS + channel, mine);
        if (!arrived_last(work.counters + group * kLossCounterStride, members, last)) return;
        total = sum_entries(work.partials + size_t(first) * NTC_HIP_DEV_MAX_CHANNELS, int(members), scratch);
    } else {
        if (part == 0) sums[channel] = mine;
        __syncthreads();
        total = sums[threadIdx.x & (NTC_HIP_DEV_MAX_CHANNELS - 1)];
    }
    // To the host in one trip: each half of a double is stored together with the serial number, so that every word
    // says for itself whether it has arrived.  Stores of system scope go past the caches.  (Plain stores and a release
    // behind them write back the die's whole L2.)
    if (threadIdx.x >= 64) return;
    uint64_t const sum = __builtin_bit_cast(uint64_t, __shfl(total, lane >> 1, 64));
    uint64_t const word = uint64_t(work.serial) << 32 | ((lane & 1) ? sum >> 32 : sum & 0xffffffffu);
    if (lane < 2 * NTC_HIP_DEV_MAX_CHANNELS)
        __hip_atomic_store(&work.rows[group].words[lane], word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Squared difference of two texels' first or second halves (SHIFT = 0, 16).
template <int SHIFT> __device__ __forceinline__ float square(uint32_t a, uint32_t b)
{
    auto const half = [](uint32_t w) { return float(__builtin_bit_cast(_Float16, uint16_t(w >> SHIFT))); };
    float const d = half(a) - half(b);
    return d * d;
}

// Large images without a mask channel.  The internal layout is row after row of channel pairs, so that whole rows are one piece of memory,
// which the workgroup goes through in order, 4 KB of each image a load; STEPS of a pair's row and PAIRS pairs are under way
// together, eight loads a lane (sixteen do not leave the registers for four waves per SIMD).  The workgroups' shares differ
// by PAIRS pairs of a row at most: with whole rows, as many in each, 2500 x 2500 took 92 us and 1920 x 1080 41, now 84 and 39
// (86.5 and 39 with 8-byte loads by lanes of two texels, see below).  Bound by memory for large
// mips, by the launch and the way to the host below 512 x 512.  Whole calls of 16 channels, 4096 x 4096, 2048 x 2048, 1024 x
// 1024 and 512 x 512: 189, 51, 23 and 16.5 us; 197, 56, 29 and 18.5 with 8-byte loads of all pairs by lanes of two texels,
// and the groups' counters on one line (6 channels: 80, 28, 16.5 and 15.5; 111, 37, 25 and 18); 209, 51, 30 and 26 with a
// wave for each pair, whose rows lie a power of two apart.  A kernel that does nothing but read the two images of 16
// channels takes 172, 38 and 10 for the first three, a call of nothing 11.
template <int STEPS, int PAIRS, bool ODD>
__global__ void __launch_bounds__(256, 4)
image_loss_kernel(uint16_t const* __restrict__ a, uint16_t const* __restrict__ b, int width, int height, int setChannels, int share, int more, int log2Lanes,
                  uint32_t validChannelMask, uint32_t blocks, uint32_t groupSize, LossWorkspace work)
{
    constexpr int MAX_PAIRS = NTC_HIP_DEV_MAX_CHANNELS / 2;
    int const pairs = setChannels >> 1, stride = 4 << log2Lanes, first = (int(threadIdx.x) & ((1 << log2Lanes) - 1)) * 4;
    double acc[NTC_HIP_DEV_MAX_CHANNELS];
#pragma unroll
    for (int c = 0; c < NTC_HIP_DEV_MAX_CHANNELS; ++c) acc[c] = 0.0;
    auto const add = [&](int p, u32x4_a4 const& va, u32x4_a4 const& vb) {
#pragma unroll
        for (int k = 0; k < 4; k += 2) {
            float const s0 = square<0>(va[k], vb[k]), t0 = square<0>(va[k + 1], vb[k + 1]);
            float const s1 = square<16>(va[k], vb[k]), t1 = square<16>(va[k + 1], vb[k + 1]);
            if constexpr (ODD) {
                acc[2 * p] += double(s0); acc[2 * p] += double(t0);
                acc[2 * p + 1] += double(s1); acc[2 * p + 1] += double(t1);
            } else {
                acc[2 * p] += double(s0 + t0);
                acc[2 * p + 1] += double(s1 + t1);
            }
        }
    };
    // Units of PAIRS pairs of the rows that the lanes take together: `share` to a workgroup, and one more to the first `more`.
    int const block = int(blockIdx.x), together = 256 >> log2Lanes, groups = (pairs + PAIRS - 1) / PAIRS;
    int const firstUnit = block * share + min(block, more), endUnit = firstUnit + share + (block < more ? 1 : 0);
    int const begin = firstUnit / groups * together;
    // (addresses: the workgroup's rows, the pair and the step in scalar registers, the lane's place in 32 bits)
    size_t const rows = size_t(begin) * size_t(setChannels) * size_t(width);
    char const* const ra = reinterpret_cast<char const*>(a + rows);
    char const* const rb = reinterpret_cast<char const*>(b + rows);
    int y = begin + (int(threadIdx.x) >> log2Lanes);
    for (int unit = firstUnit - firstUnit % groups; unit < endUnit; unit += groups, y += together) {
        if (y >= height) continue;
        uint32_t const row = uint32_t(y - begin) * uint32_t(pairs) * uint32_t(width) * 4u;
#pragma unroll
        for (int p0 = 0; p0 < MAX_PAIRS; p0 += PAIRS) {
            if (unit + p0 / PAIRS < firstUnit) continue;     // uniform, as the next
            if (p0 >= pairs || unit + p0 / PAIRS >= endUnit) break;
            size_t offset[PAIRS];                            // (no branch around a load: pairs that the set does not have read its last one again, and their sums are dropped)
#pragma unroll
            for (int p = 0; p < PAIRS; ++p) offset[p] = size_t(min(p0 + p, pairs - 1)) * size_t(width) * 4u;
            int x = first;
            for (; x + (STEPS - 1) * stride + 4 <= width; x += STEPS * stride) {
                uint32_t const lane = row + uint32_t(x) * 4u;
                u32x4_a4 va[PAIRS][STEPS], vb[PAIRS][STEPS];
#pragma unroll
                for (int p = 0; p < PAIRS; ++p)
#pragma unroll
                    for (int k = 0; k < STEPS; ++k) {
                        va[p][k] = *reinterpret_cast<u32x4_a4 const*>(ra + offset[p] + size_t(k) * size_t(stride) * 4u + lane);
                        vb[p][k] = *reinterpret_cast<u32x4_a4 const*>(rb + offset[p] + size_t(k) * size_t(stride) * 4u + lane);
                    }
                __builtin_amdgcn_sched_barrier(0);           // keep the loads ahead of the arithmetic
#pragma unroll
                for (int p = 0; p < PAIRS; ++p)
#pragma unroll
                    for (int k = 0; k < STEPS; ++k) add(p0 + p, va[p][k], vb[p][k]);
            }
#pragma unroll 1
            for (; x < width; x += stride) {                 // what is left of the row, its last one to three texels alone
                uint32_t const lane = row + uint32_t(x) * 4u;
#pragma unroll
                for (int p = 0; p < PAIRS; ++p) {
                    char const* const la = ra + offset[p] + lane;
                    char const* const lb = rb + offset[p] + lane;
                    u32x4_a4 va{}, vb{};
                    if (x + 4 <= width) {
                        va = *reinterpret_cast<u32x4_a4 const*>(la);
                        vb = *reinterpret_cast<u32x4_a4 const*>(lb);
                    } else {
#pragma unroll
                        for (int k = 0; k < 3; ++k) if (x + k < width) { va[k] = reinterpret_cast<uint32_t const*>(la)[k]; vb[k] = reinterpret_cast<uint32_t const*>(lb)[k]; }
                    }
                    add(p0 + p, va, vb);
                }
            }
        }
    }
    hand_over_sums(acc, setChannels, validChannelMask, blockIdx.x, blocks, groupSize, work);
}

// With a mask channel, or without one for images that the other kernel does not take.  A lane takes PX adjacent texels
// (2 when the width is even: 8-byte loads) of rowsPerWave rows, all pairs of them together, because every channel counts by the mask's, and all
// loads of a row are issued before its arithmetic.
template <int PX, bool MASKED>
__global__ void __launch_bounds__(256)
texel_loss_kernel(uint16_t* __restrict__ a, uint16_t const* __restrict__ b, int width, int height, int setChannels, int rowsPerWave,
                   uint32_t validChannelMask, int maskChannel, int discardMaskedOut, uint32_t gridX, uint32_t blocks, uint32_t groupSize, LossWorkspace work)
{
    constexpr int PAIRS = NTC_HIP_DEV_MAX_CHANNELS / 2;
    int const lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int const x = (blockIdx.x * 64 + lane) * PX;
    int const pairs = setChannels >> 1;
    double acc[NTC_HIP_DEV_MAX_CHANNELS];
#pragma unroll
    for (int c = 0; c < NTC_HIP_DEV_MAX_CHANNELS; ++c) acc[c] = 0.0;
    for (int r = 0; r < rowsPerWave; ++r) {
        int const y = (blockIdx.y * 4 + wave) * rowsPerWave + r;
        if (x >= width || y >= height) continue;             // width is a multiple of PX
        size_t const base = size_t(y) * size_t(width) * size_t(setChannels) + size_t(x) * 2;
        uint32_t va[PAIRS][PX], vb[PAIRS][PX];
#pragma unroll
        for (int p = 0; p < PAIRS; ++p) {
            // no branch around a load (the loads of a row must all be in flight together): pairs the
            // set does not have re-read its last pair, and their sums are dropped at the end
            size_t const at = base + size_t(2 * min(p, pairs - 1)) * size_t(width);
            if constexpr (PX == 2) {
                uint2 const u = *reinterpret_cast<uint2 const*>(a + at), v = *reinterpret_cast<uint2 const*>(b + at);
                va[p][0] = u.x; va[p][1] = u.y; vb[p][0] = v.x; vb[p][1] = v.y;
            } else {
                va[p][0] = *reinterpret_cast<uint32_t const*>(a + at);
                vb[p][0] = *reinterpret_cast<uint32_t const*>(b + at);
            }
        }
        __builtin_amdgcn_sched_barrier(0);                   // keep the loads ahead of the arithmetic
        [[maybe_unused]] bool maskedOut[PX];
        if constexpr (MASKED) {
#pragma unroll
            for (int k = 0; k < PX; ++k) maskedOut[k] = false;
#pragma unroll
            for (int p = 0; p < PAIRS; ++p) {
                if ((maskChannel >> 1) != p || !discardMaskedOut) continue;          // uniform
#pragma unroll
                for (int k = 0; k < PX; ++k) maskedOut[k] = (((maskChannel & 1) ? vb[p][k] >> 16 : vb[p][k]) & 0x7FFFu) == 0;
            }
        }
#pragma unroll
        for (int p = 0; p < PAIRS; ++p) {
            float s0 = 0.f, s1 = 0.f;
#pragma unroll
            for (int k = 0; k < PX; ++k) {
                float a0 = float(__builtin_bit_cast(_Float16, uint16_t(va[p][k])));
                float a1 = float(__builtin_bit_cast(_Float16, uint16_t(va[p][k] >> 16)));
                if constexpr (MASKED) {
                    if ((maskChannel >> 1) == p) {              // uniform; the mask channel is below setChannels
                        if (maskChannel & 1) a1 = a1 > 0.f ? fminf(a1, 1.f) : 0.f;
                        else                 a0 = a0 > 0.f ? fminf(a0, 1.f) : 0.f;
                        uint32_t const clamped = uint32_t(__builtin_bit_cast(uint16_t, _Float16(a0)))
                                               | uint32_t(__builtin_bit_cast(uint16_t, _Float16(a1))) << 16;
                        if (clamped != va[p][k]) *reinterpret_cast<uint32_t*>(a + base + size_t(2 * p) * size_t(width) + size_t(2 * k)) = clamped;
                    }
                }
                float d0 = a0 - float(__builtin_bit_cast(_Float16, uint16_t(vb[p][k])));
                float d1 = a1 - float(__builtin_bit_cast(_Float16, uint16_t(vb[p][k] >> 16)));
                if constexpr (MASKED) {
                    if (maskedOut[k] && maskChannel != 2 * p) d0 = 0.f;
                    if (maskedOut[k] && maskChannel != 2 * p + 1) d1 = 0.f;
                }
                s0 += d0 * d0;
                s1 += d1 * d1;
            }
            acc[2 * p] += double(s0);
            acc[2 * p + 1] += double(s1);
        }
    }
    hand_over_sums(acc, setChannels, validChannelMask, blockIdx.y * gridX + blockIdx.x, blocks, groupSize, work);
}

hipError_t launch_image_loss(uint16_t* a, uint16_t const* b, int width, int height, int setChannels, uint32_t validChannelMask,
                             int maskChannel, int discardMaskedOut, LossWorkspace const& work, hipStream_t stream, hipEvent_t done)
{
    LossGrid const grid = image_loss_grid(width, height, compute_units_of_current_device());
    uint32_t const blocks = grid.x * grid.y;
    // Without a mask: 2^log2Lanes lanes to a row, as few as cover a narrow one with four texels each, all 256 at most.  Rows are
    // divided among the workgroups that are resident together; the others, and those that this leaves no row, hand over zeros.
    int log2Lanes = 0;
    while (log2Lanes < 8 && (4 << log2Lanes) < width) ++log2Lanes;
    uint32_t const together = 256u >> log2Lanes, turns = (uint32_t(height) + together - 1u) / together;
    uint32_t const busy = min(blocks, 4u * uint32_t(compute_units_of_current_device())), rows = (turns + busy - 1u) / busy * together;
    // The other kernel's are images of less than 131072 texels, a trip to memory or two for a workgroup, which it makes with
    // all pairs' loads at once and without a tail of a row (300 x 200 and 150 x 100 of 16 channels 15.5 and 15.2 us, 17.1 and
    // 20.4 by whole rows; 400 x 300 16.3 and 17.7, 512 x 512 18.5 and 16.5); rows of less than four texels; rows beyond 31 bits
    // of offsets; and wide images of few rows, which leave most workgroups none (16384 x 1 30 us, 15.6 the other way;
    // 8192 x 8 22 and 16.5; 4096 x 64 19.5 and 17.1; 2048 x 128, twice the even share, 17.5 and 17.7).
    uint64_t const share = uint64_t(rows) * uint64_t(width), even = uint64_t(width) * uint64_t(height) / busy;
    bool const shared = share <= 2u * (even < 1024u ? 1024u : even);
    if (maskChannel < 0 && width >= 4 && uint64_t(width) * uint64_t(height) >= 131072u && shared && share * uint64_t(setChannels) * 2u < 0x80000000u) {
        auto launch = [&](auto steps, auto pairs, auto odd) {
            uint32_t const units = turns * ((uint32_t(setChannels) / 2u + decltype(pairs)::value - 1u) / decltype(pairs)::value);
            return launch_kernel_with_event<image_loss_kernel<decltype(steps)::value, decltype(pairs)::value, decltype(odd)::value>>(dim3(blocks), dim3(256), 0, stream, done,
                                         a, b, width, height, setChannels, int(units / busy), int(units % busy), log2Lanes, validChannelMask, blocks, grid.groupSize, work);
        };
        // Of the three shapes the one with the fewest trips to memory for a row: whole ones of its steps, then what is left a
        // step at a time.  16 channels of images not read before, by the first, the second and the third shape of
        // 2100 x 2100: -, 68 and 65.5 us; 3500 x 2000 -, 96 and 92.5; 5000 x 3000 180, - and 178; with even shares of rows.
        uint32_t const pairs = uint32_t(setChannels) / 2u, w = uint32_t(width);
        auto const trips = [&](uint32_t steps, uint32_t pairsTogether) {
            return (pairs + pairsTogether - 1u) / pairsTogether * (w / (1024u * steps) + (w % (1024u * steps) + 1023u) / 1024u);
        };
        uint32_t const four = trips(4, 1), two = trips(2, 2), one = trips(1, 4);
        auto of_steps = [&](auto odd) {
            if (four <= two && four <= one) return launch(std::integral_constant<int, 4>{}, std::integral_constant<int, 1>{}, odd);
            if (two <= one) return launch(std::integral_constant<int, 2>{}, std::integral_constant<int, 2>{}, odd);
            return launch(std::integral_constant<int, 1>{}, std::integral_constant<int, 4>{}, odd);
        };
        return (width & 1) == 0 ? of_steps(std::false_type{}) : of_steps(std::true_type{});
    }
    auto launch = [&](auto perLane, auto masked) {
        return launch_kernel_with_event<texel_loss_kernel<decltype(perLane)::value, decltype(masked)::value>>(dim3(grid.x, grid.y), dim3(256), 0, stream, done,
                                     a, b, width, height, setChannels, grid.rowsPerWave, validChannelMask, maskChannel, discardMaskedOut, grid.x, blocks, grid.groupSize, work);
    };
    auto of_width = [&](auto perLane) { return maskChannel >= 0 ? launch(perLane, std::true_type{}) : launch(perLane, std::false_type{}); };
    return (width & 1) == 0 ? of_width(std::integral_constant<int, 2>{}) : of_width(std::integral_constant<int, 1>{});
}

// ---- image difference (src/shaders/ImageDifference.hlsl) -------------------------------------------
//
// A workgroup covers 64 x 64 pixels of the extent, as the reference's does (16 x 16 threads of 4 x 4
// pixels); here lane = column and each wave walks 16 rows, so that the loads of a wave are one
// contiguous row piece.  Every thread adds its 16 squared differences in row order, the 64 lanes
// of a wave are combined by an xor butterfly (offsets 32 ... 1), the four waves in order.  Squares
// and sums are separate fp32 operations (no fused multiply-add).  The workgroup's sums are divided
// by width * height, scaled by 2^16, split into floor and fraction * 2^32 and added to the 64-bit
// accumulators (ImageDifference.hlsl:103-127; the integer atomics make the total independent of
// the order in which workgroups finish).
//
// Images of four channels in one UNORM or float format, the usual ones, are read as whole pixels, all of a thread's
// rows (or as many as 32 registers hold) before any arithmetic, and UNORM8 codes are divided by the corrected
// reciprocal.  A workgroup takes several tiles and adds its 64-bit sums to the accumulators once (four workgroups a compute unit: with eight, the atomics on four addresses add 9 us, with two
// there are too few waves: 4 us).  4096 x 4096 RGBA8:
// 33 us (the bytes take 27), 156 with four byte loads a pixel, one row after the other.
__device__ __forceinline__ float diff_channel(DiffImageArgs const& im, uint8_t const* px, int c)
{
    if (c >= im.numChannels) return c == 3 ? 1.f : 0.f;
    switch (im.format) {
    case NTC_HIP_DEV_FORMAT_UNORM8:  return float(px[c]) / 255.f;
    case NTC_HIP_DEV_FORMAT_UNORM16: return float(reinterpret_cast<uint16_t const*>(px)[c]) / 65535.f;
    case NTC_HIP_DEV_FORMAT_FLOAT16: return float(reinterpret_cast<_Float16 const*>(px)[c]);
    case NTC_HIP_DEV_FORMAT_FLOAT32: return reinterpret_cast<float const*>(px)[c];
    default:                         return float(reinterpret_cast<uint32_t const*>(px)[c]);
    }
}

// A pixel of four channels of FORMAT as dwords, at whatever alignment it has.
template <int FORMAT>
__device__ __forceinline__ void load_pixel(uint8_t const* px, uint32_t (&words)[bytes_per_channel(FORMAT)])
{
    if constexpr (bytes_per_channel(FORMAT) == 1) {
        words[0] = *reinterpret_cast<u32_any const*>(px);
    } else if constexpr (bytes_per_channel(FORMAT) == 2) {
        u32x2_any const v = *reinterpret_cast<u32x2_any const*>(px);
        words[0] = v[0]; words[1] = v[1];
    } else {
        u32x4_any const v = *reinterpret_cast<u32x4_any const*>(px);
        words[0] = v[0]; words[1] = v[1]; words[2] = v[2]; words[3] = v[3];
    }
}
template <int FORMAT>
__device__ __forceinline__ float pixel_channel(uint32_t const (&words)[bytes_per_channel(FORMAT)], int c)
{
    constexpr int BPC = bytes_per_channel(FORMAT);
    uint32_t const w = words[(c * BPC) >> 2] >> (8 * ((c * BPC) & 3));
    if constexpr (FORMAT == NTC_HIP_DEV_FORMAT_UNORM8)       return divide_by_top(float(w & 0xffu), 255.f, 1.f / 255.f);
    else if constexpr (FORMAT == NTC_HIP_DEV_FORMAT_UNORM16) return divide_by_top(float(w & 0xffffu), 65535.f, 1.f / 65535.f);
    else if constexpr (FORMAT == NTC_HIP_DEV_FORMAT_FLOAT16) return float(__builtin_bit_cast(_Float16, uint16_t(w)));
    else                                                     return __builtin_bit_cast(float, w);
}

// A tile's sum as it is added to the accumulators.
__device__ __forceinline__ unsigned long long fixed_share(float total, int width, int height)
{
    total = __fdiv_rn(total, float(width * height));
    total = __fmul_rn(total, 65536.f);
    float const whole = floorf(total);
    // float -> uint32 conversions saturate; a NaN (from NaN pixels) adds nothing
    unsigned long long const high = uint32_t(whole), low = uint32_t(floorf(__fmul_rn(__fsub_rn(total, whole), 4294967296.f)));
    return (high << 32) | low;
}

// FORMAT: of both images, four channels each; 0: any two images.
template <int FORMAT, bool MSLE>
__global__ void __launch_bounds__(256)
image_difference_kernel(ImageDifferenceArgs a, int tilesX, int tiles, int step)
{
    __shared__ float sums[4][4];
    int const lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned long long fixed = 0;                            // threads 0 ... 3: the workgroup's share of a channel's sum
    for (int tile = blockIdx.x; tile < tiles; tile += step) {
        int const tileY = tile / tilesX, tileX = tile - tileY * tilesX;
        int const x = tileX * 64 + lane, yBegin = tileY * 64 + wave * 16;
        float mse[4] = { 0.f, 0.f, 0.f, 0.f };
        auto add_pixel = [&](float const (&t1)[4], float const (&t2)[4]) {
            float diff[4];
#pragma unroll
            for (int c = 0; c < 4; ++c)
                diff[c] = MSLE ? __fsub_rn(logf(fabsf(t1[c]) + 1.f), logf(fabsf(t2[c]) + 1.f)) : __fsub_rn(t1[c], t2[c]);
            if (a.useAlphaThreshold && t1[3] < a.alphaThreshold && t2[3] < a.alphaThreshold) { diff[0] = 0.f; diff[1] = 0.f; diff[2] = 0.f; }
#pragma unroll
            for (int c = 0; c < 4; ++c) mse[c] = __fadd_rn(mse[c], __fmul_rn(diff[c], diff[c]));
        };
        if constexpr (FORMAT != 0) {
            constexpr int BPC = bytes_per_channel(FORMAT), ROWS = BPC == 1 ? 16 : BPC == 2 ? 8 : 4;
            int const xIn = min(x, a.width - 1) + a.left;    // (pixels outside the extent are read inside it and dropped)
            for (int first = 0; first < 16 && yBegin + first < a.height; first += ROWS) {
                uint32_t wa[ROWS][BPC], wb[ROWS][BPC];
#pragma unroll
                for (int r = 0; r < ROWS; ++r) {
                    size_t const y = size_t(min(yBegin + first + r, a.height - 1) + a.top);
                    load_pixel<FORMAT>(a.a.data + y * a.a.rowPitch + size_t(xIn) * a.a.pixelStride, wa[r]);
                    load_pixel<FORMAT>(a.b.data + y * a.b.rowPitch + size_t(xIn) * a.b.pixelStride, wb[r]);
                }
                __builtin_amdgcn_sched_barrier(0);           // keep the loads ahead of the arithmetic
#pragma unroll
                for (int r = 0; r < ROWS; ++r) {
                    if (x >= a.width || yBegin + first + r >= a.height) continue;
                    float t1[4], t2[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c) { t1[c] = pixel_channel<FORMAT>(wa[r], c); t2[c] = pixel_channel<FORMAT>(wb[r], c); }
                    add_pixel(t1, t2);
                }
            }
        } else {
            for (int r = 0; r < 16; ++r) {
                int const y = yBegin + r;
                if (x >= a.width || y >= a.height) continue;
                uint8_t const* const pa = a.a.data + size_t(y + a.top) * a.a.rowPitch + size_t(x + a.left) * a.a.pixelStride;
                uint8_t const* const pb = a.b.data + size_t(y + a.top) * a.b.rowPitch + size_t(x + a.left) * a.b.pixelStride;
                float t1[4], t2[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) { t1[c] = diff_channel(a.a, pa, c); t2[c] = diff_channel(a.b, pb, c); }
                add_pixel(t1, t2);
            }
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float v = mse[c];
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) v = __fadd_rn(v, __shfl_xor(v, off, 64));
            if (lane == 0) sums[wave][c] = v;
        }
        __syncthreads();
        if (threadIdx.x < 4) {
            int const c = threadIdx.x;
            float total = __fadd_rn(__fadd_rn(__fadd_rn(sums[0][c], sums[1][c]), sums[2][c]), sums[3][c]);
            fixed += fixed_share(total, a.width, a.height);
        }
        __syncthreads();
    }
    if (threadIdx.x < 4 && fixed) atomicAdd(a.output + threadIdx.x, fixed);
}

// MSE of pixels of at most eight bytes without padding, in images of many tiles: four waves take four tiles side by side, a
// wave sixteen rows of all four, a lane four columns, 16 bytes a load.  A column's sum is made by one lane in row order as
// above; the butterfly's offsets 32 ... 4 are rotations of a tile's sixteen lanes (what is below the rotation's bit is equal
// by then), 2 and 1 are between a lane's own columns.  TEAMS of four waves share a workgroup's four atomics: a thousand
// workgroups that end together wait for each other's.  Bound by memory.  RGBA8, 2048 x 2048, 3072 x 3072, 4096 x 4096 and
// 8192 x 4096: 11.3, 19.8, 23.7 and 49 us (17.6, 24, 30 and 51 with four-byte loads; one team 26.3 and four 31.4 of the
// third, 48 and 45.5 of the last; a wave to a tile, whose loads are four row pieces a power of two apart, 22 and 27 of the
// second and third); halves, the first three: 14, 27.8 and 39.4 (19.6, 30.3 and 43.5).  MSLE, bound by logarithms, gains
// from more waves, not from wider loads (3072 x 3072 39 us, 47 here), and pixels of four floats are 16-byte loads anyway.
template <int CONTROL> __device__ __forceinline__ float add_rotated(float v)
{
    return __fadd_rn(v, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CONTROL, 0xF, 0xF, true)));
}
template <int FORMAT, int TEAMS>
__global__ void __launch_bounds__(256 * TEAMS, 4)
image_difference_wide_kernel(ImageDifferenceArgs a, int groupsX, int groups, int step)
{
    constexpr int BPC = bytes_per_channel(FORMAT), ROWS = 4 / BPC;
    __shared__ float sums[2][TEAMS][4][16];                  // [turn][team][part][4 * tile + channel]
    __shared__ unsigned long long shares[TEAMS][4];
    int const lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6) & 3, team = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 8);
    float const threshold = a.useAlphaThreshold ? a.alphaThreshold : -__builtin_inff();
    unsigned long long fixed = 0;                            // threads 0 ... 15: the workgroup's share of a channel's sum, of the nth tiles
    int turn = 0;
    for (int base = blockIdx.x * TEAMS; base < groups; base += step, turn ^= 1) {
        int const group = base + team;                       // (beyond the last one: below the extent, nothing is read)
        int const groupY = group / groupsX, groupX = group - groupY * groupsX;
        int const x = groupX * 256 + lane * 4, y = groupY * 64 + wave * 16;
        float mse[4][4];                                     // [column][channel]
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int c = 0; c < 4; ++c) mse[i][c] = 0.f;
        u32x4_any wordsA[ROWS][BPC], wordsB[ROWS][BPC];      // rows of four pixels: a row gone through is loaded over
        auto const add_row = [&](int r, int columns) {
            __builtin_amdgcn_sched_barrier(0);               // (a row at a time, or the channels of more pixels than there are registers for)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (i >= columns) break;
                uint32_t wa[BPC], wb[BPC];
#pragma unroll
                for (int d = 0; d < BPC; ++d) { int const at = i * BPC + d; wa[d] = wordsA[r][at >> 2][at & 3]; wb[d] = wordsB[r][at >> 2][at & 3]; }
                float t1[4], t2[4], diff[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    t1[c] = pixel_channel<FORMAT>(wa, c); t2[c] = pixel_channel<FORMAT>(wb, c);
                    diff[c] = __fsub_rn(t1[c], t2[c]);
                }
                if (t1[3] < threshold && t2[3] < threshold) { diff[0] = 0.f; diff[1] = 0.f; diff[2] = 0.f; }
#pragma unroll
                for (int c = 0; c < 4; ++c) mse[i][c] = __fadd_rn(mse[i][c], __fmul_rn(diff[c], diff[c]));
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        if (groupX * 256 + 256 <= a.width && groupY * 64 + 64 <= a.height) {
            uint8_t const* pa = a.a.data + size_t(y + a.top) * a.a.rowPitch + size_t(x + a.left) * (4 * BPC);
            uint8_t const* pb = a.b.data + size_t(y + a.top) * a.b.rowPitch + size_t(x + a.left) * (4 * BPC);
            auto const load = [&](int r) {
#pragma unroll
                for (int v = 0; v < BPC; ++v) {
                    wordsA[r][v] = reinterpret_cast<u32x4_any const*>(pa)[v];
                    wordsB[r][v] = reinterpret_cast<u32x4_any const*>(pb)[v];
                }
                pa += a.a.rowPitch; pb += a.b.rowPitch;
            };
#pragma unroll
            for (int r = 0; r < ROWS; ++r) load(r);
#pragma unroll 1
            for (int first = 0; first < 16; first += ROWS) {
#pragma unroll
                for (int r = 0; r < ROWS; ++r) {
                    add_row(r, 4);
                    if (first + ROWS < 16) load(r);
                }
            }
        } else {
            int const columns = a.width - x;                 // (pixels outside the extent are read inside it and dropped)
#pragma unroll 1
            for (int first = 0; first < 16 && y + first < a.height; first += ROWS) {
#pragma unroll
                for (int r = 0; r < ROWS; ++r) {
                    size_t const row = size_t(min(y + first + r, a.height - 1) + a.top);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        size_t const column = size_t(min(x + i, a.width - 1) + a.left) * (4 * BPC);
                        uint32_t wa[BPC], wb[BPC];
                        load_pixel<FORMAT>(a.a.data + row * a.a.rowPitch + column, wa);
                        load_pixel<FORMAT>(a.b.data + row * a.b.rowPitch + column, wb);
#pragma unroll
                        for (int d = 0; d < BPC; ++d) { int const at = i * BPC + d; wordsA[r][at >> 2][at & 3] = wa[d]; wordsB[r][at >> 2][at & 3] = wb[d]; }
                    }
                }
#pragma unroll
                for (int r = 0; r < ROWS; ++r) add_row(r, y + first + r < a.height ? columns : 0);
            }
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = add_rotated<0x121>(add_rotated<0x122>(add_rotated<0x124>(add_rotated<0x128>(mse[i][c]))));
            float const sum = __fadd_rn(__fadd_rn(v[0], v[2]), __fadd_rn(v[1], v[3]));
            if ((lane & 15) == c) sums[turn][team][wave][4 * (lane >> 4) + c] = sum;
        }
        __syncthreads();                                     // (the next turn's sums lie elsewhere, and the one after it is behind the next barrier)
        if (wave == 0 && lane < 16) {
            float const (&of)[4][16] = sums[turn][team];
            fixed += fixed_share(__fadd_rn(__fadd_rn(__fadd_rn(of[0][lane], of[1][lane]), of[2][lane]), of[3][lane]), a.width, a.height);
        }
    }
    if (wave == 0 && lane < 16) {
        fixed += __shfl_down(fixed, 8, 16);
        fixed += __shfl_down(fixed, 4, 16);
        if (lane < 4) shares[team][lane] = fixed;
    }
    if constexpr (TEAMS > 1) __syncthreads();
    if (threadIdx.x < 4) {
#pragma unroll
        for (int t = 1; t < TEAMS; ++t) fixed += shares[t][lane];
        if (fixed) atomicAdd(a.output + threadIdx.x, fixed);
    }
}

hipError_t launch_image_difference(ImageDifferenceArgs const& a, hipStream_t stream)
{
    int const tilesX = (a.width + 63) / 64, tiles = tilesX * ((a.height + 63) / 64);
    int const resident = 4 * compute_units_of_current_device();
    int const workgroups = tiles < resident ? tiles : resident;
    auto of_format = [&](auto format) {
        constexpr int FORMAT = decltype(format)::value;
        if constexpr (FORMAT != 0 && bytes_per_channel(FORMAT) <= 2) {
            constexpr uint64_t PIXEL = 4 * bytes_per_channel(FORMAT);
            int const groupsX = (a.width + 255) / 256, groups = groupsX * ((a.height + 63) / 64);
            // (with fewer groups of tiles than compute units the other kernel's are more waves: 2048 x 1024 11.2 us)
            if (!a.useMSLE && groups >= compute_units_of_current_device() && a.a.pixelStride == PIXEL && a.b.pixelStride == PIXEL)
                return groups < resident ? launch_kernel<image_difference_wide_kernel<FORMAT, 1>>(dim3(groups), dim3(256), 0, stream, a, groupsX, groups, groups)
                                         : launch_kernel<image_difference_wide_kernel<FORMAT, 2>>(dim3(resident / 2), dim3(512), 0, stream, a, groupsX, groups, resident);
        }
        return a.useMSLE ? launch_kernel<image_difference_kernel<FORMAT, true>>(dim3(workgroups), dim3(256), 0, stream, a, tilesX, tiles, workgroups)
                         : launch_kernel<image_difference_kernel<FORMAT, false>>(dim3(workgroups), dim3(256), 0, stream, a, tilesX, tiles, workgroups);
    };
    bool const alike = a.a.format == a.b.format && a.a.numChannels == 4 && a.b.numChannels == 4;
    switch (alike ? a.a.format : 0) {
    case NTC_HIP_DEV_FORMAT_UNORM8:  return of_format(std::integral_constant<int, NTC_HIP_DEV_FORMAT_UNORM8>{});
    case NTC_HIP_DEV_FORMAT_UNORM16: return of_format(std::integral_constant<int, NTC_HIP_DEV_FORMAT_UNORM16>{});
    case NTC_HIP_DEV_FORMAT_FLOAT16: return of_format(std::integral_constant<int, NTC_HIP_DEV_FORMAT_FLOAT16>{});
    case NTC_HIP_DEV_FORMAT_FLOAT32: return of_format(std::integral_constant<int, NTC_HIP_DEV_FORMAT_FLOAT32>{});
    default:                         return of_format(std::integral_constant<int, 0>{});
    }
}

template <int FORMAT>
static hipError_t launch_read_format(ReadChannelsArgs const& a, dim3 grid, bool plain, hipStream_t stream)
{
    return plain ? launch_kernel<read_channels_kernel<FORMAT, true>>(grid, dim3(256), 0, stream, a)
                 : launch_kernel<read_channels_kernel<FORMAT, false>>(grid, dim3(256), 0, stream, a);
}

template <int FORMAT>
static hipError_t launch_read_groups_of(GroupsArgs const& args, int dstChannels, bool dithering, GroupLaunch const& plan, hipStream_t stream)
{
    auto launch = [&](auto channels) -> hipError_t {
        constexpr int CHANNELS = decltype(channels)::value;
        if constexpr (CHANNELS * bytes_per_channel(FORMAT) <= 8) {
            constexpr bool unorm = FORMAT == NTC_HIP_DEV_FORMAT_UNORM8 || FORMAT == NTC_HIP_DEV_FORMAT_UNORM16;   // (dithering changes only these)
            if (unorm && dithering) return launch_kernel<read_groups_kernel<FORMAT, CHANNELS, unorm>>(dim3(plan.grid.step), dim3(plan.threads), plan.ldsBytes, stream, args);
            return launch_kernel<read_groups_kernel<FORMAT, CHANNELS, false>>(dim3(plan.grid.step), dim3(plan.threads), plan.ldsBytes, stream, args);
        } else {
            return hipErrorInvalidValue;
        }
    };
    switch (dstChannels) {
    case 1: return launch(std::integral_constant<int, 1>{});
    case 2: return launch(std::integral_constant<int, 2>{});
    case 3: return launch(std::integral_constant<int, 3>{});
    case 4: return launch(std::integral_constant<int, 4>{});
    case 5: return launch(std::integral_constant<int, 5>{});
    case 6: return launch(std::integral_constant<int, 6>{});
    case 7: return launch(std::integral_constant<int, 7>{});
    case 8: return launch(std::integral_constant<int, 8>{});
    default: return hipErrorInvalidValue;
    }
}

static hipError_t launch_read_groups(ReadChannelsArgs const& a, hipStream_t stream)
{
    GroupLaunch const plan = plan_groups(a.width, a.height, a.srcColorSpaces, a.dstColorSpaces, a.numChannels < a.dstChannels ? a.numChannels : a.dstChannels, true);
    GroupsArgs const args{ const_cast<uint16_t*>(a.planarPairs), a.dst, a.rowPitch, a.width, a.height, plan.grid, plan.transfers,
                           uint8_t(a.setChannels), uint8_t(a.firstChannel), uint8_t(a.numChannels), a.dstColorSpaces[3], 0 };
    bool const dithering = a.useDithering != 0;
    switch (a.format) {
    case NTC_HIP_DEV_FORMAT_UNORM8:  return launch_read_groups_of<NTC_HIP_DEV_FORMAT_UNORM8>(args, a.dstChannels, dithering, plan, stream);
    case NTC_HIP_DEV_FORMAT_UNORM16: return launch_read_groups_of<NTC_HIP_DEV_FORMAT_UNORM16>(args, a.dstChannels, dithering, plan, stream);
    case NTC_HIP_DEV_FORMAT_FLOAT16: return launch_read_groups_of<NTC_HIP_DEV_FORMAT_FLOAT16>(args, a.dstChannels, dithering, plan, stream);
    case NTC_HIP_DEV_FORMAT_FLOAT32: return launch_read_groups_of<NTC_HIP_DEV_FORMAT_FLOAT32>(args, a.dstChannels, dithering, plan, stream);
    case NTC_HIP_DEV_FORMAT_UINT32:  return launch_read_groups_of<NTC_HIP_DEV_FORMAT_UINT32>(args, a.dstChannels, dithering, plan, stream);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_read_channels(ReadChannelsArgs const& args, hipStream_t stream)
{
    ReadChannelsArgs a = args;
    if (a.dstWidth > 0) {                                    // resampling copy
        dim3 const grid((a.dstWidth + 63) / 64, (a.dstHeight + 3) / 4);
        switch (a.format) {
        case NTC_HIP_DEV_FORMAT_UNORM8:  return launch_kernel<read_channels_resize_kernel<NTC_HIP_DEV_FORMAT_UNORM8>>(grid, dim3(256), 0, stream, a);
        case NTC_HIP_DEV_FORMAT_UNORM16: return launch_kernel<read_channels_resize_kernel<NTC_HIP_DEV_FORMAT_UNORM16>>(grid, dim3(256), 0, stream, a);
        case NTC_HIP_DEV_FORMAT_FLOAT16: return launch_kernel<read_channels_resize_kernel<NTC_HIP_DEV_FORMAT_FLOAT16>>(grid, dim3(256), 0, stream, a);
        case NTC_HIP_DEV_FORMAT_FLOAT32: return launch_kernel<read_channels_resize_kernel<NTC_HIP_DEV_FORMAT_FLOAT32>>(grid, dim3(256), 0, stream, a);
        case NTC_HIP_DEV_FORMAT_UINT32:  return launch_kernel<read_channels_resize_kernel<NTC_HIP_DEV_FORMAT_UINT32>>(grid, dim3(256), 0, stream, a);
        default: return hipErrorInvalidValue;
        }
    }
    if (a.dstChannels * bytes_per_channel(a.format) <= 8) return launch_read_groups(a, stream);
    dim3 const grid = copy_grid(a.width, a.height, a.xShift);
    bool const plain = plain_copy(a.srcColorSpaces, a.dstColorSpaces, a.useDithering);
    switch (a.format) {
    case NTC_HIP_DEV_FORMAT_UNORM8:  return launch_read_format<NTC_HIP_DEV_FORMAT_UNORM8>(a, grid, plain, stream);
    case NTC_HIP_DEV_FORMAT_UNORM16: return launch_read_format<NTC_HIP_DEV_FORMAT_UNORM16>(a, grid, plain, stream);
    case NTC_HIP_DEV_FORMAT_FLOAT16: return launch_read_format<NTC_HIP_DEV_FORMAT_FLOAT16>(a, grid, plain, stream);
    case NTC_HIP_DEV_FORMAT_FLOAT32: return launch_read_format<NTC_HIP_DEV_FORMAT_FLOAT32>(a, grid, plain, stream);
    case NTC_HIP_DEV_FORMAT_UINT32:  return launch_read_format<NTC_HIP_DEV_FORMAT_UINT32>(a, grid, plain, stream);
    default: return hipErrorInvalidValue;
    }
}

// ---------------------------------------------------------------------------------------------
// Byte fill (what a memset does, as a kernel: the library clears memory only this way).  The
// 16-byte-aligned middle goes out as uint4 stores, the unaligned ends byte by byte.
__global__ void __launch_bounds__(256)
fill_kernel(uint8_t* dst, uint32_t pattern, uint64_t headBytes, uint64_t vectors, uint64_t tailBytes)
{
    uint64_t const stride = uint64_t(gridDim.x) * blockDim.x, first = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    uint4* const body = reinterpret_cast<uint4*>(dst + headBytes);
    for (uint64_t i = first; i < vectors; i += stride) body[i] = make_uint4(pattern, pattern, pattern, pattern);
    if (first < headBytes) dst[first] = uint8_t(pattern);
    if (first < tailBytes) dst[headBytes + vectors * 16u + first] = uint8_t(pattern);
}

hipError_t launch_fill(uint8_t* dst, uint8_t value, uint64_t bytes, hipStream_t stream)
{
    if (bytes == 0) return hipSuccess;
    uint64_t const misaligned = reinterpret_cast<uintptr_t>(dst) & 15u;
    uint64_t const headBytes = misaligned ? (16u - misaligned < bytes ? 16u - misaligned : bytes) : 0u;
    uint64_t const vectors = (bytes - headBytes) / 16u, tailBytes = bytes - headBytes - vectors * 16u;
    uint64_t const groups = (vectors + 255u) / 256u;
    uint32_t const grid = uint32_t(groups < 1u ? 1u : (groups > 16384u ? 16384u : groups));
    hipLaunchKernelGGL(fill_kernel, dim3(grid), dim3(256), 0, stream, dst, uint32_t(value) * 0x01010101u, headBytes, vectors, tailBytes);
    return hipGetLastError();
}

} // namespace ntc_hip_dev
