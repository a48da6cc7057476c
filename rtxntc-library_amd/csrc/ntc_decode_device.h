// ntc_decode_device.h - device helpers shared by the decode kernels (int8 network: ntc_decode_kernel.hip,
// FP8 network: ntc_decode_fp8_kernel.hip): vector types, latent loads, the float sampling footprint, output
// conversion and the stores of one wave tile.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "ntc_decode_kernel.h"
#include "ntc_launch.h"
#include <type_traits>

namespace ntc_hip_dev {

typedef int   v4i __attribute__((ext_vector_type(4)));
// Latent grids live in global memory; saying so lets loads use "scalar base + 32-bit lane offset"
// addressing instead of 64-bit flat addresses built per lane.
typedef __attribute__((address_space(1))) uint16_t const* GlobalU16Ptr;
typedef __attribute__((address_space(1))) uint8_t const*  GlobalU8Ptr;

// One u16 at a uniform base plus a 32-bit byte offset per lane (global_load_ushort v, v_off, s[base]).
__device__ __forceinline__ uint32_t load_u16(GlobalU8Ptr base, uint32_t byteOffset)
{
    return *reinterpret_cast<GlobalU16Ptr>(base + byteOffset);
}

// 24-bit multiply, full rate.  Inline assembly because the compiler turns the builtin back into the
// quarter-rate 32-bit multiply in places.  Only for the input stages: the compiler inserts the wait states that
// matrix instructions in flight need around instructions it can see, and an assembly statement is opaque to it.
// The input stage of a tile runs when none is in flight - after the previous tile's results were read for
// its stores and before this tile's first matrix instruction, in a basic block of its own.
__device__ __forceinline__ uint32_t mul24(uint32_t a, uint32_t b)
{
    uint32_t r;
    asm("v_mul_u32_u24 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// Footprint of one axis of a bilinear tap pair in integers, for power-of-two sizes: with
// p = u*grid - 1/2 = N / 2^n, N = ((2x+1) << shl) - (1 << sublog) (the packed axis word of DevMip),
// floor and fraction are a shift and a mask, and the two cells wrap by masking.
struct AxisFoot { uint32_t c0, c1, f; };

__device__ __forceinline__ AxisFoot axis_fast(int x, uint32_t packedAxis, int gridSize)
{
    int const shl = int(packedAxis & 0xffu), n = int((packedAxis >> 8) & 0xffu), sublog = int((packedAxis >> 16) & 0xffu);
    int const N = ((2 * x + 1) << shl) - (1 << sublog);
    int const b = N >> n;                                    // arithmetic shift = floor
    AxisFoot a;
    a.f = uint32_t(N) & ((1u << n) - 1u);
    a.c0 = uint32_t(b) & uint32_t(gridSize - 1);             // wrap addressing
    a.c1 = uint32_t(b + 1) & uint32_t(gridSize - 1);
    return a;
}

// 24-bit multiply-add, full rate: a * b + c.  Input stages only, like mul24.
__device__ __forceinline__ uint32_t mad24(uint32_t a, uint32_t b, uint32_t c)
{
    uint32_t r;
    asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kWaveTexels  = 64;

// The entries of a launch's table, which is the kernel's FIRST argument.  The arguments are addressed where they lie:
// indexed as a by-value parameter the table would be copied to scratch first.  Both sources are constant memory for
// the whole launch, so uniform reads stay scalar loads.
__device__ __forceinline__ DevMip const* table_entries(DevMip const* entries)
{
    typedef __attribute__((address_space(4))) DevMip const* ConstantMips;
    ConstantMips const inlined = (ConstantMips)__builtin_amdgcn_kernarg_segment_ptr();
    ConstantMips const stored = (ConstantMips)(uintptr_t)entries;
    return (DevMip const*)(entries ? stored : inlined);
}

// Launches a kernel whose first argument is the table, and no other kind: that is what table_entries() relies on.
template <class Kernel> struct TableFirst { static constexpr bool value = false; };
template <class... Others> struct TableFirst<void (*)(MipTable, Others...)> { static constexpr bool value = true; };
static_assert(std::is_standard_layout_v<MipTable> && std::is_trivially_copyable_v<MipTable>, "offsets in a kernel's arguments are those of the struct");
template <auto KERNEL, class... ARGS>
inline hipError_t launch_with_table(dim3 grid, dim3 block, size_t ldsBytes, hipStream_t stream, MipTable const& table, ARGS const&... args)
{
    static_assert(TableFirst<decltype(KERNEL)>::value, "the table lies where the arguments begin");
    return launch_kernel<KERNEL>(grid, block, ldsBytes, stream, table, args...);
}

// ---- small device helpers -----------------------------------------------------------

// ---- sampling footprints in floats: any sizes --------------------------------------------------
//
// FeatureGrid::SetupBilinearFilter (src/FeatureGridDevice.h:51-57) with wrap addressing.  The results are defined by
// these binary32 operations; what could be shortened without changing a bit is the division, the wrap, the unpacking of
// the cells and the addresses (32-bit offsets from scalar bases, all loads of a texel in flight before the first is
// used): 1920 x 1080 texels of sixteen features, sixteen channels, took 91 us with divisions, 64-bit addresses per lane
// and a wait for each grid, 83 now (71 for the integer stage on as many texels).

// The middle of a texel: (x + 1/2) / size, as correctly rounded as the division: an integer below 2^17 over one of at
// most 2^17 (times powers of two) lies at least 2^-42 of itself away from the middle between two numbers, and the
// corrected quotient of a refined reciprocal is within 2^-45 before its last rounding.
__device__ __forceinline__ float texel_centre(int x, int size)
{
    float const a = float(x) + 0.5f, b = float(size);
    float r = __builtin_amdgcn_rcpf(b);
    r = __builtin_fmaf(__builtin_fmaf(-b, r, 1.f), r, r);
    float const q = a * r;
    return __builtin_fmaf(__builtin_fmaf(-q, b, a), r, q);
}

__device__ __forceinline__ uint32_t umin3(uint32_t a, uint32_t b, uint32_t c)
{
    uint32_t r;
    asm("v_min3_u32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// One axis: the two cells and the second one's weight.
struct FloatAxis { uint32_t c0, c1; float d; };
__device__ __forceinline__ FloatAxis axis_general(float u, int gridSize)
{
    float const x = u * float(gridSize) - 0.5f;
    float const fx = floorf(x);
    FloatAxis a;
    a.d = x - fx;
    // u lies in (0, 1), so the floor is in [-1, gridSize - 1] (gridSize itself only through rounding); a negative number
    // is a large unsigned one, so the smallest of c, c + gridSize, c - gridSize is the wrapped cell
    uint32_t const c = uint32_t(int(fx)), g = uint32_t(gridSize);
    a.c0 = umin3(c, c + g, c - g);
    a.c1 = min(a.c0 + 1u, a.c0 + 1u - g);
    return a;
}

// The four taps' weights as filter4 takes them: times 2^24 and 2^20.
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
struct FloatTaps {
    float lower[4], upper[4];
    __device__ __forceinline__ FloatTaps(FloatAxis const& x, FloatAxis const& y)
    {
        float const x0 = (1.f - x.d) * 0x1p24f, x1 = x.d * 0x1p24f, y0 = 1.f - y.d, y1 = y.d;
        lower[0] = x0 * y0; lower[1] = x1 * y0; lower[2] = x0 * y1; lower[3] = x1 * y1;
#pragma unroll
        for (int k = 0; k < 4; ++k) upper[k] = lower[k] * 0x1p-4f;
    }
};

// The cells of all layers at the four taps.  (Grids whose layers reach beyond 32-bit byte offsets take 64-bit ones.)
template <int LAYERS>
__device__ __forceinline__ void load_cells(uint16_t const* grid, int gridWidth, int gridHeight, FloatAxis const& x, FloatAxis const& y, uint32_t (&cells)[LAYERS][4])
{
    uint64_t const layerBytes = uint64_t(uint32_t(gridWidth)) * uint32_t(gridHeight) * 2u;
    if (layerBytes >> 32) {
        GlobalU16Ptr const g = (GlobalU16Ptr)grid;
        size_t const r0 = size_t(y.c0) * uint32_t(gridWidth), r1 = size_t(y.c1) * uint32_t(gridWidth);
#pragma unroll
        for (int L = 0; L < LAYERS; ++L) {
            GlobalU16Ptr const layer = g + L * (layerBytes / 2);
            cells[L][0] = layer[r0 + x.c0]; cells[L][1] = layer[r0 + x.c1]; cells[L][2] = layer[r1 + x.c0]; cells[L][3] = layer[r1 + x.c1];
        }
        return;
    }
    GlobalU8Ptr const g = (GlobalU8Ptr)grid;
    uint32_t const r0 = y.c0 * uint32_t(gridWidth), r1 = y.c1 * uint32_t(gridWidth);
    uint32_t const a00 = (r0 + x.c0) << 1, a10 = (r0 + x.c1) << 1, a01 = (r1 + x.c0) << 1, a11 = (r1 + x.c1) << 1;
#pragma unroll
    for (int L = 0; L < LAYERS; ++L) {
        GlobalU8Ptr const layer = g + L * layerBytes;
        cells[L][0] = load_u16(layer, a00); cells[L][1] = load_u16(layer, a10); cells[L][2] = load_u16(layer, a01); cells[L][3] = load_u16(layer, a11);
    }
}

// Four 4-bit features of the four taps, filtered.  A cell c = f0 | f1<<4 | f2<<8 | f3<<12.  The bits 0 to 3 of a half
// are a subnormal, the number they hold times 2^-24, the bits 4 to 7 sixteen times that: multiplied by a weight times 2^24
// or 2^20 either gives the products and the roundings of the feature itself, and the multiply-add that takes halves needs no
// conversion.  Two cells to a dword, a mask for each feature of the two, and the two upper ones shifted by a byte: 28
// instructions a layer for 40 when bytes were converted (with the floors below 1920 x 1080 of sixteen features decoded in
// 95.4 us for 98.9, 1500 x 900 with e4m3 weights in 88.5 for 91.9; the FP8 network, bound otherwise, as before).
__device__ __forceinline__ void filter4(FloatTaps const& tp, uint32_t const (&cells)[4], float (&t)[4])
{
    uint32_t two[2] = { cells[0] | cells[1] << 16, cells[2] | cells[3] << 16 };
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float const* const w = (i & 1) ? tp.upper : tp.lower;
        if (i == 2) { two[0] >>= 8; two[1] >>= 8; }
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            v2h const h = __builtin_bit_cast(v2h, two[k >> 1] & ((i & 1) ? 0x00f000f0u : 0x000f000fu));
            s = __builtin_fmaf(w[k], float(h[k & 1]), s);
        }
        t[i] = s;
    }
}

// The floors of four numbers below 256, given times 2^-24, as bytes: rounded towards zero to a half, such a number is a
// subnormal whose bits are its floor.  Two conversions and a permutation for four floors and four conversions.
__device__ __forceinline__ uint32_t floors_of(float a, float b, float c, float d)
{
    uint32_t const low = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a, b)), high = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(c, d));
    return __builtin_amdgcn_perm(high, low, 0x06040200u);
}

// floor(17 * t) - 128 for four features at once, returned as four packed bytes.
__device__ __forceinline__ uint32_t bilinear4(FloatTaps const& tp, uint32_t const (&cells)[4])
{
    float t[4];
    filter4(tp, cells, t);
    constexpr float k = 17.f * 0x1p-24f;
    return floors_of(t[0] * k, t[1] * k, t[2] * k, t[3] * k) ^ 0x80808080u;  // -128 on every byte
}

typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float    v2f __attribute__((ext_vector_type(2)));

// ---- weights ------------------------------------------------------------------------------------

// Four OCP e4m3 (1-4-3, bias 7, no infinities) bytes -> the integers 512*value (the conversion is exact and so is the
// product: at most 448 * 512).  The two NaN encodings decode as 0.
__device__ __forceinline__ void e4m3_times_512(uint32_t bytes, int32_t (&w)[4])
{
    v2f const lo = __builtin_amdgcn_cvt_pk_f32_fp8(int(bytes), false), hi = __builtin_amdgcn_cvt_pk_f32_fp8(int(bytes), true);
    float const f[4] = { lo[0], lo[1], hi[0], hi[1] };
#pragma unroll
    for (int r = 0; r < 4; ++r) w[r] = f[r] == f[r] ? int32_t(f[r] * 512.f) : 0;
}

__device__ __forceinline__ uint32_t halves_of_bytes(uint32_t v, int firstByte)     // two int8 -> two fp16 (exact)
{
    v2h const h = { _Float16(int(int8_t(v >> (8 * firstByte)))), _Float16(int(int8_t(v >> (8 * firstByte + 8)))) };
    return __builtin_bit_cast(uint32_t, h);
}

// The lane's number in its wave from the execution mask: no register has to keep the thread id alive for it.
__device__ __forceinline__ int lane_id()
{
    return int(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)));
}

// Two network outputs -> two fp16 in one dword.  The output is an fp32 product that is THEN
// rounded to half (round-nearest-even); a half that would be Inf/NaN is stored as zero
// (IsHalfSpecial, Inference.cu:125-126).  |o| >= 65520 is exactly the set that rounds to
// Inf.  The empty asm keeps the compiler from folding multiply + convert into
// v_fma_mixlo_f16, which rounds the exact product once, straight to half.
// CHECKED = false is for callers that know |a|, |b| stay far below 65520.
template <bool CHECKED = true>
__device__ __forceinline__ uint32_t to_half2_bits(float a, float b)
{
    asm("" : "+v"(a));
    asm("" : "+v"(b));
    if constexpr (CHECKED) {
        a = (__builtin_fabsf(a) < 65520.f) ? a : 0.f;
        b = (__builtin_fabsf(b) < 65520.f) ? b : 0.f;
    }
    v2h const h = __builtin_convertvector(v2f{a, b}, v2h);
    return __builtin_bit_cast(uint32_t, h);
}

// WriteImageChannel UNORM8 (src/ImageProcessing.cu:146-149): u8(clamp(roundf(v * 255), 0, 255)) of
// the stored half.  v*255 is exact in fp32 (11-bit x 8-bit significands).  v_cvt_pk_u8_f32 rounds to nearest
// even and saturates to [0, 255]; that equals roundf (half away from zero) here because the only tie inside
// the range is v = 1/2 (v*255 = k + 1/2 needs 255 | 2k + 1 for a dyadic v): 127.5 -> 128 under both rules.
// The result drops into byte `slot` of `packed`.
__device__ __forceinline__ uint32_t pack_unorm8(_Float16 h, uint32_t slot, uint32_t packed)
{
    return __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(float(h), 255.f, 0.f), slot, packed);
}

typedef __attribute__((address_space(1))) uint8_t* GlobalOutPtr;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// A uniform 64-bit address, pinned to scalar registers so that stores take the "scalar base + 32-bit lane
// offset" form instead of a 64-bit address computed per lane.
__device__ __forceinline__ GlobalOutPtr uniform_pointer(uint64_t address)
{
    uint32_t const lo = __builtin_amdgcn_readfirstlane(uint32_t(address));
    uint32_t const hi = __builtin_amdgcn_readfirstlane(uint32_t(address >> 32));
    return (GlobalOutPtr)((uint64_t(hi) << 32) | lo);
}

// Stores of one 16-texel block row.  `row` is uniform (start of image row y in the output), `laneOff` the
// lane's byte offset inside the row (`laneOff2` that of the second channel pair of planar output), h01/h23 the
// lane's four channels as halves.  Four channels of a pixel go out as one store at whatever alignment the pixels have,
// fewer as up to two.
typedef __attribute__((address_space(1))) uint16_t* GlobalHalfOutPtr;
typedef uint32_t __attribute__((aligned(1))) u32_any;
typedef uint16_t __attribute__((aligned(1))) u16_any;
typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t __attribute__((aligned(2))) u32_a2;
typedef __attribute__((address_space(1))) u32_any*  GlobalU32AnyPtr;
typedef __attribute__((address_space(1))) u16_any*  GlobalU16AnyPtr;
typedef __attribute__((address_space(1))) u32x2_a2* GlobalU32x2A2Ptr;
typedef __attribute__((address_space(1))) u32_a2*   GlobalU32A2OutPtr;

// One to three channels of a pixel format (`count` uniform in the lanes that are active): u8 as packed bytes.
__device__ __forceinline__ void store_few_bytes(GlobalOutPtr dst, uint32_t u8, int count)
{
    if (count & 2) { *reinterpret_cast<GlobalU16AnyPtr>(dst) = uint16_t(u8); u8 >>= 16; dst += 2; }
    if (count & 1) *dst = uint8_t(u8);
}
__device__ __forceinline__ void store_few_halves(GlobalOutPtr dst, uint32_t h01, uint32_t h23, int count)
{
    if (count & 2) { *reinterpret_cast<GlobalU32A2OutPtr>(dst) = h01; h01 = h23; dst += 4; }
    if (count & 1) *reinterpret_cast<GlobalHalfOutPtr>(dst) = uint16_t(h01);
}

__device__ __forceinline__ uint32_t unorm8_of_halves(uint32_t h01, uint32_t h23)
{
    v2h const a = __builtin_bit_cast(v2h, h01), b = __builtin_bit_cast(v2h, h23);
    return pack_unorm8(b[1], 3, pack_unorm8(b[0], 2, pack_unorm8(a[1], 1, pack_unorm8(a[0], 0, 0u))));
}

template <int FORMAT>
__device__ __forceinline__ void store_channels(GlobalOutPtr row, uint32_t laneOff, uint32_t laneOff2,
                                               uint32_t h01, uint32_t h23, int nch)
{
    GlobalOutPtr const dst = row + laneOff;
    if constexpr (FORMAT == NTC_HIP_DEV_OUT_FP16_PLANAR_PAIRS) {
        // src/RegressionKernels.h:36-45; whole half2 pairs (Inference.cu:131-134)
        *reinterpret_cast<__attribute__((address_space(1))) uint32_t*>(dst) = h01;
        if (nch > 2) *reinterpret_cast<__attribute__((address_space(1))) uint32_t*>(row + laneOff2) = h23;
    } else if constexpr (FORMAT == NTC_HIP_DEV_OUT_FP16_PIXELS) {
        if (nch == 4) *reinterpret_cast<GlobalU32x2A2Ptr>(dst) = u32x2_a2{ h01, h23 };
        else          store_few_halves(dst, h01, h23, nch);
    } else {
        uint32_t const u8 = unorm8_of_halves(h01, h23);
        if (nch == 4) *reinterpret_cast<GlobalU32AnyPtr>(dst) = u8;
        else          store_few_bytes(dst, u8, nch);
    }
}

// What the tile loop and the stores need of a mip for every tile, held by value (in scalar registers) for a run
// of tiles of one mip; the input stages read the rest through `full`.
struct RunMip {
    DevMip const& full;
    uint8_t* out;
    uint64_t outRowPitch;
    int32_t width, height, numChannels, outPixelStride, outFormat;
    uint32_t fast;
    __device__ __forceinline__ explicit RunMip(DevMip const& m)
        : full(m), out(m.out), outRowPitch(m.outRowPitch), width(m.width), height(m.height), numChannels(m.numChannels),
          outPixelStride(m.outPixelStride), outFormat(m.outFormat), fast(m.fast) {}
};

// Look-ups in the table of a decode call (one entry per mip of every set, sorted by tileStart).  Both go through
// the table a wave at a time - one load per lane and a ballot - where a loop over the entries pays a memory round
// trip for each: a workgroup does this once per segment of its share, twelve entries further for a full mip chain.
// Every wave computes the same, uniform, result.  Used by decode_fp8_kernel (-0.6 % on a 4096 x 4096 decode) and by the
// kernels for few tiles.  decode_kernel finds the first entry of a table in its arguments by inlined_entry_of(), and keeps
// the plain loops for longer tables and for a segment's end: there this took 1.3 % off a batch of eight sets and added 0.3 - 3 %
// to single sets, through the tile loop's register allocation.

// The last entry at or after `entry` whose tiles begin at or before `tile`.
__device__ __forceinline__ int table_entry_of(DevMip const* __restrict__ mips, int numMips, int entry, int tile)
{
    int const lane = threadIdx.x & 63;
    for (int base = entry + 1; base < numMips; base += 64) {
        int const k = base + lane;
        bool const before = k < numMips && mips[k].tileStart <= tile;
        int const n = __popcll(__ballot(before));
        entry += n;
        if (n < 64) break;
    }
    return entry;
}

// Where the tiles that use `blob` (the weights of entry `entry`) end: the first tile of the next entry with other
// weights, at most tileEnd.
__device__ __forceinline__ int segment_end(DevMip const* __restrict__ mips, int numMips, int entry, int tileEnd, uint8_t const* blob)
{
    int const lane = threadIdx.x & 63;
    for (int base = entry + 1; base < numMips; base += 64) {
        int const k = base + lane;
        int start = 0x7fffffff;
        bool other = false;
        if (k < numMips) { start = mips[k].tileStart; other = mips[k].weights != blob; }
        uint64_t const hit = __ballot(other || start >= tileEnd);       // another set's entry, or one beyond the share
        if (hit) return min(tileEnd, __builtin_amdgcn_readlane(start, __ffsll((unsigned long long)hit) - 1));
    }
    return tileEnd;
}

// What a lane's stores of one wave tile share: channel count, byte offsets inside an output row, row size.
template <int FORMAT, class Mip>
struct StorePlace {
    int nch;
    uint32_t laneOff, laneOff2;
    size_t rowBytes;
    __device__ __forceinline__ StorePlace(Mip const& m, int x, int chBase)
    {
        nch = (x < m.width) ? min(4, m.numChannels - chBase) : 0;
        uint32_t const C2 = uint32_t((m.numChannels + 1) & ~1);
        laneOff = (FORMAT == NTC_HIP_DEV_OUT_FP16_PLANAR_PAIRS)
            ? (uint32_t(chBase) * uint32_t(m.width) + uint32_t(x) * 2u) * 2u
            : uint32_t(x) * uint32_t(m.outPixelStride) + uint32_t(chBase) * (FORMAT == NTC_HIP_DEV_OUT_FP16_PIXELS ? 2u : 1u);
        laneOff2 = laneOff + uint32_t(m.width) * 4u;
        rowBytes = (FORMAT == NTC_HIP_DEV_OUT_FP16_PLANAR_PAIRS) ? size_t(m.width) * C2 * 2 : size_t(m.outRowPitch);
    }
};

// The lane's four channels of one texel of image row y (uniform, inside the image): outputs = accumulators times
// scales, rounded to half.
template <int FORMAT, bool CHECKED, class AccV, class Mip>
__device__ __forceinline__ void store_row(Mip const& m, StorePlace<FORMAT, Mip> const& at, AccV D, v4f S, int y)
{
    uint32_t const h01 = to_half2_bits<CHECKED>(float(D[0]) * S[0], float(D[1]) * S[1]);
    uint32_t const h23 = to_half2_bits<CHECKED>(float(D[2]) * S[2], float(D[3]) * S[3]);
    GlobalOutPtr const row = uniform_pointer(reinterpret_cast<uint64_t>(m.out) + size_t(y) * at.rowBytes);
    store_channels<FORMAT>(row, at.laneOff, at.laneOff2, h01, h23, at.nch);
}

// The stores of one wave tile: D[b] holds the lane's four channels of the texel in column `x` of block b, where block
// b of 16 texels begins 16 * (b & 1) texels further right, in row y0 + (b >> 1).
template <int FORMAT, bool CHECKED = true, class Acc, class Mip>
__device__ __forceinline__ void store_tile(Mip const& m, Acc const (&D)[4], v4f S, int x, int y0, int chBase)
{
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        int const y = y0 + (b >> 1);
        if (y >= m.height) break;                            // uniform
        StorePlace<FORMAT, Mip> const at(m, x + 16 * (b & 1), chBase);
        if (at.nch > 0) store_row<FORMAT, CHECKED>(m, at, D[b], S, y);
    }
}

// The stores of a wave tile at an image edge: the general form above, in the mip's format, with the checked conversion
// (it equals the unchecked one wherever that is allowed).  Not inlined: tiles like these are few, and inlined next to
// the fast form the six instantiations cost the kernels registers.
template <class Acc>
__device__ __attribute__((noinline)) void store_tile_general(DevMip const* mip, Acc D0, Acc D1, Acc D2, Acc D3, v4f S, int x, int y0, int chBase)
{
    RunMip const m(*mip);
    Acc const D[4] = { D0, D1, D2, D3 };
    if (m.outFormat == NTC_HIP_DEV_OUT_FP16_PLANAR_PAIRS)  store_tile<NTC_HIP_DEV_OUT_FP16_PLANAR_PAIRS, true>(m, D, S, x, y0, chBase);
    else if (m.outFormat == NTC_HIP_DEV_OUT_FP16_PIXELS)   store_tile<NTC_HIP_DEV_OUT_FP16_PIXELS, true>(m, D, S, x, y0, chBase);
    else                                                   store_tile<NTC_HIP_DEV_OUT_UNORM8_PIXELS, true>(m, D, S, x, y0, chBase);
}

// The stores of a wave tile that lies inside the image: no bounds to test, every lane stores its channels of all four
// blocks (block b: 16 texels from x0 + 16 * (b & 1) in row y0 + (b >> 1)), and the row addresses are one uniform
// base plus multiples of the row size - a handful of scalar additions instead of a 64-bit product, a test and a
// branch per row.  x0, y0: first texel of the wave tile; lane = (j, g) holds channels 4g..4g+3 of texel column j.
//
// A channel count that is no multiple of four leaves the lanes of one group with one to three channels: a second,
// uniform part stores those (planar pairs: the group's first pair only, or both).  1920 x 1080 texels of nine unorm8
// channels took 13 us more than of sixteen planar ones when such mips took the general form, 5 now.
template <int FORMAT, bool CHECKED, class Acc, class Mip>
__device__ __forceinline__ void store_tile_inside(Mip const& m, Acc const (&D)[4], v4f S, int x0, int y0, int j, int g)
{
    typedef __attribute__((address_space(1))) uint32_t* DwordPtr;
    constexpr bool PLANAR = FORMAT == NTC_HIP_DEV_OUT_FP16_PLANAR_PAIRS;
    int const rest = m.numChannels & 3;                                          // uniform
    int const mine = m.numChannels - 4 * g;                                      // channels from the lane's first on
    size_t rowBytes;
    uint32_t laneOff;
    GlobalOutPtr tile;
    if (mine <= 0) return;                                                       // lanes of channel groups the mip does not have
    if constexpr (PLANAR) {
        rowBytes = size_t(m.width) * size_t((m.numChannels + 1) & ~1) * 2;       // fp16, whole pairs
        laneOff = uint32_t(g) * (uint32_t(m.width) * 8u) + uint32_t(j) * 4u;     // (4g * width + 2j) halves
        tile = (GlobalOutPtr)m.out + (size_t(y0) * rowBytes + size_t(x0) * 4);
    } else {
        rowBytes = size_t(m.outRowPitch);
        laneOff = uint32_t(j) * uint32_t(m.outPixelStride) + uint32_t(g) * (FORMAT == NTC_HIP_DEV_OUT_FP16_PIXELS ? 8u : 4u);
        tile = (GlobalOutPtr)m.out + (size_t(y0) * rowBytes + size_t(x0) * size_t(m.outPixelStride));
    }
    uint32_t laneOff2 = laneOff + uint32_t(m.width) * 4u;                        // planar: the lane's second channel pair
    // The offsets stay 32-bit values of this tile (hoisted out of the tile loop they become 64-bit lane addresses, and
    // the stores lose their "scalar base + 32-bit lane offset" form).
    asm volatile("" : "+v"(laneOff), "+v"(laneOff2));
    auto const row_of = [&](int b) -> GlobalOutPtr {
        return tile + size_t(b >> 1) * rowBytes + ((b & 1) ? size_t(16) * (PLANAR ? size_t(4) : size_t(m.outPixelStride)) : size_t(0));
    };
    auto const halves = [&](int b, uint32_t& h01, uint32_t& h23) {
        h01 = to_half2_bits<CHECKED>(float(D[b][0]) * S[0], float(D[b][1]) * S[1]);
        h23 = to_half2_bits<CHECKED>(float(D[b][2]) * S[2], float(D[b][3]) * S[3]);
    };
    if (mine >= 4) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            uint32_t h01, h23;
            halves(b, h01, h23);
            if constexpr (PLANAR) {
                *reinterpret_cast<DwordPtr>(row_of(b) + laneOff) = h01;
                *reinterpret_cast<DwordPtr>(row_of(b) + laneOff2) = h23;
            } else if constexpr (FORMAT == NTC_HIP_DEV_OUT_FP16_PIXELS) {
                *reinterpret_cast<GlobalU32x2A2Ptr>(row_of(b) + laneOff) = u32x2_a2{ h01, h23 };
            } else {
                *reinterpret_cast<GlobalU32AnyPtr>(row_of(b) + laneOff) = unorm8_of_halves(h01, h23);
            }
        }
    }
    if (rest != 0 && mine < 4) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            uint32_t h01, h23;
            halves(b, h01, h23);
            if constexpr (PLANAR) {
                *reinterpret_cast<DwordPtr>(row_of(b) + laneOff) = h01;
                if (rest == 3) *reinterpret_cast<DwordPtr>(row_of(b) + laneOff2) = h23;
            } else if constexpr (FORMAT == NTC_HIP_DEV_OUT_FP16_PIXELS) {
                store_few_halves(row_of(b) + laneOff, h01, h23, rest);
            } else {
                store_few_bytes(row_of(b) + laneOff, unorm8_of_halves(h01, h23), rest);
            }
        }
    }
}

// One row of a wave tile in the mip's own format (checked conversion): the stores of the int8-only network path,
// which produces the wave's four blocks of 16 texels one after the other.
template <class AccV, class Mip>
__device__ __forceinline__ void store_row_any_format(Mip const& m, AccV D, v4f S, int x, int y, int chBase)
{
    if (y >= m.height) return;
    if (m.outFormat == NTC_HIP_DEV_OUT_FP16_PLANAR_PAIRS) {
        StorePlace<NTC_HIP_DEV_OUT_FP16_PLANAR_PAIRS, Mip> const at(m, x, chBase);
        if (at.nch > 0) store_row<NTC_HIP_DEV_OUT_FP16_PLANAR_PAIRS, true>(m, at, D, S, y);
    } else if (m.outFormat == NTC_HIP_DEV_OUT_FP16_PIXELS) {
        StorePlace<NTC_HIP_DEV_OUT_FP16_PIXELS, Mip> const at(m, x, chBase);
        if (at.nch > 0) store_row<NTC_HIP_DEV_OUT_FP16_PIXELS, true>(m, at, D, S, y);
    } else {
        StorePlace<NTC_HIP_DEV_OUT_UNORM8_PIXELS, Mip> const at(m, x, chBase);
        if (at.nch > 0) store_row<NTC_HIP_DEV_OUT_UNORM8_PIXELS, true>(m, at, D, S, y);
    }
}

// ---- random-access decode: pieces shared by the query kernels ----------------------------------

// Two adjacent u16 cells as one 32-bit load (2-byte aligned).
typedef uint32_t __attribute__((aligned(2))) u32_align2;
typedef __attribute__((address_space(1))) u32_align2 const* GlobalU32A2Ptr;

// The query-ordered copy of a grid: bricks of T x T cells (T = 4, or 8 for a one-layer grid),
// [brick row][brick column][cell row][cell column][layer], so that all layers of a cell are one load of 2, 4,
// 6 or 8 bytes and a 2 x 2 footprint usually lies in one or two cache lines.
typedef __attribute__((address_space(1))) u32x2 const* GlobalU32x2Ptr;

// Byte offset of a cell in the brick order: the sum of what its column and its row say, each taken once for two taps.
// (Below 2^32: a grid holds less than 2^31 bytes.)
template <int LAYERS>
__device__ __forceinline__ uint32_t brick_column(uint32_t cx)
{
    constexpr uint32_t T = brick_side_log2(LAYERS), MASK = (1u << T) - 1u;
    return (cx >> T) * uint32_t(brick_bytes(LAYERS)) + (cx & MASK) * uint32_t(2 * LAYERS);
}
template <int LAYERS>
__device__ __forceinline__ uint32_t brick_row(uint32_t cy, uint32_t log2GridWidth)
{
    constexpr uint32_t T = brick_side_log2(LAYERS), MASK = (1u << T) - 1u;
    uint32_t const lgBricksX = log2GridWidth > T ? log2GridWidth - T : 0u;
    return ((cy >> T) << lgBricksX) * uint32_t(brick_bytes(LAYERS)) + (cy & MASK) * uint32_t(2 * LAYERS << T);
}

template <int LAYERS> __device__ __forceinline__ void load_brick_cell(GlobalU8Ptr base, uint32_t off, uint32_t (&out)[2]);
// The cells of the four taps: (x0, y0), (x1, y0), (x0, y1), (x1, y1).
template <int LAYERS>
__device__ __forceinline__ void load_brick_cells(GlobalU8Ptr base, uint32_t x0, uint32_t x1, uint32_t y0, uint32_t y1, uint32_t log2GridWidth, uint32_t (&out)[4][2])
{
    uint32_t const c0 = brick_column<LAYERS>(x0), c1 = brick_column<LAYERS>(x1);
    uint32_t const r0 = brick_row<LAYERS>(y0, log2GridWidth), r1 = brick_row<LAYERS>(y1, log2GridWidth);
    load_brick_cell<LAYERS>(base, r0 + c0, out[0]);
    load_brick_cell<LAYERS>(base, r0 + c1, out[1]);
    load_brick_cell<LAYERS>(base, r1 + c0, out[2]);
    load_brick_cell<LAYERS>(base, r1 + c1, out[3]);
}

// All layers of one cell: layer L in the low or high half of out[L / 2].
template <int LAYERS>
__device__ __forceinline__ void load_brick_cell(GlobalU8Ptr base, uint32_t off, uint32_t (&out)[2])
{
    out[0] = 0; out[1] = 0;
    if constexpr (LAYERS == 1) {
        out[0] = load_u16(base, off);
    } else if constexpr (LAYERS == 2) {
        out[0] = *reinterpret_cast<GlobalU32A2Ptr>(base + off);
    } else if constexpr (LAYERS == 3) {
        out[0] = *reinterpret_cast<GlobalU32A2Ptr>(base + off);
        out[1] = load_u16(base, off + 4u);
    } else {
        u32x2 const v = *reinterpret_cast<GlobalU32x2Ptr>(base + off);
        out[0] = v[0]; out[1] = v[1];
    }
}

// The lane's query of the 64 of a wave, the call's last one again beyond it.  Whole waves, all but one of a call, read and
// write at lane offsets from scalar addresses: a store takes half the instructions.  (With the
// taps' offsets by column and row, 2^24 queries of the headline network 588.8 -> 575.7 us, 2^22 of the 0.9.2 one 163 -> 158.)
__device__ __forceinline__ DevQuery load_query(DevQuery const* queries, uint64_t q0, uint64_t numQueries, int lane)
{
    if (q0 + 64u <= numQueries) {                            // uniform
        GlobalU8Ptr const first = (GlobalU8Ptr)uniform_pointer(reinterpret_cast<uint64_t>(queries + q0));
        __attribute__((address_space(1))) DevQuery const* const own = reinterpret_cast<__attribute__((address_space(1))) DevQuery const*>(first + uint32_t(lane) * uint32_t(sizeof(DevQuery)));
        return DevQuery{ own->u, own->v, own->mip };
    }
    return queries[min(q0 + uint64_t(lane), numQueries - 1)];
}

// Four outputs of a query, zeros where its mip does not exist.
__device__ __forceinline__ void store_query_outputs(uint16_t* out, v4f F, v4f S, bool valid)
{
    uint32_t h01 = to_half2_bits(F[0] * S[0], F[1] * S[1]);
    uint32_t h23 = to_half2_bits(F[2] * S[2], F[3] * S[3]);
    if (!valid) { h01 = 0; h23 = 0; }
    *reinterpret_cast<u32x2*>(out) = u32x2{ h01, h23 };
}

// The outputs of a whole wave of queries, none of which can overflow a half: lane (j, g) holds channels 4g..4g+3 of query
// q0 + 16b + j.  valid: the bit of each query whose mip exists; the others' outputs are zeros.  (With one in twenty that does not,
// so that hardly a wave is without, 65 536 queries of the 0.9.2 network take 7.8 us and 2^22 151; where such waves stored as
// the last, partial one does, lane by lane and checked, 8.0 and 155.)
template <class ACC>
__device__ __forceinline__ void store_whole_queries(uint16_t* out, uint64_t q0, int j, int g, ACC const (&D)[4], v4f S, uint64_t valid)
{
    GlobalOutPtr const first = uniform_pointer(reinterpret_cast<uint64_t>(out + q0 * 16u));
    uint32_t const own = uint32_t(j) * 32u + uint32_t(g) * 8u;
    auto const store = [&](auto every) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            uint32_t h01 = to_half2_bits<false>(float(D[b][0]) * S[0], float(D[b][1]) * S[1]);
            uint32_t h23 = to_half2_bits<false>(float(D[b][2]) * S[2], float(D[b][3]) * S[3]);
            if (!decltype(every)::value && !((uint32_t(valid >> (16 * b)) >> j) & 1u)) { h01 = 0; h23 = 0; }
            *reinterpret_cast<__attribute__((address_space(1))) u32x2*>(first + (own + 512u * uint32_t(b))) = u32x2{ h01, h23 };
        }
    };
    if (valid == ~uint64_t(0)) store(std::true_type{});      // uniform
    else                       store(std::false_type{});
}

// What a query needs of its mip, kept in LDS: every lane of a wave may address another mip, and
// fetching these fields per lane from the table in global memory put a long dependent load in
// front of the latent gathers.
struct QueryMip {
    uint16_t const* hr;
    uint16_t const* lr;
    uint32_t hrAxisX, hrAxisY, lrAxisX, lrAxisY;
    int32_t hrWidth, hrHeight, lrWidth, lrHeight;
    int32_t width, height;
    uint32_t posMask, fast;
    float positionLod;
    uint32_t pad[3];
    uint8_t const* hrBricks;
    uint8_t const* lrBricks;
};
static_assert(sizeof(QueryMip) == 96, "QueryMip layout");

} // namespace ntc_hip_dev
