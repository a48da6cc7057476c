// ntc_bc7_kernel.hip - BC7 block compression of a decoded image (gfx950).
//
// The reference's BC7 pass (IContext::MakeBlockCompressionComputePass with BlockCompressedFormat::BC7,
// src/shaders/CompressBC7.hlsl) as compute kernels: the full search, which the waves of a workgroup share, and one that
// encodes given modes, a block per lane.
//
// Full search, per block: opaque blocks try the three-subset modes 0 and 2 and the two-subset modes
// 1 and 3, each on the partition whose bounding-box endpoints give the smallest estimated error over
// all 64 partitions; every block then tries modes 4 and 5 in the four channel rotations, mode 6 and
// mode 7.  A candidate = bounding-box endpoints per subset (ends paired by covariance sign), two
// rounds of least-squares refinement, quantisation with the mode's p-bit rule, indices along the
// dequantised endpoints; its error is measured on what a decoder will show, and it replaces the
// current block when the error is not larger.  With a mode buffer (9 bits per block: mode and
// partition, MakeBC7ModeBuffer) only that candidate is encoded and no error is computed.
//
// All float arithmetic is IEEE binary32, unfused, in the order written here.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <float.h>
#include "ntc_decode_kernel.h"
#include "ntc_bc_source.h"

namespace ntc_hip_dev {

namespace {

#define BC7_INLINE __device__ __forceinline__

// Table.P2 and Table.P3 of the BPTC format specification (ARB_texture_compression_bptc), packed: the
// subset of texel t in bits 2t, 2t+1.  Anchor tables A2, A3a, A3b of the same specification.
__constant__ uint32_t kTwoSubsets[64] = {
    0x50505050u, 0x40404040u, 0x54545454u, 0x54505040u, 0x50404000u, 0x55545450u, 0x55545040u, 0x54504000u,
    0x50400000u, 0x55555450u, 0x55544000u, 0x54400000u, 0x55555440u, 0x55550000u, 0x55555500u, 0x55000000u,
    0x55150100u, 0x00004054u, 0x15010000u, 0x00405054u, 0x00004050u, 0x15050100u, 0x05010000u, 0x40505054u,
    0x00404050u, 0x05010100u, 0x14141414u, 0x05141450u, 0x01155440u, 0x00555500u, 0x15014054u, 0x05414150u,
    0x44444444u, 0x55005500u, 0x11441144u, 0x05055050u, 0x05500550u, 0x11114444u, 0x41144114u, 0x44111144u,
    0x15055054u, 0x01055040u, 0x05041050u, 0x05455150u, 0x14414114u, 0x50050550u, 0x41411414u, 0x00141400u,
    0x00041504u, 0x00105410u, 0x10541000u, 0x04150400u, 0x50410514u, 0x41051450u, 0x05415014u, 0x14054150u,
    0x41050514u, 0x41505014u, 0x40011554u, 0x54150140u, 0x50505500u, 0x00555050u, 0x15151010u, 0x54540404u,
};
__constant__ uint32_t kThreeSubsets[64] = {
    0xaa685050u, 0x6a5a5040u, 0x5a5a4200u, 0x5450a0a8u, 0xa5a50000u, 0xa0a05050u, 0x5555a0a0u, 0x5a5a5050u,
    0xaa550000u, 0xaa555500u, 0xaaaa5500u, 0x90909090u, 0x94949494u, 0xa4a4a4a4u, 0xa9a59450u, 0x2a0a4250u,
    0xa5945040u, 0x0a425054u, 0xa5a5a500u, 0x55a0a0a0u, 0xa8a85454u, 0x6a6a4040u, 0xa4a45000u, 0x1a1a0500u,
    0x0050a4a4u, 0xaaa59090u, 0x14696914u, 0x69691400u, 0xa08585a0u, 0xaa821414u, 0x50a4a450u, 0x6a5a0200u,
    0xa9a58000u, 0x5090a0a8u, 0xa8a09050u, 0x24242424u, 0x00aa5500u, 0x24924924u, 0x24499224u, 0x50a50a50u,
    0x500aa550u, 0xaaaa4444u, 0x66660000u, 0xa5a0a5a0u, 0x50a050a0u, 0x69286928u, 0x44aaaa44u, 0x66666600u,
    0xaa444444u, 0x54a854a8u, 0x95809580u, 0x96969600u, 0xa85454a8u, 0x80959580u, 0xaa141414u, 0x96960000u,
    0xaaaa1414u, 0xa05050a0u, 0xa0a5a5a0u, 0x96000000u, 0x40804080u, 0xa9a8a9a8u, 0xaaaaaa44u, 0x2a4a5254u,
};
__constant__ uint8_t kAnchorSecondOfTwo[64] = {
    15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15,
    15,  2,  8,  2,  2,  8,  8, 15,  2,  8,  2,  2,  8,  8,  2,  2,
    15, 15,  6,  8,  2,  8, 15, 15,  2,  8,  2,  2,  2, 15, 15,  6,
     6,  2,  6,  8, 15, 15,  2,  2, 15, 15, 15, 15, 15,  2,  2, 15,
};
__constant__ uint8_t kAnchorSecondOfThree[64] = {
     3,  3, 15, 15,  8,  3, 15, 15,  8,  8,  6,  6,  6,  5,  3,  3,
     3,  3,  8, 15,  3,  3,  6, 10,  5,  8,  8,  6,  8,  5, 15, 15,
     8, 15,  3,  5,  6, 10,  8, 15, 15,  3, 15,  5, 15, 15, 15, 15,
     3, 15,  5,  5,  5,  8,  5, 10,  5, 10,  8, 13, 15, 12,  3,  3,
};
__constant__ uint8_t kAnchorThirdOfThree[64] = {
    15,  8,  8,  3, 15, 15,  3,  8, 15, 15, 15, 15, 15, 15, 15,  8,
    15,  8, 15,  3, 15,  8, 15,  8,  3, 15,  6, 10, 15, 15, 10,  8,
    15,  3, 15, 10, 10,  8,  9, 10,  6, 15,  8, 15,  3,  6,  6,  8,
    15,  3, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15,  3, 15, 15,  8,
};
// Subset masks in "spread" form: bit 2t set when texel t belongs to the subset.
constexpr uint32_t kAllTexels = 0x55555555u;
BC7_INLINE uint32_t spread_mask(uint32_t partitionWord, uint32_t subset)
{
    uint32_t const x = partitionWord ^ (subset * kAllTexels);
    return ~(x | (x >> 1)) & kAllTexels;
}
BC7_INLINE bool has_texel(uint32_t mask, int t) { return (mask >> (2 * t)) & 1u; }

template <int SUBSETS> BC7_INLINE uint32_t partition_word(int partition)
{
    if constexpr (SUBSETS == 1) return 0u;
    else if constexpr (SUBSETS == 2) return kTwoSubsets[partition];
    else return kThreeSubsets[partition];
}
template <int SUBSETS> BC7_INLINE int subset_anchor(int partition, int s)
{
    if (s == 0) return 0;
    if constexpr (SUBSETS == 2) return kAnchorSecondOfTwo[partition];
    else if constexpr (SUBSETS == 3) return s == 1 ? kAnchorSecondOfThree[partition] : kAnchorThirdOfThree[partition];
    else return 0;
}

template <int C> struct Color { float c[C]; };
template <int C> struct Quantized { int c[C]; };

BC7_INLINE float saturate(float v) { return fminf(fmaxf(v, 0.f), 1.f); }        // a NaN becomes 0
template <int C> BC7_INLINE float dot(Color<C> const& a, Color<C> const& b)
{
    float s = a.c[0] * b.c[0];
#pragma unroll
    for (int k = 1; k < C; ++k) s += a.c[k] * b.c[k];
    return s;
}
template <int C> BC7_INLINE Color<C> sub(Color<C> const& a, Color<C> const& b)
{
    Color<C> r;
#pragma unroll
    for (int k = 0; k < C; ++k) r.c[k] = a.c[k] - b.c[k];
    return r;
}

template <int C> BC7_INLINE void min_max(Color<C> const (&px)[16], uint32_t mask, Color<C>& lo, Color<C>& hi)
{
#pragma unroll
    for (int k = 0; k < C; ++k) { lo.c[k] = FLT_MAX; hi.c[k] = -FLT_MAX; }
#pragma unroll
    for (int t = 0; t < 16; ++t)
        if (has_texel(mask, t)) {
#pragma unroll
            for (int k = 0; k < C; ++k) { lo.c[k] = min_f32(lo.c[k], px[t].c[k]); hi.c[k] = max_f32(hi.c[k], px[t].c[k]); }
        }
}

// With the first component whose ends differ as the axis, the ends of later components are swapped
// where their covariance with the axis is negative.
template <int C> BC7_INLINE void orient(Color<C> const (&px)[16], uint32_t mask, Color<C>& e0, Color<C>& e1)
{
    Color<C> center;
#pragma unroll
    for (int k = 0; k < C; ++k) center.c[k] = 0.f;
#pragma unroll
    for (int t = 0; t < 16; ++t)
        if (has_texel(mask, t)) {
#pragma unroll
            for (int k = 0; k < C; ++k) center.c[k] += px[t].c[k];
        }
    float const count = float(__popc(mask));
#pragma unroll
    for (int k = 0; k < C; ++k) center.c[k] /= count;
    float cov[C][C];
#pragma unroll
    for (int a = 0; a < C; ++a)
#pragma unroll
        for (int b = 0; b < C; ++b) cov[a][b] = 0.f;
#pragma unroll
    for (int t = 0; t < 16; ++t)
        if (has_texel(mask, t)) {
            Color<C> const d = sub(px[t], center);
#pragma unroll
            for (int a = 0; a < C; ++a)
#pragma unroll
                for (int b = a + 1; b < C; ++b) cov[a][b] += d.c[a] * d.c[b];
        }
    bool done = false;
#pragma unroll
    for (int a = 0; a + 1 < C; ++a) {
        if (!done && e0.c[a] != e1.c[a]) {
#pragma unroll
            for (int b = a + 1; b < C; ++b)
                if (cov[a][b] < 0.f) { float const t = e0.c[b]; e0.c[b] = e1.c[b]; e1.c[b] = t; }
            done = true;
        }
    }
}

// Two rounds of: project the texels on the endpoint axis, snap to the index grid, solve the
// least-squares problem for new endpoints.  Components sitting exactly on 0 or 1 stay.
template <int C> BC7_INLINE void refine(Color<C> const (&px)[16], uint32_t mask, Color<C>& e0, Color<C>& e1, int indexBits)
{
    float const scale = float((1u << indexBits) - 1u), iscale = 1.f / scale;
#pragma unroll 1
    for (int iter = 0; iter < 2; ++iter) {
        Color<C> const axis = sub(e1, e0);
        float mul = dot(axis, axis);
        if (mul > 0.f) mul = 1.f / mul;
        float a2 = 0.f, b2 = 0.f, ab = 0.f;
        Color<C> ax, bx;
#pragma unroll
        for (int k = 0; k < C; ++k) ax.c[k] = bx.c[k] = 0.f;
#pragma unroll
        for (int t = 0; t < 16; ++t)
            if (has_texel(mask, t)) {
                float const f = saturate(dot(sub(px[t], e0), axis) * mul);
                float const beta = rintf(f * scale) * iscale, alpha = 1.f - beta;
                a2 += alpha * alpha; b2 += beta * beta; ab += alpha * beta;
#pragma unroll
                for (int k = 0; k < C; ++k) { ax.c[k] += alpha * px[t].c[k]; bx.c[k] += beta * px[t].c[k]; }
            }
        float const denom = a2 * b2 - ab * ab;
        if (!(fabsf(denom) > 0.0001f)) break;
        float const factor = 1.f / denom;
#pragma unroll
        for (int k = 0; k < C; ++k) {
            float const a = saturate((ax.c[k] * b2 - bx.c[k] * ab) * factor), b = saturate((bx.c[k] * a2 - ax.c[k] * ab) * factor);
            if (!(e0.c[k] == 0.f || e0.c[k] == 1.f)) e0.c[k] = a;
            if (!(e1.c[k] == 0.f || e1.c[k] == 1.f)) e1.c[k] = b;
        }
    }
}

BC7_INLINE int quantize(float v, int bits) { return int(rintf(saturate(v) * float((1u << bits) - 1u))); }
BC7_INLINE int expand8(int q, int bits) { return (q << (8 - bits)) | (q >> (2 * bits - 8)); }

// Indices of the subset's texels along the dequantised endpoints, each in its place in the block: `two` for 2-bit ones, `more`
// for those of three bits and four, whichever BITS says; for 0 both, and `indexBits` tells which of them is meant.
template <int C, int BITS> BC7_INLINE void assign(Color<C> const (&px)[16], uint32_t mask, int indexBits, int endpointBits,
                                                  Quantized<C> const& q0, Quantized<C> const& q1, uint32_t& two, uint64_t& more)
{
    Color<C> e0, e1;
#pragma unroll
    for (int k = 0; k < C; ++k) {
        e0.c[k] = unorm_quotient(float(expand8(q0.c[k], endpointBits)), 255.f, 1.f / 255.f);
        e1.c[k] = unorm_quotient(float(expand8(q1.c[k], endpointBits)), 255.f, 1.f / 255.f);
    }
    Color<C> const axis = sub(e1, e0);
    float mul = dot(axis, axis);
    if (mul > 0.f) mul = 1.f / mul;
#pragma unroll
    for (int t = 0; t < 16; ++t)
        if (has_texel(mask, t)) {
            uint32_t const index = uint32_t(quantize(dot(sub(px[t], e0), axis) * mul, indexBits));
            if constexpr (BITS == 0 || BITS == 2) two |= index << (2 * t);
            if constexpr (BITS == 0)              more |= uint64_t(index) << (3 * t);
            else if constexpr (BITS > 2)          more |= uint64_t(index) << (BITS * t);
        }
}

// A field of a block from bit `at` on, and the removal of the anchors' top index bits, which are zero.
BC7_INLINE void put_indices(uint64_t& lo, uint64_t& hi, int at, uint64_t v)
{
    if (at < 64) { lo |= v << at; hi |= at ? v >> (64 - at) : 0; }
    else hi |= v << (at - 64);
}
// The three bits of each index of a subset.
BC7_INLINE uint64_t three_bits_of(uint32_t spreadMask)
{
    uint64_t x = 0;
#pragma unroll
    for (int t = 0; t < 16; ++t) x |= uint64_t((spreadMask >> (2 * t)) & 1u) << (3 * t);
    return x * 7u;
}
BC7_INLINE uint64_t without_bit(uint64_t v, int at)
{
    uint64_t const below = (uint64_t(1) << at) - 1u;
    return (v & below) | ((v >> 1) & ~below);
}

struct Bits {
    uint64_t lo = 0, hi = 0;
    int at = 0;
    BC7_INLINE void put(int length, uint32_t value)
    {
        uint64_t const v = value & ((1u << length) - 1u);
        if (at < 64) { lo |= v << at; if (at + length > 64) hi |= v >> (64 - at); }
        else hi |= v << (at - 64);
        at += length;
    }
};

struct Best { float error; uint64_t lo, hi; };
struct Block { uint64_t lo, hi; };

enum { kNoPBit = 0, kPBitPerEndpoint = 1, kPBitPerSubset = 2 };
template <int ID, int SUBSETS_, int PARTITION_BITS, int ENDPOINT_BITS /* with the p-bit */, int INDEX_BITS, int PBIT>
struct Mode {
    static constexpr int id = ID, subsets = SUBSETS_, partitionBits = PARTITION_BITS, endpointBits = ENDPOINT_BITS, indexBits = INDEX_BITS, pbit = PBIT;
};
using Mode0 = Mode<0, 3, 4, 5, 3, kPBitPerEndpoint>;
using Mode1 = Mode<1, 2, 6, 7, 3, kPBitPerSubset>;
using Mode2 = Mode<2, 3, 6, 5, 2, kNoPBit>;
using Mode3 = Mode<3, 2, 6, 8, 2, kPBitPerEndpoint>;
using Mode6 = Mode<6, 1, 0, 8, 4, kPBitPerEndpoint>;
using Mode7 = Mode<7, 2, 6, 6, 2, kPBitPerEndpoint>;

// Endpoint quantisation with the mode's p-bit rule: the shared lowest bit is the majority of the
// components' lowest bits; with alpha, an alpha of exactly 1 forces it to 1 and a quantised alpha of 0
// to 0, which keeps both exact.
template <class M, int C> BC7_INLINE void quantize_endpoints(Color<C> const (&e)[2 * M::subsets], Quantized<C> (&q)[2 * M::subsets])
{
    constexpr int N = 2 * M::subsets;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int k = 0; k < C; ++k) q[i].c[k] = quantize(e[i].c[k], M::endpointBits);
    if constexpr (M::pbit == kPBitPerEndpoint) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            int odd = 0;
#pragma unroll
            for (int k = 0; k < C; ++k) odd += q[i].c[k] & 1;
            int lsb = odd >= 2 ? 1 : 0;
            if constexpr (C == 4) lsb = ((odd >= 2 && q[i].c[3] != 0) || e[i].c[3] == 1.f) ? 1 : 0;
#pragma unroll
            for (int k = 0; k < C; ++k) q[i].c[k] = (q[i].c[k] & 0xFE) | lsb;
        }
    } else if constexpr (M::pbit == kPBitPerSubset) {
#pragma unroll
        for (int i = 0; i < N; i += 2) {
            int odd = 0;
#pragma unroll
            for (int k = 0; k < C; ++k) odd += (q[i].c[k] & 1) + (q[i + 1].c[k] & 1);
            int const lsb = odd >= 4 ? 1 : 0;
#pragma unroll
            for (int k = 0; k < C; ++k) { q[i].c[k] = (q[i].c[k] & 0xFE) | lsb; q[i + 1].c[k] = (q[i + 1].c[k] & 0xFE) | lsb; }
        }
    }
}

// Refines the start endpoints of every subset, quantises, assigns indices and encodes the block.
template <class M, int C> BC7_INLINE Block finish(Color<C> const (&px)[16], int partition, Color<C> const (&start)[2 * M::subsets])
{
    constexpr int N = 2 * M::subsets, top = M::indexBits - 1;
    uint32_t const word = partition_word<M::subsets>(partition);
    Color<C> e[N];
    Quantized<C> q[N];
#pragma unroll
    for (int i = 0; i < N; ++i) e[i] = start[i];
#pragma unroll
    for (int s = 0; s < M::subsets; ++s) refine(px, spread_mask(word, s), e[2 * s], e[2 * s + 1], M::indexBits);
    quantize_endpoints<M, C>(e, q);
    uint64_t indices = 0;
    int anchors[M::subsets];
#pragma unroll
    for (int s = 0; s < M::subsets; ++s) {
        uint32_t const mask = spread_mask(word, s);
        uint32_t two = 0;
        uint64_t more = 0;
        assign<C, M::indexBits>(px, mask, M::indexBits, M::endpointBits, q[2 * s], q[2 * s + 1], two, more);
        uint64_t const own = M::indexBits == 2 ? uint64_t(two) : more;
        indices |= own;
        // a decoder assumes the anchor's top index bit to be 0: if it is 1 the subset's indices are complemented and its
        // endpoints trade places
        anchors[s] = subset_anchor<M::subsets>(partition, s);
        if ((own >> (anchors[s] * M::indexBits + top)) & 1u) {
            indices ^= M::indexBits == 2 ? uint64_t(mask * 3u) : M::indexBits == 4 ? ~uint64_t(0) : three_bits_of(mask);
            Quantized<C> const t = q[2 * s]; q[2 * s] = q[2 * s + 1]; q[2 * s + 1] = t;
        }
    }
    Bits b;
    b.put(M::id + 1, 1u << M::id);
    b.put(M::partitionBits, uint32_t(partition));
    constexpr int drop = M::pbit == kNoPBit ? 0 : 1;
#pragma unroll
    for (int k = 0; k < C; ++k)
#pragma unroll
        for (int i = 0; i < N; ++i) b.put(M::endpointBits - drop, uint32_t(q[i].c[k]) >> drop);
    if constexpr (M::pbit == kPBitPerEndpoint) {
#pragma unroll
        for (int i = 0; i < N; ++i) b.put(1, uint32_t(q[i].c[0]));
    }
    if constexpr (M::pbit == kPBitPerSubset) {
#pragma unroll
        for (int s = 0; s < M::subsets; ++s) b.put(1, uint32_t(q[2 * s].c[0]));
    }
    if constexpr (M::subsets == 3) {
        indices = without_bit(indices, max(anchors[1], anchors[2]) * M::indexBits + top);
        indices = without_bit(indices, min(anchors[1], anchors[2]) * M::indexBits + top);
    } else if constexpr (M::subsets == 2) {
        indices = without_bit(indices, anchors[1] * M::indexBits + top);
    }
    indices = without_bit(indices, top);
    put_indices(b.lo, b.hi, b.at, indices);
    return { b.lo, b.hi };
}

// Start endpoints of every subset of a partition: the subset's bounding box, oriented if asked.
template <int SUBSETS, int C, bool ORIENT> BC7_INLINE void partition_ends(Color<C> const (&px)[16], int partition, Color<C> (&ends)[2 * SUBSETS])
{
    uint32_t const word = partition_word<SUBSETS>(partition);
#pragma unroll
    for (int s = 0; s < SUBSETS; ++s) {
        uint32_t const mask = spread_mask(word, s);
        min_max(px, mask, ends[2 * s], ends[2 * s + 1]);
        if constexpr (ORIENT) orient(px, mask, ends[2 * s], ends[2 * s + 1]);
    }
}

// Modes 4 and 5: a colour plane of three channels and a scalar plane, each with its own endpoints and
// indices; the scalar plane takes channel {A, R, G, B}[rotation] and alpha takes its place.
BC7_INLINE void split_planes(Color<4> const (&rgba)[16], uint32_t rotation, Color<3> (&rgb)[16], Color<1> (&a)[16])
{
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        Color<4> const& p = rgba[t];
        rgb[t].c[0] = rotation == 1 ? p.c[3] : p.c[0];
        rgb[t].c[1] = rotation == 2 ? p.c[3] : p.c[1];
        rgb[t].c[2] = rotation == 3 ? p.c[3] : p.c[2];
        a[t].c[0] = rotation == 0 ? p.c[3] : rotation == 1 ? p.c[0] : rotation == 2 ? p.c[1] : p.c[2];
    }
}
template <int C> struct Ends { Color<C> e0, e1; };

// The block of the two modes from the refined endpoints of both planes.  Mode 4's fields are 8 bits of mode, rotation and
// choice, 42 of endpoints, its 2-bit indices and its 3-bit ones; mode 5's 8 bits, 58, the colours' indices, the scalars'.
BC7_INLINE Block finish_dual_plane(int mode, bool wideColorIndex, Color<3> const (&rgb)[16], Color<1> const (&a)[16], Ends<3> const& color, Ends<1> const& alpha,
                                   uint32_t rotation)
{
    int const colorIndexBits = mode == 5 ? 2 : (wideColorIndex ? 3 : 2), alphaIndexBits = mode == 5 ? 2 : (wideColorIndex ? 2 : 3);
    int const colorBits = mode == 5 ? 7 : 5, alphaBits = mode == 5 ? 8 : 6;
    Quantized<3> q0, q1;
#pragma unroll
    for (int k = 0; k < 3; ++k) { q0.c[k] = quantize(color.e0.c[k], colorBits); q1.c[k] = quantize(color.e1.c[k], colorBits); }
    Quantized<1> qa0, qa1;
    qa0.c[0] = quantize(alpha.e0.c[0], alphaBits); qa1.c[0] = quantize(alpha.e1.c[0], alphaBits);
    // indices of one plane with the first one's top bit taken out; true: they are complemented and the endpoints trade places
    auto const packed = [](int bits, uint32_t two, uint64_t three, uint64_t& indices) {
        indices = bits == 2 ? uint64_t(two) : three;
        bool const flip = (uint32_t(indices) >> (bits - 1)) & 1u;
        if (flip) indices ^= bits == 2 ? 0xffffffffull : 0xffffffffffffull;
        uint64_t const below = bits == 2 ? 1u : 3u;
        indices = (indices & below) | ((indices >> 1) & ~below);
        return flip;
    };
    uint64_t colorIndices, alphaIndices, three = 0;
    uint32_t two = 0;
    assign<3, 0>(rgb, kAllTexels, colorIndexBits, colorBits, q0, q1, two, three);
    if (packed(colorIndexBits, two, three, colorIndices)) { Quantized<3> const t = q0; q0 = q1; q1 = t; }
    two = 0; three = 0;
    assign<1, 0>(a, kAllTexels, alphaIndexBits, alphaBits, qa0, qa1, two, three);
    if (packed(alphaIndexBits, two, three, alphaIndices)) { Quantized<1> const t = qa0; qa0 = qa1; qa1 = t; }
    uint64_t ends = uint32_t(qa1.c[0]) << alphaBits | uint32_t(qa0.c[0]);
#pragma unroll
    for (int k = 2; k >= 0; --k) ends = ends << (2 * colorBits) | (uint32_t(q1.c[k]) << colorBits | uint32_t(q0.c[k]));
    uint32_t const head = mode == 5 ? 0x20u | rotation << 6 : 0x10u | rotation << 5 | (wideColorIndex ? 0x80u : 0u);
    Block block{ uint64_t(head) | ends << 8, ends >> 56 };
    bool const alphaFirst = mode == 4 && wideColorIndex;
    int const at = mode == 5 ? 66 : 50;                      // then 31 bits of 2-bit indices
    put_indices(block.lo, block.hi, at, alphaFirst ? alphaIndices : colorIndices);
    put_indices(block.lo, block.hi, at + 31, alphaFirst ? colorIndices : alphaIndices);
    return block;
}

template <int C> BC7_INLINE Ends<C> box_of(Color<C> const (&px)[16])
{
    Ends<C> e;
    min_max(px, kAllTexels, e.e0, e.e1);
    if constexpr (C > 1) orient(px, kAllTexels, e.e0, e.e1);
    return e;
}
template <int C> BC7_INLINE Ends<C> refined(Color<C> const (&px)[16], Ends<C> e, int indexBits)
{
    refine(px, kAllTexels, e.e0, e.e1, indexBits);
    return e;
}

BC7_INLINE Block fixed_dual_plane(int mode, bool wideColorIndex, Color<4> const (&rgba)[16], uint32_t rotation)
{
    Color<3> rgb[16];
    Color<1> a[16];
    split_planes(rgba, rotation, rgb, a);
    int const colorIndexBits = mode == 5 ? 2 : (wideColorIndex ? 3 : 2), alphaIndexBits = mode == 5 ? 2 : (wideColorIndex ? 2 : 3);
    return finish_dual_plane(mode, wideColorIndex, rgb, a, refined(rgb, box_of(rgb), colorIndexBits), refined(a, box_of(a), alphaIndexBits), rotation);
}

// One block with a given mode and partition (for modes 4 / 5: rotation in bits 0-1 of the partition, "wide colour
// index" in bit 2).  `list` says the mode but for 4 and 5, and is uniform.
BC7_INLINE Block bc7_encode_fixed(Color<4> const (&px)[16], int list, int mode, int partition)
{
    if (list <= 3) {
        Color<3> rgb[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) { rgb[t].c[0] = px[t].c[0]; rgb[t].c[1] = px[t].c[1]; rgb[t].c[2] = px[t].c[2]; }
        if (list <= 1) {
            Color<3> ends[6];
            partition_ends<3, 3, true>(rgb, partition, ends);
            return list == 0 ? finish<Mode0>(rgb, partition, ends) : finish<Mode2>(rgb, partition, ends);
        }
        Color<3> ends[4];
        partition_ends<2, 3, true>(rgb, partition, ends);
        return list == 2 ? finish<Mode1>(rgb, partition, ends) : finish<Mode3>(rgb, partition, ends);
    }
    if (list == 5) return fixed_dual_plane(mode, mode == 4 && (partition & 4), px, uint32_t(partition) & 3u);
    if (list == 6) {
        Color<4> ends[2];
        partition_ends<1, 4, true>(px, 0, ends);
        return finish<Mode6>(px, 0, ends);
    }
    Color<4> ends[4];
    partition_ends<2, 4, false>(px, partition, ends);
    return finish<Mode7>(px, partition, ends);
}

BC7_INLINE void load_block(BlockCompressArgs const& a, int bx, int by, Color<4> (&px)[16])
{
    float values[4][4][4];
    source_rows<4, 4>(a, a.srcLeft + bx * 4, a.srcTop + by * 4, 0, values);
#pragma unroll
    for (int t = 0; t < 16; ++t)
#pragma unroll
        for (int k = 0; k < 4; ++k) px[t].c[k] = values[t >> 2][t & 3][k];
}
BC7_INLINE void store_block(BlockCompressArgs const& a, int bx, int by, uint64_t lo, uint64_t hi)
{
    uint64_t* const dst = reinterpret_cast<uint64_t*>(a.dst + size_t(by + a.dstOffsetY) * a.dstRowPitch) + size_t(bx + a.dstOffsetX) * 2;
    dst[0] = lo; dst[1] = hi;
}

} // namespace

// ---- full search --------------------------------------------------------------------------------------
//
// A workgroup of WAVES waves encodes GROUPS x 64 blocks; the lanes of a wave are blocks, and the waves divide the search
// among themselves.  The texels lie in LDS.
//   1. A search is for the partition with the smallest estimated error of 64 blocks: of two and of three subsets for
//      opaque blocks, of two subsets for mode 7.  Tasks of a range of its partitions bound the errors from below, all
//      lanes with the same partition; when a search's are done, one more task estimates the error of the partition with
//      the smallest bound and queues those whose bounds do not exceed it: one to seven of 64 on textures with detail.
//      Beside them a task for each group: lower bounds of the errors of the four channel rotations of modes 4 and 5 and of
//      mode 6, then the three forms of the rotation with the smallest one, whose error leaves out what is bounded above it.
//      (Or, where it is the chain that counts, a task for each rotation and one for mode 6: see all_by_bounds.)
//   2. Tasks of 64 queued estimates, from any blocks of a search; tasks of 64 rotations or of 64 blocks of mode 6 that were
//      not left out; tasks of one candidate, from its endpoints to the encoded block, where every lane has a partition of
//      its own and walks its own list of texels.
//   3. A thread per block goes through the candidates in the order given at the top with "not larger replaces".
// Blocks with and without alpha are gathered in groups of their own for the tasks that only one kind has.  Waves take the
// tasks of a phase in turn; one that builds upon others waits for their count.
//
// The search is bound by vector instruction issue where it fills the GPU and by the length of one lane's chain where it
// does not.  One lane per block with the texels in 255 registers took 0.9 ms for any image of up to 1024 x 1024; with the
// search divided and every partition estimated, 64 x 64 took 98 us, 512 x 512 102, 1024 x 1024 274 and 2048 x 2048 927 (half
// of it opaque; 183 M vector instructions at 1024 x 1024, seven of ten of them estimates); with bounds first 79, 88, 191
// and 721 (140 M).  Bounds cost a third of an estimate and leave few to make where texels have noise or detail in three
// channels; where a block's colours lie near a line, because channels are proportional or an edge between two colours runs
// through it, most partitions' bounds are below the smallest error.  Searches with many such blocks are estimated as a whole
// without bounds (kMostExpected): 1024 x 1024 opaque, by estimates of every partition / by bounds first, whole where a queue
// overflows or 48 of 64 blocks are near a line / now: grey 272 / 239 / 239 us, noise of 1.5 codes on proportional channels
// 273 / 275 / 240 and of 4 codes 274 / 307 / 240, hard edges in every block 276 / 299 / 243 and with noise 275 / 306 / 245,
// antialiased boxes and strokes 278 / 317 / 244 and with noise 275 / 317 / 241; not antialiased 272 / 174 / 187.
// Rotations and mode 6 by their bounds: of the half opaque image all blocks' mode 6 but 12 to 14 %, 2 of 5 (opaque) or of 2
// (others) rotations; where alphas are 1 their planes have two channels: 1024 x 1024 opaque noise 187 -> 162 us, a smooth
// image 234 -> 226, grey 240 -> 234, hard edges 243 -> 237, ramps 191 -> 183, one colour 151 -> 149.
//
// Wave priorities fall from phase to phase.  With equal ones the older of the two workgroups of a compute unit runs ahead
// through the first phase and leaves the younger one alone with half the waves at the end (347 and 485 thousand cycles at
// 1024 x 1024); a workgroup that is behind now comes first (365 and 422 thousand; 209 -> 188 us).
// Slots of candidates: modes 0, 2, 1, 3, the rotations after the first in their order, modes 6 and 7.
enum { kSlotRotations = 4, kSlotSix = 7, kSlotSeven, kSlots };
enum : uint32_t { kKeepRotation = 4, kKeepSix = 64 };
enum { kPickThree = 0, kPickTwo, kPickTwoAlpha, kPicks };
enum : uint32_t { kBelowOne = 1, kNotOne = 2 };              // what some alpha of a block is (one above 1 or a NaN is only the second)

// The searches of a workgroup: its opaque groups' partitions of two subsets, then of three, then the partitions for mode 7
// of all groups, the opaque ones first.  (128 blocks are two groups of one kind, or three of both.)
enum { kSearches = 7, kQueued = 14 * 64, kWholeChunk = 8 };
// Of 128 blocks, candidates take the bounds' place when the picks are made; of 64, whose workgroup has a compute unit to itself,
// they have one of their own and some are made beside the bounds.
template <int BLOCKS> struct SearchBounds { uint32_t codes[kPicks][16][BLOCKS]; };         // of four partitions each
template <int BLOCKS> struct SearchCandidates { uint4 words[kSlots][BLOCKS]; float errors[kSlots][BLOCKS]; };
template <int BLOCKS> struct SearchScratch { union { SearchBounds<BLOCKS> bounds; SearchCandidates<BLOCKS> late; }; };
template <> struct SearchScratch<64> { SearchBounds<64> bounds; SearchCandidates<64> late; };

template <int BLOCKS_>
struct SearchLds {
    static constexpr int BLOCKS = BLOCKS_;
    float4 texels[16][BLOCKS];
    uint64_t picks[kPicks][BLOCKS];                          // error bits << 32 | partition
    float scale[kPicks][BLOCKS];                             // of errors before they become codes; 0: the block has no bounds
    uint32_t lowest[kPicks][BLOCKS];                         // the smallest bound's bits, the low six replaced by its partition
    SearchScratch<BLOCKS> scratch;
    struct { uint4 words[BLOCKS]; float errors[BLOCKS]; } early;                   // the first rotation's candidate (before: least errors of all four)
    uint32_t plans[BLOCKS];                                  // the first rotation; kKeepRotation << r and kKeepSix
    uint16_t flatRotations[2 * BLOCKS], rotations[3 * BLOCKS];                     // those kept, rotation << 7 | block: with planes of two channels, of three
    uint8_t sixes[BLOCKS];                                   // blocks that mode 6 is kept for
    uint16_t queues[kSearches][kQueued];                     // partition << 7 | block
    int queued[kSearches];
    uint8_t whole[kSearches];                                // searches that estimate every partition
    uint32_t alphas[BLOCKS];                                 // kBelowOne | kNotOne
    uint8_t blocks[2][BLOCKS];                               // numbers of the opaque blocks, of those with alpha
    int counts[2], next[2], wholes, kept[3];                 // kept: rotations of both kinds, mode 6
    int bounded[kSearches], selected, rotated, estimated;    // tasks done: those of a search's bounds, of selections, first rotations and estimates
};
static_assert(2 * sizeof(SearchLds<128>) <= 160 * 1024, "two workgroups share a compute unit's memory: one works while the other waits for its last task");
template <class S> using SearchPtr = __attribute__((address_space(3))) S*;

// The tasks are functions of their own (arguments reach them per lane: what is uniform is made so again): in one body
// the compiler keeps the texels of several of them in registers and spills three thousand.
#define BC7_TASK __device__ __attribute__((noinline))

template <int C, class S> BC7_INLINE Color<C> texel(SearchPtr<S> lds, int b, int t)
{
    Color<C> p;
    p.c[0] = lds->texels[t][b].x; p.c[1] = lds->texels[t][b].y; p.c[2] = lds->texels[t][b].z;
    if constexpr (C == 4) p.c[3] = lds->texels[t][b].w;
    return p;
}
BC7_INLINE int first_texel(uint32_t mask) { return __builtin_ctz(mask) >> 1; }           // (of a mask that has one)

// Endpoints' swaps of orient() from the finished covariances.
template <int C> BC7_INLINE void orient_by(float const (&cov)[C][C], Color<C>& e0, Color<C>& e1)
{
    bool done = false;
#pragma unroll
    for (int a = 0; a + 1 < C; ++a) {
        if (!done && e0.c[a] != e1.c[a]) {
#pragma unroll
            for (int b = a + 1; b < C; ++b)
                if (cov[a][b] < 0.f) { float const t = e0.c[b]; e0.c[b] = e1.c[b]; e1.c[b] = t; }
            done = true;
        }
    }
}
template <int C> BC7_INLINE void add_covariance(float (&cov)[C][C], Color<C> const& d)
{
#pragma unroll
    for (int a = 0; a < C; ++a)
#pragma unroll
        for (int b = a + 1; b < C; ++b) cov[a][b] += d.c[a] * d.c[b];
}
template <int C> BC7_INLINE float inverse_square(Color<C> const& axis) { float const l = dot(axis, axis); return l > 0.f ? 1.f / l : l; }

// ---- bounds of the partitions' errors
//
// The estimated error of a subset is the texels' squared distance from points of its box's diagonal, at least that from
// the diagonal itself, D.  With h the middle of the box, a its diagonal, M the second moments about h,
//     D = trace M - (a M a) / |a|^2,
// which takes sums over the texels instead of a pass over them for each of centre, covariance, and error, and of the
// largest subset not even those: its sums are what the others leave of the block's.  All sums are of offsets from texel 0.
// How far D as computed can be from its true value, and the estimate as computed below its true value: the terms' sizes
// add up to less than 42 T, T the sum of the block's squared offsets (|h|^2 and the squared mean are at most the subset's
// share of T, and a subset has at most 13 texels), and none passes through more than 34 roundings: together less than
// 1100 units of roundoff of T.  kBoundError, of 2048 units, is taken off each bound.
// The other 948 units, more than 2^-63 because T is at least kLeastOffsets, are for what does not shrink with T:
//  * products that round among subnormal numbers, by up to 2^-150.  Those that end a M a, five of a subset at most, are
//    multiplied by 1 / (|a|^2 + kLeastLength), at most 2^72: together less than 2^-74.  All others are multiplied by a
//    component of a as well, which leaves 2^36 of an offset at most, or by no more than offsets.
//  * kLeastLength itself, which makes (a M a) / |a|^2 too small by up to kLeastLength / |a|^2 of it: by 13 / 4 of
//    kLeastLength in a subset, because no texel is further from h than |a| / 2; together less than 2^-68.
constexpr float kBoundError = 0x1p-13f, kLeastLength = 0x1p-72f;
// Which components' ends trade places depends on the covariances' signs as orient_by() finds them.  Where one could be
// 0 within the errors of either evaluation (texel by texel about a rounded mean, which is off by 16 units of roundoff of
// the texels' size; by sums here, off by 100 units of T), the nearest of the four diagonals counts.
constexpr float kUnsureOfOffsets = 0x1p-16f, kUnsureOfTexels = 0x1p-35f;
// Bounds are kept as codes of eight bits: errors over T, four bits of the exponent (2^-16 ... 1) and four of the mantissa,
// rounded down.  Blocks whose T is no number between these have no bounds, and all of their partitions are estimated.
// Blocks near a line: what the partitions leave of their distances is less than the steps along the diagonals, and the
// bounds tell little.  How many partitions they leave in the searches for modes 0 to 3 goes by the block's squared distances
// over its squared diagonal (eight points leave 16 / 588 of it), much the same for noise, edges and gradients: 2 above 1 / 8, 5 to 18
// down to 1 / 16, 9 to 33, 14 to 47 and 16 to 57 down to 1 / 24, 1 / 37 and 1 / 64, 25 to 63 below.  The weights in bound_task()
// add up to the smaller ones.  Where more than kMostExpected of a group's 4096 are expected the search goes without bounds: 14 a
// block overflow its queue, 9 are as slow as estimating all, and 5 because the slowest group is what counts (hard edges with
// noise 283, 272, 257, 245 and 241 us with 10, 8, 6, 5 and 4, smooth images 241, 241, 232, 234 and 235, boxes that are not
// antialiased 185, 185, 185, 187 and 195).  Blocks of two colours are left out for two subsets, where one partition has no error.
constexpr float kNearLine = 1.f / 64.f;
constexpr int kMostExpected = 5 * 64;
// (The least T of halves that are not all equal is 2^-48.)
constexpr float kLeastOffsets = 0x1p-48f, kMostOffsets = 0x1p60f;
BC7_INLINE uint32_t error_code(float error, float scale)
{
    constexpr uint32_t first = (127u - 16u) << 4;
    uint32_t const bits = __float_as_uint(error * scale) >> 19;                  // (a NaN: the last code)
    return min(max(bits, first) - first, 255u);
}

template <int C> struct Sums {
    float s[C], q[C][C];                                     // of q the upper triangle
    BC7_INLINE Sums()
    {
#pragma unroll
        for (int i = 0; i < C; ++i) {
            s[i] = 0.f;
#pragma unroll
            for (int j = i; j < C; ++j) q[i][j] = 0.f;
        }
    }
    BC7_INLINE void add(Color<C> const& x)
    {
#pragma unroll
        for (int i = 0; i < C; ++i) {
            s[i] += x.c[i];
#pragma unroll
            for (int j = i; j < C; ++j) q[i][j] = __builtin_fmaf(x.c[i], x.c[j], q[i][j]);
        }
    }
    BC7_INLINE void remove(Sums const& o)
    {
#pragma unroll
        for (int i = 0; i < C; ++i) {
            s[i] -= o.s[i];
#pragma unroll
            for (int j = i; j < C; ++j) q[i][j] -= o.q[i][j];
        }
    }
    BC7_INLINE float trace() const
    {
        float t = q[0][0];
#pragma unroll
        for (int i = 1; i < C; ++i) t += q[i][i];
        return t;
    }
};

// The box of a subset (uniform, of N texels), and its sums if SUMS.
template <int C, int N, bool SUMS, class S>
BC7_INLINE void subset_box(SearchPtr<S> lds, int b, uint32_t mask, Color<C> const& origin, Color<C>& lo, Color<C>& hi, Sums<C>& sums)
{
    Color<C> px[N];
#pragma unroll
    for (int t = 0; t < N; ++t) {
        px[t] = texel<C, S>(lds, b, first_texel(mask));
        if constexpr (SUMS) px[t] = sub(px[t], origin);
        mask &= mask - 1;
    }
    lo = hi = px[0];
#pragma unroll
    for (int k = 0; k < C; ++k) {
#pragma unroll
        for (int t = 1; t + 1 < N; t += 2) { lo.c[k] = min3_f32(lo.c[k], px[t].c[k], px[t + 1].c[k]); hi.c[k] = max3_f32(hi.c[k], px[t].c[k], px[t + 1].c[k]); }
        if constexpr (!(N & 1)) { lo.c[k] = min_f32(lo.c[k], px[N - 1].c[k]); hi.c[k] = max_f32(hi.c[k], px[N - 1].c[k]); }
    }
    if constexpr (SUMS) {
#pragma unroll
        for (int t = 0; t < N; ++t) sums.add(px[t]);
    } else {
        lo = sub(lo, origin); hi = sub(hi, origin);          // (rounding is monotone: the box of the offsets)
    }
}

// The squared distances of a subset's n texels from the diagonal `a` of its box, whose middle is `middle2` / 2.  w: twice
// the texels' sum less n times the middle.
template <int C>
BC7_INLINE float distances(Sums<C> const& sums, Color<C> const& middle2, Color<C> const& w, Color<C> const& a, float inverse)
{
    float along = 0.f;                                       // sum of (a . offset from the middle)^2
#pragma unroll
    for (int i = 0; i < C; ++i) {
        float row = a.c[i] * sums.q[i][i];
#pragma unroll
        for (int j = i + 1; j < C; ++j) row = __builtin_fmaf(a.c[j] + a.c[j], sums.q[i][j], row);
        along = i == 0 ? a.c[i] * row : __builtin_fmaf(a.c[i], row, along);
    }
    float am = a.c[0] * middle2.c[0], aw = a.c[0] * w.c[0], mw = middle2.c[0] * w.c[0];
#pragma unroll
    for (int k = 1; k < C; ++k) { am = __builtin_fmaf(a.c[k], middle2.c[k], am); aw = __builtin_fmaf(a.c[k], w.c[k], aw); mw = __builtin_fmaf(middle2.c[k], w.c[k], mw); }
    along = __builtin_fmaf(-0.5f * am, aw, along);
    return __builtin_fmaf(-along, inverse, __builtin_fmaf(-0.5f, mw, sums.trace()));
}

// Adds a subset's squared distances from its box's diagonal: from the one that orient_by() chooses if ORIENTED, from lo to hi
// if PLAIN.  n: its number of texels.
template <int C, bool ORIENTED, bool PLAIN>
BC7_INLINE void add_distances(float n, Sums<C> const& sums, Color<C> const& lo, Color<C> const& hi, float unsure, float& oriented, float& plain)
{
    Color<C> const a = sub(hi, lo);
    Color<C> middle2, w;
    float length = kLeastLength;
#pragma unroll
    for (int k = 0; k < C; ++k) {
        middle2.c[k] = lo.c[k] + hi.c[k];
        w.c[k] = __builtin_fmaf(-0.5f * n, middle2.c[k], sums.s[k] + sums.s[k]);
        length = __builtin_fmaf(a.c[k], a.c[k], length);
    }
    float const inverse = __builtin_amdgcn_rcpf(length);
    if constexpr (PLAIN) plain += distances(sums, middle2, w, a, inverse);
    if constexpr (ORIENTED) {
        static_assert(C == 3, "");
        float const mean = sums.s[0] * __builtin_amdgcn_rcpf(n);
        float const c1 = __builtin_fmaf(-mean, sums.s[1], sums.q[0][1]), c2 = __builtin_fmaf(-mean, sums.s[2], sums.q[0][2]);
        float least = distances(sums, middle2, w, Color<C>{ a.c[0], copysignf(a.c[1], c1), copysignf(a.c[2], c2) }, inverse);
        bool const sure = min_f32(fabsf(c1), fabsf(c2)) > unsure;                // (a[0] = 0 is not)
        if (__any(!sure)) {
            float all = distances(sums, middle2, w, a, inverse);
            all = fminf(all, distances(sums, middle2, w, Color<C>{ a.c[0], -a.c[1], a.c[2] }, inverse));
            all = fminf(all, distances(sums, middle2, w, Color<C>{ a.c[0], a.c[1], -a.c[2] }, inverse));
            all = fminf(all, distances(sums, middle2, w, Color<C>{ a.c[0], -a.c[1], -a.c[2] }, inverse));
            if (!sure) least = all;
        }
        oriented += least;
    }
}

// Bounds of the partitions [first, last), multiples of four, of one or both picks.
template <class S, int SUBSETS, int C, bool ORIENTED, bool PLAIN>
BC7_TASK void bound_task(SearchPtr<S> lds, int b, int first, int last)
{
    first = __builtin_amdgcn_readfirstlane(first);
    last = __builtin_amdgcn_readfirstlane(last);
    constexpr int kind = SUBSETS == 3 ? kPickThree : kPickTwo;
    Color<C> const origin = texel<C, S>(lds, b, 0);
    Sums<C> total;
#pragma unroll 5
    for (int t = 1; t < 16; ++t) total.add(sub(texel<C, S>(lds, b, t), origin));
    float const offsets = total.trace();
    bool const bounded = offsets >= kLeastOffsets && offsets <= kMostOffsets;
    float const scale = bounded ? __builtin_amdgcn_rcpf(offsets) : 0.f, error = offsets * kBoundError;
    float const unsure = __builtin_fmaf(offsets, kUnsureOfOffsets, dot(origin, origin) * kUnsureOfTexels);
    if constexpr (ORIENTED) lds->scale[kind][b] = scale;
    if constexpr (PLAIN) lds->scale[kPickTwoAlpha][b] = scale;
    // Whether bounds are in vain (see kNearLine): then every partition is estimated (lowest stays as it is).
    {
        Color<C> lo, hi;
        subset_box<C, 16, false, S>(lds, b, kAllTexels, origin, lo, hi, total);
        float oriented = 0.f, plain = 0.f;
        add_distances<C, ORIENTED, !ORIENTED>(16.f, total, lo, hi, unsure, oriented, plain);
        Color<C> const a = sub(hi, lo);
        float const square = dot(a, a), distances = ORIENTED ? oriented : plain;
        bool counts = bounded;
        if constexpr (ORIENTED && SUBSETS == 2) {            // two colours lie at the ends of the diagonal
            float about = offsets;
#pragma unroll
            for (int k = 0; k < C; ++k) {
                float const middle2 = lo.c[k] + hi.c[k];
                about = __builtin_fmaf(-middle2, __builtin_fmaf(-4.f, middle2, total.s[k]), about);
            }
            counts = counts && about < square * 3.996f;
        }
        auto const near = [&](float limit) { return __popcll(__ballot(counts && distances < square * limit)); };
        if constexpr (ORIENTED) {
            if (2 * __popcll(__ballot(bounded)) + 5 * near(1.f / 8.f) + 5 * near(1.f / 16.f) + 6 * near(1.f / 24.f) + 7 * near(1.f / 37.f)
                + 15 * near(kNearLine) > kMostExpected) return;
        } else {
            if (near(kNearLine) >= 48) return;
        }
    }
    uint32_t lowestOriented = ~0u, lowestPlain = ~0u, codesOriented = 0, codesPlain = 0;
#pragma unroll 1
    for (int p = first; p < last; ++p) {
        uint32_t const word = partition_word<SUBSETS>(p);
        uint32_t masks[SUBSETS];                             // the largest subset last
#pragma unroll
        for (int s = 0; s < SUBSETS; ++s) masks[s] = spread_mask(word, uint32_t(s));
#pragma unroll
        for (int s = 0; s + 1 < SUBSETS; ++s)
            if (__popc(masks[s]) > __popc(masks[SUBSETS - 1])) { uint32_t const m = masks[s]; masks[s] = masks[SUBSETS - 1]; masks[SUBSETS - 1] = m; }
        Sums<C> rest = total;
        float oriented = 0.f, plain = 0.f;
        uint32_t mask = masks[0];
#pragma unroll 1
        for (int s = 0; s + 1 < SUBSETS; ++s) {
            Sums<C> sums;
            Color<C> lo, hi;
            mask = __builtin_amdgcn_readfirstlane(mask);
            switch (__popc(mask)) {                          // the sizes that the partitions' smaller subsets have
            case 2:  if constexpr (SUBSETS == 3) subset_box<C, 2, true, S>(lds, b, mask, origin, lo, hi, sums); break;
            case 3:  subset_box<C, 3, true, S>(lds, b, mask, origin, lo, hi, sums); break;
            case 4:  subset_box<C, 4, true, S>(lds, b, mask, origin, lo, hi, sums); break;
            case 5:  subset_box<C, 5, true, S>(lds, b, mask, origin, lo, hi, sums); break;
            case 6:  subset_box<C, 6, true, S>(lds, b, mask, origin, lo, hi, sums); break;
            default: if constexpr (SUBSETS == 2) subset_box<C, 8, true, S>(lds, b, mask, origin, lo, hi, sums); break;
            }
            add_distances<C, ORIENTED, PLAIN>(float(__popc(mask)), sums, lo, hi, unsure, oriented, plain);
            rest.remove(sums);
            mask = masks[SUBSETS - 2];
        }
        Sums<C> none;
        Color<C> lo, hi;
        mask = __builtin_amdgcn_readfirstlane(masks[SUBSETS - 1]);
        switch (__popc(mask)) {                              // and their largest
        case 6:  if constexpr (SUBSETS == 3) subset_box<C, 6, false, S>(lds, b, mask, origin, lo, hi, none); break;
        case 7:  if constexpr (SUBSETS == 3) subset_box<C, 7, false, S>(lds, b, mask, origin, lo, hi, none); break;
        case 8:  subset_box<C, 8, false, S>(lds, b, mask, origin, lo, hi, none); break;
        case 10: if constexpr (SUBSETS == 2) subset_box<C, 10, false, S>(lds, b, mask, origin, lo, hi, none); break;
        case 11: if constexpr (SUBSETS == 2) subset_box<C, 11, false, S>(lds, b, mask, origin, lo, hi, none); break;
        case 12: subset_box<C, 12, false, S>(lds, b, mask, origin, lo, hi, none); break;
        default: if constexpr (SUBSETS == 2) subset_box<C, 13, false, S>(lds, b, mask, origin, lo, hi, none); break;
        }
        add_distances<C, ORIENTED, PLAIN>(float(__popc(mask)), rest, lo, hi, unsure, oriented, plain);
        auto const consider = [&](float distances, uint32_t& lowest, uint32_t& codes) {
            float const bound = bounded ? fmaxf(distances - error, 0.f) : 0.f;
            lowest = min(lowest, (__float_as_uint(bound) & ~63u) | uint32_t(p));
            codes = codes >> 8 | error_code(bound, scale) << 24;
        };
        if constexpr (ORIENTED) consider(oriented, lowestOriented, codesOriented);
        if constexpr (PLAIN) consider(plain, lowestPlain, codesPlain);
        if ((p & 3) == 3) {
            if constexpr (ORIENTED) lds->scratch.bounds.codes[kind][p >> 2][b] = codesOriented;
            if constexpr (PLAIN) lds->scratch.bounds.codes[kPickTwoAlpha][p >> 2][b] = codesPlain;
        }
    }
    if constexpr (ORIENTED) __hip_atomic_fetch_min(&lds->lowest[kind][b], lowestOriented, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if constexpr (PLAIN) __hip_atomic_fetch_min(&lds->lowest[kPickTwoAlpha][b], lowestPlain, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Sums of one refinement round (refine() above) and its solution; false when the system is singular.
template <int C> struct Refinement {
    float a2 = 0.f, b2 = 0.f, ab = 0.f;
    Color<C> ax, bx;
    BC7_INLINE Refinement()
    {
#pragma unroll
        for (int k = 0; k < C; ++k) ax.c[k] = bx.c[k] = 0.f;
    }
    // f: the texel's saturated place between the ends
    BC7_INLINE void add(float f, Color<C> const& p, int indexBits)
    {
        float const scale = float((1u << indexBits) - 1u), iscale = 1.f / scale;
        float const beta = rintf(f * scale) * iscale, alpha = 1.f - beta;
        a2 += alpha * alpha; b2 += beta * beta; ab += alpha * beta;
#pragma unroll
        for (int k = 0; k < C; ++k) { ax.c[k] += alpha * p.c[k]; bx.c[k] += beta * p.c[k]; }
    }
    BC7_INLINE bool solve(Color<C>& e0, Color<C>& e1) const
    {
        float const denom = a2 * b2 - ab * ab;
        if (!(fabsf(denom) > 0.0001f)) return false;
        float const factor = 1.f / denom;
#pragma unroll
        for (int k = 0; k < C; ++k) {
            float const a = saturate((ax.c[k] * b2 - bx.c[k] * ab) * factor), b = saturate((bx.c[k] * a2 - ax.c[k] * ab) * factor);
            if (!(e0.c[k] == 0.f || e0.c[k] == 1.f)) e0.c[k] = a;
            if (!(e1.c[k] == 0.f || e1.c[k] == 1.f)) e1.c[k] = b;
        }
        return true;
    }
};

// Start ends of the lane's own subset: its box, oriented if asked.
template <int C, bool ORIENT, class S> BC7_INLINE void listed_ends(SearchPtr<S> lds, int b, uint32_t mask, Color<C>& e0, Color<C>& e1)
{
    Color<C> center;
#pragma unroll
    for (int k = 0; k < C; ++k) { e0.c[k] = FLT_MAX; e1.c[k] = -FLT_MAX; center.c[k] = 0.f; }
    for (uint32_t m = mask; m; m &= m - 1) {
        Color<C> const p = texel<C, S>(lds, b, first_texel(m));
#pragma unroll
        for (int k = 0; k < C; ++k) { e0.c[k] = min_f32(e0.c[k], p.c[k]); e1.c[k] = max_f32(e1.c[k], p.c[k]); center.c[k] += p.c[k]; }
    }
    if constexpr (ORIENT) {
        float const count = float(__popc(mask));
#pragma unroll
        for (int k = 0; k < C; ++k) center.c[k] /= count;
        float cov[C][C] = {};
        for (uint32_t m = mask; m; m &= m - 1) add_covariance(cov, sub(texel<C, S>(lds, b, first_texel(m)), center));
        orient_by(cov, e0, e1);
    }
}
// The estimated error of the lane's own partition, into the pick of its kind: the smallest of these numbers is the smallest
// error (errors are not negative) and the first partition that has it.
template <class S> BC7_INLINE void put_estimate(SearchPtr<S> lds, int kind, int b, int partition, float error)
{
    uint64_t const key = uint64_t(__float_as_uint(error)) << 32 | uint32_t(partition);
    __hip_atomic_fetch_min(&lds->picks[kind][b], key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// For the modes 0 to 3: squared error if every texel took the nearest of eight points between its subset's oriented ends.
template <class S, int SUBSETS>
BC7_TASK void estimate_task(SearchPtr<S> lds, int b, int partition)
{
    constexpr float maxIndex = 7.f, indexScale = 1.f / maxIndex;
    uint32_t const word = partition_word<SUBSETS>(partition);
    float error = 0.f;
#pragma unroll 1
    for (int s = 0; s < SUBSETS; ++s) {
        uint32_t const mask = spread_mask(word, uint32_t(s));
        Color<3> e0, e1;
        listed_ends<3, true, S>(lds, b, mask, e0, e1);
        Color<3> const axis = sub(e1, e0);
        float const mul = inverse_square(axis);
        float e = 0.f;
        for (uint32_t m = mask; m; m &= m - 1) {
            Color<3> const p = sub(texel<3, S>(lds, b, first_texel(m)), e0);
            float const f = rintf(dot(p, axis) * mul * maxIndex) * indexScale;
            Color<3> diff;
#pragma unroll
            for (int k = 0; k < 3; ++k) diff.c[k] = f * axis.c[k] - p.c[k];
            e += dot(diff, diff);
        }
        error = s == 0 ? e : error + e;
    }
    put_estimate<S>(lds, SUBSETS == 3 ? kPickThree : kPickTwo, b, partition, error);
}

// For mode 7: of four points between the corners of its subset's box.  The bounds leave the most partitions of this kind,
// so that lists of texels, whose addresses are a chain, would be the longest part of the search: here all texels are
// loaded at once and go through the code of both subsets, as NaNs (which minima and maxima leave out) or zeros where they
// belong to the other.
template <class S, int C>
BC7_TASK void estimate_corners_task(SearchPtr<S> lds, int b, int partition)
{
    constexpr float maxIndex = 3.f, indexScale = 1.f / maxIndex;
    uint32_t const word = partition_word<2>(partition);
    Color<C> px[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) px[t] = texel<C, S>(lds, b, t);
    auto const second = [&](int t) { return uint32_t(int32_t(word << (31 - 2 * t)) >> 31); };        // all ones if the texel is in subset 1
    auto const ored = [](float v, uint32_t m) { return __uint_as_float(__float_as_uint(v) | m); };
    Color<C> lo[2], axis[2];
#pragma unroll
    for (int k = 0; k < C; ++k) {
        float l0 = FLT_MAX, h0 = -FLT_MAX, l1 = FLT_MAX, h1 = -FLT_MAX;
#pragma unroll
        for (int t = 0; t < 16; t += 2) {
            float const a0 = ored(px[t].c[k], second(t)), b0 = ored(px[t + 1].c[k], second(t + 1));
            float const a1 = ored(px[t].c[k], ~second(t)), b1 = ored(px[t + 1].c[k], ~second(t + 1));
            l0 = min3_f32(l0, a0, b0); h0 = max3_f32(h0, a0, b0);
            l1 = min3_f32(l1, a1, b1); h1 = max3_f32(h1, a1, b1);
        }
        lo[0].c[k] = l0; axis[0].c[k] = h0 - l0;
        lo[1].c[k] = l1; axis[1].c[k] = h1 - l1;
    }
    float const mul0 = inverse_square(axis[0]), mul1 = inverse_square(axis[1]);
    float error0 = 0.f, error1 = 0.f;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        uint32_t const m = second(t);
        Color<C> p, ax, diff;
#pragma unroll
        for (int k = 0; k < C; ++k) { p.c[k] = px[t].c[k] - (m ? lo[1].c[k] : lo[0].c[k]); ax.c[k] = m ? axis[1].c[k] : axis[0].c[k]; }
        float const f = rintf(dot(p, ax) * (m ? mul1 : mul0) * maxIndex) * indexScale;
#pragma unroll
        for (int k = 0; k < C; ++k) diff.c[k] = f * ax.c[k] - p.c[k];
        float const d = dot(diff, diff);
        error0 += m ? 0.f : d;
        error1 += m ? d : 0.f;
    }
    put_estimate<S>(lds, kPickTwoAlpha, b, partition, error0 + error1);
}

enum { kThree = 0, kTwo, kCorners3, kCorners4 };            // what a search estimates: pick kinds, the last by channels
template <class S> BC7_INLINE void estimate_one(SearchPtr<S> lds, int what, int b, int partition)      // what: uniform
{
    if (what == kThree)         estimate_task<S, 3>(lds, b, partition);
    else if (what == kTwo)      estimate_task<S, 2>(lds, b, partition);
    else if (what == kCorners3) estimate_corners_task<S, 3>(lds, b, partition);
    else                        estimate_corners_task<S, 4>(lds, b, partition);
}

// With all bounds of a search there: the error of the partition with the smallest one, and the partitions whose bounds do
// not exceed it into the search's queue.  `mine`: the lane is its block's only one.  Where that leaves more of them than
// one in five all are estimated, with code for their subsets' sizes, which is then the quicker way.
template <class S>
BC7_TASK void select_task(SearchPtr<S> lds, int b, int what, int search, int mine)
{
    what = __builtin_amdgcn_readfirstlane(what);
    search = __builtin_amdgcn_readfirstlane(search);
    int const kind = what == kCorners4 ? int(kPickTwoAlpha) : what;
    uint32_t const lowest = lds->lowest[kind][b];
    uint64_t mask = 0;
    if (__any(lowest != ~0u)) {                              // (else there are no bounds)
        estimate_one<S>(lds, what, b, int(lowest & 63u));
        uint64_t const pick = lds->picks[kind][b];
        uint32_t const bits = uint32_t(pick >> 32), code = error_code(__uint_as_float(bits), lds->scale[kind][b]);
#pragma unroll 4
        for (int j = 0; j < 16; ++j) {
            uint32_t const codes = lds->scratch.bounds.codes[kind][j][b];
            uint32_t four = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) four |= ((codes >> (8 * i)) & 0xffu) <= code ? 1u << i : 0u;
            mask |= uint64_t(four) << (4 * j);
        }
        // not the picked one again; where it leaves no error only those before it can take its place
        uint64_t const picked = uint64_t(1) << (uint32_t(pick) & 63u);
        mask &= bits == 0u ? picked - 1u : ~picked;
        if (!mine) mask = 0;
        int const n = __popcll(mask);
        int place = n ? atomicAdd((int*)&lds->queued[search], n) : 0;
        if (!__any(place + n > kQueued)) {
            for (; mask; mask &= mask - 1u, ++place) lds->queues[search][place] = uint16_t(__builtin_ctzll(mask) << 7 | b);
            return;
        }
    }
    if ((threadIdx.x & 63) == 0) {
        lds->queued[search] = 0;
        lds->whole[atomicAdd((int*)&lds->wholes, 1)] = uint8_t(search);
    }
}

// ---- estimates of whole ranges of partitions
//
// All lanes take the same partition: for each subset its texels are read into registers and go through code for exactly
// that many.

// Squared error of N texels if each took the nearest of the 2^BITS points between e0 and e1.
template <int BITS, int C, int N> BC7_INLINE float estimate_of(Color<C> const (&px)[N], Color<C> const& e0, Color<C> const& e1)
{
    Color<C> const axis = sub(e1, e0);
    float const mul = inverse_square(axis);
    constexpr float maxIndex = float((1u << BITS) - 1u), indexScale = 1.f / maxIndex;
    float error = 0.f;
#pragma unroll
    for (int t = 0; t < N; ++t) {
        Color<C> const p = sub(px[t], e0);
        float const f = rintf(dot(p, axis) * mul * maxIndex) * indexScale;
        Color<C> diff;
#pragma unroll
        for (int k = 0; k < C; ++k) diff.c[k] = f * axis.c[k] - p.c[k];
        error += dot(diff, diff);
    }
    return error;
}

// Estimated errors of the subset `mask` (uniform, of N texels): with oriented ends and eight points (three-channel modes 0
// to 3) if ORIENTED, with the box's own corners and four points (mode 7) if PLAIN.
struct SubsetErrors { float oriented, plain; };
template <int C, int N, bool ORIENTED, bool PLAIN, class S> BC7_INLINE SubsetErrors subset_errors(SearchPtr<S> lds, int b, uint32_t mask)
{
    Color<C> px[N];
#pragma unroll
    for (int t = 0; t < N; ++t) { px[t] = texel<C, S>(lds, b, first_texel(mask)); mask &= mask - 1; }
    Color<C> lo, hi;
#pragma unroll
    for (int k = 0; k < C; ++k) {
        lo.c[k] = FLT_MAX; hi.c[k] = -FLT_MAX;
#pragma unroll
        for (int t = 0; t + 1 < N; t += 2) { lo.c[k] = min3_f32(lo.c[k], px[t].c[k], px[t + 1].c[k]); hi.c[k] = max3_f32(hi.c[k], px[t].c[k], px[t + 1].c[k]); }
        if constexpr (N & 1) { lo.c[k] = min_f32(lo.c[k], px[N - 1].c[k]); hi.c[k] = max_f32(hi.c[k], px[N - 1].c[k]); }
    }
    SubsetErrors e{ 0.f, 0.f };
    if constexpr (PLAIN) e.plain = estimate_of<2>(px, lo, hi);
    if constexpr (ORIENTED) {
        Color<C> center;
#pragma unroll
        for (int k = 0; k < C; ++k) {
            center.c[k] = 0.f;
#pragma unroll
            for (int t = 0; t < N; ++t) center.c[k] += px[t].c[k];
            center.c[k] /= float(N);
        }
        float cov[C][C] = {};
#pragma unroll
        for (int t = 0; t < N; ++t) add_covariance(cov, sub(px[t], center));
        orient_by(cov, lo, hi);
        e.oriented = estimate_of<3>(px, lo, hi);
    }
    return e;
}

// Of the partitions [first, last) of `pick` the one with the smallest estimated error (the first of equals), as error bits
// << 32 | partition: errors are not negative, so the smallest such number over several ranges is the same over all of them.
template <class S, int SUBSETS, int C, bool ORIENTED, bool PLAIN>
BC7_TASK void pick_task(SearchPtr<S> lds, int b, int first, int last)
{
    first = __builtin_amdgcn_readfirstlane(first);
    last = __builtin_amdgcn_readfirstlane(last);
    uint64_t bestOriented = ~uint64_t(0), bestPlain = ~uint64_t(0);
#pragma unroll 1
    for (int p = first; p < last; ++p) {
        uint32_t const word = partition_word<SUBSETS>(p);
        SubsetErrors error{ 0.f, 0.f };
#pragma unroll 1
        for (int s = 0; s < SUBSETS; ++s) {
            uint32_t const mask = spread_mask(word, uint32_t(s));
            SubsetErrors e{ 0.f, 0.f };
            switch (__popc(mask)) {                          // the sizes that the partitions' subsets have
            case 2:  if constexpr (SUBSETS == 3) e = subset_errors<C, 2, ORIENTED, PLAIN, S>(lds, b, mask); break;
            case 3:  e = subset_errors<C, 3, ORIENTED, PLAIN, S>(lds, b, mask); break;
            case 4:  e = subset_errors<C, 4, ORIENTED, PLAIN, S>(lds, b, mask); break;
            case 5:  e = subset_errors<C, 5, ORIENTED, PLAIN, S>(lds, b, mask); break;
            case 6:  e = subset_errors<C, 6, ORIENTED, PLAIN, S>(lds, b, mask); break;
            case 7:  if constexpr (SUBSETS == 3) e = subset_errors<C, 7, ORIENTED, PLAIN, S>(lds, b, mask); break;
            case 8:  e = subset_errors<C, 8, ORIENTED, PLAIN, S>(lds, b, mask); break;
            case 10: if constexpr (SUBSETS == 2) e = subset_errors<C, 10, ORIENTED, PLAIN, S>(lds, b, mask); break;
            case 11: if constexpr (SUBSETS == 2) e = subset_errors<C, 11, ORIENTED, PLAIN, S>(lds, b, mask); break;
            case 12: e = subset_errors<C, 12, ORIENTED, PLAIN, S>(lds, b, mask); break;
            case 13: if constexpr (SUBSETS == 2) e = subset_errors<C, 13, ORIENTED, PLAIN, S>(lds, b, mask); break;
            default: break;
            }
            error.oriented = s == 0 ? e.oriented : error.oriented + e.oriented;
            error.plain = s == 0 ? e.plain : error.plain + e.plain;
        }
        auto const consider = [&](uint64_t& best, float e) {
            uint64_t const key = uint64_t(__float_as_uint(e)) << 32 | uint32_t(p);
            best = key < best ? key : best;
        };
        if constexpr (ORIENTED) consider(bestOriented, error.oriented);
        if constexpr (PLAIN) consider(bestPlain, error.plain);
    }
    if constexpr (ORIENTED) __hip_atomic_fetch_min(&lds->picks[SUBSETS == 3 ? kPickThree : kPickTwo][b], bestOriented, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if constexpr (PLAIN) __hip_atomic_fetch_min(&lds->picks[kPickTwoAlpha][b], bestPlain, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <int C, int INDEX_BITS, class S> BC7_INLINE void listed_refine(SearchPtr<S> lds, int b, uint32_t mask, Color<C>& e0, Color<C>& e1)
{
#pragma unroll 1
    for (int iter = 0; iter < 2; ++iter) {
        Color<C> const axis = sub(e1, e0);
        float const mul = inverse_square(axis);
        Refinement<C> sums;
        for (uint32_t m = mask; m; m &= m - 1) {
            Color<C> const p = texel<C, S>(lds, b, first_texel(m));
            sums.add(saturate(dot(sub(p, e0), axis) * mul), p, INDEX_BITS);
        }
        if (!sums.solve(e0, e1)) break;
    }
}

// Dequantised endpoints: where texels fall between them and what a decoder shows there.
template <int C, int INDEX_BITS> struct Decoded {
    Color<C> e0, axis;
    float mul;
    int base[C], step[C];
    BC7_INLINE Decoded(Quantized<C> const& q0, Quantized<C> const& q1, int endpointBits)
    {
        Color<C> e1;
#pragma unroll
        for (int k = 0; k < C; ++k) {
            int const x0 = expand8(q0.c[k], endpointBits), x1 = expand8(q1.c[k], endpointBits);
            base[k] = 64 * x0 + 32; step[k] = x1 - x0;
            e0.c[k] = unorm_quotient(float(x0), 255.f, 1.f / 255.f); e1.c[k] = unorm_quotient(float(x1), 255.f, 1.f / 255.f);
        }
        axis = sub(e1, e0);
        mul = inverse_square(axis);
    }
    // The texel's index, and its error added.  Weights of complemented indices on swapped endpoints are complements
    // themselves, so the error is that of the final form whichever way the anchor turns out.
    BC7_INLINE uint32_t index(Color<C> const& p, float& error) const
    {
        constexpr float top = float((1u << INDEX_BITS) - 1u);
        float const place = rintf(saturate(dot(sub(p, e0), axis) * mul) * top);
        int const w = int(rintf(place * (64.f / top)));
        Color<C> diff;
#pragma unroll
        for (int k = 0; k < C; ++k) diff.c[k] = unorm_quotient(float((base[k] + __mul24(step[k], w)) >> 6), 255.f, 1.f / 255.f) - p.c[k];
        error += dot(diff, diff);
        return uint32_t(place);
    }
};

template <class W, class E> BC7_INLINE void put_candidate(W words, E errors, float error, uint64_t lo, uint64_t hi)
{
    *errors = error;
    words->x = uint32_t(lo); words->y = uint32_t(lo >> 32); words->z = uint32_t(hi); words->w = uint32_t(hi >> 32);
}

template <class S, class M, int C, bool ORIENT>
BC7_TASK void finish_task(SearchPtr<S> lds, int b, int pick, int slot)
{
    pick = __builtin_amdgcn_readfirstlane(pick);
    slot = __builtin_amdgcn_readfirstlane(slot);
    constexpr int N = 2 * M::subsets;
    int partition = 0;
    bool none = false;
    if constexpr (M::subsets > 1) {
        // A NaN or infinite texel can leave every partition without a finite estimate: then none is "best", and
        // partition 0 is tried with endpoints of zero.
        uint64_t const key = lds->picks[pick][b];
        none = uint32_t(key >> 32) >= __float_as_uint(FLT_MAX);
        partition = none ? 0 : int(uint32_t(key));
    }
    if (partition >= (1 << M::partitionBits)) {              // mode 0 has sixteen partitions only
        lds->scratch.late.errors[slot][b] = __uint_as_float(0x7f800000u);    // never taken
        return;
    }
    uint32_t const word = partition_word<M::subsets>(partition);
    Color<C> e[N];
    Quantized<C> q[N];
#pragma unroll
    for (int s = 0; s < M::subsets; ++s) {
        uint32_t const mask = spread_mask(word, uint32_t(s));
        listed_ends<C, ORIENT, S>(lds, b, mask, e[2 * s], e[2 * s + 1]);
        if (none) {
#pragma unroll
            for (int k = 0; k < C; ++k) e[2 * s].c[k] = e[2 * s + 1].c[k] = 0.f;
        }
        listed_refine<C, M::indexBits, S>(lds, b, mask, e[2 * s], e[2 * s + 1]);
    }
    quantize_endpoints<M, C>(e, q);
    uint64_t indices = 0;
    float error = 0.f;
    int anchors[M::subsets];
#pragma unroll
    for (int s = 0; s < M::subsets; ++s) {
        Decoded<C, M::indexBits> const ends(q[2 * s], q[2 * s + 1], M::endpointBits);
        float e2 = 0.f;
        uint64_t ones = 0;
        for (uint32_t m = spread_mask(word, uint32_t(s)); m; m &= m - 1) {
            int const t = first_texel(m);
            uint64_t const one = uint64_t(1) << (t * M::indexBits);
            indices |= uint64_t(ends.index(texel<C, S>(lds, b, t), e2)) << (t * M::indexBits);
            ones |= one;
        }
        error = s == 0 ? e2 : error + e2;
        // a decoder assumes the anchor's top index bit to be 0: if it is 1 the endpoints trade places
        anchors[s] = subset_anchor<M::subsets>(partition, s);
        if ((indices >> (anchors[s] * M::indexBits + M::indexBits - 1)) & 1u) {
            indices ^= ones * ((1u << M::indexBits) - 1u);
            Quantized<C> const x = q[2 * s]; q[2 * s] = q[2 * s + 1]; q[2 * s + 1] = x;
        }
    }
    Bits bits;
    bits.put(M::id + 1, 1u << M::id);
    bits.put(M::partitionBits, uint32_t(partition));
    constexpr int drop = M::pbit == kNoPBit ? 0 : 1;
#pragma unroll
    for (int k = 0; k < C; ++k)
#pragma unroll
        for (int i = 0; i < N; ++i) bits.put(M::endpointBits - drop, uint32_t(q[i].c[k]) >> drop);
    if constexpr (M::pbit == kPBitPerEndpoint) {
#pragma unroll
        for (int i = 0; i < N; ++i) bits.put(1, uint32_t(q[i].c[0]));
    }
    if constexpr (M::pbit == kPBitPerSubset) {
#pragma unroll
        for (int s = 0; s < M::subsets; ++s) bits.put(1, uint32_t(q[2 * s].c[0]));
    }
    constexpr int top = M::indexBits - 1;
    if constexpr (M::subsets == 3) {
        indices = without_bit(indices, max(anchors[1], anchors[2]) * M::indexBits + top);
        indices = without_bit(indices, min(anchors[1], anchors[2]) * M::indexBits + top);
    } else if constexpr (M::subsets == 2) {
        indices = without_bit(indices, anchors[1] * M::indexBits + top);
    }
    indices = without_bit(indices, top);
    put_indices(bits.lo, bits.hi, bits.at, indices);
    put_candidate(&lds->scratch.late.words[slot][b], &lds->scratch.late.errors[slot][b], error, bits.lo, bits.hi);
}

// The colour plane and the scalar plane of a texel under the lane's channel rotation.  C = 2: every alpha of the lane's
// block is 1 and the rotation takes a colour channel out, so that the plane is the other two and that 1 in its place: its
// differences are zeros, which sums do not see, and its ends stay 1, which decodes to 1.
template <int C, class S> BC7_INLINE void planes_of(SearchPtr<S> lds, int b, int t, int rotation, Color<C>& plane, Color<1>& a)
{
    Color<4> const p = texel<4, S>(lds, b, t);
    if constexpr (C == 2) {
        plane.c[0] = rotation == 1 ? p.c[1] : p.c[0];
        plane.c[1] = rotation == 3 ? p.c[1] : p.c[2];
        a.c[0] = rotation == 1 ? p.c[0] : rotation == 2 ? p.c[1] : p.c[2];
    } else {
        plane.c[0] = rotation == 1 ? p.c[3] : p.c[0];
        plane.c[1] = rotation == 2 ? p.c[3] : p.c[1];
        plane.c[2] = rotation == 3 ? p.c[3] : p.c[2];
        a.c[0] = rotation == 0 ? p.c[3] : rotation == 1 ? p.c[0] : rotation == 2 ? p.c[1] : p.c[2];
    }
}

template <int FORM> struct DualForm {                        // mode 4 with 2-bit colour indices, with 3-bit ones, mode 5
    static constexpr int mode = FORM == 2 ? 5 : 4, colorIndexBits = FORM == 1 ? 3 : 2, alphaIndexBits = FORM == 0 ? 3 : 2;
    static constexpr int colorBits = FORM == 2 ? 7 : 5, alphaBits = FORM == 2 ? 8 : 6;
};

template <class S, int FORM, int C>
BC7_TASK void dual_plane_form(SearchPtr<S> lds, int b, int rotation, Ends<C> color, Ends<1> alpha, Best& best)
{
    using F = DualForm<FORM>;
    Quantized<C> q0, q1;
    Quantized<1> qa0, qa1;
#pragma unroll
    for (int k = 0; k < C; ++k) { q0.c[k] = quantize(color.e0.c[k], F::colorBits); q1.c[k] = quantize(color.e1.c[k], F::colorBits); }
    qa0.c[0] = quantize(alpha.e0.c[0], F::alphaBits); qa1.c[0] = quantize(alpha.e1.c[0], F::alphaBits);
    Decoded<C, F::colorIndexBits> const colorEnds(q0, q1, F::colorBits);
    Decoded<1, F::alphaIndexBits> const alphaEnds(qa0, qa1, F::alphaBits);
    uint64_t colorIndices = 0, alphaIndices = 0;
    float colorError = 0.f, alphaError = 0.f;
#pragma unroll 4
    for (int t = 0; t < 16; ++t) {
        Color<C> rgb;
        Color<1> a;
        planes_of<C, S>(lds, b, t, rotation, rgb, a);
        colorIndices |= uint64_t(colorEnds.index(rgb, colorError)) << (t * F::colorIndexBits);
        alphaIndices |= uint64_t(alphaEnds.index(a, alphaError)) << (t * F::alphaIndexBits);
    }
    float const error = colorError + alphaError;
    if (error > best.error) return;
    auto const complemented = [](uint64_t v, int bits) { return bits == 2 ? v ^ 0xffffffffull : v ^ 0xffffffffffffull; };
    if (colorIndices & (1u << (F::colorIndexBits - 1))) { colorIndices = complemented(colorIndices, F::colorIndexBits); Quantized<C> const x = q0; q0 = q1; q1 = x; }
    if (alphaIndices & (1u << (F::alphaIndexBits - 1))) { alphaIndices = complemented(alphaIndices, F::alphaIndexBits); Quantized<1> const x = qa0; qa0 = qa1; qa1 = x; }
    Bits bits;
    bits.put(F::mode + 1, 1u << F::mode);
    bits.put(2, uint32_t(rotation));
    if constexpr (F::mode == 4) bits.put(1, FORM == 1 ? 1u : 0u);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        uint32_t v0, v1;
        if constexpr (C == 2) {                              // the alpha's place is that of the rotation
            constexpr uint32_t one = (1u << F::colorBits) - 1u;
            v0 = rotation == k + 1 ? one : uint32_t(k == 0 ? q0.c[0] : k == 2 ? q0.c[1] : rotation == 1 ? q0.c[0] : q0.c[1]);
            v1 = rotation == k + 1 ? one : uint32_t(k == 0 ? q1.c[0] : k == 2 ? q1.c[1] : rotation == 1 ? q1.c[0] : q1.c[1]);
        } else {
            v0 = uint32_t(q0.c[k]); v1 = uint32_t(q1.c[k]);
        }
        bits.put(F::colorBits, v0); bits.put(F::colorBits, v1);
    }
    bits.put(F::alphaBits, uint32_t(qa0.c[0])); bits.put(F::alphaBits, uint32_t(qa1.c[0]));
    colorIndices = without_bit(colorIndices, F::colorIndexBits - 1);
    alphaIndices = without_bit(alphaIndices, F::alphaIndexBits - 1);
    // mode 4 stores its 2-bit indices first, then the 3-bit ones; mode 5 colour first, then the scalar
    constexpr int firstBits = 16 * (FORM == 1 ? F::alphaIndexBits : F::colorIndexBits) - 1;
    put_indices(bits.lo, bits.hi, bits.at, FORM == 1 ? alphaIndices : colorIndices);
    put_indices(bits.lo, bits.hi, bits.at + firstBits, FORM == 1 ? colorIndices : alphaIndices);
    best.error = error; best.lo = bits.lo; best.hi = bits.hi;
}

// The refined ends of one rotation's planes, for 2-bit and for 3-bit indices: mode 5 shares its colour ends with mode
// 4's narrow form and its scalar ends with the wide form.
template <class S, int C>
BC7_TASK void dual_plane_ends(SearchPtr<S> lds, int b, int rotation, Ends<C> (&color)[2], Ends<1> (&alpha)[2])
{
    Ends<C> c;
    Ends<1> s;
    {
        Color<C> center;
        for (int k = 0; k < C; ++k) { c.e0.c[k] = FLT_MAX; c.e1.c[k] = -FLT_MAX; center.c[k] = 0.f; }
        s.e0.c[0] = FLT_MAX; s.e1.c[0] = -FLT_MAX;
#pragma unroll 4
        for (int t = 0; t < 16; ++t) {
            Color<C> rgb;
            Color<1> a;
            planes_of<C, S>(lds, b, t, rotation, rgb, a);
#pragma unroll
            for (int k = 0; k < C; ++k) { c.e0.c[k] = min_f32(c.e0.c[k], rgb.c[k]); c.e1.c[k] = max_f32(c.e1.c[k], rgb.c[k]); center.c[k] += rgb.c[k]; }
            s.e0.c[0] = min_f32(s.e0.c[0], a.c[0]); s.e1.c[0] = max_f32(s.e1.c[0], a.c[0]);
        }
#pragma unroll
        for (int k = 0; k < C; ++k) center.c[k] /= 16.f;
        float cov[C][C] = {};
#pragma unroll 4
        for (int t = 0; t < 16; ++t) {
            Color<C> rgb;
            Color<1> a;
            planes_of<C, S>(lds, b, t, rotation, rgb, a);
            add_covariance(cov, sub(rgb, center));
        }
        orient_by(cov, c.e0, c.e1);
    }
    color[0] = color[1] = c;
    alpha[0] = alpha[1] = s;
    bool colorGoesOn[2] = { true, true }, alphaGoesOn[2] = { true, true };
#pragma unroll 1
    for (int iter = 0; iter < 2; ++iter) {
        Refinement<C> colorSums[2];
        Refinement<1> alphaSums[2];
        Color<C> axis[2];
        Color<1> range[2];
        float mul[2], scale[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            axis[i] = sub(color[i].e1, color[i].e0); mul[i] = inverse_square(axis[i]);
            range[i] = sub(alpha[i].e1, alpha[i].e0); scale[i] = inverse_square(range[i]);
        }
#pragma unroll 2
        for (int t = 0; t < 16; ++t) {
            Color<C> rgb;
            Color<1> a;
            planes_of<C, S>(lds, b, t, rotation, rgb, a);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                colorSums[i].add(saturate(dot(sub(rgb, color[i].e0), axis[i]) * mul[i]), rgb, 2 + i);
                alphaSums[i].add(saturate(dot(sub(a, alpha[i].e0), range[i]) * scale[i]), a, 2 + i);
            }
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if (colorGoesOn[i]) colorGoesOn[i] = colorSums[i].solve(color[i].e0, color[i].e1);
            if (alphaGoesOn[i]) alphaGoesOn[i] = alphaSums[i].solve(alpha[i].e0, alpha[i].e1);
        }
    }
}

// ---- what rotations cannot win
//
// A decoder shows a plane of three channels as points of a line, each component rounded to eight bits, so that the plane's
// error is at least the squared distances from the best line, trace less largest eigenvalue of the centred moments, with the
// roundings taken off: sqrt(error) >= sqrt(distances) - 4 sqrt(3) / 510, sixteen texels of three components that round by 1/510
// (two where the third is an alpha of 1, which is shown exactly).  That holds for modes 4 and 5 of the rotation and for
// mode 6, whose line lies in four channels, with any three of them.
// Moments are of offsets from texel 0, T the sum of their squares, within 40 units of roundoff of T each, so that distances are
// within 240: kBoundError covers them.  The eigenvalue is bounded by m + 2 p, m the mean eigenvalue and 6 p^2 the squared
// deviations from it, and brought down by Newton's steps, which stay above the largest root of the characteristic
// polynomial; in units of the trace that and its derivative are within 2^-17 of themselves, which the steps leave out.
// Blocks whose T is no number between kLeastOffsets and kMostOffsets have no bounds.
template <class S> BC7_TASK void bound_rotations(SearchPtr<S> lds, int b)
{
    Color<4> const origin = texel<4, S>(lds, b, 0);
    Sums<4> sums;
#pragma unroll 5
    for (int t = 1; t < 16; ++t) sums.add(sub(texel<4, S>(lds, b, t), origin));
    float const offsets = sums.trace();
    bool const bounded = offsets >= kLeastOffsets && offsets <= kMostOffsets, ones = !(lds->alphas[b] & kNotOne);
    float m[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = i; j < 4; ++j) m[i][j] = m[j][i] = __builtin_fmaf(sums.s[i] * (-1.f / 16.f), sums.s[j], sums.q[i][j]);
    float least[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        int const x = r == 1 ? 3 : 0, y = r == 2 ? 3 : 1, z = r == 3 ? 3 : 2;
        float const trace = m[x][x] + m[y][y] + m[z][z], unit = __builtin_amdgcn_rcpf(trace);
        float const xx = m[x][x] * unit, yy = m[y][y] * unit, zz = m[z][z] * unit, xy = m[x][y] * unit, xz = m[x][z] * unit, yz = m[y][z] * unit;
        float const mixed = __builtin_fmaf(xy, xy, __builtin_fmaf(xz, xz, yz * yz));
        float const squares = __builtin_fmaf(xx, xx, __builtin_fmaf(yy, yy, __builtin_fmaf(zz, zz, mixed + mixed)));
        float const c1 = __builtin_fmaf(xx, yy, __builtin_fmaf(xx, zz, __builtin_fmaf(yy, zz, -mixed)));
        float const c0 = __builtin_fmaf(xx, __builtin_fmaf(yy, zz, -yz * yz), __builtin_fmaf(2.f * xy, xz * yz, -__builtin_fmaf(xz * xz, yy, xy * xy * zz)));
        float root = __builtin_fmaf(2.f, __builtin_amdgcn_sqrtf((fmaxf(squares - 1.f / 3.f, 0.f) + 0x1p-20f) * (1.f / 6.f)), 1.f / 3.f);
#pragma unroll
        for (int step = 0; step < 3; ++step) {
            float const value = __builtin_fmaf(root, __builtin_fmaf(root, root - 1.f, c1), -c0), slope = __builtin_fmaf(root, __builtin_fmaf(3.f, root, -2.f), c1);
            root = __builtin_fmaf(-fmaxf(value - 0x1p-17f, 0.f), __builtin_amdgcn_rcpf(fmaxf(slope, 0.f) + 0x1p-16f), root);
        }
        float const distances = __builtin_fmaf(trace, 1.f - 0x1p-16f - root, -kBoundError * offsets);
        float const rounding = (r != 0 && ones ? 1.4142f : 1.7321f) * (4.f * 1.001f / 510.f);
        float const rest = fmaxf(__builtin_amdgcn_sqrtf(fmaxf(distances, 0.f)) - rounding, 0.f);           // (a NaN: 0)
        least[r] = bounded ? rest * rest * (1.f - 0x1p-10f) : 0.f;
    }
    lds->early.words[b].x = __float_as_uint(least[0]); lds->early.words[b].y = __float_as_uint(least[1]);
    lds->early.words[b].z = __float_as_uint(least[2]); lds->early.words[b].w = __float_as_uint(least[3]);
}
// The rotation of the smallest bound; where alphas are 1 not 0, whose plane has all that leaves the other ones' lines.
template <class S> BC7_INLINE int first_rotation(SearchPtr<S> lds, int b)
{
    bool const ones = !(lds->alphas[b] & kNotOne);
    float const least[4] = { __uint_as_float(lds->early.words[b].x), __uint_as_float(lds->early.words[b].y), __uint_as_float(lds->early.words[b].z), __uint_as_float(lds->early.words[b].w) };
    int const low = ones || least[1] < least[0] ? 1 : 0, high = least[3] < least[2] ? 3 : 2;
    return fminf(least[2], least[3]) < (low ? least[1] : least[0]) ? high : low;
}
// With the first rotation's error: the other rotations and mode 6 into their lists where their bounds do not exceed it.
template <class S> BC7_INLINE void keep_candidates(SearchPtr<S> lds, int b, int first, float error, bool mine)
{
    float const least[4] = { __uint_as_float(lds->early.words[b].x), __uint_as_float(lds->early.words[b].y), __uint_as_float(lds->early.words[b].z), __uint_as_float(lds->early.words[b].w) };
    bool const ones = !(lds->alphas[b] & kNotOne);
    uint32_t plan = uint32_t(first);
#pragma unroll
    for (int r = 0; r < 4; ++r) if (r != first && !(least[r] > error)) plan |= kKeepRotation << r;
    if (!(fmaxf(fmaxf(least[0], least[1]), fmaxf(least[2], least[3])) > error)) plan |= kKeepSix;
    if (!mine) return;
    lds->plans[b] = plan;
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (plan & (kKeepRotation << r)) {
            if (r > 0 && ones) lds->flatRotations[atomicAdd((int*)&lds->kept[0], 1)] = uint16_t(r << 7 | b);
            else               lds->rotations[atomicAdd((int*)&lds->kept[1], 1)] = uint16_t(r << 7 | b);
        }
    if (plan & kKeepSix) lds->sixes[atomicAdd((int*)&lds->kept[2], 1)] = uint8_t(b);
}

// Modes 4 and 5 of the lane's rotation: the best of their three forms.
template <class S, int C> BC7_INLINE Best dual_planes(SearchPtr<S> lds, int b, int rotation)
{
    Ends<C> color[2];                                        // refined for 2-bit and 3-bit indices
    Ends<1> alpha[2];
    dual_plane_ends<S, C>(lds, b, rotation, color, alpha);
    Best best{ FLT_MAX, 0, 0 };
    dual_plane_form<S, 0, C>(lds, b, rotation, color[0], alpha[1], best);
    dual_plane_form<S, 1, C>(lds, b, rotation, color[1], alpha[0], best);
    dual_plane_form<S, 2, C>(lds, b, rotation, color[0], alpha[0], best);
    return best;
}

template <int GROUPS, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, 4)
bc7_compress_kernel(BlockCompressArgs a)
{
    // (a task of bounds sums the block first: as many partitions in one as leave a task for each wave)
    constexpr int BLOCKS = 64 * GROUPS, THREADS = 64 * WAVES, CHUNK = GROUPS == 1 ? 8 : 16, CHUNKS = 64 / CHUNK;
    constexpr bool ALONE = GROUPS == 1;                      // on its compute unit
    static_assert(THREADS >= 4 * BLOCKS && BLOCKS <= 128, "a thread per row of a block at least; seven bits number a block");
    using S = SearchLds<BLOCKS>;
    __shared__ S shared;
    SearchPtr<S> const lds = (SearchPtr<S>)&shared;
    int const tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Blocks: 8 x 8 per group, the groups side by side.  (Which blocks share a compute unit where all workgroups are
    // resident is no rule's to choose: with the lower half's columns turned by half a row 1024 x 1024 with alpha, or texture
    // beside grey, in the right half took 173 and 207 us for 181 and 235, in two opposite quadrants 183 and 235 for 175 and
    // 205.  A workgroup's groups half an image apart: 196 and 213, 198 and 215, for kinds then meet in one workgroup.)
    auto const block_x = [&](int b) { return int(blockIdx.x) * 8 * GROUPS + (b >> 6) * 8 + (b & 7); };
    auto const block_y = [&](int b) { return int(blockIdx.y) * 8 + ((b >> 3) & 7); };
    // the next of the tasks that the waves take in turn
    auto const next_task = [&](int counter) {
        int task = 0;
        if (lane == 0) task = atomicAdd(&shared.next[counter], 1);
        return __builtin_amdgcn_readfirstlane(task);
    };

    for (int i = tid; i < BLOCKS; i += THREADS) {
        shared.alphas[i] = 0u;
        for (int k = 0; k < kPicks; ++k) { shared.picks[k][i] = ~uint64_t(0); shared.lowest[k][i] = ~0u; }
    }
    if (tid < kSearches) shared.queued[tid] = shared.bounded[tid] = 0;
    if (tid < 2) shared.next[tid] = 0;
    if (tid == 0) shared.wholes = shared.selected = shared.rotated = shared.estimated = shared.kept[0] = shared.kept[1] = shared.kept[2] = 0;
    __syncthreads();
    if (int const b = tid % BLOCKS, row = tid / BLOCKS; row < 4) {
        int const bx = block_x(b), by = block_y(b);
        bool const inside = bx < a.widthInBlocks && by < a.heightInBlocks;
        uint32_t alphas = 0;
        float texels[1][4][4] = {};
        if (inside) source_rows<4, 1>(a, a.srcLeft + bx * 4, a.srcTop + by * 4 + row, 0, texels);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float const (&c)[4] = texels[0][i];
            alphas |= (c[3] < 1.f ? kBelowOne : 0u) | (c[3] != 1.f ? kNotOne : 0u);
            shared.texels[4 * row + i][b] = make_float4(c[0], c[1], c[2], c[3]);
        }
        if (alphas && inside) atomicOr(&shared.alphas[b], alphas);
    }
    __syncthreads();
    if (wave < 2) {                                          // wave 0 lists the opaque blocks, wave 1 those with alpha
        int count = 0;
        for (int g = 0; g < GROUPS; ++g) {
            int const b = 64 * g + lane;
            bool const mine = block_x(b) < a.widthInBlocks && block_y(b) < a.heightInBlocks && int(shared.alphas[b] & kBelowOne) == wave;
            uint64_t const ballot = __ballot(mine);
            if (mine) shared.blocks[wave][count + int(__builtin_amdgcn_mbcnt_hi(uint32_t(ballot >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(ballot), 0u)))] = uint8_t(b);
            count += __popcll(ballot);
        }
        if (lane == 0) shared.counts[wave] = count;
    }
    __syncthreads();
    int const opaque = __builtin_amdgcn_readfirstlane(shared.counts[0]), withAlpha = __builtin_amdgcn_readfirstlane(shared.counts[1]);
    int const opaqueGroups = (opaque + 63) / 64, alphaGroups = (withAlpha + 63) / 64, groups = opaqueGroups + alphaGroups;
    // the lane's block of a group of one kind (lanes beyond the last block repeat it)
    auto const block_of = [&](int kind, int group) { return int(shared.blocks[kind][min(64 * group + lane, (kind ? withAlpha : opaque) - 1)]); };
    auto const block_of_group = [&](int group) { return group < opaqueGroups ? block_of(0, group) : block_of(1, group - opaqueGroups); };
    auto const own_lane = [&](int group) { return 64 * (group < opaqueGroups ? group : group - opaqueGroups) + lane < (group < opaqueGroups ? opaque : withAlpha); };

    // Waits for the earlier tasks that a task builds upon: each was taken before it, by a wave that comes to its end.
    auto const wait_for = [&](int& counter, int count) {
        while (__hip_atomic_load(&counter, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < count) __builtin_amdgcn_s_sleep(1);
    };
    // (Lane 0's release is for what all lanes of the wave wrote: it waits until the wave's LDS operations are done, which are
    // counted for the wave and complete in order.)
    auto const add_one = [&](int& counter) { if (lane == 0) __hip_atomic_fetch_add(&counter, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP); };
    // Mode 7's partition comes with the two subsets where every alpha is 1, whose terms are zeros.  Opaque blocks of float
    // images can hold alphas above 1 and NaNs: their groups bound it over four channels, as blocks with alpha.
    auto const all_ones = [&](int b) { return __ballot(shared.alphas[b] & kNotOne) == 0; };

    // what a search is about, the lanes' blocks, and the search whose tasks give its bounds
    auto const kind_of = [&](int search) { return search < opaqueGroups ? int(kPickTwo) : search < 2 * opaqueGroups ? int(kPickThree) : int(kPickTwoAlpha); };
    auto const group_of = [&](int search) { return search < opaqueGroups ? search : search < 2 * opaqueGroups ? search - opaqueGroups : search - 2 * opaqueGroups; };
    auto const what_of = [&](int search, int b) { return kind_of(search) != kPickTwoAlpha ? kind_of(search) : group_of(search) < opaqueGroups && all_ones(b) ? int(kCorners3) : int(kCorners4); };
    auto const bounds_of = [&](int search) { return kind_of(search) == kPickTwoAlpha && group_of(search) < opaqueGroups ? group_of(search) : search; };

    // ---- 1. bounds of the partitions' errors; one rotation of modes 4 and 5 for each block; the errors of the first partitions
    __builtin_amdgcn_s_setprio(3);
    int const searches = 2 * opaqueGroups + groups, boundTasks = (2 * opaqueGroups + alphaGroups) * CHUNKS;
    auto const rotate_first = [&](int group) {
        int const b = block_of_group(group);
        bound_rotations<S>(lds, b);
        int const first = first_rotation<S>(lds, b);
        Best const best = all_ones(b) ? dual_planes<S, 2>(lds, b, first) : dual_planes<S, 3>(lds, b, first);
        keep_candidates<S>(lds, b, first, best.error, own_lane(group));
        put_candidate(&lds->early.words[b], &lds->early.errors[b], best.error, best.lo, best.hi);
        add_one(shared.rotated);
    };
    // Whether rotations and mode 6 are left out by their bounds for blocks with alpha, too.  A workgroup with a compute unit to
    // itself takes as long as its chains; few blocks with alpha have more to do than mode 7's search, and one rotation after
    // the other was the longer chain (256 x 256 of alpha, smooth 47.0 us with all at once behind the bounds, 61.3 by bounds, 43.0
    // with all at once beside them, behind the selections in the list and in priority; flat 44.5, 54.6, 36.7; with an opaque
    // background 83.5, 86.0, 81.3).  But where it has opaque blocks near lines, too, all of whose partitions it estimates, it is
    // the work that counts: grey 95, 92.6, and 98.  (Opaque blocks, bounds / all at once: flat 65 / 61, detail 74 / 76, grey 75 / 77.)
    auto const all_by_bounds = [&] {
        if (!ALONE) return true;
        if (opaqueGroups == 0) return false;
        int const b = block_of(0, 0);
        wait_for(shared.bounded[0], CHUNKS);
        return __any(lds->scale[kPickTwo][b] != 0.f) && !__any(lds->lowest[kPickTwo][b] != ~0u);
    };
    int const early = ALONE ? opaqueGroups : groups, late = ALONE ? 5 * alphaGroups : 0;       // tasks before the selections and after them
    for (int taken = next_task(0); taken < boundTasks + early + searches + late; taken = next_task(0)) {
        int const task = taken < boundTasks ? taken : taken < boundTasks + early ? taken - boundTasks - early : taken - early;
        if (ALONE && task >= boundTasks + searches) {
            int const nth = task - boundTasks - searches, rotation = nth / alphaGroups, group = nth % alphaGroups, b = block_of(1, group);
            if (all_by_bounds()) {
                if (rotation == 0) rotate_first(opaqueGroups + group);
                continue;
            }
            __builtin_amdgcn_s_setprio(0);
            if (rotation == 4) { finish_task<S, Mode6, 4, true>(lds, b, 0, kSlotSix); continue; }
            Best const best = dual_planes<S, 3>(lds, b, rotation);
            if (rotation == 0) {
                lds->plans[b] = 7u * (kKeepRotation << 1) | kKeepSix;
                put_candidate(&lds->early.words[b], &lds->early.errors[b], best.error, best.lo, best.hi);
            } else {
                int const slot = kSlotRotations + rotation - 1;
                put_candidate(&lds->scratch.late.words[slot][b], &lds->scratch.late.errors[slot][b], best.error, best.lo, best.hi);
            }
        } else if (task < 0) {
            rotate_first(task + early);
        } else if (task < boundTasks) {
            int const first = (task % CHUNKS) * CHUNK, nth = task / CHUNKS, search = nth < 2 * opaqueGroups ? nth : nth + opaqueGroups;
            int const b = block_of_group(group_of(search));
            if (kind_of(search) == kPickThree) {
                bound_task<S, 3, 3, true, false>(lds, b, first, first + CHUNK);
            } else if (kind_of(search) == kPickTwo && all_ones(b)) {
                bound_task<S, 2, 3, true, true>(lds, b, first, first + CHUNK);
            } else {
                if (kind_of(search) == kPickTwo) bound_task<S, 2, 3, true, false>(lds, b, first, first + CHUNK);
                bound_task<S, 2, 4, false, true>(lds, b, first, first + CHUNK);
            }
            add_one(shared.bounded[search]);
        } else {
            int const search = task - boundTasks, group = group_of(search);
            int const b = block_of_group(group);
            wait_for(shared.bounded[bounds_of(search)], CHUNKS);
            select_task<S>(lds, b, what_of(search, b), search, own_lane(group));
            add_one(shared.selected);
        }
    }
    __builtin_amdgcn_s_setprio(1);
    wait_for(shared.selected, searches);
    bool const byBounds = all_by_bounds();

    // ---- 2. the errors of the partitions that are left, then candidates: first those that need no partition
    int const wholeTasks = __builtin_amdgcn_readfirstlane(shared.wholes) * (64 / kWholeChunk);
    int estimates = wholeTasks;
    for (int search = 0; search < searches; ++search) estimates += (__builtin_amdgcn_readfirstlane(shared.queued[search]) + 63) / 64;
    for (int task = next_task(1);; task = next_task(1)) {
        if (task < wholeTasks) {
            int const search = __builtin_amdgcn_readfirstlane(int(shared.whole[task / (64 / kWholeChunk)])), first = task % (64 / kWholeChunk) * kWholeChunk;
            int const b = block_of_group(group_of(search)), what = what_of(search, b);
            if (what == kThree)         pick_task<S, 3, 3, true, false>(lds, b, first, first + kWholeChunk);
            else if (what == kTwo)      pick_task<S, 2, 3, true, false>(lds, b, first, first + kWholeChunk);
            else if (what == kCorners3) pick_task<S, 2, 3, false, true>(lds, b, first, first + kWholeChunk);
            else                        pick_task<S, 2, 4, false, true>(lds, b, first, first + kWholeChunk);
            add_one(shared.estimated);
            continue;
        }
        if (task < estimates) {
            int search = 0, piece = task - wholeTasks, count = 0;
            for (;; ++search) {                              // (ends: the task is a piece of one of the queues)
                count = __builtin_amdgcn_readfirstlane(shared.queued[search]);
                if (piece < (count + 63) / 64) break;
                piece -= (count + 63) / 64;
            }
            int const what = what_of(search, block_of_group(group_of(search)));
            if (piece * 64 + lane < count) {
                int const item = shared.queues[search][piece * 64 + lane];
                estimate_one<S>(lds, what, item & 127, item >> 7);
            }
            add_one(shared.estimated);
            continue;
        }
        __builtin_amdgcn_s_setprio(0);
        wait_for(shared.rotated, byBounds ? groups : opaqueGroups);
        int const keptFlat = __builtin_amdgcn_readfirstlane(shared.kept[0]), keptRotations = __builtin_amdgcn_readfirstlane(shared.kept[1]);
        int const keptSixes = __builtin_amdgcn_readfirstlane(shared.kept[2]);
        int const flatTasks = (keptFlat + 63) / 64, rotationTasks = flatTasks + (keptRotations + 63) / 64, sixTasks = (keptSixes + 63) / 64, candidate = task - estimates;
        if (candidate >= rotationTasks + sixTasks + 4 * opaqueGroups + groups) break;        // uniform: every wave gets here
        if (candidate < rotationTasks) {
            bool const flat = candidate < flatTasks;
            int const item = flat ? shared.flatRotations[min(candidate * 64 + lane, keptFlat - 1)] : shared.rotations[min((candidate - flatTasks) * 64 + lane, keptRotations - 1)];
            int const b = item & 127, rotation = item >> 7;
            Best const best = flat ? dual_planes<S, 2>(lds, b, rotation) : dual_planes<S, 3>(lds, b, rotation);
            int const slot = kSlotRotations + rotation - (rotation > int(shared.plans[b] & 3u) ? 1 : 0);
            put_candidate(&lds->scratch.late.words[slot][b], &lds->scratch.late.errors[slot][b], best.error, best.lo, best.hi);
            continue;
        }
        if (candidate < rotationTasks + sixTasks) {
            finish_task<S, Mode6, 4, true>(lds, shared.sixes[min((candidate - rotationTasks) * 64 + lane, keptSixes - 1)], 0, kSlotSix);
            continue;
        }
        wait_for(shared.estimated, estimates);
        int const picked = candidate - rotationTasks - sixTasks;
        if (picked < 4 * opaqueGroups) {
            int const which = picked & 3, b = block_of(0, picked >> 2);
            if (which == 0)      finish_task<S, Mode0, 3, true>(lds, b, kPickThree, 0);
            else if (which == 1) finish_task<S, Mode2, 3, true>(lds, b, kPickThree, 1);
            else if (which == 2) finish_task<S, Mode1, 3, true>(lds, b, kPickTwo, 2);
            else                 finish_task<S, Mode3, 3, true>(lds, b, kPickTwo, 3);
        } else {
            finish_task<S, Mode7, 4, false>(lds, block_of_group(picked - 4 * opaqueGroups), kPickTwoAlpha, kSlotSeven);
        }
    }
    __syncthreads();

    // ---- 3. the best candidate
    if (tid < BLOCKS) {
        int const b = tid, bx = block_x(b), by = block_y(b);
        if (bx < a.widthInBlocks && by < a.heightInBlocks) {
            float bestError = FLT_MAX;
            uint4 best = make_uint4(0u, 0u, 0u, 0u);
            uint32_t const plan = shared.plans[b];
            auto const consider = [&](float error, uint4 const& words) { if (!(error > bestError)) { bestError = error; best = words; } };
            auto const consider_late = [&](int slot) { consider(shared.scratch.late.errors[slot][b], shared.scratch.late.words[slot][b]); };
            if (!(shared.alphas[b] & kBelowOne))
                for (int slot = 0; slot < kSlotRotations; ++slot) consider_late(slot);
            for (int r = 0; r < 4; ++r) {
                if (r == int(plan & 3u))             consider(shared.early.errors[b], shared.early.words[b]);
                else if (plan & (kKeepRotation << r)) consider_late(kSlotRotations + r - (r > int(plan & 3u) ? 1 : 0));
            }
            if (plan & kKeepSix) consider_late(kSlotSix);
            consider_late(kSlotSeven);
            store_block(a, bx, by, uint64_t(best.x) | uint64_t(best.y) << 32, uint64_t(best.z) | uint64_t(best.w) << 32);
        }
    }
}

// With a mode buffer.  A workgroup covers SIDE x SIDE blocks; it first reads their entries and sorts the blocks by mode
// into lists in LDS (the reference's ReorderThreadsByMode, CompressBC7.hlsl:1445-1509), then its waves take pieces of 64
// blocks of one list each, the longest modes first, so that a wave runs one mode only (modes 4 and 5 are one piece of
// code).  Sorting 256 blocks among as many threads left each wave with three or four modes: 2048 x 2048 blocks, modes 4 and
// 5 on five blocks of six, took 86 us, with every block in one mode 27 to 50; 50 us from lists of 1024 blocks, with a wave's
// pixels loaded one after the other for a third of the time; 38.5 with all of them under way and the map's words loaded and
// counted at once; 34.0 with indices packed two and three bits at a time as they are made.  Images of no more than 256 blocks
// per compute unit sort 256 (1024 x 1024: 71 us before, 31, 23.5, and 21.3; 128 x 128 22.3 -> 20.4 by the packing).
// What is left is 19 pieces for 12 waves, unequal ones.  Which lane encodes which block depends on the order the LDS counters
// are hit in; what is written for a block does not.
// Three waves per SIMD (168 registers) serve this kernel best.
template <int SIDE, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, 3)
bc7_compress_modes_kernel(BlockCompressArgs a)
{
    constexpr int BLOCKS = SIDE * SIDE, THREADS = 64 * WAVES, LISTS = 7;
    // lists in this order: modes 0, 2, 1, 3, 7, 4 and 5, 6
    __shared__ uint32_t tasks[LISTS][BLOCKS];                // mode << 16 | partition << 10 | block
    __shared__ int counts[LISTS], next;
    static_assert(BLOCKS <= 1024, "ten bits number a block");
    int const tid = threadIdx.x, lane = tid & 63;
    if (tid < LISTS) counts[tid] = 0;
    if (tid == LISTS) next = 0;
    __syncthreads();
    // 9 bits per block of the mode map, which lie in one word or two; all loads before the first entry is looked at
    constexpr int TURNS = (BLOCKS + THREADS - 1) / THREADS;
    uint32_t words[TURNS][2];
    uint32_t shifts[TURNS];
    bool mapped[TURNS];
    int64_t const lastWord = ((int64_t(a.modeMapWidthInBlocks) * a.modeMapHeightInBlocks * 9 + 31) >> 5) - 1;
#pragma unroll
    for (int turn = 0; turn < TURNS; ++turn) {
        int const b = tid + turn * THREADS;
        int64_t const mx = int64_t(blockIdx.x) * SIDE + b % SIDE + a.modeMapOffsetX, my = int64_t(blockIdx.y) * SIDE + b / SIDE + a.modeMapOffsetY;
        mapped[turn] = mx >= 0 && my >= 0 && mx < a.modeMapWidthInBlocks && my < a.modeMapHeightInBlocks;
        int64_t const bit = mapped[turn] ? (my * a.modeMapWidthInBlocks + mx) * 9 : 0;
        words[turn][0] = a.modeBuffer[bit >> 5];
        words[turn][1] = a.modeBuffer[min((bit >> 5) + 1, lastWord)];
        shifts[turn] = uint32_t(bit & 31);
    }
#pragma unroll
    for (int turn = 0; turn < TURNS; ++turn) {
        int const b = tid + turn * THREADS, bx = int(blockIdx.x) * SIDE + b % SIDE, by = int(blockIdx.y) * SIDE + b / SIDE;
        int list = -1;
        uint32_t entry = 0;
        if (b < BLOCKS && bx < a.widthInBlocks && by < a.heightInBlocks) {
            // 0 = no entry, 0x1BF stands for mode 0 partition 0
            if (mapped[turn]) entry = uint32_t((uint64_t(words[turn][1]) << 32 | words[turn][0]) >> shifts[turn]) & 0x1FFu;
            if (entry == 0u) {
                store_block(a, bx, by, 0x0001f00000f80004ull, 0x1f9e00003ff0001full);     // the reference's marker: black, red, green and blue squares
            } else {
                if (entry == 0x1BFu) entry = 0u;
                list = int((0x46553120u >> (4u * (entry >> 6))) & 15u);
            }
        }
        // one atomic per wave, a lane for each list
        uint64_t ofList[LISTS];
        int count = 0, at = 0;
#pragma unroll
        for (int l = 0; l < LISTS; ++l) {
            ofList[l] = __ballot(list == l);
            if (lane == l) count = int(__popcll(ofList[l]));
        }
        if (lane < LISTS && count) at = atomicAdd(&counts[lane], count);
#pragma unroll
        for (int l = 0; l < LISTS; ++l) {
            int const start = __builtin_amdgcn_readlane(at, l);
            if (list == l) tasks[l][start + int(__builtin_amdgcn_mbcnt_hi(uint32_t(ofList[l] >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(ofList[l]), 0u)))] = entry << 10 | uint32_t(b);
        }
    }
    __syncthreads();
    for (;;) {
        int piece = 0;
        if (lane == 0) piece = atomicAdd(&next, 1);
        piece = __builtin_amdgcn_readfirstlane(piece);
        int list = 0;
        for (; list < LISTS; ++list) {
            int const pieces = (__builtin_amdgcn_readfirstlane(counts[list]) + 63) / 64;
            if (piece < pieces) break;
            piece -= pieces;
        }
        if (list == LISTS) break;                            // uniform: every wave gets here after the last piece
        if (piece * 64 + lane >= counts[list]) continue;
        uint32_t const task = tasks[list][piece * 64 + lane];
        int const b = int(task & 1023u), bx = int(blockIdx.x) * SIDE + b % SIDE, by = int(blockIdx.y) * SIDE + b / SIDE;
        Color<4> px[16];
        load_block(a, bx, by, px);
        Block const block = bc7_encode_fixed(px, list, int(task >> 16), int(task >> 10) & 63);
        store_block(a, bx, by, block.lo, block.hi);
    }
}

hipError_t launch_bc7_compress(BlockCompressArgs const& a, hipStream_t stream)
{
    if (a.modeBuffer) {
        int const small = ((a.widthInBlocks + 15) / 16) * ((a.heightInBlocks + 15) / 16);
        if (small <= compute_units_of_current_device())
            hipLaunchKernelGGL((bc7_compress_modes_kernel<16, 8>), dim3((a.widthInBlocks + 15) / 16, (a.heightInBlocks + 15) / 16), dim3(512), 0, stream, a);
        else
            hipLaunchKernelGGL((bc7_compress_modes_kernel<32, 12>), dim3((a.widthInBlocks + 31) / 32, (a.heightInBlocks + 31) / 32), dim3(768), 0, stream, a);
    } else {
        // One group of 64 blocks per workgroup while there are no more groups than compute units (sixteen waves then
        // have a unit to themselves), else two and half the waves, two workgroups to a unit: the groups' blocks with
        // and without alpha fill their tasks' lanes better, and one workgroup works while the other waits for its
        // last task.  (With every partition estimated: 512 x 512 111 us, 174 with two groups; 1024 x 1024 290, 427 with one.)
        int const groupsX = (a.widthInBlocks + 7) / 8, groupsY = (a.heightInBlocks + 7) / 8;
        if (int64_t(groupsX) * groupsY <= compute_units_of_current_device())
            hipLaunchKernelGGL((bc7_compress_kernel<1, 16>), dim3(groupsX, groupsY), dim3(1024), 0, stream, a);
        else
            hipLaunchKernelGGL((bc7_compress_kernel<2, 8>), dim3((groupsX + 1) / 2, groupsY), dim3(512), 0, stream, a);
    }
    return hipGetLastError();
}

} // namespace ntc_hip_dev
