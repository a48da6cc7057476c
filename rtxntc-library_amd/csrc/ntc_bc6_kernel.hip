// ntc_bc6_kernel.hip - BC6H (unsigned half float) block compression of a decoded image (gfx950).
//
// The reference's BC6 pass (IContext::MakeBlockCompressionComputePass with BlockCompressedFormat::BC6,
// src/shaders/CompressBC6.hlsl) as a compute kernel.  Two candidates, the
// smaller luminance-weighted mean squared log2 error wins:
//   * one subset, 10-bit endpoints, 4-bit indices (mode 11 of the format): bounding box, pulled inwards in
//     log2 space by at most 1/32 of its extent, one least-squares refit in half-code space;
//   * two subsets with 3-bit indices on the partition (of the format's first 32) whose texels lie closest
//     to the diagonals of the subsets' bounding boxes; endpoints stored as 7-bit base + 6-bit deltas (mode
//     2) or 9-bit base + 5-bit deltas (mode 6), whichever decodes closer.
// Where the shader uses the hardware's log2 / exp2 / rcp / rsqrt, this kernel uses the functions below,
// built from plain binary32 operations (and correctly rounded division and square root), so that the CPU
// checker can reproduce every bit.  Half conversion rounds to nearest even.  Texels are clamped to
// [0, 65504] (a NaN becomes 0).  All float arithmetic is unfused, in the order written here.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "ntc_decode_kernel.h"
#include "ntc_bc_source.h"

namespace ntc_hip_dev {

namespace {

#define BC6_INLINE __device__ __forceinline__

// The format's first 32 two-subset partitions (Table.P2 of the BPTC specification): bit t = subset of
// texel t; and the anchor texel of the second subset (table A2).
__constant__ uint16_t kSecondSubset[32] = {
    0xcccc, 0x8888, 0xeeee, 0xecc8, 0xc880, 0xfeec, 0xfec8, 0xec80, 0xc800, 0xffec, 0xfe80, 0xe800, 0xffe8, 0xff00, 0xfff0, 0xf000,
    0xf710, 0x008e, 0x7100, 0x08ce, 0x008c, 0x7310, 0x3100, 0x8cce, 0x088c, 0x3110, 0x6666, 0x366c, 0x17e8, 0x0ff0, 0x718e, 0x399c,
};
__constant__ uint8_t kSecondAnchor[32] = { 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 2, 8, 2, 2, 8, 8, 15, 2, 8, 2, 2, 8, 8, 2, 2 };

// a / b in fewer instructions than the compiler's division, which scales its operands against overflow and always
// refines the hardware's reciprocal and the quotient as far as the worst operands need.  REFINED: how often the
// reciprocal is; then the quotient is corrected once by its remainder, which leaves it within 2^-44 of itself before the
// last rounding.  Where it is used the result is the correctly rounded one.  <0>: integers below 2^17, whose quotients
// are no nearer than 2^-42 to the middle between two numbers; (m - 1) / (m + 1), m in [0.70, 1.42], compared with the
// division for every m.  <1>: (y + 1) / (x + 1) with y a half and x a half, a UNORM code over its maximum or an integer
// up to 65504, compared for every pair.  quotient_by() is the compiler's own sequence without the scaling, which none of
// the operands needs where texels are no FLOAT32.
BC6_INLINE float corrected(float a, float b, float r)
{
    float const q = a * r;
    return __builtin_fmaf(__builtin_fmaf(-q, b, a), r, q);
}
template <int REFINED> BC6_INLINE float reciprocal(float b)
{
    float r = __builtin_amdgcn_rcpf(b);
    if constexpr (REFINED == 1) r = __builtin_fmaf(__builtin_fmaf(-b, r, 1.f), r, r);
    return r;
}
template <int REFINED> BC6_INLINE float quotient(float a, float b) { return corrected(a, b, reciprocal<REFINED>(b)); }
BC6_INLINE float quotient_by(float a, float b, float r)      // r = reciprocal<1>(b)
{
    float const q = corrected(a, b, r);
    return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-q, b, a), r, q), b, a);
}

// log2 for x >= 0 (0 -> -inf); NaN for a negative or NaN argument.  Argument reduction to [sqrt(1/2), sqrt 2),
// then the series of atanh; a few units in the last place.
// (normal_log2: of a normal number's bits, the exponent raised by `e`.)
BC6_INLINE float normal_log2(uint32_t bits, int e)
{
    int const above = int(bits - 0x3f3504f4u);               // of the number that follows 1.41421354 / 2
    e += above >> 23;
    float const m = __uint_as_float(bits - (uint32_t(above) & 0xff800000u));
    float const t = quotient<0>(m - 1.f, m + 1.f), t2 = t * t;
    float p = t2 * (1.f / 9.f) + (1.f / 7.f);
    p = p * t2 + 0.2f;
    p = p * t2 + (1.f / 3.f);
    p = p * t2 + 1.f;
    return float(e) + p * t * 2.88539004f;
}
BC6_INLINE float det_log2(float x)
{
    if (!(x >= 0.f)) return __uint_as_float(0x7fc00000u);
    if (x == 0.f) return __uint_as_float(0xff800000u);
    uint32_t b = __float_as_uint(x);
    if (b >= 0x7f800000u) return x;
    int e = 0;
    if (b < 0x00800000u) { x *= 8388608.f; b = __float_as_uint(x); e = -23; }
    return normal_log2(b, e);
}

// 2^x for the x that occur here: logarithms of numbers between 1 and 65505.
BC6_INLINE float exp2_of_log(float x)
{
    float const n = rintf(x), g = (x - n) * 0.693147182f;
    float p = g * (1.f / 5040.f) + (1.f / 720.f);
    p = p * g + (1.f / 120.f);
    p = p * g + (1.f / 24.f);
    p = p * g + (1.f / 6.f);
    p = p * g + 0.5f;
    p = p * g + 1.f;
    p = p * g + 1.f;
    return p * __uint_as_float(uint32_t(int(n) + 127) << 23);
}

struct V3 { float x, y, z; };
BC6_INLINE V3 operator+(V3 a, V3 b) { return { a.x + b.x, a.y + b.y, a.z + b.z }; }
BC6_INLINE V3 operator-(V3 a, V3 b) { return { a.x - b.x, a.y - b.y, a.z - b.z }; }
BC6_INLINE V3 operator*(V3 a, float s) { return { a.x * s, a.y * s, a.z * s }; }
BC6_INLINE V3 operator*(V3 a, V3 b) { return { a.x * b.x, a.y * b.y, a.z * b.z }; }
BC6_INLINE float dot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
BC6_INLINE V3 vmin(V3 a, V3 b) { return { min_f32(a.x, b.x), min_f32(a.y, b.y), min_f32(a.z, b.z) }; }
BC6_INLINE V3 vmax(V3 a, V3 b) { return { max_f32(a.x, b.x), max_f32(a.y, b.y), max_f32(a.z, b.z) }; }
BC6_INLINE float clampf(float v, float lo, float hi) { return fminf(fmaxf(v, lo), hi); }
// A float as the number of its half-precision bit pattern, and back (the latter truncates to an integer first).
// (a NaN always gives the code 0x7e00, whatever its sign and payload)
BC6_INLINE float number_to_half_bits(float v) { return float(__builtin_bit_cast(uint16_t, _Float16(v))); }
BC6_INLINE float to_half_bits(float v) { return v != v ? 32256.f : number_to_half_bits(v); }
BC6_INLINE float from_half_bits(float v) { return float(__builtin_bit_cast(_Float16, uint16_t(uint32_t(v)))); }
BC6_INLINE V3 to_half_bits(V3 v) { return { to_half_bits(v.x), to_half_bits(v.y), to_half_bits(v.z) }; }

constexpr float kHalfMax = 65504.f;
constexpr float kHalfMaxCode = 31743.f;         // 0x7bff, the code of 65504

// One texel against what a decoder shows: WIDE texels come from a FLOAT32 image and can be any number up to 65504,
// others are halves, UNORM quotients or integers.
template <bool WIDE> struct Msle {
    V3 a, r;                                                 // the texel plus 1, its reciprocals
    BC6_INLINE explicit Msle(V3 texel) : a(texel + V3{ 1.f, 1.f, 1.f })
    {
        if constexpr (!WIDE) r = V3{ reciprocal<1>(a.x), reciprocal<1>(a.y), reciprocal<1>(a.z) };
    }
    BC6_INLINE float operator()(V3 b) const
    {
        V3 d;
        uint32_t const largest = max(max(__float_as_uint(b.x), __float_as_uint(b.y)), __float_as_uint(b.z));
        if (WIDE || largest >= 0x7f800000u) {                // (endpoints near the top decode to infinity or NaN)
            d = V3{ det_log2((b.x + 1.f) / a.x), det_log2((b.y + 1.f) / a.y), det_log2((b.z + 1.f) / a.z) };
        } else {
            d = V3{ normal_log2(__float_as_uint(corrected(b.x + 1.f, a.x, r.x)), 0), normal_log2(__float_as_uint(corrected(b.y + 1.f, a.y, r.y)), 0),
                    normal_log2(__float_as_uint(corrected(b.z + 1.f, a.z, r.z)), 0) };
        }
        V3 const sq = d * d * V3{ 0.299f, 0.587f, 0.114f };
        return sq.x + sq.y + sq.z;
    }
    // With the hardware's logarithm: within 2^-19 of its value, 0 where that is 0, infinite or no number where that is not
    // a number of normal size.
    BC6_INLINE float estimate(V3 b) const
    {
        V3 const n = b + V3{ 1.f, 1.f, 1.f };
        V3 q;
        if constexpr (WIDE) q = V3{ n.x / a.x, n.y / a.y, n.z / a.z };
        else                q = V3{ corrected(n.x, a.x, r.x), corrected(n.y, a.y, r.y), corrected(n.z, a.z, r.z) };
        V3 const d{ __builtin_amdgcn_logf(q.x), __builtin_amdgcn_logf(q.y), __builtin_amdgcn_logf(q.z) };
        V3 const sq = d * d;
        return __builtin_fmaf(sq.z, 0.114f, __builtin_fmaf(sq.y, 0.587f, sq.x * 0.299f));
    }
};

// (the quotients by constants here and below are those of integers, times a power of two)
BC6_INLINE V3 quantize(V3 v, float levels)
{
    V3 const h = to_half_bits(v);
    return { corrected(h.x * levels, 31744.f, 1.f / 31744.f), corrected(h.y * levels, 31744.f, 1.f / 31744.f), corrected(h.z * levels, 31744.f, 1.f / 31744.f) };
}
BC6_INLINE V3 unquantize(V3 v, float levels)
{
    return { (v.x * 65536.f + 32768.f) / levels, (v.y * 65536.f + 32768.f) / levels, (v.z * 65536.f + 32768.f) / levels };
}
BC6_INLINE V3 interpolate(V3 e0, V3 e1, float weight)
{
    V3 const c = (e0 * (64.f - weight) + e1 * weight + V3{ 32.f, 32.f, 32.f }) * (31.f / 4096.f);
    return { from_half_bits(c.x), from_half_bits(c.y), from_half_bits(c.z) };
}
// The same of the two-subset endpoints, integers whose products are exact.
BC6_INLINE V3 interpolate_integers(V3 e0, V3 e1, float weight)
{
    float const w0 = 64.f - weight;
    V3 const c = V3{ __builtin_fmaf(e0.x, w0, __builtin_fmaf(e1.x, weight, 32.f)), __builtin_fmaf(e0.y, w0, __builtin_fmaf(e1.y, weight, 32.f)),
                     __builtin_fmaf(e0.z, w0, __builtin_fmaf(e1.z, weight, 32.f)) } * (31.f / 4096.f);
    return { from_half_bits(c.x), from_half_bits(c.y), from_half_bits(c.z) };
}
BC6_INLINE uint32_t index_of(float pos, float e0, float e1, float scale, float bias, float top)
{
    float const a = pos - e0, b = e1 - e0;                   // half codes: integers
    float const r = __builtin_amdgcn_div_fixupf(quotient<0>(a, b), b, a);
    return uint32_t(clampf(r * scale + bias + 0.5f, 0.f, top));      // a NaN (coinciding ends) gives 0
}
BC6_INLINE uint32_t index3(float pos, float e0, float e1) { return index_of(pos, e0, e1, 6.98182f, 0.00909f, 7.f); }
BC6_INLINE uint32_t index4(float pos, float e0, float e1) { return index_of(pos, e0, e1, 14.93333f, 0.03333f, 15.f); }
// The format's weights of those indices, floor(64 index / 7 + 1/2) and floor(64 index / 15 + 1/2).
constexpr uint32_t weight3(uint32_t index) { return 9u * index + (index >> 2); }
constexpr uint32_t weight4(uint32_t index) { return (273u * index + 32u) >> 6; }
constexpr bool weights_agree()
{
    for (uint32_t i = 0; i < 16; ++i)
        if ((i < 8 && weight3(i) != (128u * i + 7u) / 14u) || weight4(i) != (128u * i + 15u) / 30u) return false;
    return true;
}
static_assert(weights_agree());
template <bool WIDE> BC6_INLINE V3 divided(V3 v, float s)
{
    if constexpr (WIDE) return { v.x / s, v.y / s, v.z / s };
    float const r = reciprocal<1>(s);
    return { quotient_by(v.x, s, r), quotient_by(v.y, s, r), quotient_by(v.z, s, r) };
}
template <bool WIDE> BC6_INLINE V3 direction(V3 lo, V3 hi) { V3 const d = hi - lo; return divided<WIDE>(d, d.x + d.y + d.z); }

BC6_INLINE float log1(float c) { return normal_log2(__float_as_uint(c + 1.f), 0); }
BC6_INLINE float exp1(float c) { return exp2_of_log(c) - 1.f; }

// ---- the workgroup ------------------------------------------------------------------------------------
//
// Four waves encode 64 blocks, whose texels lie in LDS; the lanes of a wave are blocks.
//   1. one wave: the one-subset endpoints; then all: bounds of the patterns' scores, patterns taken in turn, and the
//      scores of those that the bounds leave;
//   2. a wave per subset of each block's pattern: its endpoints; beside them the other two waves, eight texels each: the
//      one-subset candidate's indices and the estimate of its error;
//   3. each wave four of the sixteen texels: the same for the two-subset candidates, and the errors as they are defined
//      where the estimates are too close to tell;
//   4. one wave: the block.
// Bound by the issue of vector instructions and by waves that wait for the one that works alone: 68 % of the slots with four
// workgroups on a compute unit.  31.5 KB of LDS (what one part leaves, the next one overwrites) and 96 registers let five be
// there: 141 us at 2048 x 2048 with four, 133 with five, 137 with six, which takes texels in three planes and registers kept
// in scratch.  Each part is a function with registers of its own, so that nothing is spilled in a loop; the search is one
// call because a call saves registers to scratch (a call per two patterns: 257 us at 2048 x 2048 instead of 204).  One lane
// per block, all parts in one body with 168 registers, took 121 us at 64 x 64, 151 at 1024 x 1024 and 287 at 2048 x 2048:
// small images waited for the chain of one lane's scores, large ones for its spills and longer divisions.  Shared by the
// waves: 30, 61 and 204 (195 beside other kernels), of which the 32 scores, 625 instructions each, were more than half;
// with their bounds first 165 beside others, 29, 47 and 147 alone; with estimated errors (the logarithms were 13 % of the
// instructions) and five workgroups 26.6, 42 and 124, 4096 x 4096 520 -> 417; with the one-subset errors beside the subsets'
// endpoints 25.7, 41 and 123.  (Bounds from offsets to the block's corner, with the smaller subset's sums only: 8 % fewer
// instructions and no time, because what goes issues two at a time and the minima and maxima that stay do not.)
struct Bc6Lds {
    float4 texels[16][64];
    float one[11][64];                                       // one subset: lo, hi, direction, codes of the ends along it
    union {
        float least[32][64];                                 // until the pattern is picked: lower bounds of the scores
        struct {
            float two[2][11][64];                            // each of two subsets
            float errors[3][4][64];                          // of four texels, estimated: one subset, 7 + 6 bits, 9 + 5 bits
        };
    };
    uint32_t indices[2][4][64];                              // of four texels: 4 bits each, 3 bits each
    int next;
    uint64_t pick[64];                                       // score bits << 32 | pattern
    uint32_t bound[64], candidates[64], unbounded[64];       // smallest upper bound of a score; patterns that it leaves; some have no bounds
                                                             // (at the end: choices by the errors as they are defined; the blocks that need them)
    uint32_t unscored[64];                                   // pattern 0's score is a NaN: the search stays there
};
using Bc6Ptr = __attribute__((address_space(3))) Bc6Lds*;
#define BC6_TASK __device__ __attribute__((noinline))        // (separate register allocation; uniform arguments are made so again)

BC6_INLINE V3 texel(Bc6Ptr lds, int b, int t) { return { lds->texels[t][b].x, lds->texels[t][b].y, lds->texels[t][b].z }; }
struct SubsetEnds { V3 lo, hi, dir; float e0, e1; };
template <class P> BC6_INLINE void store_ends(P to, int b, SubsetEnds const& s)
{
    to[0][b] = s.lo.x; to[1][b] = s.lo.y; to[2][b] = s.lo.z; to[3][b] = s.hi.x; to[4][b] = s.hi.y; to[5][b] = s.hi.z;
    to[6][b] = s.dir.x; to[7][b] = s.dir.y; to[8][b] = s.dir.z; to[9][b] = s.e0; to[10][b] = s.e1;
}
template <class P> BC6_INLINE SubsetEnds load_ends(P from, int b)
{
    return { { from[0][b], from[1][b], from[2][b] }, { from[3][b], from[4][b], from[5][b] }, { from[6][b], from[7][b], from[8][b] }, from[9][b], from[10][b] };
}

// Pulls the box inwards in log2(1 + x) space: towards the smallest / largest values that are not the
// extremes themselves, by at most 1/32 of the extent.
BC6_INLINE void inset_box(Bc6Ptr lds, int b, V3& lo, V3& hi)
{
    V3 innerLo = hi, innerHi = lo;
#pragma unroll 4
    for (int t = 0; t < 16; ++t) {
        V3 const p = texel(lds, b, t);
        innerLo = vmin(innerLo, V3{ p.x == lo.x ? innerLo.x : p.x, p.y == lo.y ? innerLo.y : p.y, p.z == lo.z ? innerLo.z : p.z });
        innerHi = vmax(innerHi, V3{ p.x == hi.x ? innerHi.x : p.x, p.y == hi.y ? innerHi.y : p.y, p.z == hi.z ? innerHi.z : p.z });
    }
    V3 const logInnerHi{ log1(innerHi.x), log1(innerHi.y), log1(innerHi.z) }, logInnerLo{ log1(innerLo.x), log1(innerLo.y), log1(innerLo.z) };
    V3 logHi{ log1(hi.x), log1(hi.y), log1(hi.z) }, logLo{ log1(lo.x), log1(lo.y), log1(lo.z) };
    V3 const ext = (logHi - logLo) * (1.f / 32.f);
    logLo = logLo + vmin(logInnerLo - logLo, ext);
    logHi = logHi - vmin(logHi - logInnerHi, ext);
    lo = V3{ exp1(logLo.x), exp1(logLo.y), exp1(logLo.z) };
    hi = V3{ exp1(logHi.x), exp1(logHi.y), exp1(logHi.z) };
}

// Least-squares endpoints, in half-code space, for the indices the current endpoints give to the texels
// of `members` (bit t = texel t takes part).  False when the system is singular.
template <bool WIDE, bool FOUR_BIT>
BC6_INLINE bool refit(Bc6Ptr lds, int b, uint32_t members, V3 lo, V3 hi, V3& outLo, V3& outHi)
{
    V3 const dir = direction<WIDE>(lo, hi);
    float const e0 = to_half_bits(dot(lo, dir)), e1 = to_half_bits(dot(hi, dir));
    V3 alphaSum{ 0.f, 0.f, 0.f }, betaSum{ 0.f, 0.f, 0.f };
    float ab = 0.f, aa = 0.f, bb = 0.f;
    for (uint32_t m = members; m; m &= m - 1) {
        V3 const p = texel(lds, b, __ffs(int(m)) - 1);
        float const pos = to_half_bits(dot(p, dir));
        uint32_t const index = FOUR_BIT ? index4(pos, e0, e1) : index3(pos, e0, e1);
        constexpr float top = FOUR_BIT ? 15.f : 7.f;
        float const beta = clampf(corrected(float(index), top, 1.f / top), 0.f, 1.f), alpha = 1.f - beta;
        V3 const h{ number_to_half_bits(p.x), number_to_half_bits(p.y), number_to_half_bits(p.z) };
        alphaSum = alphaSum + h * alpha; betaSum = betaSum + h * beta;
        ab += alpha * beta; aa += alpha * alpha; bb += beta * beta;
    }
    float const det = aa * bb - ab * ab;
    if (!(fabsf(det) > 0.00001f)) return false;
    float const rcp = 1.f / det;
    V3 const u = (alphaSum * bb - betaSum * ab) * rcp, v = (betaSum * aa - alphaSum * ab) * rcp;
    // (the shader clamps these codes to 65504, which lets the codes of infinities and NaNs through)
    outLo = V3{ from_half_bits(clampf(u.x, 0.f, kHalfMaxCode)), from_half_bits(clampf(u.y, 0.f, kHalfMaxCode)), from_half_bits(clampf(u.z, 0.f, kHalfMaxCode)) };
    outHi = V3{ from_half_bits(clampf(v.x, 0.f, kHalfMaxCode)), from_half_bits(clampf(v.y, 0.f, kHalfMaxCode)), from_half_bits(clampf(v.z, 0.f, kHalfMaxCode)) };
    return true;
}

// 128-bit field writer for constant positions.
struct Bits {
    uint64_t lo = 0, hi = 0;
    BC6_INLINE void put(int at, uint32_t value, int n)
    {
        uint64_t const v = value & ((1u << n) - 1u);
        if (at < 64) { lo |= v << at; if (at + n > 64) hi |= v >> (64 - at); }
        else hi |= v << (at - 64);
    }
};

// Endpoints of the one-subset candidate, in the order that gives texel 0 an index below 8 (`lo` and the first code are
// the first endpoint's).
template <bool WIDE>
BC6_TASK void one_subset_ends(Bc6Ptr lds, int b)
{
    V3 lo = texel(lds, b, 0), hi = lo;
#pragma unroll 5
    for (int t = 1; t < 16; ++t) { V3 const p = texel(lds, b, t); lo = vmin(lo, p); hi = vmax(hi, p); }
    V3 const boxLo = lo, boxHi = hi;
    inset_box(lds, b, lo, hi);
    V3 fitLo, fitHi;
    if (refit<WIDE, true>(lds, b, 0xffffu, lo, hi, fitLo, fitHi)) {
        lo = vmin(vmax(fitLo, boxLo), boxHi);
        hi = vmin(vmax(fitHi, boxLo), boxHi);
    }
    SubsetEnds s{ lo, hi, direction<WIDE>(lo, hi), 0.f, 0.f };
    s.e0 = to_half_bits(dot(lo, s.dir)); s.e1 = to_half_bits(dot(hi, s.dir));
    if (index4(to_half_bits(dot(texel(lds, b, 0), s.dir)), s.e0, s.e1) > 7) {
        float const e = s.e0; s.e0 = s.e1; s.e1 = e;
        V3 const v = s.lo; s.lo = s.hi; s.hi = v;
    }
    store_ends(lds->one, b, s);
}

template <bool WIDE> BC6_INLINE V3 normalized(V3 v) { return divided<WIDE>(v, sqrtf(dot(v, v))); }
BC6_INLINE float distance_to_line2(V3 origin, V3 dir, V3 p)
{
    V3 const w = p - origin, x = w - dir * dot(w, dir);
    return dot(x, x);
}

// A pattern's score is the sum of the texels' squared distances from the diagonal of their subset's bounding box; the
// pattern of the first smallest score is wanted, not the score.  It is bounded first, by the difference of the sums of
// |w|^2 and (w . d)^2 over the offsets w from the box's corner: half the operations, in any order.  Both that sum and
// the score as it is defined lie within a hundred units of roundoff of the sum of |w|^2 from the true value, so kScoreError
// of 512 units separates all patterns but the nearly equal ones, which alone are evaluated as defined.
constexpr float kScoreError = 0x1p-15f;
// Squared diagonals below this (texels of a FLOAT32 image can be that close) leave the bounds to underflow.
constexpr float kShortDiagonal = 1e-30f;

// Adds the two sums over the N texels of a subset (uniform) and takes the minimum of the diagonals' squares, -1 for a
// subset of equal texels: it has no direction, which makes the pattern's score a NaN.
template <int N> BC6_INLINE void bound_subset(Bc6Ptr lds, int b, uint32_t members, float& lengths, float& along, float& shortest)
{
    V3 p[N];
#pragma unroll
    for (int i = 0; i < N; ++i) { p[i] = texel(lds, b, __ffs(int(members)) - 1); members &= members - 1; }
    V3 lo = p[0], hi = p[0];
#pragma unroll
    for (int i = 1; i + 1 < N; i += 2) {
        lo = V3{ min3_f32(lo.x, p[i].x, p[i + 1].x), min3_f32(lo.y, p[i].y, p[i + 1].y), min3_f32(lo.z, p[i].z, p[i + 1].z) };
        hi = V3{ max3_f32(hi.x, p[i].x, p[i + 1].x), max3_f32(hi.y, p[i].y, p[i + 1].y), max3_f32(hi.z, p[i].z, p[i + 1].z) };
    }
    if constexpr (!(N & 1)) { lo = vmin(lo, p[N - 1]); hi = vmax(hi, p[N - 1]); }
    V3 const v = hi - lo;
    float const square = dot(v, v);
    V3 const d = v * __builtin_amdgcn_rsqf(square);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        V3 const w = p[i] - lo;
        lengths = __builtin_fmaf(w.x, w.x, lengths);
        lengths = __builtin_fmaf(w.y, w.y, lengths);
        lengths = __builtin_fmaf(w.z, w.z, lengths);
        float const c = __builtin_fmaf(w.z, d.z, __builtin_fmaf(w.y, d.y, w.x * d.x));
        along = __builtin_fmaf(c, c, along);
    }
    // (equal texels: -1)
    shortest = fminf(shortest, v.x == 0.f && v.y == 0.f && v.z == 0.f ? -1.f : square);
}
BC6_INLINE void bound_members(Bc6Ptr lds, int b, uint32_t members, float& lengths, float& along, float& shortest)
{
    switch (__popc(members)) {                               // the sizes that the patterns' subsets have
    case 3:  bound_subset<3>(lds, b, members, lengths, along, shortest); break;
    case 4:  bound_subset<4>(lds, b, members, lengths, along, shortest); break;
    case 6:  bound_subset<6>(lds, b, members, lengths, along, shortest); break;
    case 8:  bound_subset<8>(lds, b, members, lengths, along, shortest); break;
    case 10: bound_subset<10>(lds, b, members, lengths, along, shortest); break;
    case 12: bound_subset<12>(lds, b, members, lengths, along, shortest); break;
    default: bound_subset<13>(lds, b, members, lengths, along, shortest); break;
    }
}

// The least value of each score of the patterns that this wave takes (infinity for a NaN, -1 if there are no bounds), and
// in `pick` the smallest greatest value.
BC6_TASK void bound_scores(Bc6Ptr lds, int b)
{
    float best = __builtin_inff();
#pragma unroll 1
    for (;;) {
        int p = 0;
        if (b == 0) p = __hip_atomic_fetch_add(&lds->next, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        p = __builtin_amdgcn_readfirstlane(p);
        if (p >= 32) break;                                  // uniform: every wave gets here
        uint32_t members = kSecondSubset[p];
        float lengths = 0.f, along = 0.f, shortest = 1.f;
#pragma unroll 1
        for (int s = 0; s < 2; ++s, members ^= 0xffffu) bound_members(lds, b, members, lengths, along, shortest);
        float const score = lengths - along, error = lengths * kScoreError;
        float least = fmaxf(score - error, 0.f);
        if (shortest < kShortDiagonal) least = shortest < 0.f ? __builtin_inff() : -1.f;
        else best = fminf(best, score + error);
        lds->least[p][b] = least;
        if (p == 0) lds->unscored[b] = shortest < 0.f;
    }
    __hip_atomic_fetch_min(&lds->bound[b], __float_as_uint(fmaxf(best, 0.f)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Which of the eight patterns 8 * wave ... could have the smallest score.
BC6_INLINE uint32_t candidate_patterns(Bc6Ptr lds, int b, int wave)
{
    float const bound = __uint_as_float(lds->bound[b]);
    uint32_t mask = 0;
    bool unbounded = false;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        float const least = lds->least[8 * wave + i][b];
        if (least <= bound && least < __builtin_inff()) mask |= 1u << i;
        unbounded |= least < 0.f;
    }
    __hip_atomic_fetch_or(&lds->candidates[b], mask << (8 * wave), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (unbounded) lds->unbounded[b] = 1u;
    return mask;
}

// Scores, as they are defined, of the candidates among the eight patterns 8 * wave ... of blocks with more than one, each
// lane with a pattern of its own.
template <bool WIDE>
BC6_TASK void score_candidates(Bc6Ptr lds, int b, int wave, uint32_t mask)
{
    wave = __builtin_amdgcn_readfirstlane(wave);
    uint64_t best = ~uint64_t(0);
#pragma unroll 1
    for (; mask; mask &= mask - 1u) {
        int const p = 8 * wave + __ffs(int(mask)) - 1;
        uint32_t const second = kSecondSubset[p];
        V3 lo0{ kHalfMax, kHalfMax, kHalfMax }, hi0{ 0.f, 0.f, 0.f }, lo1 = lo0, hi1 = hi0;
#pragma unroll 4
        for (int t = 0; t < 16; ++t) {
            V3 const q = texel(lds, b, t);
            if ((second >> t) & 1u) { lo1 = vmin(lo1, q); hi1 = vmax(hi1, q); }
            else                    { lo0 = vmin(lo0, q); hi0 = vmax(hi0, q); }
        }
        V3 const dir0 = normalized<WIDE>(hi0 - lo0), dir1 = normalized<WIDE>(hi1 - lo1);
        float score = 0.f;
#pragma unroll 4
        for (int t = 0; t < 16; ++t) {
            bool const s = (second >> t) & 1u;
            V3 const lo{ s ? lo1.x : lo0.x, s ? lo1.y : lo0.y, s ? lo1.z : lo0.z }, dir{ s ? dir1.x : dir0.x, s ? dir1.y : dir0.y, s ? dir1.z : dir0.z };
            score += distance_to_line2(lo, dir, texel(lds, b, t));
        }
        // scores are not negative, a NaN's bits are above all numbers': the smallest key is the first smallest score
        uint64_t const key = uint64_t(__float_as_uint(score) & 0x7fffffffu) << 32 | uint32_t(p);
        best = key < best ? key : best;
        if (p == 0) lds->unscored[b] = score != score;
    }
    __hip_atomic_fetch_min(&lds->pick[b], best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

BC6_INLINE int picked_pattern(Bc6Ptr lds, int b) { return lds->unscored[b] ? 0 : int(uint32_t(lds->pick[b])); }

// Endpoints of subset s of the picked pattern, in the order that gives its anchor an index below 4.
template <bool WIDE>
BC6_TASK void subset_ends(Bc6Ptr lds, int b, int s)
{
    s = __builtin_amdgcn_readfirstlane(s);
    int const pattern = picked_pattern(lds, b);
    uint32_t const members = s ? uint32_t(kSecondSubset[pattern]) : ~uint32_t(kSecondSubset[pattern]) & 0xffffu;
    V3 lo{ kHalfMax, kHalfMax, kHalfMax }, hi{ 0.f, 0.f, 0.f };
    for (uint32_t m = members; m; m &= m - 1) { V3 const p = texel(lds, b, __ffs(int(m)) - 1); lo = vmin(lo, p); hi = vmax(hi, p); }
    V3 fitLo, fitHi;
    if (refit<WIDE, false>(lds, b, members, lo, hi, fitLo, fitHi)) { lo = fitLo; hi = fitHi; }
    SubsetEnds e{ lo, hi, direction<WIDE>(lo, hi), 0.f, 0.f };
    e.e0 = to_half_bits(dot(lo, e.dir)); e.e1 = to_half_bits(dot(hi, e.dir));
    if (index3(to_half_bits(dot(texel(lds, b, s ? int(kSecondAnchor[pattern]) : 0), e.dir)), e.e0, e.e1) > 3) {
        float const x = e.e0; e.e0 = e.e1; e.e1 = x;
        V3 const v = e.lo; e.lo = e.hi; e.hi = v;
    }
    store_ends(lds->two[s], b, e);
}

BC6_INLINE uint32_t field(float v, int bits) { return uint32_t(int(v)) & ((1u << bits) - 1u); }      // two's complement of a small integer
BC6_INLINE V3 floor3(V3 v) { return { floorf(v.x), floorf(v.y), floorf(v.z) }; }
BC6_INLINE V3 clamp3(V3 v, float limit) { return { clampf(v.x, -limit, limit), clampf(v.y, -limit, limit), clampf(v.z, -limit, limit) }; }

// The two-subset endpoints as a base and three signed deltas.
BC6_INLINE void base_and_deltas(Bc6Ptr lds, int b, float levels, float limit, V3 (&q)[4])
{
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        auto const& from = lds->two[i >> 1];
        int const at = 3 * (i & 1);
        q[i] = floor3(quantize(V3{ from[at][b], from[at + 1][b], from[at + 2][b] }, levels));
    }
#pragma unroll
    for (int i = 1; i < 4; ++i) q[i] = clamp3(q[i] - q[0], limit);
}

// Indices of four texels under the one-subset candidate and, as an estimate, what they add to its error.
template <bool WIDE>
BC6_TASK void estimate_one_subset(Bc6Ptr lds, int b, int quarter)
{
    quarter = __builtin_amdgcn_readfirstlane(quarter);
    SubsetEnds const one = load_ends(lds->one, b);
    V3 const u0 = unquantize(quantize(one.lo, 1024.f), 1024.f), u1 = unquantize(quantize(one.hi, 1024.f), 1024.f);
    uint32_t indices4 = 0;
    float error1 = 0.f;
#pragma unroll 2
    for (int i = 0; i < 4; ++i) {
        V3 const p = texel(lds, b, 4 * quarter + i);
        uint32_t const index = index4(to_half_bits(dot(p, one.dir)), one.e0, one.e1);
        indices4 |= index << (4 * i);
        error1 += Msle<WIDE>(p).estimate(interpolate(u0, u1, float(weight4(index))));
    }
    lds->indices[0][quarter][b] = indices4;
    lds->errors[0][quarter][b] = error1;
}

// The same under the two candidates with two subsets.
template <bool WIDE>
BC6_TASK void estimate_two_subsets(Bc6Ptr lds, int b, int quarter)
{
    quarter = __builtin_amdgcn_readfirstlane(quarter);
    V3 u7[4], u9[4];
    {
        V3 q[4];
        base_and_deltas(lds, b, 128.f, 31.f, q);
        u7[0] = unquantize(q[0], 128.f);
#pragma unroll
        for (int i = 1; i < 4; ++i) u7[i] = unquantize(q[0] + q[i], 128.f);
        base_and_deltas(lds, b, 512.f, 15.f, q);
        u9[0] = unquantize(q[0], 512.f);
#pragma unroll
        for (int i = 1; i < 4; ++i) u9[i] = unquantize(q[0] + q[i], 512.f);
    }
    uint32_t const second = kSecondSubset[picked_pattern(lds, b)] >> (4 * quarter);
    uint32_t indices3 = 0;
    float error7 = 0.f, error9 = 0.f;
#pragma unroll 2
    for (int i = 0; i < 4; ++i) {
        V3 const p = texel(lds, b, 4 * quarter + i);
        Msle<WIDE> const error(p);
        bool const s = (second >> i) & 1u;
        V3 const dir{ lds->two[s][6][b], lds->two[s][7][b], lds->two[s][8][b] };
        uint32_t const inSubset = index3(to_half_bits(dot(p, dir)), lds->two[s][9][b], lds->two[s][10][b]);
        indices3 |= inSubset << (3 * i);
        float const weight = float(weight3(inSubset));
        error7 += error.estimate(interpolate_integers(s ? u7[2] : u7[0], s ? u7[3] : u7[1], weight));
        error9 += error.estimate(interpolate_integers(s ? u9[2] : u9[0], s ? u9[3] : u9[1], weight));
    }
    lds->indices[1][quarter][b] = indices3;
    lds->errors[1][quarter][b] = error7; lds->errors[2][quarter][b] = error9;
}

// What the estimates say of the choice between the candidates; 3: nothing.  An estimate and the error as it is defined
// are sums of 48 terms that differ by 2^-19, in different orders: within 2^-18.5 of each other.
BC6_INLINE int estimated_choice(Bc6Ptr lds, int b)
{
    float e[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) e[c] = (lds->errors[c][0][b] + lds->errors[c][1][b]) + (lds->errors[c][2][b] + lds->errors[c][3][b]);
    constexpr float kSure = 1.f - 0x1p-17f;
    auto const less = [&](int x, int y) { return e[x] < e[y] * kSure; };
    if (less(0, 1) && less(0, 2)) return 0;
    if (less(1, 2) && less(1, 0)) return 1;
    if (less(2, 1) && less(2, 0)) return 2;
    return 3;
}

// The choice between the candidates of one block (by its lanes, sixteen to a block, a texel each) by their errors as they
// are defined, added up in texel order.
template <bool WIDE>
BC6_TASK int defined_choice(Bc6Ptr lds, int b, int t)
{
    V3 const p = texel(lds, b, t);
    Msle<WIDE> const error(p);
    float of[3], sum[3] = { 0.f, 0.f, 0.f };
    {
        SubsetEnds const s = load_ends(lds->one, b);
        V3 const u0 = unquantize(quantize(s.lo, 1024.f), 1024.f), u1 = unquantize(quantize(s.hi, 1024.f), 1024.f);
        of[0] = error(interpolate(u0, u1, float(weight4((lds->indices[0][t >> 2][b] >> (4 * (t & 3))) & 15u))));
    }
    int const s = (kSecondSubset[picked_pattern(lds, b)] >> t) & 1;
    float const weight = float(weight3((lds->indices[1][t >> 2][b] >> (3 * (t & 3))) & 7u));
#pragma unroll 1
    for (int c = 1; c < 3; ++c) {
        float const levels = c == 1 ? 128.f : 512.f;
        V3 q[4];
        base_and_deltas(lds, b, levels, c == 1 ? 31.f : 15.f, q);
        V3 const u0 = unquantize(s ? q[0] + q[2] : q[0], levels), u1 = unquantize(q[0] + (s ? q[3] : q[1]), levels);
        float const e = error(interpolate_integers(u0, u1, weight));
        of[1] = c == 1 ? e : of[1]; of[2] = e;
    }
    int const lane = int(threadIdx.x) & 63;
#pragma unroll
    for (int k = 0; k < 16; ++k)
#pragma unroll
        for (int c = 0; c < 3; ++c) sum[c] += __shfl(of[c], (lane & 48) + k, 64);
    float const least = fminf(sum[1], sum[2]);
    return !(least < sum[0]) ? 0 : least == sum[1] ? 1 : 2;
}

// The block of the candidate: 0 one subset, 1 two with 7 + 6 bits, 2 two with 9 + 5 bits.
BC6_INLINE void final_block(Bc6Ptr lds, int b, int choice, uint64_t& outLo, uint64_t& outHi)
{
    Bits bits;
    if (choice == 0) {
        V3 const q0 = quantize(V3{ lds->one[0][b], lds->one[1][b], lds->one[2][b] }, 1024.f), q1 = quantize(V3{ lds->one[3][b], lds->one[4][b], lds->one[5][b] }, 1024.f);
        bits.put(0, 0x03, 5);
        bits.put(5, uint32_t(q0.x), 10); bits.put(15, uint32_t(q0.y), 10); bits.put(25, uint32_t(q0.z), 10);
        bits.put(35, uint32_t(q1.x), 10); bits.put(45, uint32_t(q1.y), 10); bits.put(55, uint32_t(q1.z), 10);
        uint64_t const indices = uint64_t(lds->indices[0][0][b]) | uint64_t(lds->indices[0][1][b]) << 16 | uint64_t(lds->indices[0][2][b]) << 32 | uint64_t(lds->indices[0][3][b]) << 48;
        // texel 0 has three bits from bit 65 on, the others four each
        outLo = bits.lo;
        outHi = bits.hi | (indices & 7u) << 1 | (indices & ~uint64_t(15));
        return;
    }
    int const pattern = picked_pattern(lds, b), anchor1 = kSecondAnchor[pattern];
    bool const sevenSix = choice == 1;
    V3 q[4];
    base_and_deltas(lds, b, sevenSix ? 128.f : 512.f, sevenSix ? 31.f : 15.f, q);
    int const baseBits = sevenSix ? 7 : 9, deltaBits = sevenSix ? 6 : 5;
    V3 const w = q[0], x = q[1], y = q[2], z = q[3];
    uint32_t const rw = field(w.x, baseBits), gw = field(w.y, baseBits), bw = field(w.z, baseBits);
    uint32_t const rx = field(x.x, deltaBits), gx = field(x.y, deltaBits), bx = field(x.z, deltaBits);
    uint32_t const ry = field(y.x, deltaBits), gy = field(y.y, deltaBits), by = field(y.z, deltaBits);
    uint32_t const rz = field(z.x, deltaBits), gz = field(z.y, deltaBits), bz = field(z.z, deltaBits);
    if (sevenSix) {         // mode 2 of the format: 7.666
        bits.put(0, 0x01, 2);
        bits.put(2, gy >> 5, 1); bits.put(3, gz >> 4, 1); bits.put(4, gz >> 5, 1);
        bits.put(5, rw, 7); bits.put(12, bz, 1); bits.put(13, bz >> 1, 1); bits.put(14, by >> 4, 1);
        bits.put(15, gw, 7); bits.put(22, by >> 5, 1); bits.put(23, bz >> 2, 1); bits.put(24, gy >> 4, 1);
        bits.put(25, bw, 7); bits.put(32, bz >> 3, 1); bits.put(33, bz >> 5, 1); bits.put(34, bz >> 4, 1);
        bits.put(35, rx, 6); bits.put(41, gy, 4); bits.put(45, gx, 6); bits.put(51, gz, 4); bits.put(55, bx, 6); bits.put(61, by, 4);
        bits.put(65, ry, 6); bits.put(71, rz, 6);
    } else {                // mode 6 of the format: 9.555
        bits.put(0, 0x0E, 5);
        bits.put(5, rw, 9); bits.put(14, by >> 4, 1); bits.put(15, gw, 9); bits.put(24, gy >> 4, 1); bits.put(25, bw, 9); bits.put(34, bz >> 4, 1);
        bits.put(35, rx, 5); bits.put(40, gz >> 4, 1); bits.put(41, gy, 4); bits.put(45, gx, 5); bits.put(50, bz, 1); bits.put(51, gz, 4);
        bits.put(55, bx, 5); bits.put(60, bz >> 1, 1); bits.put(61, by, 4); bits.put(65, ry, 5); bits.put(70, bz >> 2, 1); bits.put(71, rz, 5); bits.put(76, bz >> 3, 1);
    }
    bits.put(77, uint32_t(pattern), 5);
    // three bits per texel from bit 82 on, the anchors' (texel 0 and anchor1) without the top one, which is zero
    uint64_t indices = uint64_t(lds->indices[1][0][b]) | uint64_t(lds->indices[1][1][b]) << 12 | uint64_t(lds->indices[1][2][b]) << 24 | uint64_t(lds->indices[1][3][b]) << 36;
    uint64_t const below = (uint64_t(1) << (3 * anchor1 + 2)) - 1u;
    indices = (indices & below) | ((indices >> 1) & ~below);
    indices = (indices & 3u) | ((indices >> 1) & ~uint64_t(3));
    outLo = bits.lo;
    outHi = bits.hi | indices << 18;
}

} // namespace

template <bool WIDE>
__global__ void __launch_bounds__(256, 5)
bc6_compress_kernel(BlockCompressArgs a)
{
    __shared__ Bc6Lds shared;
    Bc6Ptr const lds = (Bc6Ptr)&shared;
    int const tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int const bx = blockIdx.x * 8 + (lane & 7), by = blockIdx.y * 8 + (lane >> 3);
    bool const inside = bx < a.widthInBlocks && by < a.heightInBlocks;
    // a row of the block per wave; lanes outside encode black
    float texels[1][4][3] = {};
    if (inside) source_rows<3, 1>(a, a.srcLeft + bx * 4, a.srcTop + by * 4 + wave, 0, texels);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float const (&c)[3] = texels[0][i];
        shared.texels[4 * wave + i][lane] = make_float4(clampf(c[0], 0.f, kHalfMax), clampf(c[1], 0.f, kHalfMax), clampf(c[2], 0.f, kHalfMax), 0.f);
    }
    if (wave == 0) {
        shared.pick[lane] = ~uint64_t(0);
        shared.bound[lane] = 0x7f800000u; shared.candidates[lane] = shared.unbounded[lane] = 0u;
        if (lane == 0) shared.next = 0;
    }
    __syncthreads();
    if (wave == 0) one_subset_ends<WIDE>(lds, lane);
    bound_scores(lds, lane);
    __syncthreads();
    uint32_t mask = candidate_patterns(lds, lane, wave);
    __syncthreads();
    uint32_t const candidates = shared.candidates[lane];
    if ((candidates & (candidates - 1u)) == 0u && !shared.unbounded[lane]) {
        if (mask) shared.pick[lane] = uint32_t(8 * wave + __ffs(int(mask)) - 1);
        mask = 0u;
    }
    if (__any(mask != 0u)) score_candidates<WIDE>(lds, lane, wave, mask);
    __syncthreads();
    // (two waves for the subsets, the others for the candidate that has none: as much work)
    if (wave < 2) {
        subset_ends<WIDE>(lds, lane, wave);
    } else {
        estimate_one_subset<WIDE>(lds, lane, 2 * wave - 4);
        estimate_one_subset<WIDE>(lds, lane, 2 * wave - 3);
    }
    __syncthreads();
    estimate_two_subsets<WIDE>(lds, lane, wave);
    __syncthreads();
    int choice = estimated_choice(lds, lane);
    uint64_t const open = __ballot(choice == 3);             // the same in all waves, few
    if (open) {
        if (choice == 3) shared.candidates[__popcll(open & ((uint64_t(1) << lane) - 1u))] = uint32_t(lane);
        __syncthreads();
        int const last = __popcll(open) - 1;
        for (int first = 4 * wave; first <= last; first += 16) {
            int const b = int(shared.candidates[min(first + (lane >> 4), last)]);
            shared.bound[b] = uint32_t(defined_choice<WIDE>(lds, b, lane & 15));
        }
        __syncthreads();
        if (choice == 3) choice = int(shared.bound[lane]);
    }
    if (wave != 0 || !inside) return;
    uint64_t lo, hi;
    final_block(lds, lane, choice, lo, hi);
    uint64_t* const dst = reinterpret_cast<uint64_t*>(a.dst + size_t(by + a.dstOffsetY) * a.dstRowPitch) + size_t(bx + a.dstOffsetX) * 2;
    dst[0] = lo; dst[1] = hi;
}

hipError_t launch_bc6_compress(BlockCompressArgs const& a, hipStream_t stream)
{
    dim3 const grid((a.widthInBlocks + 7) / 8, (a.heightInBlocks + 7) / 8);
    if (a.format == NTC_HIP_DEV_FORMAT_FLOAT32) hipLaunchKernelGGL(bc6_compress_kernel<true>, grid, dim3(256), 0, stream, a);
    else                                        hipLaunchKernelGGL(bc6_compress_kernel<false>, grid, dim3(256), 0, stream, a);
    return hipGetLastError();
}

} // namespace ntc_hip_dev
