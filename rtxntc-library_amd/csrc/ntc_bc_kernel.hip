// ntc_bc_kernel.hip - BC1 .. BC5 block compression of a decoded image (gfx950).
//
// The step after decode in a load path that hands block-compressed textures to a renderer:
// the reference runs it as a graphics compute pass (IContext::MakeBlockCompressionComputePass,
// src/shaders/CompressBC1.hlsl .. CompressBC5.hlsl, src/shaders/BlockCompressCommon.hlsli).
// (One thread encodes a 4 x 4 block there; here waves share the candidates of 64 blocks.)
//
// BC4 (one channel; BC5 = two of them, BC3 = one for alpha).  The encoder tries both BC4 palettes.
// Eight-value palette (endpoint 0 > endpoint 1): start from the
// block's extremes pulled inwards by 1/34 of the range (extremes of exactly 0 or 255 stay), assign
// every texel its nearest palette entry, then up to eight rounds of "least-squares endpoints for
// the current assignment, re-assign", stopping when the error no longer falls or the assignment
// repeats.  Six-value palette (endpoint 0 <= endpoint 1, entries 6 and 7 are 0 and 255): the same
// from the extremes that are not 0 / 255.  The candidate with the smaller squared error wins, the
// eight-value one on a tie.
//
// BC1 colour (also the colour half of BC2 and BC3).  Candidates, the first of the smallest squared
// error (over r, g, b and alpha against 1) wins:
//   * BC1 only: the all-transparent block;
//   * one colour: the block's mean, each component through a table of the endpoint pair whose
//     1/3 : 2/3 mix comes nearest to it;
//   * four-colour mode: endpoints from the bounding box of the block (corners paired by the sign of
//     the covariances, pulled inwards by 1/16), then up to four rounds of nearest-entry assignment
//     + least-squares endpoints + rounding to 5:6:5;
//   * BC1 only: three-colour mode with transparent texels (alpha <= threshold) left out, one round.
// BC2 alpha is 4 bits per texel.
//
// All float arithmetic is IEEE binary32, unfused, in the order written here.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include "ntc_decode_kernel.h"
#include "ntc_bc_source.h"

namespace ntc_hip_dev {

namespace {

// A block of one channel: four texels of a row a word, and in 16-bit lanes, of each row the texels 0 and 2, 1 and 3.
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
struct Bc4Texels {
    uint32_t rows[4];
    u16x2 even[4], odd[4];
    uint32_t lo, hi, squares;                                // extremes, sum of squares
};

// A block's endpoints, and where its texels lie between them: a position a byte, four texels a word.  Position 0 is
// endpoint 0, the last one (7, or 5 in the six-value palette) endpoint 1; 6 and 7 of the six-value palette are 0 and 255.
struct Bc4 { uint32_t e0, e1, positions[4]; };

// The block: endpoints and, of sixteen texels, the 3-bit indices that their positions stand for.
template <bool EIGHT>
__device__ __forceinline__ uint64_t bc4_bits(Bc4 const& block)
{
    uint64_t bits = uint64_t(block.e0) | (uint64_t(block.e1) << 8);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        uint32_t const k = __builtin_amdgcn_perm(EIGHT ? 0x01070605u : 0x07060105u, 0x04030200u, block.positions[r]);
        bits |= uint64_t(__builtin_amdgcn_udot4(k, 0x00400801u, (k >> 24) << 9, false)) << (16 + 12 * r);
    }
    return bits;
}

// The eight values that two endpoints stand for, times eight.  With e0 > e1 entry k + 1 is ((7 - k) e0 + k e1 + 3) / 7,
// else ((5 - k) e0 + k e1 + 2) / 5 and the last two are 0 and 255 (the reference's rounding biases); a product and a
// shift are those quotients for every numerator that occurs.
__device__ __forceinline__ void bc4_palette8(uint32_t e0, uint32_t e1, uint32_t (&p)[8])
{
    bool const eight = e0 > e1;
    uint32_t const multiplier = eight ? 9363u : 13108u, step = e1 - e0;
    uint32_t n = eight ? 7u * e0 + 3u : 5u * e0 + 2u;
    p[0] = e0 << 3; p[1] = e1 << 3;
#pragma unroll
    for (int k = 2; k < 8; ++k) {
        n += step;
        p[k] = (__umul24(n, multiplier) >> 13) & ~7u;
    }
    if (!eight) { p[6] = 0u; p[7] = 255u << 3; }
}

// The entries between two endpoints R apart, and where a texel lies among them.  The entry at position j is
// q(j) = (j R + LAST / 2) / LAST away from endpoint 0 (that is what the biased quotients come to).  A texel d away from it
// takes the nearest entry, of equally near ones the first in the order of the indices: the earlier position, but the last
// one before those between the ends.  In sixteen bits and for 0 <= d <= R that position is
//     (scale * d + start + kink * max(d - before, 0)) >> 13:
// the steps of a line while all ties fall to one side, lifted at its end (kink) where the last two entries tie.  Scale and
// start are found by trial, as the compiler runs, for every d that there is.
struct alignas(16) Bc4Range { uint32_t near, far, line, bend; };         // q(0) ... q(3), q(4) ... q(7), scale | start << 16, kink | before << 16
template <uint32_t LAST> struct Bc4Ranges { Bc4Range of[256]; };
template <uint32_t LAST>
constexpr Bc4Ranges<LAST> bc4_ranges()
{
    Bc4Ranges<LAST> table{};
    for (uint32_t range = 0; range < 256; ++range) {
        uint32_t q[8] = {}, position[256] = {};
        for (uint32_t j = 0; j <= LAST; ++j) q[j] = (j * range + LAST / 2) / LAST;
        Bc4Range& entry = table.of[range];
        entry.near = q[0] | q[1] << 8 | q[2] << 16 | q[3] << 24;
        entry.far = q[4] | q[5] << 8 | q[6] << 16 | q[7] << 24;
        if (range == 0) continue;                            // position 0
        uint32_t const first = (q[LAST - 1] + range + 1) / 2;                    // the last position's first texel
        for (uint32_t d = 0, j = 0; d < first; ++d) {
            while (2 * d > q[j] + q[j + 1]) ++j;
            uint32_t same = j;
            while (same > 0 && q[same - 1] == q[same]) --same;
            position[d] = same;
        }
        bool found = false;
        // (from the line through the ends outwards; two entries of range 2 lie four positions apart)
        uint32_t const middle = LAST == 7 && range == 2 ? 2 * 8192 : LAST * 8192 / range;
        for (uint32_t trial = 0; trial < 8 && !found; ++trial) {
            uint32_t const scale = trial & 1 ? middle - trial / 2 - 1 : middle + trial / 2;
            int32_t from = 0, to = 8191;
            for (uint32_t d = 0; d < first; ++d) {
                int32_t const least = int32_t(position[d] * 8192) - int32_t(d * scale);
                if (least > from) from = least;
                if (least + 8191 < to) to = least + 8191;
                if (from > to) break;
            }
            if (from > to) continue;
            uint32_t const start = uint32_t(to), reached = first * scale + start, kink = reached < LAST * 8192 ? LAST * 8192 - reached : 0;
            found = range * scale + start + (range - first + 1) * kink < (LAST + 1) * 8192;
            entry.line = scale | start << 16;
            entry.bend = kink | (first - 1) << 16;
        }
        if (!found) __builtin_unreachable();                 // (does not compile)
    }
    return table;
}
struct Bc4Tables { Bc4Ranges<7> eight; Bc4Ranges<5> six; };
__device__ constexpr Bc4Tables kBc4Tables{ bc4_ranges<7>(), bc4_ranges<5>() };

// Copies them to the workgroup's memory: every thread takes part, they are there after the next barrier.
__device__ __forceinline__ void bc4_stage(Bc4Tables& tables, uint32_t threads)
{
    for (uint32_t i = threadIdx.x; i < 256; i += threads) {
        tables.eight.of[i] = kBc4Tables.eight.of[i];
        tables.six.of[i] = kBc4Tables.six.of[i];
    }
}

// Nearest palette entry for every texel, from the definition: the palette that the endpoints' order stands for, whatever
// palette is searched for.
template <bool EIGHT>
__device__ __forceinline__ uint32_t bc4_assign_defined(Bc4Texels const& texels, Bc4& block)
{
    uint32_t p[8], total = 0;
    bc4_palette8(block.e0, block.e1, p);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        uint32_t indices = 0;
#pragma unroll 1
        for (int i = 0; i < 32; i += 8) {
            uint32_t const value8 = ((texels.rows[r] >> i) & 0xffu) << 3;
            uint32_t best = ~0u;
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) best = min(best, uint32_t(abs(int(value8) - int(p[k]))) | k);
            total += (best >> 3) * (best >> 3);
            indices |= (best & 7u) << i;
        }
        block.positions[r] = __builtin_amdgcn_perm(EIGHT ? 0x06050403u : 0x07060403u, EIGHT ? 0x02010700u : 0x02010500u, indices);
    }
    return total;
}

// Nearest palette entry for every texel (the first of equally near ones); returns the summed squared error.
// Positions by a line in packed 16-bit arithmetic, entries by byte permutes, the error from byte dot products as
// sum v^2 - 2 sum v p + sum p^2: 14 instructions for four texels.  (The distances to all eight entries and their minima took 70.)
template <bool EIGHT>
__device__ __forceinline__ uint32_t bc4_assign(Bc4Texels const& texels, Bc4Tables const& tables, Bc4& block)
{
    if (EIGHT ? block.e0 <= block.e1 : block.e0 > block.e1) return bc4_assign_defined<EIGHT>(texels, block);   // the other palette: rare
    uint32_t const range = EIGHT ? block.e0 - block.e1 : block.e1 - block.e0, base = block.e0 * 0x01010101u;
    Bc4Range const entry = EIGHT ? tables.eight.of[range] : tables.six.of[range];
    uint32_t const near = EIGHT ? base - entry.near : base + entry.near;         // (no byte borrows or carries)
    uint32_t const far = EIGHT ? base - entry.far : ((base + entry.far) & 0xffffu) | 0xff000000u;
    uint16_t const e0 = uint16_t(block.e0), r16 = uint16_t(range), scale = uint16_t(entry.line), start = uint16_t(entry.line >> 16);
    uint16_t const kink = uint16_t(entry.bend), before = uint16_t(entry.bend >> 16);
    auto const place = [&](u16x2 v) {
        u16x2 d = EIGHT ? __builtin_elementwise_sub_sat(u16x2(e0), v) : __builtin_elementwise_sub_sat(v, u16x2(e0));
        d = __builtin_elementwise_min(d, u16x2(r16));
        return __builtin_elementwise_sub_sat(d, u16x2(before)) * kink + (d * scale + start);
    };
    u16x2 even[4], odd[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) { even[r] = place(texels.even[r]); odd[r] = place(texels.odd[r]); }
    if constexpr (!EIGHT) {
        // texels nearer to 0 than to endpoint 0, or to 255 than to endpoint 1: positions 0 and 5 (0 if the endpoints are
        // one) become 6 and 7
        if (__any(2u * texels.lo < block.e0 || 2u * texels.hi > 255u + block.e1)) {
            uint16_t const top = uint16_t(255u + block.e1), from5 = uint16_t((range ? 2u : 7u) << 13);
            auto const ends = [&](u16x2& s, u16x2 v) {
                u16x2 const twice = v + v, one = u16x2(uint16_t(1));
                s += __builtin_elementwise_min(__builtin_elementwise_sub_sat(u16x2(e0), twice), one) * uint16_t(6 << 13);
                s += __builtin_elementwise_min(__builtin_elementwise_sub_sat(twice, u16x2(top)), one) * from5;
            };
#pragma unroll
            for (int r = 0; r < 4; ++r) { ends(even[r], texels.even[r]); ends(odd[r], texels.odd[r]); }
        }
    }
    uint32_t square = texels.squares, product = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        uint32_t const high = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, odd[r]), __builtin_bit_cast(uint32_t, even[r]), 0x07030501u);
        block.positions[r] = (high >> 5) & 0x07070707u;
        uint32_t const p = __builtin_amdgcn_perm(far, near, block.positions[r]);
        square = __builtin_amdgcn_udot4(p, p, square, false);
        product = __builtin_amdgcn_udot4(p, texels.rows[r], product, false);
    }
    return square - 2u * product;                            // at most 16 * 255^2: exact as the float sum it stands for
}

__device__ __forceinline__ float bc4_endpoint(float v) { return rintf(__builtin_amdgcn_fmed3f(v, 0.f, 255.f)); }   // a NaN becomes 0

// Least-squares endpoints for the block's current positions, as they are defined: float sums in the texels' order.  EIGHT:
// every texel takes part and the weights of endpoint 0 are 1, 0, 6/7 ... 1/7; otherwise positions 6 and 7 (the fixed 0 and
// 255) are left out and the weights are 1, 0, 4/5 ... 1/5, and a singular system leaves the endpoints alone.  w / 7 as
// w * hi + w * lo with hi + lo = 1/7, w / 5 as w * (1/5), are the correctly rounded quotients for all of them.
template <bool EIGHT>
__device__ __forceinline__ void bc4_solve_defined(Bc4Texels const& texels, Bc4 const& block, float& e0, float& e1)
{
    float aa = 0.f, bb = 0.f, ab = 0.f, ax = 0.f, bx = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        uint32_t const weights = EIGHT ? 0x07070707u - block.positions[r] : __builtin_amdgcn_perm(0x00000001u, 0x02030405u, block.positions[r]);
#pragma unroll
        for (int i = 0; i < 32; i += 8) {
            float const w = float((weights >> i) & 0xffu), x = float((texels.rows[r] >> i) & 0xffu);
            float alpha, beta;
            if constexpr (EIGHT) {
                alpha = __builtin_fmaf(w, 1.f / 7.f, w * float(1.0 / 7.0 - double(1.f / 7.f)));
                beta = 1.f - alpha;
            } else {
                alpha = w * (1.f / 5.f);
                beta = ((block.positions[r] >> i) & 0xffu) >= 6u ? 0.f : 1.f - alpha;        // adding zeros is leaving the texel out
            }
            aa += alpha * alpha; bb += beta * beta; ab += alpha * beta;
            ax += alpha * x; bx += beta * x;
        }
    }
    if constexpr (EIGHT) {
        float const factor = 1.f / (aa * bb - ab * ab);
        e0 = bc4_endpoint((ax * bb - bx * ab) * factor);
        e1 = bc4_endpoint((bx * aa - ax * ab) * factor);
    } else {
        float const det = aa * bb - ab * ab;
        if (det == 0.f) { e0 = float(block.e0); e1 = float(block.e1); return; }
        e0 = bc4_endpoint((ax * bb - bx * ab) / det);
        e1 = bc4_endpoint((bx * aa - ax * ab) / det);
    }
}

// The endpoints that bc4_solve_defined() comes to.  Its sums are those of small integers over LAST or LAST^2, which byte
// dot products give exactly; where no rounding boundary is nearer to the quotient of these than the floats can be off,
// both round alike.  Relative errors in units of 2^-24: 15 of the additions and at most 2.6 of the terms in a sum, so 36.3 of
// the products' magnitudes in a numerator and 36 in the determinant, the quotient's own two and four here: 44 with the
// products of errors, 2 % while the determinant is within 1 % (if it is not, the 51 makes `off` greater than 1/2).  One
// lane in a hundred cannot tell; most of those are at exact ties, which the floats' errors decide.
template <bool EIGHT>
__device__ __forceinline__ void bc4_refit(Bc4Texels const& texels, Bc4& block, bool keep255, bool keep0)
{
    uint32_t aa = 0, bb = 0, ab = 0, ax = 0, bx = 0;
    if constexpr (EIGHT) {
        uint32_t sum = 0, x = 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            uint32_t const j = block.positions[r];
            sum = __builtin_amdgcn_udot4(j, 0x01010101u, sum, false);
            x = __builtin_amdgcn_udot4(texels.rows[r], 0x07070707u, x, false);
            bb = __builtin_amdgcn_udot4(j, j, bb, false);
            bx = __builtin_amdgcn_udot4(j, texels.rows[r], bx, false);
        }
        aa = 16u * 49u - 14u * sum + bb; ab = 7u * sum - bb; ax = x - bx;        // weights 7 - j
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            uint32_t const w = __builtin_amdgcn_perm(0x00000001u, 0x02030405u, block.positions[r]);
            uint32_t const j = __builtin_amdgcn_perm(0x00000504u, 0x03020100u, block.positions[r]);
            aa = __builtin_amdgcn_udot4(w, w, aa, false); bb = __builtin_amdgcn_udot4(j, j, bb, false); ab = __builtin_amdgcn_udot4(w, j, ab, false);
            ax = __builtin_amdgcn_udot4(w, texels.rows[r], ax, false); bx = __builtin_amdgcn_udot4(j, texels.rows[r], bx, false);
        }
    }
    constexpr float kLast = EIGHT ? 7.f : 5.f, kUnits = 44.f * 0x1p-24f;
    uint32_t const axbb = __umul24(ax, bb), bxab = __umul24(bx, ab), bxaa = __umul24(bx, aa), axab = __umul24(ax, ab), aabb = __umul24(aa, bb), abab = __umul24(ab, ab);
    float const perDet = __builtin_amdgcn_rcpf(float(aabb - abab)), unit = kUnits * perDet, dets = float(aabb + abab) * unit;
    float const q0 = float(int32_t(axbb - bxab)) * kLast * perDet, q1 = float(int32_t(bxaa - axab)) * kLast * perDet;
    float const off0 = __builtin_fmaf(float(axbb + bxab) * kLast, unit, max_f32(fabsf(q0), 51.f) * dets);
    float const off1 = __builtin_fmaf(float(bxaa + axab) * kLast, unit, max_f32(fabsf(q1), 51.f) * dets);
    bool const sure0 = fabsf(__builtin_amdgcn_fractf(q0) - 0.5f) > off0, sure1 = fabsf(__builtin_amdgcn_fractf(q1) - 0.5f) > off1;      // (a NaN is not)
    float e0 = bc4_endpoint(q0), e1 = bc4_endpoint(q1);
    if (!((EIGHT && keep255) || sure0) || !((EIGHT && keep0) || sure1)) bc4_solve_defined<EIGHT>(texels, block, e0, e1);
    block.e0 = uint32_t(e0); block.e1 = uint32_t(e1);
    if constexpr (EIGHT) {
        if (keep255) block.e0 = 255u;
        if (keep0) block.e1 = 0u;
        uint32_t const top = max(block.e0, block.e1);
        block.e1 = min(block.e0, block.e1); block.e0 = top;
    }
}

// Up to eight rounds of refit + re-assign from the endpoints (e0, e1); returns the best block and its error.  No round betters
// an error of 0, and none moves endpoints that both stay, or that no texel lies between.  (The last have a singular system,
// which bc4_refit() leaves to the float sums: 256 x 256 with a few such blocks, a ramp from 255 back to 0, BC4 5.4 us, 3.2 without
// their round; 2048 x 2048 9.1 and 5.5.)
template <bool EIGHT>
__device__ __forceinline__ Bc4 bc4_refine(Bc4Texels const& texels, Bc4Tables const& tables, uint32_t e0, uint32_t e1, bool keep255, bool keep0, uint32_t& bestError)
{
    Bc4 block{ e0 & 0xffu, e1 & 0xffu, {} };
    bestError = bc4_assign<EIGHT>(texels, tables, block);
    Bc4 best = block;
    uint32_t const fixed = block.positions[0] & block.positions[1] & block.positions[2] & block.positions[3] & 0x06060606u;
    if (bestError == 0 || (EIGHT ? keep255 && keep0 : fixed == 0x06060606u)) return best;
#pragma unroll 1
    for (int round = 0; round < 8; ++round) {
        bc4_refit<EIGHT>(texels, block, keep255, keep0);
        uint32_t const error = bc4_assign<EIGHT>(texels, tables, block);
        if (error >= bestError) break;
        uint32_t moved = 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) moved |= block.positions[r] ^ best.positions[r];
        best = block;
        if (moved == 0) break;
        bestError = error;
    }
    return best;
}

// The candidate of one palette.
template <bool EIGHT>
__device__ __forceinline__ Bc4 bc4_candidate(Bc4Texels const& texels, Bc4Tables const& tables, uint32_t& error)
{
    uint32_t const lo = texels.lo, hi = texels.hi;
    if constexpr (EIGHT) {
        bool const keep0 = lo == 0, keep255 = hi == 255u;
        uint32_t const inset = (hi - lo) / 34u;
        error = 0;
        if (lo == hi) return Bc4{ hi, lo, {} };              // (a palette of six that has the value)
        return bc4_refine<true>(texels, tables, keep255 ? 255u : hi - inset, keep0 ? 0u : lo + inset, keep255, keep0, error);
    } else {
        // extremes among the values that are not 0 / not 255
        uint32_t inner = 255u, outer = 0;
        if (lo != 0 && hi != 255u) { inner = lo; outer = hi; }
        else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int i = 0; i < 32; i += 8) {
                    uint32_t const v = (texels.rows[r] >> i) & 0xffu;
                    if (v != 0) inner = min(inner, v);
                    if (v != 255u) outer = max(outer, v);
                }
        }
        // eight values hold a range of seven, and 0 with 255, without error, and win then
        error = ~0u;
        if (hi - lo <= 7u || inner > outer) return Bc4{ 0u, 0u, {} };
        uint32_t const inset = (outer - inner) / 34u;
        return bc4_refine<false>(texels, tables, inner + inset, outer - inset, false, false, error);
    }
}

__device__ __forceinline__ uint32_t bc4_value(float texel)
{
    float const s = fminf(fmaxf(texel, 0.f), 1.f);           // saturate: a NaN becomes 0
    return uint32_t(rintf(s * 255.f));
}

// What the searches ask of a block, from its rows.
__device__ __forceinline__ void bc4_prepare(Bc4Texels& texels)
{
    texels.squares = 0;
    u16x2 lo = u16x2(uint16_t(255)), hi = u16x2(uint16_t(0));
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        texels.even[r] = __builtin_bit_cast(u16x2, texels.rows[r] & 0x00ff00ffu);
        texels.odd[r] = __builtin_bit_cast(u16x2, (texels.rows[r] >> 8) & 0x00ff00ffu);
        lo = __builtin_elementwise_min(lo, __builtin_elementwise_min(texels.even[r], texels.odd[r]));
        hi = __builtin_elementwise_max(hi, __builtin_elementwise_max(texels.even[r], texels.odd[r]));
        texels.squares = __builtin_amdgcn_udot4(texels.rows[r], texels.rows[r], texels.squares, false);
    }
    texels.lo = min(lo[0], lo[1]); texels.hi = max(hi[0], hi[1]);
}

// Channel `c` of the sixteen texels of block (bx, by), as 8-bit values.
__device__ __forceinline__ void bc4_load(BlockCompressArgs const& a, int bx, int by, int c, Bc4Texels& texels)
{
    int const x0 = a.srcLeft + bx * 4, y0 = a.srcTop + by * 4;
    if (a.packedRows && x0 + 4 <= a.srcWidth && y0 + 4 <= a.srcHeight) {
        // UNORM8 pixels without padding, the whole block inside the image: a row of four is four dwords at most, and
        // a code is its own value (rint(code / 255 * 255) = code).  All of them are under way before the first is looked at.
        uint8_t const* px = a.src + size_t(y0) * a.rowPitch + size_t(x0) * a.pixelStride;
        auto const row = [&](int y) { return px + size_t(y) * a.rowPitch; };
        if (a.pixelStride == 1) {                            // uniform; the image has no channel 1
#pragma unroll
            for (int y = 0; y < 4; ++y) texels.rows[y] = c == 0 ? *reinterpret_cast<u32_unaligned const*>(row(y)) : 0u;
        } else if (a.pixelStride == 2) {
            u32x2_unaligned words[4];
#pragma unroll
            for (int y = 0; y < 4; ++y) words[y] = *reinterpret_cast<u32x2_unaligned const*>(row(y));
#pragma unroll
            for (int y = 0; y < 4; ++y) texels.rows[y] = __builtin_amdgcn_perm(words[y][1], words[y][0], c == 0 ? 0x06040200u : 0x07050301u);
        } else {
            uint32_t bytes[4][4];
#pragma unroll
            for (int t = 0; t < 16; ++t) bytes[t >> 2][t & 3] = row(t >> 2)[size_t(t & 3) * a.pixelStride + size_t(c)];
#pragma unroll
            for (int y = 0; y < 4; ++y) texels.rows[y] = bytes[y][0] | bytes[y][1] << 8 | bytes[y][2] << 16 | bytes[y][3] << 24;
        }
    } else {
        float values[4][4][1];
        source_rows<1, 4>(a, x0, y0, c, values);
#pragma unroll
        for (int y = 0; y < 4; ++y)
            texels.rows[y] = bc4_value(values[y][0][0]) | bc4_value(values[y][1][0]) << 8 | bc4_value(values[y][2][0]) << 16 | bc4_value(values[y][3][0]) << 24;
    }
    bc4_prepare(texels);
}

// ---------------------------------------------------------------------------------------------
// BC1 colour blocks (BlockCompressCommon.hlsli:36-493)

// For every 8-bit value the pair of 5-bit (6-bit) endpoints (a | b << 8) whose mix (2*A + B) / 3 of
// the expanded endpoints A, B (integer division) is nearest, with 3 % of |a - b| added so that close
// endpoints win among equals; pairs are tried with b in the outer loop, a in the inner one, and the
// first best is kept.  This regenerates the reference's c_ColorMatch5bit / c_ColorMatch6bit
// (hlsli:40-78), the single-colour tables of NVTT.
__device__ uint16_t g_match5[256];
__device__ uint16_t g_match6[256];

__device__ __forceinline__ uint32_t nearest_pair(int value, int bits)
{
    int const n = 1 << bits;
    int best = 0x7fffffff;
    uint32_t pick = 0;
    for (int b = 0; b < n; ++b)
        for (int a = 0; a < n; ++a) {
            int const A = bits == 5 ? (a << 3) | (a >> 2) : (a << 2) | (a >> 4);
            int const B = bits == 5 ? (b << 3) | (b >> 2) : (b << 2) | (b >> 4);
            int const cost = abs((2 * A + B) / 3 - value) * 100 + abs(a - b) * 3;
            if (cost < best) { best = cost; pick = uint32_t(a) | (uint32_t(b) << 8); }
        }
    return pick;
}

struct Rgb { float r, g, b; };
struct Rgba { float r, g, b, a; };

__device__ __forceinline__ float saturate(float v) { return __builtin_amdgcn_fmed3f(v, 0.f, 1.f); }      // a NaN becomes 0
__device__ __forceinline__ Rgb rgb_of(Rgba const& p) { return Rgb{ p.r, p.g, p.b }; }
__device__ __forceinline__ float distance2(Rgb const& a, Rgb const& b)
{
    float const dr = a.r - b.r, dg = a.g - b.g, db = a.b - b.b;
    return dr * dr + dg * dg + db * db;
}
__device__ __forceinline__ Rgb mix(Rgb const& a, Rgb const& b, float t)
{
    return Rgb{ a.r + (b.r - a.r) * t, a.g + (b.g - a.g) * t, a.b + (b.b - a.b) * t };
}
// k / 31 and k / 63: the product with the reciprocal, corrected by its remainder, is the correctly rounded quotient for
// every k below 64.
__device__ __forceinline__ float code_quotient(float k, float d, float r)
{
    float const q = k * r;
    return __builtin_fmaf(__builtin_fmaf(-q, d, k), r, q);
}
__device__ __forceinline__ Rgb of_codes(uint32_t r, uint32_t g, uint32_t b)
{
    return Rgb{ code_quotient(float(r), 31.f, 1.f / 31.f), code_quotient(float(g), 63.f, 1.f / 63.f), code_quotient(float(b), 31.f, 1.f / 31.f) };
}
__device__ __forceinline__ Rgb expand565(uint32_t w) { return of_codes((w >> 11) & 31u, (w >> 5) & 63u, w & 31u); }
__device__ __forceinline__ Rgb round565(Rgb const& v, uint32_t& w)
{
    uint32_t const r = uint32_t(rintf(saturate(v.r) * 31.f)), g = uint32_t(rintf(saturate(v.g) * 63.f)), b = uint32_t(rintf(saturate(v.b) * 31.f));
    w = (r << 11) | (g << 5) | b;
    return of_codes(r, g, b);
}

// Of four distances the smallest; pairs (0, 1) and (2, 3) are compared first, ties go to the later
// pair and, inside a pair, to its second member (hlsli:116-144).
__device__ __forceinline__ uint32_t nearest_of_four(float d0, float d1, float d2, float d3, float& error)
{
    bool const first = d0 < d1, third = d2 < d3, earlier = min_f32(d0, d1) < min_f32(d2, d3);
    float const e01 = first ? d0 : d1, e23 = third ? d2 : d3;
    uint32_t const k01 = first ? 0u : 1u, k23 = third ? 2u : 3u;
    error = earlier ? e01 : e23;
    return earlier ? k01 : k23;
}

// Palette index of a texel in four-colour mode: entries hi, lo, 1/3 and 2/3 of the way from hi to lo.  OPAQUE: the texel's
// alpha is 1, and 0 need not be added to its distances.
template <bool OPAQUE>
__device__ __forceinline__ uint32_t index_of_four(Rgba const& p, Rgb const& hi, Rgb const& lo, float& error)
{
    Rgb const c = rgb_of(p), third = mix(hi, lo, 1.f / 3.f), twoThirds = mix(hi, lo, 2.f / 3.f);
    if constexpr (OPAQUE) return nearest_of_four(distance2(hi, c), distance2(lo, c), distance2(third, c), distance2(twoThirds, c), error);
    float const alphaTerm = (1.f - p.a) * (1.f - p.a);
    return nearest_of_four(distance2(hi, c) + alphaTerm, distance2(lo, c) + alphaTerm,
                           distance2(third, c) + alphaTerm, distance2(twoThirds, c) + alphaTerm, error);
}

// Three-colour mode: entries hi, lo, their midpoint and transparent black; texels at or below the
// alpha threshold take the last at no cost.
__device__ __forceinline__ uint32_t index_of_three(Rgba const& p, Rgb const& hi, Rgb const& lo, float alphaThreshold, float& error)
{
    if (p.a <= alphaThreshold) { error = 0.f; return 3; }
    Rgb const c = rgb_of(p), middle = mix(hi, lo, 0.5f);
    float const alphaTerm = (1.f - p.a) * (1.f - p.a);
    return nearest_of_four(distance2(hi, c) + alphaTerm, distance2(lo, c) + alphaTerm, distance2(middle, c) + alphaTerm,
                           p.r * p.r + p.g * p.g + p.b * p.b + p.a * p.a, error);
}

struct ColorBlock { uint32_t endpoints, indices; float error; };

__device__ __forceinline__ uint32_t table_index(float mean)     // values outside [0, 1] use the table's ends (the reference reads outside its table there)
{
    return uint32_t(fminf(fmaxf(rintf(mean * 255.f), 0.f), 255.f));
}

__device__ __forceinline__ ColorBlock bc1_single_color(Rgba const (&px)[16])
{
    Rgb sum{ 0.f, 0.f, 0.f };
#pragma unroll
    for (int t = 0; t < 16; ++t) { sum.r += px[t].r; sum.g += px[t].g; sum.b += px[t].b; }
    uint32_t const mr = g_match5[table_index(sum.r / 16.f)], mg = g_match6[table_index(sum.g / 16.f)], mb = g_match5[table_index(sum.b / 16.f)];
    uint32_t const c0 = ((mr & 31u) << 11) | ((mg & 63u) << 5) | (mb & 31u);
    uint32_t const c1 = (((mr >> 8) & 31u) << 11) | (((mg >> 8) & 63u) << 5) | ((mb >> 8) & 31u);
    ColorBlock out;
    // c0 carries weight 2/3: index 3 when the larger word has to come first (four-colour mode), else index 2
    if (c0 < c1) { out.endpoints = (c0 << 16) | c1; out.indices = 0xffffffffu; }
    else         { out.endpoints = (c1 << 16) | c0; out.indices = 0xaaaaaaaau; }
    Rgb const shown = mix(expand565(c0), expand565(c1), 1.f / 3.f);
    out.error = 0.f;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        float const dr = px[t].r - shown.r, dg = px[t].g - shown.g, db = px[t].b - shown.b, da = px[t].a - 1.f;
        out.error += dr * dr + dg * dg + db * db + da * da;
    }
    return out;
}

// Bounding box of the texels that take part, its corners paired along the block's main direction:
// with red (or, if red is constant, green) as the axis, the other components' ends are swapped where
// their covariance with the axis is negative.  Then both ends move inwards by extent / divisor.
struct Box { Rgb lo, hi; };
__device__ __forceinline__ void orient_and_inset(Box& box, float covRG, float covRB, float covGB, float divisor)
{
    if (box.lo.r != box.hi.r) {
        if (covRG < 0.f) { float const t = box.lo.g; box.lo.g = box.hi.g; box.hi.g = t; }
        if (covRB < 0.f) { float const t = box.lo.b; box.lo.b = box.hi.b; box.hi.b = t; }
    } else if (box.lo.g != box.hi.g) {
        if (covGB < 0.f) { float const t = box.lo.b; box.lo.b = box.hi.b; box.hi.b = t; }
    }
    Rgb const inset{ (box.hi.r - box.lo.r) / divisor, (box.hi.g - box.lo.g) / divisor, (box.hi.b - box.lo.b) / divisor };
    box.hi = Rgb{ saturate(box.hi.r - inset.r), saturate(box.hi.g - inset.g), saturate(box.hi.b - inset.b) };
    box.lo = Rgb{ saturate(box.lo.r + inset.r), saturate(box.lo.g + inset.g), saturate(box.lo.b + inset.b) };
}

// Sums of the least-squares problem "texel = alpha * A + beta * B".
struct Fit {
    float aa = 0.f, bb = 0.f, ab = 0.f;
    Rgb ax{ 0.f, 0.f, 0.f }, bx{ 0.f, 0.f, 0.f };
    __device__ __forceinline__ void add(float beta, Rgba const& p)
    {
        float const alpha = 1.f - beta;
        aa += alpha * alpha; bb += beta * beta; ab += alpha * beta;
        ax.r += alpha * p.r; ax.g += alpha * p.g; ax.b += alpha * p.b;
        bx.r += beta * p.r;  bx.g += beta * p.g;  bx.b += beta * p.b;
    }
    // false when the system is (nearly) singular
    __device__ __forceinline__ bool solve(Rgb& A, Rgb& B) const
    {
        float const det = aa * bb - ab * ab;
        if (!(fabsf(det) > 0.0001f)) return false;
        float const factor = 1.f / det;
        A = Rgb{ (ax.r * bb - bx.r * ab) * factor, (ax.g * bb - bx.g * ab) * factor, (ax.b * bb - bx.b * ab) * factor };
        B = Rgb{ (bx.r * aa - ax.r * ab) * factor, (bx.g * aa - ax.g * ab) * factor, (bx.b * aa - ax.b * ab) * factor };
        return true;
    }
};
// An endpoint component that sits exactly on 0 or 1 stays there.
__device__ __forceinline__ float unless_pinned(float current, float fitted) { return (current == 0.f || current == 1.f) ? current : saturate(fitted); }
__device__ __forceinline__ Rgb unless_pinned(Rgb const& current, Rgb const& fitted)
{
    return Rgb{ unless_pinned(current.r, fitted.r), unless_pinned(current.g, fitted.g), unless_pinned(current.b, fitted.b) };
}

template <bool OPAQUE>
__device__ __forceinline__ ColorBlock bc1_four_colors(Rgba const (&px)[16])
{
    Rgb sum{ 0.f, 0.f, 0.f };
    Box box{ Rgb{ 1.f, 1.f, 1.f }, Rgb{ 0.f, 0.f, 0.f } };
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        sum.r += px[t].r; sum.g += px[t].g; sum.b += px[t].b;
        box.lo = Rgb{ min_f32(box.lo.r, px[t].r), min_f32(box.lo.g, px[t].g), min_f32(box.lo.b, px[t].b) };
        box.hi = Rgb{ max_f32(box.hi.r, px[t].r), max_f32(box.hi.g, px[t].g), max_f32(box.hi.b, px[t].b) };
    }
    Rgb const center{ sum.r / 16.f, sum.g / 16.f, sum.b / 16.f };
    float covRG = 0.f, covRB = 0.f, covGB = 0.f;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        float const r = px[t].r - center.r, g = px[t].g - center.g, b = px[t].b - center.b;
        covRG += r * g; covRB += r * b; covGB += g * b;
    }
    orient_and_inset(box, covRG, covRB, covGB, 16.f);

    uint32_t c0 = 0, c1 = 0;
#pragma unroll 1
    for (int round = 0; round < 4; ++round) {
        Fit fit;
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            float unused;
            uint32_t const k = index_of_four<OPAQUE>(px[t], box.hi, box.lo, unused);
            // (selected, not divided: 1/3 and 2/3 rounded)
            fit.add((k & 2u) ? ((k & 1u) ? 2.f / 3.f : 1.f / 3.f) : float(k & 1u), px[t]);
        }
        Rgb A, B;
        if (fit.solve(A, B)) {
            box.lo = unless_pinned(box.lo, B);
            box.hi = unless_pinned(box.hi, A);
        }
        uint32_t n0, n1;
        box.hi = round565(box.hi, n0);
        box.lo = round565(box.lo, n1);
        if (n0 == c0 && n1 == c1) break;
        c0 = n0; c1 = n1;
    }
    // the first word must be the larger one, or a decoder takes the block for three-colour mode
    if (c0 == c1) {
        if (c0 == 0) { c0 = 1; box.hi = expand565(c0); }
        else         { c1 = c0 - 1; box.lo = expand565(c1); }
    } else if (c0 < c1) {
        Rgb const t = box.hi; box.hi = box.lo; box.lo = t;
        uint32_t const w = c0; c0 = c1; c1 = w;
    }
    ColorBlock out{ (c1 << 16) | c0, 0u, 0.f };
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        float e;
        out.indices |= index_of_four<OPAQUE>(px[t], box.hi, box.lo, e) << (2 * t);
        out.error += e;
    }
    return out;
}

__device__ __forceinline__ ColorBlock bc1_three_colors(Rgba const (&px)[16], float alphaThreshold)
{
    Rgb sum{ 0.f, 0.f, 0.f };
    Box box{ Rgb{ 1.f, 1.f, 1.f }, Rgb{ 0.f, 0.f, 0.f } };
    int opaque = 0;
#pragma unroll
    for (int t = 0; t < 16; ++t)
        if (!(px[t].a <= alphaThreshold)) {
            sum.r += px[t].r; sum.g += px[t].g; sum.b += px[t].b;
            box.lo = Rgb{ min_f32(box.lo.r, px[t].r), min_f32(box.lo.g, px[t].g), min_f32(box.lo.b, px[t].b) };
            box.hi = Rgb{ max_f32(box.hi.r, px[t].r), max_f32(box.hi.g, px[t].g), max_f32(box.hi.b, px[t].b) };
            ++opaque;
        }
    float const count = float(opaque);
    Rgb const center = opaque > 0 ? Rgb{ sum.r / count, sum.g / count, sum.b / count } : Rgb{ 0.f, 0.f, 0.f };
    float covRG = 0.f, covRB = 0.f, covGB = 0.f;
#pragma unroll
    for (int t = 0; t < 16; ++t)
        if (!(px[t].a <= alphaThreshold)) {
            float const r = px[t].r - center.r, g = px[t].g - center.g, b = px[t].b - center.b;
            covRG += r * g; covRB += r * b; covGB += g * b;
        }
    orient_and_inset(box, covRG, covRB, covGB, count);      // no opaque texel: -1 / 0, the ends saturate to hi = 1, lo = 0

    Fit fit;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        float unused;
        uint32_t const k = index_of_three(px[t], box.hi, box.lo, alphaThreshold, unused);
        if (k != 3) fit.add((k & 2u) ? 0.5f : float(k & 1u), px[t]);
    }
    Rgb A, B;
    if (fit.solve(A, B)) {
        // as in the reference (hlsli:453-455): the solution for the entry-0 end goes to `lo` and vice versa
        box.lo = unless_pinned(box.lo, A);
        box.hi = unless_pinned(box.hi, B);
    }
    uint32_t c0, c1;
    box.hi = round565(box.hi, c0);
    box.lo = round565(box.lo, c1);
    if (c0 > c1) {              // first word <= second word selects three-colour mode
        Rgb const t = box.hi; box.hi = box.lo; box.lo = t;
        uint32_t const w = c0; c0 = c1; c1 = w;
    }
    ColorBlock out{ (c1 << 16) | c0, 0u, 0.f };
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        float e;
        out.indices |= index_of_three(px[t], box.hi, box.lo, alphaThreshold, e) << (2 * t);
        out.error += e;         // 0 for transparent texels
    }
    return out;
}

// The candidates without rounds of refinement: one colour and (BC1) all transparent.
template <bool TRANSPARENT>
__device__ __forceinline__ ColorBlock bc1_simple_candidates(Rgba const (&px)[16], float alphaThreshold)
{
    ColorBlock best = bc1_single_color(px);
    if constexpr (TRANSPARENT) {
        float transparentError = 0.f;
#pragma unroll
        for (int t = 0; t < 16; ++t)
            if (!(px[t].a <= alphaThreshold)) transparentError += px[t].r * px[t].r + px[t].g * px[t].g + px[t].b * px[t].b + px[t].a * px[t].a;
        if (!(best.error < transparentError)) best = ColorBlock{ 0u, 0xffffffffu, transparentError };
    }
    return best;
}

// BC2 alpha: 4 bits per texel, texel 0 in the lowest bits.
__device__ __forceinline__ uint64_t bc2_alpha(float const (&alpha)[16])
{
    uint64_t bits = 0;
#pragma unroll
    for (int t = 0; t < 16; ++t) bits |= uint64_t(uint32_t(rintf(saturate(alpha[t]) * 15.f))) << (4 * t);
    return bits;
}

} // namespace

// A wave encodes one channel of 64 blocks (16 x 4) with one palette, so that the palettes' refinements, each a chain of
// up to nine passes over the texels, run side by side and not one after the other: a workgroup is the two palettes of
// both channels of 64 blocks (BC5) or of one channel of 128 (BC4).  The waves of the six-value palette leave their
// candidates in LDS for those of the eight-value one to choose from.  Bound by vector issue: 870 instructions a wave, two
// thirds of them the refits and passes of the few lanes that go on longest.  2048 x 2048: BC5 29.4 us, BC4 17.9 (57.7 and 34 with
// the distances to all eight entries and float sums for every refit, 2 200 instructions a wave); 64 x 64: 6.5 us each (8.6).
// Six, seven or eight waves per SIMD instead of five, with fewer registers, measure the same or 1 us more.
template <int CHANNELS>
__global__ void __launch_bounds__(256)
bc4_compress_kernel(BlockCompressArgs a)
{
    __shared__ Bc4Tables tables;
    __shared__ uint64_t candidates[2][64];
    __shared__ uint32_t errors[2][64];
    int const wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63, pair = wave >> 1;
    int const bx = blockIdx.x * 16 + (lane & 15), by = (CHANNELS == 1 ? blockIdx.y * 8 + pair * 4 : blockIdx.y * 4) + (lane >> 4);
    bool const inside = bx < a.widthInBlocks && by < a.heightInBlocks;
    int const channel = CHANNELS == 1 ? 0 : pair;
    bool const eight = (wave & 1) == 0;
    Bc4Texels texels;
    bc4_stage(tables, 256);
    if (inside) bc4_load(a, bx, by, channel, texels);
    __syncthreads();
    uint64_t mine = 0;
    uint32_t error = 0;
    if (inside) {
        if (eight) {
            mine = bc4_bits<true>(bc4_candidate<true>(texels, tables, error));
        } else {
            candidates[pair][lane] = bc4_bits<false>(bc4_candidate<false>(texels, tables, error));
            errors[pair][lane] = error;
        }
    }
    __syncthreads();
    if (!inside || !eight) return;
    if (errors[pair][lane] < error) mine = candidates[pair][lane];
    reinterpret_cast<uint64_t*>(a.dst + size_t(by + a.dstOffsetY) * a.dstRowPitch)[size_t(bx + a.dstOffsetX) * CHANNELS + channel] = mine;
}

// BC1 (8 bytes per block), BC2 and BC3 (alpha block, then colour block), bound by vector instructions: a block's
// candidates are chains of passes over its texels.
//
// bc1_compress_split_kernel: the waves of a workgroup encode the same 64 blocks (16 x 4), a candidate each, and leave what
// they found in LDS for the first to choose from: that one refines the four-colour endpoints, up to five passes and the
// longest by far; the second takes the simple candidates and, BC1, the three-colour one, BC2, the alpha, BC3, the
// six-value alpha palette; BC3's third wave the eight-value one.  A wave waits for the first one's end, so this is for
// images that do not fill the device anyway.
// bc1_compress_kernel: a lane per block, all candidates one after the other.
//
// 64 x 64 and 1024 x 1024: BC1 27 and 29 us in one lane before, 15 and 16 split; BC2 19 and 20, 15 and 15; BC3 25 and 33,
// 15 and 19.  2048 x 2048: BC1 58 before, 51 (two waves per SIMD with everything in registers; 82 with three that spill; 55
// split), 46.5 with all pixels loaded at once; BC2 38, 34 (47 split), 31.6; BC3 61, 52 (72 split), 40.5 with the alpha search in
// integers, 33 with it behind the colours and nothing spilled (with hard edges in alpha 50 before, 53 and 36).  Thirds are selected
// and not divided, and k / 31 is a product.
struct Bc1Exchange { float4 texels[16][64]; uint32_t words[6][64]; uint64_t alpha[64]; uint32_t sixError[64]; };
struct NoTables {};
template <int FORMAT> using Bc1Tables = std::conditional_t<FORMAT == 3, Bc4Tables, NoTables>;          // of the alpha search
template <int FORMAT> constexpr int kBc1Waves = FORMAT == 3 ? 3 : 2;

template <int FORMAT>
__device__ __forceinline__ ColorBlock bc1_refined_candidate(Rgba const (&px)[16])
{
    if constexpr (FORMAT != 1) return bc1_four_colors<true>(px);
    bool opaque = true;
#pragma unroll
    for (int t = 0; t < 16; ++t) opaque = opaque && px[t].a == 1.f;
    return __all(opaque) ? bc1_four_colors<true>(px) : bc1_four_colors<false>(px);     // (of the active lanes)
}

// The colour word, and in front of it the alpha word of BC2 and BC3.
template <int FORMAT>
__device__ __forceinline__ uint64_t* bc1_place(BlockCompressArgs const& a, int bx, int by)
{
    constexpr int WORDS = FORMAT == 1 ? 1 : 2;
    return reinterpret_cast<uint64_t*>(a.dst + size_t(by + a.dstOffsetY) * a.dstRowPitch) + size_t(bx + a.dstOffsetX) * WORDS;
}

template <int FORMAT>
__global__ void __launch_bounds__(64 * kBc1Waves<FORMAT>) __attribute__((amdgpu_waves_per_eu(4)))
bc1_compress_split_kernel(BlockCompressArgs a)
{
    __shared__ Bc1Exchange exchange;
    __shared__ Bc1Tables<FORMAT> tables;
    if constexpr (FORMAT == 3) bc4_stage(tables, 64 * kBc1Waves<FORMAT>);
    int const wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
    int const bx = blockIdx.x * 16 + (lane & 15), by = blockIdx.y * 4 + (lane >> 4);
    bool const inside = bx < a.widthInBlocks && by < a.heightInBlocks;
    int const x0 = a.srcLeft + bx * 4, y0 = a.srcTop + by * 4;
    if (inside) {
        auto const store = [&](int t, auto packed) {
            float c[4];
            if constexpr (decltype(packed)::value) source_packed_pixel(a, x0 + (t & 3), y0 + (t >> 2), c);
            else                                   source_pixel(a, x0 + (t & 3), y0 + (t >> 2), c);
            exchange.texels[t][lane] = make_float4(c[0], c[1], c[2], c[3]);
        };
        if (a.packedRgba8) {                                 // uniform: one load a texel, all in flight
#pragma unroll
            for (int k = 0; k < (16 + kBc1Waves<FORMAT> - 1) / kBc1Waves<FORMAT>; ++k)
                if (wave + k * kBc1Waves<FORMAT> < 16) store(wave + k * kBc1Waves<FORMAT>, std::true_type{});
        } else {
#pragma unroll 2
            for (int t = wave; t < 16; t += kBc1Waves<FORMAT>) store(t, std::false_type{});
        }
    }
    __syncthreads();
    auto const alpha_candidate = [&](auto eight, auto const& tables, uint32_t& error) {
        Bc4Texels texels;
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            texels.rows[y] = 0;
#pragma unroll
            for (int x = 0; x < 4; ++x) texels.rows[y] |= bc4_value(exchange.texels[4 * y + x][lane].w) << (8 * x);
        }
        bc4_prepare(texels);
        return bc4_bits<decltype(eight)::value>(bc4_candidate<decltype(eight)::value>(texels, tables, error));
    };
    ColorBlock best{ 0u, 0u, 0.f };
    uint64_t alphaBlock = 0;
    uint32_t alphaError = 0;
    if (inside) {
        if (wave == 2) {
            if constexpr (FORMAT == 3) alphaBlock = alpha_candidate(std::true_type{}, tables, alphaError);
        } else {
            Rgba px[16];
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                float4 const v = exchange.texels[t][lane];
                px[t] = Rgba{ v.x, v.y, v.z, FORMAT == 1 ? v.w : 1.f };
            }
            if (wave == 0) {
                best = bc1_refined_candidate<FORMAT>(px);
            } else {
                ColorBlock const simple = bc1_simple_candidates<FORMAT == 1>(px, a.alphaThreshold);
                exchange.words[0][lane] = simple.endpoints; exchange.words[1][lane] = simple.indices; exchange.words[2][lane] = __float_as_uint(simple.error);
                if constexpr (FORMAT == 1) {
                    ColorBlock const three = bc1_three_colors(px, a.alphaThreshold);
                    exchange.words[3][lane] = three.endpoints; exchange.words[4][lane] = three.indices; exchange.words[5][lane] = __float_as_uint(three.error);
                } else if constexpr (FORMAT == 2) {
                    float alpha[16];
#pragma unroll
                    for (int t = 0; t < 16; ++t) alpha[t] = exchange.texels[t][lane].w;
                    exchange.alpha[lane] = bc2_alpha(alpha);
                } else {
                    exchange.alpha[lane] = alpha_candidate(std::false_type{}, tables, alphaError);
                    exchange.sixError[lane] = alphaError;
                }
            }
        }
    }
    __syncthreads();
    if (!inside || wave == 1) return;
    uint64_t* const dst = bc1_place<FORMAT>(a, bx, by);
    if (wave == 2) {
        dst[0] = exchange.sixError[lane] < alphaError ? exchange.alpha[lane] : alphaBlock;
        return;
    }
    ColorBlock chosen{ exchange.words[0][lane], exchange.words[1][lane], __uint_as_float(exchange.words[2][lane]) };
    if (best.error < chosen.error) chosen = best;
    if constexpr (FORMAT == 1) {
        float const error = __uint_as_float(exchange.words[5][lane]);
        if (error < chosen.error) chosen = ColorBlock{ exchange.words[3][lane], exchange.words[4][lane], error };
    }
    uint64_t const color = uint64_t(chosen.endpoints) | (uint64_t(chosen.indices) << 32);
    if constexpr (FORMAT == 1) {
        dst[0] = color;
    } else {
        if constexpr (FORMAT == 2) dst[0] = exchange.alpha[lane];
        dst[1] = color;
    }
}

template <int FORMAT>
__global__ void __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(FORMAT == 1 ? 2 : 4)))
bc1_compress_kernel(BlockCompressArgs a)
{
    int const bx = blockIdx.x * 16 + (threadIdx.x & 15), by = blockIdx.y * 8 + (threadIdx.x >> 4);
    __shared__ Bc1Tables<FORMAT> tables;
    if constexpr (FORMAT == 3) {
        bc4_stage(tables, 128);
        __syncthreads();
    }
    if (bx >= a.widthInBlocks || by >= a.heightInBlocks) return;
    Rgba px[16];
    float alpha[16];
    float texels[4][4][4];
    source_rows<4, 4>(a, a.srcLeft + bx * 4, a.srcTop + by * 4, 0, texels);
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        float (&c)[4] = texels[t >> 2][t & 3];
        px[t] = Rgba{ c[0], c[1], c[2], FORMAT == 1 ? c[3] : 1.f };
        alpha[t] = c[3];
    }
    uint64_t* const dst = bc1_place<FORMAT>(a, bx, by);
    if constexpr (FORMAT == 2) dst[0] = bc2_alpha(alpha);
    uint32_t rows[4];                                        // BC3: alpha is encoded when the colours are done with
    if constexpr (FORMAT == 3) {
#pragma unroll
        for (int y = 0; y < 4; ++y)
            rows[y] = bc4_value(alpha[4 * y]) | bc4_value(alpha[4 * y + 1]) << 8 | bc4_value(alpha[4 * y + 2]) << 16 | bc4_value(alpha[4 * y + 3]) << 24;
    }
    ColorBlock best = bc1_simple_candidates<FORMAT == 1>(px, a.alphaThreshold);
    ColorBlock const four = bc1_four_colors<FORMAT != 1>(px);
    if (four.error < best.error) best = four;
    if constexpr (FORMAT == 1) {
        ColorBlock const three = bc1_three_colors(px, a.alphaThreshold);
        if (three.error < best.error) best = three;
    }
    dst[FORMAT == 1 ? 0 : 1] = uint64_t(best.endpoints) | (uint64_t(best.indices) << 32);
    if constexpr (FORMAT == 3) {
        Bc4Texels texels;
        uint32_t error8, error6;
#pragma unroll
        for (int y = 0; y < 4; ++y) texels.rows[y] = rows[y];
        bc4_prepare(texels);
        Bc4 const block8 = bc4_candidate<true>(texels, tables, error8), block6 = bc4_candidate<false>(texels, tables, error6);
        dst[0] = error6 < error8 ? bc4_bits<false>(block6) : bc4_bits<true>(block8);
    }
}

template <int FORMAT>
static void launch_bc1(BlockCompressArgs const& a, hipStream_t stream)
{
    unsigned const x = unsigned(a.widthInBlocks + 15) / 16, y = unsigned(a.heightInBlocks + 3) / 4;
    // (BC3: split 19 us with four workgroups per compute unit, 42 with eight; unsplit 29 with either)
    if (uint64_t(x) * y <= 5u * uint64_t(compute_units_of_current_device()))
        hipLaunchKernelGGL(bc1_compress_split_kernel<FORMAT>, dim3(x, y), dim3(64 * kBc1Waves<FORMAT>), 0, stream, a);
    else
        hipLaunchKernelGGL(bc1_compress_kernel<FORMAT>, dim3(x, unsigned(a.heightInBlocks + 7) / 8), dim3(128), 0, stream, a);
}

__global__ void __launch_bounds__(256)
bc1_tables_kernel()
{
    g_match5[threadIdx.x] = uint16_t(nearest_pair(int(threadIdx.x), 5));
    g_match6[threadIdx.x] = uint16_t(nearest_pair(int(threadIdx.x), 6));
}

hipError_t launch_color_tables(hipStream_t stream)
{
    hipLaunchKernelGGL(bc1_tables_kernel, dim3(1), dim3(256), 0, stream);
    return hipGetLastError();
}

hipError_t launch_block_compress(BlockCompressArgs const& a, int dstFormat, hipStream_t stream)
{
    dim3 const grid((a.widthInBlocks + 15) / 16, (a.heightInBlocks + 3) / 4);
    switch (dstFormat) {
    case 1: launch_bc1<1>(a, stream); break;
    case 2: launch_bc1<2>(a, stream); break;
    case 3: launch_bc1<3>(a, stream); break;
    case 4: hipLaunchKernelGGL(bc4_compress_kernel<1>, dim3(grid.x, (a.heightInBlocks + 7) / 8), dim3(256), 0, stream, a); break;
    case 5: hipLaunchKernelGGL(bc4_compress_kernel<2>, grid, dim3(256), 0, stream, a); break;
    case 6: return launch_bc6_compress(a, stream);
    case 7: return launch_bc7_compress(a, stream);
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

} // namespace ntc_hip_dev
