// exact_functions.hip - the kernels' shortcuts for divisions and for storing colours, against what they stand for, over
// every operand they are used on (tests/test_exact_functions.py).  Compiled together with one kernel file at a time, whose
// functions it calls: SUBJECT_COPY, SUBJECT_BC, SUBJECT_BC6 or SUBJECT_DECODE.
#if defined(SUBJECT_COPY)
#include "../rtxntc-library_amd/csrc/ntc_copy_kernel.hip"
#elif defined(SUBJECT_BC)
#include "../rtxntc-library_amd/csrc/ntc_bc_kernel.hip"
#elif defined(SUBJECT_BC6)
#include "../rtxntc-library_amd/csrc/ntc_bc6_kernel.hip"
#else
#include "../rtxntc-library_amd/csrc/ntc_decode_device.h"
#endif

using namespace ntc_hip_dev;

namespace {

struct Report { unsigned long long tried, wrong, example; };

// CHECK: number of a case -> 0 not one, 1 right, 2 wrong.  Every wave ends after its share of the cases.
template <class CHECK>
__global__ void __launch_bounds__(256) sweep_kernel(uint64_t cases, Report* report)
{
    unsigned long long tried = 0, wrong = 0, example = 0;
    for (uint64_t i = uint64_t(blockIdx.x) * 256u + threadIdx.x; i < cases; i += uint64_t(gridDim.x) * 256u) {
        int const r = CHECK::check(i);
        tried += r != 0;
        if (r == 2) { ++wrong; example = i; }
    }
    atomicAdd(&report->tried, tried);
    if (wrong) { atomicAdd(&report->wrong, wrong); report->example = example; }
}
template <class CHECK> int sweep(Report* out)
{
    Report* device = nullptr;
    hipError_t e = hipMalloc(reinterpret_cast<void**>(&device), sizeof(Report));
    if (e != hipSuccess) return int(e);
    *out = Report{};
    e = hipMemcpy(device, out, sizeof(Report), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(sweep_kernel<CHECK>, dim3(4096), dim3(256), 0, nullptr, CHECK::cases, device);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(out, device, sizeof(Report), hipMemcpyDeviceToHost);
    (void)hipFree(device);
    return int(e);
}

__device__ bool same(float a, float b) { return __float_as_uint(a) == __float_as_uint(b) || (a != a && b != b); }
__device__ int verdict(bool right) { return right ? 1 : 2; }
[[maybe_unused]] __device__ float half_of(uint32_t bits) { return float(__builtin_bit_cast(_Float16, uint16_t(bits))); }

#if defined(SUBJECT_COPY)

// encoded_half(): every float.
template <int SPACE> struct EncodedHalf {
    static constexpr uint64_t cases = uint64_t(1) << 32;
    static __device__ int check(uint64_t i)
    {
        float const v = __uint_as_float(uint32_t(i));
        uint32_t const got = encoded_half(SPACE, v), want = stored_half(encode_color_space(SPACE, v));
        return verdict(got == want);
    }
};
// divide_by_top(): every code and every offset that a draw can have.
template <int TOP> struct DivideByTop {
    static constexpr uint64_t cases = (uint64_t(1) << 23) + TOP + 1;
    static __device__ int check(uint64_t i)
    {
        float const a = i <= TOP ? float(uint32_t(i)) : __uint_as_float(uint32_t(i - TOP - 1) | 0x3f800000u) - 1.5f;
        return verdict(same(divide_by_top(a, float(TOP), 1.f / float(TOP)), a / float(TOP)));
    }
};

// put_unorm8(): every float, at a byte of its own choice.
struct PutUnorm8 {
    static constexpr uint64_t cases = uint64_t(1) << 32;
    static __device__ int check(uint64_t i)
    {
        float const v = __uint_as_float(uint32_t(i));
        uint32_t const at = uint32_t(i ^ (i >> 13)) & 3u, others = ~(0xffu << (8u * at));
        return verdict(put_unorm8(v, at, 0x93a5c7e1u & others) == ((0x93a5c7e1u & others) | unorm_code(v, 255.f) << (8u * at)));
    }
};

#elif defined(SUBJECT_BC)

// code_quotient(): five and six bits.
struct CodeQuotient {
    static constexpr uint64_t cases = 32 + 64;
    static __device__ int check(uint64_t i)
    {
        float const k = float(uint32_t(i < 32 ? i : i - 32)), d = i < 32 ? 31.f : 63.f;
        return verdict(same(code_quotient(k, d, 1.f / d), k / d));
    }
};
// bc4_palette8(): every pair of endpoints.
struct Bc4Palette {
    static constexpr uint64_t cases = 65536;
    static __device__ int check(uint64_t i)
    {
        uint32_t const e0 = uint32_t(i) >> 8, e1 = uint32_t(i) & 255u;
        uint32_t p[8];
        bc4_palette8(e0, e1, p);
        bool right = p[0] == 8u * e0 && p[1] == 8u * e1;
        for (uint32_t k = 1; k < 7; ++k) {
            uint32_t want;
            if (e0 > e1)    want = ((7 - k) * e0 + k * e1 + 3) / 7;
            else if (k < 5) want = ((5 - k) * e0 + k * e1 + 2) / 5;
            else            want = k == 5 ? 0 : 255;
            right = right && p[k + 1] == 8u * want;
        }
        return verdict(right);
    }
};

// bc4_assign(): every pair of endpoints and every value, sixteen values a block, in the search that the pair belongs to.
struct Bc4Positions {
    static constexpr uint64_t cases = 65536 * 16;
    static __device__ int check(uint64_t i)
    {
        uint32_t const e0 = uint32_t(i >> 12), e1 = uint32_t(i >> 4) & 255u, first = (uint32_t(i) & 15u) * 16u;
        Bc4Texels texels;
        for (uint32_t r = 0; r < 4; ++r) texels.rows[r] = (first + 4u * r) * 0x01010101u + 0x03020100u;
        bc4_prepare(texels);
        Bc4 got{ e0, e1, {} }, want{ e0, e1, {} };
        uint32_t const gotError = e0 > e1 ? bc4_assign<true>(texels, kBc4Tables, got) : bc4_assign<false>(texels, kBc4Tables, got);
        uint32_t const wantError = e0 > e1 ? bc4_assign_defined<true>(texels, want) : bc4_assign_defined<false>(texels, want);
        bool right = gotError == wantError;
        for (int r = 0; r < 4; ++r) right = right && got.positions[r] == want.positions[r];
        return verdict(right);
    }
};
// bc4_refit(): 2^24 blocks, smooth ones, noise and blocks of few values, whose ties the float sums decide.
struct Bc4Refit {
    static constexpr uint64_t cases = uint64_t(1) << 24;
    template <bool EIGHT> static __device__ bool same_endpoints(Bc4Texels const& texels, Bc4 block)
    {
        Bc4 got = block;
        bc4_refit<EIGHT>(texels, got, false, false);
        float e0, e1;
        bc4_solve_defined<EIGHT>(texels, block, e0, e1);
        return EIGHT ? got.e0 == uint32_t(fmaxf(e0, e1)) && got.e1 == uint32_t(fminf(e0, e1)) : got.e0 == uint32_t(e0) && got.e1 == uint32_t(e1);
    }
    static __device__ int check(uint64_t i)
    {
        uint64_t h = (i + 1) * 0x9e3779b97f4a7c15ull;
        auto const next = [&] { h ^= h >> 29; h *= 0xbf58476d1ce4e5b9ull; h ^= h >> 32; return uint32_t(h); };
        uint32_t const kind = uint32_t(i) & 3u, base = next() & 127u, pool = next();
        Bc4Texels texels;
        for (int r = 0; r < 4; ++r) {
            uint32_t const bits = next();
            texels.rows[r] = 0;
            for (int x = 0; x < 4; ++x) {
                uint32_t const b = (bits >> (8 * x)) & 255u;
                uint32_t const v = kind == 0 ? b : kind == 1 ? base + (b & 15u) + 8u * uint32_t(r + x) : kind == 2 ? (pool >> (8u * (b & 3u))) & 255u : base + (b & 31u);
                texels.rows[r] |= v << (8 * x);
            }
        }
        bc4_prepare(texels);
        uint32_t const hi = texels.hi, lo = texels.lo;
        Bc4 eight{ hi, lo, {} }, six{ lo + (hi - lo) / 8u, hi - (hi - lo) / 8u, {} };
        bc4_assign_defined<true>(texels, eight);
        bc4_assign_defined<false>(texels, six);
        return verdict(same_endpoints<true>(texels, eight) && same_endpoints<false>(texels, six));
    }
};

#elif defined(SUBJECT_BC6)

// quotient<0>(): integers below 2^17.
struct QuotientOfIntegers {
    static constexpr uint64_t cases = uint64_t(1) << 34;
    static __device__ int check(uint64_t i)
    {
        float const a = float(uint32_t(i) & 0x1ffffu), b = float(uint32_t(i >> 17));
        return b == 0.f ? 0 : verdict(same(quotient<0>(a, b), a / b));
    }
};
// quotient<0>(): the mantissas that normal_log2() reduces to.
struct QuotientOfLog2 {
    static constexpr uint64_t cases = uint64_t(1) << 25;
    static __device__ int check(uint64_t i)
    {
        float const m = __uint_as_float(0x3f000000u + uint32_t(i));
        return m < 0.70f || m > 1.42f ? 0 : verdict(same(quotient<0>(m - 1.f, m + 1.f), (m - 1.f) / (m + 1.f)));
    }
};
// corrected() by reciprocal<1>(), as Msle does it: 1 + a half over 1 + a texel of any format but FLOAT32.
struct QuotientOfMsle {
    static constexpr uint64_t kHalves = 0x7c00, kTexels = kHalves + 256 + 65536 + 65505;
    static constexpr uint64_t cases = kHalves * kTexels;
    static __device__ int check(uint64_t i)
    {
        uint32_t const texel = uint32_t(i / kHalves);
        float x;
        if (texel < kHalves)                    x = half_of(texel);
        else if (texel < kHalves + 256)         x = float(texel - uint32_t(kHalves)) / 255.f;
        else if (texel < kHalves + 256 + 65536) x = float(texel - uint32_t(kHalves + 256)) / 65535.f;
        else                                    x = float(texel - uint32_t(kHalves + 256 + 65536));
        float const a = half_of(uint32_t(i % kHalves)) + 1.f, b = x + 1.f;
        return verdict(same(corrected(a, b, reciprocal<1>(b)), a / b));
    }
};
// Msle::estimate(): the hardware's logarithm of every quotient that can occur is within 2^-21 of normal_log2(), and 0 where that is 0.
struct LogEstimate {
    static constexpr uint64_t cases = uint64_t(34) << 23;
    static __device__ int check(uint64_t i)
    {
        uint32_t const bits = ((127u - 17u) << 23) + uint32_t(i);
        float const log = normal_log2(bits, 0);
        return verdict(fabsf(__builtin_amdgcn_logf(__uint_as_float(bits)) - log) <= fabsf(log) * 0x1p-21f);
    }
};
// quantize() and the indices' places.
struct QuotientOfCodes {
    static constexpr uint64_t cases = 3 * 65536 + 64;
    static __device__ int check(uint64_t i)
    {
        if (i < 3 * 65536) {
            float const levels = i < 65536 ? 128.f : i < 2 * 65536 ? 512.f : 1024.f, a = float(uint32_t(i & 65535u)) * levels;
            return verdict(same(corrected(a, 31744.f, 1.f / 31744.f), a / 31744.f));
        }
        uint32_t const k = uint32_t(i) & 15u, kind = (uint32_t(i) >> 4) & 3u;
        float const top = (kind & 1u) ? 15.f : 7.f, a = float(k) * ((kind & 2u) ? 64.f : 1.f);
        return verdict(same(corrected(a, top, 1.f / top), a / top));
    }
};
// quotient_by(): a component over the sum or the length of three, halves of all magnitudes.  (There are 2^45 such triples;
// these are 2^30 of them.)
struct QuotientOfDiagonals {
    static constexpr uint64_t cases = uint64_t(1) << 30;
    static __device__ int check(uint64_t i)
    {
        uint64_t h = (i + 1) * 0x9e3779b97f4a7c15ull;
        h ^= h >> 29; h *= 0xbf58476d1ce4e5b9ull; h ^= h >> 32;
        float const x = half_of(uint32_t(h) % 0x7c00u), y = half_of(uint32_t(h >> 16) % 0x7c00u), z = half_of(uint32_t(h >> 32) % 0x7c00u);
        float const s = (i & 1) ? x + y + z : sqrtf(x * x + y * y + z * z);
        return verdict(same(quotient_by(x, s, reciprocal<1>(s)), x / s));
    }
};

#else

// texel_centre(): every texel of every size that a mip can have.
struct TexelCentre {
    static constexpr uint64_t cases = uint64_t(1) << 32;
    static __device__ int check(uint64_t i)
    {
        int const x = int(uint32_t(i) & 0xffffu), size = int(i >> 16) + 1;
        return x >= size ? 0 : verdict(same(texel_centre(x, size), (float(x) + 0.5f) / float(size)));
    }
};

// floors_of(): every float of [0, 256), in every place beside numbers of its neighbourhood.
struct FloorsOf {
    static constexpr uint64_t cases = 0x43800000u;
    static __device__ int check(uint64_t i)
    {
        uint32_t const bits = uint32_t(i), top = 0x437fffffu;
        float const v[4] = { __uint_as_float(bits), __uint_as_float(min(bits + 1u, top)), __uint_as_float(bits ^ (bits >= 0x80u ? 0x55u : 0u)), __uint_as_float(top - bits) };
        uint32_t expected = 0;
        for (int k = 0; k < 4; ++k) expected |= uint32_t(floorf(v[k])) << (8 * k);
        return verdict(floors_of(v[0] * 0x1p-24f, v[1] * 0x1p-24f, v[2] * 0x1p-24f, v[3] * 0x1p-24f) == expected);
    }
};

// filter4() and bilinear4() against the definition, for scattered cells and fractions: zeros, the largest below 1, few and
// many bits, products of two that are subnormal.
struct FilteredFeatures {
    static constexpr uint64_t cases = uint64_t(1) << 26;
    static __device__ uint32_t hash(uint32_t h) { h ^= h >> 16; h *= 0x7feb352du; h ^= h >> 15; h *= 0x846ca68bu; return h ^ h >> 16; }
    static __device__ float fraction(uint32_t h)
    {
        switch (h & 7u) {
        case 0: return 0.f;
        case 1: return 0x1.fffffep-1f;
        case 2: return float(h >> 28) * 0x1p-4f;
        case 3: return float(h >> 8) * 0x1p-24f * __builtin_ldexpf(1.f, -int(h >> 3 & 31u) * 4);
        default: return float(h >> 8) * 0x1p-24f;
        }
    }
    static __device__ int check(uint64_t i)
    {
        uint32_t const h = hash(uint32_t(i)), c = hash(h + 1u), e = hash(h + 2u);
        FloatAxis const x{ 0, 0, fraction(hash(h + 3u)) }, y{ 0, 0, fraction(hash(h + 4u)) };
        uint32_t const cells[4] = { c & 0xffffu, c >> 16, e & 0xffffu, e >> 16 };
        FloatTaps const taps(x, y);
        float t[4];
        filter4(taps, cells, t);
        float const dxn = 1.f - x.d, dyn = 1.f - y.d, w00 = dxn * dyn, w10 = x.d * dyn, w01 = dxn * y.d, w11 = x.d * y.d;
        uint32_t bytes = 0;
        bool right = true;
        for (int f = 0; f < 4; ++f) {
            float q[4];
            for (int k = 0; k < 4; ++k) q[k] = float((cells[k] >> (4 * f)) & 15u);
            float const s = __builtin_fmaf(w11, q[3], __builtin_fmaf(w01, q[2], __builtin_fmaf(w10, q[1], w00 * q[0])));
            right = right && (same(t[f], s) || (fabsf(s) < 0x1p-100f && fabsf(t[f] - s) < 0x1p-120f));       // (the definition's weights are subnormal there)
            bytes |= ((uint32_t(floorf(17.f * s)) + 128u) & 0xffu) << (8 * f);
        }
        return verdict(right && bilinear4(taps, cells) == bytes);
    }
};

#endif

} // namespace

extern "C" {
#if defined(SUBJECT_COPY)
int exact_encoded_half_srgb(Report* r) { return sweep<EncodedHalf<1>>(r); }
int exact_encoded_half_hlg(Report* r) { return sweep<EncodedHalf<2>>(r); }
int exact_put_unorm8(Report* r) { return sweep<PutUnorm8>(r); }
int exact_divide_by_255(Report* r) { return sweep<DivideByTop<255>>(r); }
int exact_divide_by_65535(Report* r) { return sweep<DivideByTop<65535>>(r); }
#elif defined(SUBJECT_BC)
int exact_code_quotient(Report* r) { return sweep<CodeQuotient>(r); }
int exact_bc4_palette(Report* r) { return sweep<Bc4Palette>(r); }
int exact_bc4_positions(Report* r) { return sweep<Bc4Positions>(r); }
int exact_bc4_refit(Report* r) { return sweep<Bc4Refit>(r); }
#elif defined(SUBJECT_BC6)
int exact_quotient_of_integers(Report* r) { return sweep<QuotientOfIntegers>(r); }
int exact_quotient_of_log2(Report* r) { return sweep<QuotientOfLog2>(r); }
int exact_quotient_of_msle(Report* r) { return sweep<QuotientOfMsle>(r); }
int exact_log_estimate(Report* r) { return sweep<LogEstimate>(r); }
int exact_quotient_of_codes(Report* r) { return sweep<QuotientOfCodes>(r); }
int exact_quotient_of_diagonals(Report* r) { return sweep<QuotientOfDiagonals>(r); }
#else
int exact_texel_centre(Report* r) { return sweep<TexelCentre>(r); }
int exact_floors_of(Report* r) { return sweep<FloorsOf>(r); }
int exact_filtered_features(Report* r) { return sweep<FilteredFeatures>(r); }
// (on the host: the same code as on the device)
void tiles_of_workgroup(int byDie, int totalTiles, int workgroups, int workgroup, int* range)
{
    ntc_hip_dev::TileShares const shares = ntc_hip_dev::tile_shares(totalTiles, workgroups);
    ntc_hip_dev::TileRange const t = byDie ? ntc_hip_dev::tiles_of_workgroup<true>(shares, uint32_t(workgroup)) : ntc_hip_dev::tiles_of_workgroup<false>(shares, uint32_t(workgroup));
    range[0] = t.begin; range[1] = t.end;
}
#endif
}
