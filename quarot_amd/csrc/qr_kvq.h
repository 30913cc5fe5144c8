// Asymmetric int4 quantiser of the KV cache (quarot/transformers/kv_cache.py:10-33): the code forms shared by kv.hip
// and attn.hip, and the quantiser of ONE 128-wide vector by one wave, for kernels that quantise the vector they are
// about to use.
#pragma once
#include "qr_paged.h"

// Eight codes clamp(round_half_even(fp16(fp16(x + zero) / scale)), 0, 15) for all-finite input: the
// add is one packed fp16 add, the division the one-multiplication form of sym_codes8_fast (the
// shifted value is an fp16 number like any other), the rounding the +1536 trick.
// CLAMP = false leaves the clamp out: the shifted values lie in [0, range] by construction, so with a
// scale that is a NORMAL fp16 number (relative rounding error <= 2^-11: range >= 2^-10 is enough) the
// quotient is at most 15 (1 + 2^-11) and rounds to 15 at most.  A subnormal scale can be off by several
// per cent and needs the clamp (range / 15 = 10.5 units of 2^-24 -> scale 10 units -> quotient 15.75).
// A pair's two codes come as the low nibbles of the halves of a word.
template <bool CLAMP>
__device__ __forceinline__ u32 asym_pair_fast(u32 v, f16x2 zero, FastRecip f) {
    const f16x2 sh = as_f16x2(v) + zero;
    // the quotient straight from the packed pair to the packed fp16 quotient (one mixed-precision instruction per
    // value; see sym_pair_fast for why its single rounding is still the correctly rounded division), then + 1536
    f16x2 h = {(f16)__builtin_fmaf((float)sh[0], f.r, 0.0f), (f16)__builtin_fmaf((float)sh[1], f.r, 0.0f)};
    h = h + f16x2{(f16)1536.0f, (f16)1536.0f};
    if (!CLAMP) return __builtin_bit_cast(u32, h);
    // on the bit patterns: 1536 + code in [1536, 1551] is 0x6600 .. 0x660f; patterns of positive halves order
    // like signed 16-bit integers, negative sums are negative integers, +inf (0x7c00) lies above
    typedef short i16x2 __attribute__((ext_vector_type(2)));
    i16x2 c = __builtin_bit_cast(i16x2, h);
    c = __builtin_elementwise_max(c, i16x2{0x6600, 0x6600});
    c = __builtin_elementwise_min(c, i16x2{0x660f, 0x660f});
    return __builtin_bit_cast(u32, c);
}
template <bool CLAMP = true>
__device__ __forceinline__ u32 asym_codes8_fast(u32x4 v, f16 zero, FastRecip f) {
    u32 b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) b[i] = asym_pair_fast<CLAMP>(v[i], f16x2{zero, zero}, f);
    return pack_nibbles8(b);
}
// A vector's minimum decides the sign of a zero `zero` (= -min): a vector that holds both zeros must give the same one in
// every kernel, whatever the order of its reduction.  All minima of the quantisers are therefore taken with the
// hardware's minimum instructions, for which -0 is below +0 (a comparison and a selection returns whichever of two
// zeros stands second): -0.0 if the vector holds one, and +0.0 -- hence zero = -0.0, as -min gives -- if all its zeros are +0.0.
__device__ __forceinline__ f16 min_of_pair(f16x2 v) { return __builtin_fminf16(v[0], v[1]); }
// ranges from which the clamp-free form is exact (see above)
__device__ __forceinline__ bool asym_range_normal(f16 rng) { return rng >= (f16)0.0009765625f; }

// One fp16 vector of 128 values through (had) H_128 * hscale and the asymmetric int4 quantiser, by ONE wave, a pair of values per
// lane, with the arithmetic of kv_had128_kernel operation for operation: codes and parameters are the bits that kernel writes for the
// vector.  The transform is that kernel's matrix instructions on its operand layout, where the 32 columns of the second operand are 32
// vectors and four accumulators hold the four quarters of the results, which differ by the signs that the first operand takes.  Here
// eight columns each are one quarter, the vector with those signs on it (a product's bits do not say which factor was negative): eight
// matrix instructions instead of 32, and sixteen results in a lane, of which it takes two.  What bounds it is the chain of one wave, and
// the instruction cache that a launch finds cold: with all 128 results in every lane it was 2.5 us and 32 KB of code of a decode step's launch,
// now 1.5 us, mostly under the latency of the walk's first loads (1 x 2048 x 32 heads 9.3 -> 8.8 us, 40 x 438 x 40 29.3 -> 26.6).
// `piece`: the vector's 16-byte piece number lane % 16 (the caller's load, so that it can be in flight early); `stage`: 256 bytes of LDS
// private to the wave.
struct OneVector {
    u32 at, byte;       // which byte of the vector's 64 this lane has (values 2 at, 2 at + 1), and the byte
    f16 sc, zp;         // in every lane
};
template <int CTRL>
__device__ __forceinline__ u32 dpp_of(u32 v) { return (u32)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true); }
__device__ __forceinline__ OneVector kv_quant_one_vector(u32x4 piece, u32x4* stage, bool had, float hscale) {
    const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
    if (lane < 16) stage[lane] = piece;
    __builtin_amdgcn_wave_barrier();                               // (LDS operations of one wave execute in order)
    OneVector r;
    u32 pair;
    if (had) {
        const f16x8 ha[2] = {sylvester8(c, (c >> 3) & h), sylvester8(c, ((c >> 3) & h) ^ (c >> 4))};
        f32x16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            // quarter c / 8 of the results: rows 32 (c / 8) .. of H_128
            const u32 flip = (((c >> 3) & (ks >> 1) & 1) ^ ((c >> 4) & (ks >> 2))) ? 0x80008000u : 0u;
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ha[ks & 1], __builtin_bit_cast(f16x8, stage[2 * ks + h] ^ flip), acc, 0, 0, 0);
        }
        // acc[i]: value 32 (c / 8) + 8 (i / 4) + 4 h + i % 4; this lane's pair is number c % 8 of its eight
        // (by masks: conditions on elements of an array become an index into one in LDS, whose place takes a load from the launch's
        // packet in host memory, 4 us)
        u32 four = (c & 4) ? ~0u : 0u, two = (c & 2) ? ~0u : 0u, one = (c & 1) ? ~0u : 0u;
        asm volatile("" : "+v"(four), "+v"(two), "+v"(one));
        auto either = [](u32 mask, u32 a, u32 b) { return (mask & a) | (~mask & b); };
        u32 t[8], u[4];
#pragma unroll
        for (int i = 0; i < 8; ++i) t[i] = either(four, __builtin_bit_cast(u32, (float)acc[8 + i]), __builtin_bit_cast(u32, (float)acc[i]));
#pragma unroll
        for (int i = 0; i < 4; ++i) u[i] = either(two, t[4 + i], t[i]);
        pair = narrow_f16x2(__builtin_bit_cast(float, either(one, u[2], u[0])) * hscale, __builtin_bit_cast(float, either(one, u[3], u[1])) * hscale);
        r.at = (u32)((c >> 3) * 16 + ((c >> 1) & 3) * 4 + h * 2 + (c & 1));
    } else {
        pair = ((const u32*)stage)[lane];
        r.at = (u32)lane;
    }
    __builtin_amdgcn_wave_barrier();
    const f16x2 x = as_f16x2(pair);
    const bool bad = (pair & 0x7c00u) == 0x7c00u || (pair & 0x7c000000u) == 0x7c000000u;
    if (__builtin_amdgcn_ballot_w64(bad) == 0) {
        f16x2 pr = {min_of_pair(x), min_of_pair(-x)};               // minimum, -maximum
        auto with = [&](u32 other) { pr = __builtin_elementwise_min(pr, as_f16x2(other)); };
        auto word = [&] { return __builtin_bit_cast(u32, pr); };
        with(dpp_of<0xB1>(word()));                                 // lanes ^ 1, ^ 2, ^ 7, then 8 round a row of 16
        with(dpp_of<0x4E>(word()));
        with(dpp_of<0x141>(word()));
        with(dpp_of<0x128>(word()));
        const auto s16 = __builtin_amdgcn_permlane16_swap(word(), word(), false, false);
        pr = __builtin_elementwise_min(as_f16x2((u32)s16[0]), as_f16x2((u32)s16[1]));
        const auto s32 = __builtin_amdgcn_permlane32_swap(word(), word(), false, false);
        pr = __builtin_elementwise_min(as_f16x2((u32)s32[0]), as_f16x2((u32)s32[1]));
        const f16 mn = pr[0], mx = -pr[1], floor_ = (f16)1e-5f;
        f16 rng = narrow_f16((float)mx - (float)mn);
        rng = rng < floor_ ? floor_ : rng;
        r.sc = narrow_f16((float)rng * (1.0f / 15.0f));
        r.zp = -mn;
        const u32 b = asym_pair_fast<true>(pair, f16x2{r.zp, r.zp}, make_fast_recip((float)r.sc));      // (the clamp acts below asym_range_normal only)
        r.byte = (b & 15u) | ((b >> 12) & 0xf0u);
    } else {
        // a NaN anywhere in the vector makes its range, scale and zero NaN and every code 0; infinities follow the
        // IEEE operations of the reference
        const float x0 = (float)x[0], x1 = (float)x[1];
        const bool has_nan = __builtin_amdgcn_ballot_w64(x0 != x0 || x1 != x1) != 0;
        float fmn = __builtin_fminf(x0, x1), fmx = __builtin_fmaxf(x0, x1);
#pragma unroll 1
        for (int mask = 1; mask < 64; mask *= 2) {
            fmn = __builtin_fminf(fmn, __shfl_xor(fmn, mask, 64));
            fmx = __builtin_fmaxf(fmx, __shfl_xor(fmx, mask, 64));
        }
        if (has_nan) fmn = fmx = __builtin_nanf("");
        f16 rng = (f16)(fmx - fmn);
        const f16 floor_ = (f16)1e-5f;
        rng = rng < floor_ ? floor_ : rng;
        r.sc = (f16)(float)((double)(float)rng / 15.0);
        r.zp = (f16)(-fmn);
        const float s = (float)r.sc, z = (float)r.zp;
        r.byte = 0;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float sh = (float)(f16)((float)x[e] + z);
            const float q = __builtin_rintf((float)(f16)(sh / s));
            int code = (int)q;
            code = code < 0 ? 0 : (code > 15 ? 15 : code);
            code = (q != q) ? 0 : code;
            r.byte |= (u32)code << (4 * e);
        }
    }
    return r;
}
