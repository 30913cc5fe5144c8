// One row of K 2^LOG2M values through OnlineHadamard -> Quantizer by the waves of ONE workgroup, one wave per 16 rows of
// hadK and 64 columns: the two matrix stages of hadamard_m64r_kernel / hadamard_m64q_kernel (same fragments, same order of
// sums: codes and scale are the same bits), cut so that a row's latency and not a grid's throughput decides.  Shared by
// the layer of one or two tokens (mm_gemv_kernel) and by the front of a few hundred rows (hadamard_row_quant_kernel).
// A kernel calls begin, request, request_table, sylvester, stage1, table, a barrier, table_read, stage2, folds the waves' maxima, codes.
#pragma once
#include "qr_common.h"

namespace {

template <int LOG2M, int KS2, int THREADS>
struct MmRow {
    static constexpr int M_ = 1 << LOG2M, CT = M_ / 16, S1K = M_ / 32, NT = 2 * KS2, CTW = 4, HV = CT / CTW;
    static constexpr int WAVES = HV * NT;        // waves with a part of T; a kernel may have more
    static constexpr int T_BYTES = CT * NT * 64 * 8, PIECES = 256 * KS2 * KS2, TP = (PIECES + THREADS - 1) / THREADS;
    int K, lane, l16, g, tile, half, r;
    bool works, dval;
    u32x4 xr[S1K];
    u32x2 tp[TP];                                // pieces tid + i THREADS of the table, or sign words (see hadamard_m64r_kernel)
    u32 sw[KS2];
    f16x8 sb[2][2];                              // Sylvester fragments: base tile of the parity of the column tile, its negative
    f16x8 hf[KS2];
    u32x2 yv[CTW];

    __device__ __forceinline__ void begin(int K_, int wave, int lane_) {
        K = K_, lane = lane_, l16 = lane & 15, g = lane >> 4;
        tile = HV == 2 ? wave >> 1 : wave, half = HV == 2 ? wave & 1 : 0;      // 16 rows of hadK; its 64 columns
        r = tile * 16 + l16;
        works = tile * 16 < K, dval = r < K;
    }
    __device__ __forceinline__ void request(const f16* x, int64_t row) {
#pragma unroll
        for (int c = 0; c < S1K; ++c) xr[c] = *((const u32x4*)x + row * (K * (M_ / 8)) + (dval ? r * (M_ / 8) + 4 * c + g : 0));
    }
    // (a lane's own fragments, eight bytes from each of sixteen rows per load, kept the CU's address path busy for longer than the
    // row itself: the table comes as it lies in memory and is dealt out through LDS)
    __device__ __forceinline__ void request_table(const void* hadK, int signs) {
        if (signs) {
#pragma unroll
            for (int ks = 0; ks < KS2; ++ks) sw[ks] = ((const u32*)hadK)[dval ? r * KS2 + ks : 0];
        } else {
#pragma unroll
            for (int i = 0; i < TP; ++i) {
                const int at = (int)threadIdx.x + i * THREADS;
                tp[i] = ((const u32x2*)hadK)[at < K * (K >> 2) ? at : 0];
            }
        }
    }
    __device__ __forceinline__ void sylvester() {
#pragma unroll
        for (int o = 0; o < 2; ++o) {
            sb[o][0] = sylvester8(l16, (g & (l16 >> 3)) ^ ((g >> 1) & o));
            sb[o][1] = negated(sb[o][0]);
        }
    }
    // T = X . H_m for this wave's 16 rows and four column tiles, rounded to fp16 with the scale; tiles beyond K: zeros.
    // Tl: [CT][KS2][64 lanes][2 tiles], so that stage 2 reads a contraction step's fragment as 16 bytes
    __device__ __forceinline__ void stage1(u32x2* Tl, float scale) {
        if (works) {
            u32x4 af[S1K];
#pragma unroll
            for (int c = 0; c < S1K; ++c) af[c] = dval ? xr[c] : u32x4{0, 0, 0, 0};
#pragma unroll
            for (int cc = 0; cc < CTW; ++cc) {
                // the column tile is half * 4 + cc: its bits above the lowest decide the signs of the contraction's steps
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < S1K; ++c) {
                    const f16x8 a = __builtin_bit_cast(f16x8, af[c]);
                    if (HV == 2 && (c & 2)) {    // (popcount(c & (ct >> 1)) with ct >> 1 = 2 half + cc / 2)
                        const bool odd = ((__builtin_popcount(c & (cc >> 1)) + half) & 1) != 0;
                        acc = odd ? __builtin_amdgcn_mfma_f32_16x16x32_f16(a, sb[cc & 1][1], acc, 0, 0, 0)
                                  : __builtin_amdgcn_mfma_f32_16x16x32_f16(a, sb[cc & 1][0], acc, 0, 0, 0);
                    } else {
                        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, sb[cc & 1][__builtin_popcount(c & (cc >> 1)) & 1], acc, 0, 0, 0);
                    }
                }
                Tl[(((half * CTW + cc) * KS2 + (tile >> 1)) * 64 + lane) * 2 + (tile & 1)] = u32x2{narrow_f16x2(acc[0] * scale, acc[1] * scale),
                                                                        narrow_f16x2(acc[2] * scale, acc[3] * scale)};
            }
        } else if (tile < NT) {
#pragma unroll
            for (int cc = 0; cc < CTW; ++cc) Tl[(((half * CTW + cc) * KS2 + (tile >> 1)) * 64 + lane) * 2 + (tile & 1)] = u32x2{0, 0};
        }
    }
    // the table's fragments from sign words, or the table to LDS (table_read: behind the barrier), under the other waves' stage 1.  Sign words need no zeros: columns beyond K meet zeros of T, and rows
    // beyond K are kept out of the maximum and are not stored.
    __device__ __forceinline__ void table(u32x2* Hl, int signs) {
        if (signs) {
#pragma unroll
            for (int ks = 0; ks < KS2; ++ks) {
                const u32 w = sw[ks] >> (4 * g);                          // bits 0 .. 3 and 16 .. 19 are this lane's
                const u32x2 f0 = sign_halves(w), f1 = sign_halves(w >> 16);
                hf[ks] = __builtin_bit_cast(f16x8, u32x4{f0[0], f0[1], f1[0], f1[1]});
            }
        } else {
#pragma unroll
            for (int i = 0; i < TP; ++i) {
                const int at = (int)threadIdx.x + i * THREADS;
                if (at < K * (K >> 2)) Hl[at] = tp[i];
            }
        }
    }
    __device__ __forceinline__ void table_read(const u32x2* Hl, int signs) {
        if (signs) return;
#pragma unroll
        for (int ks = 0; ks < KS2; ++ks) {
            u32x4 fr;
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                const int hc = ks * 32 + hh * 16 + g * 4;
                const bool ok = dval && hc < K;
                const u32x2 v = Hl[ok ? (r * K + hc) >> 2 : 0];
                fr[hh * 2] = ok ? v[0] : 0u;
                fr[hh * 2 + 1] = ok ? v[1] : 0u;
            }
            hf[ks] = __builtin_bit_cast(f16x8, fr);
        }
    }
    // Y^T = T^T . hadK^T into registers; returns the bits of the wave's largest magnitude
    __device__ __forceinline__ u32 stage2(const u32x2* Tl) {
        float mxf = 0.f, probe = 0.f;
#pragma unroll
        for (int cc = 0; cc < CTW; ++cc) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            if (works) {
#pragma unroll
                for (int ks = 0; ks < KS2; ++ks)
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        __builtin_bit_cast(f16x8, ((const u32x4*)Tl)[((half * CTW + cc) * KS2 + ks) * 64 + lane]), hf[ks], acc, 0, 0, 0);
            }
            if (cc == 0) probe = acc[0];
            yv[cc] = u32x2{cvt_f16x2(acc[0], acc[1]), cvt_f16x2(acc[2], acc[3])};
            mxf = __builtin_fmaxf(__builtin_fmaxf(mxf, __builtin_fabsf(acc[0])), __builtin_fabsf(acc[1]));
            mxf = __builtin_fmaxf(__builtin_fmaxf(mxf, __builtin_fabsf(acc[2])), __builtin_fabsf(acc[3]));
        }
        u32 mx = dval ? f16_bits((f16)mxf) : 0u;
        if (__builtin_amdgcn_ballot_w64(mx >= 0x7c00u || probe != probe) != 0) {         // something non-finite: the exact form
            u16x2 m2 = {0, 0};
#pragma unroll
            for (int cc = 0; cc < CTW; ++cc) {
                m2 = __builtin_elementwise_max(m2, __builtin_bit_cast(u16x2, dval ? yv[cc][0] & 0x7fff7fffu : 0u));
                m2 = __builtin_elementwise_max(m2, __builtin_bit_cast(u16x2, dval ? yv[cc][1] & 0x7fff7fffu : 0u));
            }
            mx = m2[0] > m2[1] ? m2[0] : m2[1];
        }
        return wave_max_u32_dpp(mx);
    }
    // sixteen codes of the row whose largest magnitude is mx and whose scale is sp: 8 bytes that belong at place() of the row
    __device__ __forceinline__ u32x2 codes(u32 mx, float sp, float clip) {
        u32 c01, c23;
        auto codes_from = [&](auto pair) {
            u32 b0[4], b1[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                b0[w] = pair(yv[w >> 1][w & 1]);
                b1[w] = pair(yv[2 + (w >> 1)][w & 1]);
            }
            c01 = pack_nibbles8(b0);
            c23 = pack_nibbles8(b1);
        };
        if (fast_quant_ok(mx, sp)) {
            const FastRecip fq = make_fast_recip(sp);
            if (clamp_cannot_act(clip, sp)) codes_from([&](u32 w) { return sym_pair_fast<false>(w, fq); });
            else codes_from([&](u32 w) { return sym_pair_fast<true>(w, fq); });
        } else {
            const bool fs_ok = scale_fast_ok(sp);
            const float rs = fs_ok ? 1.0f / sp : 0.0f;
            c01 = sym_codes8(u32x4{yv[0][0], yv[0][1], yv[1][0], yv[1][1]}, sp, rs, fs_ok);
            c23 = sym_codes8(u32x4{yv[2][0], yv[2][1], yv[3][0], yv[3][1]}, sp, rs, fs_ok);
        }
        const auto s1 = __builtin_amdgcn_permlane32_swap(c01, c23, false, false);
        const u32 ev = __builtin_amdgcn_perm(s1[1], s1[0], 0x05040100u);
        const u32 od = __builtin_amdgcn_perm(s1[1], s1[0], 0x07060302u);
        const auto s2 = __builtin_amdgcn_permlane16_swap(ev, od, false, false);
        return u32x2{__builtin_amdgcn_perm(s2[1], s2[0], 0x05040100u), __builtin_amdgcn_perm(s2[1], s2[0], 0x07060302u)};
    }
    __device__ __forceinline__ int place() const { return r * CT + half * CTW + g; }     // of lanes with dval; 8-byte units
};

}  // namespace
