// Epilogue pieces shared by the GEMM kernels: the row-contiguous store of a wave's output slab and the
// fp16 dequantisation of four accumulators of one token.
#pragma once
#include "qr_common.h"

namespace {

// Row-contiguous output of one wave's 32 x (32 NJ) fp16 slab.  In the accumulator layout a lane owns
// 4 consecutive columns of one row, so a direct store instruction would write 16-byte pieces of 32
// different rows and leave every 128-byte line to be assembled from eight partial writes in L2
// (measured: 2.6x the output bytes written to memory on outputs larger than L2).  Instead the slab
// goes through a wave-private LDS region and leaves as 16 bytes per lane with NJ*4 consecutive lanes
// covering one row segment, i.e. whole lines per instruction.
//   o[jj][gq] = this lane's columns jj*32 + gq*8 + (lane/32)*4 .. +3 of row lane%32.
//   region: 32 * NJ * 8 slots of 8 bytes; the 8-byte slot index within a row is XORed with a key made
//   from the row so that the 32 rows written by one instruction spread over all banks.
//   rows: how many of the slab's 32 rows exist in the output (the last row tile of a token count that
//   is no multiple of the tile height); the others are computed on clamped inputs and not stored.
template <int NJ>
__device__ __forceinline__ void store_slab_rows(u32x2* region, const f16x4 (&o)[NJ][4], int lane, f16* ybase, int N,
                                                int rows = 32) {
    constexpr int U = NJ * 8;                   // 8-byte slots per row
    constexpr int LPR = U / 2;                  // lanes (16 bytes each) per row on the way out
    constexpr int RPP = 64 / LPR;               // rows per store instruction
    const int r = lane & 31, khalf = lane >> 5;
#pragma unroll
    for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
        for (int gq = 0; gq < 4; ++gq) {
            const int u = jj * 8 + gq * 2 + khalf;
            region[r * U + (u ^ ((r * U / 32) & (U - 1)))] = __builtin_bit_cast(u32x2, o[jj][gq]);
        }
    const u32x4* region16 = (const u32x4*)region;
    const int s = lane % LPR;
#pragma unroll
    for (int pass = 0; pass < 32 / RPP; ++pass) {
        const int rr = lane / LPR + pass * RPP;
        const int key = (rr * U / 32) & (U - 1);
        u32x4 v = region16[rr * LPR + (s ^ (key >> 1))];
        if (key & 1) v = u32x4{v[2], v[3], v[0], v[1]};
        // (nontemporal: the output is not read again by this launch, and written this way it disturbs the operands
        // in L2 less -- measured 1-4 % off whole GEMM launches at 2048 and 32768 tokens, int8 and FP6 kernels alike)
        if (rr < rows) __builtin_nontemporal_store(v, (u32x4*)(ybase + (int64_t)rr * N + s * 8));
    }
}

// A wave's 32 x 64 slab of an fp16 output, in two steps, so that the next slab can be computed between them.
//   slab_turn   the accumulator layout (a lane owns 4 consecutive columns of one row) becomes 16 bytes per lane with eight
//               consecutive lanes covering a 128-byte line: lane swaps make 16-byte pieces (upper against lower 32 lanes), a wave-private
//               LDS region of 4 KB turns them (position of a piece within its row XORed with the row: no bank conflicts).
//               (Lines by lane swaps alone, rows in consecutive lanes: the stores take four times as long, 64 bytes at a time.)
//   SlabOut     buffer stores: rows past the end of the output lie beyond the buffer's range and are dropped, columns past its end are
//               sent there.  No branches: with one around each store and its LDS read, the 256 x 256 tile of gemm_e2m3.hip
//               took 4.6 us to put out.
//   o[jj][gq] = this lane's columns jj * 32 + gq * 8 + (lane / 32) * 4 .. + 3 of row lane % 32
struct Slab {
    u32x4 v[4];                                 // rows lane / 8 + 8 p, 8 columns from (lane % 8) * 8 on
};
__device__ __forceinline__ Slab slab_turn(char* region, const f16x4 (&o)[2][4], int lane) {
    char* const put = region + (lane & 31) * 128 + (((lane >> 5) ^ (lane & 7)) * 16);
#pragma unroll
    for (int c = 0; c < 4; ++c) {               // pieces 2 c (lanes below 32) and 2 c + 1 of a row
        const u32x2 e = __builtin_bit_cast(u32x2, o[c >> 1][(c & 1) * 2]), f = __builtin_bit_cast(u32x2, o[c >> 1][(c & 1) * 2 + 1]);
        const auto s0 = __builtin_amdgcn_permlane32_swap(e[0], f[0], false, false);
        const auto s1 = __builtin_amdgcn_permlane32_swap(e[1], f[1], false, false);
        *(u32x4*)(region + ((u32)(put - region) ^ (u32)(c * 32))) = u32x4{s0[0], s1[0], s0[1], s1[1]};
    }
    const char* const get = region + (lane >> 3) * 128 + (((lane & 7) ^ ((lane >> 3) & 7)) * 16);
    Slab s;
#pragma unroll
    for (int p = 0; p < 4; ++p) s.v[p] = *(const u32x4*)(get + p * 1024);
    return s;
}
// The rows of an output tile that exist, `rows` from m0 on: at most 0xFFFFFF00 bytes of them (offsets of 32 bits)
struct SlabOut {
    __amdgpu_buffer_rsrc_t rsrc;
    u32 lane_at;                                // byte offset of this lane's first piece in a slab
    int N;
    bool wide, half;                            // rows are whole, aligned 16-byte (8-byte) pieces
};
__device__ __forceinline__ SlabOut slab_out(f16* Y, int m0, int rows, int N, int lane) {
    // (A workgroup that walks its tiles carries m0 round a loop, where the compiler loses sight that all lanes have the same one: it
    // would wrap every store in a loop over the distinct descriptors of a wave, 13 instructions each.  8191 x 5120 x 5120 + front 139.7 -> 136.1 us.)
    m0 = __builtin_amdgcn_readfirstlane(m0), rows = __builtin_amdgcn_readfirstlane(rows);
    return SlabOut{__builtin_amdgcn_make_buffer_rsrc((void*)(Y + (int64_t)m0 * N), 0, (int)((u32)rows * (u32)N * 2u), 0x00020000),
                   ((u32)(lane >> 3) * (u32)N + (u32)((lane & 7) * 8)) * 2u, N, (N & 7) == 0 && (((uintptr_t)Y) & 15) == 0, (N & 3) == 0};
}
// rows from `row` of the tile on, columns from col0 of the output up to `end`.  A caller whose outputs are all wide says so in WIDE, and has the code
// of whole pieces alone.
template <bool WIDE = false>
__device__ __forceinline__ void slab_store(const SlabOut& out, const Slab& s, int end, int row, int col0, int lane) {
    constexpr u32 GONE = 0xFFFFFF00u;           // beyond the range of every buffer here
    const u32 at = out.lane_at + ((u32)row * (u32)out.N + (u32)col0) * 2u, rows8 = (u32)out.N * 16u;
    const int left = end - col0 - (lane & 7) * 8;           // columns from the piece on
    // (nontemporal: the output is not read again by this launch, and written this way it disturbs the operands in L2 less --
    // measured 1-4 % off whole GEMM launches at 2048 and 32768 tokens)
    if (WIDE || out.wide) {
        const u32 off = left > 0 ? at : GONE, step = left > 0 ? rows8 : 0u;
#pragma unroll
        for (int p = 0; p < 4; ++p) __builtin_amdgcn_raw_buffer_store_b128(s.v[p], out.rsrc, off + step * (u32)p, 0, 2);
    } else if (out.half) {
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                __builtin_amdgcn_raw_buffer_store_b64(u32x2{s.v[p][2 * h], s.v[p][2 * h + 1]}, out.rsrc,
                                                      left > 4 * h ? at + rows8 * (u32)p + 8u * h : GONE, 0, 0);
    } else {
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int e = 0; e < 8; ++e)
                __builtin_amdgcn_raw_buffer_store_b16((unsigned short)(s.v[p][e >> 1] >> (16 * (e & 1))), out.rsrc,
                                                      left > e ? at + rows8 * (u32)p + 2u * e : GONE, 0, 0);
    }
}

// Four dequantised outputs of one row: fp16( fp16(sa * sb) * fp16(acc >> 8) ) (+ bias), the three
// (four) fp16 operations as packed instructions on column pairs -- each lane of a packed fp16
// multiply or add rounds exactly like the scalar instruction.
__device__ __forceinline__ f16x4 dequant4(int a0, int a1, int a2, int a3, f16 sa, f16x4 sb, f16x4 bi, bool with_bias) {
    const f16x2 s2 = {sa, sa};
    const f16x2 q01 = as_f16x2(narrow_f16x2((float)(a0 >> 8), (float)(a1 >> 8)));
    const f16x2 q23 = as_f16x2(narrow_f16x2((float)(a2 >> 8), (float)(a3 >> 8)));
    f16x2 y01 = (s2 * f16x2{sb[0], sb[1]}) * q01;
    f16x2 y23 = (s2 * f16x2{sb[2], sb[3]}) * q23;
    if (with_bias) {
        y01 = y01 + f16x2{bi[0], bi[1]};
        y23 = y23 + f16x2{bi[2], bi[3]};
    }
    return f16x4{y01[0], y01[1], y23[0], y23[1]};
}

// the same for accumulators that are exact integers held as fp32 (the FP6 matrix path)
__device__ __forceinline__ f16x4 dequant4_f32(float a0, float a1, float a2, float a3, f16 sa, f16x4 sb, f16x4 bi, bool with_bias) {
    const f16x2 s2 = {sa, sa};
    const f16x2 q01 = as_f16x2(narrow_f16x2(a0, a1));
    const f16x2 q23 = as_f16x2(narrow_f16x2(a2, a3));
    f16x2 y01 = (s2 * f16x2{sb[0], sb[1]}) * q01;
    f16x2 y23 = (s2 * f16x2{sb[2], sb[3]}) * q23;
    if (with_bias) {
        y01 = y01 + f16x2{bi[0], bi[1]};
        y23 = y23 + f16x2{bi[2], bi[3]};
    }
    return f16x4{y01[0], y01[1], y23[0], y23[1]};
}

// the same for sums held as 1/64 of the integer: the multiplication by 64 follows the rounding to fp16, which it commutes with
// (|sum| / 64 >= 2^-6 or 0 is far from fp16's subnormals; what rounds beyond 65504 becomes an infinity either way).
// bi is always added: -0 where there is no bias, which leaves every value as it is.
__device__ __forceinline__ f16x4 dequant4_f32x64(float a0, float a1, float a2, float a3, f16 sa, f16x4 sb, f16x4 bi) {
    const f16x2 s2 = {sa, sa}, x64 = {(f16)64.0f, (f16)64.0f};
    const f16x2 q01 = as_f16x2(cvt_f16x2(a0, a1)) * x64;
    const f16x2 q23 = as_f16x2(cvt_f16x2(a2, a3)) * x64;
    const f16x2 y01 = (s2 * f16x2{sb[0], sb[1]}) * q01 + f16x2{bi[0], bi[1]};
    const f16x2 y23 = (s2 * f16x2{sb[2], sb[3]}) * q23 + f16x2{bi[2], bi[3]};
    return f16x4{y01[0], y01[1], y23[0], y23[1]};
}

// A slab of two accumulator tiles, likewise.  One wave per SIMD has nobody to hide a chain of five dependent instructions behind: the 32
// values go through each step together (in chains the slab took 1200 cycles, 8 per instruction).  No addition where there is no bias.
__device__ __forceinline__ void dequant_slab_f32x64(const f32x16& a0, const f32x16& a1, f16 sa, const f16x4 (&sb)[2][4], const f16x4 (&bi)[2][4],
                                                    bool with_bias, f16x4 (&o)[2][4]) {
    const f16x2 s2 = {sa, sa}, x64 = {(f16)64.0f, (f16)64.0f};
    float v[32];
#pragma unroll
    for (int k = 0; k < 32; ++k) {
        v[k] = k < 16 ? a0[k] : a1[k - 16];
        asm volatile("" : "+v"(v[k]));
    }
    f16x2 q[16], s[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) q[k] = as_f16x2(cvt_f16x2(v[2 * k], v[2 * k + 1]));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const f16x4 b = sb[k >> 3][(k >> 1) & 3];
        s[k] = s2 * ((k & 1) ? f16x2{b[2], b[3]} : f16x2{b[0], b[1]});
        q[k] = q[k] * x64;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < 16; ++k) q[k] = s[k] * q[k];
    if (with_bias) {
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const f16x4 b = bi[k >> 3][(k >> 1) & 3];
            q[k] = q[k] + ((k & 1) ? f16x2{b[2], b[3]} : f16x2{b[0], b[1]});
        }
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k >> 2][k & 3] = f16x4{q[2 * k][0], q[2 * k][1], q[2 * k + 1][0], q[2 * k + 1][1]};
}

}  // namespace
