// int4 x int4 GEMM on the FP6 matrix path with ONE operand spread to six bits in memory first, exact: outputs that fill the compute units
// with tiles of 256 rows of one operand and 128 .. 256 of the other.
//
// gemm_e2m3.hip spreads the nibbles of both operands inside its loop, every fragment in two waves: 112 vector instructions per 16 matrix
// instructions, where a wave alone on its SIMD hides six per matrix instruction.  Here the operand with fewer rows (X; a prompt's weights,
// mostly) is spread by a pass of its own into the caller's scratch, and the other one (U) inside the loop, by the one wave that has its
// rows: 28.  X holds the codes as they are, sign and magnitude / 8 (E2M3 has a sign bit); U holds u = code + 8, the plain binary integer / 8.  Then
//   sum a b = sum x u - 8 sum x,
// and the sums of X's rows come with the spreading: the accumulators start from -8 sum x, and no matrix instruction adds up rows, as those
// of gemm_e2m3.hip must.  Every partial sum is an integer / 64: at most 64 per k that is multiplied and 64 per k that is not yet, 64 K < 2^24.
#include "qr_e2m3.h"
#include "qr_epilogue.h"

namespace {

typedef int i32x6 __attribute__((ext_vector_type(6)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef int i32x12 __attribute__((ext_vector_type(12)));

// X in memory: blocks of 32 rows x 128 k, 3072 bytes each, in the order in which a wave takes them as matrix operands: three planes of 16
// bytes per lane, lane = row % 32 + 32 * half; words 0 .. 5 of a lane's twelve are its fields of the first 64 k (32 of them per half), words
// 6 .. 11 those of the second.  [rows / 32][K / 128, even][3][64][16].  Rows and k beyond the operand are zeros, whatever U holds there.
constexpr int kBlock = 3072;

// Sixteen codes of two words -> three words of fields with sign and magnitude.  (Negative nibbles: 8 - their low three bits, a sum
// that stays within the nibble; the sign is bit 5 of a field: where kSpreadX's fields start, five bits on, and kSpreadY's.)
__device__ __forceinline__ void spread_signed(u32 x, u32 y, u32 (&d)[3]) {
    auto magnitude = [](u32 p, u32 s) { return ((p & 0x77777777u) ^ (s * 7u)) + s; };
    auto rotl = [](u32 v, int n) { return __builtin_amdgcn_alignbit(v, v, 32 - n); };
    const u32 sx = (x >> 3) & 0x11111111u, sy = (y >> 3) & 0x11111111u;
    const u32 mx = magnitude(x, sx), my = rotl(magnitude(y, sy), 2), tx = rotl(sx, 5), ty = rotl(sy, 7);
    d[0] = (mx & kSpreadX[0]) | (my & kSpreadY[0]) | (tx & 0x20020020u) | (ty & 0x00800800u);
    d[1] = (mx & kSpreadX[1]) | (my & kSpreadY[1]) | (tx & 0x00200200u) | (ty & 0x08008008u);
    d[2] = (mx & kSpreadX[2]) | (my & kSpreadY[2]) | (tx & 0x02002002u) | (ty & 0x80080080u);
}

// Spreads `rows` rows (a multiple of 32 in the output), R of them per workgroup over all of K, and leaves -(sum of the codes) / 8 of
// each.  Memory-bound: half a byte in, three quarters out per code (11008 x 4096 13 us).  Eight rows make whole lines of 128 bytes; 32 where
// that many workgroups fill the chip.
template <int R>
__global__ __launch_bounds__(512) void spread_x6_kernel(const uint8_t* __restrict__ P, int rows, int Kb, int units, uint8_t* __restrict__ X,
                                                        float* __restrict__ sums) {
    __shared__ int total[R];
    const int tid = threadIdx.x;
    if (tid < R) total[tid] = 0;
    __syncthreads();
    const int r = tid % R, half = (tid / R) & 1, row = blockIdx.x * R + r;
    const bool real = row < rows;
    const uint8_t* const from = P + (int64_t)(real ? row : 0) * Kb;
    uint8_t* const to = X + ((int64_t)(row >> 5) * units) * kBlock + ((row & 31) + 32 * half) * 16;
    int sum = 0;
#pragma unroll 4
    for (int u = tid / (2 * R); u < units; u += 256 / R) {
        u32x4 in[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int at = u * 64 + e * 32 + half * 16;
            in[e] = real && at < Kb ? *(const u32x4*)(from + at) : u32x4{0, 0, 0, 0};
        }
        u32 d[12];
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                u32 t[3];
                spread_signed(in[e][2 * h], in[e][2 * h + 1], t);
#pragma unroll
                for (int i = 0; i < 3; ++i) d[e * 6 + h * 3 + i] = t[i];
                sum = __builtin_amdgcn_sdot8((int)in[e][2 * h], 0x11111111, sum, false);
                sum = __builtin_amdgcn_sdot8((int)in[e][2 * h + 1], 0x11111111, sum, false);
            }
#pragma unroll
        for (int p = 0; p < 3; ++p) *(u32x4*)(to + (int64_t)u * kBlock + p * 1024) = u32x4{d[4 * p], d[4 * p + 1], d[4 * p + 2], d[4 * p + 3]};
    }
    atomicAdd(&total[r], sum);
    __syncthreads();
    if (tid < R) sums[blockIdx.x * R + tid] = (float)total[tid] * -0.125f;
}

// LDS: two stages of U (256 rows x 256 k, packed), three units of X (256 rows x 128 k), scales of two tiles ([256] sB, bias, sA in fp16) and
// the output slabs of four waves
constexpr int kStageU = 256 * 128, kUnitX = 8 * kBlock, kAtX = 2 * kStageU, kScales = 3 * 256;
constexpr int kLds = kAtX + 3 * kUnitX + 2 * kScales * 2 + 16384;

// Four waves, one per SIMD, each with 64 rows of U and all 32 NX rows of X: 2 NX accumulator tiles, up to all 256 accumulation registers.  XB:
// X is B (the weights), else A.  A workgroup takes `count` tiles, place(0), place(1) .., without a gap, as in gemm_e2m3.hip.
//
// A stage is 256 k, a unit 128, a sub-step 64.  U goes into LDS as it is, a line of 128 bytes per row and stage (keyed by permuting which 16
// bytes a lane fetches); a sub-step's fragments are read two sub-steps ahead and spread one ahead.  X goes there in blocks that need no key and
// no address arithmetic, twelve words per lane, fragment and unit: its fragments are read as the matrix instructions of the unit before let go
// of their words (the first four are free after the unit's first sub-step, the others as the second one goes; the last fragment's arrive
// in the first slots of the next unit, where it is used last).
// One barrier per unit, in its first sub-step: unit u + 1 of X and the stage that holds its part of U have landed, and nobody reads unit u any
// more.  Then unit u + 3 of X goes where unit u was, and after the second unit of a stage the stage after next of U where that stage was:
// two units' time for either.
//
// What bounds it is power: 32768 x 4096 x 11008 at NX = 8 takes 41 cycles of 1.67 GHz per matrix instruction, where gemm_e2m3.hip takes 57 of 2.11
// and the matrix unit alone 34 of 1.7.  Without the loads of its loop it would take 13 % less time, without spreading U 8 %, without reading X
// from LDS 7 % (with all three gone 6.96e15 operations per second, what the instruction sustains by itself): what is left costs energy, not issue.  As
// 2 x 2 waves of 128 x 128 (U spread twice, X read twice instead of four times) 635 us, so 605; sixteen matrix instructions in an order in
// which one operand stays, 1 % of that.  Measured, spreading included, against the kernels of gemm_e2m3.hip: 32768 x 4096 x 11008 703 -> 600
// us, 32768 x 11008 x 4096 795 -> 690, 16384 x 8192 x 8192 530 -> 472, 2048 x 8192 x 28672 222 -> 205, 8191 x 5120 x 5120 122 -> 112 (NX = 7: 2.9
// rounds of tiles), 2048 x 5120 x 13824 90 -> 80 (NX = 6).  A tile's end costs 8000 cycles: 3000 of arithmetic, 2700 to turn the slabs through LDS.
template <bool XB, int NX, class Place>
__device__ __forceinline__ void x6_tiles(const uint8_t* __restrict__ U, const uint8_t* __restrict__ X, const float* __restrict__ xsums,
                                         int M, int N, int Kb, f16* __restrict__ Y, const f16* __restrict__ sA, const f16* __restrict__ sB,
                                         const f16* __restrict__ bias, int count, Place place) {
    extern __shared__ u32x4 x6_smem[];
    char* const lds = (char*)x6_smem;
    f16* scales = (f16*)(lds + kAtX + 3 * kUnitX);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int stages = (Kb + 127) / 128;                    // two and more
    const int u_rows = XB ? M : N, x_rows = XB ? N : M, x_groups = (x_rows + 31) / 32;
    const u32 x_pitch = (u32)stages * 2u * (u32)kBlock;     // bytes of 32 rows of X

    // loads of U: chunk tid + i * 256 of a stage is 16 bytes of row tid / 8 + 32 i, at LDS position (row, tid % 8)
    const int srow = tid >> 3, piece = ((tid & 7) ^ ((srow >> 1) & 7)) * 16;
    Origin at = place(0);
    u32 goff[8];
    // X: load k of this wave's LX is KB number wave * LX + k of a unit (waves that would load past it repeat its last one)
    constexpr int LX = (3 * NX + 3) / 4;
    u32 xa[LX], xb[LX];                                     // bases of the loads of a stage's first and second unit (they differ where the second is the next tile's)
    u32 xa_at = 0, xb_at = 0, u_at = 0;                     // and how far along K
    auto aim = [&](Origin o) {
        int row0 = srow + (XB ? o.m0 : o.n0);
        asm volatile("" : "+v"(row0));                      // (computed here, not kept over the tiles)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int row = row0 + i * 32;
            goff[i] = (u32)(row < u_rows ? row : u_rows - 1) * (u32)Kb + (u32)piece;
        }
        int g0 = (XB ? o.n0 : o.m0) / 32;
        asm volatile("" : "+v"(g0));
#pragma unroll
        for (int k = 0; k < LX; ++k) {
            const int kb = wave * LX + k < 3 * NX ? wave * LX + k : 3 * NX - 1, g = g0 + kb / 3;
            xb[k] = (u32)(g < x_groups ? g : x_groups - 1) * x_pitch + (u32)(kb % 3) * 1024u + (u32)lane * 16u;
        }
    };
    aim(at);
    // (pieces past the end of a row of U are the next row's, or zeros beyond the operand: they meet zeros of X)
    const __amdgpu_buffer_rsrc_t rsrc_u = __builtin_amdgcn_make_buffer_rsrc((void*)U, 0, (int)((u32)u_rows * (u32)Kb), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc((void*)X, 0, (int)((u32)x_groups * x_pitch), 0x00020000);
    using Lds = __attribute__((address_space(3))) void*;
    auto load_u = [&](int i, int buf, u32 from) __attribute__((always_inline)) {
        const u32 off = goff[i];
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_u, (Lds)(lds + buf + (i * 256 + wave * 64) * 16), 16, off, from, 0, 0);
    };
    auto load_x = [&](int k, int buf, const u32 (&from)[LX], u32 along) __attribute__((always_inline)) {
        const int kb = wave * LX + k < 3 * NX ? wave * LX + k : 3 * NX - 1;
        const u32 off = from[k];
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_x, (Lds)(lds + kAtX + buf + kb * 1024), 16, off, along, 0, 0);
    };

    f32x16 acc[NX][2];                                       // [fragment of X][fragment of U]
    // addresses of U's first fragment in sub-step u (the others 4096 bytes apart), of X's first plane
    int base_u[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int row = wave * 64 + (lane & 31), chunk = 2 * u + (lane >> 5);
        base_u[u] = (row * 8 + (chunk ^ ((row >> 1) & 7))) * 16;
    }
    const int base_x = kAtX + lane * 16;
    struct Fragment {
        i32x12 w;
    };
    Fragment xf[NX];
    u32x4 raw[2];
    u32 ops[2][2][6];
    auto read_u = [&](int u, int g, int buf) __attribute__((always_inline)) { raw[g] = *(const u32x4*)(lds + (base_u[u] + buf) + g * 4096); };
    auto read_x = [&](auto fc, auto pc, int buf) __attribute__((always_inline)) {
        constexpr int f = decltype(fc)::value, p = decltype(pc)::value;
        const i32x4 v = *(const i32x4*)(lds + (base_x + buf) + f * kBlock + p * 1024);
#pragma unroll
        for (int i = 0; i < 4; ++i) xf[f].w[4 * p + i] = v[i];
    };

    u32 x0, x1, x2, y0, y1, y2, c0, c1, c2;                 // (one operand of a vector instruction may be scalar: kSpreadX in vector registers)
    asm("v_mov_b32 %0, %1" : "=v"(x0) : "n"(kSpreadX[0]));
    asm("v_mov_b32 %0, %1" : "=v"(x1) : "n"(kSpreadX[1]));
    asm("v_mov_b32 %0, %1" : "=v"(x2) : "n"(kSpreadX[2]));
    asm("s_mov_b32 %0, %1" : "=s"(y0) : "n"(kSpreadY[0]));
    asm("s_mov_b32 %0, %1" : "=s"(y1) : "n"(kSpreadY[1]));
    asm("s_mov_b32 %0, %1" : "=s"(y2) : "n"(kSpreadY[2]));
    asm("s_mov_b32 %0, %1" : "=s"(c0) : "n"(kSpreadFlip[0]));
    asm("s_mov_b32 %0, %1" : "=s"(c1) : "n"(kSpreadFlip[1]));
    asm("s_mov_b32 %0, %1" : "=s"(c2) : "n"(kSpreadFlip[2]));
    // instruction n of the 28 that spread a sub-step's two fragments
    auto spread1 = [&](u32 (&o)[2][6], int n) __attribute__((always_inline)) {
        constexpr u32 AND_XOR = 0x6a;                       // (a & b) ^ c
        const int t = n / 7, kind = n % 7, g = t >> 1, h = t & 1;
        u32* d = &o[g][3 * h];
        const u32 x = raw[g][2 * h], y = raw[g][2 * h + 1];
        if (kind == 0) raw[g][2 * h + 1] = __builtin_amdgcn_alignbit(y, y, 30);
        else if (kind == 1) d[0] = __builtin_amdgcn_bitop3_b32(x, x0, c0, AND_XOR);
        else if (kind == 2) d[1] = __builtin_amdgcn_bitop3_b32(x, x1, c1, AND_XOR);
        else if (kind == 3) d[2] = __builtin_amdgcn_bitop3_b32(x, x2, c2, AND_XOR);
        else if (kind == 4) d[0] = __builtin_amdgcn_bitop3_b32(y, y0, d[0], AND_XOR);
        else if (kind == 5) d[1] = __builtin_amdgcn_bitop3_b32(y, y1, d[1], AND_XOR);
        else d[2] = __builtin_amdgcn_bitop3_b32(y, y2, d[2], AND_XOR);
    };
    auto mfma1 = [&](auto second, const u32 (&o)[2][6], int f, int g) __attribute__((always_inline)) {
        constexpr int S = decltype(second)::value * 6;
        const i32x8 u = {(int)o[g][0], (int)o[g][1], (int)o[g][2], (int)o[g][3], (int)o[g][4], (int)o[g][5], 0, 0};
        const i32x8 x = __builtin_shufflevector(xf[f].w, xf[f].w, S, S + 1, S + 2, S + 3, S + 4, S + 5, -1, -1);
        acc[f][g] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(XB ? x : u, XB ? u : x, acc[f][g], 2, 2, 0, 0, 0, 0);
    };

    // Slots of a sub-step, a matrix instruction and its share of everything else each.  SUB: which one of its stage.  u_buf: the buffer of U that
    // holds sub-step SUB + 2; x_buf: of X, the one that this sub-step reads from (the next unit in a second sub-step; in a first one its own, for the last
    // fragment), x_next_buf: of the next unit; load_x_buf, load_u_buf: where the unit's loads go.  stores: the STORES or more of an epilogue are
    // behind the loads that its barrier waits for, and need not have arrived.
    constexpr int SLOTS = 2 * NX, BARRIER = SLOTS * 3 / 8;
    auto substep = [&](auto subc, int stores, int u_buf, int x_buf, int x_next_buf, int load_x_buf, int load_u_buf, const u32 (&x_from)[LX], u32 x_along)
        __attribute__((always_inline)) {
        constexpr int SUB = decltype(subc)::value, STORES = 4 * (XB ? (NX + 1) / 2 * 2 : NX);
        constexpr bool SECOND = SUB & 1;
        constexpr int LOADS = SUB < 2 ? LX : LX + 8;        // of the unit: X's, in the stage's second unit U's too, evenly over the slots behind the barrier
        constexpr int AHEAD = SUB < 2 ? LX + 8 : LX;        // of the unit before
        auto& cur = ops[SUB & 1];
        auto& nxt = ops[1 - (SUB & 1)];
        static_for<SLOTS>([&](auto qc) __attribute__((always_inline)) {
            constexpr int q = decltype(qc)::value, f = q / 2, g = q % 2;
            if constexpr (!SECOND && g == 0) asm volatile("" : "+v"(xf[f].w));      // (twelve registers in a row: six of them are an operand as they are)
            mfma1(IC<SECOND>(), cur, f, f & 1 ? 1 - g : g);     // (one of two operands stays from slot to slot: 1 % off long K, where power is the limit)
            constexpr int N0 = q * 28 / SLOTS, N1 = (q + 1) * 28 / SLOTS;
            static_for<N1 - N0>([&](auto nc) __attribute__((always_inline)) { spread1(nxt, N0 + decltype(nc)::value); });
            if constexpr (!SECOND && q < 2) read_x(IC<NX - 1>(), IC<q + 1>(), x_buf);
            if constexpr (SECOND && q >= 2) read_x(IC<f - 1>(), IC<1 + g>(), x_buf);
            if constexpr (!SECOND && q == BARRIER)
                asm volatile("s_cmp_lg_u32 %0, 0\n\ts_cbranch_scc1 1f\n\ts_waitcnt vmcnt(%1)\n1:\ts_waitcnt vmcnt(%2) lgkmcnt(0)\n\ts_barrier"
                             ::"s"(stores), "n"(AHEAD), "n"(AHEAD + STORES) : "memory", "scc");
            if constexpr (!SECOND && q > BARRIER && q < SLOTS - 2) read_x(IC<q - BARRIER - 1>(), IC<0>(), x_next_buf);
            if constexpr (!SECOND && q == SLOTS - 1) {
                static_for<NX - (SLOTS - 3 - BARRIER)>([&](auto ec) { read_x(IC<SLOTS - 3 - BARRIER + decltype(ec)::value>(), IC<0>(), x_next_buf); });
            }
            if constexpr (q == NX - 1 || q == SLOTS - 1) read_u((SUB + 2) & 3, q / NX, u_buf);
            static_for<LOADS>([&](auto kc) __attribute__((always_inline)) {
                constexpr int k = decltype(kc)::value, at = BARRIER + 1 + k * (2 * SLOTS - BARRIER - 1) / LOADS;
                if constexpr (at == q + SECOND * SLOTS) {
                    if constexpr (k < LX) load_x(k, load_x_buf, x_from, x_along);
                    else load_u(k - LX, load_u_buf, u_at);
                }
            });
            __builtin_amdgcn_sched_barrier(0);
        });
    };

    f16 pre_sb = (f16)0, pre_bi = (f16)-0.0f, pre_sa = (f16)0;
    float xs[NX];                                            // -(sum of a row of X) / 8, of the lane's row of every fragment
    auto fetch_scales = [&](Origin o) {
        const int col = o.n0 + tid < N ? o.n0 + tid : N - 1, row = o.m0 + tid < M ? o.m0 + tid : M - 1;
        pre_sb = sB[col], pre_sa = sA[row];
        if (bias) pre_bi = bias[col];
        int r = (XB ? o.n0 : o.m0) + (lane & 31);
        asm volatile("" : "+v"(r));
#pragma unroll
        for (int f = 0; f < NX; ++f) xs[f] = xsums[r + f * 32 < x_rows ? r + f * 32 : x_rows - 1];
    };
    auto park_scales = [&] { scales[tid] = pre_sb, scales[256 + tid] = pre_bi, scales[512 + tid] = pre_sa; };
    fetch_scales(at);

    // the pipeline's start: stage 0, units 0, 1, stage 1, unit 2
    int xc = 0, xn = kUnitX, xt = 2 * kUnitX;               // buffers of this unit of X, the next one and the one after that
    int uc = 0, un = kStageU;                               // buffers of this stage of U and the next one
#pragma unroll
    for (int k = 0; k < LX; ++k) xa[k] = xb[k];
#pragma unroll
    for (int i = 0; i < 8; ++i) load_u(i, 0, 0);
#pragma unroll
    for (int k = 0; k < LX; ++k) load_x(k, 0, xa, 0);
#pragma unroll
    for (int k = 0; k < LX; ++k) load_x(k, kUnitX, xa, kBlock);
#pragma unroll
    for (int i = 0; i < 8; ++i) load_u(i, kStageU, 128);
#pragma unroll
    for (int k = 0; k < LX; ++k) load_x(k, 2 * kUnitX, xa, 2 * kBlock);
    xa_at = 3 * kBlock, xb_at = 4 * kBlock, u_at = 256;
    park_scales();
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * LX + 8) : "memory");
#pragma unroll
    for (int g = 0; g < 2; ++g) read_u(0, g, 0);
    static_for<28>([&](auto nc) __attribute__((always_inline)) { spread1(ops[0], decltype(nc)::value); });
#pragma unroll
    for (int g = 0; g < 2; ++g) read_u(1, g, 0);
    auto read_all = [&](int buf) __attribute__((always_inline)) {
        static_for<NX - 1>([&](auto fc) { static_for<3>([&](auto pc) { read_x(fc, pc, buf); }); });
        read_x(IC<NX - 1>(), IC<0>(), buf);             // (the others in the first slots)
    };
    read_all(0);

    auto stage = [&](int stores) __attribute__((always_inline)) {
        substep(IC<0>(), stores, uc, xc, xn, xc, uc, xa, xa_at);
        substep(IC<1>(), stores, uc, xn, xn, xc, uc, xa, xa_at);
        substep(IC<2>(), stores, un, xn, xt, xn, uc, xb, xb_at);
        substep(IC<3>(), stores, un, xt, xt, xn, uc, xb, xb_at);
        const int t0 = xc, t1 = xn;                         // (two units on)
        xc = xt, xn = t0, xt = t1;
        uc = kStageU - uc, un = kStageU - un;
        xa_at = xb_at + kBlock, xb_at += 2 * kBlock, u_at += 128;
    };
    const int turn = stages - 2;                            // from this stage's second unit on, the loads are the next tile's
    for (int t = 0;;) {
        Origin then{0, 0};
#pragma unroll
        for (int f = 0; f < NX; ++f)
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                f32x16 none;
#pragma unroll
                for (int v = 0; v < 16; ++v) none[v] = 0.f;
                const float s = lane < 32 ? xs[f] : 0.f;
                float one = 1.f;
                asm volatile("" : "+v"(one));               // (or the compiler makes one tile and copies it, 16 moves a time)
                acc[f][g] = __builtin_amdgcn_mfma_f32_32x32x2f32(XB ? s : one, XB ? one : s, none, 0, 0, 0);
            }
        auto prepare = [&] {
            if (t + 1 >= count) return;                     // (what is loaded past the last tile nobody uses)
            then = place(t + 1);
            aim(then);
            fetch_scales(then);
            xb_at = 0, u_at = 0;
        };
        int stores = t;                                     // (of the epilogue before: its 32 or more may pass the first stage's barriers)
        for (int ks = 0; ks < stages;) {
            if (ks == turn) prepare();
            if (ks == turn + 1) {
#pragma unroll
                for (int k = 0; k < LX; ++k) xa[k] = xb[k];
            }
            const int stop = ks < turn ? turn : ks == turn ? turn + 1 : stages;
            for (; ks < stop; ++ks) {
                stage(stores);
                stores = 0;
            }
        }
        const bool last = t + 1 == count;
        if (last) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (loads still landing in LDS that may be somebody else's soon)

        // Epilogue: lane l, register v -> column (v / 4) * 8 + (l / 32) * 4 + v % 4 of the B tile, token l % 32
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const int kh = ln >> 5;
        char* const region = lds + kAtX + 3 * kUnitX + 2 * kScales * 2 + wave * 4096;
        const int rows = XB ? 256 : 32 * NX;
        const SlabOut out = slab_out(Y, at.m0, M - at.m0 < rows ? M - at.m0 : rows, N, ln);
        Slab slab;
        constexpr int JB = XB ? NX : 2, IB = XB ? 2 : NX;   // groups of 32 columns and of 32 rows of this wave
        const int m1 = XB ? wave * 64 : 0, n1 = XB ? 0 : wave * 64;
        const int end = at.n0 + (XB ? 32 * NX : 256), limit = end < N ? end : N;
        f16 sa[IB];
#pragma unroll
        for (int i = 0; i < IB; ++i) sa[i] = scales[512 + m1 + i * 32 + (ln & 31)];
#pragma unroll
        for (int jb = 0; jb < JB; jb += 2) {
            f16x4 sbh[2][4], bih[2][4];
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                for (int gq = 0; gq < 4; ++gq) {
                    const int col = n1 + (jb + jj) * 32 + gq * 8 + kh * 4;
                    sbh[jj][gq] = *(const f16x4*)(scales + col);
                    bih[jj][gq] = *(const f16x4*)(scales + 256 + col);
                }
#pragma unroll
            for (int i = 0; i < IB; ++i) {
                // (a slab of an odd last group of columns is half empty)
                constexpr int odd = XB && NX % 2;
                f32x16 &a0 = XB ? acc[jb][i] : acc[i][jb], &a1 = XB ? acc[jb + 1 < JB || !odd ? jb + 1 : jb][i] : acc[i][jb + 1];
                asm volatile("" : "+a"(a0), "+a"(a1));      // (moved out of their registers here, not before)
                f16x4 o[2][4];
                dequant_slab_f32x64(a0, a1, sa[i], sbh, bih, bias != nullptr, o);
                if (jb + i > 0)
                    slab_store<true>(out, slab, limit, m1 + (i > 0 ? i - 1 : IB - 1) * 32, at.n0 + n1 + (i > 0 ? jb : jb - 2) * 32, ln);
                slab = slab_turn(region, o, ln);
            }
        }
        slab_store<true>(out, slab, limit, m1 + (IB - 1) * 32, at.n0 + n1 + (JB - 1) / 2 * 64, ln);
        if (last) return;
        // the next tile's scales into the other half of their place (a slower wave may still read this tile's)
        scales = scales == (f16*)(lds + kAtX + 3 * kUnitX) ? scales + kScales : (f16*)(lds + kAtX + 3 * kUnitX);
        park_scales();
        // (X's fragments again, rather than kept in 96 registers over the epilogue)
        read_all(xc);
        at = then;
        ++t;
    }
}

// Tiles are dealt to the XCDs in runs of `per_xcd`, and workgroup b takes every (gridDim / nxcd)-th of its XCD's run
template <bool XB, int NX>
__global__ __launch_bounds__(256) void gemm_x6_kernel(const uint8_t* __restrict__ U, const uint8_t* __restrict__ X,
                                                      const float* __restrict__ xsums, int M, int N, int Kb, f16* __restrict__ Y,
                                                      const f16* __restrict__ sA, const f16* __restrict__ sB, const f16* __restrict__ bias,
                                                      int tiles_m, int tiles_n, int nxcd) {
    const int tiles = tiles_m * tiles_n, per_xcd = (tiles + nxcd - 1) / nxcd, xcd = blockIdx.x % nxcd;
    const int run = tiles - xcd * per_xcd < per_xcd ? tiles - xcd * per_xcd : per_xcd;
    const int first = blockIdx.x / nxcd, step = gridDim.x / nxcd;
    if (first >= run) return;
    x6_tiles<XB, NX>(U, X, xsums, M, N, Kb, Y, sA, sB, bias, (run - first + step - 1) / step, [=](int t) {
        const TilePlace p = tile_place(xcd * per_xcd + first + t * step, tiles_m, tiles_n);
        return XB ? Origin{p.tm * 256, p.tn * 32 * NX} : Origin{p.tm * 32 * NX, p.tn * 256};
    });
}

}  // namespace

// Bytes of scratch for `rows` rows of K codes: blocks, then a float per row
size_t qr_internal_x6_bytes(int64_t rows, int64_t Kb) {
    const int64_t groups = (rows + 31) / 32, units = (Kb + 127) / 128 * 2;
    return (size_t)(groups * units * kBlock + groups * 32 * 4);
}

// The operand with fewer rows is spread into `scratch` (qr_internal_x6_bytes of it, 16-byte aligned, below 4 GiB), then the product.  K of two
// stages and more; operands below 4 GiB, outputs within qr_e2m3_reach(256).
int qr_internal_gemm_x6(int nx, const void* A, const void* B, int M, int N, int Kb, void* Y, const void* sA, const void* sB, const void* bias,
                        void* scratch, hipStream_t st) {
    const bool xb = N <= M;
    const int rows = xb ? N : M, groups = (rows + 31) / 32, units = (Kb + 127) / 128 * 2;
    const int64_t bytes = (int64_t)groups * units * kBlock;
    if (Kb <= 128 || (int64_t)M * Kb >= (1LL << 32) || (int64_t)N * Kb >= (1LL << 32) || bytes >= (1LL << 32) || !qr_e2m3_reach(256, N, true))
        return QR_E_UNSUPPORTED;                            // (the dispatcher routes these away)
    uint8_t* const X = (uint8_t*)scratch;
    float* const sums = (float*)(X + bytes);
    if (groups >= 256) spread_x6_kernel<32><<<dim3(groups), dim3(512), 0, st>>>((const uint8_t*)(xb ? B : A), rows, Kb, units, X, sums);
    else spread_x6_kernel<8><<<dim3(groups * 4), dim3(512), 0, st>>>((const uint8_t*)(xb ? B : A), rows, Kb, units, X, sums);
    const int bm = xb ? 256 : 32 * nx, bn = xb ? 32 * nx : 256;
    const int tiles_m = (M + bm - 1) / bm, tiles_n = (N + bn - 1) / bn, nxcd = qr_device().xcds, cus = qr_device().cus;
    const int64_t tiles = (int64_t)tiles_m * tiles_n, all = (tiles + nxcd - 1) / nxcd * nxcd;
    const int64_t grid = cus % nxcd == 0 && all > cus ? cus : all;
    if (grid > 0x3fffffff) return QR_E_SHAPE;
    using Kern = void (*)(const uint8_t*, const uint8_t*, const float*, int, int, int, f16*, const f16*, const f16*, const f16*, int, int, int);
    static const Kern table[2][5] = {
        {gemm_x6_kernel<false, 4>, gemm_x6_kernel<false, 5>, gemm_x6_kernel<false, 6>, gemm_x6_kernel<false, 7>, gemm_x6_kernel<false, 8>},
        {gemm_x6_kernel<true, 4>, gemm_x6_kernel<true, 5>, gemm_x6_kernel<true, 6>, gemm_x6_kernel<true, 7>, gemm_x6_kernel<true, 8>}};
    const Kern kern = table[xb][nx - 4];
    const hipError_t e = qr_allow_dynamic_lds((const void*)kern, kLds);
    if (e != hipSuccess) return (int)e;
    kern<<<dim3((unsigned)grid), dim3(256), kLds, st>>>((const uint8_t*)(xb ? A : B), X, sums, M, N, Kb, (f16*)Y, (const f16*)sA,
                                                        (const f16*)sB, (const f16*)bias, tiles_m, tiles_n, nxcd);
    return qr_launch_status();
}
