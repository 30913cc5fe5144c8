// int4 x int4 GEMM for prompts of a few hundred tokens (and other outputs of too few 128 x 256 tiles for the 256 CUs):
// small tiles, K split among the waves of a workgroup.  C[M, N] = unpack(A)[M, K] . unpack(B)[N, K]^T, operands, packing
// and the x16 feeding of the int8 matrix instruction as in gemm.hip.
//
// What bounds these shapes is not the matrix pipe but how fast the CUs take their operands in: a CU pulls at most
// ~65 GB/s from L2, a tile needs (BM + BN) * K / 2 bytes, and with 64 x 256 tiles (the kernel this one replaces) a prompt
// of 333 tokens against 4096 weight rows gave 96 of 256 CUs 40 KB per 256 k each.  Tiles of 64 x 128, 128 x 128 and
// 64 x 64 spread the same bytes over all CUs.  Every wave owns a 64 x 64 wave tile (6 unpacking instructions per MFMA,
// affordable where the pipe idles anyway); WK groups of waves take the 64-k sub-steps of a 256-k stage (a 128-byte line
// per row) in turn, so a small tile still keeps eight waves busy, and add their accumulators through LDS at the end.
// One tile of 96 x 64 per CU takes in 160 rows per stage where one of 64 x 128 takes 192 and two of 64 x 64 take 256: 333 x 4096 x 4096
// 11.3 -> 10.2 us, 192 x 8192 x 8192 16.8 -> 15.3, 333 x 4096 x 11008 20.7 -> 18.5, 180 x 8192 x 28672 58 -> 47.
// Stages go straight from global memory into LDS (buffer_load ... lds), NBUF - 1 stages ahead, one barrier per stage;
// while a stage's MFMAs run, the wave's fragments of the next sub-step are read and unpacked.
// K need not be a multiple of 256: a sub-step beyond K is skipped (its loads repeat the stage's first piece).
// STREAM (up to 64 tokens: one row of tiles, every weight used once): the weights' loads are nontemporal, so that they do not
// push the tokens' codes out of the caches, and tile t starts its walk over K at stage t (integer sums do not depend on the order),
// so that the workgroups do not all ask the same memory channels at a time where the row pitch is a power of two.  With
// weights that come from memory (more of them in turn than the last-level cache holds), 48 tokens against 12288 x 4096: 11.2 -> 9.1 us, 8192 x 8192
// 17.2 -> 13.1, 28672 x 8192 30.9 -> 26.4.
#include "qr_common.h"
#include "qr_epilogue.h"

namespace {

template <int TM, int BN, int WK, int NBUF, bool DEQ, bool STREAM, int IM = 2>
__global__ __launch_bounds__(64 * (TM / 64) * (BN / 64) * WK) void gemm_mid_kernel(
    const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, int M, int N, int Kb, int32_t* __restrict__ C,
    f16* __restrict__ Y, const f16* __restrict__ sA, const f16* __restrict__ sB, const f16* __restrict__ bias,
    int tiles_m, int tiles_n, int ksplit, int nxcd) {
    constexpr int WM = TM / 64, WN = BN / 64, NT = 64 * WM * WN * WK;
    constexpr int BM = 32 * IM * WM;                        // rows of the tile: TM, or half as many again (IM = 3)
    constexpr int NF = IM + 2, NMF = 4 * IM, UNP = 12 * NF; // fragments, matrix and unpacking instructions of a sub-step
    constexpr int CH = (BM + BN) * 8;                       // 16-byte pieces per stage
    constexpr int NL = CH / NT;                             // ... per thread
    constexpr int RPL = NT / 8;                             // rows per load instruction of the workgroup
    constexpr int SUB = 4 / WK;                             // sub-steps per wave and stage
    static_assert(IM == 2 || (IM == 3 && TM == 64 && BN == 64 && WK == 4 && !STREAM), "wave tiles of 64 x 64 or 96 x 64");
    static_assert((WK == 2 || WK == 4) && CH % NT == 0 && BM % RPL == 0 && RPL % 16 == 0, "tile shape");
    extern __shared__ u32x4 mid_lds[];                      // [NBUF][CH]; later the accumulator exchange, then the output slabs

    // the slices of a tile are neighbours, and the tiles of an XCD's L2 share rows of both operands
    const int per_xcd = gridDim.x / nxcd;
    const int unit = (blockIdx.x % nxcd) * per_xcd + blockIdx.x / nxcd;
    if (unit >= tiles_m * tiles_n * ksplit) return;
    const int tile = unit / ksplit, split = unit - tile * ksplit;
    constexpr int GROUP_M = 8;
    const int group_sz = GROUP_M * tiles_n;
    const int gr = tile / group_sz;
    const int gm0 = gr * GROUP_M;
    const int gh = (tiles_m - gm0) < GROUP_M ? (tiles_m - gm0) : GROUP_M;
    const int m0 = (gm0 + (tile - gr * group_sz) % gh) * BM, n0 = ((tile - gr * group_sz) / gh) * BN;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave / (WM * WN), wxy = wave % (WM * WN), wm = wxy / WN, wn = wxy % WN;
    const int khalf = lane >> 5;
    const int all_stages = (Kb + 127) / 128;
    if (ksplit > 1) C += (int64_t)split * M * N;
    const int s0 = (int)((int64_t)all_stages * split / ksplit);
    const int stages = (int)((int64_t)all_stages * (split + 1) / ksplit) - s0;      // >= 1: ksplit <= all_stages
    const int rot = STREAM && (Kb & 127) == 0 ? tile % stages : 0;     // (a last stage that ends inside K stays the last)
    auto slot8 = [](int row, int chunk) { return row * 8 + (chunk ^ ((row >> 1) & 7)); };

    // ---- staging: a thread fetches, for its rows srow + i RPL, the piece that the XOR-keyed layout keeps at its place
    const int srow = tid >> 3;
    const int piece = ((tid & 7) ^ ((srow >> 1) & 7)) * 16;
    u32 goff[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int row = srow + i * RPL;
        int g = row < BM ? m0 + row : n0 + row - BM;
        const int lim = row < BM ? M - 1 : N - 1;
        g = g < lim ? g : lim;
        goff[i] = (u32)g * (u32)Kb;
    }
    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, (int)((u32)M * (u32)Kb), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void*)B, 0, (int)((u32)N * (u32)Kb), 0x00020000);
    auto request1 = [&](int st, int buf, int i) {           // load i of stage st into stage buffer buf
        const int at = st + rot;
        const int kb = (s0 + (STREAM && at >= stages ? at - stages : at)) * 128;
        __attribute__((address_space(3))) void* dst =
            (__attribute__((address_space(3))) void*)(mid_lds + buf * CH + i * NT + wave * 64);
        const u32 o = goff[i] + (u32)(kb + piece < Kb ? piece : 0);
        if (i * RPL < BM) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, dst, 16, o, kb, 0, 0);
        else __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, dst, 16, o, kb, 0, STREAM ? 2 : 0);
    };

    // ---- fragments.  A K-group holds its accumulator tiles permuted so that the ones it finalises are always the first:
    // WK = 4: register r is tile r ^ kg of the 2 x 2 (row tile (r ^ kg) >> 1, column tile (r ^ kg) & 1), tile kg is its own;
    // WK = 2: the row tiles swapped in group 1, row tile kg is its own.  96-row tiles: six tiles for four groups, summed row by row instead.
    const int fi = IM == 3 ? 0 : WK == 4 ? kg >> 1 : kg, fj = IM == 2 && WK == 4 ? kg & 1 : 0;
    i32x16 acc[IM][2];
#pragma unroll
    for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0;
    int fslot[SUB][NF];                                     // LDS slots of the wave's fragments (IM of A, two of B)
#pragma unroll
    for (int u = 0; u < SUB; ++u) {
        const int chunk = 2 * (kg * SUB + u) + khalf;
#pragma unroll
        for (int t = 0; t < IM; ++t) fslot[u][t] = slot8(wm * 64 + (t ^ fi) * 32 + (lane & 31), chunk);
#pragma unroll
        for (int t = 0; t < 2; ++t) fslot[u][IM + t] = slot8(BM + wn * 64 + (t ^ fj) * 32 + (lane & 31), chunk);
    }
    struct Packed {
        u32x4 f[NF];
    };
    struct Ops {
        i32x4 lo[NF], hi[NF];
    };
    auto read1 = [&](int buf, int u, int t, Packed& p) { p.f[t] = mid_lds[buf * CH + fslot[u][t]]; };
    // unpacking as 12 NF single instructions: dword d = n / 3 of the packed dwords, n % 3 = 0: lo = p << 4; 1: lo &= mask;
    // 2: hi = p & mask
    auto unpack1 = [&](const Packed& p, Ops& o, int n) {
        const int d = n / 3, f = d >> 2, e = d & 3, kind = n % 3;
        if (kind == 0) o.lo[f][e] = (int)(p.f[f][e] << 4);
        else if (kind == 1) o.lo[f][e] = o.lo[f][e] & (int)0xF0F0F0F0u;
        else o.hi[f][e] = (int)(p.f[f][e] & 0xF0F0F0F0u);
    };
    auto mfma1 = [&](const Ops& o, int q) {
        const int i = (q >> 1) % IM, j = q & 1;
        if (q < 2 * IM) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(o.lo[IM + j], o.lo[i], acc[i][j], 0, 0, 0);
        else acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(o.hi[IM + j], o.hi[i], acc[i][j], 0, 0, 0);
    };
    // One 64-k sub-step = NMF slots, each an MFMA of the current operands, a share of the next sub-step's unpacking (its
    // fragments are read in slot 0; UNP instructions from slot S0 on) and at most one load request; a full scheduling
    // barrier after every slot keeps the two waves of a SIMD from unpacking and multiplying in step.
    constexpr int S0 = 3;
    auto substep = [&](const Ops& cur, Ops& nxt, int rbuf, int ru, auto&& req) {
        Packed pk;
#pragma unroll
        for (int q = 0; q < NMF; ++q) {
            mfma1(cur, q);
            if (q == 0) {
#pragma unroll
                for (int t = 0; t < NF; ++t) read1(rbuf, ru, t, pk);
            }
            if (q >= 1 && q <= NL) req(q - 1);
            if (q >= S0) {
#pragma unroll
                for (int n = (q - S0) * UNP / (NMF - S0); n < (q - S0 + 1) * UNP / (NMF - S0); ++n) unpack1(pk, nxt, n);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto fill = [&](int rbuf, int ru, Ops& o) {             // the same without a multiplication under it
        Packed pk;
#pragma unroll
        for (int t = 0; t < NF; ++t) read1(rbuf, ru, t, pk);
#pragma unroll
        for (int n = 0; n < UNP; ++n) unpack1(pk, o, n);
    };
    // sub-step (st, u) lies inside K (K is a multiple of 64; uniform over the wave)
    auto inside = [&](int st, int u) { return (s0 + st) * 128 + (kg * SUB + u) * 32 < Kb; };
    auto multiply = [&](int st, int u, const Ops& o) {
        if (inside(st, u)) {
#pragma unroll
            for (int q = 0; q < NMF; ++q) mfma1(o, q);
        }
    };

    // Stage s lives in buffer s % NBUF.  Before its last sub-step of stage s a wave passes the barrier that says: stage s + 1
    // has landed and everybody has read all of stage s (reads precede the barrier by its lgkmcnt wait); stage s + NBUF is then
    // requested into the buffer of stage s, and stage s + 1 is read under the MFMAs.
#define QR_MID_WAIT(LEFT) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LEFT) : "memory")
    auto wait = [&](int left) {                             // stages that may still be in flight behind the one needed
        if (left <= 0) QR_MID_WAIT(0);
        else if (left == 1) QR_MID_WAIT(NL);
        else if (left == 2) QR_MID_WAIT(2 * NL);
        else if (left == 3) QR_MID_WAIT(3 * NL);
        else QR_MID_WAIT(4 * NL);
    };
    static_assert(NBUF >= 3 && NBUF <= 5, "waits are spelled for at most four stages behind the needed one");
    // (IM = 3) the epilogue's scales and bias: rows tid / 8 + 32 p, columns (tid % 8) * 8 .. + 7; -0 where there is no bias, which leaves every
    // value as it is
    const bool lines = DEQ && n0 + BN <= N && (N & 7) == 0 && (((uintptr_t)Y) & 15) == 0;
    f16 sa3[3];
    f16x8 sb8, bi8;
    if (IM == 3 && lines) {
#pragma unroll
        for (int p = 0; p < 3; ++p) sa3[p] = sA[min(m0 + (tid >> 3) + 32 * p, M - 1)];
        typedef f16x8 any_f16x8 __attribute__((aligned(2)));           // (weight scales and bias may start anywhere: views of larger tensors)
        sb8 = *(const any_f16x8*)(sB + n0 + (tid & 7) * 8);
        if (bias) bi8 = *(const any_f16x8*)(bias + n0 + (tid & 7) * 8);
        else
#pragma unroll
            for (int e = 0; e < 8; ++e) bi8[e] = (f16)-0.0f;
    }
    // (the buffers beyond three are asked for when the first stage has landed, which they would delay for all workgroups: 64 x 64 tiles with four, see
    // below, 128 x 128 tiles 0.8 % faster over 26 shapes, 64 tokens x 11008 x 4096 9.56 -> 9.40 us.  All at once where little is delayed or the walk
    // is short: the larger stages of 96-row tiles, 333 x 4096 x 4096 three times 35.0 us behind two fronts, 35.3 the other way; few rows of x, 8 x
    // 12288 x 4096 8.52, 8.62; slices of K, 24 x 1000 x 12288 9.53, 9.65)
    const int first = IM == 3 || (STREAM && (ksplit > 1 || M <= 16)) ? NBUF : 3;
    for (int st = 0; st < first && st < stages; ++st)
#pragma unroll
        for (int i = 0; i < NL; ++i) request1(st, st, i);
    wait(stages - 1 < first - 1 ? stages - 1 : first - 1);
    for (int st = first; st < NBUF && st < stages; ++st)
#pragma unroll
        for (int i = 0; i < NL; ++i) request1(st, st, i);
    Ops ops[2];
    fill(0, 0, ops[0]);
    int buf = 0, s = 0;
    const auto none = [](int) {};
    auto turn = [&](Ops& cur, Ops& nxt) {                   // SUB = 1: cur holds (s, 0) and nxt receives (s + 1, 0)
        const int nb = buf == NBUF - 1 ? 0 : buf + 1;
        if (SUB == 2) substep(cur, nxt, buf, 1, none);
        QR_MID_WAIT((NBUF - 2) * NL);
        const int fb = buf;
        auto req = [&](int i) { request1(s + NBUF, fb, i); };
        if (SUB == 2) substep(nxt, cur, nb, 0, req);
        else substep(cur, nxt, nb, 0, req);
        buf = nb;
        ++s;
    };
    if (SUB == 2) {
        while (s + NBUF < stages) turn(ops[0], ops[1]);
    } else {
        while (s + NBUF + 1 < stages) {
            turn(ops[0], ops[1]);
            turn(ops[1], ops[0]);
        }
        if (s + NBUF < stages) {
            turn(ops[0], ops[1]);
            ops[0] = ops[1];
        }
    }
    for (; s + 1 < stages; ++s) {                           // nothing left to request; these stages are whole
        const int nb = buf == NBUF - 1 ? 0 : buf + 1;
        if (SUB == 2) substep(ops[0], ops[1], buf, 1, none);
        wait(stages - 2 - s);
        if (SUB == 2) {
            substep(ops[1], ops[0], nb, 0, none);
        } else {
            substep(ops[0], ops[1], nb, 0, none);
            ops[0] = ops[1];
        }
        buf = nb;
    }
    multiply(s, 0, ops[0]);                                 // the last stage may end inside
    if (SUB == 2) {
        fill(buf, 1, ops[1]);
        multiply(s, 1, ops[1]);
    }
#undef QR_MID_WAIT

    // ---- the K-groups' sums: every group sends the tiles it does not finalise through LDS and adds what it receives
    __syncthreads();                                        // stage buffers free
    if constexpr (IM == 3) {
        // Every group puts all its sums out, [group][96 rows][16 pieces of four columns], pieces XORed with the row; a thread adds up the four
        // groups' eight columns (tid % 8) * 8 .. of rows tid / 8 + 32 p and stores them, eight threads a line.
        const int key = lane & 15;
#pragma unroll
        for (int i = 0; i < IM; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int qv = 0; qv < 4; ++qv)
                    mid_lds[(kg * 96 + i * 32 + (lane & 31)) * 16 + ((j * 8 + qv * 2 + khalf) ^ key)] =
                        u32x4{(u32)acc[i][j][qv * 4], (u32)acc[i][j][qv * 4 + 1], (u32)acc[i][j][qv * 4 + 2], (u32)acc[i][j][qv * 4 + 3]};
        __syncthreads();
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            const int r = (tid >> 3) + 32 * p, row = m0 + r, col = n0 + (tid & 7) * 8;
            i32x4 v[2] = {i32x4{0, 0, 0, 0}, i32x4{0, 0, 0, 0}};
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    v[h] += __builtin_bit_cast(i32x4, mid_lds[(g * 96 + r) * 16 + (((tid & 7) * 2 + h) ^ (r & 15))]);
            if (row >= M) continue;
            if (lines) {
                u32x4 o;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const f16x4 y = dequant4(v[h][0], v[h][1], v[h][2], v[h][3], sa3[p], f16x4{sb8[4 * h], sb8[4 * h + 1], sb8[4 * h + 2], sb8[4 * h + 3]},
                                             f16x4{bi8[4 * h], bi8[4 * h + 1], bi8[4 * h + 2], bi8[4 * h + 3]}, true);
                    const u32x2 w = __builtin_bit_cast(u32x2, y);
                    o[2 * h] = w[0], o[2 * h + 1] = w[1];
                }
                __builtin_nontemporal_store(o, (u32x4*)(Y + (int64_t)row * N + col));
                continue;
            }
            const f16 s = DEQ ? sA[row] : (f16)0;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (!DEQ && col + 4 * h + 4 <= N && (N & 3) == 0) {
                    *(i32x4*)(C + (int64_t)row * N + col + 4 * h) = i32x4{v[h][0] >> 8, v[h][1] >> 8, v[h][2] >> 8, v[h][3] >> 8};
                    continue;
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int c = col + 4 * h + e;
                    if (c >= N) continue;
                    if (DEQ) {
                        f16 yv = (f16)(s * sB[c]) * (f16)(float)(v[h][e] >> 8);
                        if (bias) yv = yv + bias[c];
                        Y[(int64_t)row * N + c] = yv;
                    } else {
                        C[(int64_t)row * N + c] = v[h][e] >> 8;
                    }
                }
            }
        }
        return;
    }
    if (WK == 4) {
#pragma unroll
        for (int r = 1; r < 4; ++r)
#pragma unroll
            for (int qv = 0; qv < 4; ++qv) {
                const i32x16& t = acc[r >> 1][r & 1];
                mid_lds[(((wxy * 4 + (r ^ kg)) * 3 + r - 1) * 4 + qv) * 64 + lane] =
                    u32x4{(u32)t[qv * 4], (u32)t[qv * 4 + 1], (u32)t[qv * 4 + 2], (u32)t[qv * 4 + 3]};
            }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int qv = 0; qv < 4; ++qv) {
                const u32x4 p = mid_lds[(((wxy * 4 + kg) * 3 + r) * 4 + qv) * 64 + lane];
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[0][0][qv * 4 + e] += (int)p[e];
            }
    } else {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int qv = 0; qv < 4; ++qv) {
                const i32x16& t = acc[1][j];
                mid_lds[((wxy * 2 + 1 - kg) * 8 + j * 4 + qv) * 64 + lane] =
                    u32x4{(u32)t[qv * 4], (u32)t[qv * 4 + 1], (u32)t[qv * 4 + 2], (u32)t[qv * 4 + 3]};
            }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int qv = 0; qv < 4; ++qv) {
                const u32x4 p = mid_lds[((wxy * 2 + kg) * 8 + j * 4 + qv) * 64 + lane];
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[0][j][qv * 4 + e] += (int)p[e];
            }
    }
    __syncthreads();                                        // exchange buffers free for the output slabs

    // ---- epilogue: this wave's 32 rows (tokens) x 32 NJ columns; lane l, register v -> n = (v/4)*8 + (l/32)*4 + v%4, m = l%32
    constexpr int NJ = WK == 4 ? 1 : 2;
    const int row0 = m0 + wm * 64 + fi * 32, col0 = n0 + wn * 64 + fj * 32;
    if (row0 >= M) return;
    const int row = row0 + (lane & 31);
    if (lines) {
        const f16 sa = sA[min(row, M - 1)];                 // (rows past M: computed on a clamped scale, not stored)
        f16x4 o[NJ][4];
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int gq = 0; gq < 4; ++gq) {
                const int col = col0 + j * 32 + gq * 8 + khalf * 4;
                const f16x4 sb = *(const f16x4*)(sB + col);
                const f16x4 bi = bias ? *(const f16x4*)(bias + col) : f16x4{(f16)0, (f16)0, (f16)0, (f16)0};
                o[j][gq] = dequant4(acc[0][j][gq * 4], acc[0][j][gq * 4 + 1], acc[0][j][gq * 4 + 2], acc[0][j][gq * 4 + 3], sa, sb,
                                    bi, bias != nullptr);
            }
        store_slab_rows<NJ>((u32x2*)(mid_lds + wave * (32 * NJ * 8 / 2)), o, lane, Y + (int64_t)row0 * N + col0, N, M - row0);
        return;
    }
    if (row >= M) return;
    const f16 sa = DEQ ? sA[row] : (f16)0;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int gq = 0; gq < 4; ++gq) {
            const int col = col0 + j * 32 + gq * 8 + khalf * 4;
            int v4[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v4[e] = acc[0][j][gq * 4 + e] >> 8;
            if (!DEQ && col + 4 <= N && (N & 3) == 0) {
                *(i32x4*)(C + (int64_t)row * N + col) = i32x4{v4[0], v4[1], v4[2], v4[3]};
                continue;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (col + e < N) {
                    if (DEQ) {
                        f16 yv = (f16)(sa * sB[col + e]) * (f16)(float)v4[e];
                        if (bias) yv = yv + bias[col + e];
                        Y[(int64_t)row * N + col + e] = yv;
                    } else {
                        C[(int64_t)row * N + col + e] = v4[e];
                    }
                }
        }
}

template <int TM, int BN, int WK, int NBUF, bool STREAM = false, int IM = 2>
int launch_mid(const void* A, const void* B, int M, int N, int Kb, void* C, void* Y, const void* sA, const void* sB,
               const void* bias, hipStream_t st, int ksplit) {
    constexpr int NT = 64 * (TM / 64) * (BN / 64) * WK, BM = TM / 2 * IM;
    constexpr size_t STAGES = (size_t)NBUF * (BM + BN) * 128;
    constexpr size_t XCH = IM == 3 ? (size_t)WK * BM * BN * 4 : (size_t)(TM / 64) * (BN / 64) * WK * (WK == 4 ? 3 : 2) * 4096;
    constexpr size_t LDS = STAGES > XCH ? STAGES : XCH;
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    const int64_t tiles = (int64_t)tiles_m * tiles_n * ksplit;
    if (tiles > 0x3fffffff) return QR_E_SHAPE;
    if ((int64_t)M * Kb >= (1LL << 32) || (int64_t)N * Kb >= (1LL << 32)) return QR_E_UNSUPPORTED;   // (32-bit buffer offsets)
    const int nxcd = qr_device().xcds;                      // the grid is a whole number of rounds over the XCDs
    const unsigned grid = (unsigned)((tiles + nxcd - 1) / nxcd * nxcd);
    auto kern = Y ? gemm_mid_kernel<TM, BN, WK, NBUF, true, STREAM, IM> : gemm_mid_kernel<TM, BN, WK, NBUF, false, STREAM, IM>;
    const hipError_t e = qr_allow_dynamic_lds((const void*)kern, LDS);
    if (e != hipSuccess) return (int)e;
    kern<<<dim3(grid), dim3(NT), LDS, st>>>((const uint8_t*)A, (const uint8_t*)B, M, N, Kb, (int32_t*)C, (f16*)Y, (const f16*)sA,
                                            (const f16*)sB, (const f16*)bias, tiles_m, tiles_n, ksplit, nxcd);
    return qr_launch_status();
}

}  // namespace

// shape: 0 = 64 x 64, 1 = 64 x 128, 2 = 128 x 128 tiles; 3 = 64 x 64 in the STREAM form (M <= 64); 4 = 96 x 64.  Three stage buffers of 16 KB
// let three 64 x 64 workgroups share a CU.  A 64 x 128 or 128 x 128 one has a CU to itself: eight waves exchange 96 KB of
// accumulators through LDS at the end, more than the 72 KB of its three stage buffers, and four buffers are 128 KB.
// One 64 x 64 workgroup to a CU at most and weights beyond 10 MB: four buffers.  Weights that come from memory, as a model's do layer by layer, have
// more to wait for: 256 x 4096 x 11008 19.6 -> 17.1 us, 128 x 5120 x 5120 11.8 -> 10.8, 128 x 8192 x 8192 16.7 -> 14.9, 128 x 8192 x 28672
// 47.7 -> 41.1; out of the last-level cache it is level (15.5 and 15.6, 9.2, 12.7).  (128 x 4096 x 4096 10.2 -> 9.1, but 8.1 -> 8.2 out of that cache, which
// holds thirty of these.  The line is not a capacity: below it a loop over few layers loses 1 %, and a model of many would gain there too.)  With two and three workgroups to a CU three buffers are ahead (512 x 5120 x 5120 18.2 us against 20.1), and
// 64 x 128 with five was no faster (11.8 against 11.2 us at 128 x 4096 x 4096): the loads are bound by rate there.  96 x 64 has a CU to itself as well (the
// exchange is 96 KB) and four waves: four buffers 10.2, five 10.8 us at 333 x 4096 x 4096.  The STREAM form's come from memory:
// with at most a workgroup per CU it takes five buffers, 64 KB in flight (48 x
// 5120 x 13824 in two slices of K 17.8 -> 15.7 us), with more workgroups three (48 x 22016 x 4096 14.3 -> 13.5).  Slices of K are short
// walks, in which every further buffer delays the first stages of all: four (32 x 5120 x 13824 13.5 -> 13.1 us, 48 14.3 -> 14.0, 48 x 5120 x 20480
// 17.6 -> 17.2; three 18.6, six 3 % and eight 7 % slower than five); whole walks are level or better with five (48 x 8192 x 8192 13.1, with four 13.4).
__attribute__((visibility("hidden"))) int qr_internal_gemm_mid(int shape, const void* A, const void* B, int M, int N, int Kb,
                                                               void* C, void* Y, const void* sA, const void* sB,
                                                               const void* bias, hipStream_t st, int ksplit) {
    if (ksplit > 1 && Y) return QR_E_UNSUPPORTED;           // partial sums exist only as int32
    if (shape == 0) {
        if ((int64_t)((M + 63) / 64) * ((N + 63) / 64) * ksplit <= qr_device().cus && (int64_t)N * Kb > 10000000)
            return launch_mid<64, 64, 4, 4>(A, B, M, N, Kb, C, Y, sA, sB, bias, st, ksplit);
        return launch_mid<64, 64, 4, 3>(A, B, M, N, Kb, C, Y, sA, sB, bias, st, ksplit);
    }
    if (shape == 1) return launch_mid<64, 128, 4, 3>(A, B, M, N, Kb, C, Y, sA, sB, bias, st, ksplit);
    if (shape == 4) return launch_mid<64, 64, 4, 4, false, 3>(A, B, M, N, Kb, C, Y, sA, sB, bias, st, ksplit);
    if (shape == 3) {
        if (M > 64) return QR_E_UNSUPPORTED;
        if (ksplit > 1 && (int64_t)((N + 63) / 64) * ksplit <= qr_device().cus)
            return launch_mid<64, 64, 4, 4, true>(A, B, M, N, Kb, C, Y, sA, sB, bias, st, ksplit);
        if ((int64_t)((N + 63) / 64) * ksplit <= qr_device().cus)
            return launch_mid<64, 64, 4, 5, true>(A, B, M, N, Kb, C, Y, sA, sB, bias, st, ksplit);
        return launch_mid<64, 64, 4, 3, true>(A, B, M, N, Kb, C, Y, sA, sB, bias, st, ksplit);
    }
    return launch_mid<128, 128, 2, 4>(A, B, M, N, Kb, C, Y, sA, sB, bias, st, ksplit);
}
