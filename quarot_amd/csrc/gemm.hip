// int4 x int4 -> int32 GEMM on the gfx950 int8 matrix cores, with an optional fused fp16 dequant
// epilogue.  C[M, N] = unpack(A)[M, K] . unpack(B)[N, K]^T, both operands K-contiguous, packed two
// nibbles per byte (even k in the low nibble).
//
// Feeding int4 to an int8 MFMA without sign extension: for a 32-bit word p holding 8 nibbles,
//     lo = (p << 4) & 0xF0F0F0F0   holds 16 * v[even k] in each byte (as a signed int8)
//     hi =  p       & 0xF0F0F0F0   holds 16 * v[odd k]
// Both operands are scaled by 16, so every product is 256 * a * b and the accumulator is exactly
// 256 * (the int4 dot product); an arithmetic shift by 8 at the end restores it.  Even and odd k
// go to different MFMA issues; that permutation of k is the same for A and B, so dot products are
// unchanged.  |acc| <= 256 * 64 * K requires K < 131072.
//
// The MFMA's first operand is the W (B-matrix) fragment and its second the X (A-matrix) fragment,
// so in the 32x32 accumulator a lane owns one token (m = lane % 32) and runs of 4 consecutive
// output features n: stores are 8 bytes (fp16) or 16 bytes (int32) per lane.
//
// Issue budget: a 32x32x32 int8 MFMA occupies the matrix pipe for 32 cycles and a wave's VALU op
// takes 4; measured on MI355X, up to ~5 VALU ops per MFMA are hidden.  Unpacking costs 3 VALU ops per
// packed dword, i.e. 6 (IM + JN) / (IM JN) per MFMA for a wave tile of IM x JN MFMA tiles: 64x128 per
// wave (4.5) is the smallest tile that fits where the matrix pipe is to stay busy.  (Outputs of few tiles, bound by
// the CUs' intake of operands instead, take the 64x64 wave tiles of gemm_mid.hip, and those that fill the CUs with large tiles
// the FP6 matrix path, gemm_e2m3.hip.)
#include "qr_common.h"
#include "qr_epilogue.h"
#include <type_traits>

namespace {

// LDS holds, per stage, (BM + BN) rows of 64 packed bytes (128 k values) as four 16-byte chunks.
// The chunk position is XOR-swizzled with bits 2..3 of the row so that the 16 rows a quarter-wave
// reads in one ds_read_b128 beat fall in 16 different 16-byte bank groups.
__device__ __forceinline__ int lds_slot(int row, int chunk) { return row * 4 + (chunk ^ ((row >> 2) & 3)); }

template <int BM, int BN, int WAVES_M, int WAVES_N, bool DEQ>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N) void gemm_i4_kernel(
    const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, int M, int N, int Kb, int32_t* __restrict__ C,
    f16* __restrict__ Y, const f16* __restrict__ sA, const f16* __restrict__ sB, const f16* __restrict__ bias,
    int tiles_m, int tiles_n, int nxcd) {
    constexpr int NT = 64 * WAVES_M * WAVES_N;              // threads per workgroup
    constexpr int TM = BM / WAVES_M, TN = BN / WAVES_N;     // per-wave output tile
    constexpr int IM = TM / 32, JN = TN / 32;               // 32x32 MFMA tiles per wave
    constexpr int CH = (BM + BN) * 4;                       // 16-byte chunks per stage
    constexpr int NL = (CH + NT - 1) / NT;                  // chunks each thread moves per stage
    static_assert(TM % 32 == 0 && TN % 32 == 0, "tile shape");
    // two stage buffers; the same memory later stages the fp16 output slabs (one per wave)
    constexpr int SLAB = 32 * 64 * 2 / 16;                  // 16-byte units of a 32-row x 64-column fp16 slab
    static_assert(2 * CH >= WAVES_M * WAVES_N * SLAB, "output slabs must fit in the stage buffers");
    __shared__ u32x4 lds_raw[2 * CH];
    u32x4(*lds)[CH] = (u32x4(*)[CH])lds_raw;

    // Workgroups are dealt round-robin to the nxcd XCDs (each with its own L2).  Give every XCD a
    // contiguous range of tile ids, and walk tiles in groups of GROUP_M rows so that the tiles in
    // flight on one XCD share A rows and B rows.
    const int per_xcd = gridDim.x / nxcd;
    int tile = (blockIdx.x % nxcd) * per_xcd + blockIdx.x / nxcd;
    if (tile >= tiles_m * tiles_n) return;
    constexpr int GROUP_M = 8;
    const int group_sz = GROUP_M * tiles_n;
    const int g = tile / group_sz;
    const int gm0 = g * GROUP_M;
    const int gh = (tiles_m - gm0) < GROUP_M ? (tiles_m - gm0) : GROUP_M;
    const int tm = gm0 + (tile - g * group_sz) % gh;
    const int tn = (tile - g * group_sz) / gh;
    const int m0 = tm * BM, n0 = tn * BN;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;

    // Global -> LDS staging: chunk id = tid + i * NT; 4 consecutive threads fetch one row's 64 bytes.
    // Rows beyond M (or N) are clamped to the last valid row: they are read but never stored.
    const uint8_t* src[NL];
    int dst[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        int qid = tid + i * NT;
        if (qid >= CH) qid = CH - 1;        // CH not a multiple of NT: the tail repeats the last chunk
        const int row = qid >> 2, c = qid & 3;
        if (row < BM) {
            int gr = m0 + row;
            gr = gr < M ? gr : M - 1;
            src[i] = A + (int64_t)gr * Kb + c * 16;
        } else {
            int gr = n0 + row - BM;
            gr = gr < N ? gr : N - 1;
            src[i] = B + (int64_t)gr * Kb + c * 16;
        }
        dst[i] = lds_slot(row, c);
    }

    i32x16 acc[IM][JN];
#pragma unroll
    for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0;

    const int arow = wm * TM + (lane & 31);
    const int brow = BM + wn * TN + (lane & 31);
    const int khalf = lane >> 5;

    // One stage = 64 packed bytes per row = two sub-steps of 64 k values (two MFMA issues each).
    auto compute = [&](const u32x4* buf, int nsub) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if (s < nsub) {
                i32x4 alo[IM], ahi[IM], blo[JN], bhi[JN];
#pragma unroll
                for (int i = 0; i < IM; ++i) {
                    u32x4 p = buf[lds_slot(arow + i * 32, s * 2 + khalf)];
                    alo[i] = (i32x4)((p << 4) & 0xF0F0F0F0u);
                    ahi[i] = (i32x4)(p & 0xF0F0F0F0u);
                }
#pragma unroll
                for (int j = 0; j < JN; ++j) {
                    u32x4 p = buf[lds_slot(brow + j * 32, s * 2 + khalf)];
                    blo[j] = (i32x4)((p << 4) & 0xF0F0F0F0u);
                    bhi[j] = (i32x4)(p & 0xF0F0F0F0u);
                }
                // all even-k issues first, then all odd-k ones: consecutive MFMAs never share an accumulator
#pragma unroll
                for (int i = 0; i < IM; ++i)
#pragma unroll
                    for (int j = 0; j < JN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(blo[j], alo[i], acc[i][j], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < IM; ++i)
#pragma unroll
                    for (int j = 0; j < JN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bhi[j], ahi[i], acc[i][j], 0, 0, 0);
            }
        }
    };

    // K % 64 == 0, so a row is a whole number of 32-byte half-stages: `full` whole stages, then
    // possibly one half stage (chunks 0 and 1 only).
    const int full = Kb / 64;
    const bool half_tail = (Kb & 63) != 0;
    // Global loads run TWO stages ahead of the MFMAs (HBM/L2 latency exceeds one stage of compute):
    // stage ks+2 is requested into one register set at the top of iteration ks, while the other
    // set (stage ks+1, requested an iteration earlier) is written to LDS at the bottom.
    u32x4 preA[NL], preB[NL];
    if (full > 0) {
#pragma unroll
        for (int i = 0; i < NL; ++i) preA[i] = *(const u32x4*)(src[i]);
#pragma unroll
        for (int i = 0; i < NL; ++i) lds[0][dst[i]] = preA[i];
    }
    if (full > 1) {
#pragma unroll
        for (int i = 0; i < NL; ++i) preA[i] = *(const u32x4*)(src[i] + 64);      // stage 1
    }
    __syncthreads();
    auto iteration = [&](int ks, u32x4(&cur)[NL], u32x4(&nxt)[NL]) {
        // `cur` holds stage ks+1 (in flight or landed); `nxt` receives stage ks+2
        if (ks + 2 < full) {
#pragma unroll
            for (int i = 0; i < NL; ++i) nxt[i] = *(const u32x4*)(src[i] + (int64_t)(ks + 2) * 64);
        }
        compute(lds[ks & 1], 2);
        if (ks + 1 < full) {
#pragma unroll
            for (int i = 0; i < NL; ++i) lds[(ks + 1) & 1][dst[i]] = cur[i];
        }
        __syncthreads();
    };
    {
        int ks = 0;
        for (; ks + 1 < full; ks += 2) {
            iteration(ks, preA, preB);
            iteration(ks + 1, preB, preA);
        }
        if (ks < full) iteration(ks, preA, preB);
    }
#pragma unroll
    for (int i = 0; i < NL; ++i) src[i] += (int64_t)(full > 0 ? full - 1 : 0) * 64;   // last full stage
    if (half_tail) {
        // chunks 2 and 3 of this last stage lie beyond the row: only chunks 0/1 are fetched and used
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            int qid = tid + i * NT;
            if (qid >= CH) qid = CH - 1;
            if ((qid & 3) < 2) lds[0][dst[i]] = *(const u32x4*)(src[i] + (full > 0 ? 64 : 0));
        }
        __syncthreads();
        compute(lds[0], 1);
    }

    // Epilogue.  Accumulator layout (first operand = W rows, second = X rows): lane l, register v ->
    // n = (v/4)*8 + (l/32)*4 + v%4, m = l%32.
    // Tiles of an fp16 output whose columns all exist leave as full rows through LDS, 64 columns (one
    // line) at a time; a last row tile stores the rows that exist.
    const bool by_rows = DEQ && n0 + BN <= N && (N & 7) == 0 && (((uintptr_t)Y) & 15) == 0;
    if (DEQ && by_rows) {
        constexpr int NJ = JN > 2 ? 2 : JN;                 // MFMA tiles per slab
        __syncthreads();                                    // every wave is done with the stage buffers
#pragma unroll
        for (int jb = 0; jb < JN; jb += NJ) {
            f16x4 sbh[NJ][4], bih[NJ][4];
#pragma unroll
            for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
                for (int gq = 0; gq < 4; ++gq) {
                    const int col = n0 + wn * TN + (jb + jj) * 32 + gq * 8 + khalf * 4;
                    sbh[jj][gq] = *(const f16x4*)(sB + col);
                    bih[jj][gq] = bias ? *(const f16x4*)(bias + col) : f16x4{(f16)0, (f16)0, (f16)0, (f16)0};
                }
#pragma unroll
            for (int i = 0; i < IM; ++i) {
                const int row0 = m0 + wm * TM + i * 32;       // (rows past M: computed on a clamped scale, not stored)
                if (row0 >= M) continue;
                const f16 sa = sA[min(row0 + (lane & 31), M - 1)];
                f16x4 o[NJ][4];
#pragma unroll
                for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
                    for (int gq = 0; gq < 4; ++gq)
                        o[jj][gq] = dequant4(acc[i][jb + jj][gq * 4], acc[i][jb + jj][gq * 4 + 1], acc[i][jb + jj][gq * 4 + 2],
                                             acc[i][jb + jj][gq * 4 + 3], sa, sbh[jj][gq], bih[jj][gq], bias != nullptr);
                store_slab_rows<NJ>((u32x2*)(lds_raw + wave * SLAB), o, lane,
                                    Y + (int64_t)row0 * N + n0 + wn * TN + jb * 32, N, M - row0);
            }
        }
        return;
    }
    // column scales (and bias) of this lane's 4-column groups, fetched up front as 8-byte vectors
    f16x4 sb4[JN][4], bi4[JN][4];
    if (DEQ) {
#pragma unroll
        for (int j = 0; j < JN; ++j)
#pragma unroll
            for (int gq = 0; gq < 4; ++gq) {
                const int col = n0 + wn * TN + j * 32 + gq * 8 + khalf * 4;
                if (col + 4 <= N && (N & 3) == 0) {
                    sb4[j][gq] = *(const f16x4*)(sB + col);
                    if (bias) bi4[j][gq] = *(const f16x4*)(bias + col);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int cc = col + e < N ? col + e : N - 1;
                        sb4[j][gq][e] = sB[cc];
                        if (bias) bi4[j][gq][e] = bias[cc];
                    }
                }
            }
    }
#pragma unroll
    for (int i = 0; i < IM; ++i) {
        const int row = m0 + wm * TM + i * 32 + (lane & 31);
        if (row >= M) continue;
        f16 sa = (f16)0;
        if (DEQ) sa = sA[row];
#pragma unroll
        for (int j = 0; j < JN; ++j) {
#pragma unroll
            for (int gq = 0; gq < 4; ++gq) {
                const int col = n0 + wn * TN + j * 32 + gq * 8 + khalf * 4;
                if (col >= N) continue;
                int v4[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v4[e] = acc[i][j][gq * 4 + e] >> 8;
                const bool whole = (col + 4 <= N) && ((N & 3) == 0);
                if (DEQ) {
                    f16 o[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        f16 yv = (f16)(sa * sb4[j][gq][e]) * (f16)(float)v4[e];
                        if (bias) yv = yv + bi4[j][gq][e];
                        o[e] = yv;
                    }
                    f16* yp = Y + (int64_t)row * N + col;
                    if (whole) {
                        *(f16x4*)yp = f16x4{o[0], o[1], o[2], o[3]};
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (col + e < N) yp[e] = o[e];
                    }
                } else {
                    int32_t* cp = C + (int64_t)row * N + col;
                    if (whole) {
                        *(i32x4*)cp = i32x4{v4[0], v4[1], v4[2], v4[3]};
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (col + e < N) cp[e] = v4[e];
                    }
                }
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------
// Decode (M <= 64) with too few column tiles for the tiled kernels, or few tokens.  A workgroup of
// eight waves owns 8 / KW groups of 32 weight rows; the KW waves of a group split K into contiguous
// ranges and their partial 32 x M tiles are summed through LDS and dequantised (KW = 8 when K is
// long and N small, 2 or 4 when a wave would otherwise get only a handful of steps).  Nothing is shared between waves in the main loop, so there
// are no barriers in it: every wave streams its own slices of W and X with coalesced 16-byte loads
// (SB / 16 lanes per row piece of SB bytes, PF steps ahead in a register ring) and turns them into
// MFMA fragments (lane = row) through a wave-private LDS buffer.  Loading fragments straight from
// global memory makes every instruction touch 32 different lines and was measured 1.5-2x slower.
// XL = load instructions per step that carry rows of X (64 / CPR rows each): with few tokens only
// the first ceil(M / (64 / CPR)) of them are issued and staged; the remaining rows of the 32-row
// MFMA operand keep whatever the buffer holds, and the output rows they produce are never stored.
template <int MT, int SB, int XL, int PF, int KW, bool DEQ>
__global__ __launch_bounds__(512) void decode_i4_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B,
                                                        int M, int N, int Kb, int32_t* __restrict__ C,
                                                        f16* __restrict__ Y, const f16* __restrict__ sA,
                                                        const f16* __restrict__ sB, const f16* __restrict__ bias) {
    constexpr int CPR = SB / 16;                            // 16-byte chunks per row and step (4, 8 or 16)
    constexpr int ROWS = (1 + MT) * 32;                     // staged rows per wave: 32 of W, then 32 MT of X
    constexpr int NLW = 32 * CPR / 64;                      // chunks per lane and step: rows of W ...
    constexpr int NLD = NLW + XL;                           // ... plus the rows of X that exist
    static_assert(XL >= 1 && XL <= MT * 32 * CPR / 64, "X load groups");
    constexpr int STAGE = ROWS * CPR;                       // u32x4 per wave
    constexpr int RED = MT * 4 * 64;                        // i32x4 per wave for the final sum
    extern __shared__ u32x4 dec_smem[];                     // 8 * max(STAGE, RED)
    i32x4* red = (i32x4*)dec_smem;                          // [wave][m tile][4-register group][lane]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 31, h = lane >> 5;
    constexpr int RG = 8 / KW;                              // groups of 32 weight rows per workgroup
    const int kw = wave % KW;                               // this wave's share of K within its row group
    const int n0 = (blockIdx.x * RG + wave / KW) * 32;
    const int steps = (Kb + SB - 1) / SB;
    const int s_begin = (int)((int64_t)steps * kw / KW), s_end = (int)((int64_t)steps * (kw + 1) / KW);
    u32x4* stage = dec_smem + wave * STAGE;
    // chunk position XOR-keyed by the row: the 16 rows of a fragment read spread over all bank groups
    auto slot = [](int row, int chunk) {
        return CPR == 4 ? row * 4 + (chunk ^ ((row >> 2) & 3))
               : CPR == 8 ? row * 8 + (chunk ^ ((row >> 1) & 7)) : row * 16 + (chunk ^ (row & 15));
    };

    // chunk i of this lane: row (lane + 64 i) / CPR, 16-byte piece lane % CPR
    const int piece = lane % CPR;
    const uint8_t* src[NLD];
    int dst[NLD];
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int row = lane / CPR + (64 / CPR) * i;
        if (row < 32) {
            int nr = n0 + row;
            nr = nr < N ? nr : N - 1;
            src[i] = B + (int64_t)nr * Kb;
        } else {
            int mr = row - 32;
            mr = mr < M ? mr : M - 1;
            src[i] = A + (int64_t)mr * Kb;
        }
        dst[i] = slot(row, piece);
    }
    // K % 64 == 0: a row is a whole number of 32-byte pairs of pieces.  Pieces of the last step that
    // lie beyond the row re-read piece 0 or 1 of that step and are deposited as zeros.
    struct Step {
        u32x4 v[NLD];
    };
    auto fetch = [&](int sidx, Step& st) {
        const int sc = sidx < steps ? sidx : steps - 1;
        const bool dead = sc * SB + piece * 16 >= Kb;
        const int off = sc * SB + (dead ? (piece & 1) : piece) * 16;
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            // weights are used once: streaming loads keep the tokens' codes, which every workgroup
            // re-reads, in the caches
            if (i < NLW) st.v[i] = __builtin_nontemporal_load((const u32x4*)(src[i] + off));
            else st.v[i] = *(const u32x4*)(src[i] + off);
        }
    };
    i32x16 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[t][v] = 0;
    auto deposit = [&](int sidx, const Step& st) {
        const bool dead = sidx * SB + piece * 16 >= Kb;
        // LDS operations of one wave execute in order: these writes follow the previous step's reads
#pragma unroll
        for (int i = 0; i < NLD; ++i) stage[dst[i]] = dead ? u32x4{0, 0, 0, 0} : st.v[i];
    };
    auto multiply = [&]() {
#pragma unroll
        for (int c = 0; c < CPR / 2; ++c) {                 // lane half h takes pieces 2c + h of both operands
            const u32x4 wq = stage[slot(r, 2 * c + h)];
            const i32x4 wlo = (i32x4)((wq << 4) & 0xF0F0F0F0u), whi = (i32x4)(wq & 0xF0F0F0F0u);
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                const u32x4 xq = stage[slot(32 + t * 32 + r, 2 * c + h)];
                const i32x4 xlo = (i32x4)((xq << 4) & 0xF0F0F0F0u), xhi = (i32x4)(xq & 0xF0F0F0F0u);
                acc[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wlo, xlo, acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(whi, xhi, acc[t], 0, 0, 0);
            }
        }
    };
    Step ring[PF];
#pragma unroll
    for (int p = 0; p < PF; ++p) fetch(s_begin + p, ring[p]);
    // whole turns of the ring run without a branch, so that every wait inside them counts exactly the
    // loads issued after the step it needs (a branch in the loop body makes the compiler wait for all
    // outstanding loads once per turn)
    // The loads that refill a ring slot are issued as soon as the slot has been written to LDS, before
    // the step's multiplications; the scheduling barriers keep the compiler from moving them later.
    int s = s_begin;
    for (; s + PF <= s_end; s += PF) {
#pragma unroll
        for (int p = 0; p < PF; ++p) {
            deposit(s + p, ring[p]);
            __builtin_amdgcn_sched_barrier(0);
            fetch(s + p + PF, ring[p]);                     // indices past the end re-read the last step (unused)
            __builtin_amdgcn_sched_barrier(0);
            multiply();
        }
    }
#pragma unroll
    for (int p = 0; p < PF - 1; ++p)
        if (s + p < s_end) {
            deposit(s + p, ring[p]);
            multiply();
        }
    __syncthreads();                                        // the staging buffers become the reduction buffer
    // ---- sum the eight partial tiles
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int gq = 0; gq < 4; ++gq)
            red[((wave * MT + t) * 4 + gq) * 64 + lane] = i32x4{acc[t][gq * 4], acc[t][gq * 4 + 1], acc[t][gq * 4 + 2], acc[t][gq * 4 + 3]};
    __syncthreads();
    // unit u = (row group, m tile, register group): the waves take them in turn
    for (int u = wave; u < RG * MT * 4; u += 8) {
        const int g = u / (MT * 4), t = (u >> 2) % MT, gq = u & 3;
        i32x4 sum = {0, 0, 0, 0};
#pragma unroll
        for (int w = 0; w < KW; ++w) sum += red[(((g * KW + w) * MT + t) * 4 + gq) * 64 + lane];
        const int row = t * 32 + r;
        const int col = (blockIdx.x * RG + g) * 32 + gq * 8 + h * 4;
        if (row < M && col < N) {
            const bool whole = (col + 4 <= N) && ((N & 3) == 0);
            if (DEQ) {
                const f16 sa = sA[row];
                f16 o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int cc = col + e < N ? col + e : N - 1;
                    f16 yv = (f16)(sa * sB[cc]) * (f16)(float)(sum[e] >> 8);
                    if (bias) yv = yv + bias[cc];
                    o[e] = yv;
                }
                f16* yp = Y + (int64_t)row * N + col;
                if (whole) {
                    *(f16x4*)yp = f16x4{o[0], o[1], o[2], o[3]};
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (col + e < N) yp[e] = o[e];
                }
            } else {
                int32_t* cp = C + (int64_t)row * N + col;
                if (whole) {
                    *(i32x4*)cp = i32x4{sum[0] >> 8, sum[1] >> 8, sum[2] >> 8, sum[3] >> 8};
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (col + e < N) cp[e] = sum[e] >> 8;
                }
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------
// Decode (M <= 64) with many weight rows: a workgroup owns R groups of 32 weight rows (R = 4 .. 8,
// chosen by the host so that the workgroups spread evenly over the CUs: 57344 rows are 256 workgroups
// of 7 groups) and walks K in stages of 128 packed bytes per row.
// * Twelve waves in two roles.  Waves 8..11 only FETCH: eight consecutive threads one 128-byte line,
//   MT + R chunks per thread and stage, into RD register sets that rotate RD stages ahead of the LDS
//   fill; three LDS stage buffers rotate; one barrier per stage.  Waves 0..R-1 only MULTIPLY: wave w
//   takes row group w against all tokens.  With every wave doing both, a wave waits for its loads and
//   then multiplies, the whole CU in step: the multiplications were not hidden behind the memory time
//   (64 tokens: 47 us; with the roles split 42 us, the same as 8 tokens).
// * The tokens' codes are fetched ONCE per workgroup and stage and shared through LDS -- with
//   wave-private staging every wave would pull its own copy through the vector cache, twice the weight
//   bytes at 64 tokens -- and the thread that fetched a chunk of them stores it already unpacked into
//   its two int8 planes, so that no multiplying wave unpacks tokens.
// * The multiplications are software-pipelined over the 64-k sub-steps (see `substep`).
// * Workgroup b starts its walk over K at stage b % stages and wraps around (integer sums do not depend
//   on the order): with a row pitch that is a power of two, workgroups marching through K in step
//   would all be reading the same few memory channels at any one time (measured 49 -> 41 us at
//   57344 x 8192).  With such a pitch, stage b / 8: 7 tokens x 28672 x 8192 22.2 -> 21.9 us, 24 22.2 -> 21.6, 7 x 57344 x 8192 39.2 -> 38.2,
//   16 x 28672 x 4096 13.0 -> 12.7; with others it is no better (32 x 27648 x 5120 16.2 -> 16.5).
template <int MT, int R, int RD, bool DEQ>
__global__ __launch_bounds__(768) void decode_xs_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B,
                                                        int M, int N, int Kb, int32_t* __restrict__ C,
                                                        f16* __restrict__ Y, const f16* __restrict__ sA,
                                                        const f16* __restrict__ sB, const f16* __restrict__ bias) {
    constexpr int XR = MT * 32;                             // staged rows of X
    constexpr int NL = MT + R;                              // 16-byte chunks per loader thread and stage: 32 rows each
    constexpr int XPLANES = XR * 16;                        // slots of the tokens' planes (32 bytes per packed chunk)
    constexpr int CH = XPLANES + R * 32 * 8;                // slots per stage buffer
    constexpr int NBUF = 3;
    extern __shared__ u32x4 xs_lds[];                       // [NBUF][CH]; later the output slabs
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 31, h = lane >> 5;
    const bool loader = wave >= 8;                          // waves 8..11 fetch, waves 0..R-1 multiply
    const int n0 = blockIdx.x * (R * 32);
    const int stages = (Kb + 127) / 128;
    const bool ragged = (Kb & 127) != 0;
    auto slot8 = [](int row, int chunk) { return row * 8 + (chunk ^ ((row >> 1) & 7)); };
    auto slot16 = [](int row, int chunk, int plane) {
        return row * 16 + ((chunk ^ (row & 7)) << 1) + (plane ^ ((row >> 3) & 1));
    };

    const int ltid = tid & 255;
    const int srow = ltid >> 3, piece = ltid & 7;           // chunk i of a loader thread: row srow + 32 i, same piece
    const uint8_t* src[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        if (i < MT) {
            const int mr = srow + 32 * i;
            src[i] = A + (int64_t)(mr < M ? mr : M - 1) * Kb;
        } else {
            const int nr = n0 + srow + 32 * (i - MT);
            src[i] = B + (int64_t)(nr < N ? nr : N - 1) * Kb;
        }
    }
    const int wdst0 = XPLANES + slot8(srow, piece);         // rows differ by multiples of 32: same swizzle
    const int xdst0 = slot16(srow, piece, 0);
    // (consecutive workgroups are on different XCDs: the eight of a run start together, those of an XCD one stage after the other)
    const int s0 = ((Kb & (Kb - 1)) == 0 ? blockIdx.x >> 3 : blockIdx.x) % stages;
    auto stage_of = [&](int st) {                           // absolute stage of this workgroup's st-th step
        const int a = (st < stages ? st : stages - 1) + s0;
        return a >= stages ? a - stages : a;
    };
    auto fetch = [&](int st, u32x4(&v)[NL]) {
        const int kb = stage_of(st) * 128;
        const int off = (kb + piece * 16 < Kb) ? kb + piece * 16 : kb;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            // weights are used once: streaming loads keep the tokens' codes, which every workgroup
            // re-reads, in the caches
            if (i >= MT) v[i] = __builtin_nontemporal_load((const u32x4*)(src[i] + off));
            else v[i] = *(const u32x4*)(src[i] + off);
        }
    };
    // stages past the end are written too (into a buffer nobody reads again): without a branch every
    // wait counts exactly the loads issued after the ones it needs
    auto deposit = [&](int st, int buf, const u32x4(&v)[NL]) {
        const bool zero = ragged && stage_of(st) * 128 + piece * 16 >= Kb;
        u32x4* base = xs_lds + buf * CH;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const u32x4 q = zero ? u32x4{0, 0, 0, 0} : v[i];
            if (i < MT) {
                base[xdst0 + i * 32 * 16] = (q << 4) & 0xF0F0F0F0u;
                base[(xdst0 ^ 1) + i * 32 * 16] = q & 0xF0F0F0F0u;
            } else {
                base[wdst0 + (i - MT) * 32 * 8] = q;
            }
        }
    };
    i32x16 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[t][v] = 0;
    // logical chunk 2u + h of weight row q sits at slot8(q, h) ^ (2u); plane p of a token row's chunk
    // 2u + h at slot16(q, h, 0) ^ (4u + p): the swizzles only touch the low bits
    const bool computes = wave < R;                         // (waves R..7 only keep the barriers' count)
    const int wslot = XPLANES + slot8((computes ? wave : 0) * 32 + r, h), xslot = slot16(r, h, 0);
    // The multiplications are software-pipelined over the 64-k sub-steps: while the 2 MT MFMAs of one
    // sub-step run, the operands of the next one (the first of the next stage after the last: that
    // buffer became visible with the previous barrier) are read from LDS and the weights unpacked.
    // Written as slots of one MFMA plus its share of the reads and unpacking, with a scheduling barrier
    // after every slot: left to itself the compiler reads, unpacks and multiplies in three phases, and
    // with the two waves of a SIMD in step after every barrier the three pipes then take turns
    // (measured: LDS, vector and matrix time added up to the whole launch).
    struct Ops {
        u32x4 w;
        i32x4 wlo, whi, xlo[MT], xhi[MT];
    };
    Ops ops[2];
    auto read_w = [&](const u32x4* base, int uu, Ops& o) { o.w = base[wslot ^ (2 * uu)]; };
    auto read_x = [&](const u32x4* base, int uu, int t, int plane, Ops& o) {
        const i32x4 q = (i32x4)base[(xslot ^ (4 * uu + plane)) + t * 32 * 16];
        if (plane) o.xhi[t] = q;
        else o.xlo[t] = q;
    };
    auto unpack_lo = [&](Ops& o) { o.wlo = (i32x4)((o.w << 4) & 0xF0F0F0F0u); };
    auto unpack_hi = [&](Ops& o) { o.whi = (i32x4)(o.w & 0xF0F0F0F0u); };
    auto substep = [&](const Ops& cur, Ops& nxt, const u32x4* nbase, int nu) {
        // slot 0
        acc[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(cur.wlo, cur.xlo[0], acc[0], 0, 0, 0);
        read_w(nbase, nu, nxt);
        read_x(nbase, nu, 0, 0, nxt);
        if (MT == 1) read_x(nbase, nu, 0, 1, nxt);
        __builtin_amdgcn_sched_barrier(0);
        if (MT == 2) {
            acc[MT - 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(cur.wlo, cur.xlo[MT - 1], acc[MT - 1], 0, 0, 0);
            read_x(nbase, nu, 0, 1, nxt);
            read_x(nbase, nu, MT - 1, 0, nxt);
            __builtin_amdgcn_sched_barrier(0);
        }
        acc[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(cur.whi, cur.xhi[0], acc[0], 0, 0, 0);
        if (MT == 2) read_x(nbase, nu, MT - 1, 1, nxt);
        unpack_lo(nxt);
        if (MT == 1) unpack_hi(nxt);
        __builtin_amdgcn_sched_barrier(0);
        if (MT == 2) {
            acc[MT - 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(cur.whi, cur.xhi[MT - 1], acc[MT - 1], 0, 0, 0);
            unpack_hi(nxt);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    if (loader) {
        u32x4 regs[RD][NL];
#pragma unroll
        for (int q = 0; q < RD; ++q) fetch(q, regs[q]);
        deposit(0, 0, regs[0]);
        fetch(RD, regs[0]);
        deposit(1, 1, regs[1 % RD]);
        fetch(RD + 1, regs[1 % RD]);
        __syncthreads();                                    // stages 0 and 1 visible
        int bfill = 2;
        auto iteration = [&](int ks, u32x4(&v)[NL]) {
            deposit(ks + 2, bfill, v);
            __builtin_amdgcn_sched_barrier(0);
            fetch(ks + 2 + RD, v);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            bfill = bfill == NBUF - 1 ? 0 : bfill + 1;
        };
        int ks0 = 0;
        for (; ks0 + RD <= stages; ks0 += RD) {
#pragma unroll
            for (int q = 0; q < RD; ++q) iteration(ks0 + q, regs[(q + 2) % RD]);
        }
#pragma unroll
        for (int q = 0; q < RD - 1; ++q)
            if (ks0 + q < stages) iteration(ks0 + q, regs[(q + 2) % RD]);
        return;
    }
    // The outputs' scales and bias, read here, where a multiplying wave waits for the first stages anyway: behind the loop they
    // were a memory latency at the end of every launch (7 tokens x 28672 x 8192 23.5 -> 22.6 us, 48 27.6 -> 26.5,
    // 7 x 57344 x 8192 39.0 -> 38.0; in decode_i4_kernel, whose waves all stream, they stand in front of the stream and cost 2 %).
    const int c0 = n0 + wave * 32;
    f16x4 sb4[4], bi4[4];
    f16 sa[MT];
    if (DEQ && computes) {
#pragma unroll
        for (int gq = 0; gq < 4; ++gq)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int col = c0 + gq * 8 + h * 4 + e, cc = col < N ? col : N - 1;
                sb4[gq][e] = sB[cc];
                bi4[gq][e] = bias ? bias[cc] : (f16)0;
            }
#pragma unroll
        for (int t = 0; t < MT; ++t) sa[t] = sA[t * 32 + r < M ? t * 32 + r : M - 1];
    }
    __syncthreads();                                        // stages 0 and 1 visible
    if (computes) {
        read_w(xs_lds, 0, ops[0]);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            read_x(xs_lds, 0, t, 0, ops[0]);
            read_x(xs_lds, 0, t, 1, ops[0]);
        }
        unpack_lo(ops[0]);
        unpack_hi(ops[0]);
    }
    {
        int bcur = 0;
        for (int ks = 0; ks < stages; ++ks) {
            const int bnext = bcur == NBUF - 1 ? 0 : bcur + 1;
            if (computes) {
                const u32x4* cb = xs_lds + bcur * CH;
                substep(ops[0], ops[1], cb, 1);
                substep(ops[1], ops[0], cb, 2);
                substep(ops[0], ops[1], cb, 3);
                substep(ops[1], ops[0], xs_lds + bnext * CH, 0);   // after the last stage: read, never used
            }
            __syncthreads();
            bcur = bnext;
        }
    }

    // ---- epilogue: lane l, register v -> weight row (v/4)*8 + (l/32)*4 + v%4 of the group, token l%32
    auto finish = [&](const i32x16& a, int t) {
        const int row = t * 32 + r;
        const bool by_rows = DEQ && c0 + 32 <= N && (N & 7) == 0 && (((uintptr_t)Y) & 15) == 0 && t * 32 + 32 <= M;
        if (DEQ && by_rows) {
            f16x4 o[1][4];
#pragma unroll
            for (int gq = 0; gq < 4; ++gq)
                o[0][gq] = dequant4(a[gq * 4], a[gq * 4 + 1], a[gq * 4 + 2], a[gq * 4 + 3], sa[t], sb4[gq], bi4[gq], bias != nullptr);
            store_slab_rows<1>((u32x2*)(xs_lds + wave * 128), o, lane, Y + (int64_t)(t * 32) * N + c0, N);
            return;
        }
        if (row >= M) return;
#pragma unroll
        for (int gq = 0; gq < 4; ++gq) {
            const int col = c0 + gq * 8 + h * 4;
            if (col >= N) continue;
            const bool whole = (col + 4 <= N) && ((N & 3) == 0);
            if (DEQ) {
                const f16x4 o = dequant4(a[gq * 4], a[gq * 4 + 1], a[gq * 4 + 2], a[gq * 4 + 3], sa[t], sb4[gq], bi4[gq],
                                         bias != nullptr);
                f16* yp = Y + (int64_t)row * N + col;
                if (whole) {
                    *(f16x4*)yp = o;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (col + e < N) yp[e] = o[e];
                }
            } else {
                int32_t* cp = C + (int64_t)row * N + col;
                if (whole) {
                    *(i32x4*)cp = i32x4{a[gq * 4] >> 8, a[gq * 4 + 1] >> 8, a[gq * 4 + 2] >> 8, a[gq * 4 + 3] >> 8};
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (col + e < N) cp[e] = a[gq * 4 + e] >> 8;
                }
            }
        }
    };
    if (!computes) return;
#pragma unroll
    for (int t = 0; t < MT; ++t) finish(acc[t], t);
}

// ------------------------------------------------------------------------------------------------
// Decode with very few tokens (M <= 8): a matrix-vector style kernel on the native int4 dot product
// (v_dot8_i32_i4: eight signed 4-bit products per lane and instruction, no unpacking).  A wave owns
// groups of four weight rows and walks K in 1 KB segments: lane l loads bytes [l*16, l*16+16) of
// each row's segment -- every load instruction reads 1 KB of contiguous weight bytes -- and the
// matching 16 bytes of each token's codes (shared by the four rows, L1/L2 resident).  A wave takes
// `ng` consecutive row groups as one flattened sequence of segments, so the loads of the next group
// are already in flight while the current one finishes.  The 64 partial sums of each (row, token)
// pair are added across the wave by a halving exchange (each step gives away half of the values a
// lane still holds), which costs one cross-lane move per value instead of six.
template <int MB, bool DEQ>
__global__ __launch_bounds__(256) void gemv_i4_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B,
                                                      int M, int N, int Kb, int ng, int32_t* __restrict__ C,
                                                      f16* __restrict__ Y, const f16* __restrict__ sA,
                                                      const f16* __restrict__ sB, const f16* __restrict__ bias) {
    constexpr int R = 4;                                    // rows per group
    constexpr int NV = R * MB;                              // sums per group
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g0 = (blockIdx.x * 4 + wave) * ng;            // first row group of this wave
    const int groups = (N + R - 1) / R;
    if (g0 >= groups) return;
    const int gcount = groups - g0 < ng ? groups - g0 : ng;
    const int nseg = (Kb + 1023) / 1024;
    const int total = gcount * nseg;                        // flattened (group, segment) items
    const uint8_t* xp[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        const int mr = m < M ? m : M - 1;
        xp[m] = A + (int64_t)mr * Kb + lane * 16;
    }
    // which of a group's NV sums this lane stores at the end of the exchange below (log2(NV) lane
    // bits from bit 5 downwards), and its token's scale
    constexpr int LV = NV == 4 ? 2 : NV == 8 ? 3 : NV == 16 ? 4 : 5;
    const int vidx = lane >> (6 - LV);
    const int my_m = vidx / R, my_r = vidx % R;
    f16 my_sa = (f16)0;
    if (DEQ) my_sa = sA[my_m < M ? my_m : M - 1];
    struct Seg {
        u32x4 w[R], x[MB];
        f16 sb, bi;                                         // column scale and bias of the lane's output
    };
    // fetch side: position (fg, fs) runs ahead of the consume side
    int fg = 0, fs = 0;
    auto fetch = [&](Seg& g) {
        // a lane whose 16 bytes lie beyond the row end re-reads the row start and contributes nothing;
        // items past the end of the sequence re-read the last one
        const int off = (fs * 1024 + lane * 16 < Kb) ? fs * 1024 + lane * 16 : 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            int nr = (g0 + fg) * R + r;
            nr = nr < N ? nr : N - 1;
            g.w[r] = __builtin_nontemporal_load((const u32x4*)(B + (int64_t)nr * Kb + off));
        }
#pragma unroll
        for (int m = 0; m < MB; ++m) g.x[m] = *(const u32x4*)(xp[m] - lane * 16 + off);
        // every segment carries its group's scale along: loading it at the group's end would make
        // the wave wait for everything it has in flight
        if (DEQ) {
            int col = (g0 + fg) * R + my_r;
            col = col < N ? col : N - 1;
            g.sb = sB[col];
            g.bi = (bias ? bias : sB)[col];                 // (no bias: a harmless second read of the scale)
        }
        if (fs + 1 < nseg) ++fs;
        else if (fg + 1 < gcount) { ++fg; fs = 0; }
    };
    int acc[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[v] = 0;
    int cg = 0, cs = 0;
    auto consume = [&](const Seg& g) {
        // lanes beyond the row end multiply by zero (no branch around the products: a branch here
        // makes the compiler wait for every outstanding load once per turn of the ring)
        const bool live = cs * 1024 + lane * 16 < Kb;
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const int xv = live ? (int)g.x[m][d] : 0;
#pragma unroll
                for (int r = 0; r < R; ++r)
                    acc[m * R + r] = __builtin_amdgcn_sdot8((int)g.w[r][d], xv, acc[m * R + r], false);
            }
        if (++cs < nseg) return;
        // ---- end of a row group: halving exchange.  After the steps with offsets 32, 16, ... a lane
        // holds the sum of value index (bits of its lane id, most significant first) over the lanes
        // that agree with it on those bits; the remaining offsets finish the sum.
        int vals[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) vals[v] = acc[v];
        int off = 32;
#pragma unroll
        for (int cur = NV; cur > 1; cur >>= 1) {
            const bool upper = (lane & off) != 0;
#pragma unroll
            for (int i = 0; i < cur / 2; ++i) {
                const int give = upper ? vals[i] : vals[i + cur / 2];
                const int keep = upper ? vals[i + cur / 2] : vals[i];
                vals[i] = keep + __shfl_xor(give, off, QR_WAVE);
            }
            off >>= 1;
        }
        int sum = vals[0];
        for (; off > 0; off >>= 1) sum += __shfl_xor(sum, off, QR_WAVE);
        if ((lane & ((1 << (6 - LV)) - 1)) == 0) {
            const int col = (g0 + cg) * R + my_r;
            if (my_m < M && col < N) {
                if (DEQ) {
                    f16 yv = (f16)(my_sa * g.sb) * (f16)(float)sum;
                    if (bias) yv = yv + g.bi;
                    Y[(int64_t)my_m * N + col] = yv;
                } else {
                    C[(int64_t)my_m * N + col] = sum;
                }
            }
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) acc[v] = 0;
        cs = 0;
        ++cg;
    };
    Seg ga, gb, gc;
    fetch(ga);
    fetch(gb);
    fetch(gc);
    int it = 0;
    for (; it + 3 <= total; it += 3) {                      // whole turns of the ring: no branch around the loads
        consume(ga);
        fetch(ga);
        consume(gb);
        fetch(gb);
        consume(gc);
        fetch(gc);
    }
    if (it < total) consume(ga);
    if (it + 1 < total) consume(gb);
}

int launch_gemv(const void* A, const void* B, int M, int N, int Kb, void* C, void* Y, const void* sA, const void* sB,
                const void* bias, hipStream_t st) {
    const int groups = (N + 3) / 4;
    // row groups per wave: about 64 KB of weights per wave, but keep >= 8 waves per CU when N allows ...
    int ng = (65536 + 4 * Kb - 1) / (4 * Kb);
    const int cus = qr_device().cus;
    while (ng > 1 && groups / ng < 8 * cus) --ng;
    // ... and, when all workgroups are resident at once (up to five per CU), a count that spreads
    // evenly over the CUs: 3.5 workgroups per CU run as long as 4.  Among ng / 2 ... 2 ng the
    // value nearest to ng whose last round over the CUs is at least 97 % full, else the fullest.
    {
        auto fill = [&](int g) {
            const int wgs = ((groups + g - 1) / g + 3) / 4;
            if (wgs > 5 * cus) return 1.0;
            return (double)wgs / (double)(((wgs + cus - 1) / cus) * cus);
        };
        int best = ng;
        double best_fill = fill(ng);
        for (int d = 1; d <= ng && best_fill < 0.97; ++d) {
            const int cand[2] = {ng - d, ng + d};
            for (int c = 0; c < 2; ++c) {
                const int g = cand[c];
                if (g < 1 || 2 * g < ng || g > 2 * ng) continue;
                const double f = fill(g);
                if (f >= 0.97 ? best_fill < 0.97 : f > best_fill) {
                    best = g;
                    best_fill = f;
                }
            }
        }
        ng = best;
    }
    const int waves = (groups + ng - 1) / ng;
    const unsigned grid = (unsigned)((waves + 3) / 4);
#define QR_GEMV(MB)                                                                                                   \
    do {                                                                                                              \
        if (Y)                                                                                                        \
            gemv_i4_kernel<MB, true><<<dim3(grid), dim3(256), 0, st>>>((const uint8_t*)A, (const uint8_t*)B, M, N, Kb, \
                                                                       ng, nullptr, (f16*)Y, (const f16*)sA,          \
                                                                       (const f16*)sB, (const f16*)bias);             \
        else                                                                                                          \
            gemv_i4_kernel<MB, false><<<dim3(grid), dim3(256), 0, st>>>((const uint8_t*)A, (const uint8_t*)B, M, N,   \
                                                                        Kb, ng, (int32_t*)C, nullptr, nullptr,        \
                                                                        nullptr, nullptr);                            \
    } while (0)
    if (M <= 1) QR_GEMV(1);
    else if (M <= 2) QR_GEMV(2);
    else if (M <= 4) QR_GEMV(4);
    else QR_GEMV(8);
#undef QR_GEMV
    return qr_launch_status();
}

int launch_decode(const void* A, const void* B, int M, int N, int Kb, void* C, void* Y, const void* sA, const void* sB,
                  const void* bias, hipStream_t st, int kw = 0) {
#define QR_DEC(MT, SB, XL, PF, KW)                                                                                          \
    do {                                                                                                              \
        constexpr int STAGE = (1 + MT) * 32 * (SB / 16), RED = MT * 4 * 64;                                           \
        constexpr size_t LDS = (size_t)8 * (STAGE > RED ? STAGE : RED) * 16;                                          \
        hipError_t e;                                                                                                 \
        if (Y) {                                                                                                      \
            auto kern = decode_i4_kernel<MT, SB, XL, PF, KW, true>;                                                       \
            e = qr_allow_dynamic_lds((const void*)kern, LDS);                                                         \
            if (e != hipSuccess) return (int)e;                                                                       \
            kern<<<dim3((unsigned)((N + 32 * (8 / KW) - 1) / (32 * (8 / KW)))), dim3(512), LDS, st>>>(                \
                (const uint8_t*)A, (const uint8_t*)B, M, N, Kb, nullptr,                                              \
                                                     (f16*)Y, (const f16*)sA, (const f16*)sB, (const f16*)bias);      \
        } else {                                                                                                      \
            auto kern = decode_i4_kernel<MT, SB, XL, PF, KW, false>;                                                      \
            e = qr_allow_dynamic_lds((const void*)kern, LDS);                                                         \
            if (e != hipSuccess) return (int)e;                                                                       \
            kern<<<dim3((unsigned)((N + 32 * (8 / KW) - 1) / (32 * (8 / KW)))), dim3(512), LDS, st>>>(                \
                (const uint8_t*)A, (const uint8_t*)B, M, N, Kb, (int32_t*)C,                                          \
                                                     nullptr, nullptr, nullptr, nullptr);                             \
        }                                                                                                             \
    } while (0)
    // a load instruction carries eight rows of X (128-byte pieces): issue only those that exist
    // K is split KW ways within a row group (8 / KW row groups per workgroup).  One workgroup is
    // resident per CU, so the launch takes rounds(workgroups / 256) times a workgroup's time, which
    // is a fixed part (start, first loads, final sum: about six steps' worth) plus its steps per wave.
    if (kw == 0) {
        kw = 8;
        const int cus = qr_device().cus;
        if (M <= 32) {
            const int steps = (Kb + 127) / 128;
            double best = 0;
            for (int c = 8; c >= 2; c >>= 1) {
                const int wgs = (N + 32 * (8 / c) - 1) / (32 * (8 / c));
                const double cost = (double)((wgs + cus - 1) / cus) * (6.0 + (double)steps / c);
                if (c == 8 || cost < best) {
                    best = cost;
                    kw = c;
                }
            }
        }
    }
    if (M <= 8) {
        if (kw == 2) QR_DEC(1, 128, 1, 3, 2);
        else if (kw == 4) QR_DEC(1, 128, 1, 3, 4);
        else QR_DEC(1, 128, 1, 3, 8);
    } else if (M <= 16) {
        if (kw == 2) QR_DEC(1, 128, 2, 3, 2);
        else if (kw == 4) QR_DEC(1, 128, 2, 3, 4);
        else QR_DEC(1, 128, 2, 3, 8);
    } else if (M <= 32) {
        if (kw == 2) QR_DEC(1, 128, 4, 3, 2);
        else if (kw == 4) QR_DEC(1, 128, 4, 3, 4);
        else QR_DEC(1, 128, 4, 3, 8);
    } else if (M <= 48) QR_DEC(2, 128, 6, 3, 8);
    else QR_DEC(2, 128, 8, 3, 8);
#undef QR_DEC
    return qr_launch_status();
}

// Row groups per workgroup for the shared-token decode kernel: the count among 4 .. 8 with the least
// work on the busiest CU (rounds of workgroups over the CUs times groups per workgroup), larger counts first
// (fewer copies of the tokens' codes).  0: too few row groups to fill the CUs this way.
int decode_xs_groups(int N) {
    const int groups = (N + 31) / 32, cus = qr_device().cus;
    int best = 0, best_cost = 0;
    for (int rg = 8; rg >= 4; --rg) {
        const int wgs = (groups + rg - 1) / rg;
        if (wgs < cus * 3 / 4) continue;
        const int cost = ((wgs + cus - 1) / cus) * rg;
        if (best == 0 || cost < best_cost) {
            best = rg;
            best_cost = cost;
        }
    }
    return best;
}

int launch_decode_xs(const void* A, const void* B, int M, int N, int Kb, void* C, void* Y, const void* sA,
                     const void* sB, const void* bias, hipStream_t st, int rg) {
    const unsigned grid = (unsigned)(((N + 31) / 32 + rg - 1) / rg);
#define QR_XS(MT, R)                                                                                                  \
    do {                                                                                                              \
        constexpr int RD = 3;   /* deeper rings were measured slower (4: +3 %, 5: +6 %) */                            \
        constexpr size_t LDS = (size_t)3 * (MT * 32 * 16 + ((MT * 32 + R * 32 + 63) / 64 * 64 - MT * 32) * 8) * 16;       \
        hipError_t e;                                                                                                 \
        if (Y) {                                                                                                      \
            auto kern = decode_xs_kernel<MT, R, RD, true>;                                                            \
            e = qr_allow_dynamic_lds((const void*)kern, LDS);                                                         \
            if (e != hipSuccess) return (int)e;                                                                       \
            kern<<<dim3(grid), dim3(768), LDS, st>>>((const uint8_t*)A, (const uint8_t*)B, M, N, Kb, nullptr, (f16*)Y, \
                                                     (const f16*)sA, (const f16*)sB, (const f16*)bias);               \
        } else {                                                                                                      \
            auto kern = decode_xs_kernel<MT, R, RD, false>;                                                           \
            e = qr_allow_dynamic_lds((const void*)kern, LDS);                                                         \
            if (e != hipSuccess) return (int)e;                                                                       \
            kern<<<dim3(grid), dim3(768), LDS, st>>>((const uint8_t*)A, (const uint8_t*)B, M, N, Kb, (int32_t*)C,     \
                                                     nullptr, nullptr, nullptr, nullptr);                             \
        }                                                                                                             \
    } while (0)
#define QR_XS_R(MT)                                                                                                   \
    do {                                                                                                              \
        if (rg == 8) QR_XS(MT, 8);                                                                                    \
        else if (rg == 7) QR_XS(MT, 7);                                                                               \
        else if (rg == 6) QR_XS(MT, 6);                                                                               \
        else if (rg == 5) QR_XS(MT, 5);                                                                               \
        else QR_XS(MT, 4);                                                                                            \
    } while (0)
    if (M <= 32) QR_XS_R(1);
    else QR_XS_R(2);
#undef QR_XS_R
#undef QR_XS
    return qr_launch_status();
}

template <int BM, int BN, int WAVES_M, int WAVES_N>
int launch_cfg(const void* A, const void* B, int M, int N, int Kb, void* C, void* Y, const void* sA, const void* sB,
               const void* bias, hipStream_t st) {
    constexpr int NT = 64 * WAVES_M * WAVES_N;
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    const int64_t tiles = (int64_t)tiles_m * tiles_n;
    if (tiles > 0x3fffffff) return QR_E_SHAPE;
    const int nxcd = qr_device().xcds;                      // the grid is a whole number of rounds over the XCDs
    const unsigned grid = (unsigned)((tiles + nxcd - 1) / nxcd * nxcd);
    if (Y)
        gemm_i4_kernel<BM, BN, WAVES_M, WAVES_N, true><<<dim3(grid), dim3(NT), 0, st>>>(
            (const uint8_t*)A, (const uint8_t*)B, M, N, Kb, nullptr, (f16*)Y, (const f16*)sA, (const f16*)sB,
            (const f16*)bias, tiles_m, tiles_n, nxcd);
    else
        gemm_i4_kernel<BM, BN, WAVES_M, WAVES_N, false><<<dim3(grid), dim3(NT), 0, st>>>(
            (const uint8_t*)A, (const uint8_t*)B, M, N, Kb, (int32_t*)C, nullptr, nullptr, nullptr, nullptr, tiles_m,
            tiles_n, nxcd);
    return qr_launch_status();
}

// ---- K split across workgroups (shapes with too few tiles to fill the CUs) ------------------------
// y = fp16(fp16(sA[r] * sB[c]) * fp16(acc[r, c])) (+ bias[c] as a fourth rounded operation), acc = the sum
// of `slabs` partial products: the epilogue of the fused kernels, applied to the K slices' results.
// Four columns per thread when rows are whole groups of four.
__global__ __launch_bounds__(256) void dequant_slabs_kernel(const int32_t* __restrict__ part, int slabs,
                                                            const f16* __restrict__ sA, const f16* __restrict__ sB,
                                                            const f16* __restrict__ bias, int64_t M, int64_t N,
                                                            f16* __restrict__ Y) {
    const int64_t cells = M * N;
    const int64_t stride = (int64_t)gridDim.x * 256;
    if ((N & 3) == 0) {
        for (int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x; g < cells / 4; g += stride) {
            const int64_t i = g * 4, r = i / N, c = i - r * N;
            i32x4 acc = *(const i32x4*)(part + i);
            for (int s = 1; s < slabs; ++s) acc += *(const i32x4*)(part + (int64_t)s * cells + i);
            const f16 sa = sA[r];
            const f16x4 sb = *(const f16x4*)(sB + c);
            f16x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                f16 yv = (f16)(sa * sb[e]) * (f16)(float)acc[e];
                if (bias) yv = yv + bias[c + e];
                o[e] = yv;
            }
            *(f16x4*)(Y + i) = o;
        }
    } else {
        for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < cells; i += stride) {
            const int64_t r = i / N, c = i - r * N;
            int acc = part[i];
            for (int s = 1; s < slabs; ++s) acc += part[(int64_t)s * cells + i];
            f16 yv = (f16)(sA[r] * sB[c]) * (f16)(float)acc;
            if (bias) yv = yv + bias[c];
            Y[i] = yv;
        }
    }
}

// 8 .. 64 tokens against a weight with too few rows for the shared-token kernel: the barrier-free kernel, or 64 x 64 tiles in
// the STREAM form of gemm_mid_kernel, with K in slices over several workgroups (int32 slabs in the caller's scratch and a
// second launch that adds them) where that fills CUs.  In the barrier-free kernel every group of 32 weight rows pulls all the tokens'
// codes through its CU, which takes in some 60 GB/s, and a 64-row tile halves that; but its fixed path is shorter (one barrier).
// Estimates in microseconds, st = stages of 256 k, fitted to both kernels at 5 .. 64 tokens x 1041 .. 22016 weight rows x K = 1024
// .. 28672, with weights in the last-level cache and from memory (which differ by less than the kernels do):
//   barrier-free   3 + st (0.12 + 0.0028 M), 1.2 more for a second tile of tokens; up to 3.5 more between 4096 and 8192 rows where K is longer
//                  than the waves' rings; the whole times 0.8 + rows / 12500 beyond 8192 rows (less where K is short)
//   STREAM tiles   4.4 + st / slices x (0.235 + 0.0009 M up to 128 workgroups, 0.28 + 0.002 M up to a workgroup per CU,
//                  0.25 + 0.0012 M for each of several), at least the weights at 6.2 TB/s; slices: + 2.5, 0.3 for each beyond
//                  three, the slabs' way out and back at 4 TB/s, 4 where rows are no whole number of 16-byte pieces
// From memory, before / after: 48 x 12288 x 4096 14.2 / 9.1 us, 48 x 13824 x 5120 19.8 / 11.1, 48 x 22016 x 4096 20.6 / 13.5, 48 x 5120 x
// 13824 17.6 / 13.3, 48 x 4096 x 11008 14.9 / 12.0, 25 x 12288 x 8192 17.0 / 14.3; 32 x 4096 x 4096 stays (6.1 against 8.3).  Below eight tokens
// the two are within 5 % of each other where the tiles lead at all.  Slices only where three or more fit, or where two save 4 us
// (40 tokens and K = 16384 on): the scratch that callers are asked for grows with them.
// (The fit is older than the slices' four stage buffers.  4843 shapes of 8 .. 64 tokens with weights from memory: the choice costs 1.1 % more than the best, of
// which 0.3 is the readings' spread; 24 % and more in one of a hundred, wide weights with a short K: 35 x 21824 x 1536 in 15.8 us on the barrier-free
// kernel, 9.0 on tiles.)
struct DecodePlan {
    bool tiles;
    int split;
};
DecodePlan decode_plan(int64_t M, int64_t N, int64_t Kb, int64_t max_split) {
    DecodePlan best{false, 1};
    if (M < 8 || M > 64 || decode_xs_groups((int)N) != 0) return best;
    const int64_t cus = qr_device().cus, st = (Kb + 127) / 128, tiles = (N + 63) / 64;
    const double m = (double)M, s = (double)st;
    double t_best = 3.0 + s * (0.12 + 0.0028 * m) + (M > 32 ? 1.2 : 0.0);
    if (N > 8192) t_best = 3.0 + (t_best * (0.8 + (double)N / 12500.0) - 3.0) * (s < 16.0 ? s / 16.0 : 1.0);
    else if (N > 4096 && st > 24) t_best += 3.5 * (double)(N - 4096) / 4096.0;
    const int64_t most = tiles * 3 <= cus || (M >= 40 && Kb >= 8192) ? (max_split < 8 ? max_split : 8) : 1;
    for (int64_t ks = 1; ks <= most && (ks == 1 || (ks <= st / 4 && tiles * ks <= cus)); ++ks) {
        const int64_t wgs = tiles * ks;
        const double slope = wgs * 2 <= cus ? 0.235 + 0.0009 * m
                             : wgs <= cus   ? 0.28 + 0.002 * m : (0.25 + 0.0012 * m) * (double)((wgs + cus - 1) / cus);
        const double walk = (double)((st + ks - 1) / ks) * slope, stream = (double)N * (double)Kb / 6.2e6;
        double t = 4.4 + (walk > stream ? walk : stream);
        if (ks > 1) t += 2.5 + (ks > 3 ? 0.3 * (double)(ks - 3) : 0.0) + 2.0 * (double)ks * m * (double)N * 4.0 / 4.0e6 + (N % 4 ? 4.0 : 0.0);
        if (t < t_best) {
            t_best = t;
            best = DecodePlan{true, (int)ks};
        }
    }
    return best;
}

// How many int32 slabs of [M, N] a caller is asked to provide (qr_workspace_bytes).  Up to 64 tokens: what decode_plan uses.  For
// prompts of a few hundred tokens it is a contract, not a plan: these are the shapes and slices that the first kernel of this
// path could use (64 x 256 tiles: 6 us, 1.0 per stage and round of tiles, the slabs), and what earlier versions asked for, also of
// the callers of qr_linear_i4_f16_static.  mid_plan takes at most so many slices and, with tiles that fill the CUs by
// themselves, none at most of these shapes; qr_linear_plan says how many, which is what the Python package allocates.
int ks_split(int64_t M, int64_t N, int64_t Kb) {
    if (M <= 64) return decode_plan(M, N, Kb, 8).split;
    if (N <= 128) return 1;
    const int64_t tn = (N + 255) / 256;
    const int64_t cus = qr_device().cus;
    if (((M + 127) / 128) * tn >= cus / 2) return 1;
    const int64_t tiles = ((M + 63) / 64) * tn;
    const int64_t all_stages = (Kb + 127) / 128;
    const double t_unsplit = 6.0 + 1.0 * (double)all_stages * (double)((tiles + cus - 1) / cus);
    int best = 1;
    double t_best = 0.8 * t_unsplit;
    for (int64_t ks = 2; ks <= 16 && ks <= all_stages / 4; ++ks) {
        const double slabs_us = 2.0 * (double)ks * (double)M * (double)N * 4.0 / 4.0e6;
        const double t = 8.0 + 1.0 * (double)((all_stages + ks - 1) / ks) * (double)((tiles * ks + cus - 1) / cus) + slabs_us;
        if (t < t_best) {
            t_best = t;
            best = (int)ks;
        }
    }
    return best;
}

// Which kernel takes an output of more than 64 tokens, by an estimate in microseconds (st = stages of 256 k, n = tiles on the
// busiest of the CUs):
//   64 x 64 tiles   3.9 + st 0.264 (n = 1; 0.30 heavy), 4.6 + st 0.42 (n = 2; 0.46 heavy), 3.9 + n (0.75 + 0.21 st) beyond (0.60 for 0.75 at n = 3):
//                   three workgroups share a CU; heavy = K > 8192 and weights over 36 MB: 0.23 for 0.21 from n = 5 on, and 0.25 where K > 4096
//                   and weights are over 96 MB: they are read once per 64 tokens there and once per 128 or more by the larger tiles, from
//                   memory (111 x 28736 x 9024 63 us, 45 on 128 x 128 tiles; with 72 MB, which the last-level cache keeps, 27 / 31).
//   96 x 64         5.1 + st 0.325 (n = 1; 0.37 heavy), 8.0 + st 0.69 (n = 2; 0.85 for one row of tiles, none of whose weights is shared), 5.1 + n (2.0 + 0.335 st)
//   64 x 128        4.9 + st 0.40 (n = 1), 7.6 + st 0.90 (n = 2), 4.9 + n (2.4 + 0.453 st)
//   128 x 128       5.5 + st 0.73 (n = 1; int32 6.2), 9.7 + st 1.50 (n = 2), 5.5 + n (3.6 + 0.755 st)
//   128 / 192 / 256 x 256 (e2m3 kernels)   1.7 + n ({8.1, 6.8, 8.9} + {0.99, 1.56, 1.76} st (1 - {0.25, 0.18, 0.22} idle)), idle = share of
//                   the rounds' places without a tile (the clock is higher then)
//   256 and 128     whole rounds of 256-row tiles and the rest as 128-row ones in the same launch, where that rest is at most half a round
// and what the output adds.  The small tiles put whole tiles of 16-byte pieces out as lines and anything else element by element; the
// e2m3 kernels' stores drop what lies beyond the edge.  A last column of tiles that the edge cuts, by the columns left in it: 0.07 us each
// up to 3.2, 3.3 (96 x 64), 0.045 up to 3.3, 0.085 up to 5.7 for the four small shapes (133 x 11112 x 1024 9.1 us on 64 x 64 tiles, 14.4 on
// 128 x 128, which the estimate without it took), none for the large ones; rows of no whole pieces (N % 8): 3.5 / 4 / 4 / 6 and 0.8 us per
// million elements, 3 / 5.5 / 7.5 for the large ones (5.5 for 256 and 128); rows that start within a line (N % 64): 0.20 / 0.35 / 0.40 us
// per million elements for the large ones; int32 sums: 1.8 / 2.8 / 3.2 for the large ones, 6 more where N % 4.  Outputs of more than 100 MB leave the
// last-level cache: 0.19 / 0.5 / 0.23 / 0.08 us per MB beyond for the small shapes, whose stores come in smaller pieces.
// Fitted with every kernel forced, weights from memory and from cache, to 3600 shapes of 65 .. 8192 tokens x 64 .. 28672 weight rows at
// K = 64 .. 28672, three quarters of them of whole lines, 1200 of N = 128 .. 28672 in steps of 8, 108 of 4.2 million rows and more, and 700
// of few tiles and a long K with up to eight slices.  The choice costs 0.2 % more than the best of all kernels (geometric mean; 0.1 % up to
// K = 1536, 0.3 % at N in steps of 8, 0.7 % where K may be sliced; without the output's terms and those of heavy weights 1.6, 3.2, 1.9 and
// 1.1 %, 2 x at worst).
// The fit is older than the fourth stage buffer of 64 x 64 tiles with a CU each, which take up to 14 % less from memory than it says.  Of the present
// kernels, 814 shapes of 65 .. 1500 tokens with weights from memory: the choice, spread operands among them, costs 1.2 % more than the best (the readings'
// own spread is 0.5 of it), 3 % or more in one of ten, 23 % at worst (268 x 8232 x 8768, on 64 x 64 tiles instead of 128 x 128).
// The small tiles are bound by the CUs' intake of operands, the large ones by instruction issue and power, so the small ones lead
// while the large ones leave CUs idle: 333 x 4096 x 4096 11.2 us against 22, 777 x 4096 x 4096 17.7 (22), 512 x 8192 x 8192 32.1 (34).
// Very few tiles and a long K: slices of K over several workgroups with int32 slabs in the caller's scratch and a second
// launch that adds them (+ 3 us, 4.5 more where N % 4, and the slabs' way out and back at 4 TB/s).
struct MidPlan {
    int kernel;         // 0 .. 2: qr_internal_gemm_mid's shapes; 3 .. 6: qr_internal_gemm_e2m3's; 7: 96 x 64 tiles
    int split;
    double us;
};
MidPlan mid_plan(int64_t M, int64_t N, int64_t Kb, int64_t max_split, bool fp16) {
    const int64_t cus = qr_device().cus;
    const double st = (double)((Kb + 127) / 128);
    auto tiles = [&](int64_t bm, int64_t bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
    auto loaded = [&](int64_t t) { return (double)((t + cus - 1) / cus); };
    const bool heavy = Kb > 4096 && N * Kb > 36000000, stream = Kb > 2048 && N * Kb > 96000000;
    const bool odd = fp16 && N % 8 != 0;                    // rows of the output of no whole 16-byte pieces
    const double elements = (double)M * (double)N * 1e-6, megabytes = elements * (fp16 ? 2.0 : 4.0);
    const double far = megabytes > 100.0 ? megabytes - 100.0 : 0.0;
    // what the output adds on the small tiles: a last column that the edge cuts, rows of no whole pieces, what leaves the caches
    auto put = [&](int64_t bn, double column, double most, double ragged, double beyond) {
        const double cut = fp16 ? column * (double)(N % bn) : 0.0;
        return far * beyond + (odd ? ragged + 0.8 * elements : cut < most ? cut : most);
    };
    auto t64 = [&](int64_t t, double stages) {
        const double n = loaded(t);
        if (n <= 2) return n == 1 ? 3.9 + (heavy ? 0.30 : 0.264) * stages : 4.6 + (heavy ? 0.46 : 0.42) * stages;
        return 3.9 + n * ((n == 3 ? 0.60 : 0.75) + (stream ? 0.25 : n >= 5 && heavy ? 0.23 : 0.21) * stages);
    };
    MidPlan best{0, 1, t64(tiles(64, 64), st) + put(64, 0.07, 3.2, 3.5, 0.19)};
    auto consider = [&](int kernel, int split, double t) {
        if (t < best.us) best = MidPlan{kernel, split, t};
    };
    const double n96 = loaded(tiles(96, 64));
    consider(7, 1, put(64, 0.4, 3.3, 4.0, 0.5) + (n96 == 1 ? 5.1 + (heavy ? 0.37 : 0.325) * st : n96 == 2 ? 8.0 + (M <= 96 ? 0.85 : 0.69) * st : 5.1 + n96 * (2.0 + 0.335 * st)));
    const double n128 = loaded(tiles(64, 128)), nsq = loaded(tiles(128, 128));
    consider(1, 1, put(128, 0.045, 3.3, 4.0, 0.23) + (n128 == 1 ? 4.9 + 0.40 * st : n128 == 2 ? 7.6 + 0.90 * st : 4.9 + n128 * (2.4 + 0.453 * st)));
    consider(2, 1, put(128, 0.085, 5.7, 6.0, 0.08) + (nsq == 1 ? (fp16 ? 5.5 : 6.2) + 0.73 * st : nsq == 2 ? 9.7 + 1.50 * st : 5.5 + nsq * (3.6 + 0.755 * st)));
    const double fixed[3] = {8.1, 6.8, 8.9}, slope[3] = {0.99, 1.56, 1.76}, easier[3] = {0.25, 0.18, 0.22};
    const double within[4] = {0.20, 0.35, 0.40, 0.40}, ragged[4] = {3.0, 5.5, 7.5, 5.5}, sums[4] = {1.8, 2.8, 3.2, 3.2};      // (the last: 256 and 128)
    auto round = [&](int i, double idle) { return fixed[i] + slope[i] * st * (1.0 - easier[i] * idle); };
    auto put256 = [&](int i) { return odd ? ragged[i] : fp16 ? (N % 64 != 0 ? within[i] * elements : 0.0) : sums[i] + (N % 4 != 0 ? 6.0 : 0.0); };
    auto reach = [&](int64_t rows) { return qr_e2m3_reach(rows, N, fp16); };
    for (int i = 2; i >= 0; --i) {                          // (ties go to the taller tile)
        if (!reach(128 + 64 * i)) continue;
        const int64_t t = tiles(128 + 64 * i, 256);
        const double n = loaded(t);
        consider(3 + i, 1, 1.7 + put256(i) + n * round(i, 1.0 - (double)t / (n * (double)cus)));
    }
    const int64_t whole = tiles(256, 256) / cus, left = tiles(256, 256) % cus;
    if (reach(256) && Kb > 128 && cus % qr_device().xcds == 0 && whole > 0 && left > 0 && 2 * left <= cus)
        consider(6, 1, 1.7 + put256(3) + (double)whole * round(2, 0.0) + round(0, 1.0 - 2.0 * (double)left / (double)cus));
    const int64_t all_stages = (Kb + 127) / 128;
    for (int64_t ks = 2; ks <= max_split && ks <= all_stages / 4; ++ks)
        consider(0, (int)ks, t64(tiles(64, 64) * ks, (double)((all_stages + ks - 1) / ks)) + (N % 4 != 0 ? 7.5 : 3.0) +
                                 2.0 * (double)ks * (double)M * (double)N * 4.0 / 4.0e6);
    return best;
}

// The same product with the operand of fewer rows spread in memory first (gemm_x6.hip), by tiles of 256 rows of the other operand and 32 nx of
// that one, in microseconds: 5.8 + 0.307 per MB that is written, n times (0.26 + 0.675 nx) (1 - 0.23 idle) + st times a stage of (0.406 + 0.144 nx)
// (1 - 0.285 idle), and 0.25 per million elements where rows of the output start within a line.  Where x is spread and the weights stay packed, they
// come from memory: a stage takes 1.15 at least (with two stage buffers each is asked for one stage ahead; 1.05 where a CU has several tiles, whose
// first stages come under the tile before), all of them what their bytes take at 5 TB/s.  Without these limits, which the last-level cache hides,
// prompts of 65 .. 550 tokens against wide weights took this way: 400 tokens x 13824 x 5120 35.6 us, 29.7 without, 200 x 27648 x 5120 36.5 / 31.8,
// 512 x 11008 x 4096 27.1 / 23.6, 100 x 57344 x 8192 63.7 / 60.0 (out of that cache they lose 4 % by the limits).
// The terms are fitted to 2200 shapes of 100 .. 32768 tokens x 512 .. 57344 weight rows, 1e9 .. 6e12 operations, all five nx forced; the limits and
// the lead of 1.2 us that it must have over mid_plan's kernels to 8693 more of 65 .. 32768 tokens, every nx forced, weights from memory and from cache, codes
// uniform and as quantisers leave them (Gaussian: with few bits toggling, these kernels' clock is higher).  With the latter, from memory the choice
// is 1.073 x as fast as without these kernels (1.076 with the best of all; 1.062 without the limits, when a seventh of the shapes that took them
// were 3 % and more slower, by up to 25 %; now a hundredth, 14 % at worst), from cache 1.103 x (1.109, 1.106).  With uniform codes 1.044 and 1.066 x.
// About half of the shapes take them, nine in ten from 3e11 operations on.
// What it does not take: rows of the output that are no whole 16-byte pieces, a K of one stage, scratch beyond 512 MiB (a weight of 26000 x 26000).
struct SpreadPlan {
    int nx;             // 4 .. 8; 0: not this way
    double us;
};
SpreadPlan spread_plan(int64_t M, int64_t N, int64_t Kb) {
    SpreadPlan best{0, 0.0};
    const int64_t rows = N <= M ? N : M, others = N <= M ? M : N, cus = qr_device().cus;
    const int64_t bytes = (int64_t)qr_internal_x6_bytes(rows, Kb);
    if (Kb <= 128 || N % 8 != 0 || bytes > (512LL << 20) || !qr_e2m3_reach(256, N, true)) return best;
    const double st = (double)((Kb + 127) / 128), fixed = 5.8 + 0.307e-6 * (double)bytes + (N % 64 != 0 ? 0.25e-6 * (double)M * (double)N : 0.0);
    const double bytes_us = (double)N * (double)Kb / 5.0e6;
    for (int nx = 8; nx >= 4; --nx) {
        const int64_t tiles = ((others + 255) / 256) * ((rows + 32 * nx - 1) / (32 * nx));
        const double n = (double)((tiles + cus - 1) / cus), idle = 1.0 - (double)tiles / (n * (double)cus);
        const double stage = (0.406 + 0.144 * nx) * (1.0 - 0.285 * idle);
        const double least = N <= M ? 0.0 : n > 1.0 ? 1.05 : 1.15;
        double walk = n * st * (stage < least ? least : stage);
        if (N > M && walk < bytes_us) walk = bytes_us;
        const double t = fixed + n * (0.26 + 0.675 * nx) * (1.0 - 0.23 * idle) + walk;
        if (best.nx == 0 || t < best.us) best = SpreadPlan{nx, t};
    }
    return best;
}

// The kernel that takes a shape, with so many bytes of scratch, and the slices of K that it runs in.  (pieces: the output is 16-byte aligned.)
enum class Gemm { large, gemv, shared_tokens, decode, stream64, mid64, mid64x128, mid128, spk, sp192, sp256, sp256_tail, mid96, x6 };
struct GemmPlan {
    Gemm kernel;
    int split;          // (x6: nx)
    size_t scratch;
};
GemmPlan gemm_plan(int64_t M, int64_t N, int64_t Kb, size_t scratch, bool fp16, bool pieces = true) {
    // An operand of 4 GiB or more: every specialised kernel below addresses its operands through 32-bit offsets;
    // the plain tiled kernel computes 64-bit row addresses and takes any shape (rows beyond M or N are clamped).
    if (M * Kb >= (1LL << 32) || N * Kb >= (1LL << 32)) return GemmPlan{Gemm::large, 1, 0};
    const size_t slab = (size_t)M * (size_t)N * 4;
    const int64_t max_split = scratch ? (int64_t)(scratch / slab) : 1;
    auto sliced = [&](Gemm kernel, int split) { return GemmPlan{kernel, split, split > 1 ? slab * (size_t)split : 0}; };
    if (M > 64) {
        const MidPlan plan = mid_plan(M, N, Kb, max_split, fp16);
        constexpr Gemm kernels[] = {Gemm::mid64, Gemm::mid64x128, Gemm::mid128, Gemm::spk, Gemm::sp192, Gemm::sp256, Gemm::sp256_tail, Gemm::mid96};
        const size_t x6 = fp16 && pieces && scratch ? qr_internal_x6_bytes(N <= M ? N : M, Kb) : 0;
        if (x6 && x6 <= scratch) {
            const SpreadPlan spread = spread_plan(M, N, Kb);
            if (spread.nx && spread.us + 1.2 < plan.us) return GemmPlan{Gemm::x6, spread.nx, x6};
        }
        return sliced(kernels[plan.kernel], plan.split);
    }
    // one to four tokens: the dot-product kernel -- except two to four tokens against a weight with enough rows for the
    // shared-token kernel, which is ahead there (57344 x 8192: 40.2 against 42.9 us)
    const bool xs = decode_xs_groups((int)N) != 0;
    if (M == 1 || (M <= 4 && !xs)) return GemmPlan{Gemm::gemv, 1, 0};
    const DecodePlan plan = decode_plan(M, N, Kb, max_split);
    if (plan.tiles) return sliced(Gemm::stream64, plan.split);
    // weight streaming: with enough groups of 32 rows to fill the CUs the kernel that shares the
    // tokens' codes through LDS (they are read once per workgroup); otherwise the barrier-free
    // kernel in which the waves of a workgroup split K over groups of 32 rows
    return GemmPlan{xs ? Gemm::shared_tokens : Gemm::decode, 1, 0};
}

int gemm_dispatch(const void* A, const void* B, int64_t M, int64_t N, int64_t K, void* C, void* Y, const void* sA,
                  const void* sB, const void* bias, hipStream_t st, void* ws = nullptr, size_t ws_bytes = 0) {
    if (M < 0 || N < 0 || K < 0) return QR_E_SHAPE;
    if (M == 0 || N == 0) return QR_OK;
    if (K == 0 || K % 64 != 0 || K > 131008 || M > 0x7fffffff || N > 0x7fffffff) return QR_E_SHAPE;
    if (!A || !B || (!C && !Y)) return QR_E_NULL;
    if (((uintptr_t)A & 15) || ((uintptr_t)B & 15)) return QR_E_ALIGN;
    if (Y ? ((uintptr_t)Y & 7) : ((uintptr_t)C & 15)) return QR_E_ALIGN;
    const int m = (int)M, n = (int)N, kb = (int)(K / 2);
    // the slabs of a K split and a spread operand go to scratch from the caller; without it (or with too little) the single-launch kernels run
    const bool scratch = Y && ws && ((uintptr_t)ws & 15) == 0;
    const GemmPlan plan = gemm_plan(M, N, kb, scratch ? ws_bytes : 0, Y != nullptr, ((uintptr_t)Y & 15) == 0);
    if (plan.kernel == Gemm::x6) return qr_internal_gemm_x6(plan.split, A, B, m, n, kb, Y, sA, sB, bias, ws, st);
    const int mid = plan.kernel == Gemm::stream64 ? 3 : plan.kernel == Gemm::mid96 ? 4 : (int)plan.kernel - (int)Gemm::mid64;      // qr_internal_gemm_mid's shape
    if (plan.split > 1) {
        const int rc = qr_internal_gemm_mid(mid, A, B, m, n, kb, ws, nullptr, nullptr, nullptr, nullptr, st, plan.split);
        if (rc != QR_OK) return rc;
        int64_t db = (M * N / 4 + 255) / 256;
        db = db < 1 ? 1 : (db > 4096 ? 4096 : db);
        dequant_slabs_kernel<<<dim3((unsigned)db), dim3(256), 0, st>>>((const int32_t*)ws, plan.split, (const f16*)sA,
                                                                      (const f16*)sB, (const f16*)bias, M, N, (f16*)Y);
        return qr_launch_status();
    }
    switch (plan.kernel) {
        case Gemm::large:
            if (M <= 128) return launch_cfg<128, 128, 2, 2>(A, B, m, n, kb, C, Y, sA, sB, bias, st);
            return launch_cfg<256, 256, 4, 2>(A, B, m, n, kb, C, Y, sA, sB, bias, st);
        case Gemm::gemv: return launch_gemv(A, B, m, n, kb, C, Y, sA, sB, bias, st);
        case Gemm::shared_tokens: return launch_decode_xs(A, B, m, n, kb, C, Y, sA, sB, bias, st, decode_xs_groups(n));
        case Gemm::decode: return launch_decode(A, B, m, n, kb, C, Y, sA, sB, bias, st);
        case Gemm::spk:
        case Gemm::sp192:
        case Gemm::sp256:
        case Gemm::sp256_tail:
            return qr_internal_gemm_e2m3((int)plan.kernel - (int)Gemm::spk, A, B, m, n, kb, C, Y, sA, sB, bias, st);
        default: return qr_internal_gemm_mid(mid, A, B, m, n, kb, C, Y, sA, sB, bias, st, 1);
    }
}

}  // namespace

extern "C" int qr_matmul_i4_i32(const void* A, const void* B, int64_t M, int64_t N, int64_t K, void* C, void* stream) {
    if (M > 0 && N > 0 && !C) return QR_E_NULL;
    return gemm_dispatch(A, B, M, N, K, C, nullptr, nullptr, nullptr, nullptr, (hipStream_t)stream);
}

extern "C" int qr_linear_i4_f16(const void* A, const void* sA, const void* W, const void* sW, const void* bias_or_null,
                                int64_t M, int64_t N, int64_t K, void* y, void* stream) {
    if (M > 0 && N > 0 && (!y || !sA || !sW)) return QR_E_NULL;
    return gemm_dispatch(A, W, M, N, K, nullptr, y, sA, sW, bias_or_null, (hipStream_t)stream);
}

extern "C" size_t qr_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 64 != 0) return 0;
    const int split = ks_split(M, N, K / 2);
    return split > 1 ? (size_t)split * (size_t)M * (size_t)N * 4 : 0;
}

extern "C" size_t qr_linear_spread_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 64 || N <= 0 || K <= 0 || K % 64 != 0 || K > 131008 || M > 0x7fffffff || N > 0x7fffffff) return 0;
    const size_t slabs = qr_workspace_bytes(M, N, K), x6 = qr_internal_x6_bytes(N <= M ? N : M, K / 2);
    const GemmPlan plan = gemm_plan(M, N, K / 2, x6 > slabs ? x6 : slabs, true);
    return plan.kernel == Gemm::x6 ? plan.scratch : 0;
}

extern "C" const char* qr_linear_plan(int64_t M, int64_t N, int64_t K, size_t workspace_bytes, size_t* scratch_bytes) {
    if (scratch_bytes) *scratch_bytes = 0;
    if (M <= 0 || N <= 0 || K <= 0 || K % 64 != 0 || K > 131008 || M > 0x7fffffff || N > 0x7fffffff) return nullptr;
    const GemmPlan plan = gemm_plan(M, N, K / 2, workspace_bytes, true);
    const bool slices = plan.scratch > 0;
    if (scratch_bytes) *scratch_bytes = plan.scratch;
    switch (plan.kernel) {
        case Gemm::large: return "gemm_i4_kernel";
        case Gemm::gemv: return "gemv_i4_kernel";
        case Gemm::shared_tokens: return "decode_xs_kernel";
        case Gemm::decode: return "decode_i4_kernel";
        case Gemm::stream64:
        case Gemm::mid64: return slices ? "gemm_mid_kernel<64,64> (K sliced) + dequant_slabs_kernel" : "gemm_mid_kernel<64,64>";
        case Gemm::mid96: return "gemm_mid_kernel<96,64>";
        case Gemm::mid64x128: return "gemm_mid_kernel<64,128>";
        case Gemm::mid128: return "gemm_mid_kernel<128,128>";
        case Gemm::spk: return "gemm_spk_kernel";
        case Gemm::sp192:
        case Gemm::sp256: return "gemm_sp256_kernel";
        case Gemm::sp256_tail: return "gemm_sp256_tail_kernel";
        case Gemm::x6: {
            static const char* const names[2][5] = {
                {"spread_x6_kernel + gemm_x6_kernel<128,256> (x spread)", "spread_x6_kernel + gemm_x6_kernel<160,256> (x spread)",
                 "spread_x6_kernel + gemm_x6_kernel<192,256> (x spread)", "spread_x6_kernel + gemm_x6_kernel<224,256> (x spread)",
                 "spread_x6_kernel + gemm_x6_kernel<256,256> (x spread)"},
                {"spread_x6_kernel + gemm_x6_kernel<256,128> (W spread)", "spread_x6_kernel + gemm_x6_kernel<256,160> (W spread)",
                 "spread_x6_kernel + gemm_x6_kernel<256,192> (W spread)", "spread_x6_kernel + gemm_x6_kernel<256,224> (W spread)",
                 "spread_x6_kernel + gemm_x6_kernel<256,256> (W spread)"}};
            return names[N <= M][plan.split - 4];
        }
    }
    return nullptr;
}

// ---- the entry point that allocates nothing ---------------------------------------------------------
// Slabs of int32 partial sums for the K split, held by the library itself: one array per GPU, alive
// until the process ends.  Host code must never hand the array's NAME to a kernel (in host code it is a
// stand-in, not a device address): the per-device address comes from hipGetSymbolAddress, once per
// device, and only that pointer is used afterwards.
static __device__ __align__(256) unsigned char scratch[QR_STATIC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
void* scratch_ptr[kMaxDevices];                 // per device: its own copy of `scratch`, at its own address
std::mutex scratch_guard;

// Address of `scratch` on the current device (looked up on the first call on that device).
int static_scratch(void** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= kMaxDevices) return QR_E_UNSUPPORTED;
    std::lock_guard<std::mutex> lock(scratch_guard);
    if (!scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return (int)e;
        if (!p) return (int)hipErrorInvalidSymbol;
        scratch_ptr[dev] = p;
    }
    *out = scratch_ptr[dev];
    return QR_OK;
}
}  // namespace

extern "C" int qr_linear_i4_f16_static(const void* A, const void* sA, const void* W, const void* sW,
                                       const void* bias_or_null, int64_t M, int64_t N, int64_t K, void* y, void* stream) {
    if (M > 0 && N > 0 && (!y || !sA || !sW)) return QR_E_NULL;
    // Decode batches use the buffer from 40 tokens and K = 16384 on only, as the header promises, though decode_plan would slice K
    // from 8 tokens on: calls of the other sizes share nothing and may overlap.
    const size_t need = M > 64 || (M >= 40 && K >= 16384) ? qr_workspace_bytes(M, N, K) : 0;
    if (need > (size_t)QR_STATIC_SCRATCH_BYTES) return QR_E_SCRATCH_LIMIT;
    void* ws = nullptr;
    if (need) {                                  // every slab cell is written before it is read: nothing to clear
        const int rc = static_scratch(&ws);
        if (rc != QR_OK) return rc;
    }
    return gemm_dispatch(A, W, M, N, K, nullptr, y, sA, sW, bias_or_null, (hipStream_t)stream, ws, need);
}

extern "C" int qr_linear_i4_f16_ws(const void* A, const void* sA, const void* W, const void* sW,
                                   const void* bias_or_null, int64_t M, int64_t N, int64_t K, void* y, void* workspace,
                                   size_t workspace_bytes, void* stream) {
    if (M > 0 && N > 0 && (!y || !sA || !sW)) return QR_E_NULL;
    return gemm_dispatch(A, W, M, N, K, nullptr, y, sA, sW, bias_or_null, (hipStream_t)stream, workspace, workspace_bytes);
}
